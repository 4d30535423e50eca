"""The finalize launch's split of a table: tensors of more than four chunks
take a workgroup (64 tensors looked at together, more than 1,024 tensors
shared out among 1,024 workgroups), the others a lane per role.  Tensors of
both kinds at the ends and edges of the table, against the oracle."""

import pytest
import torch

from config_util import SampledPair, normal_grad

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda")
CHUNK = 2048


@pytest.mark.parametrize("count", [1, 3, 1024, 1030, 66000])
def test_tensors_of_many_and_few_chunks(count):
    # 5 and 9 chunks (a workgroup), 4 and 1 (a lane), the rest one element
    special = {0: 5 * CHUNK - 1, 1: 4 * CHUNK, 1023: 9 * CHUNK, 1024: 4 * CHUNK + 1,
               1025: CHUNK + 1, 65535: 4 * CHUNK + 8, 65536: 8 * CHUNK + 3,
               count - 2: 3, count - 1: 6 * CHUNK}
    sizes = [special.get(i, 1) for i in range(count)]
    gen = torch.Generator(device=DEV).manual_seed(count)
    params = (torch.randn(sum(sizes), device=DEV, generator=gen) * 0.02).split(sizes)
    params = [p.clone() for p in params]
    sample = [i for i in sorted(set(special)) if 0 <= i < count]
    pair = SampledPair(params, sample)
    pair.opt._get_engine(params[0].device).chunk_elems = CHUNK
    for t in range(1, 4):
        g = torch.Generator(device=DEV).manual_seed(900 + t)
        flat = normal_grad((sum(sizes),), 1e-3, g, DEV, torch.float32, outliers=1e-2)
        gd = list(flat.split(sizes))
        pair.step(gd, {i: gd[i].cpu() for i in sample})
        pair.check()
