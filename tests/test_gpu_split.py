"""LUMA_FLAG_SPLIT: records of a small set split into parts, and its medium
tensors in a workgroup each or in wavefronts beside the parts.  The parts
change which threads step an element and nothing else, so a split launch
equals the unsplit one bit for bit; the unsplit routes (one wavefront per medium tensor among them) are compared
with the oracle here, the split ones by every other parity test."""

import pytest
import torch

from config_util import SampledPair, normal_grad
from luma_amd import LUMA
from luma_amd import _lib as L
from luma_amd import functional as F

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda")
MEDIUM = [513, 600, 2047, 2048, 2049, 4095, 4097, 8191, 8192, 8193, 1, 257, 256, 70000, 9000]
# parts of 2,048 / 4,096 / 8,192 elements, records not split, edges of each
SETS = {
    "one element": [1],
    "edges": [2047, 2048, 2049, 4095, 4096, 4097, 8191, 8193, 16383, 16384, 16385, 256, 257, 3],
    "small only": [1, 200, 256] * 3,
    "parts of 4096": [700001, 300, 90000],
    "parts of 8192": [5000003, 12000, 100],
    "many": [300 + 37 * i for i in range(250)] + [16385] * 30 + [9] * 100,
    "wide, parts of 8192": [20000] * 60 + [300 + 52 * i for i in range(150)],
    "medium wavefronts beside parts": [16385] * 60 + [300 + i for i in range(150)] + [9] * 30,
    "medium only, wide and split": [257 + 80 * i for i in range(99)],
    "medium only, wavefronts": [257 + i % 256 for i in range(701)],
}
# the part length, and whether the medium tensors take a workgroup each
PLANS = {
    "one element": (16384, False),
    "edges": (2048, True),
    "small only": (16384, False),
    "parts of 4096": (4096, True),
    "parts of 8192": (8192, False),
    "many": (16384, True),
    "wide, parts of 8192": (8192, True),
    "medium wavefronts beside parts": (4096, False),
    "medium only, wide and split": (4096, True),
    "medium only, wavefronts": (16384, False),
}


def _pair(sizes, dtype, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    a = [(torch.randn(n, device=DEV, generator=gen) * 0.02).requires_grad_(True) for n in sizes]
    b = [p.detach().clone().requires_grad_(True) for p in a]
    for p in a + b:
        p.grad_dtype = None
    oa, ob = LUMA(a, lr=1e-3, weight_decay=0.01), LUMA(b, lr=1e-3, weight_decay=0.01)
    ob._base_seed = oa._base_seed

    def step(t):
        for p, q in zip(a, b):
            g = normal_grad(p.shape, 1e-3, gen, DEV, dtype, outliers=1e-2, zeros=0.01)
            p.grad, q.grad = g, g.clone()
        oa.step()
        ob.step()
        torch.cuda.synchronize()
        sa, sb = oa.state_dict()["state"], ob.state_dict()["state"]
        for i, (p, q) in enumerate(zip(a, b)):
            assert torch.equal(sa[i]["Q_m"], sb[i]["Q_m"]), (t, i)
            assert torch.equal(sa[i]["Q_w"], sb[i]["Q_w"]), (t, i)
            assert sa[i]["S_m"] == sb[i]["S_m"] and sa[i]["S_v"] == sb[i]["S_v"], (t, i)
            assert torch.equal(p.detach(), q.detach()), (t, i)
    return oa, ob, step


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("name", list(SETS))
def test_split_equals_unsplit(name, dtype):
    print("case", name, dtype, flush=True)
    oa, ob, step = _pair(SETS[name], dtype, 31)
    ob._get_engine(next(iter(ob.param_groups[0]["params"])).device).split = False
    for t in range(4):
        step(t)
    assert (oa._engine._chunk, oa._engine._wide) == PLANS[name]
    assert (ob._engine._chunk, ob._engine._wide) == (16384, False)


def test_split_changes_between_steps():
    """Code summaries of one part length are not read with another."""
    oa, ob, step = _pair(SETS["edges"] + [70000], torch.float32, 32)
    step(0)
    for t, on in enumerate([True, False, True, True, False], 1):
        ob._engine.split = on
        step(t)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_unsplit_routes_match_oracle(dtype):
    gen = torch.Generator(device=DEV).manual_seed(33)
    params = [torch.randn(n, device=DEV, generator=gen) * 0.02 for n in MEDIUM]
    pair = SampledPair(params, range(len(MEDIUM)))
    pair.opt._get_engine(params[0].device).split = False
    for t in range(1, 5):
        g = torch.Generator(device=DEV).manual_seed(800 + t)
        gd = [normal_grad(p.shape, 1e-3, g, DEV, dtype, outliers=1e-2, zeros=0.02)
              for p in pair.params]
        pair.step(gd, {i: x.cpu() for i, x in enumerate(gd)})
        pair.check()


@pytest.mark.parametrize("n", [1, 2047, 16385, 62 * 16384 + 5, 4185079])
def test_per_tensor_op_equals_step(n):
    gen = torch.Generator(device=DEV).manual_seed(n)
    p = (torch.randn(n, device=DEV, generator=gen) * 0.02).requires_grad_(True)
    q = p.detach().clone()
    opt = LUMA([p], lr=1e-3, weight_decay=0.01)
    q_m = torch.zeros(n, dtype=torch.int16, device=DEV)
    q_w = torch.zeros(n, dtype=torch.int16, device=DEV)
    slot = F.new_slot(DEV)
    for t in range(3):
        p.grad = torch.randn(n, device=DEV, generator=gen) * 1e-3
        opt.step()
        F.luma_step(q, p.grad, q_m, q_w, slot, 0.9, 0.999, 1e-8, 1e-3, 0.01, 0, opt._base_seed)
        assert torch.equal(p.detach(), q), t
        s = opt.state_dict()["state"][0]
        assert torch.equal(s["Q_m"], q_m) and torch.equal(s["Q_w"], q_w), t
        assert F.slot_state(slot) == (s["step"], s["S_m"], s["S_v"]), t


def test_planned_steps_take_the_split_of_their_table():
    """How a set is split is worked out when its table changes or a setting
    does, not on each step (a step of a few tensors is host-bound)."""
    oa, ob, step = _pair(SETS["edges"], torch.float32, 34)
    step(0)
    step(1)
    calls = []
    eng = oa._engine
    splits = eng._splits
    eng._splits = lambda: calls.append(1) or splits()
    for p in oa.param_groups[0]["params"]:
        p.grad = torch.zeros_like(p)
    oa.step()                    # a planned step whose gradients moved
    oa.step()                    # and one where nothing did
    assert not calls and eng._chunk == 2048
    eng.split = False
    oa.step()
    assert calls and eng._chunk == 16384
