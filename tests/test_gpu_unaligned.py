"""Tensors that start anywhere in memory (views of packed buckets or flat
buffers, aligned to their elements only) step like aligned copies of them,
bit for bit: the gradient, the parameter, the codes and injected uniforms,
each at offsets of 0 to 7 elements, in every gradient type: through the
per-tensor op (one workgroup and several chunks), and through the optimizer
the small tensors' route and the medium tensors' by workgroups (`split`) and
by wavefronts."""

import pytest
import torch

from luma_amd import LUMA
from luma_amd import functional as F

pytestmark = pytest.mark.gpu

DEV = "cuda"
# sizes around a lane's group, a wavefront's and a workgroup's iteration
SIZES = [1, 7, 8, 9, 255, 511, 512, 513, 2047, 2048, 2049, 4104, 70001]
TYPES = [torch.float32, torch.bfloat16, torch.float16]


def _at(x, offset):
    """A copy of the flat x whose first element lies `offset` elements past
    an aligned address, with the elements around it kept to be checked."""
    buf = torch.full((x.numel() + 16,), 77, dtype=x.dtype, device=DEV)
    view = buf[offset:offset + x.numel()]
    view.copy_(x)
    return buf, view


def _around(buf, view, offset):
    rest = torch.cat([buf[:offset], buf[offset + view.numel():]])
    return bool((rest == 77).all())


@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("inject", [False, True])
@pytest.mark.parametrize("offsets", [(1, 0, 0), (3, 1, 0), (0, 0, 1), (7, 2, 5), (2, 3, 6)])
def test_op_at_offsets(offsets, inject, dtype):
    og, op, oq = offsets
    for n in SIZES:
        print("case", n, offsets, inject, dtype, flush=True)
        gen = torch.Generator(device=DEV).manual_seed(n)
        p0 = torch.randn(n, device=DEV, generator=gen) * 0.02
        pb, p1 = _at(p0, op)
        zero = torch.zeros(n, dtype=torch.int16, device=DEV)
        m0, w0 = zero.clone(), zero.clone()
        (mb, m1), (wb, w1) = _at(zero, oq), _at(zero, oq + 1)
        s0, s1 = F.new_slot(DEV), F.new_slot(DEV)
        for t in range(3):
            g = (torch.randn(n, device=DEV, generator=gen) * 1e-3).to(dtype)
            u = [torch.rand(n, device=DEV, generator=gen) for _ in range(2)] if inject else [None] * 2
            v = [_at(x, og + 1)[1] for x in u] if inject else [None] * 2
            for p, q_m, q_w, s, gr, un in ((p0, m0, w0, s0, g, u),
                                           (p1, m1, w1, s1, _at(g, og)[1], v)):
                F.luma_step(p, gr, q_m, q_w, s, 0.9, 0.999, 1e-8, 1e-3, 0.01, 3, 12345, *un)
            assert torch.equal(p0, p1) and torch.equal(m0, m1) and torch.equal(w0, w1), (n, t)
            assert F.slot_state(s0) == F.slot_state(s1), (n, t)
        assert _around(pb, p1, op) and _around(mb, m1, oq) and _around(wb, w1, oq + 1), n


@pytest.mark.parametrize("split", [True, False])
@pytest.mark.parametrize("dtype", TYPES)
def test_optimizer_with_packed_gradients(dtype, split):
    """b's gradients, and every other parameter, lie off a 16-byte boundary."""
    sizes = SIZES * 3 + [1537, 4609, 8191, 30001]
    gen = torch.Generator(device=DEV).manual_seed(5)
    a = [(torch.randn(n, device=DEV, generator=gen) * 0.02).requires_grad_(True) for n in sizes]
    bufs = [_at(p.detach(), i % 4) for i, p in enumerate(a)]
    b = [v.requires_grad_(True) for _, v in bufs]
    for p in a + b:
        p.grad_dtype = None
    oa, ob = LUMA(a, lr=1e-3), LUMA(b, lr=1e-3)
    ob._base_seed = oa._base_seed
    for o in (oa, ob):
        o._get_engine(a[0].device).split = split
    bucket = torch.zeros(sum(sizes) + 1, dtype=dtype, device=DEV)
    for q, g in zip(b, bucket[1:].split(sizes)):
        q.grad = g
    for t in range(4):
        for p, q in zip(a, b):
            p.grad = (torch.randn(p.shape, device=DEV, generator=gen) * 1e-3).to(dtype)
            q.grad.copy_(p.grad)
        oa.step()
        ob.step()
        assert oa._engine._wide == ob._engine._wide == split
    assert all(_around(buf, v.detach(), i % 4) for i, (buf, v) in enumerate(bufs))
    sa, sb = oa.state_dict()["state"], ob.state_dict()["state"]
    for i, (p, q) in enumerate(zip(a, b)):
        assert torch.equal(p.detach(), q.detach()), i
        assert torch.equal(sa[i]["Q_m"], sb[i]["Q_m"]) and torch.equal(sa[i]["Q_w"], sb[i]["Q_w"]), i
        assert sa[i]["S_m"] == sb[i]["S_m"] and sa[i]["S_v"] == sb[i]["S_v"], i
