"""import_adamw_state takes its codes from the certified fast encode and the
exact path; they are the oracle's codes bit for bit: around a lane's group,
the quantise pass's and the max pass's workgroups, over several iterations of
a workgroup and round its queues, in each log1p form, with injected and
Philox uniforms, and for values that only the exact path takes.
export_adamw_state decodes every code as the oracle does, at every remainder
and past a workgroup's first iteration."""

import numpy as np
import pytest
import torch

from luma_amd import LUMA
from luma_amd.optimizer import make_step_seed
from oracle import luma_oracle as O

pytestmark = pytest.mark.gpu

DEV = "cuda"
EPS = 1e-8


def _philox(c0, stream, key):
    """Philox4x32-10 (Salmon et al., SC'11) of counters (c0, 0, stream, 0)."""
    mask = np.uint64(0xFFFFFFFF)
    c = [c0.astype(np.uint64), np.zeros(c0.shape, np.uint64),
         np.full(c0.shape, stream, np.uint64), np.zeros(c0.shape, np.uint64)]
    k0, k1 = key & 0xFFFFFFFF, key >> 32
    for _ in range(10):
        p0, p1 = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), p1 & mask,
             (p0 >> np.uint64(32)) ^ c[3] ^ np.uint64(k1), p0 & mask]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return np.stack(c, axis=1).astype(np.uint32)          # (groups, 4 words)


def _uniforms(n, seed):
    """The framework's two 24-bit uniforms of elements 0 .. n-1: top 16 bits
    from blocks 0 and 2, low 8 bits from block 1 of each group of 8."""
    key = seed & ((1 << 64) - 1)
    groups = np.arange((n + 7) // 8)
    top = [_philox(groups, s, key).view(np.uint16).reshape(-1).astype(np.int64) for s in (0, 2)]
    low = _philox(groups, 1, key).view(np.uint8).reshape(-1).astype(np.int64)
    return tuple(torch.from_numpy(((top[i] << 8) | low[i::2]).astype(np.float32)[:n]) / 2.0 ** 24
                 for i in (0, 1))


def _check(m, v, inject, eps=EPS, u=None):
    n = m.numel()
    p = torch.nn.Parameter(torch.zeros(n, device=DEV))
    opt = LUMA([p], eps=eps)
    opt._base_seed = 12345
    if inject:
        if u is None:
            u = tuple(torch.rand(n, generator=torch.Generator().manual_seed(n + i)) for i in (1, 2))
        opt.inject_noise({p: tuple(x.to(DEV) for x in u)})
    else:
        u = _uniforms(n, make_step_seed(opt._base_seed, 0, 0))
    md, vd = m.to(DEV), v.to(DEV)
    opt.import_adamw_state({"state": {0: {"step": 3, "exp_avg": md, "exp_avg_sq": vd}}})
    q_m, q_w, s_m, s_v = O.quantize_states(m, v, eps, O.injected_draw(*u), "cr")
    s = opt.state_dict()["state"][0]
    assert torch.equal(md.cpu().view(torch.int32), m.view(torch.int32))   # inputs untouched
    assert np.array_equal([s["S_m"], s["S_v"]], [s_m, s_v], equal_nan=True)
    assert torch.equal(s["Q_m"].cpu(), q_m)
    assert torch.equal(s["Q_w"].cpu(), q_w)
    return opt


def _moments(n, scale):
    gen = torch.Generator().manual_seed(n)
    m = torch.randn(n, generator=gen) * scale
    v = torch.randn(n, generator=gen).square() * scale * scale
    zero = torch.rand(n, generator=gen) < 0.02
    return torch.where(zero, 0.0, m), torch.where(zero, 0.0, v)


@pytest.mark.parametrize("inject", [False, True])
@pytest.mark.parametrize("n", [1, 7, 8, 9, 511, 2047, 2049, 16383, 16384, 16385, 65535, 65537,
                               131073, 300007])
def test_codes_at_edges(n, inject):
    print("case", n, inject, flush=True)
    _check(*_moments(n, 1e-3), inject)


# the quantise pass gives each of 1,024 workgroups more than one iteration of
# 2,048 elements above 2,097,152: two (the last workgroup's run of one
# element), three, and six with ragged ends
LARGE = [(1 << 21) + 1, (2 << 21) + 2049, 10500003]


@pytest.mark.parametrize("inject", [False, True])
@pytest.mark.parametrize("n", LARGE)
def test_codes_over_several_iterations(n, inject):
    print("case", n, inject, flush=True)
    _check(*_moments(n, 1e-3), inject)


@pytest.mark.parametrize("inject", [False, True])
def test_every_code_through_the_queues(inject):
    """Four iterations per workgroup whose codes are all left open, 512 to a
    wavefront and iteration: the queues' rings of 1,024 entries wrap.  Every
    preconditioner code is open at an eps below 1e-10; the injected uniforms
    are 0 and every m a point of the grid, so that the momentum codes are too."""
    n = (3 << 21) + 513
    m, v = _moments(n, 1e-3)
    u = None
    if inject:
        s_m = float(m.abs().max())
        delta = np.log1p(s_m) / 32767.0
        k = torch.randint(1, 32767, (n,), generator=torch.Generator().manual_seed(3))
        grid = torch.expm1(k.double() * delta).float()
        grid[0] = s_m
        m = torch.copysign(grid, m)
        u = (torch.zeros(n), torch.zeros(n))
    print("case", n, inject, flush=True)
    _check(m, v, inject, eps=1e-20, u=u)


# S_m of about 0.05 (polynomials), 0.4 (atanh series), 40 (logarithm)
@pytest.mark.parametrize("scale", [1e-12, 0.01, 0.09, 8.0])
def test_codes_by_momentum_scale(scale):
    print("case", scale, flush=True)
    _check(*_moments(40003, scale), False)


@pytest.mark.parametrize("which", ["nan m", "inf m", "nan v", "negative v", "zeros", "tiny v",
                                   "tiny eps"])
def test_codes_of_special_values(which):
    print("case", which, flush=True)
    m, v = _moments(20011, 1e-3)
    eps = EPS
    if which == "nan m":
        m[777] = float("nan")
    elif which == "inf m":
        m[777] = float("inf")
    elif which == "nan v":
        v[777] = float("nan")
    elif which == "negative v":
        v[::3] *= -1.0
    elif which == "zeros":
        m.zero_()
        v.zero_()
    elif which == "tiny v":
        v *= 1e-36
    else:
        v[::5] *= 1e-34
        eps = 1e-20
    if which == "nan m":
        # torch's scale floor drops the NaN or keeps it by operand order; the
        # framework keeps it, every bin index is NaN and every code 0
        p = torch.nn.Parameter(torch.zeros(m.numel(), device=DEV))
        opt = LUMA([p])
        opt.import_adamw_state({"state": {0: {"step": 3, "exp_avg": m.to(DEV),
                                              "exp_avg_sq": v.to(DEV)}}})
        assert not opt.state_dict()["state"][0]["Q_m"].any()
        return
    _check(m, v, False, eps)


def test_moments_in_other_layouts():
    """Moments that are not float32 tensors laid out as the parameter are
    converted as before."""
    m, v = _moments(96 * 40, 1e-3)
    m, v = m.view(96, 40), v.view(96, 40)
    codes = []
    for conv in (lambda x: x.to(DEV), lambda x: x, lambda x: x.to(DEV).double(),
                 lambda x: x.t().contiguous().to(DEV).t()):
        p = torch.nn.Parameter(torch.zeros(96, 40, device=DEV))
        opt = LUMA([p])
        opt._base_seed = 5
        opt.import_adamw_state({"state": {0: {"step": 3, "exp_avg": conv(m),
                                              "exp_avg_sq": conv(v)}}})
        codes.append((opt.state[p]["Q_m"], opt.state[p]["Q_w"]))
    for a, b in codes[1:]:
        assert torch.equal(a, codes[0][0]) and torch.equal(b, codes[0][1])


# x_top = log1p(S_m) on both sides of 1/8 and of 1/2, and the scale of S_v
# where exp's argument passes 80 (eps 1e-30)
@pytest.mark.parametrize("s_m,s_v,eps", [(1e-9, 0.0, 1e-8), (1e-3, 1e-6, 1e-8), (0.133, 1e-4, 1e-8),
                                         (0.1332, 1e-12, 1e-8), (0.5, 1e-2, 1e-8),
                                         (0.6485, 1.0, 1e-12), (0.649, 4.0, 1e-8),
                                         (40.0, 100.0, 1e-8), (0.1, 1e4, 1e-20),
                                         (0.1, 1e16, 1e-30)])
@pytest.mark.parametrize("more", [0, 1, 2, 3])
def test_every_code_decodes_exactly(s_m, s_v, eps, more):
    _check_decode((1 << 16) + more, s_m, s_v, eps)


# a workgroup of export steps on above 2,097,152 elements
@pytest.mark.parametrize("s_m,s_v,eps", [(1e-3, 1e-6, 1e-8), (0.5, 1e-2, 1e-8), (40.0, 100.0, 1e-8)])
@pytest.mark.parametrize("n", [(1 << 21) + 3, (2 << 21) + 4097, 10500002])
def test_codes_decode_exactly_over_several_iterations(n, s_m, s_v, eps):
    _check_decode(n, s_m, s_v, eps)


def _check_decode(n, s_m, s_v, eps):
    print("case", n, s_m, s_v, eps, flush=True)
    codes = (torch.arange(n) & 0xFFFF).to(torch.int32).to(torch.int16)
    p = torch.nn.Parameter(torch.zeros(n, device=DEV))
    opt = LUMA([p], eps=eps)
    sd = opt.state_dict()
    sd["state"] = {0: {"step": 5, "param_id": 0, "Q_m": codes.to(DEV), "Q_w": codes.to(DEV),
                       "S_m": s_m, "S_v": s_v}}
    opt.load_state_dict(sd)
    out = opt.export_adamw_state()["state"][0]
    w_min, delta_m, _, delta_w, _ = O.precompute(s_m, s_v, eps)
    assert torch.equal(out["exp_avg"].cpu(), O.decode_momentum(codes, delta_m, "cr"))
    assert torch.equal(out["exp_avg_sq"].cpu(),
                       O.decode_second_moment(codes, w_min, delta_w, eps, "cr"))
