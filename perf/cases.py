"""What a user of luma_amd runs, as cases to be timed and compared.

Nearly all of an optimizer's use is ``LUMA.step()`` in the middle of a
training run, so most cases are that: the parameter lists of this
repository's benchmark and tests, from a small classifier to the
Llama-3-8B-shaped set, in each gradient type, with GradScaler, with gradients
that are views of packed buckets (DistributedDataParallel's
``gradient_as_bucket_view``), and replayed from a captured graph.  The others
are the per-tensor op (``luma_amd.functional.luma_step``), which compiled
training steps call, and the two directions of the AdamW hand-off:
``export_adamw_state`` (decode) and ``import_adamw_state`` (encode).

Every optimizer is prepared in the middle of training: its state is loaded as
a checkpoint of step ``STEP``, with momentum and preconditioner values as
Adam has them after that many steps of the case's gradients.  A list's
parameters and codes lie in flat buffers, every tensor 64-element aligned, so
that a pass returns all of them as three tensors.

A case's fields: ``call`` (step, replay, op, export, import), ``shapes`` and
the fields that name a list of shapes (``_shapes``), ``grad`` (the gradients'
type), ``std`` (their standard deviation; ``std_to``: log-uniform from std to
std_to over the tensors), ``outliers`` and ``zeros`` (shares of gradients 100
times larger, and zero), ``packed`` (gradients without padding between
them), ``scaled`` (GradScaler).
"""

import math
import random

import torch

from luma_amd import LUMA
from luma_amd import functional

DEV = "cuda"
STEP = 100                     # completed steps when a case begins
HYPER = dict(lr=1e-3, betas=(0.9, 0.999), eps=1e-8)
DECAY = 0.01                   # weight decay of matrices; vectors have none
SCALE = 65536.0                # GradScaler's scale
ALIGN = 64                     # elements: where a tensor of a flat buffer may start
TYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16, "float16": torch.float16}


# -- the cases ------------------------------------------------------------------


def _case(name, call, shapes, grad="float32", std=1e-3, **more):
    return dict({"name": name, "call": call, "shapes": shapes, "grad": grad, "std": std}, **more)


def listed():
    return [
        # a small classifier: six tensors, the smallest call a program makes
        _case("step mlp", "step", "mlp"),
        # a nanoGPT-sized model (51 tensors, 0.8M parameters): launches and latency
        _case("step nano", "step", "nano"),
        # the same step captured into a graph, as launch-bound training loops run it
        _case("replay nano", "replay", "nano"),
        # GPT-2 small, bfloat16 gradients: an ordinary training step
        _case("step gpt2 bf16", "step", "gpt2", "bfloat16"),
        # 20,000 tensors of 1 to 65,536 elements: many odd sizes in one call
        _case("step many small", "step", "log_uniform", std=1e-4, zeros=0.01, tensors=20000,
              most=65536, shape_seed=3),
        # one large weight
        _case("step 4096x4096", "step", "matrix", rows=4096, cols=4096),
        # the embeddings and 8 of the 32 layers of the Llama-3-8B-shaped set: the largest
        _case("step llama bf16", "step", "llama", "bfloat16", outliers=1e-3, layers=8,
              embeddings=True),
        # fp16 gradients of very different sizes under GradScaler
        _case("step scaled fp16", "step", "llama", "float16", std=1e-7, std_to=1e-1, layers=1,
              embeddings=False, scaled=True),
        # odd-sized weights whose gradients are views of a packed float32 bucket
        _case("step packed grads", "step", "log_uniform", tensors=200, most=2000003,
              shape_seed=7, packed=True),
        # the per-tensor op of compiled training steps, a ragged bfloat16 tensor
        _case("op 4099x1021 bf16", "op", "matrix", "bfloat16", rows=4099, cols=1021),
        # hand-off to AdamW and back: one Llama-3-8B layer (nine tensors)
        _case("export llama layer", "export", "llama", layers=1, embeddings=False),
        _case("import llama layer", "import", "llama", layers=1, embeddings=False),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: any call, a random list of odd-sized
    tensors (one for the op), any gradient type and option."""
    call = rng.choice(["step"] * 6 + ["replay", "op", "export", "import"])
    case = {"call": call, "grad": rng.choice(["float32", "bfloat16", "float16"]),
            "std": 10.0 ** rng.uniform(-5.0, -2.0)}
    if call == "op":
        n = _log_uniform(rng, 1, 1 << 26)
        cols = _log_uniform(rng, 1, min(n, 8192))
        case.update(shapes="matrix", rows=max(1, n // cols), cols=cols)
    else:
        tensors = _log_uniform(rng, 1, {"step": 2000, "replay": 300}.get(call, 24))
        most = _log_uniform(rng, 64, 1 << 26)
        while tensors * most > 1 << 30:
            most //= 2
        case.update(shapes="log_uniform", tensors=tensors, most=most,
                    shape_seed=rng.randrange(1 << 20))
    if call in ("step", "replay", "op"):
        if rng.random() < 0.3:
            case["outliers"] = 1e-3
        if rng.random() < 0.3:
            case["zeros"] = 0.01
    if call == "step":
        case["scaled"] = case["grad"] == "float16"
        if case["scaled"]:
            case["std"] = min(case["std"], 1e-3)     # outliers stay finite times SCALE
        case["packed"] = rng.random() < 0.25
    return case


# -- sizes ----------------------------------------------------------------------


def _shapes(case):
    """The case's tensors, matrices (weight decay) before vectors (none)."""
    kind = case["shapes"]
    if kind == "mlp":
        out = [(128, 64), (128,), (24, 128), (24,), (1, 24), (1,)]
    elif kind == "nano":
        out = [(28, 128), (64, 128)]
        for _ in range(4):
            out += [(128,), (128,), (384, 128), (384,), (128, 128), (128,), (128,), (128,),
                    (512, 128), (512,), (128, 512), (128,)]
        out += [(128,), (128,)]
    elif kind == "gpt2":
        out = [(50257, 768), (1024, 768)]
        for _ in range(12):
            out += [(768,), (768,), (768, 2304), (2304,), (768, 768), (768,), (768,), (768,),
                    (768, 3072), (3072,), (3072, 768), (768,)]
        out += [(768,), (768,)]
    elif kind == "llama":
        out = [(128256, 4096)] if case["embeddings"] else []
        for _ in range(case["layers"]):
            out += [(4096, 4096), (1024, 4096), (1024, 4096), (4096, 4096), (14336, 4096),
                    (14336, 4096), (4096, 14336), (4096,), (4096,)]
        out += [(4096,), (128256, 4096)] if case["embeddings"] else []
    elif kind == "matrix":
        out = [(case["rows"], case["cols"])]
    else:
        rng = random.Random(case["shape_seed"])
        out = [(_log_uniform(rng, 1, case["most"]),) for _ in range(case["tensors"])]
        if case["tensors"] < 20000:      # a few matrices among them, so that both groups exist
            out = [(1, s[0]) if i % 2 else s for i, s in enumerate(out)]
    return [s for s in out if len(s) > 1] + [s for s in out if len(s) < 2]


class _Layout:
    """Where a case's tensors lie in flat buffers: `at` with every tensor
    aligned, `packed_at` without padding."""

    def __init__(self, case):
        self.shapes = _shapes(case)
        self.numel = [math.prod(s) for s in self.shapes]
        self.matrices = sum(len(s) > 1 for s in self.shapes)
        self.padded = [-(-n // ALIGN) * ALIGN for n in self.numel]
        self.at, self.packed_at, a, b = [], [], 0, 0
        for n, p in zip(self.numel, self.padded):
            self.at.append(a)
            self.packed_at.append(b)
            a, b = a + p, b + n
        self.total, self.packed_total = a, b

    def views(self, flat, packed=False):
        at = self.packed_at if packed else self.at
        return [flat[o:o + n].view(s) for o, n, s in zip(at, self.numel, self.shapes)]

    def blocks(self, most=1 << 28):
        """Runs of consecutive tensors of at most `most` elements together
        (or one larger tensor): (first, end) tensor indices."""
        first, size = 0, 0
        for i, p in enumerate(self.padded):
            if i > first and size + p > most:
                yield first, i
                first, size = i, 0
            size += p
        yield first, len(self.padded)


# -- inputs ---------------------------------------------------------------------


def _stds(case, n):
    """The gradients' standard deviation of every tensor."""
    lo, hi = case["std"], case.get("std_to", case["std"])
    rng = random.Random(5)
    return [math.exp(rng.uniform(math.log(lo), math.log(hi))) for _ in range(n)]


def _params(case, L, gen):
    return torch.randn(L.total, generator=gen, device=DEV) * 0.02


def _grads(case, L, gen):
    """The flat gradients, in the case's type and layout (times SCALE under
    GradScaler)."""
    lens = L.numel if case.get("packed") else L.padded
    total = L.packed_total if case.get("packed") else L.total
    out = torch.empty(total, dtype=TYPES[case["grad"]], device=DEV)
    stds, at = _stds(case, len(lens)), 0
    for a, b in L.blocks():
        std = torch.tensor(stds[a:b], device=DEV).repeat_interleave(
            torch.tensor(lens[a:b], device=DEV))
        g = torch.randn(std.numel(), generator=gen, device=DEV) * std
        if case.get("outliers"):
            hit = torch.rand(g.numel(), generator=gen, device=DEV) < case["outliers"]
            g = torch.where(hit, g * 100.0, g)
        if case.get("zeros"):
            g *= torch.rand(g.numel(), generator=gen, device=DEV) >= case["zeros"]
        if case.get("scaled"):
            g *= SCALE
        out[at:at + g.numel()] = g
        at += g.numel()
    return out


def _moments(case, L, gen, a, b):
    """Adam's moments of tensors a .. b-1 (padded, concatenated) after STEP
    steps: m of about 0.3 std, v about the bias-corrected mean square with
    its spread, larger where an outlier fell within beta2's memory."""
    beta2 = HYPER["betas"][1]
    std = torch.tensor(_stds(case, len(L.numel))[a:b], device=DEV).repeat_interleave(
        torch.tensor(L.padded[a:b], device=DEV))
    m = torch.randn(std.numel(), generator=gen, device=DEV) * std * 0.3
    v = torch.randn(std.numel(), generator=gen, device=DEV)
    v = (1.0 + 0.14 * v).abs() * std * std * (1.0 - beta2 ** STEP)
    if case.get("outliers"):
        hit = torch.rand(std.numel(), generator=gen, device=DEV) < case["outliers"] * STEP
        v = torch.where(hit, v + (1.0 - beta2) * (100.0 * std) ** 2, v)
    return m, v


def _codes(case, L, gen):
    """A checkpoint's codes (flat int16, the parameters' layout) and scales
    [(S_m, S_v)]: _moments on the log grids, to the nearest code."""
    eps = HYPER["eps"]
    q_m = torch.empty(L.total, dtype=torch.int16, device=DEV)
    q_w = torch.empty(L.total, dtype=torch.int16, device=DEV)
    scales = []
    for a, b in L.blocks():
        base = L.at[a]
        m, v = _moments(case, L, gen, a, b)
        spans = [(L.at[i] - base, L.numel[i]) for i in range(a, b)]
        tops = torch.stack([torch.stack([m[o:o + n].abs().amax() for o, n in spans]),
                            torch.stack([v[o:o + n].amax() for o, n in spans])]).double()
        tops[0].clamp_(min=1e-9)
        d_m = torch.log1p(tops[0]) / 32767.0
        w_min = 1.0 / (tops[1].sqrt() + eps)
        d_w = torch.log(1.0 / (eps * w_min)).clamp_(min=0.0) / 65535.0
        lens = torch.tensor(L.padded[a:b], device=DEV)
        rep = lambda x: x.float().repeat_interleave(lens)  # noqa: E731
        end = base + m.numel()
        q = (m.abs().log1p() / rep(d_m)).round().clamp_(max=32767.0)
        q_m[base:end] = torch.copysign(q, m).to(torch.int16)
        w = 1.0 / (v.sqrt() + eps)
        q = ((w / rep(w_min)).log() / rep(d_w)).nan_to_num_(0.0, 0.0, 0.0)
        q_w[base:end] = q.round_().clamp_(0.0, 65535.0).to(torch.int32).to(torch.int16)
        scales += list(zip(*tops.tolist()))
    return q_m, q_w, scales


def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _optimizer(L, params, seed, state):
    """LUMA over `params` (matrices and vectors as two groups), resumed from
    a checkpoint with `state`."""
    groups = [dict(params=params[:L.matrices], weight_decay=DECAY),
              dict(params=params[L.matrices:], weight_decay=0.0)]
    opt = LUMA([g for g in groups if g["params"]], **HYPER)
    sd = opt.state_dict()
    sd["state"] = state
    sd["_base_seed"] = int(seed) * 7919 + 12345
    opt.load_state_dict(sd)
    return opt


# -- one case -------------------------------------------------------------------


def prepare(case, seed):
    L = _Layout(case)
    gen = _generator(seed)
    call = case["call"]
    state = {"call": call, "params": _params(case, L, gen)}
    if call == "import":
        params = [torch.nn.Parameter(v) for v in L.views(state["params"])]
        state["list"] = params
        state["opt"] = _optimizer(L, params, seed, {})
        m = torch.empty(L.total, device=DEV)
        v = torch.empty(L.total, device=DEV)
        for a, b in L.blocks():
            end = L.at[b] if b < len(L.at) else L.total
            m[L.at[a]:end], v[L.at[a]:end] = _moments(case, L, gen, a, b)
        state["adamw"] = {"state": {
            i: {"step": torch.tensor(float(STEP)), "exp_avg": x, "exp_avg_sq": y}
            for i, (x, y) in enumerate(zip(L.views(m), L.views(v)))}}
        return state

    q_m, q_w, scales = _codes(case, L, gen)
    state["q_m"], state["q_w"] = q_m, q_w
    codes = list(zip(L.views(q_m), L.views(q_w)))
    if call == "op":
        state["grad"] = L.views(_grads(case, L, gen))[0]
        state["param"] = L.views(state["params"])[0]
        state["codes"] = codes[0]
        state["slot"] = functional.new_slot(DEV)
        functional.init_slot(state["slot"], STEP, *scales[0], HYPER["eps"])
        state["seed"] = int(seed) * 7919 + 12345
        return state

    params = [torch.nn.Parameter(v) for v in L.views(state["params"])]
    state["list"] = params
    state["opt"] = opt = _optimizer(L, params, seed, {
        i: {"step": STEP, "param_id": i, "Q_m": c[0], "Q_w": c[1], "S_m": s[0], "S_v": s[1]}
        for i, (c, s) in enumerate(zip(codes, scales))})
    for p, (c_m, c_w) in zip(params, codes):
        opt.state[p]["Q_m"], opt.state[p]["Q_w"] = c_m, c_w
    if call == "export":
        return state
    packed = bool(case.get("packed"))
    for p, g in zip(params, L.views(_grads(case, L, gen), packed)):
        if g.dtype != p.dtype:
            p.grad_dtype = None       # a lower-precision gradient on a float32 parameter
        p.grad = g
    if case.get("scaled"):
        # (no growth: the scale of a timed run stays what the gradients were scaled by)
        state["scaler"] = torch.amp.GradScaler(DEV, init_scale=SCALE, growth_interval=1 << 30)
        state["scaler"].scale(torch.zeros(1, device=DEV))
    if call == "replay":
        opt.step()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            opt.step()
    return state


def run(state):
    call = state["call"]
    if call == "import":
        opt = state["opt"]
        opt.import_adamw_state(state["adamw"])
        return [[opt.state[p]["Q_m"], opt.state[p]["Q_w"]] for p in state["list"]]
    if call == "export":
        out = state["opt"].export_adamw_state()["state"]
        return [[s["exp_avg"], s["exp_avg_sq"]] for s in out.values()]
    if call == "op":
        beta1, beta2 = HYPER["betas"]
        functional.luma_step(state["param"], state["grad"], *state["codes"], state["slot"],
                             beta1, beta2, HYPER["eps"], HYPER["lr"], DECAY, 0, state["seed"])
    elif call == "replay":
        state["graph"].replay()
    elif "scaler" in state:
        state["scaler"].step(state["opt"])
        state["scaler"].update()
    else:
        state["opt"].step()
    return [state["params"], state["q_m"], state["q_w"]]


def work(case):
    """A step reads the gradient once and reads and writes the parameter and
    both codes (4 + 2 + 2 bytes each way); export reads the codes and writes
    two float32, import the other way.  The operations are float32 vector
    ones: decode, moving averages, update, two encodes and their draws."""
    n = sum(_Layout(case).numel)
    if case["call"] in ("export", "import"):
        return {"bytes": 12 * n, "flops": 20 * n if case["call"] == "export" else 40 * n}
    return {"bytes": (16 + TYPES[case["grad"]].itemsize) * n, "flops": 60 * n}


def tolerance(case):
    """Codes are whole numbers and the same for every correct implementation
    (the uniforms are fixed by the seeds): none may differ.  Parameters: one
    float32 rounding of p plus the update's few, an update being about a
    twentieth of p (measured, the fast path against the exact one: rel
    4.4e-8, max 1.24e-7; stated: four times that).  Exported moments: a few
    float32 roundings (measured against 64 bits: rel at most 2.0e-7), which
    1/w - eps enlarges where v is small."""
    if case["call"] == "import":
        return "exact"
    if case["call"] == "export":
        return {"rel": 5e-7, "max": 5e-6, "differ": 0.0}
    return {"rel": 1.8e-7, "max": 5e-7, "differ": 0.0}


# -- the same in 64 bits --------------------------------------------------------


def _decode(q_m, q_w, S_m, S_v):
    """m and v of the codes on the grids of S_m and S_v, in float64."""
    eps = HYPER["eps"]
    w_min = 1.0 / (math.sqrt(S_v) + eps)
    d_m = math.log1p(S_m) / 32767.0
    d_w = max(0.0, math.log(1.0 / (eps * w_min))) / 65535.0
    q = q_m.double()
    m = q.sign() * torch.expm1(q.abs() * d_m)
    w = w_min * torch.exp((q_w.to(torch.int32) & 0xFFFF).double() * d_w)
    return m, (1.0 / w - eps).clamp(min=0.0) ** 2


def exact(case, seed):
    call = case["call"]
    if call in ("import", "replay"):
        # import: whole codes only; replay: begins after a step whose rounding
        # draws are the framework's own
        return None
    L = _Layout(case)
    gen = _generator(seed)
    flat = _params(case, L, gen)
    q_m, q_w, scales = _codes(case, L, gen)
    codes = list(zip(L.views(q_m), L.views(q_w)))
    if call == "export":
        return [list(_decode(*c, *s)) for c, s in zip(codes, scales)]
    grads = L.views(_grads(case, L, gen), bool(case.get("packed")))
    beta1, beta2 = HYPER["betas"]
    t = STEP + 1
    eta = HYPER["lr"] / (1.0 - beta1 ** t)
    bc2 = 1.0 - beta2 ** t
    out = flat.double()
    for i, (p, c, s, g) in enumerate(zip(L.views(out), codes, scales, grads)):
        m, v = _decode(*c, *s)
        if case.get("scaled"):
            g = (g.float() / SCALE).to(g.dtype)     # as GradScaler.unscale_ stores it
        g = g.double()
        m = beta1 * m + (1.0 - beta1) * g
        v = beta2 * v + (1.0 - beta2) * g * g
        decay = 1.0 - HYPER["lr"] * (DECAY if call == "op" or i < L.matrices else 0.0)
        p.mul_(decay).sub_(eta * m / ((v / bc2).sqrt() + HYPER["eps"]))
    if call == "op":
        out = out.view(-1)
    return [out, None, None]
