"""Workloads of the framework's public entry points, from a single small call
to the largest training configuration: the fused mixer core (``chunk_scan``),
the drop-in scan (``fast_state_scan``), the token-exact mode (``wy_scan``), a
residual block and a whole LM around the core, and the outer optimizer's
``msign``.

A case is a dict of plain values; ``kind`` selects the entry point:

* ``core``  -- chunk_scan over (B, H, T, d) streams; ``layout`` "bthd" is the
  mixer's own storage (the heads of one projection output side by side),
  "bhtd" contiguous streams; ``train`` adds the backward of every input.
* ``scan``  -- fast_state_scan over per-chunk d x d matrices (B, H, N, d, d).
* ``wy``    -- wy_scan.
* ``block`` -- one residual block under bfloat16 autocast, forward + backward.
* ``lm``    -- the LM's logits without gradients under bfloat16 autocast.
* ``msign`` -- msign of the momentum updates of one block's hidden weights.
"""
import math
import os
import sys

import torch

_PKG = os.path.abspath("gmdn-gated-muon-deltanet_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

RULES = ("delta", "muon", "adam")
NS = (3.4445, -4.7750, 2.0315)  # the quintic iteration's coefficients
LOG_FLOOR = math.log(1e-6)


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # one layer call of the smallest configuration, float32: latency and launches
        dict(name="core_delta_f32_small_train", kind="core", rule="delta", dtype="f32", B=1, H=2, T=256, d=64, ns=5,
             chunk=64, layout="bhtd", train=True),
        # prefill of one long sequence: few heads, an odd number of chunks
        dict(name="core_delta_prefill", kind="core", rule="delta", dtype="bf16", B=1, H=8, T=8128, d=128, ns=5,
             chunk=64, layout="bthd", train=False),
        # the headline training configuration
        dict(name="core_delta_train", kind="core", rule="delta", dtype="bf16", B=4, H=16, T=4096, d=128, ns=5,
             chunk=64, layout="bhtd", train=True),
        # the largest: long-sequence training with the Newton-Schulz update
        dict(name="core_muon_train", kind="core", rule="muon", dtype="bf16", B=2, H=16, T=8192, d=128, ns=5, chunk=64,
             layout="bhtd", train=True),
        # training with the elementwise second-moment update at both head dims
        dict(name="core_adam_train", kind="core", rule="adam", dtype="bf16", B=2, H=8, T=4096, d=64, ns=5, chunk=64,
             layout="bhtd", train=True),
        dict(name="core_adam_d128_train", kind="core", rule="adam", dtype="bf16", B=2, H=8, T=2048, d=128, ns=5,
             chunk=64, layout="bthd", train=True),
        # training in float32 (autocast off) with the Newton-Schulz update
        dict(name="core_muon_f32_train", kind="core", rule="muon", dtype="f32", B=1, H=8, T=512, d=128, ns=3, chunk=64,
             layout="bthd", train=True),
        # the drop-in scan of an existing trainer that forms its own U, K
        dict(name="scan_delta_train", kind="scan", rule="delta", precision="tf32", B=4, H=16, N=64, d=128, ns=5,
             train=True),
        # training of the token-exact mode
        dict(name="wy_train", kind="wy", B=4, H=16, T=4096, d=128, train=True),
        # one block of the 12-layer LM in training
        dict(name="block_muon_train", kind="block", rule="muon", B=8, T=2048, D=1024, H=8, ns=3),
        # logits of the 12-layer LM for one prompt
        dict(name="lm_muon_prefill", kind="lm", rule="muon", B=1, T=1024, D=1024, H=8, ns=3, layers=12, vocab=32000),
        # the outer optimizer's orthogonalisation of three blocks' weights
        dict(name="msign_blocks", kind="msign", D=1024, blocks=3, steps=5),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["core"] * 6 + ["scan"] * 2 + ["wy"] * 2 + ["block", "lm", "msign"])
    rule = rng.choice(RULES)
    train = rng.random() < 0.6
    ns = rng.choice([1, 3, 5])
    if kind == "core":
        dtype = rng.choice(["bf16", "bf16", "bf16", "f32"])
        d = rng.choice([16, 32, 64, 64, 128, 128, 128])
        chunk = rng.choice([64] * 8 + [32, 128])
        most = 4096 if dtype == "bf16" and chunk == 64 else 512 if rule == "muon" else 1024  # tokens
        B, H = _log_int(rng, 1, 4), _log_int(rng, 1, 16)
        n = _log_int(rng, 1, most // chunk)
        return dict(kind=kind, rule=rule, dtype=dtype, B=B, H=H, T=n * chunk, d=d, ns=ns, chunk=chunk,
                    layout=rng.choice(["bhtd", "bthd"]), train=train)
    if kind == "scan":
        precision = rng.choice(["tf32", "tf32", "ieee"])
        most = 8 if rule == "muon" and precision == "ieee" else 48  # chunks
        return dict(kind=kind, rule=rule, precision=precision, B=_log_int(rng, 1, 4), H=_log_int(rng, 1, 16),
                    N=_log_int(rng, 1, most), d=rng.choice([16, 32, 64, 128]), ns=ns, train=train)
    if kind == "wy":
        return dict(kind=kind, B=_log_int(rng, 1, 4), H=_log_int(rng, 1, 16), T=64 * _log_int(rng, 1, 64),
                    d=rng.choice([64, 128]), train=train)
    if kind == "block":
        H = rng.choice([4, 8])
        return dict(kind=kind, rule="muon", B=_log_int(rng, 1, 8), T=64 * _log_int(rng, 1, 32),
                    D=H * rng.choice([64, 128]), H=H, ns=3)
    if kind == "lm":
        H = rng.choice([4, 8])
        return dict(kind=kind, rule="muon", B=_log_int(rng, 1, 4), T=64 * _log_int(rng, 1, 16),
                    D=H * rng.choice([64, 128]), H=H, ns=3, layers=rng.choice([2, 4]),
                    vocab=rng.choice([257, 4099, 32000]))
    return dict(kind="msign", D=64 * _log_int(rng, 3, 16), blocks=rng.choice([1, 2, 3]), steps=5)


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _streams(c, seed):
    """q, k (unit rows), v and the gates' values as the mixer's front-end
    gives them: float32, before the cast to the case's type."""
    g = _gen(seed)
    B, H, T, d = c["B"], c["H"], c["T"], c["d"]

    def rand(*shape):
        return torch.randn(*shape, generator=g, device="cuda")

    def stream(norm):
        x = rand(B, T, H, d)
        x = x / x.norm(dim=-1, keepdim=True).clamp_min(1e-12) if norm else x
        x = x.transpose(1, 2)
        return x if c.get("layout") == "bthd" else x.contiguous()

    q, k, v = stream(True), stream(True), stream(False)
    beta = torch.sigmoid(rand(B, H, T))
    la = torch.nn.functional.logsigmoid(rand(B, H, T) + 3.0)
    # momentum products of about 0.9 and 0.999 a chunk, different in every token
    lm = math.log(0.9) / 64 * (0.5 + torch.rand(B, H, T, generator=g, device="cuda"))
    ln = math.log(0.999) / 64 * (0.5 + torch.rand(B, H, T, generator=g, device="cuda"))
    dO = stream(False)
    return q, k, v, beta, la, lm, ln, dO


def _dtype(c):
    return torch.float32 if c.get("dtype") == "f32" else torch.bfloat16


def _core_inputs(c, seed):
    q, k, v, beta, la, lm, ln, dO = _streams(c, seed)
    dt = _dtype(c)
    ins = [q.to(dt), k.to(dt), v.to(dt), beta, la]
    if c["kind"] == "core" and c["rule"] != "delta":
        ins.append(lm)
    if c["kind"] == "core" and c["rule"] == "adam":
        ins.append(ln)
    return ins, dO.to(dt)


def _scan_inputs(c, seed):
    """U = v^T diag(w) k and K = k^T diag(w) k of 64-token chunks."""
    g = _gen(seed)
    B, H, N, d = c["B"], c["H"], c["N"], c["d"]
    k = torch.randn(B * H * N, 64, d, generator=g, device="cuda")
    k = k / k.norm(dim=-1, keepdim=True).clamp_min(1e-12)
    v = torch.randn(B * H * N, 64, d, generator=g, device="cuda") / d ** 0.5
    w = torch.rand(B * H * N, 64, 1, generator=g, device="cuda") * 0.3
    K = torch.bmm((k * w).transpose(1, 2).contiguous(), k).view(B, H, N, d, d)
    U = torch.bmm((v * w).transpose(1, 2).contiguous(), k).view(B, H, N, d, d)
    gates = [torch.rand(B, H, N, generator=g, device="cuda") * r + o
             for r, o in ((0.2, 0.75), (0.5, 0.2), (0.5, 0.3), (0.2, 0.7))]
    return [U, K, *gates], torch.randn(B, H, N, d, d, generator=g, device="cuda")


def _model(c, seed):
    from gmdn_amd.mixer import LM, Block
    with torch.random.fork_rng(devices=[torch.cuda.current_device()]), torch.device("cuda"):
        torch.manual_seed(int(seed))
        if c["kind"] == "lm":
            return LM(c["vocab"], c["D"], c["layers"], c["H"], c["rule"], 64, c["ns"])
        m = Block(c["D"], c["H"], c["rule"], 64, c["ns"])
        m.apply(LM._init)
        m.mixer.reset_gate_bias()
        return m


def _msign_shapes(c):
    D = c["D"]
    return [(3 * D, D), (D, D), (4 * D, D), (D, 4 * D)]


def _msign_inputs(c, seed):
    g = _gen(seed)
    return [torch.randn(c["blocks"], r, s, generator=g, device="cuda") * 1e-3 for r, s in _msign_shapes(c)]


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("core", "wy"):
        ins, dO = _core_inputs(case, seed)
        if case["train"]:
            ins = [t.requires_grad_() for t in ins]
        return dict(case=case, ins=ins, dO=dO)
    if kind == "scan":
        ins, dO = _scan_inputs(case, seed)
        if case["train"]:
            used = {"delta": 3, "muon": 5, "adam": 6}[case["rule"]]
            for t in ins[:2] + [ins[i] for i in range(2, 6) if i < used]:
                t.requires_grad_()
        return dict(case=case, ins=ins, dO=dO)
    if kind == "block":
        m = _model(case, seed)
        g = _gen(seed + 1)
        x = torch.randn(case["B"], case["T"], case["D"], generator=g, device="cuda").requires_grad_()
        dy = torch.randn(case["B"], case["T"], case["D"], generator=g, device="cuda")
        return dict(case=case, model=m, x=x, dy=dy)
    if kind == "lm":
        idx = torch.randint(case["vocab"], (case["B"], case["T"]), generator=_gen(seed + 1), device="cuda")
        return dict(case=case, model=_model(case, seed), idx=idx)
    return dict(case=case, updates=_msign_inputs(case, seed))


# ------------------------------------------------------------------ one pass
def run(state):
    import fast_scan
    c = state["case"]
    kind = c["kind"]
    fast_scan.set_precision(c.get("precision", "tf32"))  # a process-wide setting; split precision is the default
    if kind in ("core", "wy"):
        ins = state["ins"]
        with torch.set_grad_enabled(c["train"]):
            if kind == "wy":
                from gmdn_amd.wy import wy_scan
                o = wy_scan(*ins)
            else:
                from gmdn_amd.chunk import chunk_scan
                o = chunk_scan(*ins, rule=c["rule"], ns=c["ns"], chunk=c["chunk"])
        return [o, *torch.autograd.grad(o, ins, state["dO"])] if c["train"] else [o]
    if kind == "scan":
        ins = state["ins"]
        with torch.set_grad_enabled(c["train"]):
            S = fast_scan.fast_state_scan(*ins, RULES.index(c["rule"]), c["ns"])
        if not c["train"]:
            return [S]
        return [S, *torch.autograd.grad(S, [t for t in ins if t.requires_grad], state["dO"])]
    if kind == "block":
        with torch.autocast("cuda", torch.bfloat16):
            y = state["model"](state["x"])
        return [y, *torch.autograd.grad(y, [state["x"], *state["model"].parameters()], state["dy"])]
    if kind == "lm":
        with torch.no_grad(), torch.autocast("cuda", torch.bfloat16):
            return [state["model"](state["idx"])[0]]
    from gmdn_amd.muon import msign
    return [msign(u, c["steps"]) for u in state["updates"]]


# ------------------------------------------------------------------ what a pass cannot do without
def _core_flops(c, C, d, rule, train):
    """Products of one chunk and head: A = Q K^T, E = V - K S^T,
    o = Q S^T + A E, G = E^T diag(w) K, and the rule's update."""
    f = 4 * C * C * d + 6 * C * d * d
    if rule == "wy":
        f += 4 * C * C * d  # the triangular system's two right-hand sides
    b = 2 * f
    if rule == "muon":
        f += 6 * c["ns"] * d ** 3
        b += 16 * c["ns"] * d ** 3
    return f + (b if train else 0)


def work(case):
    c, kind = case, case["kind"]
    if kind in ("core", "wy"):
        rule = c.get("rule", "wy")
        size, gates = 4 if c.get("dtype") == "f32" else 2, {"delta": 2, "wy": 2, "muon": 3, "adam": 4}[rule]
        rows, C = c["B"] * c["H"] * c["T"], c.get("chunk", 64)
        per = 4 * size * c["d"] + 4 * gates
        if c["train"]:
            per += 7 * size * c["d"] + 8 * gates
        return {"bytes": rows * per, "flops": rows // C * _core_flops(c, C, c["d"], rule, c["train"])}
    if kind == "scan":
        d, n, ns = c["d"], c["B"] * c["H"] * c["N"], c["ns"]
        f = {"delta": 2, "adam": 2, "muon": 2 + 6 * ns}[c["rule"]]
        b = {"delta": 4, "adam": 6, "muon": 6 + 16 * ns}[c["rule"]]
        planes = 3 + (5 if c["train"] else 0)
        return {"bytes": n * (planes * d * d * 4 + 32), "flops": n * (f + (b if c["train"] else 0)) * d ** 3}
    if kind in ("block", "lm"):
        D, rows, d = c["D"], c["B"] * c["T"], c["D"] // c["H"]
        train, layers = kind == "block", c.get("layers", 1)
        weights = 12 * D * D * layers
        core = rows // 64 * c["H"] * _core_flops(c, 64, d, c["rule"], train) * layers
        f, by = 2 * rows * weights * (3 if train else 1) + core, 4 * weights + 4 * rows * D
        if train:
            by += 4 * weights + 12 * rows * D
        else:
            f += 2 * rows * D * c["vocab"]
            by += 4 * D * c["vocab"] + 2 * rows * c["vocab"]
        return {"bytes": by, "flops": f}
    by = f = 0
    for r, s in _msign_shapes(c):
        m, n = min(r, s), max(r, s)
        by += 8 * r * s * c["blocks"]
        f += c["steps"] * (4 * m * m * n + 2 * m ** 3) * c["blocks"]
    return {"bytes": by, "flops": f}


def tolerance(case):
    """About four times the largest distance from the 64-bit result measured
    over listed and drawn cases.  Adam's gradients have no typical one: the
    update divides by sqrt(V), and an element whose first chunk gradients are
    all near zero dominates every gradient it reaches (measured 1e-5 to 0.5
    over 60 draws at the same precision)."""
    c, kind = case, case["kind"]
    adam_train = c.get("rule") == "adam" and c["train"]
    if kind == "core":
        if adam_train:
            return {"rel": 0.6}
        if c["dtype"] == "bf16":
            return {"rel": 7e-3}  # the rounding of bfloat16 results: 1.7e-3
        if c["rule"] == "adam":
            return {"rel": 4e-4}
        # other chunk lengths scan in the split precision
        return {"rel": 1e-5 if c["chunk"] == 64 or c["rule"] == "delta" else 4e-4}
    if kind == "scan":
        if c["rule"] == "adam":
            return {"rel": 5e-2 if adam_train else 1e-4}
        return {"rel": 1e-5 if c["precision"] == "ieee" else 2e-5 if c["rule"] == "delta" else 4e-4}
    # block: bfloat16 projections around the core, and gate gradients that
    # cancel; lm: the same through every layer
    return {"rel": {"wy": 7e-3, "block": 0.15, "lm": 0.15, "msign": 1.3e-4}[kind]}


# ------------------------------------------------------------------ the same in 64 bits
def _frob(X):
    return X.square().sum((-2, -1), keepdim=True).sqrt()


def _msign64(M, steps):
    X = M / (_frob(M) + 1e-7)
    for _ in range(steps):
        P = X @ X.transpose(-1, -2)
        X = NS[0] * X + (NS[1] * P + NS[2] * (P @ P)) @ X
    return X


def _scan64(U, K, a, b, m, n, rule, ns):
    """States before each chunk's update; every argument has its chunks along
    dimension 2."""
    a, b, m, n = (t[..., None, None] for t in (a, b, m, n))
    S = torch.zeros_like(U[:, :, 0])
    M, V, states = S, S, []
    for i in range(U.shape[2]):
        states.append(S)
        G = U[:, :, i] - S @ K[:, :, i]
        ai, bi, mi, ni = (t[:, :, i] for t in (a, b, m, n))
        if rule == "delta":
            S = ai * S + G
        elif rule == "muon":
            M = mi * M + G
            S = ai * S + bi * _msign64(M, ns)
        else:
            M = mi * M + (1 - mi) * G
            V = ni * V + (1 - ni) * G * G
            S = ai * S + bi * M / (V.sqrt() + 1e-6)
    return torch.stack(states, 2)


def _core64(q, k, v, beta, la, lm, ln, rule, ns, C):
    B, H, T, d = q.shape
    N = T // C
    q, k, v = (t.reshape(B, H, N, C, d) for t in (q, k, v))
    beta, la = beta.reshape(B, H, N, C), la.clamp_min(LOG_FLOOR).reshape(B, H, N, C)
    lm, ln = (t.clamp_min(LOG_FLOOR).reshape(B, H, N, C) if t is not None else torch.zeros_like(la) for t in (lm, ln))
    if rule == "muon":
        w = (lm.flip(-1).cumsum(-1).flip(-1) - lm).exp()
    else:
        w = beta if rule == "delta" else torch.ones_like(beta)
    A = (q @ k.transpose(-1, -2) * beta[..., None, :]).tril()
    kw = (k * w[..., None]).transpose(-1, -2)
    vw = (v * w[..., None]).transpose(-1, -2)
    S = _scan64(vw @ k, kw @ k, la.sum(-1).exp(), beta.mean(-1), lm.sum(-1).exp(), ln.sum(-1).exp(), rule, ns)
    return ((q - A @ k) @ S.transpose(-1, -2) + A @ v).reshape(B, H, T, d)


def _wy64(q, k, v, beta, la):
    """The token recurrence S <- alpha S (1 - beta k k^T) + beta v k^T,
    o = S q, with the tokens of a chunk solved together: the increments
    x_t = beta_t (v_t - alpha_t S_{t-1} k_t) obey a unit lower triangular
    system within the chunk."""
    B, H, T, d = q.shape
    C, N = 64, T // 64
    q, k, v = (t.reshape(B, H, N, C, d) for t in (q, k, v))
    beta = beta.reshape(B, H, N, C)
    gc = la.clamp_min(LOG_FLOOR).reshape(B, H, N, C).cumsum(-1)
    low = torch.ones(C, C, dtype=torch.bool, device=q.device).tril()
    decay = (gc[..., :, None] - gc[..., None, :]).masked_fill(~low, float("-inf")).exp()
    L = (beta[..., None] * (k @ k.transpose(-1, -2)) * decay).tril(-1)
    M = q @ k.transpose(-1, -2) * decay
    rhs = torch.cat([beta[..., None] * v, (beta * gc.exp())[..., None] * k], -1)
    UW, power = rhs - L @ rhs, L @ L  # (1 + L)^-1 = (1 - L)(1 + L^2)(1 + L^4) .. (1 + L^32): L^64 = 0
    for j in range(5):
        UW = UW + power @ UW
        power = power @ power if j < 4 else power
    S, out = q.new_zeros(B, H, d, d), []
    for i in range(N):
        St = S.transpose(-1, -2)
        X = UW[:, :, i, :, :d] - UW[:, :, i, :, d:] @ St
        out.append(gc[:, :, i, :, None].exp() * (q[:, :, i] @ St) + M[:, :, i] @ X)
        tail = (gc[:, :, i, -1:] - gc[:, :, i]).exp()
        S = gc[:, :, i, -1].exp()[..., None, None] * S + (X * tail[..., None]).transpose(-1, -2) @ k[:, :, i]
    return torch.stack(out, 2).reshape(B, H, T, d)


def _rms64(x, w, eps):
    return x * (x.square().mean(-1, keepdim=True) + eps).rsqrt() * w


def _block64(p, x, c):
    """One pre-norm residual block: conv front-end, the core, head norm, MLP."""
    B, T, D = x.shape
    H = c["H"]
    d, eps, fn = D // H, torch.finfo(torch.float32).eps, torch.nn.functional
    h = _rms64(x, p["n1.weight"], eps)
    y = h @ p["mixer.qkv.weight"].T
    w = p["mixer.conv.weight"]
    y = sum(fn.pad(y, (0, 0, w.shape[-1] - 1 - j, 0))[:, :T] * w[:, 0, j] for j in range(w.shape[-1]))
    q, k, v = (t.reshape(B, T, H, d).transpose(1, 2) for t in fn.silu(y + p["mixer.conv.bias"]).chunk(3, -1))
    q, k = (t / t.norm(dim=-1, keepdim=True).clamp_min(1e-12) for t in (q, k))
    gate = (h @ p["mixer.gates.weight"].T + p["mixer.gates.bias"]).reshape(B, T, -1, H).permute(2, 0, 3, 1)
    la, beta, lm = fn.logsigmoid(gate[0]), gate[1].sigmoid(), fn.logsigmoid(gate[2])
    ln = fn.logsigmoid(gate[3]) if c["rule"] == "adam" else None
    o = _core64(q, k, v, beta, la, lm, ln, c["rule"], c["ns"], 64)
    o = _rms64(o.transpose(1, 2), p["mixer.norm.weight"], eps).reshape(B, T, D)
    x = x + o @ p["mixer.out.weight"].T
    h = _rms64(x, p["n2.weight"], eps)
    return x + fn.gelu(h @ p["mlp.0.weight"].T) @ p["mlp.2.weight"].T


def exact(case, seed):
    c, kind, s = case, case["kind"], prepare(case, seed)

    def wide(t):
        return t.detach().double().requires_grad_(t.requires_grad)

    if kind in ("core", "wy", "scan"):
        ins = [wide(t) for t in s["ins"]]
        with torch.set_grad_enabled(c["train"]):
            if kind == "wy":
                o = _wy64(*ins)
            elif kind == "scan":
                o = _scan64(*ins, c["rule"], c["ns"])
            else:
                o = _core64(*ins, *[None] * (7 - len(ins)), c["rule"], c["ns"], c["chunk"])
        if not c["train"]:
            return [o]
        if not o.requires_grad:  # one chunk: the only state is the initial one
            return [o, *[torch.zeros_like(t) for t in ins if t.requires_grad]]
        grads = torch.autograd.grad(o, [t for t in ins if t.requires_grad], s["dO"].double(), allow_unused=True,
                                    materialize_grads=True)
        return [o.detach(), *grads]
    if kind == "block":
        p = {name: wide(t) for name, t in s["model"].named_parameters()}
        x = wide(s["x"])
        y = _block64(p, x, c)
        return [y.detach(), *torch.autograd.grad(y, [x, *p.values()], s["dy"].double(), allow_unused=True,
                                                 materialize_grads=True)]
    if kind == "lm":
        with torch.no_grad():
            p = {name: t.double() for name, t in s["model"].named_parameters()}
            x = p["emb.weight"][s["idx"]]
            for i in range(c["layers"]):
                pre = "blocks.%d." % i
                x = _block64({n[len(pre):]: t for n, t in p.items() if n.startswith(pre)}, x, c)
            return [_rms64(x, p["norm_f.weight"], torch.finfo(torch.float32).eps) @ p["emb.weight"].T]
    out = []
    for u in s["updates"]:
        u = u.double()
        tall = u.shape[-2] > u.shape[-1]
        X = _msign64(u.transpose(-1, -2) if tall else u, c["steps"])
        out.append((X.transpose(-1, -2) if tall else X).contiguous())
    return out
