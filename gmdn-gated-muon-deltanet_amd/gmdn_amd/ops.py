"""``torch.ops.gmdn.*``: the C-ABI entry points as registered torch operators.

Each operator wraps one call of ``libgmdn_scan.so`` (include/gmdn_scan.h) on
the tensors' current stream.  All but ``msign`` are C++ (csrc/torch_ops.cpp,
``libgmdn_ops.so``), with autograd on the forward operators; this module
registers their shape-only fake implementations, so that ``torch.compile``
traces through the scan without a graph break (the reference trainer compiles
its model, train_ablation.py:420-422):

* ``gmdn::state_scan(U, K, a, b, m, n, rule, ns, precision, save_moments)
  -> (S_all, M_all, V_all)`` -- the drop-in scan's forward (reference
  ``_TritonScan.forward``, fast_scan.py:360-377).  Inputs are float32 and
  contiguous; ``M_all`` / ``V_all`` are the moment stacks the backward needs
  (empty unless ``save_moments`` and the rule keeps them).
* ``gmdn::state_scan_bwd(...) -> (dU, dK, da, db, dm, dn)`` (reference
  ``_TritonScan.backward``, fast_scan.py:379-396).
* ``gmdn::chunk_fwd(q, k, v, beta, g, gmu, gnu, rule, ns, eps, record)
  -> (o, states)`` -- the fused mixer core (reference train_ablation.py:142-187);
  ``states`` is the library-private state checkpoint (empty unless
  ``record``).
* ``gmdn::chunk_bwd(...) -> (dq, dk, dv, dbeta, dg, dgmu, dgnu)``.
* ``gmdn::front_fwd`` / ``gmdn::front_bwd`` -- the mixer front-end (causal
  depthwise conv, SiLU, q/k norms; train_ablation.py:124-128).
* ``gmdn::gates_fwd`` / ``gmdn::gates_bwd`` -- the gate activations and their
  clamped logs (train_ablation.py:131-134); ``gmdn::head_norm_fwd`` /
  ``gmdn::head_norm_bwd`` -- the per-head RMSNorm of the output (:188).
* ``gmdn::chunk_bwd_muon`` -- the muon core's backward.
* ``gmdn::wy_fwd`` / ``gmdn::wy_bwd`` -- the token-exact mode (gmdn_amd.wy).
* ``gmdn::msign(M, steps, eps) -> X`` -- the outer Muon optimizer's msign of
  a batch of matrices (train_ablation.py:60-73); no autograd (the optimizer
  runs it under ``no_grad``).

Operators cannot return ``None``: absent optional results are empty tensors.
There is no CPU implementation; CPU tensors never reach these operators (the
drop-in dispatcher sends them to its eager path).
"""
from __future__ import annotations

import torch
from torch import Tensor

from . import _native as nat

CHUNK = 64


def _empty(like: Tensor) -> Tensor:
    return like.new_empty((0,), dtype=torch.float32)


def chunk_desc(q: Tensor, k: Tensor, v: Tensor, o: Tensor, rule: int, ns: int, eps: float,
               precision: int = nat.PREC_TF32):
    """The ``gmdn_chunk_desc`` of a call: sizes, rule and the element strides
    of the (B, H, T, d) token streams (``precision``: rule 1's Newton-Schulz
    VJP in the backward)."""
    B, H, T, d = q.shape
    desc = nat.ChunkDesc()
    desc.B, desc.H, desc.T, desc.d, desc.C = B, H, T, d, CHUNK
    dtype = nat.DTYPE_F32 if q.dtype == torch.float32 else nat.DTYPE_BF16
    desc.rule, desc.ns, desc.dtype, desc.eps = rule, ns, dtype, eps
    desc.precision = precision
    for name, t in (("sq", q), ("sk", k), ("sv", v), ("so", o)):
        arr = getattr(desc, name)
        for i in range(3):
            arr[i] = t.stride(i)
    return desc


def _states_numel(q: Tensor, rule: int, ns: int, eps: float) -> int:
    # the checkpoint size depends on the sizes and the rule only
    return nat.load().gmdn_chunk_states_bytes(chunk_desc(q, q, q, q, rule, ns, eps)) // 4


def _keeps_states(q: Tensor, rule: int, record: bool) -> bool:
    """Whether the forward writes the chunk states: for a backward, and always
    where the output kernel reads them (muon; float32 streams, whose matrix
    form runs the drop-in scan between chunk-parallel kernels)."""
    return record or rule == 1 or q.dtype == torch.float32


def _dense_permutation(t: Tensor) -> bool:
    """Whether ``t``'s elements fill its storage extent exactly once: its
    strides are those of a contiguous tensor with permuted dimensions (no
    zero strides from ``expand``, no gaps as in a slice of a wider tensor)."""
    dims = sorted((st, sz) for st, sz in zip(t.stride(), t.shape) if sz != 1)
    want = 1
    for st, sz in dims:
        if st != want:
            return False
        want *= sz
    return True


def _kernel_strides(t: Tensor):
    """The strides of the output and gradient of token stream ``t``: its own
    when they suit the kernels (unit-stride d, B/H/T strides in multiples of
    8 elements) and ``t`` is a dense permutation (an expanded stream would
    make rows alias, a gapped one would leave holes), else contiguous.  The
    data pointer does not enter, so the real and fake implementations agree."""
    if t.stride(-1) != 1 or any(s % 8 for s in t.stride()[:3]) or not _dense_permutation(t):
        return t.new_empty(t.shape).stride()
    return t.stride()


def _wy_ckpt_numel(q: Tensor) -> int:
    return max(nat.load().gmdn_wy_fwd_workspace_bytes(chunk_desc(q, q, q, q, 0, 0, 1e-6)) // 4, 4)


# ------------------------------------------------- fake implementations
def _state_scan_fake(U, K, a, b, m, n, rule, ns, precision, save_moments):
    S_all = torch.empty_like(U)
    M_all = torch.empty_like(U) if (rule != 0 and save_moments) else _empty(U)
    V_all = torch.empty_like(U) if (rule == 2 and save_moments) else _empty(U)
    return S_all, M_all, V_all


def _state_scan_bwd_fake(U, K, a, b, m, n, S_all, M_all, V_all, gS, rule, ns, precision):
    return (torch.empty_like(U), torch.empty_like(K), *(torch.empty_like(a) for _ in range(4)))


def _chunk_fwd_fake(q, k, v, beta, g, gmu, gnu, rule, ns, eps, record):
    o = q.new_empty_strided(q.shape, _kernel_strides(q))
    keep = _keeps_states(q, rule, record)
    states = q.new_empty((_states_numel(q, rule, ns, eps),), dtype=torch.float32) if keep else _empty(q)
    return o, states


def _chunk_bwd_fake(q, k, v, beta, g, gmu, gnu, states, dO, rule, ns, eps):
    dq, dk, dv = (t.new_empty_strided(t.shape, _kernel_strides(t)) for t in (q, k, v))
    dbeta = beta.new_empty(beta.shape, dtype=torch.float32)
    dg = g.new_empty(g.shape, dtype=torch.float32)
    dgmu = gmu.new_empty(gmu.shape, dtype=torch.float32) if gmu is not None else _empty(q)
    dgnu = gnu.new_empty(gnu.shape, dtype=torch.float32) if gnu is not None else _empty(q)
    return dq, dk, dv, dbeta, dg, dgmu, dgnu


def _chunk_bwd_muon_fake(q, k, v, beta, g, gmu, states, dO, ns, precision):
    dq, dk, dv = (t.new_empty_strided(t.shape, _kernel_strides(t)) for t in (q, k, v))
    return dq, dk, dv, beta.new_empty(beta.shape), g.new_empty(g.shape), gmu.new_empty(gmu.shape)


def _wy_fwd_fake(q, k, v, beta, g, record):
    o = q.new_empty_strided(q.shape, _kernel_strides(q))
    return o, (q.new_empty((_wy_ckpt_numel(q),), dtype=torch.float32) if record else _empty(q))


def _wy_bwd_fake(q, k, v, beta, g, ckpt, dO):
    dq, dk, dv = (t.new_empty_strided(t.shape, _kernel_strides(t)) for t in (q, k, v))
    return (dq, dk, dv, beta.new_empty(beta.shape, dtype=torch.float32),
            g.new_empty(g.shape, dtype=torch.float32))


def _front_fwd_fake(y, weight, bias, dh):
    B, T, C3 = y.shape
    return tuple(y.new_empty(B, T, C3 // 3) for _ in range(3))


def _front_bwd_fake(y, weight, bias, dq, dk, dv, dh):
    return y.new_empty(y.shape), torch.empty_like(weight), torch.empty_like(bias)


def _gates_fwd_fake(y, heads, n_gates):
    B, T, C = y.shape
    return y.new_empty((n_gates, B, heads, T), dtype=torch.float32)


def _gates_bwd_fake(y, dout, heads, n_gates):
    return torch.empty_like(y, memory_format=torch.contiguous_format)


def _head_norm_fwd_fake(x, weight, eps):
    return (torch.empty_like(x, memory_format=torch.contiguous_format),
            x.new_empty(x.shape[:-1], dtype=torch.float32))


def _head_norm_bwd_fake(x, weight, rstd, dout):
    return torch.empty_like(x, memory_format=torch.contiguous_format), weight.new_empty(weight.shape)


_FAKES = {
    "state_scan": _state_scan_fake,
    "state_scan_bwd": _state_scan_bwd_fake,
    "chunk_fwd": _chunk_fwd_fake,
    "chunk_bwd": _chunk_bwd_fake,
    "chunk_bwd_muon": _chunk_bwd_muon_fake,
    "wy_fwd": _wy_fwd_fake,
    "wy_bwd": _wy_bwd_fake,
    "front_fwd": _front_fwd_fake,
    "front_bwd": _front_bwd_fake,
    "gates_fwd": _gates_fwd_fake,
    "gates_bwd": _gates_bwd_fake,
    "head_norm_fwd": _head_norm_fwd_fake,
    "head_norm_bwd": _head_norm_bwd_fake,
}
# Set by _register_fakes.  Without the native libraries the operators do not
# exist: every entry point calls ensure(), which raises what _native.load raises.
REGISTERED = False


def _register_fakes():
    global REGISTERED
    for name, fake in _FAKES.items():
        torch.library.register_fake(f"gmdn::{name}", fake)
    REGISTERED = True


nat.when_loaded(_register_fakes)
nat.available()


def ensure() -> None:
    """Load the operators if they are not registered yet (the libraries may
    have been built after this module's import)."""
    if not REGISTERED:
        nat.load()


def __getattr__(name: str):
    """The C++ operators by name, as ``msign`` is: ``ops.chunk_fwd(...)``."""
    if name in _FAKES:
        ensure()
        return getattr(torch.ops.gmdn, name)
    raise AttributeError(f"module {__name__!r} has no attribute {name!r}")


def _dtype_code(t: Tensor) -> int:
    if t.dtype == torch.bfloat16:
        return nat.DTYPE_BF16
    if t.dtype == torch.float32:
        return nat.DTYPE_F32
    raise RuntimeError(f"the mixer front-end kernels take bfloat16 or float32, got {t.dtype}")


# ------------------------------------------------------------ outer msign
@torch.library.custom_op("gmdn::msign", mutates_args=(), device_types="cuda")
def msign(M: Tensor, steps: int, eps: float) -> Tensor:
    """msign of each matrix of ``M`` (..., rows, cols), float32 or bfloat16,
    result in ``M``'s dtype (reference train_ablation.py:60-73)."""
    lib = nat.load()
    if M.dim() < 2:
        raise RuntimeError(f"msign needs a matrix or a batch of matrices, got shape {tuple(M.shape)}")
    if M.dtype not in (torch.float32, torch.bfloat16):
        raise RuntimeError(f"gmdn::msign takes float32 or bfloat16, got {M.dtype}")
    rows, cols = M.shape[-2], M.shape[-1]
    Mc = M.contiguous()
    out = torch.empty_like(Mc)
    batch = Mc.numel() // max(rows * cols, 1) if rows * cols else 0
    if batch == 0:
        return out
    ws = torch.empty(lib.gmdn_msign_workspace_bytes(batch, rows, cols), dtype=torch.uint8, device=M.device)
    with torch.cuda.device(M.device):
        rc = lib.gmdn_msign(nat.ptr(Mc), nat.ptr(out), batch, rows, cols, steps, eps, _dtype_code(Mc), nat.ptr(ws),
                            ws.numel(), nat.stream_of(Mc))
    nat.check(rc, "gmdn_msign")
    return out


@msign.register_fake
def _msign_fake(M, steps, eps):
    return torch.empty_like(M, memory_format=torch.contiguous_format)
