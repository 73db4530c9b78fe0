"""Exact WY/UT mode: the token-exact gated delta rule, chunked by the WY/UT
transform (the reference leaves this mode out and trains the chunk-frozen
E-form, train_ablation.py:12-18).

``wy_scan(q, k, v, beta, g)`` returns o (B, H, T, d) of

    S_t = alpha_t S_{t-1} (I - beta_t k_t k_t^T) + beta_t v_t k_t^T,   o_t = S_t q_t,
    alpha_t = exp(max(g_t, log 1e-6)),

for bfloat16 q, k, v (B, H, T, d) (d = 64 or 128, T a multiple of 64) and
float32 beta, g (B, H, T).  Forward and backward are HIP:

* forward (``gmdn_wy_fwd``): a chunk-parallel prep kernel (decay masks, the
  triangular inverse T = (I + A)^-1 by float32 forward substitution, and
  the products that reduce each chunk to the affine state update
  S' = a S + U_A - S K_A and the output o = Qt S^T + Ov), the drop-in delta
  scan kernels and an output kernel.  Its workspace is the backward's
  checkpoint.
* backward (``gmdn_wy_bwd``): dL/dS_i through o, the drop-in delta scan's
  reverse kernel for the state cotangents, then chunk-parallel kernels that
  differentiate the chunk algebra (T, U, W, the decay masks) back to q, k,
  v, beta and g.

Every product is split-bf16 MFMA: bf16 q, k, v enter exactly, float32
operands as hi + lo bf16 (about 2^-16 relative error per product).

``wy_chunk_terms`` restates the chunk algebra as float32 tensor operations;
it documents the prep kernel's quantities and is checked on the CPU against
the oracle's token recurrence.
"""
from __future__ import annotations

import math

import torch

from . import ops  # registers torch.ops.gmdn.*

CHUNK = 64
LOG_FLOOR = math.log(1e-6)


def __getattr__(name: str):
    """The operators ``wy_fwd`` and ``wy_bwd``."""
    if name in ("wy_fwd", "wy_bwd"):
        return getattr(ops, name)
    raise AttributeError(f"module {__name__!r} has no attribute {name!r}")


def wy_chunk_terms(q, k, v, beta, g):
    """Per chunk, in float32: a (B, H, N), U_A, K_A (B, H, N, d, d), Qt, Ov
    (B, H, N, C, d) -- the quantities the prep kernel forms."""
    B, H, T, d = q.shape
    N, C = T // CHUNK, CHUNK
    Q, K, V = (t.float().reshape(B, H, N, C, d) for t in (q, k, v))
    bt = beta.float().reshape(B, H, N, C)
    gcum = torch.cumsum(torch.clamp(g.float(), min=LOG_FLOOR).reshape(B, H, N, C), -1)
    gam = torch.exp(gcum)
    strict = torch.ones(C, C, dtype=torch.bool, device=q.device).tril(-1)
    incl = torch.ones(C, C, dtype=torch.bool, device=q.device).tril()
    # Gamma[t, s] = gamma_t / gamma_s on the causal entries; the exponent is
    # masked before exp, so the (unused) upper triangle is exp(-inf) = 0 and
    # never overflows (an inf there would turn where()'s backward into NaN)
    Gam = torch.exp(torch.where(incl, gcum.unsqueeze(-1) - gcum.unsqueeze(-2), float("-inf")))
    A = torch.where(strict, bt.unsqueeze(-1) * torch.matmul(K, K.transpose(-1, -2)) * Gam, 0.0)
    eye = torch.eye(C, dtype=torch.float32, device=q.device)
    T_ = torch.linalg.solve_triangular(eye + A, eye.expand_as(A), upper=False, unitriangular=True)
    M = torch.where(incl, torch.matmul(Q, K.transpose(-1, -2)) * Gam, 0.0)
    MT = torch.matmul(M, T_)
    kd = torch.exp(gcum[..., -1:] - gcum)
    P = torch.matmul((T_ * kd.unsqueeze(-1)).transpose(-1, -2), K)
    UA = torch.matmul((V * bt.unsqueeze(-1)).transpose(-1, -2), P)
    KA = torch.matmul((K * (bt * gam).unsqueeze(-1)).transpose(-1, -2), P)
    Qt = gam.unsqueeze(-1) * Q - torch.matmul(MT * (bt * gam).unsqueeze(-2), K)
    Ov = torch.matmul(MT * bt.unsqueeze(-2), V)
    return gam[..., -1], UA, KA, Qt, Ov


def wy_scan(q, k, v, beta, g):
    """o of the token-exact gated delta rule; see the module docstring."""
    if not q.is_cuda:
        raise RuntimeError("wy_scan needs GPU tensors")
    ops.ensure()
    if q.dim() != 4 or k.shape != q.shape or v.shape != q.shape:
        raise RuntimeError(f"q, k, v must be (B, H, T, d) of equal shape, got {tuple(q.shape)}")
    B, H, T, d = q.shape
    if d not in (64, 128) or T % CHUNK:
        raise RuntimeError(f"wy_scan supports d in (64, 128) and T a multiple of {CHUNK}, got d={d}, T={T}")
    if any(t.dtype != torch.bfloat16 for t in (q, k, v)):
        raise RuntimeError("wy_scan takes bfloat16 q, k, v")
    for name, t in (("beta", beta), ("g", g)):
        if tuple(t.shape) != (B, H, T):
            raise RuntimeError(f"{name} must be (B, H, T) = {(B, H, T)}, got {tuple(t.shape)}")
    record = torch.is_grad_enabled() and any(t.requires_grad for t in (q, k, v, beta, g))
    o, _ = torch.ops.gmdn.wy_fwd(q, k, v, beta.float(), g.float(), record)
    return o
