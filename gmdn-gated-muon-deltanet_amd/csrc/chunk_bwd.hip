// Level B backward: the fused mixer core's VJP (reference train_ablation.py:142-187
// differentiated through fast_scan.py:72-95 and :134-186).
//
// Per (b, h) and chunk i, with the forward's E-form quantities
//   A = tril(Q K^T) diag(beta),  E = V - K S_i^T,  o = Q S_i^T + A E,
//   G = E^T diag(w) K,  delta: S_{i+1} = a_i S_i + G,
// and Sb_{i+1} = dL/dS_{i+1} (Sb_N = 0), the delta rule's cotangents are
//   Gb  = Sb_{i+1}
//   dE  = A^T dO + diag(w) K Gb^T          (= dV)
//   Sb_i = a_i Sb_{i+1} + dO^T Q - dE^T K
//   dA  = tril(dO E^T)                      (before the beta scaling)
//   dQ  = dO S_i + (dA diag(beta)) K
//   dK  = (dA diag(beta))^T Q - dE S_i + diag(w) E Gb
//   dbeta_s = sum_t dA[t,s] (q_t . k_s) + [delta] (E Gb)[s,:] . k_s
//   dg_t = <Sb_{i+1}, S_i> a_i [g_t >= log 1e-6]
//
// Two kernels per rule:
//  * the reverse recurrence of Sb.  Row r of Sb_i needs only row r of Sb_{i+1}
//    (dE[:, r] = A^T dO[:, r] + diag(w) K Sb[r, :]^T), so one workgroup owns a
//    row block, with an LDS-DMA ring of the chunk's tiles, and writes Gb_i:
//    chunk_bwd_dscan (delta, odd chunks only; chunk_bwd_dscan.hip) and
//    chunk_bwd_ascan (adam at d = 64, every chunk, with the moment
//    cotangents; chunk_bwd_ascan.hip).
//  * the token gradients, chunk-parallel.  From S_i (saved by the forward)
//    and Gb_i they recompute E, A and dE and form dQ, dK, dV and the gate
//    gradients; every contraction over the state's rows is local to the
//    workgroup.  chunk_bwd_tok (adam) takes one chunk per workgroup; the
//    delta rule runs the same phases over chunk pairs (chunk_bwd_pair.hip).
//    The kernel's template still carries the delta branches those phases
//    share.  Adam at d = 64 runs the reverse scan in chunk segments with each
//    segment's token gradients beside the next segment's scan, on a second
//    stream (launch_bwd_adam below).
#include "../../include/gmdn_scan.h"
#include "chunk_b.h"
#include "chunk_prep.h"
#include "muon_bwd.h"
#include "scan_a.h"

#include <mutex>
#include <type_traits>

namespace gmdn {

// ============================================================== chunk_bwd_tok
// One wave per 16 state rows (phase I) and per 16 state columns (phase IIb):
// D / 16 waves, two per SIMD at d = 128, so one wave's global loads overlap
// another's MFMA work (the workgroup's LDS allows one workgroup per CU).
template <int D>
struct TokBwdLds {
  static constexpr int NW = D / 16;
  static constexpr int NTHR = 64 * NW;
  static constexpr int TILE = CB_C * D * 2;
  static constexpr int Q0 = 0, K0 = TILE, V0 = 2 * TILE, O0 = 3 * TILE;
  static constexpr int EH0 = 4 * TILE, EL0 = 5 * TILE;    // E (rows s, columns r), hi / lo
  static constexpr int DH0 = 6 * TILE, DL0 = 7 * TILE;    // dE
  static constexpr int AP = CB_C * CB_C * 2;
  static constexpr int AH0 = 8 * TILE, AL0 = AH0 + AP;    // dA diag(beta), transposed (rows s)
  // floats: per-wave dbeta and (muon) dw partials [NW][64] each, beta, g,
  // gmu, gnu (muon: w), per-wave da partials [NW]
  static constexpr int R0 = AL0 + AP;
  static constexpr int BYTES = R0 + (2 * NW * CB_C + 4 * CB_C + NW) * 4;
  static_assert(BYTES <= 160 * 1024, "token backward LDS exceeds the 160 KiB of a CU");
};

// Adam with four waves (d = 64) keeps its gates in registers and stores
// dbeta per wave (each wave's dA tiles share one token tile), so it needs no
// reduction area: 80 KiB, two workgroups per CU.
// (Not MAT: the drop-in scan's per-chunk gradients keep the general path.)
template <int D, int RULE, bool MAT>
constexpr bool tok_regs() { return RULE == 2 && !MAT && TokBwdLds<D>::NW == 4; }
template <int D, int RULE, bool MAT = false>
constexpr int tok_lds_bytes() { return tok_regs<D, RULE, MAT>() ? TokBwdLds<D>::R0 : TokBwdLds<D>::BYTES; }
static_assert(tok_lds_bytes<64, 2>() <= 80 * 1024, "two adam token workgroups per CU");

// MAT: S_i and Gb_i are the drop-in scan's float32 rows and the chunk
// scalars' gradients arrive as arrays [da | db | dm | dn] (B H N each) in
// p.part -- muon always, adam when its scan ran in exact float32 (d = 128)
template <int D, int RULE, bool MAT = RULE == 1>
GMDN_DEV void chunk_bwd_tok_body(const ChunkArgs& p, int64_t bh, int i) {
  using LQ = BSwz<D>;
  using LA = BSwz<CB_C>;
  using L = TokBwdLds<D>;
  constexpr int NKB = D / 32;
  constexpr int NW = L::NW;
  constexpr int NTHR = L::NTHR;
  extern __shared__ __align__(16) char smem[];
  const bf16* Qs = reinterpret_cast<const bf16*>(smem + L::Q0);
  const bf16* Ks = reinterpret_cast<const bf16*>(smem + L::K0);
  const bf16* Vs = reinterpret_cast<const bf16*>(smem + L::V0);
  const bf16* Os = reinterpret_cast<const bf16*>(smem + L::O0);
  bf16* Eh = reinterpret_cast<bf16*>(smem + L::EH0);
  bf16* El = reinterpret_cast<bf16*>(smem + L::EL0);
  bf16* Dh = reinterpret_cast<bf16*>(smem + L::DH0);
  bf16* Dl = reinterpret_cast<bf16*>(smem + L::DL0);
  bf16* Ah = reinterpret_cast<bf16*>(smem + L::AH0);
  bf16* Al = reinterpret_cast<bf16*>(smem + L::AL0);
  // dbeta and da are summed per wave into the wave's own slots, then over
  // the waves in a fixed order: the gradients are bitwise reproducible
  float* red = reinterpret_cast<float*>(smem + L::R0);
  float* pdbeta = red;               // [NW][64]
  float* pdw = red + NW * CB_C;      // [NW][64] (muon: dL/dw_t)
  float* rbeta = red + 2 * NW * CB_C;  // [64]
  float* rg = rbeta + CB_C;          // [64]
  float* rgmu = rbeta + 2 * CB_C;    // [64] (muon, adam)
  float* rgnu = rbeta + 3 * CB_C;    // [64] (adam; muon: the token weights w)
  float* pda = rbeta + 4 * CB_C;     // [NW]
  // muon reads S_i and Gb_i as float32 rows (the drop-in scan's layout), the
  // others as split pieces: the conversion waits until the rows are used
  auto piece = [](const bf16x8& x) {
    if constexpr (MAT)
      return split_piece(__builtin_bit_cast(f32x4, x));
    else
      return x;
  };

  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = lane_id(), G = l >> 4, lc = l & 15;
  const int64_t bb = bh / p.H, hh = bh % p.H;
  const int64_t t0 = (int64_t)i * CB_C;
  // adam at d = 64: beta of the wave's token tile (16 (w % 4) + lc) in a
  // register; wave 0's lanes keep g, gmu, gnu of their token (gv below)
  constexpr bool REGG = tok_regs<D, RULE, MAT>();
  const float bw = REGG ? p.beta[bh * p.T + t0 + 16 * (w & 3) + lc] : 0.f;
  const float* S = p.states + (bh * p.N + i) * (int64_t)D * D;
  const float* Gb = p.gb + (bh * p.N + i) * (int64_t)D * D;
  const int r0 = 16 * w;  // this wave's state rows (phase I) ...
  const int j0 = 16 * w;  // ... and state columns (phase IIb)

  // ---------------- phase 0: gates, then the q, k tiles (all phase I' needs),
  // the v, dO tiles and the rows r0 + lc of S_i and Gb_i (natural k order),
  // which arrive while phase I' runs
  float gv[4];
  if (threadIdx.x < CB_C) {
    const int64_t e = bh * p.T + t0 + threadIdx.x;
    gv[0] = p.beta[e];
    gv[1] = p.g[e];
    if constexpr (RULE >= 1) gv[2] = p.gmu[e];
    if constexpr (RULE == 2) gv[3] = p.gnu[e];
  }
  {
    DmaPlan<LQ, CB_C, NTHR> pq, pk, pv, po;
    pq.init(w, p.sq[2]);
    pk.init(w, p.sk[2]);
    pv.init(w, p.sv[2]);
    po.init(w, p.so[2]);
    const uint32_t lds0 = lds_addr(smem);
    pq.issue(p.q + bb * p.sq[0] + hh * p.sq[1] + t0 * p.sq[2], lds0 + L::Q0, w);
    pk.issue(p.k + bb * p.sk[0] + hh * p.sk[1] + t0 * p.sk[2], lds0 + L::K0, w);
    pv.issue(p.v + bb * p.sv[0] + hh * p.sv[1] + t0 * p.sv[2], lds0 + L::V0, w);
    po.issue(p.o + bb * p.so[0] + hh * p.so[1] + t0 * p.so[2], lds0 + L::O0, w);
  }
  bf16x8 srow[NKB][2], grow[NKB][2];  // split pieces of columns 32 kb + 8G .. +3, +4 .. +7
#pragma unroll
  for (int kb = 0; kb < NKB; ++kb) {
    const int64_t off = (int64_t)(r0 + lc) * D + 32 * kb + 8 * G;
    srow[kb][0] = *reinterpret_cast<const bf16x8*>(S + off);
    srow[kb][1] = *reinterpret_cast<const bf16x8*>(S + off + 4);
    grow[kb][0] = *reinterpret_cast<const bf16x8*>(Gb + off);
    grow[kb][1] = *reinterpret_cast<const bf16x8*>(Gb + off + 4);
  }
  // vector-memory operations complete in issue order: with the 4 NKB row
  // loads still in flight, the gates and the four tiles have landed
  wait_vmem_le<4 * NKB>();
  if (!REGG && threadIdx.x < CB_C) {
    const int e = threadIdx.x;
    rbeta[e] = gv[0];
    rg[e] = gv[1];
    if constexpr (RULE >= 1) rgmu[e] = gv[2];
    if constexpr (RULE == 2) rgnu[e] = gv[3];
    if constexpr (RULE == 1) {
      // w_t = exp(sum_{s > t} max(gmu_s, log 1e-6)) (train_ablation.py:154-156)
      const float lm = fmaxf(gv[2], LOG_FLOOR);
      const float msum = wave_sum(lm);
      float incl = lm;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const float y = __shfl_up(incl, o, 64);
        if (e >= o) incl += y;
      }
      rgnu[e] = expf(msum - incl);
    }
  }
  __syncthreads();

  // ---------------- phase I': A^T = (tril(Q K^T) diag(beta))^T, split, into the
  // dA planes (free until phase IIa): tile (tt, st), k = 4 tt + st, goes to
  // wave k % NW; tiles above the diagonal are written as zeros
#pragma unroll
  for (int kk = 0; kk < 16 / NW; ++kk) {
    const int k = w + NW * kk, tt = k >> 2, st = k & 3;
    bf16x4 ah, al;
    if (tt < st) {
      ah = al = bf16x4{(bf16)0.f, (bf16)0.f, (bf16)0.f, (bf16)0.f};
    } else {
      f32x4 X = zero4();
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
        X = mfma(row8<LQ>(Qs, 16 * tt + lc, 32 * kb), row8<LQ>(Ks, 16 * st + lc, 32 * kb), X);
      // lane (s, G) holds A[t = 16 tt + 4G + jj][s = 16 st + lc]
      const float bs = REGG ? bw : rbeta[16 * st + lc];
      f32x4 xv;
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) xv[jj] = (tt > st || 4 * G + jj >= lc) ? X[jj] * bs : 0.f;
      split4(xv, ah, al);
    }
    const int ao = LA::off(16 * st + lc, 16 * tt + 4 * G);
    *reinterpret_cast<bf16x4*>(Ah + ao) = ah;
    *reinterpret_cast<bf16x4*>(Al + ao) = al;
  }
  __syncthreads();  // the A planes published (the state rows may still be arriving)

  // ---------------- phase I: E^T, (Gb K^T) and dE^T for this wave's 16 state rows
  Op<2> Sa[NKB], Ga[NKB];  // rows r0 + lc of S_i, Gb_i (m = r, k = c natural); reused in IIb
  {
    float ws[4], dbp[4];
#pragma unroll
    for (int st = 0; st < 4; ++st) ws[st] = RULE == 0 ? rbeta[16 * st + lc] : RULE == 1 ? rgnu[16 * st + lc] : 1.f;
    // column block by column block: the MFMA chains of block kb start as soon
    // as its rows have landed (the loads complete in issue order)
    f32x4 Ets[4], GKs[4];
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      // D layout: lane (s, G) holds rows r0 + 4G + jj
      const bf16x4 vv = *reinterpret_cast<const bf16x4*>(Vs + LQ::off(16 * st + lc, r0 + 4 * G));
      Ets[st] = f32x4{-(float)vv[0], -(float)vv[1], -(float)vv[2], -(float)vv[3]};
      GKs[st] = zero4();
    }
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb) {
      Sa[kb] = join_pieces(piece(srow[kb][0]), piece(srow[kb][1]));
      Ga[kb] = join_pieces(piece(grow[kb][0]), piece(grow[kb][1]));
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        const Op<1> kr{{row8<LQ>(Ks, 16 * st + lc, 32 * kb)}};
        Ets[st] = mma<2, 1>(Sa[kb], kr, Ets[st]);
        GKs[st] = mma<2, 1>(Ga[kb], kr, GKs[st]);
      }
      __builtin_amdgcn_sched_barrier(0);  // keep each block's wait after the previous block's MFMAs
    }
    // the loop below has no cross-lane step, so the LDS reads of one token
    // tile overlap the MFMA chains of the previous one
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      const f32x4 Et = -Ets[st];  // E^T = V^T - S K^T
      const f32x4 GK = GKs[st];
      dbp[st] = dot4(Et, GK);  // dbeta's diag(w) term, this lane's 4 rows
      f32x4 dEt = GK * ws[st];
#pragma unroll
      for (int kbt = 0; kbt < 2; ++kbt) {
        if (32 * kbt + 31 < 16 * st) continue;
        const Op<1> dOt{{col8<LQ>(Os, 32 * kbt, r0)}};  // dO^T (m = r, k = t)
        const Op<2> At{{row8<LA>(Ah, 16 * st + lc, 32 * kbt), row8<LA>(Al, 16 * st + lc, 32 * kbt)}};
        dEt = mma<1, 2>(dOt, At, dEt);  // (k = t, n = s)
      }
      bf16x4 eh, el, dh, dl;
      split4(Et, eh, el);
      split4(dEt, dh, dl);
      const int eo = LQ::off(16 * st + lc, r0 + 4 * G);
      *reinterpret_cast<bf16x4*>(Eh + eo) = eh;
      *reinterpret_cast<bf16x4*>(El + eo) = el;
      *reinterpret_cast<bf16x4*>(Dh + eo) = dh;
      *reinterpret_cast<bf16x4*>(Dl + eo) = dl;
    }
    if constexpr (RULE == 0) {
      // dbeta's diag(w) term: sum_r E[s][r] (Gb k_s)[r] over the wave's rows
#pragma unroll
      for (int st = 0; st < 4; ++st) dbp[st] = group_sum(dbp[st]);
      if (G == 0) {
#pragma unroll
        for (int st = 0; st < 4; ++st) pdbeta[w * CB_C + 16 * st + lc] = dbp[st];
      }
      // delta: Gb_i = Sb_{i+1}, so da_i = <Gb_i, S_i>: the trace of this
      // wave's 16 x 16 diagonal block of Gb_i S_i^T (A = Gb rows, B = S rows)
      f32x4 T = zero4();
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb) T = mma<2, 2>(Ga[kb], Sa[kb], T);
      // lane (n, G) holds entries (4G + jj, n): the diagonal is jj = n - 4G
      const float dpart = (lc >> 2) == G ? T[lc & 3] : 0.f;
      const float da_w = wave_sum(dpart);
      if (l == 0) pda[w] = da_w;
    } else {
      if constexpr (RULE == 1) {
        // muon: sum_r E[s][r] (Gb k_s)[r] is dL/dw_s (w depends on gmu only)
#pragma unroll
        for (int st = 0; st < 4; ++st) dbp[st] = group_sum(dbp[st]);
        if (G == 0) {
#pragma unroll
          for (int st = 0; st < 4; ++st) pdw[w * CB_C + 16 * st + lc] = dbp[st];
        }
      }
      if (!REGG && G == 0) {
#pragma unroll
        for (int st = 0; st < 4; ++st) pdbeta[w * CB_C + 16 * st + lc] = 0.f;
      }
    }
  }
  __syncthreads();

  // ---------------- phase IIa: dA = tril(dO E^T), dbeta's A term, dA diag(beta) -> LDS
  // tiles k = 4 tt + st, k = w, w + NW, ...; tiles above the diagonal are zeroed
  float dbk[16 / NW];
#pragma unroll
  for (int kk = 0; kk < 16 / NW; ++kk) {
    dbk[kk] = 0.f;
    const int k = w + NW * kk, tt = k >> 2, st = k & 3;
    bf16x4 ah, al;
    if (tt < st) {
      ah = al = bf16x4{(bf16)0.f, (bf16)0.f, (bf16)0.f, (bf16)0.f};
    } else {
      f32x4 P = zero4(), QK = zero4();
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb) {
        const Op<1> dOr{{row8<LQ>(Os, 16 * tt + lc, 32 * kb)}};
        const Op<2> Er{{row8<LQ>(Eh, 16 * st + lc, 32 * kb), row8<LQ>(El, 16 * st + lc, 32 * kb)}};
        P = mma<1, 2>(dOr, Er, P);
        QK = mfma(row8<LQ>(Qs, 16 * tt + lc, 32 * kb), row8<LQ>(Ks, 16 * st + lc, 32 * kb), QK);
      }
      const float bs = REGG ? bw : rbeta[16 * st + lc];
      float db = 0.f;
      f32x4 pb;
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        const float pv = (tt > st || 4 * G + jj >= lc) ? P[jj] : 0.f;
        db += pv * QK[jj];
        pb[jj] = pv * bs;
      }
      split4(pb, ah, al);
      dbk[kk] = db;
    }
    const int ao = LA::off(16 * st + lc, 16 * tt + 4 * G);
    *reinterpret_cast<bf16x4*>(Ah + ao) = ah;
    *reinterpret_cast<bf16x4*>(Al + ao) = al;
  }
  {
    // the wave's tiles k = w + NW kk all have st = w % 4
    static_assert(NW % 4 == 0, "a wave's phase IIa tiles share one token tile");
    float db = 0.f;
#pragma unroll
    for (int kk = 0; kk < 16 / NW; ++kk) {
      const int k = w + NW * kk, tt = k >> 2, st = k & 3;
      const float v = group_sum(dbk[kk]);
      if (tt >= st) db += v;
    }
    if constexpr (REGG) {
      // adam: dbeta of the wave's tokens 16 w + lc, the A term and
      // db / 64 (b = mean(beta); db from the reverse scan's partial sums)
      if (G == 0) {
        const float* pp = p.part + (bh * p.N + i) * (int64_t)(D / 16) * 4;
        float sdb = 0.f;
#pragma unroll
        for (int r = 0; r < D / 16; ++r) sdb += pp[4 * r + 1];
        p.dbeta[bh * p.T + t0 + 16 * w + lc] = db + sdb * (1.f / CB_C);
      }
    } else {
      if (G == 0) pdbeta[w * CB_C + 16 * (w & 3) + lc] += db;
    }
  }
  __syncthreads();

  // ---------------- gate gradients and dV
  if (w == 0) {
    const int64_t o = bh * p.T + t0 + l;
    const float a = expf(wave_sum(fmaxf(REGG ? gv[1] : rg[l], LOG_FLOOR)));
    float rdb = 0.f;
    if constexpr (!REGG) {
#pragma unroll
      for (int q = 0; q < NW; ++q) rdb += pdbeta[q * CB_C + l];
    }
    if constexpr (RULE == 0) {
      float da = 0.f;
#pragma unroll
      for (int q = 0; q < NW; ++q) da += pda[q];
      p.dbeta[o] = rdb;
      p.dg[o] = rg[l] >= LOG_FLOOR ? da * a : 0.f;
    } else if constexpr (RULE == 1) {
      // da, db, dm from the drop-in scan's backward: part = [da | db | dm] (B H N each)
      const int64_t BHN = p.B * p.H * p.N, si = bh * p.N + i;
      const float da = p.part[si], db = p.part[BHN + si], dm = p.part[2 * BHN + si];
      const float m = expf(wave_sum(fmaxf(rgmu[l], LOG_FLOOR)));
      float dw = 0.f;
#pragma unroll
      for (int q = 0; q < NW; ++q) dw += pdw[q * CB_C + l];
      // d/dlm_t: m (all t) and w_s for s < t (w_s = exp(sum_{u > s} lm_u))
      const float x = dw * rgnu[l];
      float incl = x;
#pragma unroll
      for (int q = 1; q < 64; q <<= 1) {
        const float y = __shfl_up(incl, q, 64);
        if (l >= q) incl += y;
      }
      p.dbeta[o] = rdb + db * (1.f / CB_C);  // b = mean(beta)
      p.dg[o] = rg[l] >= LOG_FLOOR ? da * a : 0.f;
      p.dgmu[o] = rgmu[l] >= LOG_FLOOR ? (incl - x) + dm * m : 0.f;
    } else {
      // da, db, dm, dn: sums of the reverse scan's per-row-block partials,
      // or (MAT) the drop-in scan's per-chunk gradients
      float sc[4] = {0.f, 0.f, 0.f, 0.f};
      if constexpr (MAT) {
        const int64_t BHN = p.B * p.H * p.N, si = bh * p.N + i;
#pragma unroll
        for (int c = 0; c < 4; ++c) sc[c] = p.part[c * BHN + si];
      } else {
        const float* pp = p.part + (bh * p.N + i) * (int64_t)(D / 16) * 4;
#pragma unroll
        for (int r = 0; r < D / 16; ++r)
#pragma unroll
          for (int c = 0; c < 4; ++c) sc[c] += pp[4 * r + c];
      }
      if constexpr (REGG) {  // g, gmu, gnu of token l in this wave's registers
        const float m = expf(wave_sum(fmaxf(gv[2], LOG_FLOOR)));
        const float n = expf(wave_sum(fmaxf(gv[3], LOG_FLOOR)));
        p.dg[o] = gv[1] >= LOG_FLOOR ? sc[0] * a : 0.f;
        p.dgmu[o] = gv[2] >= LOG_FLOOR ? sc[2] * m : 0.f;
        p.dgnu[o] = gv[3] >= LOG_FLOOR ? sc[3] * n : 0.f;
      } else {
        const float m = expf(wave_sum(fmaxf(rgmu[l], LOG_FLOOR)));
        const float n = expf(wave_sum(fmaxf(rgnu[l], LOG_FLOOR)));
        p.dbeta[o] = rdb + sc[1] * (1.f / CB_C);  // b = mean(beta)
        p.dg[o] = rg[l] >= LOG_FLOOR ? sc[0] * a : 0.f;
        p.dgmu[o] = rgmu[l] >= LOG_FLOOR ? sc[2] * m : 0.f;
        p.dgnu[o] = rgnu[l] >= LOG_FLOOR ? sc[3] * n : 0.f;
      }
    }
  }
  {
    bf16* dvg = p.dv + bb * p.sv[0] + hh * p.sv[1] + t0 * p.sv[2];
    for (int e = threadIdx.x; e < CB_C * D / 8; e += NTHR) {
      const int r = e / (D / 8), c8 = (e % (D / 8)) * 8;
      *reinterpret_cast<bf16x8*>(dvg + r * p.sv[2] + c8) = *reinterpret_cast<const bf16x8*>(Dh + LQ::off(r, c8));
    }
  }

  // ---------------- phase IIb: dQ and dK for this wave's 16 state columns
  //   dQ = (dA diag(beta)) K + dO S,   dK = (dA diag(beta))^T Q - dE S + diag(w) E Gb
  // Every product has its operands swapped, so the tiles are the transposes
  // (lane <-> token, registers <-> 4 consecutive state columns) and each
  // leaves in one 8-byte store.
  bf16* dqg = p.dq + bb * p.sq[0] + hh * p.sq[1] + t0 * p.sq[2];
  bf16* dkg = p.dk + bb * p.sk[0] + hh * p.sk[1] + t0 * p.sk[2];
  f32x4 dqa[4], dka[4], des[4], eg[4];
  // the dA terms first: they are the last readers of the Q and K tiles
#pragma unroll
  for (int tt = 0; tt < 4; ++tt) {
    dqa[tt] = zero4();
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      if (32 * ks > 16 * tt + 15) continue;
      const Op<2> dA{{col8<LA>(Ah, 32 * ks, 16 * tt), col8<LA>(Al, 32 * ks, 16 * tt)}};
      dqa[tt] = mma<1, 2>(Op<1>{{col8<LQ>(Ks, 32 * ks, j0)}}, dA, dqa[tt]);
    }
  }
#pragma unroll
  for (int st = 0; st < 4; ++st) {
    dka[st] = des[st] = eg[st] = zero4();
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
      if (32 * kt + 31 < 16 * st) continue;
      const Op<2> dAT{{row8<LA>(Ah, 16 * st + lc, 32 * kt), row8<LA>(Al, 16 * st + lc, 32 * kt)}};
      dka[st] = mma<1, 2>(Op<1>{{col8<LQ>(Qs, 32 * kt, j0)}}, dAT, dka[st]);
    }
  }
  // The products over the state's rows need S_i and Gb_i by columns.  They
  // are transposed on chip: the rows still held from phase I pass through
  // the (now free) Q and K tiles one 32-row block at a time, split planes
  // of [32 rows][D], and every wave reads its 16 columns back transposed.
  bf16* Sh = reinterpret_cast<bf16*>(smem + L::Q0);
  bf16* Sl = Sh + 32 * D;
  bf16* Gh = reinterpret_cast<bf16*>(smem + L::K0);
  bf16* Gl = Gh + 32 * D;
  __syncthreads();  // Q and K tiles free
#pragma unroll
  for (int kb = 0; kb < NKB; ++kb) {
    if ((w >> 1) == kb) {  // waves 2kb, 2kb+1 hold rows 32 kb .. 32 kb + 31
      const int lr = 16 * (w & 1) + lc;
#pragma unroll
      for (int kc = 0; kc < NKB; ++kc) {
        const int so = LQ::off(lr, 32 * kc + 8 * G);
        *reinterpret_cast<bf16x8*>(Sh + so) = Sa[kc].v[0];
        *reinterpret_cast<bf16x8*>(Sl + so) = Sa[kc].v[1];
        *reinterpret_cast<bf16x8*>(Gh + so) = Ga[kc].v[0];
        *reinterpret_cast<bf16x8*>(Gl + so) = Ga[kc].v[1];
      }
    }
    __syncthreads();
    // columns j0 + lc, rows 32 kb + (k = 8G .. 8G + 7): (k = r natural, n = j)
    const Op<2> sc{{col8<LQ>(Sh, 0, j0), col8<LQ>(Sl, 0, j0)}};
    const Op<2> gc{{col8<LQ>(Gh, 0, j0), col8<LQ>(Gl, 0, j0)}};
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) dqa[tt] = mma<2, 1>(sc, Op<1>{{row8<LQ>(Os, 16 * tt + lc, 32 * kb)}}, dqa[tt]);
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      const Op<2> Er{{row8<LQ>(Eh, 16 * st + lc, 32 * kb), row8<LQ>(El, 16 * st + lc, 32 * kb)}};
      const Op<2> Dr{{row8<LQ>(Dh, 16 * st + lc, 32 * kb), row8<LQ>(Dl, 16 * st + lc, 32 * kb)}};
      eg[st] = mma<2, 2>(gc, Er, eg[st]);
      des[st] = mma<2, 2>(sc, Dr, des[st]);
    }
    if (kb + 1 < NKB) __syncthreads();  // before the next block overwrites the staging planes
  }
  // dQ and dK: staged as [64 tokens][D] bf16 tiles in the V tile and the dA
  // planes (both free since phase I / the dA terms), then stored in rows
  bf16* dqs = reinterpret_cast<bf16*>(smem + L::V0);
  bf16* dks = Ah;
  static_assert(2 * L::AP >= L::TILE, "the dA planes hold one [64][D] bf16 tile");
  // lane (t, G) of transposed tile tt holds dQ[16 tt + t][j0 + 4G .. +3]
#pragma unroll
  for (int tt = 0; tt < 4; ++tt)
    *reinterpret_cast<bf16x4*>(dqs + LQ::off(16 * tt + lc, j0 + 4 * G)) =
        to_bf16x4(dqa[tt]);
#pragma unroll
  for (int st = 0; st < 4; ++st) {
    f32x4 e = eg[st];
    if constexpr (RULE == 0) e = e * rbeta[16 * st + lc];  // diag(w) E Gb, w = beta of token 16 st + lc
    if constexpr (RULE == 1) e = e * rgnu[16 * st + lc];   // muon: w_t
    const f32x4 acc = dka[st] - des[st] + e;
    *reinterpret_cast<bf16x4*>(dks + LQ::off(16 * st + lc, j0 + 4 * G)) =
        to_bf16x4(acc);
  }
  __syncthreads();
  for (int e = threadIdx.x; e < CB_C * D / 8; e += NTHR) {
    const int r = e / (D / 8), c8 = (e % (D / 8)) * 8;
    *reinterpret_cast<bf16x8*>(dqg + r * p.sq[2] + c8) = *reinterpret_cast<const bf16x8*>(dqs + LQ::off(r, c8));
    *reinterpret_cast<bf16x8*>(dkg + r * p.sk[2] + c8) = *reinterpret_cast<const bf16x8*>(dks + LQ::off(r, c8));
  }
}

// One workgroup per (b, h, chunk).
template <int D, int RULE, bool MAT = RULE == 1>
__global__ void __launch_bounds__(TokBwdLds<D>::NTHR) chunk_bwd_tok(ChunkArgs p) {
  chunk_bwd_tok_body<D, RULE, MAT>(p, blockIdx.x / p.N, (int)(blockIdx.x % p.N));
}

// The token gradients of chunks c0 .. c1 - 1 of every (b, h): a grid-stride
// loop over (b, h, chunk), so that a launch of fewer workgroups than CUs
// leaves CUs to a reverse-scan segment running beside it.
template <int D, int RULE>
__global__ void __launch_bounds__(TokBwdLds<D>::NTHR) chunk_bwd_tok_range(ChunkArgs p, int c0, int c1) {
  const int L = c1 - c0;
  const int64_t n = p.B * p.H * (int64_t)L;
  for (int64_t u = blockIdx.x; u < n; u += gridDim.x) {
    if (u != blockIdx.x) __syncthreads();  // the previous chunk's LDS reads are done
    chunk_bwd_tok_body<D, RULE>(p, u / L, c0 + (int)(u % L));
  }
}

namespace {

// A second stream per device (default priority) and the events that order
// it against the caller's stream, created on first use; the mutex keeps one
// call's records and waits together.
struct AuxStream {
  std::mutex mu;
  bool tried = false, ok = false;
  hipStream_t s = nullptr;
  hipEvent_t ev[8] = {};
  int cus = 0;
};
AuxStream g_aux[64];

AuxStream* aux_stream() {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return nullptr;
  AuxStream& x = g_aux[dev];
  std::lock_guard<std::mutex> lk(x.mu);
  if (!x.tried) {
    x.tried = true;
    bool ok = hipStreamCreateWithFlags(&x.s, hipStreamNonBlocking) == hipSuccess &&
              hipDeviceGetAttribute(&x.cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess;
    for (int k = 0; ok && k < 8; ++k) ok = hipEventCreateWithFlags(&x.ev[k], hipEventDisableTiming) == hipSuccess;
    x.ok = ok;
  }
  return x.ok ? &x : nullptr;
}

}  // namespace

// adam at d = 64: the reverse scan in chunk segments (last chunks first) on
// the caller's stream, each segment's token gradients on the second stream
// beside the next segment's scan (chunk_bwd_tok_range on the CUs the scan's
// B H D / 16 workgroups leave), joined back before returning.  Two segments:
// the last holds the chunks whose token gradients fit one round of one
// workgroup per CU (CUs / (B H) chunks, at most half), the token launch that
// runs alone; each segment costs the scan a pipeline fill, so two beat three
// or more.  Without a carry area, with few chunks, or when the scan's
// workgroups fill more than half the CUs, one scan pass then the token
// kernel.
template <int D>
static hipError_t launch_bwd_adam(const ChunkArgs& a, float* carry, hipStream_t stream) {
  constexpr int lds2 = tok_lds_bytes<D, 2>();
  constexpr int thr2 = TokBwdLds<D>::NTHR;
  const int N = a.N;
  const int64_t scan_wgs = a.B * a.H * (D / 16);
  AuxStream* ax = carry && N >= 16 ? aux_stream() : nullptr;
  if (ax && 2 * scan_wgs > ax->cus) ax = nullptr;
  if (!ax) {
    hipError_t e = chunk_bwd_ascan_launch(a, D, carry, 0, N, stream);
    if (e != hipSuccess) return e;
    auto k2 = chunk_bwd_tok<D, 2>;
    e = hipFuncSetAttribute((const void*)k2, hipFuncAttributeMaxDynamicSharedMemorySize, lds2);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k2, dim3((unsigned)(a.B * a.H * N)), dim3(thr2), lds2, stream, a);
    return hipGetLastError();
  }
  auto kr = chunk_bwd_tok_range<D, 2>;
  hipError_t e = hipFuncSetAttribute((const void*)kr, hipFuncAttributeMaxDynamicSharedMemorySize, lds2);
  if (e != hipSuccess) return e;
  std::lock_guard<std::mutex> lk(ax->mu);
  const int64_t fit = ax->cus / (a.B * a.H);
  const int last = (int)(fit < 1 ? 1 : fit < N / 2 ? fit : N / 2);
  const int nseg = 2;
  const int len[2] = {N - last, last};
  int c1 = N;
  for (int k = 0; k < nseg; ++k) {
    const int c0 = k + 1 < nseg ? c1 - len[k] : 0;
    if ((e = chunk_bwd_ascan_launch(a, D, carry, c0, c1, stream)) != hipSuccess) return e;
    if ((e = hipEventRecord(ax->ev[k], stream)) != hipSuccess) return e;
    if ((e = hipStreamWaitEvent(ax->s, ax->ev[k], 0)) != hipSuccess) return e;
    // beside the next segment's scan: the CUs it leaves; the last segment's
    // token gradients run alone
    const int64_t units = a.B * a.H * (int64_t)(c1 - c0);
    const int64_t free_cus = ax->cus - scan_wgs;
    const int64_t grid = k + 1 < nseg && free_cus > 0 && free_cus < units ? free_cus : units;
    hipLaunchKernelGGL(kr, dim3((unsigned)grid), dim3(thr2), lds2, ax->s, a, c0, c1);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    c1 = c0;
  }
  if ((e = hipEventRecord(ax->ev[7], ax->s)) != hipSuccess) return e;
  return hipStreamWaitEvent(stream, ax->ev[7], 0);
}

template <int D, int RULE>
static hipError_t launch_bwd(const ChunkArgs& a, float* carry, hipStream_t stream) {
  if constexpr (RULE == 0) {
    // delta: the reverse scan (Gb of the odd chunks), then the token
    // gradients of chunk pairs (even checkpoints, odd Gb)
    hipError_t e = chunk_bwd_dscan_launch(a, D, stream);
    if (e != hipSuccess) return e;
    return chunk_bwd_pair_launch(a, D, stream);
  } else {
    // adam: the reverse scan of the state and moment cotangents (Gb of every
    // chunk, per-row-block partial sums), then the token gradients
    return launch_bwd_adam<D>(a, carry, stream);
  }
}

// Muon: the matrix form's per-chunk Kw, Uv and gS (chunk_prep_muon), the
// drop-in muon scan's backward on the forward's S_i, M_i (Newton-Schulz VJP,
// chunks in segments), then the token gradients with Gb_i = dU_i.
size_t chunk_bwd_muon_ws_floats(int64_t BH, int64_t N, int d, int ns) {
  const int64_t BHN = BH * N;
  // (+64: the scan's workspace starts 256-byte aligned after the scalars)
  return (size_t)(4 * BHN * (int64_t)d * d + 8 * BHN + 64 + muon_bwd_ws_total(BH, N, d, ns));
}

size_t chunk_bwd_muon_min_ws_floats(int64_t BH, int64_t N, int d, int ns) {
  const int64_t BHN = BH * N;
  const int64_t prefix = (4 * BHN * (int64_t)d * d + 8 * BHN + 63) & ~(int64_t)63;
  return (size_t)(prefix + muon_bwd_ws_segment_floats(BH, 1, d, ns));
}

// One launch of the pipelined muon backward: the reverse pass of segment k
// (blocks 0 .. nx3 - 1), then blocks for the iterates of segment k + 1, the
// matrix-form stage (Kw, Uv, gS, the chunk scalars) of chunks [p0, p0 + pcur)
// and the token gradients of chunks [t0, t0 + tcur).  Every role but the
// first is chunk-parallel and fills the CUs the B H serial reverse scans
// leave idle; each reads only what earlier launches wrote.
struct MuonPipeArgs {
  MuonSegArgs seg;
  ChunkArgs prep, tok;
  float *Kw, *Uv, *gS, *abm;
  int p0, pcur, t0, tcur;
};

template <int D>
constexpr int muon_pipe_lds() {
  constexpr int a = 2 * NSSplit<D>::BYTES + 64, b = PrepLds<D>::BYTES, c = TokBwdLds<D>::BYTES;
  return a > b ? (a > c ? a : c) : (b > c ? b : c);
}

template <int D>
__global__ void __launch_bounds__(D * 4) chunk_bwd_muon_pipe(MuonPipeArgs a) {
  static_assert(PrepLds<D>::NTHR == D * 4 && TokBwdLds<D>::NTHR == D * 4, "one block size for every role");
  int64_t b = blockIdx.x;
  const int64_t npre = a.seg.BH * a.seg.jcur, nprep = a.seg.BH * a.pcur;
  if (b < a.seg.nx3) {
    muon_x3_body<D>(a.seg, b);
    return;
  }
  b -= a.seg.nx3;
  if (b < npre) {
    muon_pre_body<D>(a.seg, b);
    return;
  }
  b -= npre;
  if (b < nprep) {
    chunk_prep_body<D, 1, true, true>(a.prep, a.Kw, a.Uv, a.gS, a.abm, b / a.pcur, a.p0 + (int)(b % a.pcur));
    return;
  }
  b -= nprep;
  chunk_bwd_tok_body<D, 1>(a.tok, b / a.tcur, a.t0 + (int)(b % a.tcur));
}

template <int D>
static hipError_t launch_bwd_muon_chunks(const ChunkArgs& a, int ns, int precision, float* ws, size_t ws_floats,
                                         hipStream_t stream) {
  const int64_t BH = a.B * a.H, BHN = BH * a.N, mat = (int64_t)D * D;
  float* Kw = ws;
  float* Uv = Kw + BHN * mat;
  float* gS = Uv + BHN * mat;
  float* dU = gS + BHN * mat;
  float* abm = dU + BHN * mat;  // a, b, m, n
  float* part = abm + 4 * BHN;  // da, db, dm, dn
  float* sws = ws + ((part + 4 * BHN - ws + 63) & ~(int64_t)63);  // 16-byte pieces: aligned
  const int64_t sws_floats = (int64_t)ws_floats - (sws - ws);
  const MuonBwdPlan plan = muon_bwd_plan(BH, a.N, D, ns, sws_floats);
  if (precision == GMDN_PREC_TF32 && plan.nbuf == 2) {
    // Segments k = 0, 1, .. of plan.nseg chunks from the end.  Launch k runs
    // segment k's reverse pass, segment k + 1's iterates, segment k + 2's
    // matrix-form stage and segment k - 1's token gradients; two launches
    // before (the first segment's stage, then its iterates with the second
    // segment's stage) and one after (the last segment's token gradients)
    // fill and drain the pipeline.
    const int N = (int)a.N, nseg = (int)plan.nseg;
    auto seg_lo = [&](int k) { return N - (k + 1) * nseg > 0 ? N - (k + 1) * nseg : 0; };
    auto seg_hi = [&](int k) { return N - k * nseg > 0 ? N - k * nseg : 0; };
    const int nsegs = (N + nseg - 1) / nseg;
    MuonPipeArgs pa{};
    MuonSegArgs& sg = pa.seg;
    sg.U = Uv; sg.K = Kw; sg.av = abm; sg.bv = abm + BHN; sg.mv = abm + 2 * BHN;
    sg.S_all = a.states; sg.M_all = a.states + BHN * mat; sg.gS = gS;
    sg.dU = dU; sg.da = part; sg.db = part + BHN; sg.dm = part + 2 * BHN; sg.dn = part + 3 * BHN; sg.ws = sws;
    sg.BH = BH; sg.N = N; sg.ns = ns; sg.nseg = nseg; sg.nbuf = 2;
    pa.prep = a;
    pa.tok = a;
    pa.tok.gb = dU;
    pa.tok.part = part;
    pa.Kw = Kw; pa.Uv = Uv; pa.gS = gS; pa.abm = abm;
    auto k = chunk_bwd_muon_pipe<D>;
    constexpr int lds = muon_pipe_lds<D>();
    hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    // x3 segment (or -1), pre segment, prep chunk range, tok segment
    auto launch = [&](int kx, int kp, int p0, int p1, int kt) {
      const bool x = kx >= 0 && kx < nsegs, pre = kp >= 0 && kp < nsegs, tok = kt >= 0 && kt < nsegs;
      sg.nx3 = x ? (int)BH : 0;
      sg.i0 = x ? seg_lo(kx) : 0; sg.i1 = x ? seg_hi(kx) : 0; sg.xbuf = x ? (kx & 1) : 0;
      sg.j0 = pre ? seg_lo(kp) : 0; sg.jcur = pre ? seg_hi(kp) - seg_lo(kp) : 0; sg.pbuf = pre ? (kp & 1) : 0;
      pa.p0 = p0; pa.pcur = p1 > p0 ? p1 - p0 : 0;
      pa.t0 = tok ? seg_lo(kt) : 0; pa.tcur = tok ? seg_hi(kt) - seg_lo(kt) : 0;
      const int64_t blocks = sg.nx3 + BH * (sg.jcur + pa.pcur + pa.tcur);
      if (blocks == 0) return hipSuccess;
      hipLaunchKernelGGL(k, dim3((unsigned)blocks), dim3(D * 4), lds, stream, pa);
      return hipGetLastError();
    };
    if (e == hipSuccess) e = launch(-1, -1, seg_lo(0), seg_hi(0), -1);
    if (e == hipSuccess) e = launch(-1, 0, seg_lo(1), seg_hi(1), -1);
    for (int kk = 0; e == hipSuccess && kk < nsegs; ++kk)
      e = launch(kk, kk + 1, kk + 2 < nsegs ? seg_lo(kk + 2) : 0, kk + 2 < nsegs ? seg_hi(kk + 2) : 0, kk - 1);
    if (e == hipSuccess) e = launch(-1, -1, 0, 0, nsegs - 1);
    return e;
  }
  hipError_t e = chunk_prep_launch(a, D, 1, true, true, Kw, Uv, gS, abm, stream);
  if (e != hipSuccess) return e;
  ScanArgs sa{};
  sa.U = Uv; sa.K = Kw; sa.a = abm; sa.b = abm + BHN; sa.m = abm + 2 * BHN; sa.n = nullptr;
  sa.S_all = a.states; sa.M_all = a.states + BHN * mat; sa.V_all = nullptr; sa.gS = gS;
  sa.dU = dU; sa.dK = nullptr;
  sa.da = part; sa.db = part + BHN; sa.dm = part + 2 * BHN; sa.dn = part + 3 * BHN;
  sa.BH = BH; sa.N = a.N; sa.dh = D; sa.rule = 1; sa.ns = ns; sa.precision = precision;
  sa.stream = stream;
  e = scan_bwd_muon_launch(sa, sws, sws_floats);
  if (e != hipSuccess) return e;
  ChunkArgs t = a;
  t.gb = dU;
  t.part = part;
  auto k = chunk_bwd_tok<D, 1>;
  e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, TokBwdLds<D>::BYTES);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k, dim3((unsigned)BHN), dim3(TokBwdLds<D>::NTHR), TokBwdLds<D>::BYTES, stream, t);
  return hipGetLastError();
}

// Adam at d = 128 (exact float32 scan): gS per chunk, the drop-in adam
// reverse scan on the forward's S, M, V and stored Kw, Uv, scalars, then the
// token gradients with Gb_i = dU_i.  states = [S | M | V | Kw | Uv | a b m n].
size_t chunk_bwd_adam_mat_ws_floats(int64_t BH, int64_t N, int d) {
  const int64_t BHN = BH * N;
  return (size_t)(2 * BHN * (int64_t)d * d + 8 * BHN + BHN * (d / 16) * 4 + 64);
}

hipError_t chunk_bwd_adam_mat_launch(const ChunkArgs& a, int d, float* ws, hipStream_t stream) {
  if (d != 128) return hipErrorNotSupported;
  constexpr int D = 128;
  const int64_t BH = a.B * a.H, BHN = BH * a.N, mat = (int64_t)D * D;
  const float* S = a.states;
  const float* Kw = S + 3 * BHN * mat;
  const float* Uv = S + 4 * BHN * mat;
  const float* abm = S + 5 * BHN * mat;
  float* gS = ws;
  float* dU = gS + BHN * mat;
  float* abm2 = dU + BHN * mat;  // the prep kernel's copy of the scalars (unused)
  float* sc = abm2 + 4 * BHN;    // da, db, dm, dn
  float* part = ws + ((sc + 4 * BHN - ws + 63) & ~(int64_t)63);
  hipError_t e = chunk_prep_launch(a, D, 2, false, true, nullptr, nullptr, gS, abm2, stream);
  if (e != hipSuccess) return e;
  ScanArgs sa{};
  sa.U = Uv; sa.K = Kw; sa.a = abm; sa.b = abm + BHN; sa.m = abm + 2 * BHN; sa.n = abm + 3 * BHN;
  sa.S_all = a.states; sa.M_all = a.states + BHN * mat; sa.V_all = a.states + 2 * BHN * mat;
  sa.gS = gS; sa.dU = dU;  // no dK: the E-form below accounts for every path through K
  sa.da = sc; sa.db = sc + BHN; sa.dm = sc + 2 * BHN; sa.dn = sc + 3 * BHN;
  sa.BH = BH; sa.N = a.N; sa.dh = D; sa.rule = 2; sa.ns = 0; sa.precision = GMDN_PREC_IEEE;
  sa.stream = stream;
  e = scan_bwd_rows_launch(sa, part);
  if (e != hipSuccess) return e;
  e = scan_bwd_dk_launch(sa, part);
  if (e != hipSuccess) return e;
  ChunkArgs t = a;
  t.gb = dU;
  t.part = sc;
  auto k = chunk_bwd_tok<D, 2, true>;
  e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, TokBwdLds<D>::BYTES);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k, dim3((unsigned)BHN), dim3(TokBwdLds<D>::NTHR), TokBwdLds<D>::BYTES, stream, t);
  return hipGetLastError();
}

hipError_t chunk_bwd_muon_launch(const ChunkArgs& a, int d, int ns, int precision, float* ws, size_t ws_floats,
                                 hipStream_t s) {
  if (d == 128) return launch_bwd_muon_chunks<128>(a, ns, precision, ws, ws_floats, s);
  if (d == 64) return launch_bwd_muon_chunks<64>(a, ns, precision, ws, ws_floats, s);
  return hipErrorNotSupported;
}

hipError_t chunk_bwd_launch(const ChunkArgs& a, int d, int rule, float* ascan_carry, hipStream_t s) {
  if (rule == 0) return d == 128 ? launch_bwd<128, 0>(a, nullptr, s) : launch_bwd<64, 0>(a, nullptr, s);
  // adam at d = 128 is refused by the caller: its VJP is ill-conditioned there
  if (rule == 2 && d == 64) return launch_bwd<64, 2>(a, ascan_carry, s);
  return hipErrorNotSupported;
}

}  // namespace gmdn
