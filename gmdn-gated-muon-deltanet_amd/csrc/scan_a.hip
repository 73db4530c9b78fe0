// Level A: the drop-in chunk state scan, fast_state_scan(U, K, a, b, m, n,
// rule, ns) (reference fast_scan.py:403-414; kernels :206-331; math :72-186).
//
// Row-separable rules (delta, adam).  Row r of G_i = U_i - S_i K_i needs only
// row r of S_i, and the delta/adam updates are elementwise, so every 16-row
// tile of S is an independent recurrence.  A workgroup owns 16 rows (exact
// float32 products: scan_fwd_rowsf, scan_bwd_rowsf) or 32 rows (bf16x3:
// scan_fwd_rows8, scan_bwd_rows8) for the whole sequence; its waves hold
// D-layout tiles of S^T (lane <-> row r, registers <-> columns c).
//
//   forward, chunk i, rows r:
//     G^T = U^T - K^T S^T       (MFMA tiles: A = K^T, B = -S^T)
//     delta: S^T <- a S^T + G^T
//     adam : M^T <- m M^T + (1-m) G^T ; V^T <- n V^T + (1-n) G^T.^2 ;
//            S^T <- a S^T + b M^T / (sqrt(V^T) + eps)
//
//   backward (reverse over chunks; Sb = dL/dS_{i+1}):
//     delta: Gb = Sb
//     adam : elementwise VJP of the moments (fast_scan.py:167-182)
//     dU_i = Gb ;  Sb <- a Sb - Gb K^T + gS_i   (A = K rows, B = -Gb^T)
//   dK_i = -S_i^T Gb_i and the scalar gradients are formed per chunk by a
//   second, chunk-parallel kernel (contraction over all rows of S).
#include "prec.h"
#include "scan_a.h"

namespace gmdn {

// blockIdx -> (bh, row block).  Workgroups are dispatched round-robin over
// the 8 XCDs; keep all row blocks of one (b, h) on one XCD so they share its
// K_i stream through that XCD's L2.
GMDN_DEV void map_rows_block(int64_t BH, int nblk, int64_t& bh, int& blk) {
  const int64_t x = blockIdx.x;
  if (BH % 8 == 0) {
    const int64_t xcd = x & 7, slot = x >> 3;
    blk = (int)(slot % nblk);
    bh = (slot / nblk) * 8 + xcd;
  } else {
    bh = x / nblk;
    blk = (int)(x % nblk);
  }
}

// ------------------------------------ exact float32: D/16 waves per 16 rows
// One workgroup of D/16 waves per 16 rows of S; wave w holds column tile w
// (one D-layout tile of S^T per lane, four values).  v_mfma_f32_16x16x4_f32
// steps take the contraction in the order k = 16 t + 4 G + e (tile t, step e,
// lane group G), so that the shared operand, the workgroup's 16 rows of S, is
// one 16-byte LDS read per tile from an exchange each wave writes one 16-byte
// piece of (padded rows: conflict-free; double buffered: one barrier a chunk).
// A wave reads its own 16 columns of K_i only, so K_i goes straight from
// global memory to the operand registers, two chunks in flight, and never
// through LDS.
//
// Bound: the MFMA pipe (D/4 products of 32 cycles per wave and chunk, two
// waves a SIMD at D = 128: 0.85 us a chunk) and the chain around it.  The
// rows used to be split over waves (16 rows x all columns a wave, K_i through
// LDS as float32): eight times the products and the elementwise update in one
// wave's chain, two of the four SIMDs idle. Measured (adam, d = 128, 32 chunks):
// 423 -> 77 us at 16 heads, 445 -> 235 us at 64; adam d = 64, 8 heads, 16
// chunks 60 -> 19 us; delta d = 128, 64 heads, 64 chunks 478 -> 330 us.
template <int D>
struct RowsfLds {
  static constexpr int LD = D + 4;          // padded row of the exchange
  static constexpr int X = 16 * LD;         // floats of one buffer
};

template <int D, int RULE>
__global__ void __launch_bounds__(D * 4)
scan_fwd_rowsf(const float* __restrict__ U, const float* __restrict__ K,
               const float* __restrict__ av, const float* __restrict__ bv,
               const float* __restrict__ mv, const float* __restrict__ nv,
               float* __restrict__ S_all, float* __restrict__ M_all,
               float* __restrict__ V_all, int64_t BH, int N) {
  constexpr int NT = D / 16;
  constexpr int LD = RowsfLds<D>::LD;
  __shared__ __align__(16) float xs[2][RowsfLds<D>::X];

  int64_t bh;
  int blk;
  map_rows_block(BH, NT, bh, blk);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = lane_id(), G = l >> 4, rl = l & 15;
  const int64_t mat = (int64_t)D * D;
  const int64_t base = bh * N * mat;
  // 32-bit lane offsets from scalar bases
  const uint32_t so = (16 * blk + rl) * D + 16 * w + 4 * G;  // this lane's piece of a state
  const uint32_t ko = 4 * G * D + 16 * w + rl;               // K columns of tile w

  struct Chunk {  // one chunk's operands of this lane
    float k[NT][4];
    f32x4 u;
    float a, b, m, n;
  };
  auto load = [&](Chunk& c, int i) {
    const int64_t o = base + i * mat;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) c.k[t][e] = (K + o + (16 * t + e) * D)[ko];
    c.u = *reinterpret_cast<const f32x4*>(U + o + so);
    const int64_t si = bh * N + i;
    c.a = av[si];
    if constexpr (RULE == 2) {
      c.b = bv[si];
      c.m = mv[si];
      c.n = nv[si];
    }
  };

  f32x4 S = zero4(), M = zero4(), V = zero4();
  auto step = [&](Chunk& c, int i) {
    float* const x = xs[i & 1];
    // pre-update state (and adam's moments); -S^T to the exchange
    *reinterpret_cast<f32x4*>(S_all + base + i * mat + so) = S;
    if constexpr (RULE == 2) {
      if (M_all) *reinterpret_cast<f32x4*>(M_all + base + i * mat + so) = M;
      if (V_all) *reinterpret_cast<f32x4*>(V_all + base + i * mat + so) = V;
    }
    *reinterpret_cast<f32x4*>(x + rl * LD + 16 * w + 4 * G) = -S;
    __syncthreads();
    // delta: two chains, 0.73 of one chain's error; adam: one, which its
    // reverse scan repeats bit for bit
    f32x4 g = c.u, g1 = zero4();
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const f32x4 s = *reinterpret_cast<const f32x4*>(x + rl * LD + 16 * t + 4 * G);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (RULE == 0 && (t & 1))
          g1 = mfma_f32(c.k[t][e], s[e], g1);
        else
          g = mfma_f32(c.k[t][e], s[e], g);
      }
    }
    if constexpr (RULE == 0) g += g1;
    const float a = c.a, b = c.b, m = c.m, n = c.n;
    if (i + 2 < N) load(c, i + 2);
    if constexpr (RULE == 0) {
      S = a * S + g;
    } else {
      M = m * M + (1.f - m) * g;
      V = n * V + (1.f - n) * g * g;
#pragma unroll
      for (int j = 0; j < 4; ++j) S[j] = a * S[j] + b * M[j] / (sqrtf(V[j]) + 1e-6f);
    }
  };

  Chunk c0, c1;
  load(c0, 0);
  load(c1, N > 1 ? 1 : 0);
  int i = 0;
  for (; i + 1 < N; i += 2) {
    step(c0, i);
    step(c1, i + 1);
  }
  if (i < N) step(c0, i);
}

// ------------------------------------- forward, 8 waves per 32 rows (bf16x3)
// The same recurrence with one workgroup of 8 waves per 32 rows of S: wave
// (rt, cq) holds rows 32 blk + 16 rt + lc and column quarter cq as D-layout
// tiles of S^T.  The contraction G = U - S K runs over all columns of S, so
// the workgroup's rows are exchanged each chunk as split bf16 planes in LDS;
// K_i is staged once per chunk, as split bf16 planes (double buffered), by
// all 512 threads from fp32 loads issued one chunk ahead.  Every MFMA operand
// is then a plain LDS read.
template <int D>
struct Rows8Lds {
  static constexpr int PLANE = D * D * 2;   // one bf16 plane of K_i (bytes)
  static constexpr int K0 = 0;              // [buffer][hi | lo]
  static constexpr int XSP = 32 * D * 2;    // the workgroup's S rows, one plane
  static constexpr int XS0 = K0 + 4 * PLANE;
  static constexpr int BYTES = XS0 + 2 * XSP;
  static_assert(BYTES <= 160 * 1024, "row scan LDS exceeds the 160 KiB of a CU");
};
constexpr int A8_THREADS = 512;

template <int D, int RULE>
__global__ void __launch_bounds__(A8_THREADS)
scan_fwd_rows8(const float* __restrict__ U, const float* __restrict__ K,
               const float* __restrict__ av, const float* __restrict__ bv,
               const float* __restrict__ mv, const float* __restrict__ nv,
               float* __restrict__ S_all, float* __restrict__ M_all,
               float* __restrict__ V_all, int64_t BH, int N) {
  using L = BSwz<D>;
  using R = Rows8Lds<D>;
  using P = PrecX3;
  constexpr int NKB = D / 32;                // k-blocks over all columns of S
  constexpr int TPW = D / 64;                // column tiles per wave
  constexpr int ROWB = D * 2;                // bytes per row of a plane
  constexpr int PR = D / 4;                  // fp32 pieces per row of K
  constexpr int NQ = D * PR / A8_THREADS;    // pieces of K_i per thread
  constexpr int RSTEP = A8_THREADS / PR;     // rows between a thread's pieces
  static_assert(NQ * A8_THREADS == D * PR && RSTEP % 16 == 0, "K pieces split in swizzle-keeping row steps");
  extern __shared__ __align__(16) float smem[];

  int64_t bh;
  int blk;
  map_rows_block(BH, D / 32, bh, blk);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = lane_id(), G = l >> 4, lc = l & 15;
  const int rt = w >> 2, cq = w & 3;
  const int row = 32 * blk + 16 * rt + lc;   // this lane's row of S
  const int64_t mat = (int64_t)D * D;
  const float* Ub = U + bh * N * mat;
  const float* Kb = K + bh * N * mat;
  const lds_ptr L0 = lds_base(smem);

  // per-lane LDS offsets (row tiles, k-blocks and planes are immediates)
  uint32_t kcol[TPW], xsw[TPW], xsr[NKB][2];
#pragma unroll
  for (int u = 0; u < TPW; ++u) {
    const int ct = cq * TPW + u;
    kcol[u] = swz_off<L>(4 * G + (lc >> 2), 16 * ct + 4 * (lc & 3));
    xsw[u] = swz_off<L>(16 * rt + lc, 16 * ct + 4 * G);
  }
#pragma unroll
  for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
    for (int h = 0; h < 2; ++h) xsr[kb][h] = swz_off<L>(16 * rt + lc, 32 * kb + 16 * h + 4 * G);
  // K staging: thread j takes pieces (j / PR + q RSTEP, 4 (j % PR))
  const int kr = threadIdx.x / PR, kc = (threadIdx.x % PR) * 4;
  const uint32_t kdst = swz_off<L>(kr, kc);
  const int64_t ksrc = (int64_t)kr * D + kc;
  auto roff = [&](int u) { return (int64_t)row * D + 16 * (cq * TPW + u) + 4 * G; };

  f32x4 Kpre[NQ];
  auto load_k = [&](int i) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) Kpre[q] = *reinterpret_cast<const f32x4*>(Kb + i * mat + ksrc + q * RSTEP * D);
  };
  auto stage_k = [&](int buf) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      bf16x4 hi, lo;
      split4(Kpre[q], hi, lo);
      const uint32_t o = R::K0 + buf * 2 * R::PLANE + kdst + q * RSTEP * ROWB;
      lds_st<bf16x4>(L0 + o, hi);
      lds_st<bf16x4>(L0 + (o + R::PLANE), lo);
    }
  };

  f32x4 S[TPW], M[TPW], V[TPW], Unext[TPW];
#pragma unroll
  for (int u = 0; u < TPW; ++u) S[u] = M[u] = V[u] = Unext[u] = zero4();
  if (N > 0) {
    load_k(0);
    stage_k(0);
#pragma unroll
    for (int u = 0; u < TPW; ++u) Unext[u] = *reinterpret_cast<const f32x4*>(Ub + roff(u));
  }
  if (N > 1) load_k(1);
  __syncthreads();

  for (int i = 0; i < N; ++i) {
    const int buf = i & 1;
    const int64_t si = bh * N + i;
    f32x4 Ucur[TPW];
#pragma unroll
    for (int u = 0; u < TPW; ++u) {
      Ucur[u] = Unext[u];
      // pre-update state (and adam's moments)
      *reinterpret_cast<f32x4*>(S_all + si * mat + roff(u)) = S[u];
      if constexpr (RULE == 2) {
        if (M_all) *reinterpret_cast<f32x4*>(M_all + si * mat + roff(u)) = M[u];
        if (V_all) *reinterpret_cast<f32x4*>(V_all + si * mat + roff(u)) = V[u];
      }
      // this wave's split S tile -> the exchange planes
      bf16x4 hi, lo;
      split4(S[u], hi, lo);
      lds_st<bf16x4>(L0 + (R::XS0 + xsw[u]), hi);
      lds_st<bf16x4>(L0 + (R::XS0 + xsw[u] + R::XSP), lo);
    }
    __syncthreads();  // S rows published (K_i staged by the last barrier)
    // B operands: this lane's row of S over every k-block (pair order)
    P::Op Sop[NKB];
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb) {
      Sop[kb].hi = cat8(lds_ld<bf16x4>(L0 + (R::XS0 + xsr[kb][0])), lds_ld<bf16x4>(L0 + (R::XS0 + xsr[kb][1])));
      Sop[kb].lo = cat8(lds_ld<bf16x4>(L0 + (R::XS0 + R::XSP + xsr[kb][0])),
                        lds_ld<bf16x4>(L0 + (R::XS0 + R::XSP + xsr[kb][1])));
    }
    const float a = av[si];
    float b = 0.f, m = 0.f, n = 0.f;
    if constexpr (RULE == 2) {
      b = bv[si];
      m = mv[si];
      n = nv[si];
    }
#pragma unroll
    for (int u = 0; u < TPW; ++u) {
      // (S K)^T tile: A = K^T (column reads of K_i), B = S^T
      f32x4 acc = zero4();
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb) {
        const uint32_t o = R::K0 + buf * 2 * R::PLANE + kcol[u] + kb * 32 * ROWB;
        P::Op A;
        A.hi = cat8(lds_tr16(L0 + o), lds_tr16(L0 + (o + 16 * ROWB)));
        A.lo = cat8(lds_tr16(L0 + (o + R::PLANE)), lds_tr16(L0 + (o + R::PLANE + 16 * ROWB)));
        acc = P::mma(A, Sop[kb], acc);
      }
      const f32x4 g = Ucur[u] - acc;  // G^T = U^T - K^T S^T
      if constexpr (RULE == 0) {
        S[u] = a * S[u] + g;
      } else {
        M[u] = m * M[u] + (1.f - m) * g;
        V[u] = n * V[u] + (1.f - n) * g * g;
#pragma unroll
        for (int j = 0; j < 4; ++j) S[u][j] = a * S[u][j] + b * M[u][j] * hw_rcp(hw_sqrt(V[u][j]) + 1e-6f);
      }
    }
    // K_{i+1} into the other buffer (last read in chunk i-1); loads of K_{i+2}, U_{i+1}
    if (i + 1 < N) {
      stage_k(buf ^ 1);
#pragma unroll
      for (int u = 0; u < TPW; ++u) Unext[u] = *reinterpret_cast<const f32x4*>(Ub + (i + 1) * mat + roff(u));
    }
    if (i + 2 < N) load_k(i + 2);
    __syncthreads();  // K_{i+1} staged; the exchange planes free
  }
}

// ---------------------- reverse scan, exact float32: D/16 waves per 16 rows
// The layout of scan_fwd_rowsf: wave w holds column tile w of Sb^T.  Delta:
// dU_i = Sb, then Sb^T <- a Sb^T + gS^T - K Sb^T with -Sb^T through the
// exchange and A = K_i rows (16-byte loads of the wave's own 16 rows, two
// chunks in flight); da is formed later from dU and S_all. Bound: vector
// memory into a CU (K_i again for each 16 rows). Measured (d = 128, 64 heads,
// 64 chunks): 508 -> 321 us against the two-wave kernel.
template <int D>
__global__ void __launch_bounds__(D * 4)
scan_bwd_rowsf(const float* __restrict__ K, const float* __restrict__ av, const float* __restrict__ gS,
               float* __restrict__ dU, int64_t BH, int N) {
  constexpr int NT = D / 16;
  constexpr int LD = RowsfLds<D>::LD;
  __shared__ __align__(16) float xs[2][RowsfLds<D>::X];

  int64_t bh;
  int blk;
  map_rows_block(BH, NT, bh, blk);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = lane_id(), G = l >> 4, rl = l & 15;
  const int64_t mat = (int64_t)D * D;
  const int64_t base = bh * N * mat;
  // 32-bit lane offsets from scalar bases
  const uint32_t to = (16 * blk + rl) * D + 16 * w + 4 * G;  // this lane's piece of a state
  const uint32_t kro = (16 * w + rl) * D + 4 * G;            // K rows of column tile w

  struct Chunk {
    f32x4 k[NT], gs;
    float a;
  };
  auto load = [&](Chunk& c, int i) {
    const int64_t o = base + i * mat;
#pragma unroll
    for (int t = 0; t < NT; ++t) c.k[t] = *reinterpret_cast<const f32x4*>(K + o + 16 * t + kro);
    c.gs = *reinterpret_cast<const f32x4*>(gS + o + to);
    c.a = av[bh * N + i];
  };
  f32x4 Sb = zero4();
  auto step = [&](Chunk& c, int i) {
    float* const x = xs[i & 1];
    *reinterpret_cast<f32x4*>(x + rl * LD + 16 * w + 4 * G) = -Sb;
    *reinterpret_cast<f32x4*>(dU + base + i * mat + to) = Sb;
    __syncthreads();
    f32x4 a0 = c.a * Sb + c.gs, a1 = zero4();
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const f32x4 gb = *reinterpret_cast<const f32x4*>(x + rl * LD + 16 * t + 4 * G);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (t & 1)
          a1 = mfma_f32(c.k[t][e], gb[e], a1);
        else
          a0 = mfma_f32(c.k[t][e], gb[e], a0);
      }
    }
    Sb = a0 + a1;
    if (i >= 2) load(c, i - 2);
  };
  Chunk c0, c1;
  load(c0, N - 1);
  load(c1, N > 1 ? N - 2 : 0);
  int i = N - 1;
  for (; i >= 1; i -= 2) {
    step(c0, i);
    step(c1, i - 1);
  }
  if (i == 0) step(c0, 0);
}

// Adam: the moment VJP needs G_i = U_i - S_i K_i again, which does not depend
// on the cotangent, so chunk i - 1's is formed in step i after the update.
// Wave w also holds column tile w of Mb^T, Vb^T.  K_i is read by rows (the
// update) in step i and by columns (G) in step i + 1, both from one LDS copy
// (LDS-DMA, two buffers); S_{i-1}'s rows, which every wave reads whole, go
// through a second exchange like -Gb's.  Per step:
//   moment VJP of chunk i; -Gb, -S_{i-1} and the partial sums to LDS | barrier
//   Sb^T <- a Sb^T + gS^T - K_i Gb^T                                | barrier
//   request K_{i-2} into K_i's buffer, and chunk i-2's tiles
//   G_{i-1}^T = U^T - K_{i-1}^T S_{i-1}^T
// The partial sums of da, db, dm, dn of each 16-row tile go to
// part[(bh*N + i) * (D/16) + tile][4].
//
// Bound: vector memory into a CU (112 KB a chunk at D = 128, most of it K_i
// from L2), then the MFMA pipe (1.7 us a chunk). Measured (d = 128, 32
// chunks): 16 heads 682 -> 155 us, 64 heads 747 -> 381 us against the two-wave
// kernel (both products and the moment VJP of 16 rows in one wave); 206 and
// 482 us with K and S operands loaded from global memory by each wave. d = 64,
// 8 heads, 16 chunks: 116 -> 35 us.
template <int D>
struct AdamfLds {
  static constexpr int K = 0;                           // two D x D float32 buffers (SwzMat)
  static constexpr int XG = 2 * D * D;                  // -Gb rows
  static constexpr int XS = XG + RowsfLds<D>::X;        // -S rows
  static constexpr int RED = XS + RowsfLds<D>::X;       // [wave][4] partial sums
  static constexpr int BYTES = (RED + D / 16 * 4) * 4;
  static_assert(BYTES <= 160 * 1024, "adam reverse scan LDS exceeds the 160 KiB of a CU");
};

template <int D>
__global__ void __launch_bounds__(D * 4)
scan_bwd_adamf(const float* __restrict__ U, const float* __restrict__ K,
               const float* __restrict__ av, const float* __restrict__ bv,
               const float* __restrict__ mv, const float* __restrict__ nv,
               const float* __restrict__ S_all, const float* __restrict__ M_all,
               const float* __restrict__ V_all, const float* __restrict__ gS,
               float* __restrict__ dU, float* __restrict__ part, int64_t BH, int N) {
  using R = AdamfLds<D>;
  using L = SwzMat<D>;
  constexpr int NT = D / 16;
  constexpr int LD = RowsfLds<D>::LD;
  extern __shared__ __align__(16) float smem[];
  float* const xg = smem + R::XG;
  float* const xsr = smem + R::XS;
  float* const red = smem + R::RED;

  int64_t bh;
  int blk;
  map_rows_block(BH, NT, bh, blk);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = lane_id(), G = l >> 4, rl = l & 15;
  const int64_t mat = (int64_t)D * D;
  const int64_t base = bh * N * mat;
  const uint32_t to = (16 * blk + rl) * D + 16 * w + 4 * G;  // this lane's piece of a state
  const int xo = rl * LD + 16 * w + 4 * G;                   // its place in the exchanges
  const float* const Kb = K + base;

  struct Tiles {  // the lane's pieces of a chunk
    f32x4 u, mp, vp, si, gs;
    float a, b, m, n;
  };
  auto load = [&](Tiles& c, int i) {
    const int64_t o = base + i * mat, sc = bh * N + i;
    c.u = *reinterpret_cast<const f32x4*>(U + o + to);
    c.mp = *reinterpret_cast<const f32x4*>(M_all + o + to);
    c.vp = *reinterpret_cast<const f32x4*>(V_all + o + to);
    c.si = *reinterpret_cast<const f32x4*>(S_all + o + to);
    c.gs = *reinterpret_cast<const f32x4*>(gS + o + to);
    c.a = av[sc];
    c.b = bv[sc];
    c.m = mv[sc];
    c.n = nv[sc];
  };
  f32x4 Sb = zero4(), Mb = zero4(), Vb = zero4();
  // g - K^T S^T of the chunk whose -S rows are in the exchange, K_j at kl: the
  // forward's chain, so that M_i, V_i are the forward's bit for bit (with the
  // sums split otherwise the gradients' errors grew 1.1- to 1.7-fold)
  auto form_g = [&](f32x4 g, const float* kl) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const f32x4 s = *reinterpret_cast<const f32x4*>(xsr + rl * LD + 16 * t + 4 * G);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        g = mfma_f32(kl[L::off(16 * t + 4 * G + e, 16 * w + rl)], s[e], g);
      }
    }
    return g;
  };

  // Step i: `c` holds chunk i's pieces, `p` chunk i-1's, g is G_i.  Buffers:
  // K_i in i & 1, K_{i-1} requested a step ago into the other.
  f32x4 g;
  auto step = [&](Tiles& c, const Tiles& p, int i) {
    f32x4 Gb;
    float pda = 0.f, pdb = 0.f, pdm = 0.f, pdn = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      // the moments contracted as in the forward, and nothing across steps
      // (of two unrolled steps the compiler would fuse one's Mb, Vb only)
#pragma clang fp contract(off)
      const float gg = g[j];
      const float Mi = fmaf(c.m, c.mp[j], (1.f - c.m) * gg);
      const float Vi = fmaf(c.n, c.vp[j], (1.f - c.n) * gg * gg);
      const float root = sqrtf(Vi);
      const float den = root + 1e-6f;
      const float sb = Sb[j];
      pda = fmaf(sb, c.si[j], pda);
      pdb = fmaf(sb, Mi / den, pdb);
      const float ub = c.b * sb;
      const float Mtot = Mb[j] + ub / den;
      const float Vtot = Vb[j] - ub * Mi / (den * den) / (2.f * fmaxf(root, 1e-12f));
      pdm = fmaf(Mtot, c.mp[j] - gg, pdm);
      pdn = fmaf(Vtot, fmaf(-gg, gg, c.vp[j]), pdn);
      Mb[j] = c.m * Mtot;
      Vb[j] = c.n * Vtot;
      Gb[j] = fmaf(1.f - c.m, Mtot, (1.f - c.n) * 2.f * gg * Vtot);
    }
    *reinterpret_cast<f32x4*>(xg + xo) = -Gb;
    const f32x2 s0 = wave_sum2(pda, pdb), s1 = wave_sum2(pdm, pdn);
    if (l < 4) red[4 * w + l] = l == 0 ? s0[0] : l == 1 ? s0[1] : l == 2 ? s1[0] : s1[1];
    *reinterpret_cast<f32x4*>(dU + base + i * mat + to) = Gb;
    __syncthreads();  // -Gb and the partial sums published; S_i's rows read
    *reinterpret_cast<f32x4*>(xsr + xo) = -p.si;
    if (w == 0 && l < 4) {
      float t = 0.f;
#pragma unroll
      for (int q = 0; q < NT; ++q) t += red[4 * q + l];
      part[((bh * N + i) * NT + blk) * 4 + l] = t;
    }
    const float* kl = smem + R::K + (i & 1) * D * D;
    Sb = c.a * Sb + c.gs;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const f32x4 k = *reinterpret_cast<const f32x4*>(kl + L::off(16 * w + rl, 16 * t + 4 * G));
      const f32x4 gb = *reinterpret_cast<const f32x4*>(xg + rl * LD + 16 * t + 4 * G);
#pragma unroll
      for (int e = 0; e < 4; ++e) Sb = mfma_f32(k[e], gb[e], Sb);
    }
    if (i == 0) return;
    wait_vmem();      // K_{i-1} landed
    __syncthreads();  // K_{i-1} and S_{i-1}'s rows published; K_i, -Gb and the sums read
    if (i >= 2) {
      lds_dma_matrix<D, D * 4>(smem + R::K + (i & 1) * D * D, Kb + (i - 2) * mat);
      load(c, i - 2);
    }
    g = form_g(p.u, smem + R::K + ((i - 1) & 1) * D * D);
  };

  Tiles c0, c1;
  lds_dma_matrix<D, D * 4>(smem + R::K + ((N - 1) & 1) * D * D, Kb + (N - 1) * mat);
  load(c0, N - 1);
  load(c1, N > 1 ? N - 2 : 0);
  *reinterpret_cast<f32x4*>(xsr + xo) = -c0.si;
  wait_vmem();
  __syncthreads();
  if (N > 1) lds_dma_matrix<D, D * 4>(smem + R::K + ((N - 2) & 1) * D * D, Kb + (N - 2) * mat);
  g = form_g(c0.u, smem + R::K + ((N - 1) & 1) * D * D);
  int i = N - 1;
  for (; i >= 1; i -= 2) {
    step(c0, c1, i);
    step(c1, c0, i - 1);
  }
  if (i == 0) step(c0, c1, 0);
}

// ------------------------------------ reverse scan, 8 waves per 32 rows (bf16x3)
// Wave (rt, cq) holds rows 32 blk + 16 rt + lc and column quarter cq of Sb as
// D-layout tiles of Sb^T (adam: also of its moment adjoints).  Per chunk the
// workgroup's -Gb rows are exchanged as split bf16 planes in LDS, since the
// update Sb <- a Sb - Gb K^T + gS contracts over every column of Gb; K_i is
// staged as split planes (double buffered) by all threads from fp32 loads
// issued one chunk ahead, read by rows for that update and by columns (adam)
// for recomputing G = U - S_i K_i, whose S_i row pieces a lane loads itself in
// the operand's k order.  Every chunk operand (gS, and adam's U, M, V, S_i)
// is loaded one chunk ahead.
template <int D, int RULE>
__global__ void __launch_bounds__(A8_THREADS)
scan_bwd_rows8(const float* __restrict__ U, const float* __restrict__ K,
               const float* __restrict__ av, const float* __restrict__ bv,
               const float* __restrict__ mv, const float* __restrict__ nv,
               const float* __restrict__ S_all, const float* __restrict__ M_all,
               const float* __restrict__ V_all, const float* __restrict__ gS,
               float* __restrict__ dU, float* __restrict__ part, int64_t BH, int N) {
  using L = BSwz<D>;
  using R = Rows8Lds<D>;
  using P = PrecX3;
  constexpr int NKB = D / 32;
  constexpr int TPW = D / 64;
  constexpr int ROWB = D * 2;
  constexpr int PR = D / 4;
  constexpr int NQ = D * PR / A8_THREADS;
  constexpr int RSTEP = A8_THREADS / PR;
  constexpr int NTILES = D / 16;
  constexpr int RED = R::BYTES;  // adam: [rt][cq][4] partial sums after the planes
  static_assert(NQ * A8_THREADS == D * PR && RSTEP % 16 == 0, "K pieces split in swizzle-keeping row steps");
  static_assert(RULE == 0 || R::BYTES + 32 * 4 <= 160 * 1024, "adam partial sums exceed the LDS");
  extern __shared__ __align__(16) float smem[];

  int64_t bh;
  int blk;
  map_rows_block(BH, D / 32, bh, blk);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = lane_id(), G = l >> 4, lc = l & 15;
  const int rt = w >> 2, cq = w & 3;
  const int row = 32 * blk + 16 * rt + lc;
  const int64_t mat = (int64_t)D * D;
  const float* Kb = K + bh * N * mat;
  const lds_ptr L0 = lds_base(smem);

  // per-lane LDS offsets: K rows 16 ct + lc over k-block kb (both halves of
  // the pair order), K columns (adam), exchange-plane writes and reads
  uint32_t krow[NKB][2], kcol[TPW], xsw[TPW], xsr[NKB][2];
#pragma unroll
  for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      krow[kb][h] = swz_off<L>(lc, 32 * kb + 16 * h + 4 * G);
      xsr[kb][h] = swz_off<L>(16 * rt + lc, 32 * kb + 16 * h + 4 * G);
    }
#pragma unroll
  for (int u = 0; u < TPW; ++u) {
    const int ct = cq * TPW + u;
    kcol[u] = swz_off<L>(4 * G + (lc >> 2), 16 * ct + 4 * (lc & 3));
    xsw[u] = swz_off<L>(16 * rt + lc, 16 * ct + 4 * G);
  }
  const int kr = threadIdx.x / PR, kc = (threadIdx.x % PR) * 4;
  const uint32_t kdst = swz_off<L>(kr, kc);
  const int64_t ksrc = (int64_t)kr * D + kc;
  auto roff = [&](int u) { return (int64_t)row * D + 16 * (cq * TPW + u) + 4 * G; };

  f32x4 Kpre[NQ];
  auto load_k = [&](int i) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) Kpre[q] = *reinterpret_cast<const f32x4*>(Kb + i * mat + ksrc + q * RSTEP * D);
  };
  auto stage_k = [&](int buf) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      bf16x4 hi, lo;
      split4(Kpre[q], hi, lo);
      const uint32_t o = R::K0 + buf * 2 * R::PLANE + kdst + q * RSTEP * ROWB;
      lds_st<bf16x4>(L0 + o, hi);
      lds_st<bf16x4>(L0 + (o + R::PLANE), lo);
    }
  };
  // chunk operands of this lane: gS tiles; adam: U, M, V tiles and the S_i row
  // pieces of every k-block (columns 32 kb + 16 h + 4G .. +3)
  f32x4 gsn[TPW], un[TPW], mn[TPW], vn[TPW], sn[NKB][2];
  auto load_chunk = [&](int i) {
    const int64_t base = (bh * N + i) * mat;
#pragma unroll
    for (int u = 0; u < TPW; ++u) gsn[u] = *reinterpret_cast<const f32x4*>(gS + base + roff(u));
    if constexpr (RULE == 2) {
#pragma unroll
      for (int u = 0; u < TPW; ++u) {
        un[u] = *reinterpret_cast<const f32x4*>(U + base + roff(u));
        mn[u] = *reinterpret_cast<const f32x4*>(M_all + base + roff(u));
        vn[u] = *reinterpret_cast<const f32x4*>(V_all + base + roff(u));
      }
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          sn[kb][h] = *reinterpret_cast<const f32x4*>(S_all + base + (int64_t)row * D + 32 * kb + 16 * h + 4 * G);
    }
  };

  f32x4 Sb[TPW], Mb[TPW], Vb[TPW];
#pragma unroll
  for (int u = 0; u < TPW; ++u) Sb[u] = Mb[u] = Vb[u] = zero4();
  if (N > 0) {
    load_k(N - 1);
    stage_k((N - 1) & 1);
    load_chunk(N - 1);
  }
  if (N > 1) load_k(N - 2);
  __syncthreads();

  for (int i = N - 1; i >= 0; --i) {
    const int buf = i & 1;
    const int64_t si = bh * N + i;
    const float a = av[si];
    f32x4 gsc[TPW], Gb[TPW];
#pragma unroll
    for (int u = 0; u < TPW; ++u) gsc[u] = gsn[u];
    if constexpr (RULE == 0) {
#pragma unroll
      for (int u = 0; u < TPW; ++u) Gb[u] = Sb[u];
    } else {
      const float b = bv[si], m = mv[si], n = nv[si];
      P::Op Sop[NKB];
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb) Sop[kb] = P::pack(-sn[kb][0], -sn[kb][1]);
      float pda = 0.f, pdb = 0.f, pdm = 0.f, pdn = 0.f;
#pragma unroll
      for (int u = 0; u < TPW; ++u) {
        // G^T = U^T - K^T S_i^T : A = K^T (column reads), B = -S_i^T
        f32x4 g = un[u];
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb) {
          const uint32_t o = R::K0 + buf * 2 * R::PLANE + kcol[u] + kb * 32 * ROWB;
          P::Op A;
          A.hi = cat8(lds_tr16(L0 + o), lds_tr16(L0 + (o + 16 * ROWB)));
          A.lo = cat8(lds_tr16(L0 + (o + R::PLANE)), lds_tr16(L0 + (o + R::PLANE + 16 * ROWB)));
          g = P::mma(A, Sop[kb], g);
        }
        const int ct = cq * TPW + u;  // this tile's S_i pieces, selected with constant indices
        f32x4 Si = sn[0][0];
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
          for (int h = 0; h < 2; ++h)
            if (2 * kb + h == ct) Si = sn[kb][h];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float gg = g[j];
          const float Mi = m * mn[u][j] + (1.f - m) * gg;
          const float Vi = n * vn[u][j] + (1.f - n) * gg * gg;
          const float root = hw_sqrt(Vi);
          const float rden = hw_rcp(root + 1e-6f);
          const float sb = Sb[u][j];
          pda += sb * Si[j];
          pdb += sb * (Mi * rden);
          const float ub = b * sb;
          const float Mtot = Mb[u][j] + ub * rden;
          const float Vtot = Vb[u][j] - ub * Mi * rden * rden * hw_rcp(2.f * fmaxf(root, 1e-12f));
          pdm += Mtot * (mn[u][j] - gg);
          pdn += Vtot * (vn[u][j] - gg * gg);
          Mb[u][j] = m * Mtot;
          Vb[u][j] = n * Vtot;
          Gb[u][j] = (1.f - m) * Mtot + (1.f - n) * 2.f * gg * Vtot;
        }
      }
      pda = wave_sum(pda);
      pdb = wave_sum(pdb);
      pdm = wave_sum(pdm);
      pdn = wave_sum(pdn);
      if (l < 4) {
        const float v = l == 0 ? pda : l == 1 ? pdb : l == 2 ? pdm : pdn;
        lds_st<float>(L0 + (RED + (w * 4 + l) * 4), v);
      }
    }
    // dU_i = Gb ; -Gb (split) -> the exchange planes
#pragma unroll
    for (int u = 0; u < TPW; ++u) {
      *reinterpret_cast<f32x4*>(dU + si * mat + roff(u)) = Gb[u];
      bf16x4 hi, lo;
      split4(-Gb[u], hi, lo);
      lds_st<bf16x4>(L0 + (R::XS0 + xsw[u]), hi);
      lds_st<bf16x4>(L0 + (R::XS0 + xsw[u] + R::XSP), lo);
    }
    __syncthreads();  // -Gb rows (and adam's partial sums) published
    if constexpr (RULE == 2) {
      if (cq == 0 && l < 4) {
        float t = 0.f;
#pragma unroll
        for (int q = 0; q < 4; ++q) t += lds_ld<float>(L0 + (RED + ((4 * rt + q) * 4 + l) * 4));
        part[(si * NTILES + 2 * blk + rt) * 4 + l] = t;
      }
    }
    P::Op Gop[NKB];
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb) {
      Gop[kb].hi = cat8(lds_ld<bf16x4>(L0 + (R::XS0 + xsr[kb][0])), lds_ld<bf16x4>(L0 + (R::XS0 + xsr[kb][1])));
      Gop[kb].lo = cat8(lds_ld<bf16x4>(L0 + (R::XS0 + R::XSP + xsr[kb][0])),
                        lds_ld<bf16x4>(L0 + (R::XS0 + R::XSP + xsr[kb][1])));
    }
    // Sb^T <- a Sb^T - K Gb^T + gS^T : A = K rows 16 ct.., B = -Gb^T
#pragma unroll
    for (int u = 0; u < TPW; ++u) {
      const int ct = cq * TPW + u;
      f32x4 acc = a * Sb[u] + gsc[u];
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb) {
        const uint32_t o0 = R::K0 + buf * 2 * R::PLANE + 16 * ct * ROWB;
        P::Op A;
        A.hi = cat8(lds_ld<bf16x4>(L0 + (o0 + krow[kb][0])), lds_ld<bf16x4>(L0 + (o0 + krow[kb][1])));
        A.lo = cat8(lds_ld<bf16x4>(L0 + (o0 + R::PLANE + krow[kb][0])),
                    lds_ld<bf16x4>(L0 + (o0 + R::PLANE + krow[kb][1])));
        acc = P::mma(A, Gop[kb], acc);
      }
      Sb[u] = acc;
    }
    // K_{i-1} into the other buffer (last read in chunk i+1); loads of K_{i-2} and chunk i-1
    if (i > 0) {
      stage_k(buf ^ 1);
      load_chunk(i - 1);
    }
    if (i > 1) load_k(i - 2);
    __syncthreads();  // K_{i-1} staged; the exchange planes free
  }
}

// Chunk-parallel part of the backward: dK_i = -S_i^T Gb_i (contraction over
// the rows of S) and the scalar gradients of chunk i, exact float32.  One
// workgroup of D/16 waves per (bh, i).  Wave w forms the tiles of dK rows
// 16 w .. 16 w + 15, transposed ((Gb^T S)[c][c']), so that a lane stores four
// consecutive columns of dK; its own S columns are loaded straight into the
// operand registers once, and Gb_i, which every wave reads whole, is staged
// in LDS (rows padded by four floats: the four lane groups' rows, four apart,
// fall on different banks).  Bound: the MFMA pipe (6.8 us a chunk at D = 128,
// two workgroups a CU). Measured (d = 128): 4096 chunks 363 -> 216 us, 2048
// chunks 165 -> 97 us against 16-byte-swizzled copies of both matrices read by
// column for every tile.
template <int D, int RULE>
__global__ void __launch_bounds__(D * 4)
scan_bwd_dkf(const float* __restrict__ S_all, const float* __restrict__ dU,
             const float* __restrict__ part, float* __restrict__ dK,
             float* __restrict__ da, float* __restrict__ db, float* __restrict__ dm,
             float* __restrict__ dn, int64_t BH, int N) {
  constexpr int NT = D / 16;
  constexpr int LD = D + 4;
  extern __shared__ __align__(16) float smem[];  // Gb_i, D rows of LD floats
  __shared__ float red[NT];
  const int64_t si = blockIdx.x;  // = bh * N + i
  const int64_t mat = (int64_t)D * D;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = lane_id(), G = l >> 4, rl = l & 15;
  const float* const Gi = dU + si * mat;
  const float* const Si = S_all + si * mat;
  const uint32_t so = 4 * G * D + 16 * w + rl;
  float s[NT][4];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) s[t][e] = (Si + (16 * t + e) * D)[so];
  {
    constexpr int PR = D / 4, NQ = D * PR / (D * 4), RSTEP = D * 4 / PR;  // 16-byte pieces
    const int r = threadIdx.x / PR, c = (threadIdx.x % PR) * 4;
    f32x4 x[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) x[q] = *reinterpret_cast<const f32x4*>(Gi + (r + q * RSTEP) * D + c);
#pragma unroll
    for (int q = 0; q < NQ; ++q) *reinterpret_cast<f32x4*>(smem + (r + q * RSTEP) * LD + c) = x[q];
  }
  __syncthreads();
  float* const out = dK + si * mat + (16 * w + rl) * D + 4 * G;
  float dot = 0.f;
#pragma unroll 2
  for (int tc = 0; tc < NT; ++tc) {
    const float* const gp = smem + 4 * G * LD + 16 * tc + rl;
    f32x4 a0 = zero4(), a1 = zero4();
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float gv = gp[(16 * t + e) * LD];
        if (t & 1)
          a1 = mfma_f32(gv, s[t][e], a1);
        else
          a0 = mfma_f32(gv, s[t][e], a0);
        if constexpr (RULE == 0) dot += tc == w ? gv * s[t][e] : 0.f;  // da_i = <Gb_i, S_i>
      }
    *reinterpret_cast<f32x4*>(out + 16 * tc) = -(a0 + a1);
  }
  if constexpr (RULE == 0) {
    dot = wave_sum(dot);
    if (l == 0) red[w] = dot;
    __syncthreads();
    if (threadIdx.x == 0) {
      float t = 0.f;
#pragma unroll
      for (int q = 0; q < NT; ++q) t += red[q];
      da[si] = t;
      db[si] = 0.f;
      dm[si] = 0.f;
      dn[si] = 0.f;
    }
  } else if constexpr (RULE == 2) {
    if (threadIdx.x < 4) {
      float t = 0.f;
#pragma unroll
      for (int q = 0; q < NT; ++q) t += part[(si * NT + q) * 4 + threadIdx.x];
      float* dst = threadIdx.x == 0 ? da : threadIdx.x == 1 ? db : threadIdx.x == 2 ? dm : dn;
      dst[si] = t;
    }
  }
  // RULE == 1: the muon backward kernel writes the scalar gradients itself
}

// The chunk-parallel part with 8 waves: S_i and Gb_i staged as split bf16
// planes (loaded as 16-byte fp32 pieces by all threads, which also form
// delta's da = <Gb_i, S_i> in fp32 on the way), every operand a transposing
// LDS read, and each output tile formed transposed, (Gb^T S)[c][c'] =
// -dK[c'][c], so that a lane writes four consecutive columns of dK.
template <int D>
struct Dk8Lds {
  static constexpr int PLANE = D * D * 2;
  static constexpr int S0 = 0;          // S_i hi, lo
  static constexpr int G0 = 2 * PLANE;  // Gb_i hi, lo
  static constexpr int RED = 4 * PLANE; // per-wave partial sums
  static constexpr int BYTES = RED + 8 * 4;
  static_assert(BYTES <= 160 * 1024, "dK LDS exceeds the 160 KiB of a CU");
};

template <int D, int RULE>
__global__ void __launch_bounds__(A8_THREADS)
scan_bwd_dk8(const float* __restrict__ S_all, const float* __restrict__ dU,
             const float* __restrict__ part, float* __restrict__ dK,
             float* __restrict__ da, float* __restrict__ db, float* __restrict__ dm,
             float* __restrict__ dn, int64_t BH, int N) {
  using L = BSwz<D>;
  using R = Dk8Lds<D>;
  using P = PrecX3;
  constexpr int NT = D / 16;
  constexpr int NKB = D / 32;
  constexpr int ROWB = D * 2;
  constexpr int PR = D / 4;
  constexpr int NQ = D * PR / A8_THREADS;
  constexpr int RSTEP = A8_THREADS / PR;
  constexpr int NW = A8_THREADS / 64;
  static_assert(NQ * A8_THREADS == D * PR && RSTEP % 16 == 0, "pieces split in swizzle-keeping row steps");
  static_assert((NT * NT) % NW == 0, "output tiles split evenly over the waves");
  extern __shared__ __align__(16) float smem[];
  const lds_ptr L0 = lds_base(smem);
  const int64_t si = blockIdx.x;  // = bh * N + i
  const int64_t mat = (int64_t)D * D;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = lane_id(), G = l >> 4, lc = l & 15;

  // ---- staging (and delta's da from the fp32 values)
  {
    const int kr = threadIdx.x / PR, kc = (threadIdx.x % PR) * 4;
    const float* sg = S_all + si * mat + (int64_t)kr * D + kc;
    const float* gg = dU + si * mat + (int64_t)kr * D + kc;
    const uint32_t dst = swz_off<L>(kr, kc);
    f32x4 xs[NQ], xg[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      xs[q] = *reinterpret_cast<const f32x4*>(sg + q * RSTEP * D);
      xg[q] = *reinterpret_cast<const f32x4*>(gg + q * RSTEP * D);
    }
    float dot = 0.f;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const uint32_t o = dst + q * RSTEP * ROWB;
      bf16x4 hi, lo;
      split4(xs[q], hi, lo);
      lds_st<bf16x4>(L0 + (R::S0 + o), hi);
      lds_st<bf16x4>(L0 + (R::S0 + R::PLANE + o), lo);
      split4(xg[q], hi, lo);
      lds_st<bf16x4>(L0 + (R::G0 + o), hi);
      lds_st<bf16x4>(L0 + (R::G0 + R::PLANE + o), lo);
      if constexpr (RULE == 0) dot += xs[q][0] * xg[q][0] + xs[q][1] * xg[q][1] + xs[q][2] * xg[q][2] + xs[q][3] * xg[q][3];
    }
    if constexpr (RULE == 0) {
      dot = wave_sum(dot);
      if (l == 0) reinterpret_cast<float*>(smem + R::RED / 4)[w] = dot;
    }
  }
  __syncthreads();

  // ---- dK tiles: (Gb^T S) tile (tc, tr) = -dK^T; A = Gb columns, B = S columns
  uint32_t pcol[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) pcol[t] = swz_off<L>(4 * G + (lc >> 2), 16 * t + 4 * (lc & 3));
  auto colop = [&](uint32_t base, int kb, int t) {
    const uint32_t o = base + pcol[t] + kb * 32 * ROWB;
    P::Op x;
    x.hi = cat8(lds_tr16(L0 + o), lds_tr16(L0 + (o + 16 * ROWB)));
    x.lo = cat8(lds_tr16(L0 + (o + R::PLANE)), lds_tr16(L0 + (o + R::PLANE + 16 * ROWB)));
    return x;
  };
  float* const dKi = dK + si * mat;
#pragma unroll
  for (int q = 0; q < NT * NT / NW; ++q) {
    const int tile = w + NW * q, tr = tile / NT, tc = tile % NT;
    f32x4 acc = zero4();
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb) acc = P::mma(colop(R::G0, kb, tc), colop(R::S0, kb, tr), acc);
    // lane (c', G) holds (Gb^T S)[16 tc + 4G + j][16 tr + c'] = -dK[16 tr + c'][16 tc + 4G + j]
    *reinterpret_cast<f32x4*>(dKi + (int64_t)(16 * tr + lc) * D + 16 * tc + 4 * G) = -acc;
  }

  // ---- scalar gradients of the chunk
  if constexpr (RULE == 0) {
    if (threadIdx.x == 0) {
      const float* red = reinterpret_cast<const float*>(smem + R::RED / 4);
      float t = 0.f;
#pragma unroll
      for (int q = 0; q < NW; ++q) t += red[q];
      da[si] = t;
      db[si] = 0.f;
      dm[si] = 0.f;
      dn[si] = 0.f;
    }
  } else if constexpr (RULE == 2) {
    if (threadIdx.x < 4) {
      float t = 0.f;
      for (int q = 0; q < D / 16; ++q) t += part[(si * (D / 16) + q) * 4 + threadIdx.x];
      float* dst = threadIdx.x == 0 ? da : threadIdx.x == 1 ? db : threadIdx.x == 2 ? dm : dn;
      dst[si] = t;
    }
  }
  // RULE == 1: the muon backward kernel writes the scalar gradients itself
}

// Adam's scalar gradients alone, from the row tiles' partial sums: thread
// 4 c + q sums value q of chunk c in the order the dK kernels use.
__global__ void __launch_bounds__(256)
scan_bwd_scalars(const float* __restrict__ part, float* __restrict__ da, float* __restrict__ db,
                 float* __restrict__ dm, float* __restrict__ dn, int64_t chunks, int tiles) {
  const int64_t x = (int64_t)blockIdx.x * 256 + threadIdx.x, c = x >> 2;
  const int q = (int)(x & 3);
  if (c >= chunks) return;
  float t = 0.f;
  for (int k = 0; k < tiles; ++k) t += part[(c * tiles + k) * 4 + q];
  float* const dst = q == 0 ? da : q == 1 ? db : q == 2 ? dm : dn;
  dst[c] = t;
}

// ---------------------------------------------------------------- launchers
template <int D, int RULE>
static hipError_t launch_fwd_rowsf(const ScanArgs& s) {
  hipLaunchKernelGGL((scan_fwd_rowsf<D, RULE>), dim3((unsigned)(s.BH * (D / 16))), dim3(D * 4), 0, s.stream, s.U, s.K,
                     s.a, s.b, s.m, s.n, s.S_all, s.M_all, s.V_all, s.BH, (int)s.N);
  return hipGetLastError();
}

template <int D>
static hipError_t launch_bwd_rowsf(const ScanArgs& s) {
  hipLaunchKernelGGL((scan_bwd_rowsf<D>), dim3((unsigned)(s.BH * (D / 16))), dim3(D * 4), 0, s.stream, s.K, s.a, s.gS,
                     s.dU, s.BH, (int)s.N);
  return hipGetLastError();
}

template <int D>
static hipError_t launch_bwd_adamf(const ScanArgs& s, float* part) {
  const int lds = AdamfLds<D>::BYTES;
  auto kern = scan_bwd_adamf<D>;
  hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3((unsigned)(s.BH * (D / 16))), dim3(D * 4), lds, s.stream, s.U, s.K, s.a, s.b, s.m, s.n,
                     s.S_all, s.M_all, s.V_all, s.gS, s.dU, part, s.BH, (int)s.N);
  return hipGetLastError();
}

template <int D, int RULE, int PREC>
static hipError_t launch_bwd_dk(const ScanArgs& s, const float* part) {
  if constexpr (PREC == 0 && D >= 64) {  // bf16x3 planes
    const int lds = Dk8Lds<D>::BYTES;
    auto k8 = scan_bwd_dk8<D, RULE>;
    hipError_t e = hipFuncSetAttribute((const void*)k8, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k8, dim3((unsigned)(s.BH * s.N)), dim3(A8_THREADS), lds, s.stream, s.S_all, s.dU, part,
                       s.dK, s.da, s.db, s.dm, s.dn, s.BH, (int)s.N);
    return hipGetLastError();
  }
  const int lds = D * (D + 4) * (int)sizeof(float);
  auto kf = scan_bwd_dkf<D, RULE>;
  hipError_t e = hipFuncSetAttribute((const void*)kf, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kf, dim3((unsigned)(s.BH * s.N)), dim3(D * 4), lds, s.stream, s.S_all, s.dU, part, s.dK, s.da,
                     s.db, s.dm, s.dn, s.BH, (int)s.N);
  return hipGetLastError();
}

template <int D, int PREC>
static hipError_t dk_rule(const ScanArgs& s, const float* part) {
  switch (s.rule) {
    case 0: return launch_bwd_dk<D, 0, PREC>(s, part);
    case 1: return launch_bwd_dk<D, 1, PREC>(s, part);
    default: return launch_bwd_dk<D, 2, PREC>(s, part);
  }
}

template <int D>
static hipError_t dk_prec(const ScanArgs& s, const float* part) {
  return s.precision == 0 ? dk_rule<D, 0>(s, part) : dk_rule<D, 1>(s, part);
}

hipError_t scan_bwd_dk_launch(const ScanArgs& s, const float* part) {
  if (!s.dK && s.rule == 2) {
    const int64_t chunks = s.BH * s.N;
    hipLaunchKernelGGL(scan_bwd_scalars, dim3((unsigned)((4 * chunks + 255) / 256)), dim3(256), 0, s.stream, part, s.da,
                       s.db, s.dm, s.dn, chunks, s.dh / 16);
    return hipGetLastError();
  }
  switch (s.dh) {
    case 32: return dk_prec<32>(s, part);
    case 64: return dk_prec<64>(s, part);
    case 128: return dk_prec<128>(s, part);
  }
  return hipErrorInvalidValue;
}

template <int D, int RULE>
static hipError_t launch_fwd_rows8(const ScanArgs& s) {
  const int lds = Rows8Lds<D>::BYTES;
  auto kern = scan_fwd_rows8<D, RULE>;
  hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3((unsigned)(s.BH * (D / 32))), dim3(A8_THREADS), lds, s.stream, s.U, s.K, s.a,
                     s.b, s.m, s.n, s.S_all, s.M_all, s.V_all, s.BH, (int)s.N);
  return hipGetLastError();
}

template <int D, int PREC>
static hipError_t fwd_rows_rule(const ScanArgs& s) {
  // bf16x3: the 8-wave kernel (at D = 32 a row block is a few products either
  // way: the float32 one)
  if constexpr (PREC == 0 && D >= 64)
    return s.rule == 0 ? launch_fwd_rows8<D, 0>(s) : launch_fwd_rows8<D, 2>(s);
  else
    return s.rule == 0 ? launch_fwd_rowsf<D, 0>(s) : launch_fwd_rowsf<D, 2>(s);
}
template <int D, int RULE>
static hipError_t launch_bwd_rows8(const ScanArgs& s, float* part) {
  const int lds = Rows8Lds<D>::BYTES + (RULE == 2 ? 32 * 4 : 0);
  auto kern = scan_bwd_rows8<D, RULE>;
  hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3((unsigned)(s.BH * (D / 32))), dim3(A8_THREADS), lds, s.stream, s.U, s.K, s.a,
                     s.b, s.m, s.n, s.S_all, s.M_all, s.V_all, s.gS, s.dU, part, s.BH, (int)s.N);
  return hipGetLastError();
}

template <int D, int PREC>
static hipError_t bwd_rows_rule(const ScanArgs& s, float* part) {
  // bf16x3: the 8-wave kernel (adam's at D = 128 would spill: the float32 one)
  if constexpr (PREC == 0 && D >= 64) {
    if (s.rule == 0) return launch_bwd_rows8<D, 0>(s, part);
    if constexpr (D == 64) return launch_bwd_rows8<D, 2>(s, part);
  }
  return s.rule == 0 ? launch_bwd_rowsf<D>(s) : launch_bwd_adamf<D>(s, part);
}

template <int D>
static hipError_t fwd_rows_prec(const ScanArgs& s) {
  return s.precision == 0 ? fwd_rows_rule<D, 0>(s) : fwd_rows_rule<D, 1>(s);
}
template <int D>
static hipError_t bwd_rows_prec(const ScanArgs& s, float* part) {
  return s.precision == 0 ? bwd_rows_rule<D, 0>(s, part) : bwd_rows_rule<D, 1>(s, part);
}

hipError_t scan_fwd_rows_launch(const ScanArgs& s) {
  switch (s.dh) {
    case 32: return fwd_rows_prec<32>(s);
    case 64: return fwd_rows_prec<64>(s);
    case 128: return fwd_rows_prec<128>(s);
  }
  return hipErrorInvalidValue;
}

hipError_t scan_bwd_rows_launch(const ScanArgs& s, float* part) {
  switch (s.dh) {
    case 32: return bwd_rows_prec<32>(s, part);
    case 64: return bwd_rows_prec<64>(s, part);
    case 128: return bwd_rows_prec<128>(s, part);
  }
  return hipErrorInvalidValue;
}

}  // namespace gmdn
