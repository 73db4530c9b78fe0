// Level B forward of the delta rule with 16-row workgroups, for launches that
// leave CUs idle.
//
// The mathematics of chunk_fwd_rows (reference train_ablation.py:142-187 with
// fast_scan.py:72-85, E-form) with the work split of chunk_fwd_adam16: per
// (b, h) and chunk i with state S_i,
//   E = V - K S_i^T,   o = Q S_i^T + tril(Q K^T) diag(beta) E,
//   S_{i+1} = a S_i + E^T diag(beta) K.
// chunk_fwd_rows keeps a 16-row block's whole recurrence in one wave (64
// products a chunk in its chain at d = 128, no exchange): the better split when
// every CU has a workgroup, since the exchange adds LDS traffic and barriers.
// With few heads most CUs have none, and the chain's latency is all there is:
// here the row block's chain runs on four waves, twice as many CUs.
//
// A workgroup of ten waves owns 16 rows of S for the whole sequence
// (B H D / 16 workgroups, the D/16 of one (b, h) on one XCD).  Two barriers a
// chunk; interval i runs from barrier i to barrier i + 1.
//  * State waves 0-3: wave q owns token tile q of E and D/64 column tiles of
//    the state (D = 128: k-block q; D = 64: half of k-block q / 2).  E's tile
//    from the published pieces of Sf = -S, -beta E published | mid-chunk barrier | Sf <- a Sf +
//    K^T (-beta E) on its columns, its pieces published | barrier.
//  * Output waves 4-7 (token tiles 0, 1, 3, 2): A^T = K Q^T, packed | mid-chunk
//    barrier | -o^T = Sf Q^T + (-beta E)^T A^T, stored.  Q rows come straight
//    from global memory two chunks ahead (each is read by one wave only), asked
//    for before the last products so that the gather's issue is hidden.
//  * Copy waves 8, 9: LDS-DMA copies of K, V, beta of chunk i + 3 (4-stage
//    ring) at the start of interval i, the chunk decays lane-parallel, 64
//    chunks at a time, and, in the training forward, the even chunks'
//    checkpoint from the staging.
//
// What bounds it: LDS reads (~150 KB a chunk at d = 128, ~1200 cycles at 128
// B/clk) behind two latency chains; 1950 cycles a chunk in all.  So operands
// that do not depend on the state are read in the half that reads less, and each
// half's reads are all issued before its first product.  K rows from global memory for the state waves cost more
// than the LDS they save (1.3x the time: 64-byte row pieces, 16 lines a load).
//
// Every sum (the decay's too) runs in chunk_fwd_rows' order, so that a head's
// bits do not depend on how many heads the call has.  Two and four shorter
// chains in place of the 8 and 14 dependent products gained nothing: 103.4
// against 103.6 us at B 1, H 8, T 8128, d 128.
//
// Measured against chunk_fwd_rows (bf16, one launch, infer / with checkpoint):
// B 1, H 8, T 8128, d 128: 158 -> 104 us / 166 -> 108 us; B 2, H 16, T 4096,
// d 128: 89 -> 64 / 92 -> 70; B 1, H 8, T 4096, d 64: 52 -> 39 / 58 -> 39;
// B 4, H 16, T 4096, d 64: 60 -> 46 / 63 -> 49.
#include "../../include/gmdn_scan.h"
#include "chunk_b.h"

#include <type_traits>

namespace gmdn {

namespace {

// An LDS base the compiler cannot see into (keeps ds_read immediates small).
GMDN_DEV lds_cptr opaque16(lds_cptr p) {
  uint32_t v = (uint32_t)(uintptr_t)p;
  asm volatile("" : "+v"(v));
  return (lds_cptr)(uintptr_t)v;
}

constexpr int FE_THREADS = 640;
constexpr int FE_RING = 4;  // LDS ring depth: chunk i + 3 is copied in interval i

template <int D>
struct FwdDelta16Lds {
  static constexpr int NKB = D / 32;
  static constexpr int TILE = CB_C * D * 2;  // one K chunk (bytes)
  static constexpr int VT = CB_C * 16 * 2;   // the workgroup's 16 columns of V
  static constexpr int GT = CB_C * 4;        // beta of a chunk
  static constexpr int K0 = 0;
  static constexpr int V0 = K0 + FE_RING * TILE;
  static constexpr int G0 = V0 + FE_RING * VT;
  // per chunk parity: Sf pieces [k-block][hi, lo][lane][tile u], 8 bytes
  static constexpr int SPB = NKB * 2 * 1024;
  // per chunk parity: -beta E pieces [token block][hi, lo][lane][tile u]
  static constexpr int EPB = 2 * 2 * 1024;
  static constexpr int SP0 = G0 + FE_RING * GT;
  static constexpr int EP0 = SP0 + 2 * SPB;
  static constexpr int SC0 = EP0 + 2 * EPB;  // a of 64 chunks, double-buffered by block parity
  // training forward: S_i of an even chunk (split pieces), unit u4 of row R
  // at slot u4 ^ R (conflict-free both ways); stored before the next even
  // chunk's is staged
  static constexpr int CK0 = SC0 + 2 * 64 * 4;
  static constexpr int BYTES = CK0 + 16 * (D / 4) * 16;
  static_assert(BYTES <= 160 * 1024, "delta forward LDS exceeds the 160 KiB of a CU");
};

}  // namespace

template <int D>
__global__ void __launch_bounds__(FE_THREADS) chunk_fwd_delta16(ChunkArgs p) {
  using LQ = RowSwz<D>;
  using LV = BSwz<16>;
  using L = FwdDelta16Lds<D>;
  constexpr int NKB = D / 32;
  constexpr int CT = D / 64;   // column tiles of a state wave
  constexpr int ROWB = D * 2;  // bytes per K row
  using DK = DmaPlan<LQ, CB_C, 128>;
  using DV = DmaPlan<LV, CB_C, 128>;
  extern __shared__ __align__(16) char smem[];

  int64_t bh;
  int blk;
  map_block(p.B * p.H, D / 16, bh, blk);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = lane_id(), G = l >> 4, lc = l & 15;
  const int64_t bb = bh / p.H, hh = bh % p.H;
  const lds_ptr L0 = lds_base(smem);
  const int N = p.N;

  if (w >= 8) {
    // ========================================================= copy waves
    const int cw = w - 8;
    const uint32_t lds0 = lds_addr(smem);
    const bf16* kg = p.k + bb * p.sk[0] + hh * p.sk[1];
    const bf16* vg = p.v + bb * p.sv[0] + hh * p.sv[1] + 16 * blk;
    DK dk;
    DV dv;
    dk.init(cw, p.sk[2]);
    dv.init(cw, p.sv[2]);
    // beta of the chunk, 16 bytes per lane of wave 8's lanes 0-15
    const float* bsrc = p.beta + bh * p.T + 4 * lc;
    auto issue_loads = [&](int i, int stg) {
      const int64_t t0 = (int64_t)i * CB_C;
      dk.issue(kg + t0 * p.sk[2], lds0 + L::K0 + stg * L::TILE, cw);
      dv.issue(vg + t0 * p.sv[2], lds0 + L::V0 + stg * L::VT, cw);
      if (cw == 0 && l < 16) lds_dma16(bsrc + t0, smem + L::G0 + stg * L::GT);
    };
    // wait until at most `ahead` (0 or 1) chunk copies issued after the awaited
    // one are still in flight (wave 8 also copies beta)
    constexpr int ND = DK::NOPS + DV::NOPS;
    auto wait_chunks = [&](int ahead) {
      if (cw == 0) {
        if (ahead == 1)
          wait_vmem_le<ND + 1>();
        else
          wait_vmem();
      } else {
        if (ahead == 1)
          wait_vmem_le<ND>();
        else
          wait_vmem();
      }
    };
    // a = exp(sum of max(g, log 1e-6)) of chunks 64 J .. 64 J + 63, lane c:
    // chunk 64 J + c (wave 8)
    auto scalar_block = [&](int J) {
      const int c = 64 * J + l;
      if (cw != 0 || c >= N) return;
      const float* x = p.g + bh * p.T + (int64_t)c * CB_C;
      // wave_sum's order: quads, quads 0 + 3 and 2 + 1 of each 16, then the rows of 16
      float row[CB_C / 16];
#pragma unroll
      for (int r = 0; r < CB_C / 16; ++r) {
        float q[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const f32x4 u = *reinterpret_cast<const f32x4*>(x + 16 * r + 4 * k);
          q[k] = (fmaxf(u[0], LOG_FLOOR) + fmaxf(u[1], LOG_FLOOR)) + (fmaxf(u[2], LOG_FLOOR) + fmaxf(u[3], LOG_FLOOR));
        }
        row[r] = (q[0] + q[3]) + (q[2] + q[1]);
      }
      lds_st<float>(L0 + (L::SC0 + (J & 1) * 256 + 4 * l), expf((row[0] + row[1]) + (row[2] + row[3])));
    };
    // the even chunks' checkpoint rows from the staging: lane L = 64 cw + l
    // stores units f = 128 k + L (row f / (D/4), columns 4 u4 .. 4 u4 + 3)
    constexpr int UPR = D / 4, NU = 16 * UPR / 128;
    uint32_t cko[NU];
    int64_t ckg[NU];
#pragma unroll
    for (int k = 0; k < NU; ++k) {
      const int f = 128 * k + 64 * cw + l, R = f / UPR, u4 = f % UPR;
      cko[k] = (uint32_t)(R * UPR * 16 + 16 * (u4 ^ R));
      ckg[k] = (int64_t)R * D + 4 * u4;
    }
    auto store_state = [&](int i) {
      if (!p.states || (i & 1)) return;
      float* sp = p.states + ((bh * ((N + 1) / 2) + i / 2) * D + 16 * blk) * (int64_t)D;
#pragma unroll
      for (int k = 0; k < NU; ++k)
        *reinterpret_cast<bf16x8*>(sp + ckg[k]) = lds_ld<bf16x8>(L0 + (L::CK0 + cko[k]));
    };
    const int pre = N < FE_RING - 1 ? N : FE_RING - 1;
    for (int i = 0; i < pre; ++i) issue_loads(i, i);
    scalar_block(0);
    wait_chunks(pre > 2 ? 1 : 0);
    __syncthreads();  // barrier 0
    for (int i = 0; i < N; ++i) {
      // the stage of chunk i - 1 was last read before the mid-chunk barrier of
      // interval i - 1 (its K^T operands and A): chunk i + 3's copies go out at
      // once; chunk i + 2 (copied since interval i - 1) lands before barrier
      // i + 1
      store_state(i);  // before the next copy, so that no copy wait waits on it
      if (i + 3 < N) issue_loads(i + 3, (i + 3) % FE_RING);
      __syncthreads();  // the mid-chunk barrier of chunk i
      if ((i & 63) == 63 && i + 1 < N) scalar_block((i + 1) >> 6);
      if (i + 2 < N) wait_chunks(i + 3 < N ? 1 : 0);
      __syncthreads();  // barrier i + 1
    }
    return;
  }

  // natural-order row operand of a K tile: lane (m, G) takes row 16 tt + m,
  // columns 32 kb + 8G .. +7 (one 16-byte read)
  lds_cptr rowK[NKB];
#pragma unroll
  for (int kb = 0; kb < NKB; ++kb) rowK[kb] = opaque16(L0 + (L::K0 + swz_off<LQ>(lc, 32 * kb + 8 * G)));
  // the k-block operands of Sf (lane l's 16 bytes) and of -beta E
  const lds_cptr spr = L0 + (L::SP0 + 16 * l);
  const lds_cptr epr = L0 + (L::EP0 + 16 * l);

  if (w < 4) {
    // ========================================================= state waves
    const int q = w;
    const int kb0 = CT == 2 ? q : q >> 1, u0 = CT == 2 ? 0 : q & 1;  // the wave's k-block and first tile of it
    // K^T operand of column tile u of k-block kb0: lane (m, G) takes K[s][c]
    // for the pair-order tokens s of block kt and column
    // c = 32 kb0 + 4u + 8 (m / 4) + m % 4 (transposing reads)
    lds_cptr colp[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c)
      colp[c] = opaque16(L0 + (L::K0 + swz_off<LQ>(4 * G + (lc >> 2), 32 * kb0 + 4 * (u0 + c) + 8 * (lc & 3))));
    // V: tokens 16 q + 4G + j of the workgroup's column lc; beta of the same tokens
    const lds_cptr vp = L0 + (L::V0 + q * 16 * 32 + swz_off<LV>(4 * G + (lc >> 2), 4 * (lc & 3)));
    const lds_cptr bp = L0 + (L::G0 + 4 * (16 * q + 4 * G));
    // this wave's slots: Sf pieces of its tiles, -beta E of token tile q
    const lds_ptr spw = L0 + (L::SP0 + kb0 * 2048 + 16 * l + 8 * u0);
    const lds_ptr epw = L0 + (L::EP0 + (q >> 1) * 2048 + 16 * l + 8 * (q & 1));
    // staging: row lc, units u4 = 8 kb0 + 2G + u0 + c
    lds_ptr ckw[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c)
      ckw[c] = L0 + (L::CK0 + lc * (D / 4) * 16 + 16 * ((8 * kb0 + 2 * G + u0 + c) ^ lc));

    f32x4 Sf[CT];  // -S, lane (r, G): columns 32 kb0 + 8G + 4 (u0 + c) + j of row r
#pragma unroll
    for (int c = 0; c < CT; ++c) Sf[c] = zero4();
    auto publish_s = [&](int i) {
      const uint32_t par = (uint32_t)(i & 1) * L::SPB;
      bf16x4 hi[CT], lo[CT];
#pragma unroll
      for (int c = 0; c < CT; ++c) split4(Sf[c], hi[c], lo[c]);
      if constexpr (CT == 2) {
        lds_st<bf16x8>(spw + par, cat8(hi[0], hi[1]));
        lds_st<bf16x8>(spw + (par + 1024), cat8(lo[0], lo[1]));
      } else {
        lds_st<bf16x4>(spw + par, hi[0]);
        lds_st<bf16x4>(spw + (par + 1024), lo[0]);
      }
      if (p.states && (i & 1) == 0 && i < N) {
#pragma unroll
        for (int c = 0; c < CT; ++c) lds_st<bf16x8>(ckw[c], neg8(cat8(hi[c], lo[c])));
      }
    };
    // E's operands of a chunk that do not depend on the state
    lds_cptr rowq[NKB];
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb)
      rowq[kb] = opaque16(L0 + (L::K0 + q * 16 * ROWB + swz_off<LQ>(lc, 32 * kb + 8 * G)));
    struct Ops {
      bf16x8 Kr[NKB];
      bf16x4 vb;
      f32x4 bt;
    };
    auto load_ops = [&](auto stg_tag) {
      constexpr int STG = decltype(stg_tag)::value;
      Ops o;
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb) o.Kr[kb] = lds_ld<bf16x8>(rowq[kb] + STG * L::TILE);
      o.vb = lds_tr16(vp + STG * L::VT);
      o.bt = lds_ld<f32x4>(bp + STG * L::GT);
      return o;
    };
    publish_s(0);
    __builtin_amdgcn_s_setprio(3);
    __syncthreads();  // barrier 0: chunks 0 and 1 landed, S_0 published
    Ops cur = load_ops(std::integral_constant<int, 0>{});

    auto state_chunk = [&](auto stg_tag, int i) {
      constexpr int STG = decltype(stg_tag)::value;
      // E = V + K Sf^T, token tile q, from every wave's Sf_i pieces
      const uint32_t so = (uint32_t)(i & 1) * L::SPB;
      bf16x8 Sr[NKB][2];
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int pc = 0; pc < 2; ++pc) Sr[kb][pc] = lds_ld<bf16x8>(spr + (so + kb * 2048 + pc * 1024));
      const float a = lds_ld<float>(L0 + (L::SC0 + ((i >> 6) & 1) * 256 + (i & 63) * 4));
      // the update's K^T operands and chunk i + 1's operands of E (landed since
      // barrier i), read under E's products
      bf16x8 Kc[CT][2];
#pragma unroll
      for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
          Kc[c][kt] = cat8(lds_tr16(colp[c] + (STG * L::TILE + 32 * kt * ROWB)),
                           lds_tr16(colp[c] + (STG * L::TILE + (32 * kt + 16) * ROWB)));
      Ops nxt;
      if (i + 1 < N) nxt = load_ops(std::integral_constant<int, (STG + 1) % FE_RING>{});
      __builtin_amdgcn_sched_barrier(0);
      f32x4 E = f32x4{(float)cur.vb[0], (float)cur.vb[1], (float)cur.vb[2], (float)cur.vb[3]};
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int pc = 0; pc < 2; ++pc) E = mfma(cur.Kr[kb], Sr[kb][pc], E);
#pragma unroll
      for (int c = 0; c < CT; ++c) Sf[c] = a * Sf[c];
      const uint32_t eo = (uint32_t)(i & 1) * L::EPB;
      {
        bf16x4 eh, el;
        split4(-(cur.bt * E), eh, el);
        lds_st<bf16x4>(epw + eo, eh);
        lds_st<bf16x4>(epw + eo + 1024, el);
      }
      __syncthreads();  // mid-chunk barrier: every token tile's -beta E published
      bf16x8 We[2][2];
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int pc = 0; pc < 2; ++pc) We[kt][pc] = lds_ld<bf16x8>(epr + eo + kt * 2048 + pc * 1024);
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int pc = 0; pc < 2; ++pc)
#pragma unroll
          for (int c = 0; c < CT; ++c) Sf[c] = mfma(Kc[c][kt], We[kt][pc], Sf[c]);
      publish_s(i + 1);
      if (i + 1 < N) cur = nxt;
      __syncthreads();  // barrier i + 1
    };
    int i = 0;
    for (; i + FE_RING <= N; i += FE_RING) {
      state_chunk(std::integral_constant<int, 0>{}, i);
      state_chunk(std::integral_constant<int, 1>{}, i + 1);
      state_chunk(std::integral_constant<int, 2>{}, i + 2);
      state_chunk(std::integral_constant<int, 3>{}, i + 3);
    }
    if (i < N) {
      state_chunk(std::integral_constant<int, 0>{}, i);
      if (i + 1 < N) {
        state_chunk(std::integral_constant<int, 1>{}, i + 1);
        if (i + 2 < N) state_chunk(std::integral_constant<int, 2>{}, i + 2);
      }
    }
    return;
  }

  // ========================================================== output waves
  // waves 4, 5, 6, 7 take token tiles 0, 1, 3, 2
  const int ow = w - 4;
  bf16* og = p.o + bb * p.so[0] + hh * p.so[1] + 16 * blk + 4 * G;

  auto run = [&](auto tt_tag) {
    constexpr int TT = decltype(tt_tag)::value;
    constexpr int NKT = TT >= 2 ? 2 : 1;  // token blocks of A with s <= t
    // Q rows of the token tile: lane (m, G) takes row 16 TT + m, columns
    // 32 kb + 8G .. +7
    const bf16* qg = p.q + bb * p.sq[0] + hh * p.sq[1] + (16 * TT + lc) * p.sq[2] + 8 * G;
    auto load_q = [&](int i, bf16x8 (&x)[NKB]) {
      const bf16* s = qg + (int64_t)(i < N ? i : N - 1) * CB_C * p.sq[2];
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb) x[kb] = *reinterpret_cast<const bf16x8*>(s + 32 * kb);
    };
    bf16x8 Q0[NKB], Q1[NKB];
    load_q(0, Q0);
    load_q(1, Q1);
    __syncthreads();  // barrier 0
    auto out_chunk = [&](auto stg_tag, bf16x8 (&Qr)[NKB], int i) {
      constexpr int STG = decltype(stg_tag)::value;
      constexpr uint32_t SK = STG * L::TILE;
      // A^T tiles (K Q^T, causal part) -> pair-order A operands of chunk i
      f32x4 At[4];
#pragma unroll
      for (int st = 0; st < 4; ++st) At[st] = zero4();
      bf16x8 Kr[NKB][TT + 1];
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int st = 0; st <= TT; ++st) Kr[kb][st] = lds_ld<bf16x8>(rowK[kb] + (SK + st * 16 * ROWB));
      __builtin_amdgcn_sched_barrier(0);  // every read issued before the first product
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int st = 0; st <= TT; ++st) At[st] = mfma(Kr[kb][st], Qr[kb], At[st]);
      // keep s <= t on the diagonal tile: lane (t, G) row 4G + j is s
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (4 * G + j > lc) At[TT][j] = 0.f;
      Op<2> Ap[NKT];
#pragma unroll
      for (int kt = 0; kt < NKT; ++kt) Ap[kt] = pack_tiles<2>(At[2 * kt], At[2 * kt + 1]);
      __builtin_amdgcn_sched_barrier(0);  // A is packed before the barrier
      __syncthreads();  // the mid-chunk barrier of chunk i: -beta E published
      // -o^T = Sf Q^T + (-beta E)^T A^T
      const uint32_t eo = (uint32_t)(i & 1) * L::EPB, sbo = (uint32_t)(i & 1) * L::SPB;
      bf16x8 Sr[NKB][2];
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int pc = 0; pc < 2; ++pc) Sr[kb][pc] = lds_ld<bf16x8>(spr + sbo + kb * 2048 + pc * 1024);
      bf16x8 We[2][2];
#pragma unroll
      for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
        for (int pc = 0; pc < 2; ++pc) We[kt][pc] = lds_ld<bf16x8>(epr + eo + kt * 2048 + pc * 1024);
      __builtin_amdgcn_sched_barrier(0);
      f32x4 O = zero4();
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int pc = 0; pc < 2; ++pc) O = mfma(Sr[kb][pc], Qr[kb], O);
      load_q(i + 2, Qr);
      __builtin_amdgcn_sched_barrier(0);
      // (hi, hi), (hi, lo), (lo, hi) of each operand pair
#pragma unroll
      for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
        for (int pc = 0; pc < 3; ++pc) O = mfma(We[kt][pc == 2 ? 1 : 0], Ap[kt].v[pc == 1 ? 1 : 0], O);
      // lane (t, G): token 16 TT + t, state rows 4G ..
      *reinterpret_cast<bf16x4*>(og + ((int64_t)i * CB_C + 16 * TT + lc) * p.so[2]) = to_bf16x4(-O);
      __syncthreads();  // barrier i + 1
    };
    // the chunks of a ring turn without branches between them: the compiler
    // then knows how many of the wave's stores and Q reads are newer than the
    // Q rows it waits for, and waits for nothing newer
    int i = 0;
    for (; i + FE_RING <= N; i += FE_RING) {
      out_chunk(std::integral_constant<int, 0>{}, Q0, i);
      out_chunk(std::integral_constant<int, 1>{}, Q1, i + 1);
      out_chunk(std::integral_constant<int, 2>{}, Q0, i + 2);
      out_chunk(std::integral_constant<int, 3>{}, Q1, i + 3);
    }
    if (i < N) {
      out_chunk(std::integral_constant<int, 0>{}, Q0, i);
      if (i + 1 < N) {
        out_chunk(std::integral_constant<int, 1>{}, Q1, i + 1);
        if (i + 2 < N) out_chunk(std::integral_constant<int, 2>{}, Q0, i + 2);
      }
    }
  };
  switch (ow) {
    case 0: run(std::integral_constant<int, 0>{}); break;
    case 1: run(std::integral_constant<int, 1>{}); break;
    case 2: run(std::integral_constant<int, 3>{}); break;
    default: run(std::integral_constant<int, 2>{}); break;
  }
}

template <int D>
static hipError_t launch_fwd_delta16(const ChunkArgs& a, hipStream_t stream) {
  auto kern = chunk_fwd_delta16<D>;
  constexpr int lds = FwdDelta16Lds<D>::BYTES;
  hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3((unsigned)(a.B * a.H * (D / 16))), dim3(FE_THREADS), lds, stream, a);
  return hipGetLastError();
}

hipError_t chunk_fwd_delta16_launch(const ChunkArgs& a, int d, hipStream_t s) {
  return d == 128 ? launch_fwd_delta16<128>(a, s) : launch_fwd_delta16<64>(a, s);
}

}  // namespace gmdn
