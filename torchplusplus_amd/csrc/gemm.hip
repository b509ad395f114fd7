// MFMA GEMM with fused epilogue for gfx950:  C[M,N] = epi(A[M,K] . B[N,K]^T)
//
// Replaces the CUTLASS SM80 tensor-op GEMM + LinearActivationFP16 epilogue of
// csrc/activation/fused_gemm.cuh:20-170 (bound at binding.cu:11-160). B is the
// nn.Linear weight [N, K] (ldb = K, "ColumnMajor" B in CUTLASS terms), so
// both operands are K-contiguous and every load is a 128-bit row segment.
//
// Epilogues (fp32 accumulator in, T out):
//   plain      C = T(acc)
//   bias+act   C = T(act(float(T(acc + bias))))  -- the reference rounds the
//              pre-activation to half before GeluHalf/SiluHalf/ReluHalf
//              (fused_gemm.cuh:93-105); its epilogue as committed reads
//              unconverted registers (:79-89), this is the intended formula.
//   SwiGLU     weight rows interleaved in blocks of 32 ([gate 32 | up 32]...):
//              C[:, 32j+c] = T(T(silu(T(g))) * T(u)), the eager FFN chain.
//
// Tiles: 32x32 to 256x256 outputs per block of v_mfma_f32_32x32x16
// accumulators, operands by LDS-DMA in 16-byte chunks, LDS rows XOR-swizzled
// (conflict-free ds_read_b128 for the MFMA operand pattern). Blocks are mapped
// XCD-aware: the hardware deals blocks round-robin to the 8 XCDs, so block
// ids are remapped so that each XCD works on a compact group of tiles that
// share A rows and B columns in its own L2.
#include "tpp_common.hpp"

namespace tpp {

enum GemmEpi { kGPlain = 0, kGBiasAct = 1, kGSwiGLU = 2 };

// LDS tiles hold 128-byte rows of eight 16-byte chunks; chunk c of row r is
// stored at position c ^ swz(r). A ds_read_b128 serves 16 lanes (16 rows of
// one fragment) per cycle from 16 distinct 16-byte bank groups only if those
// rows land in different groups: rows r and r+1 already differ in the row's
// half of the 256-byte bank space, so the XOR uses row bits 1..3 (bits 0..2
// would put rows r and r+8 on the same banks: a 2-way conflict on every read).
__device__ __forceinline__ int swz(int row) { return (row >> 1) & 7; }

// The 256x256 tile takes BK 64 in 2 ring stages (64 KB each; 4- and 5-stage
// rings of BK 32 tiles measured slower), the 128-row tiles BK 64 in as many
// stages as fit 160 KB of LDS
// (one block per CU): 5 for 128x128, 4 for 128x192, 3 for 128x256 (at the
// Linear+act shape 3 stages were 6% faster than 2, and 4 another 3%)
constexpr int kSmallBK = 64;
// below this many outputs 128-row tiles leave CUs idle: smaller tiles, chosen
// by pick_small_tile
constexpr int64_t kDmaMinMN = 256 * 128 * 128;
// the DMA kernel addresses a tile's rows by 32-bit byte offsets from its
// first row: 256 rows * ld * 2 bytes stays below 2^32 up to this pitch
constexpr int64_t kDmaMaxLd = 1 << 22;

template <typename T>
__device__ __forceinline__ f32x16 mfma32(typename VecT<T>::v8 a, typename VecT<T>::v8 b,
                                         f32x16 c) {
  if constexpr (__is_same(T, bf16))
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ void tile_coords(int pid, int nb, int ntm, int ntn, int &tm,
                                            int &tn) {
  const int q = nb >> 3, rem = nb & 7;
  const int xcd = pid & 7, idx = pid >> 3;
  const int logical =
      (xcd < rem) ? xcd * (q + 1) + idx : rem * (q + 1) + (xcd - rem) * q + idx;
  constexpr int GM = 8;
  const int width = GM * ntn;
  const int group = logical / width;
  const int first_m = group * GM;
  const int gsz = (ntm - first_m) < GM ? (ntm - first_m) : GM;
  const int within = logical - group * width;
  tm = first_m + within % gsz;
  tn = within / gsz;
}

// ---------------------------------------------------------------------------
// Outputs of a round of 128x128 tiles and more: operands go HBM/L2 -> LDS directly with
// global_load_lds_dwordx4 (no VGPR staging, no ds_write), through an
// NST-stage ring (NST-1 K tiles in flight while one is multiplied). Block
// tile (32*WM*FM) x (32*WN*FN), WM x WN waves, wave tile (32*FM) x (32*FN).
// Why big tiles: the CU's L1 delivers ~64 B/clk while its four matrix cores
// consume 4096 bf16 flop/clk, so a BM x BN tile needs (BM+BN)/(BM*BN) <=
// 1/64 byte per flop; 128x128 sits exactly at that limit, 256x256 at half.
// Measured on MI355X: 256x256 with 8 waves (4x2 of 64x128, two per SIMD)
// runs ~37-43% of MFMA peak on the prefill shapes vs ~31% for 128x128; where
// the rounds of 256x256 tiles leave CUs idle the 128-row tiles win (one block
// per CU, rings of 3 to 5 stages; pick_dma_tile has the cost of each round).
// An LDS-DMA instruction writes lane i's 16 bytes at base + 16*i; lane i of
// a row group therefore fetches the 16-byte chunk kc = (i%8) ^ swz(row), which
// lands the tile in the same XOR-swizzled layout the fragment reads expect.
// Waits are explicit (s_waitcnt vmcnt / lgkmcnt + s_barrier): a fenced
// __syncthreads() would drain every DMA in flight at each K step.
template <int N> __device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}
__device__ __forceinline__ void wait_lgkmcnt0() { __builtin_amdgcn_s_waitcnt(0xC07F); }
// Wait until at most min(later, R) K tiles' DMA (NQ instructions each, this
// wave's share) are outstanding: the ring's DMA completes in issue order, so
// every older tile has landed.
template <int NQ, int R> __device__ __forceinline__ void wait_tiles(int later) {
  if constexpr (R <= 0) {
    wait_vmcnt<0>();
  } else {
    if (later >= R) wait_vmcnt<R * NQ>();
    else wait_tiles<NQ, R - 1>(later);
  }
}

template <int BK> __device__ __forceinline__ int swzk(int row) {
  // BK = 64: 128-byte rows, two per 256-byte bank space; BK = 32: 64-byte rows,
  // four per bank space. The XOR uses the row bits above those, so the 16
  // rows one ds_read_b128 cycle serves hit 16 distinct 16-byte bank groups.
  if constexpr (BK == 64) return (row >> 1) & 7;
  else return (row >> 2) & 3;
}

// x[e] <- float(T(x[e])) for four values, converted two at a time (one
// packed conversion per pair instead of one per value)
template <typename T> __device__ __forceinline__ void round_pairs(float (&x)[4]) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef typename VecT<T>::v2 T2;
#pragma unroll
  for (int p = 0; p < 4; p += 2) {
    const f2 in = {x[p], x[p + 1]};
    const f2 out = __builtin_convertvector(__builtin_convertvector(in, T2), f2);
    x[p] = out[0];
    x[p + 1] = out[1];
  }
}

// 16-byte LDS units of a tile: the ring, or the epilogue's staging tile that
// reuses it
template <typename T, int EPI, int FM, int FN, int NST, int WM, int WN, int BK> constexpr int dma_tile_lds() {
  const int ring = NST * (32 * WM * FM + 32 * WN * FN) * (BK / 8);
  const int ows = EPI == kGSwiGLU ? FN * 16 : FN * 32;
  const int outs = WM * WN * FM * 32 * (ows + 8) * (int)sizeof(T) / 16;
  return ring > outs ? ring : outs;
}

// The output tile at (m0, n0); `smem` holds dma_tile_lds units. TAIL: K is a
// multiple of 8 only; the last K tile's chunks past K fetch the row's last
// chunk and both fragments are zeroed there.
template <typename T, int EPI, int ACT, int FM, int FN, int NST, int WM, int WN, int BK, bool TAIL = false>
__device__ __forceinline__ void gemm_dma_tile(
    typename VecT<T>::v8 *smem, const T *__restrict__ A, int64_t lda, const T *__restrict__ B,
    int64_t ldb, T *__restrict__ C, int64_t ldc, const T *__restrict__ bias, int M, int N, int K,
    int m0, int n0) {
  typedef typename VecT<T>::v8 V8;
  constexpr int BM = 32 * WM * FM, BN = 32 * WN * FN, NWV = WM * WN;
  constexpr int CPR = BK / 8;                // 16-byte chunks per tile row
  constexpr int RPI = 64 / CPR;              // tile rows per DMA instruction
  constexpr int STG = (BM + BN) * CPR;       // 16-byte slots per stage
  constexpr int NA = BM / RPI / NWV, NB = BN / RPI / NWV; // DMA instructions per wave per stage
  static_assert(NA * RPI * NWV == BM && NB * RPI * NWV == BN, "tile rows per wave");
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int wm = w / WN, wn = w % WN;

  // DMA instruction j of wave w covers tile rows (NWV*j + w)*RPI .. +RPI-1;
  // lane i fetches row +i/CPR, chunk (i%CPR)^swzk(row). swzk(row) depends on
  // w and i only (NWV is even). Source rows are clamped to the matrix: rows
  // past M / N only feed outputs that are never stored.
  const int lrow = lane / CPR, lkc = (lane % CPR) ^ swzk<BK>(RPI * w + lrow);
  // DMA sources: a uniform tile base (row m0 of A, row n0 of B, in scalar
  // registers) plus per-lane 32-bit byte offsets of the lane's clamped rows
  // relative to it, fixed for the whole K loop (the host keeps
  // BM * ld * sizeof(T) below 2^32)
  constexpr int NQ = NA + NB;
  const char *ta = reinterpret_cast<const char *>(A) + (int64_t)m0 * lda * (int64_t)sizeof(T);
  const char *tb = reinterpret_cast<const char *>(B) + (int64_t)n0 * ldb * (int64_t)sizeof(T);
  uint32_t off[NQ];
#pragma unroll
  for (int q = 0; q < NA; ++q)
    off[q] = (uint32_t)((int64_t)(min(m0 + w * RPI + lrow + RPI * NWV * q, M - 1) - m0) * lda + lkc * 8) *
             (uint32_t)sizeof(T);
#pragma unroll
  for (int q = 0; q < NB; ++q)
    off[NA + q] = (uint32_t)((int64_t)(min(n0 + w * RPI + lrow + RPI * NWV * q, N - 1) - n0) * ldb + lkc * 8) *
                  (uint32_t)sizeof(T);
  const int nk = (K + BK - 1) / BK;
  // DMA instruction q (0 .. NQ - 1) of K tile kt into a stage
  auto issue_one = [&](int stage, int kt, int q) {
    V8 *sa = smem + stage * STG, *sb = sa + BM * CPR;
    int64_t kb = (int64_t)kt * BK * (int64_t)sizeof(T);
    if (TAIL && kt == nk - 1) kb += min(0, K - 8 - (kt * BK + lkc * 8)) * (int)sizeof(T);
    if (q < NA)
      __builtin_amdgcn_global_load_lds((const void *)(ta + kb + off[q]),
                                       (__attribute__((address_space(3))) void *)(sa + (q * NWV + w) * 64),
                                       16, 0, 0);
    else
      __builtin_amdgcn_global_load_lds((const void *)(tb + kb + off[q]),
                                       (__attribute__((address_space(3))) void *)(sb + ((q - NA) * NWV + w) * 64),
                                       16, 0, 0);
  };

  f32x16 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  // The bias is added by one more MFMA per accumulator block after the K
  // loop: A' = the bias of the block's 32 W rows in K column 0, B' = ones in
  // K row 0, so acc += bias[n] . 1 with one fp32 rounding, the add of the
  // epilogue formula, with no VALU work per output. Lane l < 32 holds
  // bias[nw0 + 32 j + l] in element 0 of fragment j (requested now, so its
  // latency hides under the main loop); every other element is zero.
  const int nw0 = n0 + wn * FN * 32; // first W row (output column before SwiGLU) of the wave
  V8 bfrag[EPI == kGBiasAct ? FN : 1];
  if constexpr (EPI == kGBiasAct) {
    if (bias) { // uniform
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int c = nw0 + j * 32 + (lane & 31);
        const T bv = bias[c < N ? c : N - 1];
#pragma unroll
        for (int e = 0; e < 8; ++e) bfrag[j][e] = (T)0.0f;
        bfrag[j][0] = (lane < 32 && c < N) ? bv : (T)0.0f;
      }
    }
  }

  // Main loop. Each K tile is KS = BK/16 sub-steps of FM x FN MFMAs, with
  // the operand fragments of sub-step ks + 1 read (into the other register
  // set) while the MFMAs of ks run. The DMA of K tile kt + NST - 1 goes into
  // the slot every wave finished reading before the last barrier and is
  // spread between the MFMAs of the first half of the tile, so no wave
  // stalls on a burst of DMA issue. The wait for K tile kt + 1's DMA and the
  // barrier that publishes it sit in the middle of the last sub-step, right
  // before the next tile's first fragment reads: the second half of the
  // sub-step's MFMAs is still to issue while the barrier resolves and those
  // reads return (measured 3-4% faster on the prefill shapes than a barrier
  // at the top of each K tile).
  constexpr int KS = BK / 16;
  static_assert(KS % 2 == 0, "register sets alternate across the K-tile boundary");
  constexpr int NMF = KS * FM * FN;
  constexpr int MID = NMF - (FM * FN) / 2; // MFMAs of a K tile issued before its barrier
  constexpr int SP = (NMF / 2) / NQ > 0 ? (NMF / 2) / NQ : 1; // MFMAs per DMA instruction
  static_assert(NQ * SP <= MID, "all DMA of a K tile issued before its barrier");
#pragma unroll
  for (int p = 0; p < NST - 1; ++p)
    if (p < nk)
#pragma unroll
      for (int q = 0; q < NQ; ++q) issue_one(p, p, q);
  // K tile 0 landed (tiles 1 .. NST-2 may be in flight)
  wait_tiles<NQ, NST - 2>(nk - 1);
  __builtin_amdgcn_s_barrier();
  V8 af[2][FM], bfr[2][FN];
  auto frag = [&](const V8 *sa, int ks) {
    const V8 *sb = sa + BM * CPR;
    const int kc = ks * 2 + (lane >> 5);
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int row = wm * FM * 32 + i * 32 + (lane & 31);
      af[ks & 1][i] = sa[row * CPR + (kc ^ swzk<BK>(row))];
    }
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int col = wn * FN * 32 + j * 32 + (lane & 31);
      bfr[ks & 1][j] = sb[col * CPR + (kc ^ swzk<BK>(col))];
    }
  };
  frag(smem, 0);
  // K tile kt, with the DMA of K tile kt + NST - 1 if there is `more`. The
  // 128-row tiles run two loops, `more` known in each: no DMA instruction under
  // a branch and constant waits, 5-10% faster ([5367 x 1024] . [3072 x
  // 1024]^T 47.7 -> 43.1 us, [2048 x 3072] + bias + SiLU, K 1024, 22.4 -> 21.1
  // us); the 256x256 tile, with 32 MFMAs per sub-step, is 9% slower that way
  // (113 -> 124 us) and keeps one loop.
  auto ktile = [&](int kt, auto more) {
    constexpr bool known = !std::is_same<decltype(more), bool>::value;
    const V8 *sa = smem + (kt % NST) * STG;
    const int kn = kt + NST - 1;
    const bool next = more || kt + 1 < nk;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      if (ks + 1 < KS) frag(sa, ks + 1);
      if (TAIL && kt == nk - 1) {
        const bool past = kt * BK + ks * 16 + (lane >> 5) * 8 >= K;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
#pragma unroll
          for (int i = 0; i < FM; ++i) af[ks & 1][i][e] = past ? (T)0.0f : af[ks & 1][i][e];
#pragma unroll
          for (int j = 0; j < FN; ++j) bfr[ks & 1][j][e] = past ? (T)0.0f : bfr[ks & 1][j][e];
        }
      }
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          acc[i][j] = mfma32<T>(bfr[ks & 1][j], af[ks & 1][i], acc[i][j]);
          const int m = (ks * FM + i) * FN + j + 1;
          if (m % SP == 0 && m / SP <= NQ && more) issue_one(kn % NST, kn, m / SP - 1);
          if (m == MID && next) {
            // own DMA of K tile kt + 1 landed (tiles kt + 2 .. kt + NST - 1
            // may still be in flight). The fragment reads of tile kt must
            // all have returned before the barrier, since after it any wave
            // may refill that slot: with one row block per wave (FM = 1) the
            // fragments of the second half of this sub-step are not consumed
            // yet, so wait for every LDS read (lgkmcnt(0); the barrier does
            // not wait for them)
            if constexpr (known && std::is_same<decltype(more), std::true_type>::value) wait_vmcnt<(NST - 2) * NQ>();
            else wait_tiles<NQ, NST - 2>(nk - kt - 2);
            wait_lgkmcnt0();
            __builtin_amdgcn_s_barrier();
            frag(smem + ((kt + 1) % NST) * STG, 0);
          }
        }
    }
  };
  if constexpr (FM == 1) {
    int kt = 0;
    for (; kt + NST - 1 < nk; ++kt) ktile(kt, std::true_type{});
    for (; kt < nk; ++kt) ktile(kt, std::false_type{});
  } else {
    for (int kt = 0; kt < nk; ++kt) ktile(kt, kt + NST - 1 < nk);
  }

  if constexpr (EPI == kGBiasAct) {
    if (bias) {
      V8 ones;
#pragma unroll
      for (int e = 0; e < 8; ++e) ones[e] = (T)0.0f;
      ones[0] = lane < 32 ? (T)1.0f : (T)0.0f;
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = mfma32<T>(bfrag[j], ones, acc[i][j]);
    }
  }

  // Epilogue. The operands are swapped in the MFMA (W rows first), so the
  // 32x32 accumulator holds lane -> output row m = i*32 + (lane & 31) and
  // registers 4q..4q+3 -> four consecutive output columns
  // n = j*32 + q*8 + (lane/32)*4 + {0..3}. Each wave converts its 32FM x 32FN
  // tile, packs 4 columns per 8-byte LDS write into a padded row-major
  // staging tile (the ring is free by now), then stores whole rows with
  // 16-byte global writes.
  constexpr int OW = (EPI == kGSwiGLU) ? FN * 16 : FN * 32; // output cols per wave
  constexpr int LDR = OW + 8; // staging row pitch in elements (16-byte aligned rows)
  wait_lgkmcnt0();
  __builtin_amdgcn_s_barrier(); // every wave is done reading the ring
  T *stage = reinterpret_cast<T *>(smem) + w * (FM * 32 * LDR);
  const int half = lane >> 5, ml = lane & 31;
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    if constexpr (EPI == kGSwiGLU) {
      if (j & 1) continue;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int nl = j * 32 + q * 8 + half * 4; // wave-local W column of register 4q
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        typename VecT<T>::v4 pk;
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[i][j][4 * q + e];
        if constexpr (EPI == kGSwiGLU) {
          float u[4], sl[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) u[e] = acc[i][j + 1][4 * q + e];
          round_pairs<T>(v);
          round_pairs<T>(u);
#pragma unroll
          for (int e = 0; e < 4; ++e) sl[e] = act_silu(v[e]);
          round_pairs<T>(sl);
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = sl[e] * u[e];
        } else if constexpr (EPI == kGBiasAct) {
          round_pairs<T>(v); // the pre-activation rounded to T (bias already in acc)
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = apply_act<ACT>(v[e]);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) pk[e] = from_f32<T>(v[e]);
        const int col = (EPI == kGSwiGLU) ? (j / 2) * 32 + q * 8 + half * 4 : nl;
        *reinterpret_cast<typename VecT<T>::v4 *>(stage + (i * 32 + ml) * LDR + col) = pk;
      }
    }
  }
  wait_lgkmcnt0();
  // rows of the wave tile: OW/8 lanes per row, 16 bytes each; RPI rows per
  // pass (with OW = 96, lanes 60..63 idle)
  constexpr int LPR = OW / 8, OPR = 64 / LPR; // output rows per pass
  const int oc0 = (EPI == kGSwiGLU) ? nw0 / 2 : nw0;
  const int NO = (EPI == kGSwiGLU) ? N / 2 : N;
  const int rr = lane / LPR, cc = (lane % LPR) * 8;
  const bool vec_ok = (ldc % 8 == 0) && ((reinterpret_cast<uintptr_t>(C) & 15) == 0);
#pragma unroll
  for (int r0 = 0; r0 < FM * 32; r0 += OPR) {
    const int rl = r0 + rr;
    if (rr >= OPR || rl >= FM * 32) continue;
    const int row = m0 + wm * FM * 32 + rl;
    const typename VecT<T>::v8 v =
        *reinterpret_cast<const typename VecT<T>::v8 *>(stage + rl * LDR + cc);
    if (row >= M) continue;
    const int col = oc0 + cc;
    T *dst = C + (int64_t)row * ldc + col;
    if (vec_ok && col + 8 <= NO) {
      *reinterpret_cast<typename VecT<T>::v8 *>(dst) = v;
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (col + e < NO) dst[e] = v[e];
    }
  }
}

template <typename T, int EPI, int ACT, int FM, int FN, int NST, int WM, int WN, int BK>
__global__ __launch_bounds__(64 * WM * WN) void gemm_dma_kernel(
    const T *__restrict__ A, int64_t lda, const T *__restrict__ B, int64_t ldb,
    T *__restrict__ C, int64_t ldc, const T *__restrict__ bias, int M, int N, int K) {
  constexpr int BM = 32 * WM * FM, BN = 32 * WN * FN;
  __shared__ typename VecT<T>::v8 smem[dma_tile_lds<T, EPI, FM, FN, NST, WM, WN, BK>()];
  const int ntm = (M + BM - 1) / BM, ntn = (N + BN - 1) / BN;
  int tm, tn;
  tile_coords(blockIdx.x, ntm * ntn, ntm, ntn, tm, tn);
  gemm_dma_tile<T, EPI, ACT, FM, FN, NST, WM, WN, BK>(smem, A, lda, B, ldb, C, ldc, bias, M, N, K,
                                                       tm * BM, tn * BN);
}

// Two tile sizes in one launch: 256x256 tiles over the first Mb rows, as many
// as fill the CUs in whole rounds, and 128x128 tiles over the rest. 256x256
// tiles are the fastest per output, but 300 of them on 256 CUs take two rounds
// for 1.17 rounds of work, and smaller tiles everywhere lose their operand
// reuse: 6227 x 3072 x 1024 + bias + GeLU (bf16) 66.4 us with 256x256 tiles,
// 74.0 with 128x128, 52.4 mixed; 3000 x 6144 x 1024 SwiGLU 54.0 -> 43.8 us;
// 6227 x 5632 x 2048 + bias + GeLU 177 -> 146 us. The TAIL form takes any K % 8
// == 0, with all rows (or none) in 256x256 tiles where those (or 128x128) are
// the better plan. It took the place of a register-staged 128x128 kernel:
// 6227 x 3072 x 1000 + bias + GeLU 101 -> 55 us, 16384 x 3072 x 1000 + bias +
// SiLU 220 -> 120, 2649 x 3072 x 1000 40 -> 32, 1600 x 5632 x 2008 80 -> 53.
template <typename T, int EPI, int ACT, bool TAIL>
__global__ __launch_bounds__(512) void gemm_mixed_kernel(
    const T *__restrict__ A, int64_t lda, const T *__restrict__ B, int64_t ldb,
    T *__restrict__ C, int64_t ldc, const T *__restrict__ bias, int M, int N, int K, int Mb) {
  constexpr int LB = dma_tile_lds<T, EPI, 2, 4, 2, 4, 2, 64>(), LS = dma_tile_lds<T, EPI, 1, 2, 4, 4, 2, 64>();
  __shared__ typename VecT<T>::v8 smem[LB > LS ? LB : LS];
  const int ntb = (N + 255) / 256, nbig = Mb / 256 * ntb;
  int tm, tn;
  if ((int)blockIdx.x < nbig) {
    tile_coords(blockIdx.x, nbig, Mb / 256, ntb, tm, tn);
    gemm_dma_tile<T, EPI, ACT, 2, 4, 2, 4, 2, 64, TAIL>(smem, A, lda, B, ldb, C, ldc, bias, M, N, K, tm * 256, tn * 256);
  } else {
    const int ntm = (M - Mb + 127) / 128, ntn = (N + 127) / 128;
    tile_coords(blockIdx.x - nbig, ntm * ntn, ntm, ntn, tm, tn);
    gemm_dma_tile<T, EPI, ACT, 1, 2, 4, 4, 2, 64, TAIL>(smem, A, lda, B, ldb, C, ldc, bias, M, N, K,
                                                   Mb + tm * 128, tn * 128);
  }
}

// ---------------------------------------------------------------------------
// Persistent 256x256 variant for launches with more tiles than CUs (the
// prefill projections: 4-6 tiles per CU). One workgroup per CU loops over the
// tiles b, b + gridDim, ... (all on the workgroup's XCD: gridDim is a
// multiple of 8, and tile_coords keeps an XCD's tiles a compact group). The
// K steps of consecutive tiles form one stream through the 2-stage ring: the
// last K step of a tile issues the DMA of the next tile's first K step, and
// the epilogue, staged through the slot that K step has just finished
// reading (64 KB: 8 KB per wave, two passes), issues the next tile's second
// K step before its global stores, so neither the first DMA of a tile nor the
// store drain sits on the critical path. Measured on the prefill shapes:
// 3-7% faster than one workgroup per tile. Plain and SwiGLU epilogues only
// (a bias prefetch for the next tile does not fit the registers).
template <typename T, int EPI, int ACT>
__global__ __launch_bounds__(512) void gemm_persist_kernel(
    const T *__restrict__ A, int64_t lda, const T *__restrict__ B, int64_t ldb,
    T *__restrict__ C, int64_t ldc, const T *__restrict__ bias, int M, int N, int K) {
  typedef typename VecT<T>::v8 V8;
  typedef typename VecT<T>::v4 V4;
  static_assert(EPI == kGPlain || EPI == kGSwiGLU, "plain or SwiGLU epilogue");
  constexpr int FM = 2, FN = 4, WM = 4, WN = 2, BK = 64, NST = 2;
  constexpr int BM = 32 * WM * FM, BN = 32 * WN * FN, NWV = WM * WN;
  constexpr int CPR = BK / 8, RPI = 64 / CPR;
  constexpr int STG = (BM + BN) * CPR;
  constexpr int NA = BM / RPI / NWV, NB = BN / RPI / NWV, NQ = NA + NB;
  constexpr int KS = BK / 16, NMF = KS * FM * FN, MID = NMF - (FM * FN) / 2;
  constexpr int SP = (NMF / 2) / NQ > 0 ? (NMF / 2) / NQ : 1;
  static_assert(NQ * SP <= MID, "all DMA of a K step issued before its barrier");
  // epilogue staging per wave and pass: 64 rows x OWP output columns, read
  // back in NR rounds of 16 bytes per lane (NSTO global stores per wave)
  constexpr int OWP = (EPI == kGSwiGLU) ? 32 : 64;
  constexpr int RB = OWP * (int)sizeof(T), LPR = RB / 16, OPR = 64 / LPR;
  constexpr int NR = FM * 32 / OPR, NSTO = 2 * NR;
  static_assert(NWV * FM * 32 * RB <= STG * 16, "staging fits one ring slot");
  __shared__ V8 smem[NST * STG];

  const int ntm = (M + BM - 1) / BM, ntn = (N + BN - 1) / BN, ntiles = ntm * ntn;
  // wave index in a scalar register: every per-wave decision (DMA rows,
  // store path, wait counts) is then provably uniform
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = w / WN, wn = w % WN;
  const int half = lane >> 5, ml = lane & 31;
  const int lrow = lane / CPR, lkc = (lane % CPR) ^ swzk<BK>(RPI * w + lrow);
  const int nk = K / BK;
  int tile = blockIdx.x;
  if (tile >= ntiles) return;

  // DMA sources of a tile: uniform tile bases plus per-lane 32-bit offsets of
  // the lane's clamped rows (the host keeps BM * ld * sizeof(T) below 2^32)
  struct Src {
    const char *ta, *tb;
    uint32_t off[NQ];
    int m0, n0;
  };
  auto src_of = [&](int t, Src &s) {
    int tm, tn;
    tile_coords(t, ntiles, ntm, ntn, tm, tn);
    s.m0 = tm * BM;
    s.n0 = tn * BN;
    s.ta = reinterpret_cast<const char *>(A) + (int64_t)s.m0 * lda * (int64_t)sizeof(T);
    s.tb = reinterpret_cast<const char *>(B) + (int64_t)s.n0 * ldb * (int64_t)sizeof(T);
#pragma unroll
    for (int q = 0; q < NA; ++q)
      s.off[q] = (uint32_t)((int64_t)(min(s.m0 + w * RPI + lrow + RPI * NWV * q, M - 1) - s.m0) * lda +
                            lkc * 8) * (uint32_t)sizeof(T);
#pragma unroll
    for (int q = 0; q < NB; ++q)
      s.off[NA + q] = (uint32_t)((int64_t)(min(s.n0 + w * RPI + lrow + RPI * NWV * q, N - 1) - s.n0) * ldb +
                                 lkc * 8) * (uint32_t)sizeof(T);
  };
  auto issue = [&](const Src &s, int stage, int kt, int q) {
    V8 *sa = smem + stage * STG, *sb = sa + BM * CPR;
    const int64_t kb = (int64_t)kt * BK * sizeof(T);
    if (q < NA)
      __builtin_amdgcn_global_load_lds((const void *)(s.ta + kb + s.off[q]),
                                       (__attribute__((address_space(3))) void *)(sa + (q * NWV + w) * 64),
                                       16, 0, 0);
    else
      __builtin_amdgcn_global_load_lds((const void *)(s.tb + kb + s.off[q]),
                                       (__attribute__((address_space(3))) void *)(sb + ((q - NA) * NWV + w) * 64),
                                       16, 0, 0);
  };
  V8 af[2][FM], bfr[2][FN];
  auto frag = [&](const V8 *sa, int ks) {
    const V8 *sb = sa + BM * CPR;
    const int kc = ks * 2 + (lane >> 5);
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int row = wm * FM * 32 + i * 32 + (lane & 31);
      af[ks & 1][i] = sa[row * CPR + (kc ^ swzk<BK>(row))];
    }
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int col = wn * FN * 32 + j * 32 + (lane & 31);
      bfr[ks & 1][j] = sb[col * CPR + (kc ^ swzk<BK>(col))];
    }
  };

  Src cur, nxt;
  src_of(tile, cur);
#pragma unroll
  for (int q = 0; q < NQ; ++q) issue(cur, 0, 0, q);
  wait_vmcnt<0>();
  __builtin_amdgcn_s_barrier();
  frag(smem, 0);
  int slot = 0;
  // K step 1 of the current tile already in flight (issued in the previous
  // tile's epilogue), with `sto` store instructions of that epilogue issued
  // after it (-1: an unknown number)
  bool pre = false;
  int sto = -1;
  for (;;) {
    const int tnext = tile + (int)gridDim.x;
    const bool has_next = tnext < ntiles;
    if (has_next) src_of(tnext, nxt);
    const int nw0 = cur.n0 + wn * FN * 32; // first W row (output column before SwiGLU) of the wave
    f32x16 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    // K loop: step kt reads slot `slot`; its DMA fills the other slot with
    // K step kt + 1, or with the next tile's first K step after the last
    for (int kt = 0; kt < nk; ++kt) {
      const V8 *sa = smem + slot * STG;
      const bool last = kt + 1 == nk;
      const bool more = !last || has_next;
      const bool early = kt == 0 && pre; // this step's DMA was issued early
      const bool dma = more && !early;
      const Src &ds = last ? nxt : cur;
      const int kd = last ? 0 : kt + 1;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        if (ks + 1 < KS) frag(sa, ks + 1);
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j) {
            acc[i][j] = mfma32<T>(bfr[ks & 1][j], af[ks & 1][i], acc[i][j]);
            const int m = (ks * FM + i) * FN + j + 1;
            if (m % SP == 0 && m / SP <= NQ && dma) issue(ds, slot ^ 1, kd, m / SP - 1);
            if (m == MID && more) {
              // the other slot's DMA landed; this slot's fragment reads all
              // returned (lgkmcnt(0): the slot is refilled after the
              // barrier). Vector memory operations complete in issue order,
              // so behind an early DMA only the epilogue stores issued after
              // it may stay in flight.
              if (early && sto == NSTO) wait_vmcnt<NSTO>();
              else wait_vmcnt<0>();
              wait_lgkmcnt0();
              __builtin_amdgcn_s_barrier();
              frag(smem + (slot ^ 1) * STG, 0);
            }
          }
      }
      slot ^= 1;
    }

    // Epilogue through the slot the last K step read (slot ^ 1 now), which
    // every wave has finished with after this barrier; the next tile's first
    // K step is in the other slot (its first fragments already requested).
    // The output is converted, staged (per wave, two passes of OWP columns)
    // and read back into registers; then the next tile's second K step is
    // issued into the staging slot ahead of the global stores, so the stores
    // drain under the next tile's first K step.
    wait_lgkmcnt0();
    __builtin_amdgcn_s_barrier();
    T *stage = reinterpret_cast<T *>(smem + (slot ^ 1) * STG) + w * (FM * 32 * OWP);
    auto sw = [](int row) { return (RB == 128) ? (row >> 1) & 7 : (row >> 2) & 3; };
    const int NO = (EPI == kGSwiGLU) ? N / 2 : N;
    const int oc0 = (EPI == kGSwiGLU) ? nw0 / 2 : nw0;
    V8 ov[2][NR];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
#pragma unroll
      for (int jj = 0; jj < 2; ++jj) {
        const int j = 2 * p + jj;
        if constexpr (EPI == kGSwiGLU) {
          if (jj == 1) continue;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
#pragma unroll
          for (int i = 0; i < FM; ++i) {
            V4 pk;
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = acc[i][j][4 * q + e];
            if constexpr (EPI == kGSwiGLU) {
              float u[4], sl[4];
#pragma unroll
              for (int e = 0; e < 4; ++e) u[e] = acc[i][j + 1][4 * q + e];
              round_pairs<T>(v);
              round_pairs<T>(u);
#pragma unroll
              for (int e = 0; e < 4; ++e) sl[e] = act_silu(v[e]);
              round_pairs<T>(sl);
#pragma unroll
              for (int e = 0; e < 4; ++e) v[e] = sl[e] * u[e];
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) pk[e] = from_f32<T>(v[e]);
            const int row = i * 32 + ml;
            const int col = ((EPI == kGSwiGLU) ? 0 : jj * 32) + q * 8 + half * 4; // column in the pass
            const int byte = row * RB + (((col * (int)sizeof(T)) / 16) ^ sw(row)) * 16 +
                             (col * (int)sizeof(T)) % 16;
            *reinterpret_cast<V4 *>(reinterpret_cast<char *>(stage) + byte) = pk;
          }
        }
      }
      wait_lgkmcnt0(); // this wave's staging rows written (the staging is per wave)
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        const int rl = r * OPR + lane / LPR, ch = lane % LPR;
        ov[p][r] = *reinterpret_cast<const V8 *>(reinterpret_cast<const char *>(stage) + rl * RB +
                                                 (ch ^ sw(rl)) * 16);
      }
      wait_lgkmcnt0(); // the staging reads returned before the next pass overwrites it
    }
    // every wave is done with the staging slot: the next tile's second K step
    // may refill it
    __builtin_amdgcn_s_barrier();
    pre = has_next && nk > 1;
    if (pre) {
#pragma unroll
      for (int q = 0; q < NQ; ++q) issue(nxt, slot ^ 1, 1, q);
    }
    __builtin_amdgcn_sched_barrier(0); // the stores stay behind the DMA
    const int orow0 = cur.m0 + wm * FM * 32;
    const bool vec_ok = (ldc % 8 == 0) && ((reinterpret_cast<uintptr_t>(C) & 15) == 0);
    // whole wave tile inside the output: one 16-byte store per readback round
    const bool full = vec_ok && orow0 + FM * 32 <= M && oc0 + 2 * OWP <= NO;
    if (full) {
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          const int rl = r * OPR + lane / LPR, ch = lane % LPR;
          *reinterpret_cast<V8 *>(C + (int64_t)(orow0 + rl) * ldc + oc0 + p * OWP + ch * 8) = ov[p][r];
        }
    } else {
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          const int rl = r * OPR + lane / LPR, ch = lane % LPR;
          const int row = orow0 + rl;
          const int col = oc0 + p * OWP + ch * 8;
          if (row >= M) continue;
          T *dst = C + (int64_t)row * ldc + col;
          if (vec_ok && col + 8 <= NO) {
            *reinterpret_cast<V8 *>(dst) = ov[p][r];
          } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
              if (col + e < NO) dst[e] = ov[p][r][e];
          }
        }
    }
    sto = full ? NSTO : -1;
    if (!has_next) break;
    tile = tnext;
    cur = nxt;
  }
}

// ---------------------------------------------------------------------------
// Small outputs (short prompts, batches of decode tokens): 32FM x 32FN tiles,
// the K dimension split over the block's NW waves. Wave w takes the 64-deep K
// chunks w, w + NW, ... through its own two-slot LDS ring (LDS-DMA, no barrier
// in the K loop), then the waves' partial tiles are summed in LDS in wave
// order (deterministic) and the epilogue runs on the sums.
// What bounds it: with few outputs a 128-row tile leaves most CUs idle and
// its K steps form a serial chain of memory round trips ([230 x 3072] .
// [1024 x 3072]^T: 16 blocks, 48 steps of ~0.9 us). Small tiles fill the chip
// but read more operand bytes per CU (~60 B/clk through L1), and the NW waves'
// independent rings keep 64-128 KB of them in flight per CU, so the launch
// costs its bytes over that rate plus ~3 us of launch, first round trip and
// sum. Measured (bf16, weights cold, us; the register-staged 128x128 kernel
// first): 230x1024x3072 45.0 -> 6.8, 230x4096x1024 19.1 -> 6.8, 77x1024x3072
// + bias + GeLU 52.1 -> 7.4, 600x1024x1024 18.7 -> 6.6, 230x6144x1024 SwiGLU
// 18.7 -> 9.2. Splitting K over blocks instead would need a cross-block sum
// (~2 us); rings of 3 and 4 slots, 8 waves per 32x32 tile and 4 waves of two
// K halves per 64x64 tile were no faster.
template <int FM, int FN> constexpr int ksplit_wave_lds() { // 16-byte units per wave
  const int ring = 2 * (32 * FM + 32 * FN) * 8, part = 32 * FM * (32 * FN + 4) / 4;
  return ring > part ? ring : part;
}

template <typename T, int EPI, int ACT, int FM, int FN, int NW>
__device__ __forceinline__ void gemm_ksplit_tile(
    typename VecT<T>::v8 *smem, const T *__restrict__ A, int64_t lda, const T *__restrict__ B,
    int64_t ldb, T *__restrict__ C, int64_t ldc, const T *__restrict__ bias, int M, int N, int K,
    int m0, int n0) {
  typedef typename VecT<T>::v8 V8;
  constexpr int NST = 2; // ring slots per wave
  constexpr int BM = 32 * FM, BN = 32 * FN, ROWS = BM + BN;
  constexpr int NQ = ROWS / 8;        // DMA instructions per chunk (8 rows of 128 bytes each)
  constexpr int STG = ROWS * 8;       // 16-byte units per ring slot
  constexpr int LDR = BN + 4;         // fp32 pitch of a partial tile (odd in 16-byte units)
  constexpr int WREG = ksplit_wave_lds<FM, FN>();
  static_assert(NQ * (NST - 1) < 64, "vmcnt range");
  static_assert(EPI != kGSwiGLU || FN % 2 == 0, "whole [gate | up] pairs per tile");
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);

  // DMA instruction q: slot rows 8q .. 8q + 7 (A rows, then B rows), lane l
  // row 8q + l / 8, fetching the chunk that its slot position holds under the
  // XOR swizzle. Rows past M / N read the last row (outputs never stored).
  const char *src[NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const int r = 8 * q + (lane >> 3);
    src[q] = 8 * q < BM
                 ? reinterpret_cast<const char *>(A + (int64_t)min(m0 + r, M - 1) * lda)
                 : reinterpret_cast<const char *>(B + (int64_t)min(n0 + r - BM, N - 1) * ldb);
  }
  // k of the lane's unit in chunk 0, for even and odd q
  const int k_even = ((lane & 7) ^ (lane >> 4)) * 8, k_odd = ((lane & 7) ^ (4 + (lane >> 4))) * 8;
  V8 *const ring = smem + w * WREG;
  // units past K (the last chunk of a K that is no multiple of 64) read the
  // row's last one; the fragments zero them
  auto issue = [&](int c, int slot) {
    const uint32_t ke = (uint32_t)min(c * 64 + k_even, K - 8) * (uint32_t)sizeof(T);
    const uint32_t ko = (uint32_t)min(c * 64 + k_odd, K - 8) * (uint32_t)sizeof(T);
#pragma unroll
    for (int q = 0; q < NQ; ++q)
      __builtin_amdgcn_global_load_lds(
          (const void *)(src[q] + ((q & 1) ? ko : ke)),
          (__attribute__((address_space(3))) void *)(ring + slot * STG + q * 64), 16, 0, 0);
  };

  const int nch = (K + 63) / 64;
  const int n = w < nch ? (nch - w + NW - 1) / NW : 0; // this wave's chunks
#pragma unroll
  for (int i = 0; i < NST; ++i)
    if (i < n) issue(w + i * NW, i);

  f32x16 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  const int l32 = lane & 31, half = lane >> 5, sw = swz(l32);
  const unsigned lbase = (unsigned)(uintptr_t)(const __attribute__((address_space(3))) char *)ring + l32 * 128;
  int slot = 0;
  for (int i = 0; i < n; ++i) {
    wait_tiles<NQ, NST - 1>(n - 1 - i); // chunk i landed
    const unsigned sb = lbase + slot * (STG * 16);
    V8 f[4][FM + FN];
    static_for<4>([&](auto kk) {
      constexpr int ks = decltype(kk)::value;
      const unsigned a = sb + (((ks * 2 + half) ^ sw) << 4);
      static_for<FM + FN>([&](auto ii) {
        constexpr int r = decltype(ii)::value;
        f[ks][r] = lds_read_b128<r * 32 * 128, V8>(a);
      });
    });
    const int c = w + i * NW;
    const bool tail = c * 64 + 64 > K;
    static_for<4>([&](auto kk) {
      constexpr int ks = decltype(kk)::value;
      lds_wait_tied<(3 - ks) * (FM + FN)>(f[ks]);
      if constexpr (ks == 3) {
        // every fragment is in registers: refill the slot
        asm volatile("" ::: "memory");
        if (i + NST < n) issue(c + NST * NW, slot);
      }
      if (tail) {
        const bool past = c * 64 + (ks * 2 + half) * 8 >= K;
#pragma unroll
        for (int r = 0; r < FM + FN; ++r)
#pragma unroll
          for (int e = 0; e < 8; ++e) f[ks][r][e] = past ? (T)0.0f : f[ks][r][e];
      }
#pragma unroll
      for (int ii = 0; ii < FM; ++ii)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[ii][j] = mfma32<T>(f[ks][FM + j], f[ks][ii], acc[ii][j]);
    });
    slot = slot + 1 == NST ? 0 : slot + 1;
  }

  // Partial tiles in LDS (each wave over its own ring, drained above), W rows
  // first in the MFMA: a lane holds output row lane & 31 and four consecutive
  // columns per register group.
  float *const part = reinterpret_cast<float *>(ring);
#pragma unroll
  for (int ii = 0; ii < FM; ++ii)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[ii][j][4 * q + e];
        *reinterpret_cast<f32x4 *>(part + (ii * 32 + l32) * LDR + j * 32 + q * 8 + half * 4) = v;
      }
  __syncthreads();

  constexpr int OW = (EPI == kGSwiGLU) ? BN / 2 : BN, CPR = OW / 8; // output columns, 8-column groups
  const int NO = (EPI == kGSwiGLU) ? N / 2 : N, oc0 = (EPI == kGSwiGLU) ? n0 / 2 : n0;
  const bool vec_ok = (ldc % 8 == 0) && ((reinterpret_cast<uintptr_t>(C) & 15) == 0);
  auto total = [&](int row, int col, float (&v)[8]) {
    const float *p = reinterpret_cast<const float *>(smem) + row * LDR + col;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = 0.f;
#pragma unroll
    for (int ww = 0; ww < NW; ++ww) {
      const f32x4 a = *reinterpret_cast<const f32x4 *>(p + ww * WREG * 4);
      const f32x4 b = *reinterpret_cast<const f32x4 *>(p + ww * WREG * 4 + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += a[e], v[e + 4] += b[e];
    }
  };
  for (int idx = tid; idx < BM * CPR; idx += 64 * NW) {
    const int rl = idx / CPR, cl = (idx % CPR) * 8;
    const int row = m0 + rl, col = oc0 + cl;
    if (row >= M || col >= NO) continue;
    float v[8];
    if constexpr (EPI == kGSwiGLU) {
      // gate columns 64p .. + 31, up columns the next 32, of pair p
      const int wc = (cl / 32) * 64 + cl % 32;
      float u[8];
      total(rl, wc, v);
      total(rl, wc + 32, u);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float s = to_f32(from_f32<T>(act_silu(to_f32(from_f32<T>(v[e])))));
        v[e] = s * to_f32(from_f32<T>(u[e]));
      }
    } else {
      total(rl, cl, v);
      if constexpr (EPI == kGBiasAct) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          if (bias) v[e] += to_f32(bias[col + e < N ? col + e : N - 1]);
          v[e] = apply_act<ACT>(to_f32(from_f32<T>(v[e])));
        }
      }
    }
    V8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = from_f32<T>(v[e]);
    T *dst = C + (int64_t)row * ldc + col;
    if (vec_ok && col + 8 <= NO) {
      *reinterpret_cast<V8 *>(dst) = o;
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (col + e < NO) dst[e] = o[e];
    }
  }
}

template <typename T, int EPI, int ACT, int FM, int FN, int NW>
__global__ __launch_bounds__(64 * NW) void gemm_ksplit_kernel(
    const T *__restrict__ A, int64_t lda, const T *__restrict__ B, int64_t ldb,
    T *__restrict__ C, int64_t ldc, const T *__restrict__ bias, int M, int N, int K) {
  constexpr int BM = 32 * FM, BN = 32 * FN;
  __shared__ typename VecT<T>::v8 smem[NW * ksplit_wave_lds<FM, FN>()];
  const int ntm = (M + BM - 1) / BM, ntn = (N + BN - 1) / BN;
  int tm, tn;
  tile_coords(blockIdx.x, ntm * ntn, ntm, ntn, tm, tn);
  gemm_ksplit_tile<T, EPI, ACT, FM, FN, NW>(smem, A, lda, B, ldb, C, ldc, bias, M, N, K, tm * BM, tn * BN);
}

// Up to three plain products of one A (an attention layer's query, key and
// value projections) in one launch: the tile columns of the three outputs
// follow one another, each tile belonging to one of them. The projections of
// a layer are the width of one weight each, so apart they fill the chip badly
// (and cost a launch each). Three weights of [1024 x 1024], bf16, us, three
// launches -> one: 100 rows 11.4 -> 5.9, 640 18.8 -> 10.5, 2000 28.9 -> 22.3,
// 4500 51.0 -> 34.1; [1024 | 128 | 128], 2412 rows 20.5 -> 13.2.
struct Group3 {
  const void *B[3];
  void *C[3];
  int N[3];  // output columns (row pitch of C)
  int nt[3]; // tile columns
};
template <typename T> struct GroupTile {
  const T *B;
  T *C;
  int N, tm, tn;
};
template <typename T> __device__ __forceinline__ GroupTile<T> group_tile(const Group3 &g, int ntm) {
  const int ntn = g.nt[0] + g.nt[1] + g.nt[2];
  int tm, tn;
  tile_coords(blockIdx.x, ntm * ntn, ntm, ntn, tm, tn);
  const int i = tn < g.nt[0] ? 0 : tn < g.nt[0] + g.nt[1] ? 1 : 2;
  tn -= (i > 0 ? g.nt[0] : 0) + (i > 1 ? g.nt[1] : 0);
  return {(const T *)(i == 0 ? g.B[0] : i == 1 ? g.B[1] : g.B[2]), (T *)(i == 0 ? g.C[0] : i == 1 ? g.C[1] : g.C[2]),
          i == 0 ? g.N[0] : i == 1 ? g.N[1] : g.N[2], tm, tn};
}
template <typename T, int FM, int FN, int NST, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN) void gemm_dma_group_kernel(const T *__restrict__ A, int64_t lda,
                                                                      Group3 g, int M, int K) {
  constexpr int BM = 32 * WM * FM, BN = 32 * WN * FN;
  __shared__ typename VecT<T>::v8 smem[dma_tile_lds<T, kGPlain, FM, FN, NST, WM, WN, 64>()];
  const GroupTile<T> t = group_tile<T>(g, (M + BM - 1) / BM);
  gemm_dma_tile<T, kGPlain, TPP_ACT_NONE, FM, FN, NST, WM, WN, 64>(smem, A, lda, t.B, K, t.C, t.N, nullptr, M,
                                                                   t.N, K, t.tm * BM, t.tn * BN);
}
template <typename T, int FM, int FN, int NW>
__global__ __launch_bounds__(64 * NW) void gemm_ksplit_group_kernel(const T *__restrict__ A, int64_t lda,
                                                                    Group3 g, int M, int K) {
  constexpr int BM = 32 * FM, BN = 32 * FN;
  __shared__ typename VecT<T>::v8 smem[NW * ksplit_wave_lds<FM, FN>()];
  const GroupTile<T> t = group_tile<T>(g, (M + BM - 1) / BM);
  gemm_ksplit_tile<T, kGPlain, TPP_ACT_NONE, FM, FN, NW>(smem, A, lda, t.B, K, t.C, t.N, nullptr, M, t.N, K,
                                                         t.tm * BM, t.tn * BN);
}

// Tiles of an output of kDmaMinMN elements and more: the cheapest plan by the
// time of its rounds (tiles / CUs), in us from fits of each kernel over M 700 -
// 16384, N 1024 - 11264, K 768 - 3072 (bf16; 6-10% rms, the rounds themselves
// make steps of up to 2x): a round costs `full` or, not filled, `part` per 1024
// of K plus `round`, the launch `base`. The mixed plan fills whole rounds with
// 256x256 tiles and tiles the remaining rows by 128x128. Over 75 shapes the
// plan chosen is within 1% of the fastest on average (at most 6%) and 9%
// faster than the choice by tile area alone (up to 1.5x).
enum BigTile { kTile128x128, kTile128x192, kTile128x256, kTile256x256, kTileMixed };
struct BigPlan {
  BigTile tile;
  int64_t big_rows; // rows of the 256x256 part (mixed)
  double us;
};
// Output columns of a launch: of one matrix, or of three side by side.
struct OutCols {
  int64_t n[3];
  int count;
  int64_t tiles(int bn) const {
    int64_t t = 0;
    for (int i = 0; i < count; ++i) t += (n[i] + bn - 1) / bn;
    return t;
  }
};
static BigPlan pick_dma_tile(int64_t M, const OutCols &cols, int64_t K, bool swiglu, bool persist, int cus,
                             bool mixed = true, bool tail = false) {
  struct Cand { BigTile id; int bm, bn; double base, full, part, round; };
  const Cand cands[] = {{kTile128x128, 128, 128, 1.0, 8.7, 8.7, 3.5},
                        {kTile128x192, 128, 192, 0.0, 11.0, 12.0, 6.0},
                        {kTile128x256, 128, 256, 1.0, 15.0, 14.0, 5.5},
                        {kTile256x256, 256, 256, 1.5, 25.0, 21.0, 7.5}};
  const double k = (double)K / 1024.0;
  BigPlan best{kTile128x128, 0, 0.0};
  double best_t = -1.0;
  auto tiles_of = [&](int64_t rows, int bm, int bn) { return ((rows + bm - 1) / bm) * cols.tiles(bn); };
  for (const Cand &c : cands) {
    if (swiglu && c.id == kTile128x192) continue; // whole [gate | up] 64-column pairs per wave
    if (tail && (c.id == kTile128x192 || c.id == kTile128x256)) continue; // tiles of the mixed kernel
    const int64_t tiles = tiles_of(M, c.bm, c.bn), full = tiles / cus, part = tiles % cus ? 1 : 0;
    const bool loop = c.id == kTile256x256 && persist && tiles > cus; // the persistent kernel
    const double t = (loop ? 3.0 : c.base) + (double)full * (c.full * k + (loop ? 3.5 : c.round)) +
                     (double)part * (c.part * k + (loop ? 3.5 : c.round));
    if (best_t < 0 || t < best_t) best = {c.id, 0, t}, best_t = t;
  }
  const int64_t ntn = cols.tiles(256);
  for (int64_t r = 1; mixed && r * cus <= tiles_of(M, 256, 256) && r <= 64; ++r) {
    const int64_t rows = r * cus / ntn * 256; // row blocks that fit r rounds
    if (rows < 256 || rows >= M) continue;
    const int64_t small = (tiles_of(M - rows, 128, 128) + cus - 1) / cus;
    const double t = 2.5 + (double)r * (23.5 * k + 6.5) + (double)small * (8.7 * k + 3.5);
    if (t < best_t) best = {kTileMixed, rows, t}, best_t = t;
  }
  return best;
}

// Tile of an output below kDmaMinMN elements: the cheapest candidate by its
// measured time per round of resident tiles (1 or 2 per CU), in us per 1024 of
// K beyond the ~3 us every launch costs; one tile per CU at most is cheaper
// than a full round for the two-per-CU shapes. Measured at M 32 - 2048, N
// 1024 - 6144, K 1024 - 3072 (bf16): it picks the fastest or within 10% of it,
// e.g. 512x1024x3072: 32x32 11.0, 64x32 8.8, 64x64 11.0, 128x64 18.7 us;
// 2000x1024x1024: 16.1, 15.3, 9.7, 9.2, 128x128 11.2 us; 1000x3072x1024 +
// bias: 28.5, 27.4, 21.1, 15.6, 13.5 us.
enum SmallTile { kKs32x32, kKs64x32, kKs64x64w4, kKs64x64w2, kDma128x64, kDma128x128 };
struct SmallPlan {
  SmallTile tile;
  double us;
};
static SmallPlan pick_small_tile(int64_t M, const OutCols &cols, int64_t K, bool swiglu, bool dma_ok, int cus) {
  struct Cand { SmallTile id; int bm, bn, per_cu; double one, full; };
  const Cand cands[] = {{kKs32x32, 32, 32, 2, 1.25, 2.6},   {kKs64x32, 64, 32, 1, 1.95, 2.6},
                        {kKs64x64w4, 64, 64, 1, 3.6, 4.2},  {kKs64x64w2, 64, 64, 2, 4.5, 6.2},
                        {kDma128x64, 128, 64, 2, 6.2, 10.3}, {kDma128x128, 128, 128, 1, 9.4, 9.4}};
  SmallTile best = kKs64x64w4;
  double best_t = -1.0;
  for (const Cand &c : cands) {
    // SwiGLU needs whole [gate | up] 64-column pairs per wave
    if (swiglu && (c.bn < 64 || c.id == kDma128x64)) continue;
    if (!dma_ok && (c.id == kDma128x64 || c.id == kDma128x128)) continue;
    const int64_t tiles = ((M + c.bm - 1) / c.bm) * cols.tiles(c.bn);
    const int64_t round = (int64_t)cus * c.per_cu;
    const double t = tiles <= cus ? c.one : (double)((tiles + round - 1) / round) * c.full;
    if (best_t < 0 || t < best_t) best = c.id, best_t = t;
  }
  return {best, 3.0 + best_t * (double)K / 1024.0};
}

static int device_cus() {
  const int n = device_cu_count();
  return n > 0 ? n : 256;
}

template <typename T, int EPI, int ACT, int FM, int FN, int WM, int WN, int BK, int NST>
static void launch_dma(const void *A, int64_t lda, const void *B, int64_t ldb, void *C,
                       int64_t ldc, const void *bias, int64_t M, int64_t N, int64_t K,
                       hipStream_t st) {
  constexpr int BM = 32 * WM * FM, BN = 32 * WN * FN;
  const int64_t nb = ((M + BM - 1) / BM) * ((N + BN - 1) / BN);
  gemm_dma_kernel<T, EPI, ACT, FM, FN, NST, WM, WN, BK><<<dim3((unsigned)nb), dim3(64 * WM * WN), 0, st>>>(
      (const T *)A, lda, (const T *)B, ldb, (T *)C, ldc, (const T *)bias, (int)M, (int)N, (int)K);
}

template <typename T, int EPI, int ACT, int FM, int FN, int NW>
static void launch_ksplit(const void *A, int64_t lda, const void *B, int64_t ldb, void *C,
                          int64_t ldc, const void *bias, int64_t M, int64_t N, int64_t K,
                          hipStream_t st) {
  constexpr int BM = 32 * FM, BN = 32 * FN;
  const int64_t nb = ((M + BM - 1) / BM) * ((N + BN - 1) / BN);
  gemm_ksplit_kernel<T, EPI, ACT, FM, FN, NW><<<dim3((unsigned)nb), dim3(64 * NW), 0, st>>>(
      (const T *)A, lda, (const T *)B, ldb, (T *)C, ldc, (const T *)bias, (int)M, (int)N, (int)K);
}

// Fallback for K % 8 != 0 or unaligned operands: one thread per output.
template <typename T, int EPI, int ACT>
__global__ __launch_bounds__(256) void gemm_scalar_kernel(
    const T *__restrict__ A, int64_t lda, const T *__restrict__ B, int64_t ldb,
    T *__restrict__ C, int64_t ldc, const T *__restrict__ bias, int M, int NO, int K) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (int64_t)M * NO) return;
  const int m = (int)(t / NO), o = (int)(t % NO);
  const T *a = A + (int64_t)m * lda;
  if constexpr (EPI == kGSwiGLU) {
    const int64_t n0 = (o / 32) * 64 + (o % 32), n1 = n0 + 32;
    float g = 0.f, u = 0.f;
    for (int k = 0; k < K; ++k) {
      g += to_f32(a[k]) * to_f32(B[n0 * ldb + k]);
      u += to_f32(a[k]) * to_f32(B[n1 * ldb + k]);
    }
    const float s = to_f32(from_f32<T>(act_silu(to_f32(from_f32<T>(g)))));
    C[(int64_t)m * ldc + o] = from_f32<T>(s * to_f32(from_f32<T>(u)));
  } else {
    float v = 0.f;
    for (int k = 0; k < K; ++k) v += to_f32(a[k]) * to_f32(B[(int64_t)o * ldb + k]);
    if constexpr (EPI == kGBiasAct) {
      if (bias) v += to_f32(bias[o]);
      v = apply_act<ACT>(to_f32(from_f32<T>(v)));
    }
    C[(int64_t)m * ldc + o] = from_f32<T>(v);
  }
}

// hipBLASLt for plain GEMMs with at least one 256x256 tile per CU (gemm_lt.hip)
bool lt_gemm_wanted(int64_t M, int64_t N, int cus);
bool lt_gemm(const void *X, int64_t ldx, const void *W, int64_t ldw, void *Y, int64_t ldy,
             int64_t M, int64_t N, int64_t K, bool bf16, hipStream_t st);

template <typename T, int EPI, int ACT>
static int launch_gemm(const void *A, int64_t lda, const void *B, int64_t ldb, void *C,
                       int64_t ldc, const void *bias, int64_t M, int64_t N, int64_t K,
                       hipStream_t st, const char *name) {
  if (M == 0) return TPP_OK;
  const bool vec = (K % 8 == 0) && (lda % 8 == 0) && (ldb % 8 == 0) && aligned16(A) &&
                   aligned16(B);
  if constexpr (EPI == kGPlain) {
    if (vec && lt_gemm_wanted(M, N, device_cus()) &&
        lt_gemm(A, lda, B, ldb, C, ldc, M, N, K, __is_same(T, bf16), st))
      return check_launch(name);
  }
  const bool dma_ld = lda <= kDmaMaxLd && ldb <= kDmaMaxLd;
  if (vec && M * N >= (int64_t)kDmaMinMN && dma_ld) {
    if ((M + 127) / 128 * ((N + 127) / 128) > 0x7fffffffLL)
      return set_error(TPP_E_UNSUPPORTED, "%s: too many tiles", name);
    const int cus = device_cus();
    const bool persist = EPI != kGBiasAct && cus % 8 == 0;
    const bool tail = K % 64 != 0;
    const BigPlan pl = pick_dma_tile(M, {{N}, 1}, K, EPI == kGSwiGLU, persist && !tail, cus, true, tail);
    auto mixed = [&](int64_t big_rows, auto tl) {
      const int64_t small_rows = M > big_rows ? M - big_rows : 0;
      const int64_t nb = big_rows / 256 * ((N + 255) / 256) + (small_rows + 127) / 128 * ((N + 127) / 128);
      gemm_mixed_kernel<T, EPI, ACT, decltype(tl)::value><<<dim3((unsigned)nb), dim3(512), 0, st>>>(
          (const T *)A, lda, (const T *)B, ldb, (T *)C, ldc, (const T *)bias, (int)M, (int)N, (int)K,
          (int)big_rows);
    };
    if (tail) {
      mixed(pl.tile == kTileMixed ? pl.big_rows : pl.tile == kTile256x256 ? (M + 255) / 256 * 256 : 0,
            std::true_type{});
      return check_launch(name);
    }
    switch (pl.tile) {
    case kTile128x128: launch_dma<T, EPI, ACT, 1, 2, 4, 2, kSmallBK, 5>(A, lda, B, ldb, C, ldc, bias, M, N, K, st); break;
    case kTile128x192: launch_dma<T, EPI, ACT, 1, 3, 4, 2, kSmallBK, 4>(A, lda, B, ldb, C, ldc, bias, M, N, K, st); break;
    case kTile128x256: launch_dma<T, EPI, ACT, 1, 4, 4, 2, kSmallBK, 3>(A, lda, B, ldb, C, ldc, bias, M, N, K, st); break;
    case kTileMixed: mixed(pl.big_rows, std::false_type{}); break;
    case kTile256x256: {
      // more tiles than CUs: the persistent kernel (plain / SwiGLU epilogue)
      bool done = false;
      if constexpr (EPI != kGBiasAct) {
        const int64_t nb = ((M + 255) / 256) * ((N + 255) / 256);
        if (persist && nb > cus) {
          gemm_persist_kernel<T, EPI, ACT><<<dim3((unsigned)cus), dim3(512), 0, st>>>(
              (const T *)A, lda, (const T *)B, ldb, (T *)C, ldc, (const T *)bias, (int)M, (int)N, (int)K);
          done = true;
        }
      }
      if (!done) launch_dma<T, EPI, ACT, 2, 4, 4, 2, 64, 2>(A, lda, B, ldb, C, ldc, bias, M, N, K, st);
      break;
    }
    }
  } else if (vec && M * N < (int64_t)kDmaMinMN) {
    const bool dma_ok = K % 64 == 0 && dma_ld;
    switch (pick_small_tile(M, {{N}, 1}, K, EPI == kGSwiGLU, dma_ok, device_cus()).tile) {
    case kKs32x32:
      if constexpr (EPI != kGSwiGLU) launch_ksplit<T, EPI, ACT, 1, 1, 4>(A, lda, B, ldb, C, ldc, bias, M, N, K, st);
      break;
    case kKs64x32:
      if constexpr (EPI != kGSwiGLU) launch_ksplit<T, EPI, ACT, 2, 1, 4>(A, lda, B, ldb, C, ldc, bias, M, N, K, st);
      break;
    case kKs64x64w4: launch_ksplit<T, EPI, ACT, 2, 2, 4>(A, lda, B, ldb, C, ldc, bias, M, N, K, st); break;
    case kKs64x64w2: launch_ksplit<T, EPI, ACT, 2, 2, 2>(A, lda, B, ldb, C, ldc, bias, M, N, K, st); break;
    case kDma128x64:
      if constexpr (EPI != kGSwiGLU) launch_dma<T, EPI, ACT, 1, 1, 4, 2, kSmallBK, 3>(A, lda, B, ldb, C, ldc, bias, M, N, K, st);
      break;
    case kDma128x128: launch_dma<T, EPI, ACT, 1, 2, 4, 2, kSmallBK, 5>(A, lda, B, ldb, C, ldc, bias, M, N, K, st); break;
    }
  } else if (vec) {
    // row pitches past the DMA tiles' 32-bit offsets: the tile with 64-bit row addresses
    if ((M + 63) / 64 * ((N + 63) / 64) > 0x7fffffffLL)
      return set_error(TPP_E_UNSUPPORTED, "%s: too many tiles", name);
    launch_ksplit<T, EPI, ACT, 2, 2, 4>(A, lda, B, ldb, C, ldc, bias, M, N, K, st);
  } else {
    const int64_t NO = (EPI == kGSwiGLU) ? N / 2 : N;
    const int64_t blocks = (M * NO + 255) / 256;
    gemm_scalar_kernel<T, EPI, ACT><<<dim3((unsigned)blocks), dim3(256), 0, st>>>(
        (const T *)A, lda, (const T *)B, ldb, (T *)C, ldc, (const T *)bias, (int)M, (int)NO,
        (int)K);
  }
  return check_launch(name);
}

// Three projections of one input: one launch where the tile rules above
// expect it to take no longer than three (a weight whose 256x256 tiles fill the
// chip is faster by itself; near that line the two meet: three weights of [1024
// x 1024], us apart and in one, 3320 rows 38.4 and 29.9, 8192 rows 70.5 and
// 72.5).
struct Plan3 {
  bool one, big; // one launch; its tile is bp's, or sp's
  BigPlan bp;
  SmallPlan sp;
};
static Plan3 plan_gemm3(int64_t M, const int64_t *N, int64_t K, bool dma_ok, int cus) {
  const OutCols cols{{N[0], N[1], N[2]}, 3};
  Plan3 pl{true, M * (N[0] + N[1] + N[2]) >= (int64_t)kDmaMinMN, {kTile128x128, 0, 0.0}, {kKs64x64w4, 0.0}};
  if (pl.big && !dma_ok) pl.one = false;
  for (int i = 0; i < 3; ++i) pl.one = pl.one && ((M + 255) / 256) * ((N[i] + 255) / 256) < cus;
  if (!pl.one) return pl;
  if (pl.big) pl.bp = pick_dma_tile(M, cols, K, false, false, cus, false);
  else pl.sp = pick_small_tile(M, cols, K, false, dma_ok, cus);
  double apart = 0.0;
  for (int i = 0; i < 3; ++i)
    apart += M * N[i] >= (int64_t)kDmaMinMN ? pick_dma_tile(M, {{N[i]}, 1}, K, false, false, cus).us
                                            : pick_small_tile(M, {{N[i]}, 1}, K, false, dma_ok, cus).us;
  pl.one = (pl.big ? pl.bp.us : pl.sp.us) <= apart;
  return pl;
}

// y[i][M, N_i] = x . w[i]^T for three weights, as planned; three launches
// where the operands are not 16-byte aligned.
template <typename T>
static int launch_gemm3(const void *x, int64_t ldx, const void *const *w, void *const *y, int64_t M,
                        const int64_t *N, int64_t K, hipStream_t st, const char *name) {
  bool one = K % 8 == 0 && ldx % 8 == 0 && aligned16(x) && M > 0;
  for (int i = 0; i < 3; ++i) one = one && aligned16(w[i]);
  Plan3 pl{};
  if (one) pl = plan_gemm3(M, N, K, K % 64 == 0 && ldx <= kDmaMaxLd, device_cus());
  const bool big = pl.big;
  const BigPlan &bp = pl.bp;
  const SmallPlan &sp = pl.sp;
  if (!one || !pl.one) {
    for (int i = 0; i < 3; ++i)
      if (int e = launch_gemm<T, kGPlain, TPP_ACT_NONE>(x, ldx, w[i], K, y[i], N[i], nullptr, M, N[i], K, st, name))
        return e;
    return TPP_OK;
  }
  Group3 g;
  auto tiles = [&](int bm, int bn) {
    int64_t n = 0;
    for (int i = 0; i < 3; ++i) {
      g.B[i] = w[i], g.C[i] = y[i], g.N[i] = (int)N[i], g.nt[i] = (int)((N[i] + bn - 1) / bn);
      n += g.nt[i];
    }
    return dim3((unsigned)(n * ((M + bm - 1) / bm)));
  };
  const T *a = (const T *)x;
  if (big) {
    switch (bp.tile) {
    case kTile128x192:
      gemm_dma_group_kernel<T, 1, 3, 4, 4, 2><<<tiles(128, 192), dim3(512), 0, st>>>(a, ldx, g, (int)M, (int)K);
      break;
    case kTile128x256:
      gemm_dma_group_kernel<T, 1, 4, 3, 4, 2><<<tiles(128, 256), dim3(512), 0, st>>>(a, ldx, g, (int)M, (int)K);
      break;
    case kTile256x256:
      gemm_dma_group_kernel<T, 2, 4, 2, 4, 2><<<tiles(256, 256), dim3(512), 0, st>>>(a, ldx, g, (int)M, (int)K);
      break;
    default:
      gemm_dma_group_kernel<T, 1, 2, 5, 4, 2><<<tiles(128, 128), dim3(512), 0, st>>>(a, ldx, g, (int)M, (int)K);
      break;
    }
  } else {
    switch (sp.tile) {
    case kKs32x32: gemm_ksplit_group_kernel<T, 1, 1, 4><<<tiles(32, 32), dim3(256), 0, st>>>(a, ldx, g, (int)M, (int)K); break;
    case kKs64x32: gemm_ksplit_group_kernel<T, 2, 1, 4><<<tiles(64, 32), dim3(256), 0, st>>>(a, ldx, g, (int)M, (int)K); break;
    case kKs64x64w4: gemm_ksplit_group_kernel<T, 2, 2, 4><<<tiles(64, 64), dim3(256), 0, st>>>(a, ldx, g, (int)M, (int)K); break;
    case kKs64x64w2: gemm_ksplit_group_kernel<T, 2, 2, 2><<<tiles(64, 64), dim3(128), 0, st>>>(a, ldx, g, (int)M, (int)K); break;
    case kDma128x64:
      gemm_dma_group_kernel<T, 1, 1, 3, 4, 2><<<tiles(128, 64), dim3(512), 0, st>>>(a, ldx, g, (int)M, (int)K);
      break;
    case kDma128x128:
      gemm_dma_group_kernel<T, 1, 2, 5, 4, 2><<<tiles(128, 128), dim3(512), 0, st>>>(a, ldx, g, (int)M, (int)K);
      break;
    }
  }
  return check_launch(name);
}

static int gemm_args(const char *name, const void *x, const void *w, const void *y, int64_t M,
                     int64_t N, int64_t K, int64_t ldx) {
  if (!x || !w || !y) return set_error(TPP_E_INVALID, "%s: null pointer", name);
  if (M < 0 || N < 1 || K < 1)
    return set_error(TPP_E_INVALID, "%s: invalid shapes (M=%lld N=%lld K=%lld)", name,
                     (long long)M, (long long)N, (long long)K);
  if (M > 0x7fffffffLL || N > 0x7fffffffLL || K > 0x7fffffffLL)
    return set_error(TPP_E_UNSUPPORTED, "%s: dimension exceeds 2^31-1", name);
  if (ldx < K) return set_error(TPP_E_INVALID, "%s: ldx < K", name);
  return TPP_OK;
}

} // namespace tpp

using namespace tpp;

extern "C" int tpp_linear_act(const void *x, const void *w, const void *bias, void *y,
                              int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldy,
                              int act, int dtype, void *stream) {
  const char *name = "tpp_linear_act";
  if (int e = gemm_args(name, x, w, y, M, N, K, ldx)) return e;
  if (ldy < N) return set_error(TPP_E_INVALID, "%s: ldy < N", name);
  if (act < TPP_ACT_NONE || act > TPP_ACT_RELU)
    return set_error(TPP_E_INVALID, "%s: unknown activation %d", name, act);
  hipStream_t st = as_stream(stream);
  return TPP_DISPATCH_HALF(dtype, [&] {
    if (!bias && act == TPP_ACT_NONE)
      return launch_gemm<T, kGPlain, TPP_ACT_NONE>(x, ldx, w, K, y, ldy, nullptr, M, N, K, st,
                                                   name);
    switch (act) {
    case TPP_ACT_GELU_TANH:
      return launch_gemm<T, kGBiasAct, TPP_ACT_GELU_TANH>(x, ldx, w, K, y, ldy, bias, M, N, K,
                                                          st, name);
    case TPP_ACT_SILU:
      return launch_gemm<T, kGBiasAct, TPP_ACT_SILU>(x, ldx, w, K, y, ldy, bias, M, N, K, st,
                                                     name);
    case TPP_ACT_RELU:
      return launch_gemm<T, kGBiasAct, TPP_ACT_RELU>(x, ldx, w, K, y, ldy, bias, M, N, K, st,
                                                     name);
    default:
      return launch_gemm<T, kGBiasAct, TPP_ACT_NONE>(x, ldx, w, K, y, ldy, bias, M, N, K, st,
                                                     name);
    }
  });
}

extern "C" int tpp_linear3(const void *x, const void *const *w, void *const *y, int64_t M,
                           const int64_t *N, int64_t K, int64_t ldx, int dtype, void *stream) {
  const char *name = "tpp_linear3";
  if (!w || !y || !N) return set_error(TPP_E_INVALID, "%s: null pointer", name);
  for (int i = 0; i < 3; ++i)
    if (int e = gemm_args(name, x, w[i], y[i], M, N[i], K, ldx)) return e;
  hipStream_t st = as_stream(stream);
  return TPP_DISPATCH_HALF(dtype, [&] { return launch_gemm3<T>(x, ldx, w, y, M, N, K, st, name); });
}

extern "C" int tpp_linear_tiles(int64_t M, const int64_t *N, int outputs, int64_t K, int fused,
                                int swiglu, int32_t *tile) {
  const char *name = "tpp_linear_tiles";
  if (!N || !tile) return set_error(TPP_E_INVALID, "%s: null pointer argument", name);
  if (M < 1 || K < 8 || K % 8 != 0 || (outputs != 1 && outputs != 3) || (outputs == 3 && (fused || swiglu)))
    return set_error(TPP_E_INVALID, "%s: invalid shapes", name);
  for (int i = 0; i < outputs; ++i)
    if (N[i] < 1) return set_error(TPP_E_INVALID, "%s: invalid shapes", name);
  const int cus = device_cus();
  const bool tail = K % 64 != 0;
  bool big = M * N[0] >= (int64_t)kDmaMinMN;
  BigPlan bp{};
  SmallPlan sp{};
  tile[0] = tile[1] = tile[2] = tile[3] = 0;
  if (outputs == 3) {
    const Plan3 pl = plan_gemm3(M, N, K, !tail, cus);
    if (!pl.one) return TPP_OK;
    big = pl.big, bp = pl.bp, sp = pl.sp;
  } else {
    if (!fused && !swiglu && lt_gemm_wanted(M, N[0], cus)) return TPP_OK;
    if (big) bp = pick_dma_tile(M, {{N[0]}, 1}, K, swiglu, !fused && cus % 8 == 0 && !tail, cus, true, tail);
    else sp = pick_small_tile(M, {{N[0]}, 1}, K, swiglu, !tail, cus);
  }
  if (big) {
    const int bn[] = {128, 192, 256, 256, 128};
    tile[0] = bp.tile == kTile256x256 ? 256 : 128, tile[1] = bn[bp.tile], tile[3] = (int32_t)bp.big_rows;
  } else {
    const int bm[] = {32, 64, 64, 64, 128, 128}, bn[] = {32, 32, 64, 64, 64, 128}, nw[] = {4, 4, 4, 2, 0, 0};
    tile[0] = bm[sp.tile], tile[1] = bn[sp.tile], tile[2] = nw[sp.tile];
  }
  return TPP_OK;
}

extern "C" int tpp_linear_swiglu(const void *x, const void *w_gu, void *y, int64_t M,
                                 int64_t I, int64_t K, int64_t ldx, int64_t ldy, int dtype,
                                 void *stream) {
  const char *name = "tpp_linear_swiglu";
  if (int e = gemm_args(name, x, w_gu, y, M, 2 * I, K, ldx)) return e;
  if (I % 32 != 0)
    return set_error(TPP_E_UNSUPPORTED, "%s: intermediate size must be a multiple of 32", name);
  if (ldy < I) return set_error(TPP_E_INVALID, "%s: ldy < I", name);
  hipStream_t st = as_stream(stream);
  return TPP_DISPATCH_HALF(dtype, [&] {
    return launch_gemm<T, kGSwiGLU, TPP_ACT_NONE>(x, ldx, w_gu, K, y, ldy, nullptr, M, 2 * I,
                                                  K, st, name);
  });
}
