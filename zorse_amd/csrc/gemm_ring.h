// The small-tile MFMA GEMM for bf16 / fp16 and fp32, M, N and K off every grid
// but the 8 elements of a load or store (masked_takes in gemm.hip):
//
//   C[M, N] = op(A) op(B)^T (+ R[M, N])
//
// with the operand layouts and rounding of gemm_kernels.h.  It takes what the
// 256 x 256 pipeline is too coarse for: few tokens, widths off the 256 grid, token counts off every
// grid, and products whose large tiles would leave CUs idle.
//
// Workgroup = 4 waves in a 2 x 2 arrangement over a tile of 32 MB x 32 NB,
// each wave MB x NB blocks of v_mfma_f32_16x16x32; K advances by 64 (fp32:
// v_mfma_f32_16x16x4f32, by 32: the same 128 bytes per tile row).  Tiles
// reach LDS through buffer_load_dwordx4 ... lds.  B sits in a ring of RB
// stages and A in one of RB + 1, so loads run RB K steps ahead; operands are
// double-buffered in registers across the 32-deep substeps, and each K step
// has one barrier and one exact vmcnt wait, as in the large kernel.  With
// KS == 1 every output is summed as there (K ascending in steps of 32).  With
// KS == 2 eight waves share the tile, four on the even and four on the odd
// 32-deep substeps, and the two sums are added at the end: for grids that
// leave a CU one workgroup, where a single wave per SIMD waits out every
// barrier and LDS read.
//
// Ragged edges cost no branch in the loop: each operand's buffer resource
// ends at the operand's last element, and gfx950 writes zeros to LDS for
// lanes whose offset lies past it.  Rows past M or N (and, for a K-major
// operand, rows past K) are therefore zero, or other rows' data that only
// reaches outputs that are not stored; the columns of an NT tile past K are
// sent out of range lane by lane.  K steps past the end load zeros, so the
// loop needs no tail.
#pragma once
#include <type_traits>

#include "gemm_kernels.h"

namespace zk {
namespace gemm {

// Elements of one K step of a tile row (128 bytes).
template <typename T>
constexpr int kStep = 128 / static_cast<int>(sizeof(T));

// Swizzle of a K-major tile of COLS columns: k-row k's 16-byte chunk c sits at
// chunk position c ^ sw.  2-byte types (see kmaj_sw for 256 columns): the
// eight rows {k0 .. k0 + 3, k0 + 8 .. k0 + 11} that one transposed read of a
// 32-lane half touches go to eight different 32-byte groups of a 256-byte
// bank row.  128 columns: one row fills a bank row, as for 256.  64 columns:
// two rows share one (k & 1 picks the half), four chunk pairs remain.  fp32:
// an operand read takes one float of rows 4 (l / 16) + j, which land on four
// different 64-byte segments.
template <typename T, int COLS>
__device__ __forceinline__ int kmaj_sw_n(int k) {
  if (sizeof(T) == 4) return 4 * ((k >> 2) & 3);
  if (COLS >= 128) return 2 * ((k & 3) | ((k >> 1) & 4));
  return 2 * (((k >> 1) & 1) | ((k >> 2) & 2));
}

// One operand tile of ROWS outputs x 128 bytes of k and its loads by NW waves
// (4, or 8 for 2-byte types): ROWS / (8 NW) instructions per wave and K step.
template <typename T, int ROWS, bool KM, int NW>
struct RingTile {
  static constexpr int ES = sizeof(T);
  static constexpr int EL = ROWS * kStep<T>;         // elements of a stage
  static constexpr int NI = ROWS / 8 / NW;           // load instructions per wave
  static constexpr int RPI = 1024 / (ROWS * ES);     // K-major: k-rows per instruction
  static constexpr int LPR = ROWS * ES / 16;         // K-major: lanes per k-row
  uint32_t lane_off;  // bytes from the tile's first element
  int kcol;           // NT: this lane's first k of the tile
  int wave_by;        // LDS bytes before this wave's first instruction
  __device__ __forceinline__ void init(int64_t ld) {
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    if constexpr (KM) {
      // instruction i of wave w: k-rows kw + ki(i) .., kw from the wave and
      // ki(i) chosen so that a lane's swizzle is the same for every i
      const int kw = ES == 4 ? 4 * w : NW == 8 ? RPI * w : 8 * (w & 1) + 16 * (w >> 1);
      const int row = kw + lane / LPR;
      const int c = (lane % LPR) ^ kmaj_sw_n<T, ROWS>(row);
      lane_off = static_cast<uint32_t>(row * ld * ES + c * 16);
      wave_by = kw * ROWS * ES;
      kcol = 0;
    } else {
      const int row = tid >> 3;
      const int c = (tid & 7) ^ nt_sw(row);
      lane_off = static_cast<uint32_t>(row * ld * ES + c * 16);
      kcol = c * (16 / ES);
      wave_by = w * 1024;
    }
  }
  // first k-row (K-major) of instruction i, less the wave's
  static constexpr int ki(int i) {
    if (ES == 4) return ROWS == 128 ? 2 * (i & 1) + 16 * (i >> 1) : 16 * i;
    return NW == 4 && ROWS == 128 ? 4 * (i & 1) + 32 * (i >> 1) : 32 * i;
  }
  // instruction i of the stage at `lds` (byte address) from the resource r;
  // voff is lane_off or, past K, an offset out of range
  __device__ __forceinline__ void issue(uint32_t lds, v4i r, uint32_t voff, int64_t ld, int i) const {
    if constexpr (KM)
      dma16(r, voff, static_cast<uint32_t>(ki(i) * ld * ES), lds + wave_by + ki(i) * ROWS * ES);
    else
      dma16(r, voff, static_cast<uint32_t>(8 * NW * i * ld * ES), lds + wave_by + i * (1024 * NW));
  }
};

// One lane's operand of a 16-wide block and substep (half a K step): 8
// elements of consecutive k (2-byte types: one MFMA) or 4 (fp32: four MFMAs,
// element j at k = 4 (l / 16) + j in both operands).
template <typename T>
struct RingOp {
  typedef typename Mfma<T>::vec8 vec;
  static __device__ __forceinline__ f32x4 mma(vec a, vec b, f32x4 c) { return Mfma<T>::mma16(a, b, c); }
};
template <>
struct RingOp<float> {
  typedef f32x4 vec;
  static __device__ __forceinline__ f32x4 mma(vec a, vec b, f32x4 c) {
#pragma unroll
    for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[j], c, 0, 0, 0);
    return c;
  }
};

// LDS element offset of this lane's first K-major read for the 16-column block
// at colw (see kmaj_base); block r is at that ^ 16 r, substep 1 half a tile on.
template <typename T, int COLS>
__device__ __forceinline__ int kmaj_base_n(int colw) {
  const int lane = threadIdx.x & 63;
  if constexpr (sizeof(T) == 4) {
    const int k = 4 * (lane >> 4), col = colw + (lane & 15);
    return k * COLS + (((col >> 2) ^ kmaj_sw_n<T, COLS>(k)) << 2) + (col & 3);
  } else {
    const int k = 8 * (lane >> 4) + ((lane & 15) >> 2);
    const int col = colw + 4 * (lane & 3);
    return k * COLS + (((col >> 3) ^ kmaj_sw_n<T, COLS>(k)) << 3) + (col & 7);
  }
}
template <typename T, int COLS>
__device__ __forceinline__ typename RingOp<T>::vec kmaj_operand_n(const T* tile, int off) {
  if constexpr (sizeof(T) == 4) {
    const T* p = tile + off;
    return f32x4{p[0], p[COLS], p[2 * COLS], p[3 * COLS]};
  } else {
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
    const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(tile + off));
    const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(tile + off + 4 * COLS));
    return __builtin_bit_cast(typename RingOp<T>::vec,
                              __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
  }
}

// EPI as for gemm_tiled_kernel: 0 plain (+ residual), 1 SwiGLU (the B tile's
// first half gate rows, its second half up rows of the same features; silu in
// the IEEE form of the SwiGLU kernel), 2 RoPE on the columns below rcols
// (whole heads of 2 rhalf columns, which divide the tile's width).
template <typename T, int EPI, bool AKM, bool BKM, int MB, int NB, int RB, int WPE, int KS>
__global__ __launch_bounds__(256 * KS) __attribute__((amdgpu_waves_per_eu(WPE, WPE)))
void gemm_ring_kernel(GemmArgs args) {
  static_assert(EPI == 0 || (EPI == 3 && !AKM) || (!AKM && !BKM),
                "the SwiGLU and RoPE epilogues take NT operands");
  constexpr int TBM = 32 * MB, TBN = 32 * NB, WR = 16 * MB, WC = 16 * NB;
  typedef RingOp<T> Mm;
  typedef typename Mm::vec V8;
  constexpr int NT = 256 * KS, ES = sizeof(T), BK = kStep<T>;
  static_assert(ES == 2 || (EPI == 0 && KS == 1), "fp32: plain epilogue");
  typedef RingTile<T, TBM, AKM, 4 * KS> TA;
  typedef RingTile<T, TBN, BKM, 4 * KS> TB;
  constexpr int RA = KS == 1 ? RB + 1 : RB;  // A stages
  constexpr int LDS_EL = RA * TA::EL + RB * TB::EL;
  constexpr int EP = TBN + 4;  // pitch of the epilogue's fp32 tile
  static_assert(TBM * EP * 4 <= LDS_EL * ES, "the epilogue tile lies in the rings");
  __shared__ __attribute__((aligned(16))) T lds[LDS_EL];
  T* const As = lds;
  T* const Bs = lds + RA * TA::EL;

  const int64_t lda = args.lda, ldb = args.ldb;
  // EPI 3: the blockIdx.y-th split_k of the reduction, into C + blockIdx.y M N
  const int64_t k_first = EPI == 3 ? blockIdx.y * args.split_k : 0;
  const int64_t k_left = args.K - k_first;
  const int64_t M = args.M, N = args.N, K = EPI == 3 && args.split_k < k_left ? args.split_k : k_left;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, q4 = lane >> 4;
  const int wm = (wave >> 1) & 1, wn = wave & 1;
  // tiles in groups of GROUP_M along M, consecutive tiles on one XCD
  const int64_t n_m = (M + TBM - 1) / TBM, n_n = (N + TBN - 1) / TBN;
  const int64_t pid = xcd_order(blockIdx.x, n_m * n_n);
  const int64_t per_group = static_cast<int64_t>(GROUP_M) * n_n;
  const int64_t grp = pid / per_group;
  const int64_t mf = grp * GROUP_M;
  const int64_t gm = n_m - mf < GROUP_M ? n_m - mf : GROUP_M;
  const int64_t in_grp = pid - grp * per_group;
  const int64_t m0 = (mf + in_grp % gm) * TBM, n0 = (in_grp / gm) * TBN;
  const int64_t f0 = n0 / 2;  // EPI 1: the tile's first feature

  // first element of each operand's tile, bytes left from there to the
  // operand's end, and the bytes of one K step
  const char* Ab = static_cast<const char*>(args.a) +
                   ES * (AKM ? m0 + k_first * lda : m0 * lda + k_first);
  const int64_t a_left = ES * (AKM ? (K - 1) * lda + M - m0 : (M - 1 - m0) * lda + K);
  const int64_t a_step = AKM ? ES * BK * lda : ES * BK;
  const int64_t b_rows = EPI == 1 ? N / 2 : N, b_r0 = EPI == 1 ? f0 : n0;
  const char* Bb = static_cast<const char*>(args.b) +
                   ES * (BKM ? b_r0 + k_first * ldb : b_r0 * ldb + k_first);
  const char* B2b = EPI == 1 ? static_cast<const char*>(args.b2) + ES * b_r0 * ldb : nullptr;
  const int64_t b_left = ES * (BKM ? (K - 1) * ldb + b_rows - b_r0 : (b_rows - 1 - b_r0) * ldb + K);
  const int64_t b_step = BKM ? ES * BK * ldb : ES * BK;

  TA ta;
  TB tb;
  ta.init(lda);
  static_assert(EPI != 1 || TB::NI % 2 == 0, "gate and up rows: instructions of their own");
  tb.init(ldb);
  const uint32_t lds_a = lds_addr(As), lds_b = lds_addr(Bs);
  f32x4 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = f32x4{};

  int abase[2], bbase[2];  // operand read bases of the two substeps (elements)
  if constexpr (AKM) {
    abase[0] = kmaj_base_n<T, TBM>(wm * WR);
    abase[1] = abase[0] + BK / 2 * TBM;
  } else {
    abase[0] = nt_off(wm * WR + l16, 8 * q4) * 2 / ES;
    abase[1] = abase[0] ^ (64 / ES);
  }
  if constexpr (BKM) {
    bbase[0] = kmaj_base_n<T, TBN>(wn * WC);
    bbase[1] = bbase[0] + BK / 2 * TBN;
  } else if constexpr (EPI == 1) {
    // wave half wn: features WC / 2 wn .. of the gate rows, then of the up
    // rows (block j < NB / 2: gate, else up), so that a wave's blocks j and
    // j + NB / 2 are g and u of one element
    bbase[0] = nt_off(wn * (WC / 2) + l16, 8 * q4);
    bbase[1] = bbase[0] ^ 32;
  } else {
    bbase[0] = nt_off(wn * WC + l16, 8 * q4) * 2 / ES;
    bbase[1] = bbase[0] ^ (64 / ES);
  }
  V8 xa[2][MB], xb[2][NB];
  // operand piece r (A row blocks, then B row blocks) of substep s, stages sa / sb
  auto rd_piece = [&](int sa, int sb, int s, int r) __attribute__((always_inline)) {
    if (r < MB) {
      const T* t = As + sa * TA::EL;
      if constexpr (AKM)
        xa[s][r] = kmaj_operand_n<T, TBM>(t, abase[s] ^ (16 * r));
      else
        xa[s][r] = *reinterpret_cast<const V8*>(t + abase[s] + 16 * BK * r);
    } else {
      const int j = r - MB;
      const T* t = Bs + sb * TB::EL;
      if constexpr (BKM)
        xb[s][j] = kmaj_operand_n<T, TBN>(t, bbase[s] ^ (16 * j));
      else if constexpr (EPI == 1)
        xb[s][j] = *reinterpret_cast<const V8*>(
            t + bbase[s] + 1024 * (j % (NB / 2)) + (j / (NB / 2)) * (TBN / 2) * BK);
      else
        xb[s][j] = *reinterpret_cast<const V8*>(t + bbase[s] + 16 * BK * j);
    }
  };
  // loads of K step k (k0 = 64 k): resource of the step, lane offset
  struct Src {
    v4i r, r2;
    uint32_t voff;
  };
  auto a_src = [&](int64_t k) __attribute__((always_inline)) {
    Src s;
    s.r = rsrc_left(Ab + k * a_step, a_left - k * a_step);
    s.voff = AKM || k * BK + ta.kcol < K ? ta.lane_off : 0x80000000u;
    return s;
  };
  auto b_src = [&](int64_t k) __attribute__((always_inline)) {
    Src s;
    s.r = rsrc_left(Bb + k * b_step, b_left - k * b_step);
    if constexpr (EPI == 1) s.r2 = rsrc_left(B2b + k * b_step, b_left - k * b_step);
    s.voff = BKM || k * BK + tb.kcol < K ? tb.lane_off : 0x80000000u;
    return s;
  };
  auto load_a = [&](const Src& s, int st, int i) __attribute__((always_inline)) {
    ta.issue(lds_a + st * (ES * TA::EL), s.r, s.voff, lda, i);
  };
  auto load_b = [&](const Src& s, int st, int i) __attribute__((always_inline)) {
    if constexpr (EPI == 1) {
      // pieces of the first half: gate rows 32 i .., of the second: up rows
      if (i < TB::NI / 2)
        tb.issue(lds_b + st * (ES * TB::EL), s.r, s.voff, ldb, i);
      else
        dma16(s.r2, s.voff, static_cast<uint32_t>(32 * KS * (i - TB::NI / 2) * ldb * 2),
              lds_b + st * (ES * TB::EL) + tb.wave_by + i * (4096 * KS));
    } else {
      tb.issue(lds_b + st * (ES * TB::EL), s.r, s.voff, ldb, i);
    }
  };
  // The MB NB MFMAs of set q, row by row; after row c its share of the loads
  // (lk 1: A of step k into stage lst, 2: B) and, when rd, of the reads of
  // substep s0 in the order its MFMAs use them (A0, all of B, the other A).
  auto mm = [&](int q, int lk, int lst, int64_t k, bool rd, int ra, int rb,
                int s0) __attribute__((always_inline)) {
    Src src;
    if (lk == 1) src = a_src(k);
    if (lk == 2) src = b_src(k);
#pragma unroll
    for (int c = 0; c < MB; ++c) {
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[c][j] = Mm::mma(xa[q][c], xb[q][j], acc[c][j]);
      if (rd) {
#pragma unroll
        for (int u = c * (MB + NB) / MB; u < (c + 1) * (MB + NB) / MB; ++u)
          rd_piece(ra, rb, s0, u == 0 ? 0 : u <= NB ? MB + u - 1 : u - NB);
      }
      if (lk == 1) load_a(src, lst, c);
      if (lk == 2) {
#pragma unroll
        for (int u = c * NB / MB; u < (c + 1) * NB / MB; ++u) load_b(src, lst, u);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  const int64_t n_k = (K + BK - 1) / BK;
#pragma unroll
  for (int p = 0; p < RB; ++p) {
    const Src sa = a_src(p), sb = b_src(p);
#pragma unroll
    for (int i = 0; i < TA::NI; ++i) load_a(sa, p, i);
#pragma unroll
    for (int i = 0; i < TB::NI; ++i) load_b(sb, p, i);
  }
  if constexpr (KS == 1) {
    wait_vmcnt<(RB - 1) * (TA::NI + TB::NI)>();  // step 0 landed
    __syncthreads();
#pragma unroll
    for (int r = 0; r < MB + NB; ++r) rd_piece(0, 0, 0, r);
    int sa = 0, sb = 0;  // stages of step t
    for (int64_t t = 0;; ++t) {
      // substep 0 with A(t + RB) into the stage that step t - 1 left
      mm(0, 1, sa == 0 ? RB : sa - 1, t + RB, true, sa, sb, 1);
      if (t + 1 >= n_k) break;
      const int sa1 = sa == RB ? 0 : sa + 1, sb1 = sb == RB - 1 ? 0 : sb + 1;
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this step's reads done
      wait_vmcnt<(RB - 1) * TA::NI + (RB - 2) * TB::NI>();  // A, B of step t + 1 landed
      __syncthreads();
      // substep 1 with B(t + RB) into step t's stage, and step t + 1's reads
      mm(1, 2, sb, t + RB, true, sa1, sb1, 0);
      sa = sa1;
      sb = sb1;
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);
    mm(1, 0, 0, 0, false, 0, 0, 0);

  } else {
    // Two groups of four waves, one per 32-deep substep of a K step, each over
    // the whole tile; their sums meet in LDS below.  Step t: barrier (step
    // t + 1 landed everywhere, step t's reads done), then set t % 2 with the
    // reads of step t + 1 into the other set and the loads of step t + RB into
    // the stage step t leaves.
    constexpr int NL = TA::NI + TB::NI;
    const int grp2 = __builtin_amdgcn_readfirstlane(tid >> 8);
    const int ab = grp2 ? abase[1] : abase[0], bb = grp2 ? bbase[1] : bbase[0];
    abase[0] = abase[1] = ab;
    bbase[0] = bbase[1] = bb;
    wait_vmcnt<(RB - 1) * NL>();  // step 0 landed
    __syncthreads();
#pragma unroll
    for (int r = 0; r < MB + NB; ++r) rd_piece(0, 0, 0, r);
    int st = 0;
    auto step = [&](auto set_tag, int64_t t) __attribute__((always_inline)) {
      constexpr int q = decltype(set_tag)::value;
      const int st1 = st == RB - 1 ? 0 : st + 1;
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this step's reads done
      wait_vmcnt<(RB - 2) * NL>();         // step t + 1 landed
      __syncthreads();
      const Src sa = a_src(t + RB), sb = b_src(t + RB);
#pragma unroll
      for (int c = 0; c < MB; ++c) {
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[c][j] = Mm::mma(xa[q][c], xb[q][j], acc[c][j]);
#pragma unroll
        for (int u = c * (MB + NB) / MB; u < (c + 1) * (MB + NB) / MB; ++u)
          rd_piece(st1, st1, q ^ 1, u == 0 ? 0 : u <= NB ? MB + u - 1 : u - NB);
#pragma unroll
        for (int u = c * NL / MB; u < (c + 1) * NL / MB; ++u) {
          if (u < TA::NI)
            load_a(sa, st, u);
          else
            load_b(sb, st, u - TA::NI);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      st = st1;
    };
    int64_t t = 0;
    for (; t + 1 < n_k; t += 2) {
      step(std::integral_constant<int, 0>{}, t);
      step(std::integral_constant<int, 1>{}, t + 1);
    }
    if (t < n_k) step(std::integral_constant<int, 0>{}, t);
    __builtin_amdgcn_s_waitcnt(0xC07F);
  }

  // Epilogue: the tile in fp32 through LDS, then 8-column chunks per thread.
  // acc[i][j][e] is row 16 i + 4 (l / 16) + e, column 16 j + l % 16.
  wait_vmcnt<0>();  // the zero-filling loads past the last step
  __syncthreads();
  float* ws = reinterpret_cast<float*>(lds);
  auto stage = [&](bool add) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int col = EPI == 1 ? (j / (NB / 2)) * (TBN / 2) + wn * (WC / 2) + 16 * (j % (NB / 2))
                                   : wn * WC + 16 * j;
          float* p = &ws[(wm * WR + 16 * i + 4 * q4 + e) * EP + col + l16];
          *p = add ? acc[i][j][e] + *p : acc[i][j][e];
        }
  };
  if constexpr (KS == 2) {
    if (wave >= 4) stage(false);
    __syncthreads();
    if (wave < 4) stage(true);
  } else {
    stage(false);
  }
  __syncthreads();
  typedef T T8 __attribute__((ext_vector_type(8)));
  auto chunk = [&](int row, int col, float (&v)[8]) __attribute__((always_inline)) {
    const float4 lo = *reinterpret_cast<const float4*>(&ws[row * EP + col]);
    const float4 hi = *reinterpret_cast<const float4*>(&ws[row * EP + col + 4]);
    v[0] = lo.x; v[1] = lo.y; v[2] = lo.z; v[3] = lo.w;
    v[4] = hi.x; v[5] = hi.y; v[6] = hi.z; v[7] = hi.w;
  };
  T* const C = static_cast<T*>(args.c);
  if constexpr (EPI == 1) {
    T* const U = static_cast<T*>(args.c2);
    T* const Z = static_cast<T*>(args.z);
    constexpr int CPR = TBN / 16;  // feature chunks per row
    constexpr int NIT = TBM * CPR / NT;
    T8 zo[NIT];
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      const int id = it * NT + tid, row = id / CPR, ch = id % CPR;
      float g[8], u[8];
      chunk(row, 8 * ch, g);
      chunk(row, TBN / 2 + 8 * ch, u);
      T8 go, uo;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        go[e] = static_cast<T>(g[e]);
        uo[e] = static_cast<T>(u[e]);
        const float gv = to_f32(go[e]);
        zo[it][e] = static_cast<T>(round_to<T>(gv / (1.0f + expf(-gv))) * to_f32(uo[e]));
      }
      const int64_t gr = m0 + row, gf = f0 + 8 * ch;
      if (gr < M && gf < b_rows) {
        *reinterpret_cast<T8*>(C + gr * args.ldc + gf) = go;
        *reinterpret_cast<T8*>(U + gr * args.ldc + gf) = uo;
        *reinterpret_cast<T8*>(Z + gr * args.ldz + gf) = zo[it];
      }
    }
    if (args.zt != nullptr) {
      // z^T through an LDS tile [features][TBM tokens] (the host asks for M % 8 == 0)
      constexpr int ZP = TBM + 8;
      T* zs = lds;
      __syncthreads();
#pragma unroll
      for (int it = 0; it < NIT; ++it) {
        const int id = it * NT + tid, row = id / CPR, ch = id % CPR;
#pragma unroll
        for (int e = 0; e < 8; ++e) zs[(8 * ch + e) * ZP + row] = zo[it][e];
      }
      __syncthreads();
      T* const ZT = static_cast<T*>(args.zt);
      constexpr int RC = TBM / 8;
#pragma unroll
      for (int it = 0; it < TBN / 2 * RC / NT; ++it) {
        const int id = it * NT + tid, f = id / RC, tc = id % RC;
        if (f0 + f < b_rows && m0 + 8 * tc < M)
          *reinterpret_cast<T8*>(ZT + (f0 + f) * args.ldzt + m0 + 8 * tc) =
              *reinterpret_cast<const T8*>(&zs[f * ZP + 8 * tc]);
      }
    }
  } else {
    constexpr int CPR = TBN / 8;
    const T* const R = static_cast<const T*>(args.r);
#pragma unroll
    for (int it = 0; it < TBM * CPR / NT; ++it) {
      const int id = it * NT + tid, row = id / CPR, ch = id % CPR;
      const int64_t gr = m0 + row, gc = n0 + 8 * ch;
      if (gr >= M || gc >= N) continue;
      float v[8];
      chunk(row, 8 * ch, v);
      if constexpr (EPI == 3) {
        Vec8<float>::store(static_cast<float*>(args.c) + (blockIdx.y * M + gr) * N + gc, v);
        continue;
      }
      if constexpr (EPI == 2) if (gc < args.rcols) {
        // this chunk rotated: its pair is the chunk rhalf columns away in the
        // same head (half-split) or inside the chunk (interleaved); the
        // product is rounded to T first, as the RoPE pass would read it
        const int s = static_cast<int>(static_cast<uint32_t>(gr) % static_cast<uint32_t>(args.rS));
        int64_t pos = args.rpos != nullptr ? args.rpos[s] : s;
        pos = pos < 0 ? 0 : pos > args.rnpos - 1 ? args.rnpos - 1 : pos;
        const int hc = static_cast<int>(gc) & (2 * args.rhalf - 1);  // column in the head
        const float* cp = args.rcos + pos * args.rhalf;
        const float* sp = args.rsin + pos * args.rhalf;
        if (args.rpair == ZK_ROPE_HALF) {
          const bool second = hc >= args.rhalf;
          const int i0 = second ? hc - args.rhalf : hc;
          float w[8], cs[8], sn[8];
          chunk(row, second ? 8 * ch - args.rhalf : 8 * ch + args.rhalf, w);
          Vec8<float>::load(cp + i0, cs);
          Vec8<float>::load(sp + i0, sn);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float x1 = round_to<T>(second ? w[e] : v[e]), x2 = round_to<T>(second ? v[e] : w[e]);
            float y1, y2;
            rotate_pair<T, ZK_ROPE_HALF, false>(x1, x2, cs[e], sn[e], y1, y2);
            v[e] = second ? y2 : y1;
          }
        } else {
          const float4 c4 = *reinterpret_cast<const float4*>(cp + hc / 2);
          const float4 s4 = *reinterpret_cast<const float4*>(sp + hc / 2);
          const float cs[4] = {c4.x, c4.y, c4.z, c4.w}, sn[4] = {s4.x, s4.y, s4.z, s4.w};
          T8 o;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float x1 = round_to<T>(v[2 * e]), x2 = round_to<T>(v[2 * e + 1]);
            float y1, y2;
            rotate_pair<T, ZK_ROPE_INTERLEAVED, false>(x1, x2, cs[e], sn[e], y1, y2);
            // converted here, next to the fma, as the RoPE pass does: for fp16
            // the compiler makes one rounding of the two (v_fma_mix)
            o[2 * e] = static_cast<T>(y1);
            o[2 * e + 1] = static_cast<T>(y2);
          }
          *reinterpret_cast<T8*>(C + gr * args.ldc + gc) = o;
          continue;
        }
      }
      if (EPI == 0 && R != nullptr) {
        float rv[8];
        Vec8<T>::load(R + gr * args.ldr + gc, rv);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] += rv[e];
      }
      Vec8<T>::store(C + gr * args.ldc + gc, v);
    }
  }
}

}  // namespace gemm
}  // namespace zk
