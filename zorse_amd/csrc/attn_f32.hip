// Attention for fp32 layers, forward and backward, on the fp32 matrix cores
// (v_mfma_f32_16x16x4f32: full fp32 products and sums), any head dim up to
// 128 (zero-padded to D = 64 or 128 in registers and LDS).
//
// Workgroup = 4 waves, 16 queries (forward, dQ) or 16 keys (dK / dV) per
// wave; the other side streams through LDS in tiles of 32 rows, the next
// tile's global loads in flight in registers during the current one's math.
// The arrangement is the 16-bit kernels' (attn_fwd.hip, attn_bwd.hip): scores
// transposed in the forward and dQ (a lane owns one query and 4 keys of each
// 16-key block, so the softmax is per lane plus two exchanges), probabilities
// straight from the accumulators into the next product's operand, dQ by its
// own pass, nothing accumulated through memory.
//
// Operands.  The MFMA takes one float per lane: row (or column) l % 16 and k
// index l / 16.  Both operands of a product may permute k alike, so a 16-byte
// LDS read of elements 16 c + 4 (l / 16) .. + 3 serves four MFMAs; and the
// accumulator's rows 4 (l / 16) + e make operand e of the product that
// consumes them, whose other operand reads those rows' elements.  LDS rows
// are padded to D + 4 floats: both read patterns spread over the banks.
//
// Bound by latency at the sizes fp32 layers have (the parity layer's shape, 2
// sequences x 4 heads x 128 x 64, is 16 workgroups).  There a thread per row
// took 1770 us forward, 1955 us for dQ and 1976 us for dK / dV; these kernels
// take 16, 26 and 31 us.  Many sequences of a few tokens are a thread per row's
// still (by_rows).
#include "attn_common.h"
#include "vec.h"

namespace zk {

namespace {

constexpr int kTile = 32;  // rows per LDS tile

// Rows r0 .. r0 + 31 (of `rows`) of a [.., d] tensor, D / 8 floats per
// thread: load() issues the global loads, store() writes the LDS tile.
template <int D, bool kVec>
struct TileReg {
  static constexpr int NC = kTile * D / 4 / 256;  // 4-float chunks per thread
  float4 v[NC];
  __device__ __forceinline__ void load(const float* base, int64_t ld, int64_t r0, int64_t rows, int d) {
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int id = i * 256 + static_cast<int>(threadIdx.x);
      const int r = id / (D / 4), c = 4 * (id % (D / 4));
      float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
      if (r0 + r < rows && c < d) {
        const float* p = base + (r0 + r) * ld + c;
        if (kVec) {
          x = *reinterpret_cast<const float4*>(p);
        } else {
          x.x = p[0];
          if (c + 1 < d) x.y = p[1];
          if (c + 2 < d) x.z = p[2];
          if (c + 3 < d) x.w = p[3];
        }
      }
      v[i] = x;
    }
  }
  // returns whether one of this thread's values is an infinity or NaN
  __device__ __forceinline__ int store(float* tile) const {
    float z = 0.f;  // stays 0 for finite values, else NaN
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int id = i * 256 + static_cast<int>(threadIdx.x);
      *reinterpret_cast<float4*>(&tile[(id / (D / 4)) * (D + 4) + 4 * (id % (D / 4))]) = v[i];
      z += 0.f * v[i].x + 0.f * v[i].y + 0.f * v[i].z + 0.f * v[i].w;
    }
    return z != 0.f;
  }
};

// This lane's operand of row `row` (null: zeros): elements 16 c + 4 q4 .. + 3.
template <int D, bool kVec>
__device__ __forceinline__ void load_row(float4 (&x)[D / 16], const float* row, int d) {
  const int q4 = (threadIdx.x & 63) >> 4;
#pragma unroll
  for (int c = 0; c < D / 16; ++c) {
    const int e = 16 * c + 4 * q4;
    x[c] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (row == nullptr || e >= d) continue;
    if (kVec) {
      x[c] = *reinterpret_cast<const float4*>(row + e);
    } else {
      x[c].x = row[e];
      if (e + 1 < d) x[c].y = row[e + 1];
      if (e + 2 < d) x[c].z = row[e + 2];
      if (e + 3 < d) x[c].w = row[e + 3];
    }
  }
}

__device__ __forceinline__ f32x4 mma4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// X Y^T over d of the LDS rows row0 .. + 15 (X) and this lane's operand y.
template <int D>
__device__ __forceinline__ f32x4 dot_rows(const float* tile, int row0, const float4 (&y)[D / 16]) {
  const int l16 = threadIdx.x & 15, q4 = (threadIdx.x & 63) >> 4;
  const float* p = tile + (row0 + l16) * (D + 4) + 4 * q4;
  f32x4 s{};
#pragma unroll
  for (int c = 0; c < D / 16; ++c) {
    const float4 x = *reinterpret_cast<const float4*>(p + 16 * c);
    s = mma4(x.x, y[c].x, s);
    s = mma4(x.y, y[c].y, s);
    s = mma4(x.z, y[c].z, s);
    s = mma4(x.w, y[c].w, s);
  }
  return s;
}

// acc^T += X^T w over the 16 LDS rows row0 ..: w[e] belongs to row 4 q4 + e.
template <int D>
__device__ __forceinline__ void add_rows(f32x4 (&acc)[D / 16], const float* tile, int row0,
                                         const f32x4& w) {
  const int l16 = threadIdx.x & 15, q4 = (threadIdx.x & 63) >> 4;
  const float* p = tile + (row0 + 4 * q4) * (D + 4) + l16;
#pragma unroll
  for (int e = 0; e < 4; ++e)
#pragma unroll
    for (int nt = 0; nt < D / 16; ++nt)
      acc[nt] = mma4(p[e * (D + 4) + 16 * nt], w[e], acc[nt]);
}

// The same for a tile that holds an infinity or NaN, where a product with the
// zero weight of a masked row would be NaN: row by row, masked rows left out.
template <int D, typename Vis>
__device__ __forceinline__ void add_rows_visible(f32x4 (&acc)[D / 16], const float* tile, int row0,
                                              const f32x4& w, Vis visible) {
  const int l16 = threadIdx.x & 15, q4 = (threadIdx.x & 63) >> 4;
  for (int r = 0; r < 16; ++r) {
    float wr = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) wr = (r & 3) == e ? w[e] : wr;
    wr = __shfl(wr, (r >> 2) * 16 + l16, 64);
    if (!visible(row0 + r)) continue;
#pragma unroll
    for (int nt = 0; nt < D / 16; ++nt)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        acc[nt][e] = fmaf(wr, tile[(row0 + r) * (D + 4) + 16 * nt + 4 * q4 + e], acc[nt][e]);
  }
}

// sum / max over the four lane groups that share a column
__device__ __forceinline__ float group_sum(float x) {
  x += __shfl_xor(x, 16, 64);
  return x + __shfl_xor(x, 32, 64);
}
__device__ __forceinline__ float group_max(float x) {
  x = fmaxf(x, __shfl_xor(x, 16, 64));
  return fmaxf(x, __shfl_xor(x, 32, 64));
}

// This lane's accumulators (elements 16 nt + 4 q4 + e of its row), scaled, to
// the row at dst.
template <int D, bool kVec>
__device__ __forceinline__ void store_row(float* dst, const f32x4 (&x)[D / 16], float scale, int d) {
  const int q4 = (threadIdx.x & 63) >> 4;
#pragma unroll
  for (int nt = 0; nt < D / 16; ++nt) {
    const int e0 = 16 * nt + 4 * q4;
    if (kVec) {
      if (e0 < d)
        *reinterpret_cast<float4*>(dst + e0) = make_float4(x[nt][0] * scale, x[nt][1] * scale,
                                                           x[nt][2] * scale, x[nt][3] * scale);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (e0 + e < d) dst[e0 + e] = x[nt][e] * scale;
    }
  }
}

// The transpose of the RoPE rotation on one row of a tensor just stored
// (gradients of queries / keys the forward rotated), by the 16-lane column's
// four lanes after a barrier (lanes first, first + step, ..): pairs
// (i, i + d / 2) or (2 i, 2 i + 1), the formula of rope_inverse_regs.
__device__ __forceinline__ void rope_inverse_row(float* x, const AttnArgs& a, int64_t row,
                                                 int first, int step) {
  int64_t pos = a.rope_pos != nullptr ? a.rope_pos[row] : row;
  if (pos < 0) pos = 0;
  if (pos > a.rope_npos - 1) pos = a.rope_npos - 1;
  const int half = static_cast<int>(a.d / 2);
  const float* ct = a.rope_cos + pos * half;
  const float* st = a.rope_sin + pos * half;
  for (int i = first; i < half; i += step) {
    const int ia = a.rope_interleaved ? 2 * i : i;
    const int ib = a.rope_interleaved ? 2 * i + 1 : i + half;
    const float u = x[ia], w = x[ib];
    x[ia] = fmaf(u, ct[i], w * st[i]);
    x[ib] = fmaf(w, ct[i], -u * st[i]);
  }
}

// Rows of the other side that rows r0 .. r0 + n - 1 of one side meet, as a
// tile range [lo, hi): keys for queries (kKeys) or queries for keys.
template <bool kKeys>
__device__ __forceinline__ void tile_range(const AttnArgs& a, int64_t r0, int64_t n, int64_t& lo,
                                           int64_t& hi) {
  lo = 0;
  hi = kKeys ? a.Skv : a.Sq;
  if (kKeys) {
    if (a.causal && hi > r0 + n) hi = r0 + n;
    if (a.window > 0 && r0 - a.window + 1 > lo) lo = r0 - a.window + 1;
  } else {
    if (a.causal) lo = r0;
    if (a.window > 0 && r0 + n - 1 + a.window < hi) hi = r0 + n - 1 + a.window;
  }
  lo /= kTile;
  hi = hi > lo * kTile ? (hi + kTile - 1) / kTile : lo;
}

// A launch holds fewer than 2^32 threads along x: workgroup n of any number is
// (n % kGridX, n / kGridX), those past the last one leave at once.
constexpr int64_t kGridX = int64_t(1) << 20;
__device__ __forceinline__ int64_t group_id() {
  return static_cast<int64_t>(blockIdx.y) * kGridX + blockIdx.x;
}
dim3 group_grid(int64_t n) {
  if (n <= kGridX) return dim3(static_cast<unsigned>(n));
  return dim3(static_cast<unsigned>(kGridX), static_cast<unsigned>((n + kGridX - 1) / kGridX));
}

template <int D, bool kVec>
__global__ __launch_bounds__(256) void attn_fwd_f32(AttnArgs a, int64_t n_qt) {
  __shared__ __attribute__((aligned(16))) float Ks[kTile * (D + 4)], Vs[kTile * (D + 4)];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15, q4 = lane >> 4;
  const int64_t bid = group_id(), nbh = a.B * a.Hq;
  if (bid >= n_qt * nbh) return;
  const int64_t qt = n_qt - 1 - bid / nbh, bh = bid % nbh;
  const int64_t b = bh / a.Hq, hq = bh % a.Hq, hk = hq / (a.Hq / a.Hkv);
  const int64_t q0 = qt * 64, my_q = q0 + 16 * wave + l16;
  const int d = static_cast<int>(a.d);
  const float* K = static_cast<const float*>(a.k) + b * a.k_sb + hk * a.k_sh;
  const float* V = static_cast<const float*>(a.v) + b * a.v_sb + hk * a.v_sh;
  float4 q[D / 16];
  load_row<D, kVec>(q, my_q < a.Sq ? static_cast<const float*>(a.q) + b * a.q_sb + hq * a.q_sh +
                                         my_q * a.q_ss : nullptr, d);
  f32x4 o[D / 16];
#pragma unroll
  for (int nt = 0; nt < D / 16; ++nt) o[nt] = f32x4{};
  float m = -INFINITY, l = 0.f;
  int64_t t0, t1;
  tile_range<true>(a, q0, 64, t0, t1);
  TileReg<D, kVec> kr, vr;
  if (t0 < t1) {
    kr.load(K, a.k_ss, t0 * kTile, a.Skv, d);
    vr.load(V, a.v_ss, t0 * kTile, a.Skv, d);
  }
  for (int64_t t = t0; t < t1; ++t) {
    __syncthreads();  // the previous tile's reads are done
    kr.store(Ks);
    const bool odd = __syncthreads_or(vr.store(Vs));
    auto visible = [&](int r) __attribute__((always_inline)) {
      return attn_visible(my_q, t * kTile + r, a.Skv, a.causal, a.window);
    };
    if (t + 1 < t1) {
      kr.load(K, a.k_ss, (t + 1) * kTile, a.Skv, d);
      vr.load(V, a.v_ss, (t + 1) * kTile, a.Skv, d);
    }
    f32x4 s[2];
    float mloc = -INFINITY;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      s[h] = dot_rows<D>(Ks, 16 * h, q);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[h][e] = visible(16 * h + 4 * q4 + e) ? s[h][e] * a.scale : -INFINITY;
        mloc = fmaxf(mloc, s[h][e]);
      }
    }
    const float m_new = fmaxf(m, group_max(mloc));
    const float ref = m_new == -INFINITY ? 0.f : m_new;  // nothing visible yet
    const float alpha = expf(m - ref);
    m = m_new;
    l *= alpha;
#pragma unroll
    for (int nt = 0; nt < D / 16; ++nt) o[nt] *= alpha;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[h][e] = expf(s[h][e] - ref);
        l += s[h][e];
      }
      if (odd)
        add_rows_visible<D>(o, Vs, 16 * h, s[h], visible);
      else
        add_rows<D>(o, Vs, 16 * h, s[h]);
    }
  }
  l = group_sum(l);
  if (my_q >= a.Sq) return;
  // no weight although keys are visible: every score is -inf or NaN, and so is O
  store_row<D, kVec>(static_cast<float*>(a.out) + b * a.o_sb + hq * a.o_sh + my_q * a.o_ss, o,
                     l > 0.f ? 1.0f / l : t0 < t1 ? NAN : 0.f, d);
  if (q4 == 0) a.lse_out[(b * a.Hq + hq) * a.Sq + my_q] = l > 0.f ? m + logf(l) : -INFINITY;
}

// dQ, and delta = rowsum(dO o O) for the dK / dV kernel that follows.
template <int D, bool kVec>
__global__ __launch_bounds__(256) void attn_bwd_dq_f32(AttnArgs a, int64_t n_qt) {
  __shared__ __attribute__((aligned(16))) float Ks[kTile * (D + 4)], Vs[kTile * (D + 4)];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15, q4 = lane >> 4;
  const int64_t bid = group_id(), nbh = a.B * a.Hq;
  if (bid >= n_qt * nbh) return;
  const int64_t qt = n_qt - 1 - bid / nbh, bh = bid % nbh;
  const int64_t b = bh / a.Hq, hq = bh % a.Hq, hk = hq / (a.Hq / a.Hkv);
  const int64_t q0 = qt * 64, my_q = q0 + 16 * wave + l16;
  const int d = static_cast<int>(a.d);
  const bool in = my_q < a.Sq;
  const float* K = static_cast<const float*>(a.k) + b * a.k_sb + hk * a.k_sh;
  const float* V = static_cast<const float*>(a.v) + b * a.v_sb + hk * a.v_sh;
  const int64_t orow = b * a.o_sb + hq * a.o_sh + my_q * a.o_ss;
  float4 q[D / 16], g[D / 16];
  load_row<D, kVec>(q, in ? static_cast<const float*>(a.q) + b * a.q_sb + hq * a.q_sh + my_q * a.q_ss
                          : nullptr, d);
  load_row<D, kVec>(g, in ? static_cast<const float*>(a.dout) + orow : nullptr, d);
  float lse = INFINITY, del = 0.f;
  {
    float4 ov[D / 16];
    load_row<D, kVec>(ov, in ? static_cast<const float*>(a.o) + orow : nullptr, d);
#pragma unroll
    for (int c = 0; c < D / 16; ++c) {
      del = fmaf(ov[c].x, g[c].x, del);
      del = fmaf(ov[c].y, g[c].y, del);
      del = fmaf(ov[c].z, g[c].z, del);
      del = fmaf(ov[c].w, g[c].w, del);
    }
    del = group_sum(del);
    if (in) {
      const int64_t i = (b * a.Hq + hq) * a.Sq + my_q;
      lse = a.lse[i];  // -inf where O is NaN: the row's gradients are not finite either
      if (q4 == 0) {
        a.delta[i] = del;
        a.lse2[i] = lse;
      }
    }
  }
  f32x4 dq[D / 16];
#pragma unroll
  for (int nt = 0; nt < D / 16; ++nt) dq[nt] = f32x4{};
  int64_t t0, t1;
  tile_range<true>(a, q0, 64, t0, t1);
  TileReg<D, kVec> kr, vr;
  if (t0 < t1) {
    kr.load(K, a.k_ss, t0 * kTile, a.Skv, d);
    vr.load(V, a.v_ss, t0 * kTile, a.Skv, d);
  }
  for (int64_t t = t0; t < t1; ++t) {
    __syncthreads();
    vr.store(Vs);
    const bool odd = __syncthreads_or(kr.store(Ks));
    auto visible = [&](int r) __attribute__((always_inline)) {
      return in && attn_visible(my_q, t * kTile + r, a.Skv, a.causal, a.window);
    };
    if (t + 1 < t1) {
      kr.load(K, a.k_ss, (t + 1) * kTile, a.Skv, d);
      vr.load(V, a.v_ss, (t + 1) * kTile, a.Skv, d);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      f32x4 s = dot_rows<D>(Ks, 16 * h, q);
      const f32x4 dp = dot_rows<D>(Vs, 16 * h, g);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[e] = visible(16 * h + 4 * q4 + e) ? expf(s[e] * a.scale - lse) * (dp[e] - del) : 0.f;
      }
      if (odd)
        add_rows_visible<D>(dq, Ks, 16 * h, s, visible);
      else
        add_rows<D>(dq, Ks, 16 * h, s);
    }
  }
  float* out = static_cast<float*>(a.dq) + b * a.dq_sb + hq * a.dq_sh + my_q * a.dq_ss;
  if (in) store_row<D, kVec>(out, dq, a.scale, d);
  if (a.rope_cos != nullptr) {
    __syncthreads();  // the row's four lanes have stored it
    if (in) rope_inverse_row(out, a, my_q, q4, 4);
  }
}

// dK and dV of 64 keys per workgroup, summed over the query heads of the
// group; after attn_bwd_dq_f32 (delta, lse2).
template <int D, bool kVec>
__global__ __launch_bounds__(256) void attn_bwd_dkdv_f32(AttnArgs a, int64_t n_kt) {
  __shared__ __attribute__((aligned(16))) float Qs[kTile * (D + 4)], Gs[kTile * (D + 4)];
  __shared__ __attribute__((aligned(16))) float ls[kTile], ds[kTile];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15, q4 = lane >> 4;
  const int64_t bid = group_id(), nbh = a.B * a.Hkv;
  if (bid >= n_kt * nbh) return;
  const int64_t kt = bid / nbh, bh = bid % nbh;
  const int64_t b = bh / a.Hkv, hk = bh % a.Hkv, n_rep = a.Hq / a.Hkv;
  const int64_t k0 = kt * 64, my_k = k0 + 16 * wave + l16;
  const int d = static_cast<int>(a.d);
  const bool in = my_k < a.Skv;
  float4 k[D / 16], v[D / 16];
  load_row<D, kVec>(k, in ? static_cast<const float*>(a.k) + b * a.k_sb + hk * a.k_sh + my_k * a.k_ss
                          : nullptr, d);
  load_row<D, kVec>(v, in ? static_cast<const float*>(a.v) + b * a.v_sb + hk * a.v_sh + my_k * a.v_ss
                          : nullptr, d);
  f32x4 dk[D / 16], dv[D / 16];
#pragma unroll
  for (int nt = 0; nt < D / 16; ++nt) {
    dk[nt] = f32x4{};
    dv[nt] = f32x4{};
  }
  int64_t t0, t1;
  tile_range<false>(a, k0, 64, t0, t1);
  const int64_t nt = t1 - t0, n_it = nt * n_rep;
  TileReg<D, kVec> qr, gr;
  float lr = 0.f, dr = 0.f;
  auto load = [&](int64_t it) __attribute__((always_inline)) {
    const int64_t hq = hk * n_rep + it / nt, r0 = (t0 + it % nt) * kTile;
    qr.load(static_cast<const float*>(a.q) + b * a.q_sb + hq * a.q_sh, a.q_ss, r0, a.Sq, d);
    gr.load(static_cast<const float*>(a.dout) + b * a.o_sb + hq * a.o_sh, a.o_ss, r0, a.Sq, d);
    if (threadIdx.x < kTile) {
      const int64_t qi = r0 + threadIdx.x, i = (b * a.Hq + hq) * a.Sq + qi;
      lr = qi < a.Sq ? a.lse2[i] : INFINITY;
      dr = qi < a.Sq ? a.delta[i] : 0.f;
    }
  };
  if (n_it > 0) load(0);
  for (int64_t it = 0; it < n_it; ++it) {
    __syncthreads();
    const int odd_q = qr.store(Qs), odd_g = gr.store(Gs);
    if (threadIdx.x < kTile) {
      ls[threadIdx.x] = lr;
      ds[threadIdx.x] = dr;
    }
    const bool odd = __syncthreads_or(odd_q | odd_g);
    if (it + 1 < n_it) load(it + 1);
    const int64_t r0 = (t0 + it % nt) * kTile;
    auto visible = [&](int r) __attribute__((always_inline)) {
      return in && r0 + r < a.Sq && attn_visible(r0 + r, my_k, a.Skv, a.causal, a.window);
    };
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const f32x4 s = dot_rows<D>(Qs, 16 * h, k);
      const f32x4 dp = dot_rows<D>(Gs, 16 * h, v);
      f32x4 p, w;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = 16 * h + 4 * q4 + e;
        const bool vis = visible(r);
        p[e] = vis ? expf(s[e] * a.scale - ls[r]) : 0.f;
        w[e] = vis ? p[e] * (dp[e] - ds[r]) : 0.f;
      }
      if (odd) {
        add_rows_visible<D>(dv, Gs, 16 * h, p, visible);
        add_rows_visible<D>(dk, Qs, 16 * h, w, visible);
      } else {
        add_rows<D>(dv, Gs, 16 * h, p);
        add_rows<D>(dk, Qs, 16 * h, w);
      }
    }
  }
  float* dkp = static_cast<float*>(a.dk) + b * a.dk_sb + hk * a.dk_sh + my_k * a.dk_ss;
  if (in) {
    store_row<D, kVec>(dkp, dk, a.scale, d);
    store_row<D, kVec>(static_cast<float*>(a.dv) + b * a.dv_sb + hk * a.dv_sh + my_k * a.dv_ss, dv,
                       1.f, d);
  }
  if (a.rope_cos != nullptr) {
    __syncthreads();
    if (in) rope_inverse_row(dkp, a, my_k, q4, 4);
  }
}

// ---- many sequences of a few tokens: one thread per row --------------------
// The kernels above give each (batch, head) a workgroup of 64 rows, and with it
// a workgroup's latency however few its rows are; here a thread walks its row's
// keys (or its key's queries) by itself (by_rows below says when).

// Elements 4 c .. 4 c + 3 of a row of d, zeros from d on.
template <bool kVec>
__device__ __forceinline__ float4 row4(const float* row, int c, int d) {
  const float* p = row + 4 * c;
  if (kVec) return *reinterpret_cast<const float4*>(p);
  const int n = d - 4 * c;
  return make_float4(p[0], n > 1 ? p[1] : 0.f, n > 2 ? p[2] : 0.f, n > 3 ? p[3] : 0.f);
}
template <int D, bool kVec>
__device__ __forceinline__ float row_dot(const float* x, const float* y, int d) {
  float s = 0.f;
#pragma unroll
  for (int c = 0; c < D / 4; ++c)
    if (4 * c < d) {
      const float4 u = row4<kVec>(x, c, d), w = row4<kVec>(y, c, d);
      s = fmaf(u.x, w.x, s);
      s = fmaf(u.y, w.y, s);
      s = fmaf(u.z, w.z, s);
      s = fmaf(u.w, w.w, s);
    }
  return s;
}
// acc = f acc + w x
template <int D, bool kVec>
__device__ __forceinline__ void row_add(float4 (&acc)[D / 4], float f, float w, const float* x,
                                        int d) {
#pragma unroll
  for (int c = 0; c < D / 4; ++c)
    if (4 * c < d) {
      const float4 u = row4<kVec>(x, c, d);
      acc[c] = make_float4(fmaf(acc[c].x, f, w * u.x), fmaf(acc[c].y, f, w * u.y),
                           fmaf(acc[c].z, f, w * u.z), fmaf(acc[c].w, f, w * u.w));
    }
}
template <int D, bool kVec>
__device__ __forceinline__ void row_put(float* dst, const float4 (&x)[D / 4], float scale, int d) {
#pragma unroll
  for (int c = 0; c < D / 4; ++c)
    if (4 * c < d) {
      const float v[4] = {x[c].x * scale, x[c].y * scale, x[c].z * scale, x[c].w * scale};
      float* p = dst + 4 * c;
      if (kVec) {
        *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (4 * c + e < d) p[e] = v[e];
      }
    }
}
template <int D>
__device__ __forceinline__ void row_zero(float4 (&x)[D / 4]) {
#pragma unroll
  for (int c = 0; c < D / 4; ++c) x[c] = make_float4(0.f, 0.f, 0.f, 0.f);
}

template <int D, bool kVec>
__global__ __launch_bounds__(64) void attn_fwd_rows_f32(AttnArgs a) {
  const int64_t row = group_id() * 64 + threadIdx.x;
  if (row >= a.B * a.Hq * a.Sq) return;
  const int64_t qi = row % a.Sq, bh = row / a.Sq;
  const int64_t b = bh / a.Hq, hq = bh % a.Hq, hk = hq / (a.Hq / a.Hkv);
  const int d = static_cast<int>(a.d);
  const float* Q = static_cast<const float*>(a.q) + b * a.q_sb + hq * a.q_sh + qi * a.q_ss;
  const float* K = static_cast<const float*>(a.k) + b * a.k_sb + hk * a.k_sh;
  const float* V = static_cast<const float*>(a.v) + b * a.v_sb + hk * a.v_sh;
  float4 o[D / 4];
  row_zero<D>(o);
  float m = -INFINITY, l = 0.f;
  for (int64_t j = 0; j < a.Skv; ++j) {
    if (!attn_visible(qi, j, a.Skv, a.causal, a.window)) continue;
    const float s = row_dot<D, kVec>(Q, K + j * a.k_ss, d) * a.scale;
    const float m_new = fmaxf(m, s);
    const float ref = m_new == -INFINITY ? 0.f : m_new;  // no weight yet
    const float alpha = expf(m - ref), p = expf(s - ref);
    l = l * alpha + p;
    row_add<D, kVec>(o, alpha, p, V + j * a.v_ss, d);
    m = m_new;
  }
  row_put<D, kVec>(static_cast<float*>(a.out) + b * a.o_sb + hq * a.o_sh + qi * a.o_ss, o,
                   l > 0.f ? 1.0f / l : a.Skv > 0 ? NAN : 0.f, d);
  a.lse_out[row] = l > 0.f ? m + logf(l) : -INFINITY;
}

template <int D, bool kVec>
__global__ __launch_bounds__(64) void attn_bwd_dq_rows_f32(AttnArgs a) {
  const int64_t row = group_id() * 64 + threadIdx.x;
  if (row >= a.B * a.Hq * a.Sq) return;
  const int64_t qi = row % a.Sq, bh = row / a.Sq;
  const int64_t b = bh / a.Hq, hq = bh % a.Hq, hk = hq / (a.Hq / a.Hkv);
  const int d = static_cast<int>(a.d);
  const int64_t orow = b * a.o_sb + hq * a.o_sh + qi * a.o_ss;
  const float* Q = static_cast<const float*>(a.q) + b * a.q_sb + hq * a.q_sh + qi * a.q_ss;
  const float* G = static_cast<const float*>(a.dout) + orow;
  const float* K = static_cast<const float*>(a.k) + b * a.k_sb + hk * a.k_sh;
  const float* V = static_cast<const float*>(a.v) + b * a.v_sb + hk * a.v_sh;
  const float lse = a.lse[row], del = row_dot<D, kVec>(static_cast<const float*>(a.o) + orow, G, d);
  a.lse2[row] = lse;
  a.delta[row] = del;
  float4 dq[D / 4];
  row_zero<D>(dq);
  for (int64_t j = 0; j < a.Skv; ++j) {
    if (!attn_visible(qi, j, a.Skv, a.causal, a.window)) continue;
    const float* k = K + j * a.k_ss;
    const float p = expf(row_dot<D, kVec>(Q, k, d) * a.scale - lse);
    row_add<D, kVec>(dq, 1.f, p * (row_dot<D, kVec>(G, V + j * a.v_ss, d) - del), k, d);
  }
  float* out = static_cast<float*>(a.dq) + b * a.dq_sb + hq * a.dq_sh + qi * a.dq_ss;
  row_put<D, kVec>(out, dq, a.scale, d);
  if (a.rope_cos != nullptr) rope_inverse_row(out, a, qi, 0, 1);
}

template <int D, bool kVec>
__global__ __launch_bounds__(64) void attn_bwd_dkdv_rows_f32(AttnArgs a) {
  const int64_t row = group_id() * 64 + threadIdx.x;
  if (row >= a.B * a.Hkv * a.Skv) return;
  const int64_t kj = row % a.Skv, bh = row / a.Skv;
  const int64_t b = bh / a.Hkv, hk = bh % a.Hkv, n_rep = a.Hq / a.Hkv;
  const int d = static_cast<int>(a.d);
  const float* K = static_cast<const float*>(a.k) + b * a.k_sb + hk * a.k_sh + kj * a.k_ss;
  const float* V = static_cast<const float*>(a.v) + b * a.v_sb + hk * a.v_sh + kj * a.v_ss;
  float4 dk[D / 4], dv[D / 4];
  row_zero<D>(dk);
  row_zero<D>(dv);
  for (int64_t hq = hk * n_rep; hq < (hk + 1) * n_rep; ++hq) {
    const float* Q = static_cast<const float*>(a.q) + b * a.q_sb + hq * a.q_sh;
    const float* G = static_cast<const float*>(a.dout) + b * a.o_sb + hq * a.o_sh;
    for (int64_t qi = 0; qi < a.Sq; ++qi) {
      if (!attn_visible(qi, kj, a.Skv, a.causal, a.window)) continue;
      const int64_t i = (b * a.Hq + hq) * a.Sq + qi;
      const float* q = Q + qi * a.q_ss;
      const float* g = G + qi * a.o_ss;
      const float p = expf(row_dot<D, kVec>(q, K, d) * a.scale - a.lse2[i]);
      row_add<D, kVec>(dv, 1.f, p, g, d);
      row_add<D, kVec>(dk, 1.f, p * (row_dot<D, kVec>(g, V, d) - a.delta[i]), q, d);
    }
  }
  float* dkp = static_cast<float*>(a.dk) + b * a.dk_sb + hk * a.dk_sh + kj * a.dk_ss;
  row_put<D, kVec>(dkp, dk, a.scale, d);
  row_put<D, kVec>(static_cast<float*>(a.dv) + b * a.dv_sb + hk * a.dv_sh + kj * a.dv_ss, dv, 1.f, d);
  if (a.rope_cos != nullptr) rope_inverse_row(dkp, a, kj, 0, 1);
}

// Which kernels a pass takes, `heads` the (batch, head) pairs of its rows: a
// workgroup costs its latency over the chip (8 ns forward and 24 backward once
// there are 2048, 15 and 55 for head dims above 64), a row the walk over S keys of
// d elements, never less than 12 us forward and 20 backward in all.  Measured, us
// forward + backward, tiles / rows, at 1024, 2048 and 16384 heads:
//   S 1, d 64     47 / 37     79 / 36     527 / 40
//   S 8, d 16     46 / 39     78 / 40     544 / 73
//   S 4, d 32     51 / 45     79 / 44     545 / 71
//   S 4, d 64     47 / 67     81 / 68     549 / 135
//   S 16, d 16    46 / 65     80 / 67     541 / 215
//   S 4, d 128    84 / 126   156 / 128   1160 / 268
//   S 32, d 16    50 / 122    84 / 130    575 / 744
//   S 2, d 50     53 / 70     91 / 70     625 / 129   (not 16-byte aligned)
// and 512 heads are even up to S d = 64, slower from there.
bool by_rows(const AttnArgs& a, int64_t heads, bool vec) {
  const int64_t S = a.Sq > a.Skv ? a.Sq : a.Skv;
  const int64_t cost = vec ? S * a.d : S * a.d * 3 / 2;
  return heads >= 1024 && cost <= heads / 8 && cost <= (S <= 4 ? 512 : 256);
}

// float4 accesses: head dim and strides multiples of 4, pointers of 16 bytes
bool vec4_ok(int64_t d, std::initializer_list<int64_t> strides,
             std::initializer_list<const void*> ptrs) {
  if (d % 4 != 0) return false;
  for (int64_t s : strides)
    if (s % 4 != 0) return false;
  for (const void* p : ptrs)
    if (!aligned(p, 16)) return false;
  return true;
}

}  // namespace

#define ZK_F32_DISPATCH(KERNEL, GRID, ...)                                                   \
  do {                                                                                       \
    if (a.d <= 64 && vec)                                                                    \
      hipLaunchKernelGGL((KERNEL<64, true>), GRID, dim3(256), 0, s, __VA_ARGS__);            \
    else if (a.d <= 64)                                                                      \
      hipLaunchKernelGGL((KERNEL<64, false>), GRID, dim3(256), 0, s, __VA_ARGS__);           \
    else if (vec)                                                                            \
      hipLaunchKernelGGL((KERNEL<128, true>), GRID, dim3(256), 0, s, __VA_ARGS__);           \
    else                                                                                     \
      hipLaunchKernelGGL((KERNEL<128, false>), GRID, dim3(256), 0, s, __VA_ARGS__);          \
  } while (0)

#define ZK_F32_ROWS(KERNEL, ROWS)                                                              \
  do {                                                                                         \
    const dim3 grid = group_grid(((ROWS) + 63) / 64);                                          \
    if (a.d <= 16) {                                                                           \
      if (vec) hipLaunchKernelGGL((KERNEL<16, true>), grid, dim3(64), 0, s, a);                \
      else hipLaunchKernelGGL((KERNEL<16, false>), grid, dim3(64), 0, s, a);                   \
    } else if (a.d <= 64) {                                                                    \
      if (vec) hipLaunchKernelGGL((KERNEL<64, true>), grid, dim3(64), 0, s, a);                \
      else hipLaunchKernelGGL((KERNEL<64, false>), grid, dim3(64), 0, s, a);                   \
    } else {                                                                                   \
      if (vec) hipLaunchKernelGGL((KERNEL<128, true>), grid, dim3(64), 0, s, a);               \
      else hipLaunchKernelGGL((KERNEL<128, false>), grid, dim3(64), 0, s, a);                  \
    }                                                                                          \
  } while (0)

void launch_attn_fwd_f32(const AttnArgs& a, hipStream_t s) {
  const bool vec = vec4_ok(a.d, {a.q_sb, a.q_ss, a.q_sh, a.k_sb, a.k_ss, a.k_sh, a.v_sb, a.v_ss,
                                 a.v_sh, a.o_sb, a.o_ss, a.o_sh}, {a.q, a.k, a.v, a.out});
  if (by_rows(a, a.B * a.Hq, vec)) {
    ZK_F32_ROWS(attn_fwd_rows_f32, a.B * a.Hq * a.Sq);
    return;
  }
  const int64_t n_qt = (a.Sq + 63) / 64;
  const dim3 grid = group_grid(n_qt * a.B * a.Hq);
  ZK_F32_DISPATCH(attn_fwd_f32, grid, a, n_qt);
}

void launch_attn_bwd_f32(const AttnArgs& a, hipStream_t s) {
  const bool vec = vec4_ok(a.d, {a.q_sb, a.q_ss, a.q_sh, a.k_sb, a.k_ss, a.k_sh, a.v_sb, a.v_ss,
                                 a.v_sh, a.o_sb, a.o_ss, a.o_sh, a.dq_sb, a.dq_ss, a.dq_sh, a.dk_sb,
                                 a.dk_ss, a.dk_sh, a.dv_sb, a.dv_ss, a.dv_sh},
                           {a.q, a.k, a.v, a.o, a.dout, a.dq, a.dk, a.dv});
  const int64_t n_qt = (a.Sq + 63) / 64, n_kt = (a.Skv + 63) / 64;
  if (n_qt > 0 && by_rows(a, a.B * a.Hq, vec)) {
    ZK_F32_ROWS(attn_bwd_dq_rows_f32, a.B * a.Hq * a.Sq);
  } else if (n_qt > 0) {
    const dim3 grid = group_grid(n_qt * a.B * a.Hq);
    ZK_F32_DISPATCH(attn_bwd_dq_f32, grid, a, n_qt);
  }
  if (n_kt > 0 && by_rows(a, a.B * a.Hkv, vec)) {
    ZK_F32_ROWS(attn_bwd_dkdv_rows_f32, a.B * a.Hkv * a.Skv);
  } else if (n_kt > 0) {
    const dim3 grid = group_grid(n_kt * a.B * a.Hkv);
    ZK_F32_DISPATCH(attn_bwd_dkdv_f32, grid, a, n_kt);
  }
}

}  // namespace zk
