// Rotary position embedding, applied in place to Q and K.
//
// One thread rotates 4 pairs of one (batch, position, head) row: for the
// half-split pairing it reads elements i..i+3 and i+d/2..i+d/2+3, for the
// interleaved pairing the 8 consecutive elements 2i..2i+7.  cos/sin come
// from fp32 tables [n_pos, d/2] built by the caller with the reference's
// own formula, so the kernel only does the rotation arithmetic (rotate_pair,
// rope_math.h).
#include "rope_math.h"

namespace zk {

template <typename T, int kPairing, bool kInverse>
__global__ __launch_bounds__(256) void rope_kernel(
    T* __restrict__ q, int64_t q_sb, int64_t q_ss, int64_t q_sh,
    T* __restrict__ k, int64_t k_sb, int64_t k_ss, int64_t k_sh, int64_t B,
    int64_t S, int64_t Hq, int64_t Hkv, int64_t d,
    const float* __restrict__ cosT, const float* __restrict__ sinT,
    int64_t n_pos, const int64_t* __restrict__ positions) {
  const int64_t half = d / 2;
  const int64_t nq = (half + 3) / 4;  // quads of pairs per row
  const int64_t H = Hq + (k != nullptr ? Hkv : 0);
  const int64_t total = B * S * H * nq;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
       t < total; t += stride) {
    int64_t r = t;
    const int64_t quad = r % nq; r /= nq;
    const int64_t h = r % H; r /= H;
    const int64_t s = r % S;
    const int64_t b = r / S;
    T* row = h < Hq ? q + b * q_sb + s * q_ss + h * q_sh
                    : k + b * k_sb + s * k_ss + (h - Hq) * k_sh;
    int64_t pos = positions != nullptr ? positions[s] : s;
    if (pos < 0) pos = 0;
    if (pos >= n_pos) pos = n_pos - 1;
    const float* crow = cosT + pos * half;
    const float* srow = sinT + pos * half;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t i = quad * 4 + j;
      if (i < half) {
        const int64_t i1 = kPairing == ZK_ROPE_HALF ? i : 2 * i;
        const int64_t i2 = kPairing == ZK_ROPE_HALF ? i + half : 2 * i + 1;
        float y1, y2;
        rotate_pair<T, kPairing, kInverse>(to_f32(row[i1]), to_f32(row[i2]),
                                           crow[i], srow[i], y1, y2);
        row[i1] = from_f32<T>(y1);
        row[i2] = from_f32<T>(y2);
      }
    }
  }
}

// The rows of one tensor [B, S, H, d]: read from src, written to dst (in place
// where they and their strides are the same), strides in elements.
template <typename T>
struct RopeRows {
  T* dst;
  const T* src;
  int64_t d_sb, d_ss, d_sh, s_sb, s_ss, s_sh;
};

// One thread's 8 pairs of one (position, head) row, 16-byte accesses, from
// `in` to `row` (the same address where the pass is in place).
template <typename T, int D, int kPairing, bool kInverse>
__device__ __forceinline__ void rope_chunk8(T* row, const T* in, int i0, const float (&c)[8],
                                            const float (&sn)[8]) {
  constexpr int HALF = D / 2;
  float x1[8], x2[8], y1[8], y2[8];
  if (kPairing == ZK_ROPE_HALF) {
    Vec8<T>::load(in + i0, x1);
    Vec8<T>::load(in + i0 + HALF, x2);
  } else {
    float a[8], bb[8];
    Vec8<T>::load(in + 2 * i0, a);
    Vec8<T>::load(in + 2 * i0 + 8, bb);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      x1[j] = a[2 * j];
      x2[j] = a[2 * j + 1];
      x1[j + 4] = bb[2 * j];
      x2[j + 4] = bb[2 * j + 1];
    }
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) rotate_pair<T, kPairing, kInverse>(x1[j], x2[j], c[j], sn[j], y1[j], y2[j]);
  if (kPairing == ZK_ROPE_HALF) {
    Vec8<T>::store(row + i0, y1);
    Vec8<T>::store(row + i0 + HALF, y2);
  } else {
    float a[8], bb[8];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      a[2 * j] = y1[j];
      a[2 * j + 1] = y2[j];
      bb[2 * j] = y1[j + 4];
      bb[2 * j + 1] = y2[j + 4];
    }
    Vec8<T>::store(row + 2 * i0, a);
    Vec8<T>::store(row + 2 * i0 + 8, bb);
  }
}

// Vectorised path for head_dim 64 / 128 with 16-byte aligned rows and few
// heads: a thread rotates 8 pairs of one row; the grid is (position blocks,
// heads, batch), so no index arithmetic divides.
template <typename T, int D, int kPairing, bool kInverse>
__global__ __launch_bounds__(256) void rope_vec_kernel(
    RopeRows<T> q, RopeRows<T> k, int64_t S, int64_t Hq,
    const float* __restrict__ cosT, const float* __restrict__ sinT, int64_t n_pos,
    const int64_t* __restrict__ positions) {
  constexpr int HALF = D / 2;
  constexpr int TPR = HALF / 8;        // threads per (position, head) row
  constexpr int RPB = 256 / TPR;       // positions per workgroup
  const int64_t s = static_cast<int64_t>(blockIdx.x) * RPB + threadIdx.x / TPR;
  if (s >= S) return;
  const int64_t h = blockIdx.y, b = blockIdx.z;
  const int i0 = (threadIdx.x % TPR) * 8;  // first pair of this thread
  const RopeRows<T>& x = h < Hq ? q : k;
  const int64_t hx = h < Hq ? h : h - Hq;
  int64_t pos = positions != nullptr ? positions[s] : s;
  if (pos < 0) pos = 0;
  if (pos >= n_pos) pos = n_pos - 1;
  float c[8], sn[8];
  Vec8<float>::load(cosT + pos * HALF + i0, c);
  Vec8<float>::load(sinT + pos * HALF + i0, sn);
  rope_chunk8<T, D, kPairing, kInverse>(x.dst + b * x.d_sb + s * x.d_ss + hx * x.d_sh,
                                        x.src + b * x.s_sb + s * x.s_ss + hx * x.s_sh, i0, c, sn);
}

// Position-major path for many heads: a workgroup rotates every q and k head
// of one (batch, position) -- with heads contiguous in memory, one run of
// (Hq + Hkv) d elements -- and each thread reads its cos / sin values once
// (256 threads and HALF / 8 chunks per row: a thread's pair offset is the
// same in every head it visits).
template <typename T, int D, int kPairing, bool kInverse>
__global__ __launch_bounds__(256) void rope_pos_kernel(
    RopeRows<T> q, RopeRows<T> k, int64_t Hq, int64_t H,
    const float* __restrict__ cosT, const float* __restrict__ sinT, int64_t n_pos,
    const int64_t* __restrict__ positions) {
  constexpr int HALF = D / 2;
  constexpr int CPH = HALF / 8;  // 8-pair chunks per head row
  static_assert(256 % CPH == 0, "chunk offset must be fixed per thread");
  const int64_t s = blockIdx.x, b = blockIdx.y;
  const int i0 = (threadIdx.x % CPH) * 8;
  int64_t pos = positions != nullptr ? positions[s] : s;
  if (pos < 0) pos = 0;
  if (pos >= n_pos) pos = n_pos - 1;
  float c[8], sn[8];
  Vec8<float>::load(cosT + pos * HALF + i0, c);
  Vec8<float>::load(sinT + pos * HALF + i0, sn);
  for (int64_t h = threadIdx.x / CPH; h < H; h += 256 / CPH) {
    const RopeRows<T>& x = h < Hq ? q : k;
    const int64_t hx = h < Hq ? h : h - Hq;
    rope_chunk8<T, D, kPairing, kInverse>(x.dst + b * x.d_sb + s * x.d_ss + hx * x.d_sh,
                                          x.src + b * x.s_sb + s * x.s_ss + hx * x.s_sh, i0, c, sn);
  }
}

// Position-major path for the other head dims that are multiples of 4 (2-byte
// types, rows at even element offsets): a thread owns two neighbouring pairs,
// reads their cos / sin once and rotates them in every head it visits with
// 4-byte accesses (half of such a head dim is even, so both halves of a pair of
// pairs are 4-byte aligned).  Nothing divides inside the loop: 12 us where the
// general pass, element accesses and three divisions a thread, takes 34 (64
// heads of 100 at 2048 positions, 52 MB read and written).
template <typename T, int kPairing, bool kInverse>
__global__ __launch_bounds__(256) void rope_pos2_kernel(
    T* __restrict__ q, int64_t q_sb, int64_t q_ss, int64_t q_sh,
    T* __restrict__ k, int64_t k_sb, int64_t k_ss, int64_t k_sh, int64_t Hq, int64_t H, int half,
    const float* __restrict__ cosT, const float* __restrict__ sinT, int64_t n_pos,
    const int64_t* __restrict__ positions) {
  typedef T T2 __attribute__((ext_vector_type(2)));
  const int n2 = half / 2, hpb = 256 / n2;  // two-pair slots per head, heads per sweep
  const int h0 = static_cast<int>(threadIdx.x) / n2;
  if (h0 >= hpb) return;
  const int i0 = (static_cast<int>(threadIdx.x) - h0 * n2) * 2;
  const int64_t s = blockIdx.x, b = blockIdx.y;
  int64_t pos = positions != nullptr ? positions[s] : s;
  if (pos < 0) pos = 0;
  if (pos >= n_pos) pos = n_pos - 1;
  const float2 c = *reinterpret_cast<const float2*>(cosT + pos * half + i0);
  const float2 sn = *reinterpret_cast<const float2*>(sinT + pos * half + i0);
  T* qrow = q + b * q_sb + s * q_ss;
  T* krow = k != nullptr ? k + b * k_sb + s * k_ss : nullptr;
  // half-split: elements i0, i0 + 1 and their partners at + half;
  // interleaved: elements 2 i0 .. 2 i0 + 3
  const int e0 = kPairing == ZK_ROPE_HALF ? i0 : 2 * i0;
  const int e1 = kPairing == ZK_ROPE_HALF ? i0 + half : 2 * i0 + 2;
  for (int64_t h = h0; h < H; h += hpb) {
    T* row = h < Hq ? qrow + h * q_sh : krow + (h - Hq) * k_sh;
    const T2 u = *reinterpret_cast<const T2*>(row + e0);
    const T2 w = *reinterpret_cast<const T2*>(row + e1);
    float y[4];
    if (kPairing == ZK_ROPE_HALF) {
      rotate_pair<T, kPairing, kInverse>(to_f32(u[0]), to_f32(w[0]), c.x, sn.x, y[0], y[2]);
      rotate_pair<T, kPairing, kInverse>(to_f32(u[1]), to_f32(w[1]), c.y, sn.y, y[1], y[3]);
    } else {
      rotate_pair<T, kPairing, kInverse>(to_f32(u[0]), to_f32(u[1]), c.x, sn.x, y[0], y[1]);
      rotate_pair<T, kPairing, kInverse>(to_f32(w[0]), to_f32(w[1]), c.y, sn.y, y[2], y[3]);
    }
    const T2 a = {from_f32<T>(y[0]), from_f32<T>(y[1])}, z = {from_f32<T>(y[2]), from_f32<T>(y[3])};
    *reinterpret_cast<T2*>(row + e0) = a;
    *reinterpret_cast<T2*>(row + e1) = z;
  }
}

template <typename T>
static void launch_rope_pos2(int pairing, int inverse, void* q, int64_t q_sb, int64_t q_ss,
                             int64_t q_sh, void* k, int64_t k_sb, int64_t k_ss, int64_t k_sh,
                             int64_t B, int64_t S, int64_t Hq, int64_t H, int64_t d,
                             const float* c, const float* sn, int64_t n_pos, const int64_t* pos,
                             hipStream_t st) {
  const dim3 grid(static_cast<unsigned>(S), static_cast<unsigned>(B));
#define ZK_ROPE2(P, I)                                                                     \
  hipLaunchKernelGGL((rope_pos2_kernel<T, P, I>), grid, dim3(256), 0, st, (T*)q, q_sb,     \
                     q_ss, q_sh, (T*)k, k_sb, k_ss, k_sh, Hq, H, static_cast<int>(d / 2), c, \
                     sn, n_pos, pos)
  if (pairing == ZK_ROPE_HALF) {
    if (inverse) ZK_ROPE2(ZK_ROPE_HALF, true); else ZK_ROPE2(ZK_ROPE_HALF, false);
  } else {
    if (inverse) ZK_ROPE2(ZK_ROPE_INTERLEAVED, true); else ZK_ROPE2(ZK_ROPE_INTERLEAVED, false);
  }
#undef ZK_ROPE2
}

template <typename T, int D>
static void launch_rope_vec(int pairing, int inverse, const RopeRows<T>& q, const RopeRows<T>& k,
                            int64_t B, int64_t S, int64_t Hq, int64_t H, const float* c,
                            const float* sn, int64_t n_pos, const int64_t* pos, hipStream_t st) {
  constexpr int RPB = 256 / (D / 16);
  // position-major once a position's rows fill half a workgroup's threads
  const bool by_pos = H * (D / 16) >= 128 && S < 0x7fffffff;
  const dim3 grid = by_pos ? dim3(static_cast<unsigned>(S), static_cast<unsigned>(B))
                           : dim3(static_cast<unsigned>((S + RPB - 1) / RPB),
                                  static_cast<unsigned>(H), static_cast<unsigned>(B));
#define ZK_ROPEV(P, I)                                                                       \
  do {                                                                                       \
    if (by_pos)                                                                              \
      hipLaunchKernelGGL((rope_pos_kernel<T, D, P, I>), grid, dim3(256), 0, st, q, k, Hq, H, \
                         c, sn, n_pos, pos);                                                 \
    else                                                                                     \
      hipLaunchKernelGGL((rope_vec_kernel<T, D, P, I>), grid, dim3(256), 0, st, q, k, S, Hq, \
                         c, sn, n_pos, pos);                                                 \
  } while (0)
  if (pairing == ZK_ROPE_HALF) {
    if (inverse) ZK_ROPEV(ZK_ROPE_HALF, true); else ZK_ROPEV(ZK_ROPE_HALF, false);
  } else {
    if (inverse) ZK_ROPEV(ZK_ROPE_INTERLEAVED, true); else ZK_ROPEV(ZK_ROPE_INTERLEAVED, false);
  }
#undef ZK_ROPEV
}

template <typename T>
static void launch_rope(int pairing, int inverse, void* q, int64_t q_sb,
                        int64_t q_ss, int64_t q_sh, void* k, int64_t k_sb,
                        int64_t k_ss, int64_t k_sh, int64_t B, int64_t S,
                        int64_t Hq, int64_t Hkv, int64_t d, const float* c,
                        const float* sn, int64_t n_pos, const int64_t* pos,
                        hipStream_t st) {
  const int64_t H = Hq + (k != nullptr ? Hkv : 0);
  const int64_t total = B * S * H * ((d / 2 + 3) / 4);
  int64_t grid = (total + 255) / 256;
  const int64_t cap = static_cast<int64_t>(device_cus()) * 16;
  if (grid > cap) grid = cap;
  if (grid < 1) grid = 1;
#define ZK_ROPE(P, I)                                                          \
  hipLaunchKernelGGL((rope_kernel<T, P, I>), dim3(grid), dim3(256), 0, st,     \
                     (T*)q, q_sb, q_ss, q_sh, (T*)k, k_sb, k_ss, k_sh, B, S, Hq, \
                     Hkv, d, c, sn, n_pos, pos)
  if (pairing == ZK_ROPE_HALF) {
    if (inverse) ZK_ROPE(ZK_ROPE_HALF, true); else ZK_ROPE(ZK_ROPE_HALF, false);
  } else {
    if (inverse) ZK_ROPE(ZK_ROPE_INTERLEAVED, true); else ZK_ROPE(ZK_ROPE_INTERLEAVED, false);
  }
#undef ZK_ROPE
}

}  // namespace zk

using namespace zk;

extern "C" int zk_rope(void* q, int64_t q_sb, int64_t q_ss, int64_t q_sh,
                       void* k, int64_t k_sb, int64_t k_ss, int64_t k_sh,
                       int64_t B, int64_t S, int64_t Hq, int64_t Hkv, int64_t d,
                       const float* cos, const float* sin, int64_t n_pos,
                       const int64_t* positions, int pairing, int inverse,
                       int dtype, zk_stream_t stream) {
  ZK_REQUIRE(valid_dtype(dtype), ZK_EDTYPE, "zk_rope: bad dtype %d", dtype);
  ZK_REQUIRE(pairing == ZK_ROPE_HALF || pairing == ZK_ROPE_INTERLEAVED,
             ZK_EINVAL, "zk_rope: bad pairing %d", pairing);
  ZK_REQUIRE(B >= 0 && S >= 0 && Hq >= 0 && Hkv >= 0 && d > 0 && d % 2 == 0,
             ZK_EINVAL, "zk_rope: bad shape (d must be even, got %lld)",
             (long long)d);
  ZK_REQUIRE(q && cos && sin, ZK_EINVAL, "zk_rope: null pointer");
  ZK_REQUIRE(positions != nullptr || n_pos >= S, ZK_EINVAL,
             "zk_rope: table has %lld positions < S=%lld", (long long)n_pos,
             (long long)S);
  ZK_REQUIRE(n_pos > 0, ZK_EINVAL, "zk_rope: empty table");
  if (B == 0 || S == 0 || Hq + Hkv == 0) return ZK_OK;
  hipStream_t st = as_stream(stream);
  // 16-byte vector path: 2-byte types, d 64 / 128, aligned rows and heads,
  // grid dimensions within range
  const int64_t H = Hq + (k != nullptr ? Hkv : 0);
  bool vec = dtype != ZK_F32 && (d == 64 || d == 128) && aligned(q, 16) &&
             (k == nullptr || aligned(k, 16)) && H < 65536 && B < 65536 &&
             S / (256 / (d / 16)) < 0x7fffffff;
  vec = vec && q_sb % 8 == 0 && q_ss % 8 == 0 && q_sh % 8 == 0;
  if (k != nullptr) vec = vec && k_sb % 8 == 0 && k_ss % 8 == 0 && k_sh % 8 == 0;
  if (vec) {
#define ZK_VEC(T, D)                                                                          \
  launch_rope_vec<T, D>(pairing, inverse,                                                     \
                        RopeRows<T>{(T*)q, (const T*)q, q_sb, q_ss, q_sh, q_sb, q_ss, q_sh},  \
                        RopeRows<T>{(T*)k, (const T*)k, k_sb, k_ss, k_sh, k_sb, k_ss, k_sh},  \
                        B, S, Hq, H, cos, sin, n_pos, positions, st)
    if (dtype == ZK_BF16) {
      if (d == 128) ZK_VEC(bf16, 128); else ZK_VEC(bf16, 64);
    } else {
      if (d == 128) ZK_VEC(f16, 128); else ZK_VEC(f16, 64);
    }
#undef ZK_VEC
    return launch_status("zk_rope");
  }
  // other head dims: position-major, 4-byte accesses (tables 8-byte aligned:
  // rows of d / 2 floats, an even number)
  bool pos2 = dtype != ZK_F32 && d % 4 == 0 && d <= 1024 && aligned(q, 4) &&
              (k == nullptr || aligned(k, 4)) && aligned(cos, 8) && aligned(sin, 8) &&
              S < (int64_t(1) << 24) && B < 65536;  // 256 threads a position, below 2^32
  // A workgroup a position costs 0.5 ns, whatever its heads give it to do: with
  // less than a wavefront's work, H d / 4 < 64, the general pass is ahead.  us
  // general / position-major, at 65536 positions: 1 head of 16 7 / 35, 4 of 48
  // 25 / 35, 2 of 100 32 / 36, 16 of 16 37 / 35, 4 of 100 60 / 42; up to 8192
  // positions either takes a launch's 7 us.
  pos2 = pos2 && H * (d / 4) >= 64;
  pos2 = pos2 && q_sb % 2 == 0 && q_ss % 2 == 0 && q_sh % 2 == 0;
  if (k != nullptr) pos2 = pos2 && k_sb % 2 == 0 && k_ss % 2 == 0 && k_sh % 2 == 0;
  if (pos2) {
    if (dtype == ZK_BF16)
      launch_rope_pos2<bf16>(pairing, inverse, q, q_sb, q_ss, q_sh, k, k_sb, k_ss, k_sh, B, S, Hq, H, d, cos, sin, n_pos, positions, st);
    else
      launch_rope_pos2<f16>(pairing, inverse, q, q_sb, q_ss, q_sh, k, k_sb, k_ss, k_sh, B, S, Hq, H, d, cos, sin, n_pos, positions, st);
    return launch_status("zk_rope");
  }
  if (dtype == ZK_BF16)
    launch_rope<bf16>(pairing, inverse, q, q_sb, q_ss, q_sh, k, k_sb, k_ss, k_sh, B, S, Hq, Hkv, d, cos, sin, n_pos, positions, st);
  else if (dtype == ZK_F16)
    launch_rope<f16>(pairing, inverse, q, q_sb, q_ss, q_sh, k, k_sb, k_ss, k_sh, B, S, Hq, Hkv, d, cos, sin, n_pos, positions, st);
  else
    launch_rope<float>(pairing, inverse, q, q_sb, q_ss, q_sh, k, k_sb, k_ss, k_sh, B, S, Hq, Hkv, d, cos, sin, n_pos, positions, st);
  return launch_status("zk_rope");
}

// The rotated copies of q and k (contiguous [B, S, H, d]), head dims 64 and 128
// of 2-byte types with 16-byte aligned rows: 84 us for 8 x 2048 positions of 32
// + 32 heads of 128 (537 MB, 6.4 TB/s), where copying both and rotating in
// place took 98 + 81.
extern "C" int zk_rope_copy(const void* q, int64_t q_sb, int64_t q_ss, int64_t q_sh, void* q_out,
                            const void* k, int64_t k_sb, int64_t k_ss, int64_t k_sh, void* k_out,
                            int64_t B, int64_t S, int64_t Hq, int64_t Hkv, int64_t d,
                            const float* cos, const float* sin, int64_t n_pos, int pairing,
                            int dtype, zk_stream_t stream) {
  ZK_REQUIRE(dtype == ZK_BF16 || dtype == ZK_F16, ZK_EDTYPE, "zk_rope_copy: 2-byte dtypes only");
  ZK_REQUIRE(pairing == ZK_ROPE_HALF || pairing == ZK_ROPE_INTERLEAVED, ZK_EINVAL,
             "zk_rope_copy: bad pairing %d", pairing);
  ZK_REQUIRE((d == 64 || d == 128) && B >= 0 && S >= 0 && Hq > 0 && Hkv > 0 &&
                 Hq + Hkv < 65536 && B < 65536 && S < 0x7fffffff,
             ZK_EUNSUPPORTED, "zk_rope_copy: unsupported shape");
  if (B == 0 || S == 0) return ZK_OK;
  ZK_REQUIRE(q && q_out && k && k_out && cos && sin && n_pos >= S, ZK_EINVAL,
             "zk_rope_copy: null pointer or short table");
  const int64_t strides[] = {q_sb, q_ss, q_sh, k_sb, k_ss, k_sh};
  for (int64_t t : strides)
    ZK_REQUIRE(t % 8 == 0, ZK_EALIGN, "zk_rope_copy: strides must be multiples of 8");
  ZK_REQUIRE(aligned(q, 16) && aligned(k, 16) && aligned(q_out, 16) && aligned(k_out, 16) &&
                 aligned(cos, 16) && aligned(sin, 16),
             ZK_EALIGN, "zk_rope_copy: tensors must be 16-byte aligned");
  hipStream_t st = as_stream(stream);
#define ZK_COPY(T, D)                                                                           \
  launch_rope_vec<T, D>(                                                                        \
      pairing, 0,                                                                               \
      RopeRows<T>{(T*)q_out, (const T*)q, S * Hq * d, Hq * d, d, q_sb, q_ss, q_sh},             \
      RopeRows<T>{(T*)k_out, (const T*)k, S * Hkv * d, Hkv * d, d, k_sb, k_ss, k_sh}, B, S, Hq, \
      Hq + Hkv, cos, sin, n_pos, nullptr, st)
  if (dtype == ZK_BF16) {
    if (d == 128) ZK_COPY(bf16, 128); else ZK_COPY(bf16, 64);
  } else {
    if (d == 128) ZK_COPY(f16, 128); else ZK_COPY(f16, 64);
  }
#undef ZK_COPY
  return launch_status("zk_rope_copy");
}
