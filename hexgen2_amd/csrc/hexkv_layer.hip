// The elementwise and normalising steps between a decoder layer's matrix
// products: hexkv_add_rms_norm, hexkv_rope_split and hexkv_silu_mul.
//
// What bounds them: at decode each moves a few KB, so its launch is its cost,
// and a layer written as separate tensor operations is a chain of about 55
// launches of which 45 are these steps (a norm is 9, a rotation 12).  One
// kernel per step leaves ten launches a layer.  At a prompt they are bound by
// memory: every element is read once and written once, in 16-byte vectors.
// Measured on MI355X with a 4-layer model of TinyLlama's width (512-token
// prompt, handoff and three decode steps; q/k/v and gate/up each one product
// as well): 7.33 ms as separate operations, 2.52 ms with the three above the
// few-token products.
//
// Each row is one token; a workgroup takes a row (a piece of it where a row
// is long), so a one-token step still has its row spread over 256 lanes.
#include "hexkv_common.h"

namespace hexkv {

constexpr int kLayerThreads = 256;
constexpr int kLayerWaves = kLayerThreads / 64;

// VEC consecutive elements of T as one load or store.
template <typename T, int VEC>
struct alignas(sizeof(T) * VEC) Pack {
  T e[VEC];
};

// out = rms_norm(h + y) * weight; h + y, rounded to T, is kept in h_out.  The
// roundings are those of the separate operations (sum to T; normalised value
// to T; product to T).  NV: vectors of the row a lane keeps in registers; 0:
// any length, the row is read twice.
struct NormArgs {
  const void *h, *y, *weight;
  void *h_out, *out;
  int64_t h_stride, y_stride, h_out_stride;  // elements between rows; out rows are contiguous
  int32_t hidden;
  float eps;
};

template <typename T, int VEC>
__device__ __forceinline__ Pack<T, VEC> norm_input(const NormArgs &a, int64_t row, int i) {
  using P = Pack<T, VEC>;
  P v = *reinterpret_cast<const P *>(static_cast<const T *>(a.h) + row * a.h_stride + i);
  if (a.y) {
    const P y = *reinterpret_cast<const P *>(static_cast<const T *>(a.y) + row * a.y_stride + i);
#pragma unroll
    for (int k = 0; k < VEC; ++k)
      v.e[k] = Elem<T>::from_float(static_cast<float>(v.e[k]) + static_cast<float>(y.e[k]));
  }
  return v;
}

template <typename T, int VEC>
__device__ __forceinline__ Pack<T, VEC> norm_scale(const Pack<T, VEC> &v, const Pack<T, VEC> &w, float r) {
  Pack<T, VEC> o;
#pragma unroll
  for (int k = 0; k < VEC; ++k) {
    const T n = Elem<T>::from_float(static_cast<float>(v.e[k]) * r);
    o.e[k] = Elem<T>::from_float(static_cast<float>(n) * static_cast<float>(w.e[k]));
  }
  return o;
}

template <typename T, int VEC, int NV>
__global__ __launch_bounds__(kLayerThreads) void add_rms_norm_kernel(const NormArgs a) {
  using P = Pack<T, VEC>;
  constexpr int STEP = kLayerThreads * VEC;
  __shared__ float s_sum[kLayerWaves];
  const int64_t row = blockIdx.x;
  const int i0 = static_cast<int>(threadIdx.x) * VEC;
  T *keep = a.h_out ? static_cast<T *>(a.h_out) + row * a.h_out_stride : nullptr;
  P x[NV > 0 ? NV : 1];
  float sum = 0.f;
  auto add = [&](const P &v, int i) {
    if (keep) *reinterpret_cast<P *>(keep + i) = v;
#pragma unroll
    for (int k = 0; k < VEC; ++k) sum = fmaf(static_cast<float>(v.e[k]), static_cast<float>(v.e[k]), sum);
  };
  if constexpr (NV > 0) {
#pragma unroll
    for (int n = 0; n < NV; ++n)
      if (i0 + n * STEP < a.hidden) x[n] = norm_input<T, VEC>(a, row, i0 + n * STEP);
#pragma unroll
    for (int n = 0; n < NV; ++n)
      if (i0 + n * STEP < a.hidden) add(x[n], i0 + n * STEP);
  } else {
    for (int i = i0; i < a.hidden; i += STEP) add(norm_input<T, VEC>(a, row, i), i);
  }
  sum = sum_from<1>(sum);
  if ((threadIdx.x & 63) == 0) s_sum[threadIdx.x >> 6] = sum;
  __syncthreads();
  float total = 0.f;
#pragma unroll
  for (int w = 0; w < kLayerWaves; ++w) total += s_sum[w];
  const float r = rsqrtf(total / static_cast<float>(a.hidden) + a.eps);
  T *out = static_cast<T *>(a.out) + row * a.hidden;
  auto scale = [&](const P &v, int i) {
    const P w = *reinterpret_cast<const P *>(static_cast<const T *>(a.weight) + i);
    *reinterpret_cast<P *>(out + i) = norm_scale<T, VEC>(v, w, r);
  };
  if constexpr (NV > 0) {
#pragma unroll
    for (int n = 0; n < NV; ++n)
      if (i0 + n * STEP < a.hidden) scale(x[n], i0 + n * STEP);
  } else {
    // h_out may be h itself, which then holds the sum already: take it from
    // there (this lane wrote it), not from h and y again.
    for (int i = i0; i < a.hidden; i += STEP) {
      if (keep) scale(*reinterpret_cast<const P *>(keep + i), i);
      else scale(norm_input<T, VEC>(a, row, i), i);
    }
  }
}

// qkv rows [q heads | k heads | v heads] -> q [rows][q_heads][D] and
// kv [rows][2][kv_heads][D], q and k turned (GPT-NeoX halves) at the row's
// position.  The angle is the fp32 product of position and inv_freq, its
// sine and cosine and the turn are fp32, and the result is rounded to T once.
struct RopeArgs {
  const void *qkv;
  void *q, *kv;
  const float *inv_freq;     // [D / 2]
  const int32_t *positions;  // per sequence, or nullptr: offset + index in the sequence
  int64_t qkv_stride;        // elements between rows
  int32_t q_heads, kv_heads, head_dim, seqlen, offset;
};

template <typename T, int VEC>
__global__ __launch_bounds__(kLayerThreads) void rope_split_kernel(const RopeArgs a) {
  using P = Pack<T, VEC>;
  const int64_t row = blockIdx.x;
  const int unit = static_cast<int>(blockIdx.y * kLayerThreads + threadIdx.x);
  const int D = a.head_dim, half = D / 2, per = half / VEC;  // units of one rotated head
  const int turned = (a.q_heads + a.kv_heads) * per;
  const T *src = static_cast<const T *>(a.qkv) + row * a.qkv_stride;
  T *q = static_cast<T *>(a.q) + row * a.q_heads * D;
  T *kv = static_cast<T *>(a.kv) + row * 2 * a.kv_heads * D;
  if (unit < turned) {
    const int head = unit / per, j = (unit - head * per) * VEC;
    const P x0 = *reinterpret_cast<const P *>(src + head * D + j);
    const P x1 = *reinterpret_cast<const P *>(src + head * D + half + j);
    const int64_t b = row / a.seqlen;
    const float pos = a.positions ? static_cast<float>(a.positions[b])
                                  : static_cast<float>(a.offset + static_cast<int32_t>(row - b * a.seqlen));
    P y0, y1;
#pragma unroll
    for (int k = 0; k < VEC; ++k) {
      float sn, cs;
      sincosf(pos * a.inv_freq[j + k], &sn, &cs);
      const float u = static_cast<float>(x0.e[k]), v = static_cast<float>(x1.e[k]);
      y0.e[k] = Elem<T>::from_float(u * cs - v * sn);
      y1.e[k] = Elem<T>::from_float(v * cs + u * sn);
    }
    T *dst = head < a.q_heads ? q + head * D : kv + (head - a.q_heads) * D;
    *reinterpret_cast<P *>(dst + j) = y0;
    *reinterpret_cast<P *>(dst + half + j) = y1;
    return;
  }
  const int i = (unit - turned) * VEC;
  if (i < a.kv_heads * D)
    *reinterpret_cast<P *>(kv + a.kv_heads * D + i) =
        *reinterpret_cast<const P *>(src + (a.q_heads + a.kv_heads) * D + i);
}

// out[r][i] = silu(gate_up[r][i]) * gate_up[r][width + i], fp32 inside and
// rounded once.
template <typename T, int VEC>
__global__ __launch_bounds__(kLayerThreads) void silu_mul_kernel(const T *__restrict__ gate_up, T *__restrict__ out,
                                                                int32_t width) {
  using P = Pack<T, VEC>;
  const int64_t row = blockIdx.x;
  const int64_t i = (static_cast<int64_t>(blockIdx.y) * kLayerThreads + threadIdx.x) * VEC;
  if (i >= width) return;
  const P g = *reinterpret_cast<const P *>(gate_up + row * 2 * width + i);
  const P u = *reinterpret_cast<const P *>(gate_up + (row * 2 + 1) * width + i);
  P o;
#pragma unroll
  for (int k = 0; k < VEC; ++k) {
    const float x = static_cast<float>(g.e[k]);
    o.e[k] = Elem<T>::from_float(x / (1.f + expf(-x)) * static_cast<float>(u.e[k]));
  }
  *reinterpret_cast<P *>(out + row * width + i) = o;
}

// ------------------------------------------------- few-token products ---
//
// norm_linear_kernel: out = x W^T for up to kLinearRows tokens, x = h or
// rms_norm(h + y) * weight, out = x W^T or silu(gate) * up of its two halves.
//
// What bounds it: a few tokens use each weight once or a few times, so the
// product streams W; at the sizes of one layer (8-50 MB) a launch's ramp and
// the latency of that stream count as much as its bytes.  Every wave owns R
// rows of W (R gate and R up rows), issues its first loads of them before it
// looks at x, and keeps the next ones in flight; x is staged in LDS by each
// workgroup for itself, which costs it the norm again (4-8 KB from the L2,
// while W arrives) and saves the norm's launch.  The dot products run on the
// VALU with fp32 sums: at this few tokens the matrix cores would wait for W
// just the same.
//
// Measured on MI355X in fp16, one token, against the norm, the library's
// product and the SwiGLU as launches of their own: 64 -> 64 with norm 2.7 and
// 4.6 us, 2048 -> 2560 with norm 4.8 and 10.1, 2048 -> 2 x 5632 with norm and
// SwiGLU 10.0 and 19.3, 5632 -> 2048 7.3 and 10.5, 4096 -> 2 x 14336 36.9 and
// 40.3 (6.4 TB/s), 4096 -> 32000 with norm 40.3 and 42.8 (6.5 TB/s); with the
// heads split and turned in it as well the model call of the head comment
// goes from 1.48 to 1.41 ms.  Two tokens take 5-25% longer, the library's no
// longer.  Of 110 products of one and two tokens in fp16, bf16 and fp32 (64 to
// 14336 -> 64 to 128256, plain and with norm) four lose to the library, by
// 3-9%: 4096 -> 28672 without norm, 4096 -> 32000 with norm and two tokens in
// fp16 (45.4 and 43.2), 14336 -> 4096 in fp32 without norm (38.4 and 35.2).
// The line is at two tokens for want of instances beyond: with four, norm and
// 4096 -> 12288 took 27.9 and 23.8, and three, or the small products where
// the kernel leads most, were not measured.
constexpr int kLinearRows = 2;
constexpr int64_t kLinearLds = INT64_C(64) << 10;  // x in LDS: two workgroups a CU at least

struct LinearArgs {
  NormArgs norm;  // h, y, weight (nullptr: x = h), h_out
  const void *w;  // [n][hidden], or [2 n][hidden] gate then up
  void *out;      // [rows][n]
  int32_t n;
  RopeArgs rope;  // kLinearRope: w is the q, k and v heads, n their pairs of dimensions
};

// What becomes of the two rows of W that a wave takes together.
enum LinearKind {
  kLinearPlain,  // one row: its product
  kLinearGlu,    // gate i, up i: silu(gate) * up
  kLinearRope,   // dimensions j and j + D / 2 of a head: turned (q, k) or not (v)
};

template <typename T, int M, int R, int KIND>
__global__ __launch_bounds__(kLayerThreads) void norm_linear_kernel(const LinearArgs a) {
  using E = Elem<T>;
  constexpr int VEC = 16 / static_cast<int>(sizeof(T));
  using P = Pack<T, VEC>;
  constexpr int U = 4, RW = KIND == kLinearPlain ? R : 2 * R, KSTEP = U * 64 * VEC;
  extern __shared__ __attribute__((aligned(16))) char s_raw[];
  __shared__ float s_sum[M][kLayerWaves];
  T *s_x = reinterpret_cast<T *>(s_raw);  // [rows][K]
  const int K = a.norm.hidden, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n0 = (static_cast<int>(blockIdx.x) * kLayerWaves + wave) * R;

  // Rows past the last one repeat it (loaded in bounds, not stored).
  const T *wrow[RW];
#pragma unroll
  for (int r = 0; r < RW; ++r) {
    int64_t n = min(n0 + r % R, a.n - 1);
    if constexpr (KIND == kLinearRope) {
      const int half = a.rope.head_dim / 2;
      n += n / half * half + (r >= R ? half : 0);
    } else {
      n += r >= R ? a.n : 0;
    }
    wrow[r] = static_cast<const T *>(a.w) + n * K + lane * VEC;
  }
  using Tile = u32x4[RW][U];
  auto fetch = [&](int k0, Tile &t) {
#pragma unroll
    for (int r = 0; r < RW; ++r)
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = k0 + u * 64 * VEC;
        t[r][u] = u32x4{};
        if (k + lane * VEC < K) t[r][u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(wrow[r] + k));
      }
  };
  Tile cur;
  fetch(0, cur);

  const int i0 = static_cast<int>(threadIdx.x) * VEC;
  for (int m = 0; m < M; ++m) {
    T *keep = a.norm.h_out && blockIdx.x == 0 ? static_cast<T *>(a.norm.h_out) + m * a.norm.h_out_stride : nullptr;
    float sum = 0.f;
    for (int i = i0; i < K; i += kLayerThreads * VEC) {
      const P v = norm_input<T, VEC>(a.norm, m, i);
      *reinterpret_cast<P *>(s_x + static_cast<int64_t>(m) * K + i) = v;
      if (keep) *reinterpret_cast<P *>(keep + i) = v;
#pragma unroll
      for (int k = 0; k < VEC; ++k) sum = fmaf(static_cast<float>(v.e[k]), static_cast<float>(v.e[k]), sum);
    }
    sum = sum_from<1>(sum);
    if (lane == 0) s_sum[m][wave] = sum;
  }
  __syncthreads();
  if (a.norm.weight) {
    for (int m = 0; m < M; ++m) {
      float total = 0.f;
#pragma unroll
      for (int w = 0; w < kLayerWaves; ++w) total += s_sum[m][w];
      const float r = rsqrtf(total / static_cast<float>(K) + a.norm.eps);
      for (int i = i0; i < K; i += kLayerThreads * VEC) {
        P *x = reinterpret_cast<P *>(s_x + static_cast<int64_t>(m) * K + i);
        *x = norm_scale<T, VEC>(*x, *reinterpret_cast<const P *>(static_cast<const T *>(a.norm.weight) + i), r);
      }
    }
    __syncthreads();
  }

  float acc[M][RW];
#pragma unroll
  for (int m = 0; m < M; ++m)
#pragma unroll
    for (int r = 0; r < RW; ++r) acc[m][r] = 0.f;
  auto consume = [&](int k0, const Tile &t) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + u * 64 * VEC + lane * VEC;
      if (k >= K) continue;  // its weights are zero
#pragma unroll
      for (int m = 0; m < M; ++m) {
        const u32x4 x = *reinterpret_cast<const u32x4 *>(s_x + static_cast<int64_t>(m) * K + k);
#pragma unroll
        for (int r = 0; r < RW; ++r) acc[m][r] = E::dot(x, t[r][u], acc[m][r]);
      }
    }
  };
  int k0 = 0;
  for (; k0 + KSTEP < K; k0 += KSTEP) {
    Tile next;
    fetch(k0 + KSTEP, next);
    consume(k0, cur);
#pragma unroll
    for (int r = 0; r < RW; ++r)
#pragma unroll
      for (int u = 0; u < U; ++u) cur[r][u] = next[r][u];
  }
  consume(k0, cur);

#pragma unroll
  for (int m = 0; m < M; ++m) {
#pragma unroll
    for (int r = 0; r < RW; ++r) acc[m][r] = sum_from<1>(acc[m][r]);
    if (lane != 0) continue;
    if constexpr (KIND == kLinearRope) {
      const RopeArgs &p = a.rope;
      const int half = p.head_dim / 2, b = m / p.seqlen;
      const float pos = static_cast<float>(p.positions ? p.positions[b] : p.offset + m - b * p.seqlen);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if (n0 + r >= a.n) continue;
        const int head = (n0 + r) / half, j = n0 + r - head * half;
        float x0 = acc[m][r], x1 = acc[m][R + r];
        if (head < p.q_heads + p.kv_heads) {
          float sn, cs;
          sincosf(pos * p.inv_freq[j], &sn, &cs);
          const float u = x0, v = x1;
          x0 = u * cs - v * sn;
          x1 = v * cs + u * sn;
        }
        T *dst = head < p.q_heads
                     ? static_cast<T *>(p.q) + (static_cast<int64_t>(m) * p.q_heads + head) * p.head_dim
                     : static_cast<T *>(p.kv) + (static_cast<int64_t>(m) * 2 * p.kv_heads + head - p.q_heads) * p.head_dim;
        dst[j] = E::from_float(x0);
        dst[j + half] = E::from_float(x1);
      }
    } else {
      T *out = static_cast<T *>(a.out) + static_cast<int64_t>(m) * a.n;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        float v = acc[m][r];
        if constexpr (KIND == kLinearGlu) v = v / (1.f + expf(-v)) * acc[m][R + r];
        if (n0 + r < a.n) out[n0 + r] = E::from_float(v);
      }
    }
  }
}

// ------------------------------------------------------------------ host ---

static int dtype_size(int dtype, const char *what, int *es) {
  if (dtype != HEXKV_F16 && dtype != HEXKV_BF16 && dtype != HEXKV_F32)
    return fail(HEXKV_EINVAL, "%s: unknown dtype %d", what, dtype);
  *es = dtype == HEXKV_F32 ? 4 : 2;
  return HEXKV_OK;
}

static int check_rows(int64_t rows, const char *what) {
  if (rows < 0) return fail(HEXKV_EINVAL, "%s: negative row count", what);
  // One workgroup of 256 lanes per row, and a launch holds below 2^32 lanes.
  if (rows >= INT64_C(1) << 24) return fail(HEXKV_ERANGE, "%s: 2^24 rows or more", what);
  return HEXKV_OK;
}

template <typename T>
static void launch_norm(const NormArgs &a, bool vec16, int64_t rows, hipStream_t s) {
  constexpr int VEC = 16 / static_cast<int>(sizeof(T));
  const dim3 grid(static_cast<unsigned>(rows));
  const int64_t vectors = vec16 ? (a.hidden / VEC + kLayerThreads - 1) / kLayerThreads : 0;
  if (!vec16) add_rms_norm_kernel<T, 1, 0><<<grid, kLayerThreads, 0, s>>>(a);
  else if (vectors <= 1) add_rms_norm_kernel<T, VEC, 1><<<grid, kLayerThreads, 0, s>>>(a);
  else if (vectors <= 2) add_rms_norm_kernel<T, VEC, 2><<<grid, kLayerThreads, 0, s>>>(a);
  else if (vectors <= 4) add_rms_norm_kernel<T, VEC, 4><<<grid, kLayerThreads, 0, s>>>(a);
  else add_rms_norm_kernel<T, VEC, 0><<<grid, kLayerThreads, 0, s>>>(a);
}

template <typename T>
static void launch_rope(const RopeArgs &a, bool vec16, int64_t rows, hipStream_t s) {
  constexpr int VEC = 16 / static_cast<int>(sizeof(T));
  const int vec = vec16 ? VEC : 1;
  const int64_t units = (static_cast<int64_t>(a.q_heads) + a.kv_heads) * (a.head_dim / 2 / vec) +
                        static_cast<int64_t>(a.kv_heads) * a.head_dim / vec;
  const dim3 grid(static_cast<unsigned>(rows), static_cast<unsigned>((units + kLayerThreads - 1) / kLayerThreads));
  if (vec16) rope_split_kernel<T, VEC><<<grid, kLayerThreads, 0, s>>>(a);
  else rope_split_kernel<T, 1><<<grid, kLayerThreads, 0, s>>>(a);
}

template <typename T>
static void launch_silu(const void *gate_up, void *out, bool vec16, int64_t rows, int32_t width, hipStream_t s) {
  constexpr int VEC = 16 / static_cast<int>(sizeof(T));
  const int64_t per = static_cast<int64_t>(kLayerThreads) * (vec16 ? VEC : 1);
  const dim3 grid(static_cast<unsigned>(rows), static_cast<unsigned>((width + per - 1) / per));
  if (vec16) silu_mul_kernel<T, VEC><<<grid, kLayerThreads, 0, s>>>(static_cast<const T *>(gate_up), static_cast<T *>(out), width);
  else silu_mul_kernel<T, 1><<<grid, kLayerThreads, 0, s>>>(static_cast<const T *>(gate_up), static_cast<T *>(out), width);
}

template <typename T, int M, int KIND>
static void launch_linear(const LinearArgs &a, hipStream_t s) {
  const size_t lds = static_cast<size_t>(M) * a.norm.hidden * sizeof(T);
  // Two rows (or pairs) a wave once that still gives every CU a workgroup.
  const int R = a.n >= 2048 ? 2 : 1;
  const dim3 grid(static_cast<unsigned>((a.n + kLayerWaves * R - 1) / (kLayerWaves * R)));
  if (R == 2) norm_linear_kernel<T, M, 2, KIND><<<grid, kLayerThreads, lds, s>>>(a);
  else norm_linear_kernel<T, M, 1, KIND><<<grid, kLayerThreads, lds, s>>>(a);
}

template <typename T, int KIND>
static void dispatch_rows_of(const LinearArgs &a, int rows, hipStream_t s) {
  static_assert(kLinearRows == 2, "one instance per row count");
  if (rows == 1) launch_linear<T, 1, KIND>(a, s);
  else launch_linear<T, 2, KIND>(a, s);
}

template <int KIND>
static void dispatch_linear(const LinearArgs &a, int rows, int dtype, hipStream_t s) {
  switch (dtype) {
    case HEXKV_BF16: dispatch_rows_of<__bf16, KIND>(a, rows, s); break;
    case HEXKV_F16: dispatch_rows_of<_Float16, KIND>(a, rows, s); break;
    default: dispatch_rows_of<float, KIND>(a, rows, s); break;
  }
}

// `n` rows of `bytes` each, `stride` bytes apart.
struct Rows {
  const void *at;
  int64_t n, stride, bytes;
  bool same_as(const Rows &o) const { return at == o.at && (n == 1 || stride == o.stride); }
};

// Whether two sets of rows share a byte.
static bool meet(const Rows &a, const Rows &b) {
  if (!a.at || !b.at || a.n < 1 || b.n < 1) return false;
  const int64_t a0 = reinterpret_cast<intptr_t>(a.at), b0 = reinterpret_cast<intptr_t>(b.at);
  if (a0 + (a.n - 1) * a.stride + a.bytes <= b0 || b0 + (b.n - 1) * b.stride + b.bytes <= a0) return false;
  for (int64_t i = 0; i < a.n; ++i) {
    // rows j of b that start below this row's end and end above its start
    const int64_t lo = a0 + i * a.stride - b0 - b.bytes + 1, hi = a0 + i * a.stride + a.bytes - 1 - b0;
    if (hi < 0) continue;
    if (b.stride == 0 || b.n == 1) {
      if (lo <= 0) return true;
      continue;
    }
    const int64_t first = lo <= 0 ? 0 : (lo + b.stride - 1) / b.stride;
    if (first < b.n && first * b.stride <= hi) return true;
  }
  return false;
}

static int refuse_overlap(const char *out, const char *in, const char *what) {
  return fail(HEXKV_EINVAL, "%s: %s overlaps %s, which other workgroups read or write meanwhile", what, out, in);
}

// The checks that every norm_linear_kernel launch shares.  Every workgroup
// reads all of h and y, and workgroup 0 stores their sum, while others store
// the products: no output may share a byte with an input or another output.
static int check_linear(const NormArgs &a, const Rows &weight, const Rows (&outs)[2], int rows, int es, const char *what) {
  if (a.h_stride < 0 || a.y_stride < 0 || a.h_out_stride < 0) return fail(HEXKV_EINVAL, "%s: negative stride", what);
  const int64_t vec = 16 / es;
  if (rows > kLinearRows || static_cast<int64_t>(rows) * a.hidden * es > kLinearLds)
    return fail(HEXKV_EUNSUPPORTED, "%s: at most %d rows and %lld bytes of them", what, kLinearRows,
                static_cast<long long>(kLinearLds));
  if (a.hidden % vec || a.h_stride % vec || a.y_stride % vec || a.h_out_stride % vec || !aligned16(a.h) ||
      !aligned16(a.y) || !aligned16(a.h_out) || !aligned16(a.weight) || !aligned16(weight.at))
    return fail(HEXKV_EUNSUPPORTED, "%s: rows must be 16-byte aligned and a multiple of 16 bytes", what);
  const int64_t row = static_cast<int64_t>(a.hidden) * es;
  const Rows in[] = {{a.h, rows, a.h_stride * es, row}, {a.y, rows, a.y_stride * es, row}, {a.weight, 1, row, row}, weight};
  const Rows out[] = {{a.h_out, rows, a.h_out_stride * es, row}, outs[0], outs[1]};
  if (a.h_out && rows > 1 && a.h_out_stride < a.hidden) return fail(HEXKV_EINVAL, "%s: h_out's rows overlap", what);
  for (const Rows &o : out)
    for (const Rows &i : in)
      if (meet(o, i)) return refuse_overlap("an output", "an input", what);
  if (meet(out[0], out[1]) || meet(out[0], out[2]) || meet(out[1], out[2]))
    return refuse_overlap("an output", "another", what);
  return HEXKV_OK;
}

}  // namespace hexkv

extern "C" int hexkv_norm_linear(const void *h, int64_t h_stride, const void *y, int64_t y_stride, void *h_out,
                                 int64_t h_out_stride, const void *norm_weight, float eps, const void *weight,
                                 void *out, int rows, int hidden, int n, int glu, int dtype, hexkv_stream_t stream) {
  using namespace hexkv;
  clear_error();
  const char *what = "hexkv_norm_linear";
  int es = 0;
  const int rc = dtype_size(dtype, what, &es);
  if (rc != HEXKV_OK) return rc;
  if (rows < 0 || hidden < 1 || n < 0 || n > 1 << 28) return fail(HEXKV_EINVAL, "%s: bad sizes", what);
  if (rows == 0 || n == 0) return HEXKV_OK;
  if (!h || !weight || !out) return fail(HEXKV_EINVAL, "%s: null tensor", what);
  const LinearArgs a{NormArgs{h, y, norm_weight, h_out, nullptr, h_stride, y_stride, h_out_stride, hidden, eps},
                     weight, out, n, RopeArgs{}};
  const int64_t w_bytes = (glu ? 2 : 1) * static_cast<int64_t>(n) * hidden * es, out_row = static_cast<int64_t>(n) * es;
  const int bad = check_linear(a.norm, Rows{weight, 1, w_bytes, w_bytes}, {Rows{out, rows, out_row, out_row}, Rows{}},
                               rows, es, what);
  if (bad != HEXKV_OK) return bad;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (glu) dispatch_linear<kLinearGlu>(a, rows, dtype, s);
  else dispatch_linear<kLinearPlain>(a, rows, dtype, s);
  return check_launch(what);
}

extern "C" int hexkv_norm_rope_linear(const void *h, int64_t h_stride, const void *y, int64_t y_stride, void *h_out,
                                      int64_t h_out_stride, const void *norm_weight, float eps, const void *weight,
                                      const float *inv_freq_dev, const int32_t *positions_dev, int offset, void *q,
                                      void *kv, int rows, int seqlen, int hidden, int q_heads, int kv_heads,
                                      int head_dim, int dtype, hexkv_stream_t stream) {
  using namespace hexkv;
  clear_error();
  const char *what = "hexkv_norm_rope_linear";
  int es = 0;
  const int rc = dtype_size(dtype, what, &es);
  if (rc != HEXKV_OK) return rc;
  if (rows < 0 || hidden < 1 || q_heads < 1 || kv_heads < 1 || head_dim < 2 || head_dim % 2 || seqlen < 1 || rows % seqlen)
    return fail(HEXKV_EINVAL, "%s: bad sizes", what);
  const int64_t units = (static_cast<int64_t>(q_heads) + 2 * static_cast<int64_t>(kv_heads)) * (head_dim / 2);
  if (units > 1 << 22) return fail(HEXKV_ERANGE, "%s: rows of more than 2^23 elements", what);
  if (offset < 0 || (!positions_dev && offset > INT32_MAX - seqlen))
    return fail(HEXKV_ERANGE, "%s: position offset %d", what, offset);
  if (rows == 0) return HEXKV_OK;
  if (!h || !weight || !inv_freq_dev || !q || !kv) return fail(HEXKV_EINVAL, "%s: null tensor", what);
  const LinearArgs a{NormArgs{h, y, norm_weight, h_out, nullptr, h_stride, y_stride, h_out_stride, hidden, eps},
                     weight, nullptr, static_cast<int32_t>(units),
                     RopeArgs{nullptr, q, kv, inv_freq_dev, positions_dev, 0, q_heads, kv_heads, head_dim, seqlen, offset}};
  const int64_t w_bytes = 2 * units * hidden * es, q_row = static_cast<int64_t>(q_heads) * head_dim * es;
  const int64_t kv_row = 2 * static_cast<int64_t>(kv_heads) * head_dim * es;
  const int bad = check_linear(a.norm, Rows{weight, 1, w_bytes, w_bytes},
                               {Rows{q, rows, q_row, q_row}, Rows{kv, rows, kv_row, kv_row}}, rows, es, what);
  if (bad != HEXKV_OK) return bad;
  dispatch_linear<kLinearRope>(a, rows, dtype, static_cast<hipStream_t>(stream));
  return check_launch(what);
}

extern "C" int hexkv_add_rms_norm(const void *h, int64_t h_stride, const void *y, int64_t y_stride, void *h_out,
                                  int64_t h_out_stride, const void *weight, void *out, int64_t rows, int hidden,
                                  float eps, int dtype, hexkv_stream_t stream) {
  using namespace hexkv;
  clear_error();
  const char *what = "hexkv_add_rms_norm";
  int es = 0, rc = dtype_size(dtype, what, &es);
  if (rc == HEXKV_OK) rc = check_rows(rows, what);
  if (rc != HEXKV_OK) return rc;
  if (hidden < 1 || h_stride < 0 || y_stride < 0 || h_out_stride < 0)
    return fail(HEXKV_EINVAL, "%s: hidden below 1 or a negative stride", what);
  if (rows == 0) return HEXKV_OK;
  if (!h || !weight || !out) return fail(HEXKV_EINVAL, "%s: null tensor", what);
  const NormArgs a{h, y, weight, h_out, out, h_stride, y_stride, h_out_stride, hidden, eps};
  // A workgroup reads its own row and the weight, and each lane writes the
  // elements it read: in place row for row, but over no other row.
  const int64_t row = static_cast<int64_t>(hidden) * es;
  const Rows r_h{h, rows, h_stride * es, row}, r_y{y, rows, y_stride * es, row}, r_w{weight, 1, row, row};
  const Rows r_sum{h_out, rows, h_out_stride * es, row}, r_out{out, rows, row, row};
  if (h_out && rows > 1 && h_out_stride < hidden) return fail(HEXKV_EINVAL, "%s: h_out's rows overlap", what);
  for (const Rows &o : {r_sum, r_out}) {
    if (meet(o, r_w)) return refuse_overlap("an output", "the weight", what);
    for (const Rows &i : {r_h, r_y, r_sum})
      if (!o.same_as(i) && meet(o, i)) return refuse_overlap("an output", "rows of another tensor", what);
  }
  const int64_t vec = 16 / es;
  const bool vec16 = hidden % vec == 0 && h_stride % vec == 0 && y_stride % vec == 0 && h_out_stride % vec == 0 &&
                     aligned16(h) && aligned16(y) && aligned16(h_out) && aligned16(weight) && aligned16(out);
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case HEXKV_BF16: launch_norm<__bf16>(a, vec16, rows, s); break;
    case HEXKV_F16: launch_norm<_Float16>(a, vec16, rows, s); break;
    default: launch_norm<float>(a, vec16, rows, s); break;
  }
  return check_launch(what);
}

extern "C" int hexkv_rope_split(const void *qkv, int64_t qkv_stride, const float *inv_freq_dev,
                                const int32_t *positions_dev, int offset, void *q, void *kv, int64_t rows, int seqlen,
                                int q_heads, int kv_heads, int head_dim, int dtype, hexkv_stream_t stream) {
  using namespace hexkv;
  clear_error();
  const char *what = "hexkv_rope_split";
  int es = 0, rc = dtype_size(dtype, what, &es);
  if (rc == HEXKV_OK) rc = check_rows(rows, what);
  if (rc != HEXKV_OK) return rc;
  if (q_heads < 1 || kv_heads < 1 || head_dim < 2 || head_dim % 2 || seqlen < 1 || rows % seqlen)
    return fail(HEXKV_EINVAL, "%s: bad head counts, head_dim or seqlen", what);
  const int64_t row = (static_cast<int64_t>(q_heads) + 2 * static_cast<int64_t>(kv_heads)) * head_dim;
  if (row > INT64_C(1) << 23) return fail(HEXKV_ERANGE, "%s: rows of more than 2^23 elements", what);
  if (qkv_stride < row) return fail(HEXKV_EINVAL, "%s: rows overlap", what);
  if (offset < 0 || (!positions_dev && offset > INT32_MAX - seqlen))
    return fail(HEXKV_ERANGE, "%s: position offset %d", what, offset);
  if (rows == 0) return HEXKV_OK;
  if (!qkv || !inv_freq_dev || !q || !kv) return fail(HEXKV_EINVAL, "%s: null tensor", what);
  // One row may be split where it stands: a lane writes what it read.
  const int64_t q_row = static_cast<int64_t>(q_heads) * head_dim * es, kv_row = row * es - q_row;
  const Rows r_in{qkv, rows, qkv_stride * es, row * es}, r_q{q, rows, q_row, q_row}, r_kv{kv, rows, kv_row, kv_row};
  if ((!(rows == 1 && q == qkv) && meet(r_q, r_in)) ||
      (!(rows == 1 && kv == static_cast<const char *>(qkv) + q_row) && meet(r_kv, r_in)))
    return refuse_overlap("q or kv", "qkv", what);
  if (meet(r_q, r_kv)) return refuse_overlap("q", "kv", what);
  const RopeArgs a{qkv, q, kv, inv_freq_dev, positions_dev, qkv_stride, q_heads, kv_heads, head_dim, seqlen, offset};
  const int vec = 16 / es;
  const bool vec16 = (head_dim / 2) % vec == 0 && qkv_stride % vec == 0 && aligned16(qkv) && aligned16(q) && aligned16(kv);
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case HEXKV_BF16: launch_rope<__bf16>(a, vec16, rows, s); break;
    case HEXKV_F16: launch_rope<_Float16>(a, vec16, rows, s); break;
    default: launch_rope<float>(a, vec16, rows, s); break;
  }
  return check_launch(what);
}

extern "C" int hexkv_silu_mul(const void *gate_up, void *out, int64_t rows, int width, int dtype,
                              hexkv_stream_t stream) {
  using namespace hexkv;
  clear_error();
  const char *what = "hexkv_silu_mul";
  int es = 0, rc = dtype_size(dtype, what, &es);
  if (rc == HEXKV_OK) rc = check_rows(rows, what);
  if (rc != HEXKV_OK) return rc;
  if (width < 1 || width > 1 << 23) return fail(HEXKV_EINVAL, "%s: width %d outside [1, 2^23]", what, width);
  if (rows == 0) return HEXKV_OK;
  if (!gate_up || !out) return fail(HEXKV_EINVAL, "%s: null tensor", what);
  // One row's result may take the place of its gate or its up half.
  const int64_t half = static_cast<int64_t>(width) * es;
  const char *gate = static_cast<const char *>(gate_up);
  if (!(rows == 1 && (out == gate || out == gate + half)) &&
      meet(Rows{out, rows, half, half}, Rows{gate_up, rows, 2 * half, 2 * half}))
    return refuse_overlap("out", "gate_up", what);
  const bool vec16 = width % (16 / es) == 0 && aligned16(gate_up) && aligned16(out);
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case HEXKV_BF16: launch_silu<__bf16>(gate_up, out, vec16, rows, width, s); break;
    case HEXKV_F16: launch_silu<_Float16>(gate_up, out, vec16, rows, width, s); break;
    default: launch_silu<float>(gate_up, out, vec16, rows, width, s); break;
  }
  return check_launch(what);
}
