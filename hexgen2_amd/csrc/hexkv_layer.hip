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
// as well): 7.33 ms as separate operations, 2.52 ms with these kernels.
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
    P o;
#pragma unroll
    for (int k = 0; k < VEC; ++k) {
      const T n = Elem<T>::from_float(static_cast<float>(v.e[k]) * r);
      o.e[k] = Elem<T>::from_float(static_cast<float>(n) * static_cast<float>(w.e[k]));
    }
    *reinterpret_cast<P *>(out + i) = o;
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

}  // namespace hexkv

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
  const bool vec16 = width % (16 / es) == 0 && aligned16(gate_up) && aligned16(out);
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case HEXKV_BF16: launch_silu<__bf16>(gate_up, out, vec16, rows, width, s); break;
    case HEXKV_F16: launch_silu<_Float16>(gate_up, out, vec16, rows, width, s); break;
    default: launch_silu<float>(gate_up, out, vec16, rows, width, s); break;
  }
  return check_launch(what);
}
