// Attention of several query rows per sequence (a prompt, or a later chunk
// of one) over the KV cache: hexkv_attend with q_len > 1, but for small calls
// (rows_lead in hexkv_attend.hip).
//
// What bounds it: the decode kernels stream a row's keys once per query row,
// so a prompt of n tokens reads n / 2 times its K and V; a tile of rows that
// share a KV head reads them once, and both products are then large enough
// for the matrix cores, which bound this kernel (a softmax step per score on
// the VALU beside them).
//
// Measured on MI355X against the decode kernels row by row: Llama-3-8B's
// 8192-token layer 760-810 us and 16.9 ms, 700 TFLOP/s of the products
// without the lo halves (1.05 PFLOP/s with them; a library product reaches
// 1.2), matrix cores 55% and VALU 48% busy, LDS 27%; a Llama-2-7B chunk of
// 2 x 611 over 512 keys 55 and 1165 us.
//
// Work split: a workgroup (4 waves) takes ROWS of the q_len * group query
// rows that share one (sequence, KV head) pair, in (position, query head)
// order, so a grouped query's heads share the staged keys and a tile spans
// few positions (little work above the causal diagonal).  Consecutive
// workgroups are different pairs: with the round-robin dispatch a pair's
// tiles meet its K and V in one XCD's L2.  Tiles run from the longest rows
// down.  When the tiles alone leave CUs idle and the rows are few for their
// keys (a short chunk over a long past), the keys are cut into partitions
// merged by combine_kernel as for decode rows (tile_parts).
//
// One wave, 32 query rows (one per lane and half):
//   S^T = K Q^T   v_mfma_f32_32x32x16, K (A) from LDS, Q (B) in registers:
//                 lane (q, h) gets row q's scores of keys 8 i + 4 h + e.
//   softmax       in the log2 domain per lane, one permlane32 exchange for
//                 the maximum, the running maximum moved only when a score
//                 exceeds it by more than kSlack.
//   O^T += V^T P^T the score layout is the B operand as it stands (the
//                 contraction index of a 16-key step is key 4 h + e, then
//                 8 + 4 h + e), V^T (A) comes from row-major LDS by
//                 ds_read_b64_tr_b16 in the same order.  Every probability
//                 enters as hi + lo 16-bit values (about 2^-17 relative for
//                 bf16; 2^-22 for fp16, or 2^-36 of the row's largest),
//                 both products exact in fp32.  (The accumulators take 16
//                 products at a time, in fp32: over 2^20 keys of 2^-25 of
//                 the largest, together 2.7% of the output, they lost a
//                 fifth to a third of it; at 8192 keys the error against 64 bits is the
//                 output's own rounding.)
// A lane's accumulators all belong to its own row, so rescaling and the
// final division need no exchange.
//
// K and V tiles of 16-bit rows are staged through registers into two LDS
// buffers: the loads of tile i + 1 are in flight while tile i computes, one
// barrier per tile.
//
// Masked keys enter the products with probability 0, which is exact as long
// as V is finite.  A wave whose result holds a non-finite value recomputes
// those rows key by key (exact_row), where a masked key is not touched at
// all, so an infinity or NaN in the cache reaches exactly the rows that
// attend it.
#include "hexkv_prefill.h"

#include <algorithm>

namespace hexkv {

constexpr int kTileThreads = 256;
constexpr int kTileWaves = kTileThreads / 64;
static_assert(kTileRows == 32 * kTileWaves, "32 query rows a wave");
constexpr float kLowest = -1e30f;   // finite "minus infinity" of the running maximum

typedef short h4 __attribute__((ext_vector_type(4)));
typedef short h8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) h4 lds_h4;

__device__ __forceinline__ float tile_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Two 16-bit values per probability, and the scale they are held at: with
// the running maximum M at the last move, a score s enters as
// 2^(s - M + kShift), up to 2^(kShift + kSlack) before the maximum moves (all
// in log2 units).  The scale cancels in the division by the row's sum.
template <typename T>
struct Mma32;

template <>
struct Mma32<__bf16> {
  typedef __bf16 v8 __attribute__((ext_vector_type(8)));
  typedef __bf16 v2 __attribute__((ext_vector_type(2)));
  // bf16 has fp32's exponents: no probability is too small, and a larger
  // scale would only bring P V closer to fp32's range.
  static constexpr float kShift = 0.f, kSlack = 8.f;
  __device__ __forceinline__ static f32x16 mma(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
  }
  // (p0, p1) as packed hi and lo pairs: hi by truncation, lo the rounded rest.
  __device__ __forceinline__ static void split(float p0, float p1, unsigned int *hi, unsigned int *lo) {
    const unsigned int u0 = __float_as_uint(p0), u1 = __float_as_uint(p1);
    *hi = __builtin_amdgcn_perm(u1, u0, 0x07060302u);  // the upper halves
    const v2 r = {static_cast<__bf16>(p0 - __uint_as_float(u0 & 0xffff0000u)),
                  static_cast<__bf16>(p1 - __uint_as_float(u1 & 0xffff0000u))};
    *lo = __builtin_bit_cast(unsigned int, r);
  }
};

template <>
struct Mma32<_Float16> {
  typedef _Float16 v8 __attribute__((ext_vector_type(8)));
  typedef _Float16 v2 __attribute__((ext_vector_type(2)));
  // fp16 ends at 2^-24 (rounded: 2^-25), so at scale 1 a probability below
  // 2^-25 of the largest was lost to the product though not to the sum: one
  // high score over 65536 keys just below took the whole output.  At 2^11
  // the loss is below 2^-36 a key (2^-20 over 65536 keys), and 2^(11 + 4)
  // still lies below fp16's 65504.  A smaller slack moves the maximum more
  // often: a Llama-2-7B chunk of 2 x 611 over 512 keys takes 54.8 us with a
  // slack of 8 (scale 2^7), 55.2 with 4 and 56.0 with 2 (2^13).
  static constexpr float kShift = 11.f, kSlack = 4.f;
  __device__ __forceinline__ static f32x16 mma(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
  }
  __device__ __forceinline__ static void split(float p0, float p1, unsigned int *hi, unsigned int *lo) {
    const v2 h = {static_cast<_Float16>(p0), static_cast<_Float16>(p1)};
    const v2 r = {static_cast<_Float16>(p0 - static_cast<float>(h[0])),
                  static_cast<_Float16>(p1 - static_cast<float>(h[1]))};
    *hi = __builtin_bit_cast(unsigned int, h);
    *lo = __builtin_bit_cast(unsigned int, r);
  }
};

__device__ __forceinline__ float other_half_max(float v) {
  return xor_step<32>(v, MaxOp{});
}

// Keys row t of a sequence of `base` keys attends, clamped like row_length of
// the decode kernels.
__device__ __forceinline__ int keys_of(const TileArgs &a, int base, int t) {
  const int len = a.causal ? base - a.q_len + t + 1 : base;
  return min(len, a.max_seqlen);
}

// Row (position t, query head qh) over keys [p0, end) by one wave, key by key
// in fp32: lanes hold a key each for the scores, D / 64 outputs each for the
// values.  Used for rows whose tile result is not finite, values past
// fp32's range at the tile's scale among them, so no probability exceeds 1.
template <typename T, int D>
__device__ __forceinline__ void exact_row(const TileArgs &a, int b, int t, int qh, int p0, int end, int nparts, int part) {
  using E = Elem<T>;
  constexpr int DPL = D / 64;
  const int lane = threadIdx.x & 63;
  const int hk = qh / a.group;
  const T *q = static_cast<const T *>(a.q) + b * a.q_bs + t * a.q_rs + static_cast<int64_t>(qh) * D;
  const T *kseq = static_cast<const T *>(a.cache) + b * a.c_bs + static_cast<int64_t>(hk) * D;
  const T *vseq = kseq + a.c_kv;
  float m = kLowest, l = 0.f, o[DPL];
#pragma unroll
  for (int e = 0; e < DPL; ++e) o[e] = 0.f;
#pragma unroll 1
  for (int k0 = p0; k0 < end; k0 += 64) {
    const int pos = min(k0 + lane, end - 1);
    float s = 0.f;
#pragma unroll 1
    for (int c = 0; c < D; c += 8)
      s = E::dot(*reinterpret_cast<const u32x4 *>(q + c),
                 *reinterpret_cast<const u32x4 *>(kseq + static_cast<int64_t>(pos) * a.c_ps + c), s);
    if (k0 + lane >= end) s = -INFINITY;
    const float mt = wave_max(s) * a.scale_log2;
    if (mt > m) {
      const float c = tile_exp2(m - mt);
      m = mt;
      l *= c;
#pragma unroll
      for (int e = 0; e < DPL; ++e) o[e] *= c;
    }
    const float p = tile_exp2(fmaf(s, a.scale_log2, -m));
    l += p;
    const int n = min(64, end - k0);
#pragma unroll 1
    for (int j = 0; j < n; ++j) {
      const float pj = __shfl(p, j);
      const T *v = vseq + static_cast<int64_t>(k0 + j) * a.c_ps + lane * DPL;
#pragma unroll
      for (int e = 0; e < DPL; ++e) o[e] = fmaf(pj, static_cast<float>(v[e]), o[e]);
    }
  }
  l = sum_from<1>(l);
  if (nparts == 1) {
    T *out = static_cast<T *>(a.out) + b * a.o_bs + t * a.o_rs + static_cast<int64_t>(qh) * D + lane * DPL;
    const float inv = 1.f / l;
#pragma unroll
    for (int e = 0; e < DPL; ++e) out[e] = E::from_float(o[e] * inv);
  } else {
    const int64_t slot = ((static_cast<int64_t>(b) * a.q_len + t) * a.q_heads + qh) * a.max_parts + part;
#pragma unroll
    for (int e = 0; e < DPL; ++e) a.ws_o[slot * D + lane * DPL + e] = o[e];
    if (lane == 0) *reinterpret_cast<float2 *>(a.ws_ml + slot * 2) = float2{m, l};
  }
}

template <typename T, int D>
__global__ __launch_bounds__(kTileThreads, 2) void attend_tile_kernel(const TileArgs a) {
  using M = Mma32<T>;
  constexpr int ROWS = kTileRows;
  constexpr int NKB = 2;                  // 32-key blocks per tile
  constexpr int KT = 32 * NKB;            // keys per tile
  constexpr int NJ = D / 16;              // score k-steps
  constexpr int ND = D / 32;              // output blocks of 32 dims
  constexpr int CH = D / 8;               // 16-byte chunks per head row
  constexpr int CPT = KT * CH / kTileThreads;
  constexpr int KP = 2 * D + 16;          // LDS bytes per K row: 16 rows' chunks over all banks
  constexpr int VP = 2 * D + 64;          // per V row: the 4 rows of a transposed read over all banks
  static_assert(KT * CH % kTileThreads == 0, "the tile splits over the workgroup");
  __shared__ __attribute__((aligned(16))) char s_k[2][KT * KP];
  __shared__ __attribute__((aligned(16))) char s_v[2][KT * VP];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int c = lane & 31, h = lane >> 5;
  const int pair = static_cast<int>(blockIdx.x % static_cast<unsigned>(a.pairs));
  const int rest = static_cast<int>(blockIdx.x / static_cast<unsigned>(a.pairs));
  const int part = rest % a.max_parts;
  const int tile = a.tiles - 1 - rest / a.max_parts;
  const int b = pair / a.kv_heads, hk = pair - b * a.kv_heads;
  const int base = (a.seqlens ? a.seqlens[b] : 0) + a.bias;
  const int total = a.q_len * a.group;
  const int row0 = tile * ROWS;
  const int p0 = part * a.part;

  // The workgroup's longest row bounds the keys it walks.
  const int t_last = (min(row0 + ROWS, total) - 1) / a.group;
  if (tid == 0 && part == 0 && (a.causal ? base - a.q_len + t_last + 1 : base) > a.max_seqlen)
    raise_status(a.status, HEXKV_STATUS_LENGTH_CLAMPED);
  const int wg_end = min(keys_of(a, base, t_last), p0 + a.part);
  if (part > 0 && wg_end <= p0) return;

  // This wave's rows and this lane's; rows past the last repeat it.
  const int wrow0 = row0 + wave * 32;
  const bool live = wrow0 + c < total;
  const int row = min(wrow0 + c, total - 1);
  const int t = row / a.group, qh = hk * a.group + row - t * a.group;
  const int len = keys_of(a, base, t);
  const int lim = min(len, p0 + a.part);  // keys [p0, lim) are this lane's
  // Keys the wave walks, and those below which none of its rows masks; a wave
  // without rows (the last tile of a pair) only stages.
  const bool idle = wrow0 >= total;
  const int w_end = idle ? p0 : min(keys_of(a, base, (min(wrow0 + 32, total) - 1) / a.group), p0 + a.part);
  const int w_full = idle ? p0 : min(keys_of(a, base, wrow0 / a.group), p0 + a.part);

  u32x4 qf[NJ];
  {
    const T *q = static_cast<const T *>(a.q) + b * a.q_bs + t * a.q_rs + static_cast<int64_t>(qh) * D + h * 8;
#pragma unroll
    for (int j = 0; j < NJ; ++j) qf[j] = *reinterpret_cast<const u32x4 *>(q + j * 16);
  }
  const char *kseq = static_cast<const char *>(a.cache) +
                     (b * a.c_bs + static_cast<int64_t>(hk) * D) * static_cast<int64_t>(sizeof(T));
  const char *vseq = kseq + a.c_kv * static_cast<int64_t>(sizeof(T));
  const uint32_t row_bytes = static_cast<uint32_t>(a.c_ps * sizeof(T));
  const float scale = a.scale_log2;

  float m = kLowest, l = 0.f;  // m: the running maximum less kShift
  f32x16 acc[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d) acc[d] = f32x16{};

  // Staging: thread tid moves chunk tid % CH of rows tid / CH + k * (threads / CH).
  const int s_row = tid / CH, s_ch = tid % CH;
  u32x4 kr[CPT], vr[CPT];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      // past the last key: that key again (finite or not, it is masked)
      const int pos = min(k0 + s_row + i * (kTileThreads / CH), wg_end - 1);
      const uint32_t off = static_cast<uint32_t>(pos) * row_bytes + static_cast<uint32_t>(s_ch) * 16u;
      kr[i] = *reinterpret_cast<const u32x4 *>(kseq + off);
      vr[i] = *reinterpret_cast<const u32x4 *>(vseq + off);
    }
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int r = s_row + i * (kTileThreads / CH);
      *reinterpret_cast<u32x4 *>(&s_k[buf][r * KP + s_ch * 16]) = kr[i];
      *reinterpret_cast<u32x4 *>(&s_v[buf][r * VP + s_ch * 16]) = vr[i];
    }
  };
  const uint32_t k_read = static_cast<uint32_t>(c * KP + h * 16);
  const int s16 = lane & 15;
  const uint32_t v_read = static_cast<uint32_t>((4 * h + s16 / 4) * VP + ((lane >> 4) & 1) * 32 + (s16 % 4) * 8);

  auto compute = [&](int buf, int k0, auto masked) {
    constexpr bool MASK = decltype(masked)::value;
    f32x16 s[NKB];
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb) {
      s[kb] = f32x16{};
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        s[kb] = M::mma(*reinterpret_cast<const u32x4 *>(&s_k[buf][kb * 32 * KP + k_read + j * 32]), qf[j], s[kb]);
    }
    if constexpr (MASK) {
      const int left = lim - k0 - 4 * h;
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          s[kb][i] = kb * 32 + 8 * (i / 4) + i % 4 < left ? s[kb][i] : -INFINITY;
    }
    float mt = s[0][0];
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
      for (int i = 0; i < 16; ++i) mt = fmaxf(mt, s[kb][i]);
    mt = other_half_max(mt) * scale;
    const bool up = mt > m + (M::kShift + M::kSlack);
    if (__any(up)) {
      const float mnew = up ? mt - M::kShift : m;
      const float f = tile_exp2(m - mnew);
      m = mnew;
      l *= f;
#pragma unroll
      for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[d][i] *= f;
    }
    // The tile's sum first: a probability alone may be below half a spacing of l.
    float l0 = 0.f, l1 = 0.f;
    u32x4 hi[2 * NKB], lo[2 * NKB];
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
      for (int i = 0; i < 16; i += 2) {
        const float e0 = tile_exp2(fmaf(s[kb][i], scale, -m)), e1 = tile_exp2(fmaf(s[kb][i + 1], scale, -m));
        l0 += e0;
        l1 += e1;
        unsigned int x, y;
        M::split(e0, e1, &x, &y);
        hi[2 * kb + i / 8][i % 8 / 2] = x;
        lo[2 * kb + i / 8][i % 8 / 2] = y;
      }
    l += l0 + l1;
#pragma unroll
    for (int ks = 0; ks < 2 * NKB; ++ks)
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        const uint32_t at = static_cast<uint32_t>(buf * KT * VP + ks * 16 * VP + d * 64) + v_read;
        auto *shared = (__attribute__((address_space(3))) char *)&s_v[0][0];
        const h4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_h4 *)(shared + at));
        const h4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_h4 *)(shared + at + 8 * VP));
        const u32x4 v = __builtin_bit_cast(u32x4, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
        acc[d] = M::mma(v, hi[ks], acc[d]);
        acc[d] = M::mma(v, lo[ks], acc[d]);
      }
  };

  if (wg_end > p0) {
    fetch(p0);
    stage(0);
    __syncthreads();
    int buf = 0;
    for (int k0 = p0; k0 < wg_end; k0 += KT) {
      const bool more = k0 + KT < wg_end;
      if (more) fetch(k0 + KT);
      if (k0 + KT <= w_full) compute(buf, k0, std::false_type{});
      else if (k0 < w_end) compute(buf, k0, std::true_type{});
      if (more) stage(buf ^ 1);
      buf ^= 1;
      __syncthreads();
    }
  }

  if (idle) return;
  l = xor_step<32>(l, AddOp{});
  const int nparts = len > 0 ? (len + a.part - 1) / a.part : 0;
  const bool holds = live && (part == 0 || lim > p0);  // this lane's row has something to write
  float check = l * 0.f;
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) check = fmaf(acc[d][i], 0.f, check);
  // Decided for the row, over both lanes that hold its outputs, before either
  // stores: `out` may be `q`, and exact_row reads the row's query again.
  uint64_t redo = __ballot(holds && lim > p0 && !(check == 0.f));
  redo = (redo | redo >> 32) & 0xffffffffu;
  const bool bad = redo >> c & 1;
  if (holds && !bad) {
    if (nparts <= 1) {
      // A row without keys is zero, not its sum times zero: beside rows that
      // attend an infinity its sum of 0 * V is a NaN.
      const float inv = 1.f / l;
      T *out = static_cast<T *>(a.out) + b * a.o_bs + t * a.o_rs + static_cast<int64_t>(qh) * D + 4 * h;
#pragma unroll
      for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          f32x4 o = f32x4{acc[d][4 * i], acc[d][4 * i + 1], acc[d][4 * i + 2], acc[d][4 * i + 3]} * inv;
          if (len <= 0) o = f32x4{};
          store4(out + d * 32 + i * 8, o);
        }
    } else {
      const int64_t slot = ((static_cast<int64_t>(b) * a.q_len + t) * a.q_heads + qh) * a.max_parts + part;
      float *o = a.ws_o + slot * D + 4 * h;
#pragma unroll
      for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          *reinterpret_cast<f32x4 *>(o + d * 32 + i * 8) =
              f32x4{acc[d][4 * i], acc[d][4 * i + 1], acc[d][4 * i + 2], acc[d][4 * i + 3]};
      if (h == 0) *reinterpret_cast<float2 *>(a.ws_ml + slot * 2) = float2{m, l};
    }
  }
  while (redo) {
    const int r = __builtin_ctzll(redo);
    redo &= redo - 1;
    exact_row<T, D>(a, b, __shfl(t, r), __shfl(qh, r), p0, __shfl(lim, r), __shfl(nparts, r), part);
  }
}

bool tiles_support(int dtype, int head_dim) {
  return (dtype == HEXKV_F16 || dtype == HEXKV_BF16) && (head_dim == 64 || head_dim == 128);
}

template <typename T, int D>
static void launch_tile(const TileArgs &a, dim3 grid, hipStream_t s) {
  attend_tile_kernel<T, D><<<grid, kTileThreads, 0, s>>>(a);
}

int launch_tiles(TileArgs a, int dtype, int head_dim, int64_t batch, hipStream_t s, const char *what) {
  if (!tiles_support(dtype, head_dim)) return fail(HEXKV_EUNSUPPORTED, "%s: no tile kernel for head_dim %d", what, head_dim);
  const int64_t rows = static_cast<int64_t>(a.q_len) * a.group;
  const int64_t tiles = (rows + kTileRows - 1) / kTileRows, pairs = batch * a.kv_heads;
  if (rows > INT32_MAX || pairs * tiles * a.max_parts >= INT64_C(1) << 24)
    return fail(HEXKV_ERANGE, "%s: 2^24 row tiles or more", what);
  a.pairs = static_cast<int32_t>(pairs);
  a.tiles = static_cast<int32_t>(tiles);
  const dim3 grid(static_cast<unsigned>(pairs * tiles * a.max_parts));
  if (dtype == HEXKV_BF16) {
    if (head_dim == 128) launch_tile<__bf16, 128>(a, grid, s);
    else launch_tile<__bf16, 64>(a, grid, s);
  } else {
    if (head_dim == 128) launch_tile<_Float16, 128>(a, grid, s);
    else launch_tile<_Float16, 64>(a, grid, s);
  }
  return HEXKV_OK;
}

}  // namespace hexkv
