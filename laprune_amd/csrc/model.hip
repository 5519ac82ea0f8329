// model.hip — the element-wise parts of a decode step around the attention
// layers, one launch each.
//
// A decode step of one token per sequence moves a few kilobytes through each of
// these, so a launch is all they cost; as torch runs them, an RMSNorm is eight
// launches, the rotary tables nine and silu(gate) * up two, some 60 of a
// two-layer step's 90 (3 to 4 us each inside a captured graph).  With one launch
// each, and no mask built for one token, that step (2 of Llama-3.1-8B's layers at
// 32k, weights' and cache's reads 404 us) went from 737 to 549 us
// (414 with the projections' own kernels and the last touches below).  The arithmetic
// is that of the model code's tensor ops, rounded to the model dtype where
// they round (transformers' LlamaRMSNorm, LlamaRotaryEmbedding and LlamaMLP):
//   rms_norm     rnd(w * rnd(x * rsqrt(mean(x^2) + eps))), the mean in fp32
//   rope_tables  rnd(cos(pos * inv_freq) * scaling), and sin
//   silu_mul     rnd(rnd(g / (1 + exp(-g))) * u)
//   argmax_rows  first index of the largest value, NaN above all
#include "common.h"

namespace lap {
namespace {

template <int DT>
__device__ __forceinline__ float widen(uint16_t v) {
  return DT == LAP_DTYPE_F16 ? h2f(v) : bf2f(v);
}
template <int DT>
__device__ __forceinline__ uint16_t narrow(float f) {
  return DT == LAP_DTYPE_F16 ? f2h(f) : f2bf(f);
}

// One workgroup per row, eight elements (16 bytes) per thread and pass; a
// row of up to 8192 is read once and kept in registers.
constexpr int kNormThreads = 512, kNormPass = kNormThreads * 8, kNormKeep = 2;

template <int DT>
__global__ __launch_bounds__(kNormThreads) void rms_norm_kernel(
    const uint16_t* __restrict__ x, int64_t xs, const uint16_t* __restrict__ w, int H, float eps,
    uint16_t* __restrict__ out) {
  __shared__ float s_sum[kNormThreads / 64];
  const int tid = threadIdx.x;
  const uint16_t* xr = x + (int64_t)blockIdx.x * xs;
  uint16_t* orow = out + (int64_t)blockIdx.x * H;
  uint4 keep[kNormKeep];
  float sum = 0.f;
  auto add = [&](uint4 v) {
    const uint32_t u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float a = widen<DT>((uint16_t)u[e]), b = widen<DT>((uint16_t)(u[e] >> 16));
      sum = __builtin_fmaf(a, a, sum);
      sum = __builtin_fmaf(b, b, sum);
    }
  };
#pragma unroll
  for (int p = 0; p < kNormKeep; ++p) {
    const int i = p * kNormPass + tid * 8;
    keep[p] = i < H ? *reinterpret_cast<const uint4*>(xr + i) : make_uint4(0, 0, 0, 0);
    add(keep[p]);
  }
  for (int i = kNormKeep * kNormPass + tid * 8; i < H; i += kNormPass)
    add(*reinterpret_cast<const uint4*>(xr + i));
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) sum += __shfl_xor(sum, d, 64);
  if ((tid & 63) == 0) s_sum[tid >> 6] = sum;
  __syncthreads();
  float all = 0.f;
#pragma unroll
  for (int i = 0; i < kNormThreads / 64; ++i) all += s_sum[i];
  const float inv = rsqrtf(all / (float)H + eps);
  auto put = [&](int i, uint4 v) {
    const uint4 wv = *reinterpret_cast<const uint4*>(w + i);
    const uint32_t u[4] = {v.x, v.y, v.z, v.w}, q[4] = {wv.x, wv.y, wv.z, wv.w};
    uint32_t o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      uint32_t r = 0;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const float n = widen<DT>(narrow<DT>(widen<DT>((uint16_t)(u[e] >> (16 * h))) * inv));
        r |= (uint32_t)narrow<DT>(widen<DT>((uint16_t)(q[e] >> (16 * h))) * n) << (16 * h);
      }
      o[e] = r;
    }
    *reinterpret_cast<uint4*>(orow + i) = make_uint4(o[0], o[1], o[2], o[3]);
  };
#pragma unroll
  for (int p = 0; p < kNormKeep; ++p) {
    const int i = p * kNormPass + tid * 8;
    if (i < H) put(i, keep[p]);
  }
  for (int i = kNormKeep * kNormPass + tid * 8; i < H; i += kNormPass)
    put(i, *reinterpret_cast<const uint4*>(xr + i));
}

template <int DT>
__global__ __launch_bounds__(256) void silu_mul_kernel(const uint16_t* __restrict__ g,
                                                       const uint16_t* __restrict__ u, int64_t n,
                                                       uint16_t* __restrict__ out) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 2;
  if (i >= n) return;
  const uint32_t a = *reinterpret_cast<const uint32_t*>(g + i);
  const uint32_t b = *reinterpret_cast<const uint32_t*>(u + i);
  uint32_t r = 0;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const float x = widen<DT>((uint16_t)(a >> (16 * h)));
    const float s = widen<DT>(narrow<DT>(x / (1.0f + expf(-x))));
    r |= (uint32_t)narrow<DT>(s * widen<DT>((uint16_t)(b >> (16 * h)))) << (16 * h);
  }
  *reinterpret_cast<uint32_t*>(out + i) = r;
}

template <int DT>
__global__ __launch_bounds__(128) void rope_tables_kernel(const int64_t* __restrict__ pos,
                                                          const void* __restrict__ inv_freq,
                                                          int freq_dtype, float scaling, int half,
                                                          uint16_t* __restrict__ cos_out,
                                                          uint16_t* __restrict__ sin_out) {
  const int i = threadIdx.x;
  if (i >= half) return;
  const float f = freq_dtype == LAP_DTYPE_F32 ? static_cast<const float*>(inv_freq)[i]
                  : freq_dtype == LAP_DTYPE_F16
                      ? h2f(static_cast<const uint16_t*>(inv_freq)[i])
                      : bf2f(static_cast<const uint16_t*>(inv_freq)[i]);
  const float a = f * (float)pos[blockIdx.x];
  const uint16_t c = narrow<DT>(cosf(a) * scaling), s = narrow<DT>(sinf(a) * scaling);
  const int64_t o = (int64_t)blockIdx.x * 2 * half + i;
  cos_out[o] = c;
  cos_out[o + half] = c;
  sin_out[o] = s;
  sin_out[o + half] = s;
}

// Orderable key of a value (NaN above all, -0 as +0), then the lower index.
template <int DT>
__device__ __forceinline__ uint64_t arg_key(uint16_t v, uint32_t i) {
  const float f = widen<DT>(v);
  const uint32_t k = f != f ? 0x1ffffu : orderable16(v);
  return ((uint64_t)k << 32) | (0xffffffffu - i);
}
__device__ __forceinline__ uint64_t max64(uint64_t a, uint64_t b) { return a > b ? a : b; }

// One workgroup per row.  A thread keeps the largest value of its 16-byte
// vectors and the first vector that holds it, and looks for the element once at
// the end: 15 instructions per vector; an ordered key per element took 80 and set
// the time (128256 columns 16.0 us, now 10.2 with the copy).  The step's copy of the logits to the
// buffer its caller reads rides along (4.7 us as a launch of its own).
template <int DT>
__global__ __launch_bounds__(1024) void argmax_rows_kernel(const uint16_t* __restrict__ x,
                                                           int64_t xs, int V,
                                                           int64_t* __restrict__ out,
                                                           uint16_t* __restrict__ copy) {
  __shared__ uint64_t s_best[16];
  const int tid = threadIdx.x;
  const uint16_t* xr = x + (int64_t)blockIdx.x * xs;
  uint16_t* cr = copy ? copy + (int64_t)blockIdx.x * V : nullptr;
  const bool vec = ((reinterpret_cast<uintptr_t>(xr) | reinterpret_cast<uintptr_t>(cr)) & 15) == 0;
  const int nv = vec ? V / 8 : 0;
  const uint4* xv = reinterpret_cast<const uint4*>(xr);
  float top = -__builtin_inff();
  int at = tid;
  auto look = [&](uint4 v, int i) {
    const uint32_t u[4] = {v.x, v.y, v.z, v.w};
    float m = widen<DT>((uint16_t)u[0]);
#pragma unroll
    for (int e = 1; e < 8; ++e)
      m = __builtin_elementwise_maximum(m, widen<DT>((uint16_t)(u[e / 2] >> (16 * (e & 1)))));
    if (m > top || (m != m && top == top)) {  // ascending vectors: the first is kept
      top = m;
      at = i;
    }
  };
  int i = tid;
#pragma unroll 1
  for (; i + 7 * 1024 < nv; i += 8 * 1024) {
    uint4 v[8];
#pragma unroll
    for (int d = 0; d < 8; ++d) v[d] = xv[i + d * 1024];
#pragma unroll
    for (int d = 0; d < 8; ++d) {
      look(v[d], i + d * 1024);
      if (cr) reinterpret_cast<uint4*>(cr)[i + d * 1024] = v[d];
    }
  }
#pragma unroll 1
  for (; i < nv; i += 1024) {
    const uint4 v = xv[i];
    look(v, i);
    if (cr) reinterpret_cast<uint4*>(cr)[i] = v;
  }
  uint64_t best = 0;
  if (tid < nv)
    for (int e = 0; e < 8; ++e) best = max64(best, arg_key<DT>(xr[8 * at + e], 8 * at + e));
  for (i = 8 * nv + tid; i < V; i += 1024) {
    best = max64(best, arg_key<DT>(xr[i], i));
    if (cr) cr[i] = xr[i];
  }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1)
    best = max64(best, (uint64_t)__shfl_xor((unsigned long long)best, d, 64));
  if ((tid & 63) == 0) s_best[tid >> 6] = best;
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < 16; ++w) best = max64(best, s_best[w]);
    out[blockIdx.x] = (int64_t)(0xffffffffu - (uint32_t)best);
  }
}

bool misaligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) != 0; }

}  // namespace
}  // namespace lap

using namespace lap;

#define LAP_BY_DTYPE(KERNEL, GRID, THREADS, ...)                                             \
  do {                                                                                      \
    if (dtype == LAP_DTYPE_F16)                                                             \
      hipLaunchKernelGGL(KERNEL<LAP_DTYPE_F16>, GRID, dim3(THREADS), 0, as_stream(stream),   \
                         __VA_ARGS__);                                                      \
    else                                                                                    \
      hipLaunchKernelGGL(KERNEL<LAP_DTYPE_BF16>, GRID, dim3(THREADS), 0, as_stream(stream),  \
                         __VA_ARGS__);                                                      \
    LAP_LAUNCH_CHECK(#KERNEL);                                                              \
  } while (0)

extern "C" int lap_rms_norm(const void* x, int64_t x_row_stride, int rows, int H,
                            const void* weight, float eps, int dtype, void* out,
                            lap_stream_t stream) {
  clear_error();
  LAP_CHECK(x && weight && out, "lap_rms_norm: null pointer");
  LAP_CHECK(dtype == LAP_DTYPE_F16 || dtype == LAP_DTYPE_BF16, "lap_rms_norm: dtype fp16/bf16");
  LAP_CHECK(rows >= 0 && H > 0 && H % 8 == 0 && x_row_stride >= H && x_row_stride % 8 == 0,
            "lap_rms_norm: H and the row stride must be multiples of 8");
  LAP_CHECK(!misaligned16(x) && !misaligned16(weight) && !misaligned16(out),
            "lap_rms_norm: 16-byte aligned tensors");
  if (rows == 0) return LAP_OK;
  LAP_BY_DTYPE(rms_norm_kernel, dim3(rows), kNormThreads, static_cast<const uint16_t*>(x),
               x_row_stride, static_cast<const uint16_t*>(weight), H, eps,
               static_cast<uint16_t*>(out));
  return LAP_OK;
}

extern "C" int lap_silu_mul(const void* gate, const void* up, int64_t n, int dtype, void* out,
                            lap_stream_t stream) {
  clear_error();
  LAP_CHECK(gate && up && out, "lap_silu_mul: null pointer");
  LAP_CHECK(dtype == LAP_DTYPE_F16 || dtype == LAP_DTYPE_BF16, "lap_silu_mul: dtype fp16/bf16");
  LAP_CHECK(n >= 0 && n % 2 == 0 && n < (int64_t)1 << 38, "lap_silu_mul: n must be even");
  LAP_CHECK(((reinterpret_cast<uintptr_t>(gate) | reinterpret_cast<uintptr_t>(up) |
              reinterpret_cast<uintptr_t>(out)) & 3) == 0, "lap_silu_mul: 4-byte aligned tensors");
  if (n == 0) return LAP_OK;
  LAP_BY_DTYPE(silu_mul_kernel, dim3((unsigned)((n / 2 + 255) / 256)), 256,
               static_cast<const uint16_t*>(gate), static_cast<const uint16_t*>(up), n,
               static_cast<uint16_t*>(out));
  return LAP_OK;
}

extern "C" int lap_rope_tables(const int64_t* pos, int B, const void* inv_freq, int freq_dtype,
                               int half, float scaling, int dtype, void* cos_out, void* sin_out,
                               lap_stream_t stream) {
  clear_error();
  LAP_CHECK(pos && inv_freq && cos_out && sin_out, "lap_rope_tables: null pointer");
  LAP_CHECK(dtype == LAP_DTYPE_F16 || dtype == LAP_DTYPE_BF16, "lap_rope_tables: dtype fp16/bf16");
  LAP_CHECK(freq_dtype == LAP_DTYPE_F32 || freq_dtype == LAP_DTYPE_F16 ||
                freq_dtype == LAP_DTYPE_BF16, "lap_rope_tables: frequencies fp32/fp16/bf16");
  LAP_CHECK(B >= 0 && half > 0 && half <= 128, "lap_rope_tables: head dim 2 to 256");
  if (B == 0) return LAP_OK;
  LAP_BY_DTYPE(rope_tables_kernel, dim3(B), 128, pos, inv_freq, freq_dtype, scaling, half,
               static_cast<uint16_t*>(cos_out), static_cast<uint16_t*>(sin_out));
  return LAP_OK;
}

extern "C" int lap_argmax_rows(const void* x, int64_t x_row_stride, int rows, int V, int dtype,
                               int64_t* out, void* copy, lap_stream_t stream) {
  clear_error();
  LAP_CHECK(x && out, "lap_argmax_rows: null pointer");
  LAP_CHECK(dtype == LAP_DTYPE_F16 || dtype == LAP_DTYPE_BF16, "lap_argmax_rows: dtype fp16/bf16");
  LAP_CHECK(rows >= 0 && V > 0 && x_row_stride >= V, "lap_argmax_rows: bad sizes");
  if (rows == 0) return LAP_OK;
  LAP_BY_DTYPE(argmax_rows_kernel, dim3(rows), 1024, static_cast<const uint16_t*>(x), x_row_stride,
               V, out, static_cast<uint16_t*>(copy));
  return LAP_OK;
}
