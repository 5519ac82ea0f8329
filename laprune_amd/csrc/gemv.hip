// gemv.hip — y[n] = sum_k x[k] * w[n][k] for the projections of a decode step of
// one sequence, and the MLP's rnd(silu(gate x)) * up x as one launch.
//
// Bound by the read of the weights.  A wave takes two whole rows, so a row's sum
// ends in one wave reduction with nothing to combine; its loads of a step, four
// of 16 bytes per lane and row, are issued before the first is used, and some 16
// waves per CU keep 128 KB in flight, three times what 5 TB/s needs at this
// card's latency.  x comes from the caches.  Products are fp32 FMAs of the exact
// 16-bit values, sums are rounded once.
//
// us in a captured loop over weights larger than the caches, bf16, N x K
// (library GEMV / this kernel): 6144 x 4096 14.6 / 9.8, 4096 x 4096 15.5 / 7.6,
// 14336 x 4096 30.0 / 21.0, 4096 x 14336 26.8 / 20.9, 128256 x 4096 189 / 158
// (6.65 TB/s), 2048 x 2048 11.1 / 3.8, 64 x 176 6.2 / 2.4; the two 14336 x 4096
// products with silu and multiply 65 / 38.6.  Tried: rows x loads of 2 x 8 (11.0,
// 8.8, 23.3, 24.7, 161), 1 x 4 (9.9, 7.7, 20.2, 22.0, 154), 4 x 4 (12.3, 10.1,
// 22.8, 28.2, 160), 1 x 14 (9.8, 7.8, 20.3, 24.0, 155).  For more rows of x the
// lanes' products, not the read, set the time (four rows, 2 x 8: 17.1, 14.1,
// 34.0, 42.1, 241 against the library's 15.8, 15.6, 30.5, 27.3, 192), so
// batches keep the library's matrix-core product.
#include "common.h"

namespace lap {
namespace {

constexpr int kGemvThreads = 256, kRows = 2, kDeep = 4;

template <int DT>
__device__ __forceinline__ float lo16(uint32_t u) {
  return DT == LAP_DTYPE_F16 ? h2f((uint16_t)u) : __builtin_bit_cast(float, u << 16);
}
template <int DT>
__device__ __forceinline__ float hi16(uint32_t u) {
  return DT == LAP_DTYPE_F16 ? h2f((uint16_t)(u >> 16))
                             : __builtin_bit_cast(float, u & 0xffff0000u);
}
template <int DT>
__device__ __forceinline__ uint16_t rnd16(float f) {
  return DT == LAP_DTYPE_F16 ? f2h(f) : f2bf(f);
}
template <int DT>
__device__ __forceinline__ float round_to(float f) {
  return lo16<DT>(rnd16<DT>(f));
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

static_assert(kRows == 2, "a GLU wave holds one row of each weight");

// GLU: the wave's two rows are row n of w (gate) and of w2 (up), and
// out[n] = rnd(rnd(g / (1 + exp(-g))) * u) of their rounded sums.
template <int DT, bool GLU>
__global__ __launch_bounds__(kGemvThreads) void gemv_kernel(const uint16_t* __restrict__ x,
                                                            const uint16_t* __restrict__ w,
                                                            const uint16_t* __restrict__ w2, int N,
                                                            int K, uint16_t* __restrict__ out) {
  constexpr int R = kRows, STEP = GLU ? 1 : kRows;
  const int lane = threadIdx.x & 63;
  const int n0 = (blockIdx.x * (kGemvThreads / 64) + (threadIdx.x >> 6)) * STEP;
  if (n0 >= N) return;
  const uint16_t* wr[R];
#pragma unroll
  for (int r = 0; r < R; ++r)
    wr[r] = GLU ? (r ? w2 : w) + (int64_t)n0 * K : w + (int64_t)(n0 + r < N ? n0 + r : N - 1) * K;
  float acc[R] = {};
  auto fold = [&](const u32x4 (&wv)[R], int k) {
    const u32x4 xv = *reinterpret_cast<const u32x4*>(x + k);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float x0 = lo16<DT>(xv[e]), x1 = hi16<DT>(xv[e]);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        acc[r] = __builtin_fmaf(lo16<DT>(wv[r][e]), x0, acc[r]);
        acc[r] = __builtin_fmaf(hi16<DT>(wv[r][e]), x1, acc[r]);
      }
    }
  };
  int k = 0;
#pragma unroll 1
  for (; k + 512 * kDeep <= K; k += 512 * kDeep) {
    u32x4 wv[kDeep][R];
#pragma unroll
    for (int d = 0; d < kDeep; ++d)
#pragma unroll
      for (int r = 0; r < R; ++r)
        wv[d][r] = __builtin_nontemporal_load(
            reinterpret_cast<const u32x4*>(wr[r] + k + 512 * d + lane * 8));
#pragma unroll
    for (int d = 0; d < kDeep; ++d) fold(wv[d], k + 512 * d + lane * 8);
  }
#pragma unroll 4
  for (k += lane * 8; k < K; k += 512) {
    u32x4 wv[R];
#pragma unroll
    for (int r = 0; r < R; ++r)
      wv[r] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wr[r] + k));
    fold(wv, k);
  }
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) acc[r] += __shfl_xor(acc[r], d, 64);
  if (lane != 0) return;
  if constexpr (GLU) {
    const float g = round_to<DT>(acc[0]), u = round_to<DT>(acc[1]);
    out[n0] = rnd16<DT>(round_to<DT>(g / (1.0f + expf(-g))) * u);
  } else {
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (n0 + r < N) out[n0 + r] = rnd16<DT>(acc[r]);
  }
}

template <bool GLU>
void launch(const void* x, const void* w, const void* w2, int N, int K, int dtype, void* out,
            hipStream_t s) {
  const int per = (GLU ? 1 : kRows) * (kGemvThreads / 64);
  const dim3 grid((N + per - 1) / per), block(kGemvThreads);
  const uint16_t* xp = static_cast<const uint16_t*>(x);
  const uint16_t* wp = static_cast<const uint16_t*>(w);
  const uint16_t* w2p = static_cast<const uint16_t*>(w2);
  uint16_t* op = static_cast<uint16_t*>(out);
  if (dtype == LAP_DTYPE_F16)
    hipLaunchKernelGGL((gemv_kernel<LAP_DTYPE_F16, GLU>), grid, block, 0, s, xp, wp,
                       w2p, N, K, op);
  else
    hipLaunchKernelGGL((gemv_kernel<LAP_DTYPE_BF16, GLU>), grid, block, 0, s, xp, wp,
                       w2p, N, K, op);
}

bool misaligned(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) != 0; }

}  // namespace
}  // namespace lap

using namespace lap;

extern "C" int lap_gemv(const void* x, const void* w, int N, int K, int dtype, void* out,
                        lap_stream_t stream) {
  clear_error();
  LAP_CHECK(x && w && out, "lap_gemv: null pointer");
  LAP_CHECK(dtype == LAP_DTYPE_F16 || dtype == LAP_DTYPE_BF16, "lap_gemv: dtype fp16/bf16");
  LAP_CHECK(N > 0 && K > 0 && K % 8 == 0 && K <= 1 << 30 && N <= 1 << 30,
            "lap_gemv: K must be a multiple of 8");
  LAP_CHECK(!misaligned(x) && !misaligned(w), "lap_gemv: 16-byte aligned x and w");
  launch<false>(x, w, nullptr, N, K, dtype, out, as_stream(stream));
  LAP_LAUNCH_CHECK("gemv_kernel");
  return LAP_OK;
}

extern "C" int lap_gemv_glu(const void* x, const void* gate, const void* up, int N, int K,
                            int dtype, void* out, lap_stream_t stream) {
  clear_error();
  LAP_CHECK(x && gate && up && out, "lap_gemv_glu: null pointer");
  LAP_CHECK(dtype == LAP_DTYPE_F16 || dtype == LAP_DTYPE_BF16, "lap_gemv_glu: dtype fp16/bf16");
  LAP_CHECK(N > 0 && K > 0 && K % 8 == 0 && K <= 1 << 30 && N <= 1 << 30,
            "lap_gemv_glu: K must be a multiple of 8");
  LAP_CHECK(!misaligned(x) && !misaligned(gate) && !misaligned(up),
            "lap_gemv_glu: 16-byte aligned x and weights");
  launch<true>(x, gate, up, N, K, dtype, out, as_stream(stream));
  LAP_LAUNCH_CHECK("gemv_kernel");
  return LAP_OK;
}
