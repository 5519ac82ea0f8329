// encode_wide.h — the prompt-sized greedy encode (included by encode.hip).
//
// Same recurrence and contract as the other encode kernels: the distance
// search is a coarse fp16-MFMA pass that can only rule entries out, and every
// entry it cannot rule out is compared by the contract's fp32 distance.
//
// Work shape.  A wave owns 32 rows for all M stages and never shares them.  It
// holds them twice over, in two lane layouts:
//   search  v_mfma_f32_32x32x16_f16 with the codebook as operand A and the
//           rows as operand B: lane l ends with the scores of row l % 32
//           against 16 of a tile's 32 entries (the other 16 in lane l ^ 32), so
//           the maximum and the survivors are found inside the lane;
//   update  four neighbouring lanes hold a row's fp32 residual (two rows each:
//           row l / 4 and row 16 + l / 4), lane l the dot16 chains 4i + l % 4.
//           The vector memory unit takes four neighbouring lanes on one line
//           in a cycle and any other four in four (18 and 64 cycles measured
//           per 1 KiB instruction), and every stage reads a row of the fp32
//           codebook per residual row: one residual per lane pair, as the
//           search has them, made those reads 60 % of the kernel.
// The fp16 residual goes from the update's to the search's layout through
// 2 KiB of LDS per wave; apart from that, LDS holds the codebook's fragments
// alone, two stages of them, filled by DMA under the previous stage.
//
// Scores.  A_k = r . C'_k - h'_k with C' = 2^b C (b per stage, exact) and
// h' = 2^(b-1) cn, so that dist_k = rn - 2^(1-b) A_k; the smallest distance is
// the largest A.  h' rides in the product as one more k-step: three fp16 parts
// of h' / 64 against the constant -64.
//
// Ruling out.  Let A*_k be the value with E_k = rn - 2^(1-b) A*_k for the
// contract's fp32 distance E_k.  With c' = max_k |C'_k|, d' = max_k of the
// norm of C'_k's fp16 rounding error, h = max_k h'_k and s = sqrt(rn):
//   |A_k - A*_k| <= s d' + (2^-11 s + sqrt(D) (2^-14 + 2^-25)) (c' + d')  fp16 inputs
//                 + (D + 16) 2^-23 (s c' + h)                      fp32 MFMA sums
//                 + 20 2^-24 s c' + 2^-24 (2^b rn + 2 h + s c')    E_k's own rounding
//                 + min(h, 2^-8) (1 + 2^-10) + 2^-19               the parts of h'
// (2^-14: subnormal fp16 inputs may be flushed, of the parts of h' / 64 less than
// 2^-14 in all; the sum term takes one ulp of the largest magnitude per addition,
// in any order).  eps is above the sum, with 2^-15 for the (D + 16) 2^-23, 2^-22
// for rn's 2^-24 and 2^-18 for the last, and an entry with
// A_k < max A - 2 eps cannot attain the minimum of E, nor tie with it.  Stages
// or rows outside the fp16 range (norms that are not finite, codebook norms
// past 2^12, rows past 2^15) keep every entry.  With post-RoPE keys and
// codebooks of trained magnitudes one entry is left for about 95 % of the
// rows, and its distance need not be formed at all.
//
// Measured (1,048,576 rows, D = 128): 3.2 to 3.9 ms in six runs (3.3 to 3.6 with
// entries of trained magnitudes) against 13.6 to 14.0 for the bf16 form it
// replaced (64 rows per workgroup, a barrier-separated coarse pass, shortlist and
// recheck, 6.9 us per stage and 64 rows; here 6.4 us per 256).  What bounds it now is instruction issue: about 1120 VALU
// instructions per wave and stage (2.5 per score to find maximum and
// survivors) fill some 60 % of the cycles and the products 33 %.
#pragma once

namespace lap {
namespace {

typedef _Float16 wh8_t __attribute__((ext_vector_type(8)));
typedef _Float16 wh4_t __attribute__((ext_vector_type(4)));
typedef float wf16_t __attribute__((ext_vector_type(16)));

// Dimension that slot e (0 .. 7) of k-step s in half h of the operands stands
// for.  Quarter q = 2 (s % 2) + h of a row holds the dot16 chains 4i + q,
// i = 0 .. 3, one after another; slots 8v .. 8v + 7 of it are k-step 2v + q / 2.
template <int D>
__device__ __forceinline__ constexpr int wide_dim(int s, int e, int h) {
  constexpr int L = D / 16;
  const int q = 2 * (s & 1) + h, x = 8 * (s >> 1) + e;
  return (4 * (x / L) + q) * L + x % L;
}

__device__ __forceinline__ float wide_f16_flushed(float x) {
  const float y = h2f(f2h(x));
  return fabsf(y) < 0x1p-14f ? 0.f : y;
}

// One workgroup per stage: the scale b, the test's constants and the fp16
// fragments.  Entries past K repeat entry K - 1 (they can then neither raise
// the maximum nor be picked).
template <int D>
__global__ __launch_bounds__(1024) void encode_prep_wide(const float* __restrict__ cb, int M,
                                                         int K, const float* __restrict__ cn,
                                                         uint4* __restrict__ wide,
                                                         WideStage* __restrict__ stage) {
  constexpr int KS = D / 16, L = D / 16;
  __shared__ float s_red[16];
  const int m = blockIdx.x, tid = threadIdx.x;
  const float* cbm = cb + (int64_t)m * K * D;
  const float* cnm = cn + (int64_t)m * K;
  auto block_max = [&](float v) {
    for (int w = 32; w >= 1; w >>= 1) v = fmaxf(v, __shfl_xor(v, w, 64));
    if ((tid & 63) == 0) s_red[tid >> 6] = v;
    __syncthreads();
    float r = s_red[0];
    for (int i = 1; i < 16; ++i) r = fmaxf(r, s_red[i]);
    __syncthreads();
    return r;
  };
  const float v = tid < K ? cnm[tid] : 0.f;
  const bool bad = __syncthreads_or(!(v < 0x1p24f));  // NaN, inf or a norm of 2^12 and above
  const float cmax = block_max(v);
  int b = cmax > 0.f && !bad ? 9 - ilogbf(sqrtf(cmax)) : 0;
  b = b < -20 ? -20 : b > 60 ? 60 : b;
  const float sc = ldexpf(1.f, b);
  // the largest rounding-error norm of the stage's fp16 entries, four threads
  // per entry
  float err = 0.f;
  if (tid / 4 < K) {
    const float* row = cbm + (int64_t)(tid / 4) * D + (tid & 3) * 4;
    for (int d = 0; d < D; d += 16) {
      const float4 x = *reinterpret_cast<const float4*>(row + d);
      const float xs[4] = {x.x * sc, x.y * sc, x.z * sc, x.w * sc};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float dx = xs[e] - wide_f16_flushed(xs[e]);
        err = __builtin_fmaf(dx, dx, err);
      }
    }
  }
  err += __shfl_xor(err, 1, 64);
  err += __shfl_xor(err, 2, 64);
  const float d_ = sqrtf(block_max(err)) * 1.001f;
  if (tid == 0) {
    const float c = sqrtf(cmax) * sc * 1.001f, h = 0.5f * cmax * sc * 1.001f;
    WideStage w;
    w.e1 = 2.05f * (d_ + (0x1p-11f + 0x1p-15f + 0x1p-17f) * (c + d_));
    w.e0 = bad ? INFINITY
               : 2.05f * (sqrtf((float)D) * 0x1.01p-14f * (c + d_) + 0x1p-15f * h + 0x1p-18f +
                          1.01f * fminf(h, 0x1p-8f));
    w.e2 = 2.05f * sc * 0x1p-22f;
    w.pad = 0.f;
    stage[m] = w;
  }
  const int NT = wide_tiles(K), nf = NT * KS * 64;
  uint4* out = wide + (int64_t)m * wide_stage_uint4(K, D);
  for (int i = tid; i < nf; i += 1024) {
    const int l = i & 63, ks = (i >> 6) % KS, tile = (i >> 6) / KS;
    const int k = min(32 * tile + (l & 31), K - 1);
    const float* row = cbm + (int64_t)k * D;
    wh8_t x;
#pragma unroll
    for (int e = 0; e < 8; e += 4) {  // four slots in a row are four dimensions in a row
      static_assert(L % 4 == 0, "chains of whole float4 blocks");
      const float4 y = *reinterpret_cast<const float4*>(row + wide_dim<D>(ks, e, l >> 5));
      x[e] = __builtin_bit_cast(_Float16, f2h(y.x * sc));
      x[e + 1] = __builtin_bit_cast(_Float16, f2h(y.y * sc));
      x[e + 2] = __builtin_bit_cast(_Float16, f2h(y.z * sc));
      x[e + 3] = __builtin_bit_cast(_Float16, f2h(y.w * sc));
    }
    out[i] = __builtin_bit_cast(uint4, x);
  }
  uint2* hp = reinterpret_cast<uint2*>(out + nf);
  for (int i = tid; i < (int)(wide_stage_uint4(K, D) - nf) * 2; i += 1024) {
    float x = cnm[min(i, K - 1)] * (0.5f * sc) * 0x1p-6f;
    wh4_t y = {};
#pragma unroll
    for (int e = 0; e < 3; ++e) {
      y[e] = __builtin_bit_cast(_Float16, f2h(x));
      x = x - (float)y[e];
    }
    hp[i] = __builtin_bit_cast(uint2, y);
  }
}

// Both halves' values of x, in every lane: {lane l % 32's, lane l % 32 + 32's}.
struct HalfPair {
  uint32_t lo, hi;
};
__device__ __forceinline__ HalfPair halves(uint32_t x) {
  const auto p = __builtin_amdgcn_permlane32_swap(x, x, false, false);
  return HalfPair{p[0], p[1]};
}
__device__ __forceinline__ float half_max(float x) {
  const HalfPair p = halves(__builtin_bit_cast(uint32_t, x));
  return __builtin_elementwise_maximum(__builtin_bit_cast(float, p.lo),
                                       __builtin_bit_cast(float, p.hi));
}

// dot16 of a quarter row each in four neighbouring lanes: four chains per
// lane, the contract's fold over w = 8 and 4 inside the lane and over w = 2
// and 1 within the four (fp32 + commutes), the result in all of them.
template <int D>
__device__ __forceinline__ float wide_dot16(const float (&a)[D / 4], const float (&b)[D / 4]) {
  constexpr int L = D / 16;
  float s[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float x = 0.f;
#pragma unroll
    for (int t = 0; t < L; ++t) x = __builtin_fmaf(a[i * L + t], b[i * L + t], x);
    s[i] = x;
  }
  s[0] = s[0] + s[2];
  s[1] = s[1] + s[3];
  float x = s[0] + s[1];
  x = x + dpp_f<0x4e>(x);  // quad_perm: lane ^ 2
  x = x + dpp_f<0xb1>(x);  // quad_perm: lane ^ 1
  return x;
}

// Quarter q of an fp32 row: chains 4i + q.
template <int D>
__device__ __forceinline__ void wide_row(float (&c)[D / 4], const float* __restrict__ row, int q) {
  constexpr int L = D / 16;
#pragma unroll
  for (int i = 0; i < D / 4; i += 4) {
    const float4 v = *reinterpret_cast<const float4*>(row + 4 * (i / L) * L + i % L + q * L);
    c[i] = v.x;
    c[i + 1] = v.y;
    c[i + 2] = v.z;
    c[i + 3] = v.w;
  }
}

// Quarter q of an input row, widened to fp32; vec: its chunks are aligned.
template <int D, int DT, typename T>
__device__ __forceinline__ void wide_input(float (&r)[D / 4], const T* __restrict__ x, int q,
                                           int vec) {
  constexpr int L = D / 16;
  if (!vec) {
#pragma unroll
    for (int i = 0; i < D / 4; ++i) r[i] = load_as_f32(x, 4 * (i / L) * L + i % L + q * L, DT);
    return;
  }
  if constexpr (DT == LAP_DTYPE_F32) {
    wide_row<D>(r, x, q);
  } else {
#pragma unroll
    for (int i = 0; i < D / 4; i += 4) {
      const uint2 v = *reinterpret_cast<const uint2*>(x + 4 * (i / L) * L + i % L + q * L);
      const uint32_t w[4] = {v.x & 0xffffu, v.x >> 16, v.y & 0xffffu, v.y >> 16};
#pragma unroll
      for (int e = 0; e < 4; ++e)
        r[i + e] = DT == LAP_DTYPE_F16 ? h2f((uint16_t)w[e]) : bf2f((uint16_t)w[e]);
    }
  }
}

// x of lane `from` (ds_bpermute).
__device__ __forceinline__ uint32_t lane_read(uint32_t x, int from) {
  return (uint32_t)__builtin_amdgcn_ds_bpermute(from << 2, (int)x);
}
__device__ __forceinline__ float lane_read(float x, int from) {
  return __builtin_bit_cast(float, lane_read(__builtin_bit_cast(uint32_t, x), from));
}

// One kilobyte per call straight from global memory into LDS: lane l's 16
// bytes at src land at dst + 16 l (dst uniform).  Issued from asm: through the
// builtin the compiler would wait for it before any later LDS read, and the
// point is to let a stage's fragments arrive under the previous stage.  It has
// no result register; wide_dma_wait covers it.
__device__ __forceinline__ void wide_dma(const uint4* src, uint32_t dst) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 1\n\tglobal_load_lds_dwordx4 %0, off"
               :
               : "v"(src), "s"(dst)
               : "memory", "m0");
}
__device__ __forceinline__ void wide_dma_wait() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

template <int D, int WAVES>
constexpr size_t wide_lds_bytes(int K) {
  return (size_t)2 * wide_stage_uint4(K, D) * 16 + (size_t)WAVES * 2048;
}

// K256: all 256 entries (the tiles' addresses are then constants).
template <int D, int WAVES, bool K256>
__global__ __launch_bounds__(WAVES * 64) void encode_wide_kernel(
    RowMap rm, int N, const float* __restrict__ cb, int M, int K_arg,
    const uint4* __restrict__ wide, const WideStage* __restrict__ stage,
    const float* __restrict__ cn, float* __restrict__ rnorm, int x_vec, int polls) {
  constexpr int KS = D / 16, NV = D / 4;
  constexpr uint32_t kNone = 0x7fffu;
  const int K = K256 ? 256 : K_arg;
  extern __shared__ __attribute__((aligned(16))) char wide_smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int h = lane >> 5, n = lane & 31;   // search: half, row
  const int q = lane & 3, rho = lane >> 2;  // update: quarter, rows rho and 16 + rho
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int NT = wide_tiles(K);
  const int n16 = (int)wide_stage_uint4(K, D);
  uint4* s_frag = reinterpret_cast<uint4*>(wide_smem);
  uint4* s_tr = s_frag + 2 * n16 + wave * 128;  // this wave's 2 KiB
  const int row0 = (blockIdx.x * WAVES + wave) * 32 + rho;
  const bool live[2] = {row0 < N && rm.live(row0), row0 + 16 < N && rm.live(row0 + 16)};
  // a workgroup with no live row leaves at once
  if (rm.ranges && !__syncthreads_or(live[0] || live[1])) return;

  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)wide_smem;
  auto request = [&](int m) {
    const uint4* src = wide + (int64_t)m * n16 + lane;
    const uint32_t dst = lds0 + (uint32_t)((m & 1) * n16) * 16u;
    for (int c = wave; c < n16 / 64; c += WAVES) wide_dma(src + c * 64, dst + c * 1024);
  };
  request(0);
  // The waves run up to a stage apart, so that some search (matrix cores, LDS)
  // while others update (VALU, L2 latency): in place of a barrier, counters of
  // the waves whose share of an even or odd stage's fragments is in (0, 1) and
  // of those past the search of one (2, 3), each in turns of WAVES.  A wave
  // asks for stage m + 2 only when all are past the search of stage m, so a
  // counter never mixes two stages.
  // Waits are bounded, so that the kernel always ends.  A wait that gives up
  // marks every counter, which ends the waits of the other waves too (each
  // wave then has in_step false): from there on they neither request nor
  // count fragments in, so that no stage that is still read is overwritten,
  // and every row keeps all entries, so that the contract's distances alone
  // decide and the codes stay what they are.
  constexpr uint32_t kGaveUp = 0x80000000u;
  __shared__ uint32_t s_cnt[4];
  bool in_step = true;  // wave-uniform
  auto arrive = [&](int i) {
    if (lane == 0)
      __hip_atomic_fetch_add(&s_cnt[i], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  };
  auto await = [&](int i, uint32_t turns) {
    uint32_t v = 0;
    for (int spin = 0; spin < polls; ++spin) {
      v = (uint32_t)__builtin_amdgcn_readfirstlane((int)__hip_atomic_load(
          &s_cnt[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
      if (v >= turns) break;
      __builtin_amdgcn_s_sleep(1);
    }
    if (v < turns && lane < 4)
      __hip_atomic_fetch_or(&s_cnt[lane], kGaveUp, __ATOMIC_RELAXED,
                            __HIP_MEMORY_SCOPE_WORKGROUP);
    in_step = in_step && v >= turns && v < kGaveUp;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  };

  float r[2][NV], rn[2];
  uint8_t* crow[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
#pragma unroll
    for (int i = 0; i < NV; ++i) r[u][i] = 0.f;
    crow[u] = rm.codes;
    if (live[u]) {
      const int row = row0 + 16 * u;
      crow[u] = rm.crow(row);
      const int64_t o = rm.off(row, rm.x_sb, rm.x_sh, rm.x_st);
      if (rm.x_dtype == LAP_DTYPE_F32)
        wide_input<D, LAP_DTYPE_F32>(r[u], static_cast<const float*>(rm.x) + o, q, x_vec);
      else if (rm.x_dtype == LAP_DTYPE_F16)
        wide_input<D, LAP_DTYPE_F16>(r[u], static_cast<const uint16_t*>(rm.x) + o, q, x_vec);
      else
        wide_input<D, LAP_DTYPE_BF16>(r[u], static_cast<const uint16_t*>(rm.x) + o, q, x_vec);
    }
    rn[u] = wide_dot16<D>(r[u], r[u]);
  }

  // operand B of the h' step: the three parts times -64 (in the lower half's
  // slots; the upper half repeats the same operand A against zeros)
  wh4_t baug = {};
  if (h == 0) baug[0] = baug[1] = baug[2] = (_Float16)-64.f;
  wide_dma_wait();
  if (tid < 4) s_cnt[tid] = 0;
  lds_barrier();
  if (M > 1) request(1);

  for (int m = 0; m < M; ++m) {
    // The residual's side of the search: the fp16 residual as operand B and
    // the test's 2 eps.  Units of 16 bytes go through LDS, written by (row,
    // q) and read by (row, half); the row's slot is permuted by q so that
    // neither side's lanes meet in a bank.  DS operations of a wave stay in
    // order.
    const WideStage ws = stage[m];
    wh8_t bf[KS];
#pragma unroll
    for (int v = 0; v < KS / 2; ++v) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        wh8_t x;
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = (_Float16)r[u][8 * v + e];
        s_tr[(2 * q + u) * 16 + (rho ^ (4 * q))] = __builtin_bit_cast(uint4, x);
      }
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront", "local");
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int qq = 2 * b + h;
        bf[2 * v + b] = __builtin_bit_cast(
            wh8_t, s_tr[(2 * qq + (n >> 4)) * 16 + ((n & 15) ^ (4 * qq))]);
      }
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront", "local");
    }
    const float rn0 = lane_read(rn[0], 4 * (n & 15)), rn1 = lane_read(rn[1], 4 * (n & 15));
    const float rns = n < 16 ? rn0 : rn1;
    const float eps2 = __builtin_fmaf(__builtin_amdgcn_sqrtf(rns), ws.e1,
                                      __builtin_fmaf(rns, ws.e2, ws.e0));

    // stage 0's fragments came in before the barrier
    if (m && in_step) await(m & 1, (uint32_t)(WAVES * ((m + 1) / 2)));

    // ---- coarse scores, a tile (32 entries) at a time: the lane's running
    // maximum t1 and, per tile, its entries within 2 eps of it.  Step i of a
    // tile: product i of tile t, and 1 / (KS + 1) of the sifting of tile
    // t - 1.  Left to itself the compiler issues the products in a row and
    // the sifting after them; up to six VALU instructions fit under one.
    const uint4* fs = s_frag + (m & 1) * n16;
    const uint2* hs = reinterpret_cast<const uint2*>(fs + NT * KS * 64) + n;
    float t1 = -INFINITY, mp0, mp1, mp2, mp3 = -INFINITY;
    uint32_t mk0, mk1, mk2, mk3 = 0;
    float x = 0.f, y = 0.f, sthr = 0.f;
    uint32_t w = 0;
    // step i of sifting v, a pair's even or odd tile
    auto sift = [&](int i, bool odd, const wf16_t& v) {
      constexpr int S = KS + 1, SM = KS == 8 ? 2 : 1;  // steps for the maximum
      // elements 0 .. 15 of the maximum in steps < SM, then the threshold,
      // then the differences' signs, shifted in
      if (i == 0) x = __builtin_elementwise_maximum(v[0], v[1]);
#pragma unroll
      for (int e = 2; e < 16; e += 2)
        if (e * SM / 16 == i)
          x = __builtin_elementwise_maximum(__builtin_elementwise_maximum(x, v[e]), v[e + 1]);
      if (i == SM) {
        t1 = __builtin_elementwise_maximum(t1, x);
        sthr = t1 - eps2;
        // an even tile's entries are dropped when the odd one's maximum
        // leaves them behind
        if (odd) w = y >= sthr ? w : ~0u;
      }
#pragma unroll
      for (int e = 0; e < 16; ++e)
        if (i > SM && e * (S - SM - 1) / 16 == i - SM - 1)
          w = __builtin_amdgcn_alignbit(w, __builtin_bit_cast(uint32_t, v[e] - sthr), 31);
      if (i == S - 1) {
        if (odd) {  // entry e of tile t at bit 31 - 16 (t % 2) - e
          mk0 = mk1; mk1 = mk2; mk2 = mk3; mk3 = ~w;
          mp0 = mp1; mp1 = mp2; mp2 = mp3; mp3 = __builtin_elementwise_maximum(x, y);
        } else {
          y = x;
        }
      }
    };
    // products of tile t into a under the sifting of v
    auto tile = [&](int t, wf16_t& a, bool odd, const wf16_t& v) {
      const int tc = min(t, NT - 1);  // tiles past the last repeat it (entries past K, dropped)
      const uint4* f = fs + tc * KS * 64 + lane;
      const uint2 hp = hs[tc * 32];
      uint4 g[3];  // operand A, two steps ahead
      g[1] = f[0];
#pragma unroll
      for (int i = 0; i <= KS; ++i) {
        if (i + 2 <= KS) g[(i + 2) % 3] = f[(i + 1) * 64];
        const wf16_t z = {};
        if (i == 0)
          a = __builtin_amdgcn_mfma_f32_32x32x8f16(__builtin_bit_cast(wh4_t, hp), baug, z, 0, 0, 0);
        else
          a = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(wh8_t, g[i % 3]),
                                                     bf[i ? i - 1 : 0], a, 0, 0, 0);
        sift(i, odd, v);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    // four pairs of tiles; the first turn sifts a tile of zeros whose word is
    // shifted out again
    wf16_t ae, ao = {};
    mk0 = mk1 = mk2 = 0;
    mp0 = mp1 = mp2 = -INFINITY;
    t1 = -INFINITY;
#pragma unroll 1
    for (int p = 0; p < 4; ++p) {
      tile(2 * p, ae, true, ao);
      if (p == 0) t1 = -INFINITY;
      tile(2 * p + 1, ao, false, ae);
    }
#pragma unroll
    for (int i = 0; i <= KS; ++i) sift(i, true, ao);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    arrive(2 + (m & 1));  // this wave has read stage m's fragments
    if (m + 1 < M) {      // and its share of stage m + 1's is in
      wide_dma_wait();
      if (in_step) arrive((m + 1) & 1);
    }

    t1 = half_max(t1);
    const float thr = t1 - eps2;
    // outside the fp16 range, or no fragments
    const bool all = !(eps2 < 0x1p60f) || !(rns < 0x1p30f) || !in_step;
    mk0 = all ? ~0u : mp0 >= thr ? mk0 : 0u;
    mk1 = all ? ~0u : mp1 >= thr ? mk1 : 0u;
    mk2 = all ? ~0u : mp2 >= thr ? mk2 : 0u;
    mk3 = all ? ~0u : mp3 >= thr ? mk3 : 0u;

    // The row's lowest candidate (kNone: none): each half's own lowest, then
    // the lower of the two; drop: its half takes it out.
    auto lowest = [&](bool drop) -> uint32_t {
      const bool z0 = mk0 == 0, z1 = z0 && mk1 == 0, z2 = z1 && mk2 == 0;
      const uint32_t w = !z0 ? mk0 : !z1 ? mk1 : !z2 ? mk2 : mk3;
      const uint32_t pi = !z0 ? 0u : !z1 ? 1u : !z2 ? 2u : 3u;
      const uint32_t b = (uint32_t)__builtin_clz(w | 1u);
      const uint32_t e = 64 * pi + 32 * (b >> 4) + 8 * ((b & 15) >> 2) + 4 * h + (b & 3);
      const uint32_t f = w != 0 && e < (uint32_t)K ? e : kNone;
      const HalfPair fp = halves(f);
      const uint32_t cand = min(fp.lo, fp.hi);
      const uint32_t keep = drop && f == cand && f != kNone ? ~(0x80000000u >> b) : ~0u;
      mk0 &= pi == 0 ? keep : ~0u;
      mk1 &= pi == 1 ? keep : ~0u;
      mk2 &= pi == 2 ? keep : ~0u;
      mk3 &= pi == 3 ? keep : ~0u;
      return cand;
    };
    const float* cbm = cb + (int64_t)m * K * D;
    const float* cnm = cn + (int64_t)m * K;
    const HalfPair cnt = halves((uint32_t)(__builtin_popcount(mk0) + __builtin_popcount(mk1) +
                                           __builtin_popcount(mk2) + __builtin_popcount(mk3)));
    const uint32_t ca = lowest(false);
    uint32_t cb2 = kNone;
    if (__ballot(cnt.lo + cnt.hi > 1 || all)) {
      lowest(true);
      cb2 = lowest(true);
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const uint32_t k0 = lane_read(ca, 16 * u + rho);
      uint32_t k = lane_read(cb2, 16 * u + rho);
      int code = k0 == kNone ? 0 : (int)k0;
      float c[NV];
      wide_row<D>(c, cbm + (int64_t)code * D, q);
      if (__ballot(k != kNone)) {
        // some row has several candidates (out of range: all entries): the
        // contract's distances decide.  Candidates come in ascending order,
        // so a tie keeps the earlier; NaN and +inf never win; with no finite
        // distance (rows that keep every entry) the first, entry 0, stays.
        float best = (rn[u] + cnm[code]) - 2.0f * wide_dot16<D>(r[u], c);
        bool have = !(best != best) && best != INFINITY;
        const int first = code;
#pragma unroll 1
        do {
          if (k != kNone) {
            float d[NV];
            wide_row<D>(d, cbm + (int64_t)k * D, q);
            const float E = (rn[u] + cnm[k]) - 2.0f * wide_dot16<D>(r[u], d);
            const bool win = !(E != E) && E != INFINITY && (!have || E < best);
            best = win ? E : best;
            code = win ? (int)k : code;
            have = have || win;
          }
          k = lane_read(lowest((n >> 4) == u), 16 * u + rho);
        } while (__ballot(k != kNone));
        if (code != first) wide_row<D>(c, cbm + (int64_t)code * D, q);
      }
#pragma unroll
      for (int i = 0; i < NV; ++i) r[u][i] = r[u][i] - c[i];
      rn[u] = wide_dot16<D>(r[u], r[u]);
      if (q == 0 && live[u]) crow[u][m] = (uint8_t)code;
    }
    if (m + 2 < M && in_step) {  // stage m + 2's fragments replace stage m's
      await(2 + (m & 1), (uint32_t)(WAVES * (m / 2 + 1)));
      if (in_step) request(m + 2);
    }
  }
#pragma unroll
  for (int u = 0; u < 2; ++u)
    if (q == 0 && live[u] && rnorm) rnorm[row0 + 16 * u] = sqrtf(rn[u]);
}

// ------------------------------------------ fewer rows than the chip has waves
// The same search and update for up to about two workgroups per CU, where the
// chain of a stage's dependent steps sets the time: R = 32 or 16 rows per
// workgroup of eight waves.  Wave w searches tile w for all R rows (its
// fragments come straight from L2 into registers, the next stage's requested
// as soon as this one's products are issued) and updates R / 8 rows, sixteen
// lanes per row, lane j the dot16 chain j; a maximum and a survivor mask per
// (row, tile) and the fp16 residual change hands through LDS, two barriers per
// stage.  R = 16 (16x16x32 products, half the work between the barriers) while
// every CU gets at most one workgroup of 16 rows.
constexpr int kSplitCodes = 32;  // codes of the first stages, stored after the last

template <int D, int R>
struct SplitShared {
  uint4 b[R * (D / 8)];  // fp16 residual, 16-byte units of a row permuted by the row
  uint2 m[R][8];         // per row and tile: maximum, entries within 2 eps of it
  float eps2[R];
  uint8_t code[R][kSplitCodes];
};

typedef float wf4_t __attribute__((ext_vector_type(4)));

// Maximum and union over lanes l, l ^ 16, l ^ 32, l ^ 48, in all of them.
__device__ __forceinline__ float quarter_max(float x) {
  const uint32_t u = __builtin_bit_cast(uint32_t, half_max(x));
  const auto p = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  const uint32_t a = p[0], b = p[1];  // (a bit cast of the element itself reads element 0)
  return __builtin_elementwise_maximum(__builtin_bit_cast(float, a),
                                       __builtin_bit_cast(float, b));
}
__device__ __forceinline__ uint32_t quarter_or(uint32_t x) {
  const HalfPair h = halves(x);
  const auto p = __builtin_amdgcn_permlane16_swap(h.lo | h.hi, h.lo | h.hi, false, false);
  return p[0] | p[1];
}

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xf, 0xf, false);
}

template <int D, int R>
__global__ __launch_bounds__(512, 4) void encode_split_kernel(
    RowMap rm, int N, const float* __restrict__ cb, int M, int K,
    const uint4* __restrict__ wide, const WideStage* __restrict__ stage,
    const float* __restrict__ cn, float* __restrict__ rnorm) {
  constexpr int KS = D / 16, L = D / 16, U = D / 8;  // units per row
  constexpr uint32_t kNone = 0x7fffu;
  static_assert(R == 16 || R == 32, "rows per workgroup");
  __shared__ __attribute__((aligned(16))) SplitShared<D, R> s;
  const int tid = threadIdx.x, lane = tid & 63;
  // search: row, and the half (R = 32) or quarter of the wave
  const int n = lane & (R - 1), h = lane / R;
  const int j = lane & 15;  // update: chain
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // update: row (R = 16: the upper half of the wave repeats the lower)
  const int lrow = R / 8 * wave + ((lane >> 4) & (R / 8 - 1)), row = blockIdx.x * R + lrow;
  const int NT = wide_tiles(K);
  const int64_t n16 = wide_stage_uint4(K, D);
  const bool live = row < N && rm.live(row);
  // a workgroup with no live row leaves at once
  if (rm.ranges && !__syncthreads_or(live)) return;

  // Waves past the last tile load it again and offer nothing.
  const int tile = min(wave, NT - 1);
  // bits of a tile's mask that stand for entries (entry e at bit 31 - e)
  auto entries = [&](int t) -> uint32_t {
    const int c = K - 32 * t;
    return c >= 32 ? ~0u : c > 0 ? ~0u << (32 - c) : 0u;
  };
  const uint32_t mine = wave < NT ? entries(wave) : 0u, theirs = entries(j & 7);
  // stage m's fragments of the tile: a uniform base each, and the lane.
  // Slot i: 32 rows, k-step i; 16 rows, k-steps 2 (i / 2) and 2 (i / 2) + 1 of
  // the tile's 16 entries i % 2 (operand A's quarter q is k-step q / 2, half
  // q % 2 of the pair).
  uint4 f[KS];
  uint2 hp[R == 32 ? 1 : 2];
  auto fragment = [&](int m, int i) {
    const uint4* base = wide + m * n16 + tile * KS * 64;
    return R == 32 ? base[i * 64 + lane]
                   : base[(i & ~1) * 64 + (i & 1) * 16 + (h >> 1) * 64 + (h & 1) * 32 + n];
  };
  auto part = [&](int m, int x) {
    return reinterpret_cast<const uint2*>(wide + m * n16 + NT * KS * 64)[tile * 32 + x * 16 + n];
  };
#pragma unroll
  for (int x = 0; x < (R == 32 ? 1 : 2); ++x) hp[x] = part(0, x);
#pragma unroll
  for (int i = 0; i < KS; ++i) f[i] = fragment(0, i);

  float r[L];
#pragma unroll
  for (int t = 0; t < L; ++t) r[t] = live ? rm.xval(row, j * L + t) : 0.f;
  float rn = 0.f, eps2 = 0.f;
  // new norm, 2 eps and fp16 residual of the row
  auto publish = [&](const WideStage& ws) {
    float a = 0.f;
#pragma unroll
    for (int t = 0; t < L; ++t) a = __builtin_fmaf(r[t], r[t], a);
    rn = row_fold16(a);
    eps2 = __builtin_fmaf(__builtin_amdgcn_sqrtf(rn), ws.e1, __builtin_fmaf(rn, ws.e2, ws.e0));
    if (j == 0) s.eps2[lrow] = eps2;
    if constexpr (L == 8) {  // chain j is unit j
      wh8_t x;
#pragma unroll
      for (int t = 0; t < 8; ++t) x[t] = (_Float16)r[t];
      s.b[lrow * U + (j ^ (lrow & 15))] = __builtin_bit_cast(uint4, x);
    } else {  // L = 4: chains 8v + q and 8v + 4 + q are the halves of unit 4v + q
      wh4_t x;
#pragma unroll
      for (int t = 0; t < 4; ++t) x[t] = (_Float16)r[t];
      const int u = 4 * (j >> 3) + (j & 3);
      reinterpret_cast<uint2*>(s.b)[(lrow * U + (u ^ (lrow & 7))) * 2 + ((j >> 2) & 1)] =
          __builtin_bit_cast(uint2, x);
    }
  };
  publish(stage[0]);
  wh4_t baug = {};
  if (h == 0) baug[0] = baug[1] = baug[2] = (_Float16)-64.f;
  lds_barrier();

  for (int m = 0; m < M; ++m) {
    const int mn = min(m + 1, M - 1);
    // ---- search: rows n, tile `tile`.  Each fragment's successor is requested
    // as soon as its product is issued: the eight waves' requests take the
    // vector memory unit about 1150 cycles, and issued in one block they held
    // up the sifting (and, issued later, the candidates' rows).
    const float re = s.eps2[n];
    const WideStage ws = stage[mn];
    float x;
    uint32_t w;  // the tile's entries within 2 eps of its maximum, entry e at bit 31 - e
    const uint4* br = s.b + n * U;
    if constexpr (R == 32) {
      wf16_t a = {};
      wh8_t bf[KS];
#pragma unroll
      for (int i = 0; i < KS; ++i)
        bf[i] = __builtin_bit_cast(wh8_t, br[(2 * i + h) ^ (n & (U - 1))]);
      a = __builtin_amdgcn_mfma_f32_32x32x8f16(__builtin_bit_cast(wh4_t, hp[0]), baug, a, 0, 0, 0);
      hp[0] = part(mn, 0);
#pragma unroll
      for (int i = 0; i < KS; ++i) {
        a = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(wh8_t, f[i]), bf[i], a, 0, 0,
                                                   0);
        f[i] = fragment(mn, i);
        __builtin_amdgcn_sched_barrier(0);
      }
      float y = __builtin_elementwise_maximum(a[2], a[3]);
      x = __builtin_elementwise_maximum(a[0], a[1]);
#pragma unroll
      for (int i = 4; i < 16; i += 4) {
        x = __builtin_elementwise_maximum(__builtin_elementwise_maximum(x, a[i]), a[i + 1]);
        y = __builtin_elementwise_maximum(__builtin_elementwise_maximum(y, a[i + 2]), a[i + 3]);
      }
      x = half_max(__builtin_elementwise_maximum(x, y));
      const float thr = x - re;
      uint32_t w0 = 0, w1 = 0;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        w0 = __builtin_amdgcn_alignbit(w0, __builtin_bit_cast(uint32_t, a[i] - thr), 31);
        w1 = __builtin_amdgcn_alignbit(w1, __builtin_bit_cast(uint32_t, a[8 + i] - thr), 31);
      }
      w = ~((w0 << 8) | w1) & 0xffffu;  // register i at bit 15 - i
      // registers 4g .. 4g + 3 of half h are entries 8g + 4h ..
      w = (w | (w << 8)) & 0x00ff00ffu;
      w = (w | (w << 4)) & 0x0f0f0f0fu;
      const HalfPair wp = halves(w);
      w = (wp.lo << 4) | wp.hi;
    } else {
      wf4_t a[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
      wh8_t bf[KS / 2];
#pragma unroll
      for (int i = 0; i < KS / 2; ++i)
        bf[i] = __builtin_bit_cast(wh8_t, br[(4 * i + h) ^ (n & (U - 1))]);
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        a[e] = __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(wh4_t, hp[e]), baug, a[e],
                                                     0, 0, 0);
        hp[e] = part(mn, e);
      }
#pragma unroll
      for (int i = 0; i < KS; ++i) {
        a[i & 1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(wh8_t, f[i]),
                                                          bf[i / 2], a[i & 1], 0, 0, 0);
        f[i] = fragment(mn, i);
        __builtin_amdgcn_sched_barrier(0);
      }
      x = __builtin_elementwise_maximum(a[0][0], a[0][1]);
      float y = __builtin_elementwise_maximum(a[1][0], a[1][1]);
      x = __builtin_elementwise_maximum(__builtin_elementwise_maximum(x, a[0][2]), a[0][3]);
      y = __builtin_elementwise_maximum(__builtin_elementwise_maximum(y, a[1][2]), a[1][3]);
      x = quarter_max(__builtin_elementwise_maximum(x, y));
      const float thr = x - re;
      uint32_t w0 = 0, w1 = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        w0 = __builtin_amdgcn_alignbit(w0, __builtin_bit_cast(uint32_t, a[0][i] - thr), 31);
        w1 = __builtin_amdgcn_alignbit(w1, __builtin_bit_cast(uint32_t, a[1][i] - thr), 31);
      }
      // register i of quarter h is entry 4h + i of the 16
      w = quarter_or((((~w0 & 15u) << 16) | (~w1 & 15u)) << (12 - 4 * h));
    }
    if (h == 0)
      s.m[n][wave] = make_uint2(mine ? __builtin_bit_cast(uint32_t, x) : 0xff800000u, w & mine);
    lds_barrier();

    // ---- update: row lrow, lanes j; lanes 8 .. 15 repeat tiles 0 .. 7
    const float* cbm = cb + (int64_t)m * K * D + j * L;
    const float* cnm = cn + (int64_t)m * K;
    const uint2 mw = s.m[lrow][j & 7];
    const float mx = __builtin_bit_cast(float, mw.x);
    float top = __builtin_elementwise_maximum(mx, dpp_f<0x124>(mx));
    top = __builtin_elementwise_maximum(top, dpp_f<0x122>(top));
    top = __builtin_elementwise_maximum(top, dpp_f<0x121>(top));
    const bool all = !(eps2 < 0x1p60f) || !(rn < 0x1p30f);  // outside the fp16 range
    uint32_t keep = all ? theirs : mx >= top - eps2 ? mw.y : 0u;
    uint32_t cnt = (uint32_t)__builtin_popcount(keep);
    cnt += dpp_u32<0x124>(cnt);
    cnt += dpp_u32<0x122>(cnt);
    cnt += dpp_u32<0x121>(cnt);
    // lowest candidate of the row (kNone: none); drop: takes it out
    auto lowest = [&](bool drop) -> uint32_t {
      const uint32_t b = (uint32_t)__builtin_clz(keep | 1u);
      const uint32_t own = keep ? 32u * (uint32_t)(j & 7) + b : kNone;
      uint32_t c = min(own, dpp_u32<0x124>(own));
      c = min(c, dpp_u32<0x122>(c));
      c = min(c, dpp_u32<0x121>(c));
      if (drop && own == c && c != kNone) keep &= ~(0x80000000u >> b);
      return c;
    };
    auto fetch = [&](float (&c)[L], uint32_t k) {
#pragma unroll
      for (int t = 0; t < L; t += 4) {
        const float4 v = *reinterpret_cast<const float4*>(cbm + (int64_t)k * D + t);
        c[t] = v.x;
        c[t + 1] = v.y;
        c[t + 2] = v.z;
        c[t + 3] = v.w;
      }
    };
    const uint32_t ca = lowest(false);
    int code = ca == kNone ? 0 : (int)ca;
    float c[L];
    fetch(c, (uint32_t)code);
    if (__ballot(cnt > 1)) {
      // as in the wide kernel: the contract's distances decide between several
      // candidates, the lowest entry on a tie; NaN and +inf never win.  Rows
      // without a second candidate read entry 0.
      const float cna = cnm[code];
      if (((uint32_t)code >> 5) == (uint32_t)(j & 7)) keep &= ~(0x80000000u >> (code & 31));
      uint32_t cd = lowest(true);
      float d[L], cnd = cnm[cd == kNone ? 0 : cd];
      fetch(d, cd == kNone ? 0 : cd);
      auto distance = [&](const float (&v)[L], float cnk) {
        float dot = 0.f;
#pragma unroll
        for (int t = 0; t < L; ++t) dot = __builtin_fmaf(r[t], v[t], dot);
        return (rn + cnk) - 2.0f * row_fold16(dot);
      };
      float best = distance(c, cna);
      bool have = !(best != best) && best != INFINITY;
      for (;;) {
        const float E = distance(d, cnd);
        const bool win = cd != kNone && !(E != E) && E != INFINITY && (!have || E < best);
        best = win ? E : best;
        code = win ? (int)cd : code;
        have = have || win;
#pragma unroll
        for (int t = 0; t < L; ++t) c[t] = win ? d[t] : c[t];
        cd = lowest(true);
        if (!__ballot(cd != kNone)) break;
        cnd = cnm[cd == kNone ? 0 : cd];
        fetch(d, cd == kNone ? 0 : cd);
      }
    }
#pragma unroll
    for (int t = 0; t < L; ++t) r[t] = r[t] - c[t];
    publish(ws);
    if (j == 0) {
      if (m < kSplitCodes) s.code[lrow][m] = (uint8_t)code;
      else if (live) rm.crow(row)[m] = (uint8_t)code;
    }
    lds_barrier();
  }
  const int mc = M < kSplitCodes ? M : kSplitCodes;
  for (int i = tid; i < R * mc; i += 512) {
    const int rr = i / mc, mm = i - rr * mc, gr = blockIdx.x * R + rr;
    if (gr < N && rm.live(gr)) rm.crow(gr)[mm] = s.code[rr][mm];
  }
  if (j == 0 && live && rnorm) rnorm[row] = sqrtf(rn);
}

}  // namespace
}  // namespace lap
