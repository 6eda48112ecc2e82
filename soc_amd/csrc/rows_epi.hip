// rows_epi.hip - the second half of a ragged decode batch's projections beyond 16 rows: the split-K partial sums that
// launch_gemm_rows leaves ([split][row][N], fp32) added in split order, and what follows the projection in the layer.
// A row's result does not depend on what the other rows hold or where they stand; the number of splits, and with it the
// order of a row's sums, follows the number of row tiles (rows_plan in gemm.hip). Bound by the partials' round trip (they stay in L2 and the
// memory-side cache) and the launch; every load of a thread's sums goes out before the first add.
#include "kernels.h"

namespace soc {
namespace {

// Sum over the splits, in order, of 4 adjacent columns of a row's partials (stride: floats from split to split).
__device__ __forceinline__ f32x4 sum_splits(const float* p, size_t stride, int splits) {
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
  for (int k = 0; k < splits; k += 8) {
    f32x4 x[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) x[u] = *reinterpret_cast<const f32x4*>(p + min(k + u, splits - 1) * stride);
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (k + u < splits) v += x[u];
  }
  return v;
}

// hi = f16(y), lo = f16((y - hi) 2^11). y is materialised first: left to itself the compiler stores hi rounded from the
// fp32 product y = a b but takes lo against hi rounded from the unrounded a b (v_fma_mixlo_f16), and where the two
// roundings differ the pair is off by an ulp of hi (1e-5 to 6e-5 of a row's norm, in about one row in ten).
__device__ __forceinline__ void split_pair(const f32x4& y, f16x4* hi, f16x4* lo) {
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    float v = y[c];
    __asm__ volatile("" : "+v"(v));
    (*hi)[c] = static_cast<f16>(v);
    (*lo)[c] = static_cast<f16>((v - static_cast<float>((*hi)[c])) * 2048.0f);
  }
}

// One block per row: x += the sums, then RMSNorm(x) * gain (rms_norm_module.cpp:56-64) as a hi/lo pair for the next
// projection. V4: 4-column pieces per thread.
template <int V4>
__global__ __launch_bounds__(256) void k_rows_residual_norm(const float* part, int splits, int M, int H, float* x,
                                                             const f16* gain, float eps, f16* yh, f16* yl) {
  __shared__ float red[4];
  const int m = blockIdx.x, tid = threadIdx.x, nv = H / 4;
  const size_t stride = static_cast<size_t>(M) * H, row = static_cast<size_t>(m) * H;
  f32x4 v[V4];
  f16x4 g[V4];
  float ss = 0.0f;
#pragma unroll
  for (int e = 0; e < V4; ++e) {
    const int i = min(tid + 256 * e, nv - 1);
    const f32x4 prev = *reinterpret_cast<const f32x4*>(x + row + 4 * i);
    g[e] = *reinterpret_cast<const f16x4*>(gain + 4 * i);
    v[e] = prev + sum_splits(part + row + 4 * i, stride, splits);
    if (tid + 256 * e < nv) {
      *reinterpret_cast<f32x4*>(x + row + 4 * i) = v[e];
#pragma unroll
      for (int c = 0; c < 4; ++c) ss = fmaf(v[e][c], v[e][c], ss);
    }
  }
  ss = block_sum<256>(ss, red);
  const float scale = 1.0f / sqrtf(ss / static_cast<float>(H) + eps);
#pragma unroll
  for (int e = 0; e < V4; ++e) {
    const int i = tid + 256 * e;
    if (i >= nv) break;
    f32x4 y;
#pragma unroll
    for (int c = 0; c < 4; ++c) y[c] = v[e][c] * scale * static_cast<float>(g[e][c]);
    f16x4 hi, lo;
    split_pair(y, &hi, &lo);
    *reinterpret_cast<f16x4*>(yh + row + 4 * i) = hi;
    *reinterpret_cast<f16x4*>(yl + row + 4 * i) = lo;
  }
}

// h = silu(gate) * up of the [gate | up] sums (qwen_mlp.cpp:69-72) as a hi/lo pair; grid (column pieces, rows).
__global__ __launch_bounds__(256) void k_rows_swiglu(const float* part, int splits, int M, int I, f16* yh, f16* yl) {
  const int i = 4 * (blockIdx.x * 256 + threadIdx.x), m = blockIdx.y;
  if (i >= I) return;
  const size_t stride = static_cast<size_t>(M) * 2 * I;
  const float* p = part + static_cast<size_t>(m) * 2 * I + i;
  const f32x4 g = sum_splits(p, stride, splits), u = sum_splits(p + I, stride, splits);
  f32x4 y;
#pragma unroll
  for (int c = 0; c < 4; ++c) y[c] = silu_ref(g[c]) * u[c];
  f16x4 hi, lo;
  split_pair(y, &hi, &lo);
  const size_t o = static_cast<size_t>(m) * I + i;
  *reinterpret_cast<f16x4*>(yh + o) = hi;
  *reinterpret_cast<f16x4*>(yl + o) = lo;
}

// The attention input: one wave per (row, head); q and k heads get their RMSNorm and RoPE at pos[row]
// (qwen_attention.cpp:168-171; rope.cpp:81-84), k and v go to the fp16 cache of the row's slot.
__global__ __launch_bounds__(64) void k_rows_qkv(const float* part, int splits, QkNormRopeArgs a) {
  const int m = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  const int N = (a.nq + 2 * a.nkv) * 128;
  const size_t stride = static_cast<size_t>(a.T) * N;
  const float* p = part + static_cast<size_t>(m) * N + h * 128 + lane;
  const int pos = a.pos[m], slot = a.slots[m];
  const bool normed = h < a.nq + a.nkv;
  float g0 = 1.0f, g1 = 1.0f, c = 0.0f, sn = 0.0f;
  if (normed) {
    const f16* gn = h < a.nq ? a.q_gain : a.k_gain;
    g0 = static_cast<float>(ld_global(gn, lane));
    g1 = static_cast<float>(ld_global(gn, lane + 64));
    c = a.rope_cos[static_cast<size_t>(pos) * 64 + lane];
    sn = a.rope_sin[static_cast<size_t>(pos) * 64 + lane];
  }
  float x0 = 0.0f, x1 = 0.0f;
  for (int k = 0; k < splits; k += 8) {
    float u0[8], u1[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const float* q = p + min(k + u, splits - 1) * stride;
      u0[u] = q[0];
      u1[u] = q[64];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (k + u < splits) {
        x0 += u0[u];
        x1 += u1[u];
      }
  }
  if (normed) norm_rope_pair(x0, x1, g0, g1, a.eps, c, sn);
  if (h < a.nq) {
    float* dst = a.q_out + static_cast<size_t>(m) * a.nq * 128 + h * 128;
    dst[lane] = x0;
    dst[lane + 64] = x1;
  } else {
    const int kvh = normed ? h - a.nq : h - a.nq - a.nkv;
    f16* cache = (normed ? a.kcache : a.vcache) + static_cast<size_t>(slot) * a.slot_stride +
                 static_cast<size_t>(a.layer) * a.layer_stride +
                 (static_cast<size_t>(kvh) * a.cap + static_cast<size_t>(pos)) * 128;
    cache[lane] = static_cast<f16>(x0);
    cache[lane + 64] = static_cast<f16>(x1);
  }
}

}  // namespace

hipError_t launch_rows_residual_norm(const float* part, int splits, int M, int H, float* x, const f16* gain, float eps,
                                     f16* yh, f16* yl, hipStream_t s) {
  if (M <= 0 || splits <= 0 || H <= 0 || H % 4 != 0 || H > 16384) return hipErrorInvalidValue;
  const int nv = H / 4;
#define SOC_ROWS_NORM(V) \
  hipLaunchKernelGGL(k_rows_residual_norm<V>, dim3(M), dim3(256), 0, s, part, splits, M, H, x, gain, eps, yh, yl)
  if (nv <= 256) SOC_ROWS_NORM(1);
  else if (nv <= 512) SOC_ROWS_NORM(2);
  else if (nv <= 1024) SOC_ROWS_NORM(4);
  else SOC_ROWS_NORM(16);
#undef SOC_ROWS_NORM
  return hipGetLastError();
}

hipError_t launch_rows_swiglu(const float* part, int splits, int M, int I, f16* yh, f16* yl, hipStream_t s) {
  if (M <= 0 || splits <= 0 || I <= 0 || I % 4 != 0) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_rows_swiglu, dim3((I / 4 + 255) / 256, M), dim3(256), 0, s, part, splits, M, I, yh, yl);
  return hipGetLastError();
}

hipError_t launch_rows_qkv(const float* part, int splits, const QkNormRopeArgs& a, hipStream_t s) {
  if (a.T <= 0 || splits <= 0 || a.pos == nullptr || a.slots == nullptr) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_rows_qkv, dim3(a.T, a.nq + 2 * a.nkv), dim3(64), 0, s, part, splits, a);
  return hipGetLastError();
}

}  // namespace soc
