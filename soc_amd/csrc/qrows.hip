// qrows.hip - group-quantized projections of 1..8 activation rows (int8 / int4 codes, fp16 scale per 64 inputs) on
// matrix cores, with the steps around a decode projection fused in: y[m][n] = sum_g scale[n][g] *
// sum_{k in group g} x[m][k] * code[n][k], the products exact and summed in fp32 per group.
//
// One row runs on the vector ALUs (k_qgemv), two to eight on the matrix cores (k_qrows). MI355X, us per call, against the
// kernels these replaced: one row 2560 x 9728 int4 9.1 -> 6.6, int8 12.0 -> 8.1, 151936 x 1024 int4 16.2 -> 15.4; eight
// rows 1024 x 3072 int4 14.4 -> 5.1, 2560 x 4096 int8 33.4 -> 7.9, 100000 x 2560 int4 121 -> 33 (4.0 TB/s).
//
// A projection of a few rows is a stream of codes, K/2 or K bytes per output, and at the sizes of one layer the
// latency of its loads: a block of k_qrows takes 16 output rows at a time and its waves split K, so that even 1024 outputs keep
// 64 blocks loading and a wave has one to four 16-byte loads per lane to wait for. The activations of a wave's part of
// K are loaded once, straight into registers in the operand layout of v_mfma_f32_16x16x32_f16 (no LDS staging, no
// barrier before the first product), and stay there while the block walks its row tiles; the next tile's codes are in
// flight while the current one is multiplied. The waves' partial sums meet in LDS, one barrier per tile, added in wave
// order.
//
// An input RMSNorm (rms_norm_module.cpp:56-64) is computed by every block for itself (a row is a few KB of L2), the
// normalised value rounded to fp16 as the unfused kernels round it; the residual add and SwiGLU
// (qwen_block.cpp:70-72, qwen_mlp.cpp:69-72) happen as the sums are stored.
#include "kernels.h"

#include <algorithm>

namespace soc {
namespace {

typedef _Float16 qr_h2 __attribute__((ext_vector_type(2)));
typedef _Float16 qr_h8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ qr_h2 qr_as_h2(uint32_t v) { return __builtin_bit_cast(qr_h2, v); }

// 16 codes -> 16 exact fp16 values as two MFMA operands of 8. int8: four dwords, k in order. int4: two dwords, each
// holding 8 codes that come out in the order 0 4 1 5 2 6 3 7 (the codes are placed in the low mantissa bits of 1024.0
// by a byte permute or a mask and xor, and one packed fp16 subtract, or multiply-add for the upper nibbles, leaves the
// code; every step is exact).
__device__ __forceinline__ void qr_unpack8(const u32x4& w, qr_h8 (&out)[2]) {
  const qr_h2 bias = {static_cast<_Float16>(-1152.0f), static_cast<_Float16>(-1152.0f)};
  qr_h2 p[8];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t u = w[j] ^ 0x80808080u;  // code + 128 per byte
    p[2 * j] = qr_as_h2(__builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) + bias;
    p[2 * j + 1] = qr_as_h2(__builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) + bias;
  }
#pragma unroll
  for (int h = 0; h < 2; ++h)
    out[h] = qr_h8{p[4 * h][0], p[4 * h][1], p[4 * h + 1][0], p[4 * h + 1][1],
                   p[4 * h + 2][0], p[4 * h + 2][1], p[4 * h + 3][0], p[4 * h + 3][1]};
}
__device__ __forceinline__ qr_h8 qr_unpack4(uint32_t u) {
  const qr_h2 bias = {static_cast<_Float16>(-1032.0f), static_cast<_Float16>(-1032.0f)};
  const qr_h2 bias16 = {static_cast<_Float16>(-72.0f), static_cast<_Float16>(-72.0f)};
  const qr_h2 sixteenth = {static_cast<_Float16>(0.0625f), static_cast<_Float16>(0.0625f)};
  const uint32_t v = u >> 8;
  const qr_h2 a = qr_as_h2((u & 0x000F000Fu) ^ 0x64086408u) + bias;
  const qr_h2 b = qr_as_h2((u & 0x00F000F0u) ^ 0x64806480u) * sixteenth + bias16;
  const qr_h2 c = qr_as_h2((v & 0x000F000Fu) ^ 0x64086408u) + bias;
  const qr_h2 d = qr_as_h2((v & 0x00F000F0u) ^ 0x64806480u) * sixteenth + bias16;
  return qr_h8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

enum { QX_F16 = 0, QX_F32 = 1, QX_NORM = 2 };  // activations: fp16 rows; fp32 rows rounded; RMSNorm of fp32 rows

// A unit is one 16-byte code load per lane over 16 rows: 64 bytes of each row, 128 int4 or 64 int8 codes. Wave w of
// the eight takes units w, w + 8, ..., UW of them per pass over K, so that the waves' loads of a row are adjacent.
// Lane (r, q) = (lane % 16, lane / 16) loads row r; as the MFMA's A operand it stands for activation row r, as its D
// column for output row r. int8: the lane's 16 codes are k = 64 u + 16 q .. of group u. int4: its 32 codes are
// k = 128 u + 32 q .., and one v_permlane32_swap per dword pair gives every lane 16 codes of each of the unit's two
// groups, at k offset 16 * (0, 2, 1, 3)[q] of the group (an odd number of groups leaves the last unit half empty:
// those lanes hold zeros). With K over 8 UW units (LONG) the activations do not stay in registers: each pass of each
// tile loads its part again.
// Waves over K: KW of the eight; the block's 8 / KW wave groups take neighbouring tiles. Sums meet in LDS four tiles at a
// time, one barrier for the four and one output per thread.
template <int BITS, int UW, int KW, bool LONG, int XF, int EPI>
__global__ __launch_bounds__(512, XF == QX_F16 && KW == 8 && !LONG && UW * BITS <= (BITS == 4 ? 12 : 48) ? 4 : 2) void
k_qrows(QRowsArgs a) {
  constexpr int TW = 8 / KW;               // tiles side by side
  constexpr int TS = 4 / TW;               // tiles one after the other between barriers
  // the next tile's codes requested a tile ahead, but where holding both spills (24 of 128 registers: int8, UW = 6)
  constexpr bool AHEAD = !(BITS == 8 && UW == 6 && !LONG && XF == QX_F16);
  static_assert(KW == 8 || (XF == QX_F16 && EPI == EPI_STORE && !LONG && KW >= 2), "wave groups");
  constexpr int GPU = BITS == 4 ? 2 : 1;   // scale groups per unit
  constexpr int KU = 64 * GPU;             // codes of a row per unit
  __shared__ float red[2][4][KW][8][17];
  __shared__ float ssw[8];
  const int tid = threadIdx.x, lane = tid & 63, wid = (tid >> 6) % KW, wg = (tid >> 6) / KW;
  const int rl = lane & 15, kq = lane >> 4;
  const int K = a.K, G = K / 64, nu = (K + KU - 1) / KU, M = a.M;
  const size_t rowbytes = BITS == 4 ? static_cast<size_t>(K) / 2 : static_cast<size_t>(K);
  const int half = a.N / 2;                       // SwiGLU: gate rows [0, half), up rows [half, N)
  const int nout = EPI == EPI_SWIGLU ? half : a.N;
  constexpr int TO = EPI == EPI_SWIGLU ? 8 : 16;  // outputs per tile
  const int ntiles = (nout + TO - 1) / TO;
  const int npass = LONG ? (nu + KW * UW - 1) / (KW * UW) : 1;
  const int kb = BITS == 4 ? 16 * ((kq & 1) * 2 + (kq >> 1)) : 16 * kq;

  // The scales of four units in one load: lane (r, q) loads those of unit 4 j + q of row r (int4: both groups, one
  // dword), and two lane swaps hand each unit's to all four q (a load per unit would cost as many cache lookups as the
  // codes themselves: 16 rows, 16 lines)
  constexpr int SJ = (UW + 3) / 4;
  struct Codes {
    u32x4 w[UW];
    uint32_t s[SJ];
  };
  auto load = [&](Codes& c, int tile, int pass) {
    int row;
    if constexpr (EPI == EPI_SWIGLU) row = min(tile * 8 + (rl & 7), half - 1) + (rl >> 3) * half;
    else row = min(tile * 16 + rl, a.N - 1);
    const uint8_t* cp = static_cast<const uint8_t*>(a.codes) + row * rowbytes;
    const f16* sp = a.scales + static_cast<size_t>(row) * G;
#pragma unroll
    for (int i = 0; i < UW; ++i) {
      const int u = min(wid + KW * (pass * UW + i), nu - 1);  // units past the wave's last re-read it, unused
      const size_t off = static_cast<size_t>(u) * 64 + kq * 16;
      c.w[i] = load16(cp + (off + 16 <= rowbytes ? off : rowbytes - 16));
    }
#pragma unroll
    for (int j = 0; j < SJ; ++j) {
      const int u = min(wid + KW * (pass * UW + min(4 * j + kq, UW - 1)), nu - 1);
      if constexpr (BITS == 4) {  // (half-aligned where G is odd)
        if (G == 1) {
          c.s[j] = __builtin_bit_cast(uint16_t, ld_global(sp, 0));
        } else {
          const bool tail = 2 * u > G - 2;  // the last group alone: the upper half of the dword before
          uint32_t v;
          __builtin_memcpy(&v, sp + (tail ? G - 2 : 2 * u), 4);
          c.s[j] = tail ? v >> 16 : v;
        }
      } else {
        c.s[j] = __builtin_bit_cast(uint16_t, ld_global(sp, u));
      }
    }
  };

  // the block's tiles in steps of TW neighbours: steps blockIdx.x, blockIdx.x + gridDim.x, ... < nsteps; a wave group
  // past the last tile works on it again and stores nothing
  const int nsteps = (ntiles + TW - 1) / TW;
  Codes cur;
  int step = blockIdx.x, pass = 0;  // grid <= nsteps
  load(cur, min(step * TW + wg, ntiles - 1), 0);

  // 1 / rms of the activation rows: the block's waves share each row's squares
  float rs = 1.0f;
  if constexpr (XF == QX_NORM) {
    const int P = M > 4 ? 1 : M > 2 ? KW / 4 : M > 1 ? KW / 2 : KW;  // waves per row
    const int m = wid / P, part = wid % P;
    float ss = 0.0f;
    if (m < M) {
      const float* xr = a.x + static_cast<size_t>(m) * K;
      for (int k = part * 256 + 4 * lane; k < K; k += 256 * P) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(xr + k);
#pragma unroll
        for (int e = 0; e < 4; ++e) ss = fmaf(v[e], v[e], ss);
      }
      ss = wave_sum(ss);
    }
    if (lane == 0) ssw[wid] = ss;
    __syncthreads();
    float t = 0.0f;
    const int mr = min(rl, M - 1);
    for (int p = 0; p < P; ++p) t += ssw[mr * P + p];
    rs = 1.0f / sqrtf(t / static_cast<float>(K) + a.eps);
  }

  // the wave's activations of one pass as MFMA operands (rows past M and k past K are zeros)
  qr_h8 xa[UW][2 * GPU];
  auto load_x = [&](int ps) {
#pragma unroll
    for (int i = 0; i < UW; ++i) {
      const int u = wid + KW * (ps * UW + i);
#pragma unroll
      for (int h = 0; h < 2 * GPU; ++h) {
        const int k = u * KU + (h >> 1) * 64 + kb + (h & 1) * 8;
        const bool ok = rl < M && u < nu && k < K;
        const size_t at = static_cast<size_t>(min(rl, M - 1)) * K + min(k, K - 8);
        f16x8 v;
        if constexpr (XF == QX_F16) {
          v = as_f16x8(load16(a.xh + at));
        } else {
          const f32x4 p = *reinterpret_cast<const f32x4*>(a.x + at), q = *reinterpret_cast<const f32x4*>(a.x + at + 4);
          float f[8] = {p[0], p[1], p[2], p[3], q[0], q[1], q[2], q[3]};
          if constexpr (XF == QX_NORM) {
            const f16x8 gn = as_f16x8(load16(a.gain + min(k, K - 8)));
#pragma unroll
            for (int e = 0; e < 8; ++e) f[e] = f[e] * rs * static_cast<float>(gn[e]);
          }
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = static_cast<f16>(f[e]);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int src = BITS == 4 ? ((e & 1) * 4 + (e >> 1)) : e;
          xa[i][h][e] = ok ? v[src] : static_cast<f16>(0.0f);
        }
      }
    }
  };
  if constexpr (!LONG) load_x(0);

  int buf = 0, held = 0, first = step;  // steps whose sums wait in red[buf], and the first of them
  f32x4 acc = {0.f, 0.f, 0.f, 0.f}, acc2 = {0.f, 0.f, 0.f, 0.f};  // alternate groups: half the length of either sum
  while (step < nsteps) {
    const bool done = pass == npass - 1;  // the step's last pass
    const int nstep = done ? step + static_cast<int>(gridDim.x) : step, nps = done ? 0 : pass + 1;
    uint32_t sc[4 * SJ];  // scales of each unit, in every lane of the row
#pragma unroll
    for (int j = 0; j < SJ; ++j) {
      const auto h = __builtin_amdgcn_permlane32_swap(cur.s[j], cur.s[j], false, false);
      const auto lo = __builtin_amdgcn_permlane16_swap(h[0], h[0], false, false);
      const auto hi = __builtin_amdgcn_permlane16_swap(h[1], h[1], false, false);
      sc[4 * j] = lo[0];
      sc[4 * j + 1] = lo[1];
      sc[4 * j + 2] = hi[0];
      sc[4 * j + 3] = hi[1];
    }
    if constexpr (LONG) load_x(pass);
    Codes nxt;
    if (AHEAD && nstep < nsteps) load(nxt, min(nstep * TW + wg, ntiles - 1), nps);
#pragma unroll
    for (int i = 0; i < UW; ++i) {
      const int u = wid + KW * (pass * UW + i);
      if (u >= nu) break;  // wave-uniform
      u32x4 w = cur.w[i];
      if constexpr (BITS == 8) {
        qr_h8 p[2];
        qr_unpack8(w, p);
        f32x4 d = {0.f, 0.f, 0.f, 0.f};
        d = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[i][0], p[0], d, 0, 0, 0);
        d = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[i][1], p[1], d, 0, 0, 0);
        const float s = static_cast<float>(qr_as_h2(sc[i])[0]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (i & 1) acc2[e] = fmaf(d[e], s, acc2[e]);
          else acc[e] = fmaf(d[e], s, acc[e]);
        }
      } else {
        if (u * KU + 32 * kq >= K) w = u32x4{0, 0, 0, 0};  // the empty half of the last unit
        const auto s02 = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
        const auto s13 = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
        f32x4 d0 = {0.f, 0.f, 0.f, 0.f}, d1 = {0.f, 0.f, 0.f, 0.f};
        d0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[i][0], qr_unpack4(s02[0]), d0, 0, 0, 0);
        d0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[i][1], qr_unpack4(s13[0]), d0, 0, 0, 0);
        d1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[i][2], qr_unpack4(s02[1]), d1, 0, 0, 0);
        d1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[i][3], qr_unpack4(s13[1]), d1, 0, 0, 0);
        const float s0 = static_cast<float>(qr_as_h2(sc[i])[0]), s1 = static_cast<float>(qr_as_h2(sc[i])[1]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          acc[e] = fmaf(d0[e], s0, acc[e]);
          acc2[e] = fmaf(d1[e], s1, acc2[e]);
        }
      }
    }
    if (!AHEAD && nstep < nsteps) load(cur, min(nstep * TW + wg, ntiles - 1), nps);
    if (done) {
      // D: the lane holds activation rows 4 kq .. 4 kq + 3 of output row rl
      if (kq < 2)
#pragma unroll
        for (int e = 0; e < 4; ++e) red[buf][held * TW + wg][wid][4 * kq + e][rl] = acc[e] + acc2[e];
      acc = acc2 = f32x4{0.f, 0.f, 0.f, 0.f};
      ++held;
      if (held == TS || nstep >= nsteps) {
        __syncthreads();
        const int sl = tid >> 7, m = (tid >> 4) & 7, c = tid & 15;
        const int t = (first + (sl / TW) * static_cast<int>(gridDim.x)) * TW + sl % TW;
        if (sl < held * TW && t < ntiles && m < M && (EPI != EPI_SWIGLU || c < 8)) {
          const int n = t * TO + c;
          // the waves' sums in float64: seven fp32 roundings of the whole result less
          double vd = 0.0, gd = 0.0;
#pragma unroll
          for (int w = 0; w < KW; ++w) vd += static_cast<double>(red[buf][sl][w][m][c]);
          if constexpr (EPI == EPI_SWIGLU) {
#pragma unroll
            for (int w = 0; w < KW; ++w) gd += static_cast<double>(red[buf][sl][w][m][c + 8]);
          }
          const float v = static_cast<float>(vd), g = static_cast<float>(gd);
          if (n < nout) {
            const size_t o = static_cast<size_t>(m) * nout + n;
            if constexpr (EPI == EPI_SWIGLU) a.yh[o] = static_cast<f16>(silu_ref(v) * g);
            else if constexpr (EPI == EPI_RESIDUAL) a.y[o] += v;
            else a.y[o] = v;
          }
        }
        buf ^= 1;
        held = 0;
        first = nstep;
      }
    }
    if (AHEAD && nstep < nsteps) cur = nxt;
    step = nstep;
    pass = nps;
  }
}

// group_sum<L> with the sums of 16 lanes added in float64 (two to four terms: one rounding instead of up to two levels),
// for soc_qmm.
template <int L>
__device__ __forceinline__ float row_sum(float v) {
  if constexpr (L <= 16) {
    return group_sum<L>(v);
  } else {
    v = group_sum<16>(v);
    const double r0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0));
    const double r1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 16));
    const double r2 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 32));
    const double r3 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 48));
    if constexpr (L == 64) return static_cast<float>((r0 + r1) + (r2 + r3));
    else return static_cast<float>((threadIdx.x & 32) ? r2 + r3 : r0 + r1);
  }
}

// One activation row: the codes are a plain stream, so a wave takes whole rows, L lanes side by side on each (1 KB of a
// row per load instruction where it is long enough), and the dot products run on the vector ALUs
// (v_dot2_f32_f16 on the unpacked pairs; 16 rows of 64 bytes per load, as the matrix cores want them, stream more
// slowly). RR rows per lane group are in flight at once, U chunks of each; the first are requested before the
// activations are staged (fp16 in the codes' order, in LDS). SwiGLU: RR gate rows and their up rows.
//
// Inside a model's layers the sums keep the order of the separate kernels (k_qmm, k_rmsnorm_rows_v) that these forms
// fused: a chunk's products in one chain, a row's lanes by group_sum, the squares of RMSNorm by one wave. Every
// projection rounds its input to fp16, so another order of fp32 sums flips roundings that travel through the layers
// (3e-4 to 6e-4 of the logits over four layers, as far from 64 bits on average: 6.9e-4 and 7.0e-4). soc_qmm (QX_F16,
// EPI_STORE), whose sums are its result, takes four chains and row_sum.
template <int BITS, int L, int RR, int U, int XF, int EPI>
__global__ __launch_bounds__(256) void k_qgemv(QRowsArgs a) {
  extern __shared__ __attribute__((aligned(16))) u32x4 qx[];  // [K / 8]
  constexpr int CH = BITS == 8 ? 16 : 32;         // codes per 16-byte chunk
  constexpr int RP = 64 / L;                      // lane groups
  constexpr bool AHEAD = RR == 1;                 // (tall matrices: more waves resident instead)
  constexpr int RA = EPI == EPI_SWIGLU ? 2 * RR : RR;
  constexpr bool QMM = XF == QX_F16 && EPI == EPI_STORE;
  const int tid = threadIdx.x, lane = tid & 63, sub = lane / L, ln = lane % L;
  const int K = a.K, nch = K / CH, G = K / 64;
  const int nout = EPI == EPI_SWIGLU ? a.N / 2 : a.N;
  const size_t rowbytes = BITS == 8 ? static_cast<size_t>(K) : static_cast<size_t>(K) / 2;
  const int wave = blockIdx.x * 4 + (tid >> 6), nwaves = gridDim.x * 4;
  struct Chunks {
    u32x4 w[U][RA];
    f16 s[U][RA];
  };
  auto load = [&](Chunks& c, int base, int c0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int ch = min(c0 + u * L + ln, nch - 1);  // (chunks past the row are loaded and not used)
#pragma unroll
      for (int r = 0; r < RA; ++r) {
        const int out = min(base + (r % RR) * RP + sub, nout - 1);
        const int row = r < RR ? out : out + nout;
        c.w[u][r] = load_stream16(static_cast<const uint8_t*>(a.codes) + row * rowbytes + static_cast<size_t>(ch) * 16);
        c.s[u][r] = ld_global(a.scales, static_cast<size_t>(row) * G + ch * CH / 64);
      }
    }
  };
  int base = wave * RR * RP, c0 = 0;
  Chunks cur;
  load(cur, min(base, nout - 1), 0);

  // the row as fp16, 8 values per thread and step
  constexpr int KEEP = 2;
  float keep[KEEP][8];
  float rs = 1.0f;
  auto values = [&](int i, float (&f)[8]) {
    const f32x4 p = *reinterpret_cast<const f32x4*>(a.x + 8 * i), q = *reinterpret_cast<const f32x4*>(a.x + 8 * i + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      f[e] = p[e];
      f[4 + e] = q[e];
    }
  };
  if constexpr (XF == QX_NORM) {
#pragma unroll
    for (int u = 0; u < KEEP; ++u) values(min(tid + 256 * u, K / 8 - 1), keep[u]);
    // every wave sums the whole row's squares (a few KB of L1), four loads in flight: no barrier
    float ss = 0.0f;
    const int nv = K / 4;
    for (int i0 = lane; i0 < nv; i0 += 4 * 64) {
      f32x4 v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = *reinterpret_cast<const f32x4*>(a.x + 4 * min(i0 + 64 * u, nv - 1));
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (i0 + 64 * u < nv) {
          ss = i0 + u == lane ? fmaf(v[u][0], v[u][0], v[u][1] * v[u][1])
                              : fmaf(v[u][1], v[u][1], fmaf(v[u][0], v[u][0], ss));
          ss = fmaf(v[u][3], v[u][3], fmaf(v[u][2], v[u][2], ss));
        }
    }
    rs = 1.0f / sqrtf(wave_sum(ss) / static_cast<float>(K) + a.eps);
  }
  auto stage = [&](int i, const float (&f)[8]) {
    f16x8 v;
    if constexpr (XF == QX_NORM) {
      const f16x8 gn = as_f16x8(load16(a.gain + 8 * i));
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float y = f[e] * rs * static_cast<float>(gn[e]);
        __asm__ volatile("" : "+v"(y));  // rounded to fp32, then to fp16 (v_fma_mixlo_f16 would round once)
        v[e] = static_cast<f16>(y);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = static_cast<f16>(f[e]);
    }
    if constexpr (BITS == 4) v = f16x8{v[0], v[4], v[1], v[5], v[2], v[6], v[3], v[7]};
    qx[i] = __builtin_bit_cast(u32x4, v);
  };
  if constexpr (XF == QX_F16) {
    for (int i = tid; i < K / 8; i += 256) {
      f16x8 v = as_f16x8(load16(a.xh + 8 * i));
      if constexpr (BITS == 4) v = f16x8{v[0], v[4], v[1], v[5], v[2], v[6], v[3], v[7]};
      qx[i] = __builtin_bit_cast(u32x4, v);
    }
  } else {
#pragma unroll
    for (int u = 0; u < KEEP; ++u) {
      if (XF == QX_F32) values(min(tid + 256 * u, K / 8 - 1), keep[u]);
      if (tid + 256 * u < K / 8) stage(tid + 256 * u, keep[u]);
    }
    for (int i = tid + 256 * KEEP; i < K / 8; i += 256) {
      float f[8];
      values(i, f);
      stage(i, f);
    }
  }
  __syncthreads();

  float acc[RA];
#pragma unroll
  for (int r = 0; r < RA; ++r) acc[r] = 0.0f;
  while (base < nout) {  // no barrier below
    const bool done = c0 + U * L >= nch;
    const int nbase = done ? base + nwaves * RR * RP : base, nc0 = done ? 0 : c0 + U * L;
    Chunks nxt;
    if (AHEAD && nbase < nout) load(nxt, nbase, nc0);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int ch = c0 + u * L + ln;
      const bool in = ch < nch;
      const u32x4* xp = qx + min(ch, nch - 1) * (CH / 8);
      qr_h2 x[CH / 2];
#pragma unroll
      for (int q = 0; q < CH / 8; ++q) {
        const u32x4 v = xp[q];
#pragma unroll
        for (int t = 0; t < 4; ++t) x[4 * q + t] = qr_as_h2(v[t]);
      }
#pragma unroll
      for (int r = 0; r < RA; ++r) {
        constexpr int NC = QMM ? 4 : 1;  // chains: of four, each has a quarter of the roundings
        float ps[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if constexpr (BITS == 8) {
          qr_h8 p[2];
          qr_unpack8(cur.w[u][r], p);
#pragma unroll
          for (int q = 0; q < 8; ++q)
            ps[q % NC] = __builtin_amdgcn_fdot2(qr_h2{p[q >> 2][2 * (q & 3)], p[q >> 2][2 * (q & 3) + 1]}, x[q],
                                                ps[q % NC], false);
        } else {
#pragma unroll
          for (int d = 0; d < 4; ++d) {
            const qr_h8 p = qr_unpack4(cur.w[u][r][d]);
#pragma unroll
            for (int q = 0; q < 4; ++q)
              ps[q % NC] = __builtin_amdgcn_fdot2(qr_h2{p[2 * q], p[2 * q + 1]}, x[4 * d + q], ps[q % NC], false);
          }
        }
        const float part = QMM ? (ps[0] + ps[1]) + (ps[2] + ps[3]) : ps[0];
        acc[r] = in ? fmaf(static_cast<float>(cur.s[u][r]), part, acc[r]) : acc[r];
      }
    }
    if (done) {
#pragma unroll
      for (int r = 0; r < RA; ++r) {
        if constexpr (QMM) acc[r] = row_sum<L>(acc[r]);
        else acc[r] = group_sum<L>(acc[r]);
      }
#pragma unroll
      for (int r = 0; r < RR; ++r) {
        const int n = base + r * RP + sub;
        if (ln == 0 && n < nout) {
          if constexpr (EPI == EPI_SWIGLU) a.yh[n] = static_cast<f16>(silu_ref(acc[r]) * acc[r + RR]);
          else if constexpr (EPI == EPI_RESIDUAL) a.y[n] += acc[r];
          else a.y[n] = acc[r];
        }
      }
#pragma unroll
      for (int r = 0; r < RA; ++r) acc[r] = 0.0f;
    }
    if (nbase < nout) {
      if constexpr (AHEAD) cur = nxt;
      else load(cur, nbase, nc0);
    }
    base = nbase;
    c0 = nc0;
  }
}

template <int BITS, int L, int RR, int U, int XF, int EPI>
hipError_t launch_gemv_cfg(const QRowsArgs& a, hipStream_t s) {
  const int nout = EPI == EPI_SWIGLU ? a.N / 2 : a.N, rows = 4 * RR * (64 / L), steps = (nout + rows - 1) / rows;
  hipLaunchKernelGGL((k_qgemv<BITS, L, RR, U, XF, EPI>), dim3(std::min(steps, 2048)), dim3(256),
                     static_cast<size_t>(a.K) * 2, s, a);
  return hipGetLastError();
}

// Rows per wave: enough waves to fill the chip's slots first (and then more of a row in flight per wave), then more rows.
template <int BITS, int L, int U, int XF, int EPI>
hipError_t launch_gemv_rows(const QRowsArgs& a, hipStream_t s) {
  const int nout = EPI == EPI_SWIGLU ? a.N / 2 : a.N;
  constexpr int R4 = EPI == EPI_SWIGLU ? 2 : 4;
  if (nout >= 1024 * R4 * (64 / L)) return launch_gemv_cfg<BITS, L, R4, 1, XF, EPI>(a, s);
  return launch_gemv_cfg<BITS, L, 1, U, XF, EPI>(a, s);
}

template <int BITS, int XF, int EPI>
hipError_t launch_gemv_form(const QRowsArgs& a, hipStream_t s) {
  const int nch = a.K / (BITS == 8 ? 16 : 32);  // 16-byte chunks of a row
  if (nch > 64) return launch_gemv_rows<BITS, 64, 2, XF, EPI>(a, s);
  if (nch > 32) return launch_gemv_rows<BITS, 64, 1, XF, EPI>(a, s);
  if (nch > 16) return launch_gemv_rows<BITS, 32, 1, XF, EPI>(a, s);
  return launch_gemv_rows<BITS, 16, 1, XF, EPI>(a, s);
}

template <int BITS, int UW, int KW, bool LONG, int XF, int EPI>
hipError_t launch_cfg(const QRowsArgs& a, hipStream_t s) {
  constexpr int TW = 8 / KW;
  const int tiles = EPI == EPI_SWIGLU ? (a.N / 2 + 7) / 8 : (a.N + 15) / 16, steps = (tiles + TW - 1) / TW;
  // resident blocks by the registers of the variant; the grid shares the steps evenly among at most that many
  constexpr int c = BITS == 4 ? UW : UW / 2;  // 16 (fp16 activations) to 24 registers each
  constexpr int slots = 256 * (LONG || c > 3 ? 1 : c > 1 ? 2 : 4);
  const int per = (steps + slots - 1) / slots;
  hipLaunchKernelGGL((k_qrows<BITS, UW, KW, LONG, XF, EPI>), dim3((steps + per - 1) / per), dim3(512), 0, s, a);
  return hipGetLastError();
}

template <int XF, int EPI>
hipError_t launch_form(const QRowsArgs& a, int bits, hipStream_t s) {
  if (a.M == 1 && a.K <= 16384)  // (32 KB of LDS)
    return bits == 8 ? launch_gemv_form<8, XF, EPI>(a, s) : launch_gemv_form<4, XF, EPI>(a, s);
  const int nu = bits == 4 ? (a.K + 127) / 128 : a.K / 64;
  if constexpr (XF == QX_F16 && EPI == EPI_STORE) {
    // tall matrices of short rows: fewer waves over K, so that each has four (int4) or eight (int8) loads a tile
    if (a.N >= 32768 && bits == 4 && nu <= 8) return launch_cfg<4, 4, 2, false, XF, EPI>(a, s);
    if (a.N >= 32768 && bits == 4 && nu <= 16) return launch_cfg<4, 4, 4, false, XF, EPI>(a, s);
    if (a.N >= 32768 && bits == 8 && nu <= 16) return launch_cfg<8, 8, 2, false, XF, EPI>(a, s);
    if (a.N >= 32768 && bits == 8 && nu <= 32) return launch_cfg<8, 8, 4, false, XF, EPI>(a, s);
    // rows of up to 5120 (int4) or 4096 (int8) inputs: the activations still fit in registers
    if (bits == 4 && nu > 32 && nu <= 40) return launch_cfg<4, 5, 8, false, XF, EPI>(a, s);
    if (bits == 8 && nu > 48 && nu <= 64) return launch_cfg<8, 8, 8, false, XF, EPI>(a, s);
  }
  if (bits == 4) {
    if (nu <= 8) return launch_cfg<4, 1, 8, false, XF, EPI>(a, s);
    if (nu <= 16) return launch_cfg<4, 2, 8, false, XF, EPI>(a, s);
    if (nu <= 24) return launch_cfg<4, 3, 8, false, XF, EPI>(a, s);
    if (nu <= 32) return launch_cfg<4, 4, 8, false, XF, EPI>(a, s);
    return launch_cfg<4, XF == QX_NORM ? 2 : 4, 8, true, XF, EPI>(a, s);
  }
  if (nu <= 16) return launch_cfg<8, 2, 8, false, XF, EPI>(a, s);
  if (nu <= 32) return launch_cfg<8, 4, 8, false, XF, EPI>(a, s);
  if (nu <= 48) return launch_cfg<8, 6, 8, false, XF, EPI>(a, s);
  return launch_cfg<8, 6, 8, true, XF, EPI>(a, s);
}

}  // namespace

bool qrows_supported(const QRowsArgs& a, int bits) {
  const uintptr_t align = reinterpret_cast<uintptr_t>(a.xh) | reinterpret_cast<uintptr_t>(a.x) |
                          reinterpret_cast<uintptr_t>(a.gain) | reinterpret_cast<uintptr_t>(a.codes);
  return (bits == 4 || bits == 8) && a.M >= 1 && a.M <= 8 && a.N > 0 && a.K >= 64 && a.K % 64 == 0 &&
         align % 16 == 0;
}

hipError_t launch_qrows(const QRowsArgs& a, int bits, int epi, hipStream_t s) {
  if (!qrows_supported(a, bits) || (a.xh != nullptr) == (a.x != nullptr)) return hipErrorInvalidValue;
  if (epi == EPI_SWIGLU) {
    if (a.x == nullptr || a.gain == nullptr || a.yh == nullptr || a.N % 2 != 0) return hipErrorInvalidValue;
    return launch_form<QX_NORM, EPI_SWIGLU>(a, bits, s);
  }
  if (a.y == nullptr) return hipErrorInvalidValue;
  if (epi == EPI_STORE && a.xh != nullptr) return launch_form<QX_F16, EPI_STORE>(a, bits, s);
  if (epi == EPI_STORE && a.gain != nullptr) return launch_form<QX_NORM, EPI_STORE>(a, bits, s);
  if (epi == EPI_RESIDUAL && a.xh != nullptr) return launch_form<QX_F16, EPI_RESIDUAL>(a, bits, s);
  if (epi == EPI_RESIDUAL && a.gain == nullptr) return launch_form<QX_F32, EPI_RESIDUAL>(a, bits, s);
  return hipErrorInvalidValue;
}

}  // namespace soc
