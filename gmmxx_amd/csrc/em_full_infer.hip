// Full-covariance inference at D <= 16 and K <= 32 (predict_proba,
// score_samples, labels) by whitening on the bf16 MFMA with split operands.
//
// The tile kernel's E-step forms the row's 136 products x_d x_e and splits each
// into three bf16 parts: at D = 16 that VALU work, not the matrix core, bounds
// it.  Here the quadratic form is a squared norm, (x - μ)ᵀ Σ⁻¹ (x - μ) =
// ‖L⁻¹x - L⁻¹μ‖² (Σ = L Lᵀ; torch_fallback.py:400-432 computes the same value
// expanded, clamped at zero), and only x's 16 values are split.
//
// Two components make one 32 x 32 output tile of v_mfma_f32_32x32x16_bf16 (16
// dims of each x 32 rows), accumulated from -L⁻¹μ by the six products of the split
// operands down to 2^-24, L_h x_h first: it cancels -L⁻¹μ, and the others (L_h x_m,
// L_h x_l, L_m x_h, L_m x_m, L_l x_h) are rounded at the size of y (smallest first the scores
// of data 300 from the origin were 2.5 times as far from float64; responsibilities of
// 16 x 262144 rows, K = 32 382 -> 386 us).
// Lane l holds 8 of the 16 dims of both components for row l % 32: one swap of the
// two partial norms between lanes l and l ^ 32 and one addition leave lane half h
// with the whole norm of its own component.  The pair of step j is (j, KH + j), KH =
// ceil(K / 2): half h ends with the log2 logits of components h·KH … h·KH + KH - 1
// of its row, so the log-normaliser, the responsibilities (written as contiguous
// runs) and the first argmax need no second pass.  A wave takes 2 blocks of 32
// rows per tile; the components' operands sit in LDS for the whole launch (an odd
// K is padded with zeros and the constant -inf).
//
// Bound: the MFMAs (16 x 262144 rows, K = 32: 6 x 69 GFLOP, 215 us at the rate a pure
// MFMA loop reaches) with the squares and the softmax of 3 waves per SIMD not
// hidden behind them (MFMA busy 55 %, VALU 43 %).  A 16 x 16 tile per component and row block, the
// operands laid twice along k (96 KB of LDS: one workgroup of 8 waves per CU, four
// swaps and eight selects per norm) took 458 us for the scores, 534 with labels
// and 496 for the responsibilities; here 349, 397 and 390.  64 x 20000 rows, K = 8:
// 72 -> 50; 3000 rows, K = 32, all launches: 36 -> 25.

#include <math.h>

#include <algorithm>
#include <atomic>

#include "common.hpp"
#include "engine.hpp"

namespace gx {

namespace {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kWaves = 4;
constexpr int kRB = 2;                     // 32-row blocks per wave and tile
constexpr int kCompElems = 3 * 2 * 16 * 8; // a component's operand: [part][column half][row][8]
constexpr int kMaxPairs = kFull16MaxK / 2;

__device__ __forceinline__ f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// v_permlane32_swap(x, y): the lower lanes get (own x, partner's x), the upper lanes
// (partner's y, own y).
__device__ __forceinline__ void swap32(float x, float y, float& t0, float& t1) {
  const auto t = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
  t0 = __uint_as_float(t[0]);
  t1 = __uint_as_float(t[1]);
}
// Over lanes l and l ^ 32: the same bits in both.
__device__ __forceinline__ float sum2(float v) {
  float a, b;
  swap32(v, v, a, b);
  return a + b;
}
__device__ __forceinline__ float max2(float v) {
  float a, b;
  swap32(v, v, a, b);
  return fmaxf(a, b);
}

// v = h + m + l exactly, eight values to three bf16x8.
__device__ __forceinline__ void split8(const float (&v)[8], bf16x8& h, bf16x8& m, bf16x8& l) {
#pragma unroll
  for (int p = 0; p < 8; p += 2) {
    const f32x2 a = f32x2{v[p], v[p + 1]};
    const bf16x2 hh = __builtin_convertvector(a, bf16x2);
    const f32x2 r = a - __builtin_convertvector(hh, f32x2);
    const bf16x2 mm = __builtin_convertvector(r, bf16x2);
    const bf16x2 ll = __builtin_convertvector(r - __builtin_convertvector(mm, f32x2), bf16x2);
    h[p] = hh[0];
    h[p + 1] = hh[1];
    m[p] = mm[0];
    m[p + 1] = mm[1];
    l[p] = ll[0];
    l[p + 1] = ll[1];
  }
}

}  // namespace

// ---------------------------------------------------------------------------
// Operands per component: L⁻¹ zero-padded to 16 x 16 and split into bf16 parts
// h + m + l ([part][columns 8 g … +7][row]), -L⁻¹μ and the log2 constant
// log2 w - ½ log2(e) (D log 2π + log det Σ).
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(64) void full16_pack_kernel(Full16Args a) {
  const int k = blockIdx.x, b = blockIdx.y, t = threadIdx.x;
  const int K = a.K, D = a.D;
  const size_t bk = (size_t)b * K + k;
  const float* X = a.linv + bk * D * D;
  const float* mu = a.means + bk * D;
  __bf16* op = reinterpret_cast<__bf16*>(a.lparts) + bk * kCompElems;
  for (int e = t; e < kCompElems / 3; e += 64) {
    const int g = e / 128, i = (e / 8) % 16, d = 8 * g + e % 8;
    const float v = (i < D && d < D) ? X[i * D + d] : 0.f;
    const __bf16 h = (__bf16)v;
    const float r = v - (float)h;
    const __bf16 m = (__bf16)r;
    op[e] = h;
    op[kCompElems / 3 + e] = m;
    op[2 * kCompElems / 3 + e] = (__bf16)(r - (float)m);
  }
  if (t < 16) {
    double acc = 0.0;
    if (t < D)
      for (int j = 0; j <= t; ++j) acc = fma((double)X[t * D + j], (double)mu[j], acc);
    a.bneg[bk * 16 + t] = (float)(-acc);
  }
  if (t == 0) {
    constexpr double kLog2eD = 1.4426950408889634;
    const double c2 = (log((double)a.weights[bk]) - 0.5 * ((double)D * kLog2Pi + (double)a.logdet[bk])) * kLog2eD;
    a.c2[bk] = (float)c2;
  }
}

// ---------------------------------------------------------------------------
// Scores, labels, responsibilities
// ---------------------------------------------------------------------------

// KH = ceil(K / 2): the components per lane half (a template parameter, so every
// guard on it below is resolved at compile time).
// Workgroups per CU: four waves per SIMD while the logits fit 128 registers (at KH = 16
// four spill: scores 371 us against 364 with three), and 3 x 51 KB of LDS fit.
constexpr int groups_per_cu(int kh) { return kh <= 9 ? 4 : 3; }

template <int KH>
__global__ __launch_bounds__(64 * kWaves, groups_per_cu(KH)) void full16_infer_kernel(Full16Args a) {
  __shared__ __align__(16) __bf16 parts[KH * 2 * kCompElems];   // [pair][part][lane][8]
  __shared__ __align__(16) float bneg[KH * 32];                 // [pair][component][dim]
  __shared__ float c2s[2 * KH];
  const int b = blockIdx.y;
  const int K = a.K, D = a.D;
  const int64_t N = a.N;
  // Stage every component's operands: component k is member k / KH of pair k % KH.
  {
    const uint4* src = reinterpret_cast<const uint4*>(reinterpret_cast<const __bf16*>(a.lparts) + (size_t)b * K * kCompElems);
    uint4* dst = reinterpret_cast<uint4*>(parts);
    for (int i = threadIdx.x; i < 2 * KH * kCompElems / 8; i += 64 * kWaves) {
      const int k = i / (kCompElems / 8), c = i % (kCompElems / 8);   // c = (part, half, row)
      dst[((k % KH) * 3 + c / 32) * 64 + (c / 16 % 2) * 32 + (k / KH) * 16 + c % 16] = k < K ? src[i] : make_uint4(0, 0, 0, 0);
    }
    for (int i = threadIdx.x; i < 2 * KH * 16; i += 64 * kWaves) {
      const int k = i / 16;
      bneg[(k % KH) * 32 + (k / KH) * 16 + i % 16] = k < K ? a.bneg[(size_t)b * K * 16 + i] : 0.f;
    }
    for (int i = threadIdx.x; i < 2 * KH; i += 64 * kWaves) c2s[i] = i < K ? a.c2[(size_t)b * K + i] : -INFINITY;
  }
  __syncthreads();

  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  const int lr = lane & 31, g = lane >> 5;    // row of a 32-row block; lane half
  // The operands are staged once; the workgroup then walks its share of the
  // problem's row tiles (the grid is the device's resident capacity).
  const int64_t ntiles = (N + 32 * kRB * kWaves - 1) / (32 * kRB * kWaves);
  const float* xb = a.x + (size_t)b * N * D;
  for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const int64_t base = (tile * kWaves + wave) * (32 * kRB);
    // x parts as B operands: row lr of each block, dims 8g … +7.
    bf16x8 xh[kRB], xm[kRB], xl[kRB];
#pragma unroll
    for (int rb = 0; rb < kRB; ++rb) {
      const int64_t n = base + 32 * rb + lr;
      float v[8];
      if (n < N && a.vec_ok) {
        const f32x4 p = *reinterpret_cast<const f32x4*>(xb + (size_t)n * 16 + 8 * g);
        const f32x4 q = *reinterpret_cast<const f32x4*>(xb + (size_t)n * 16 + 8 * g + 4);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          v[u] = p[u];
          v[4 + u] = q[u];
        }
      } else {
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = (n < N && 8 * g + u < D) ? xb[(size_t)n * D + 8 * g + u] : 0.f;
      }
      split8(v, xh[rb], xm[rb], xl[rb]);
    }
    // Every LDS read below is indexed through z, zero but opaque to the compiler
    // and redefined per tile: the component operands are loop-invariant, and
    // without it their loads are hoisted out of the tile loop into registers
    // (hundreds: the kernel then spills).
    int z = 0;
    asm volatile("" : "+v"(z));
    const __bf16* opl = parts + lane * 8 + z;
    const float* bl = bneg + 4 * g + z;
    const float* cl = c2s + g * KH + z;

    float l2v[kRB][KH];
#pragma unroll
    for (int j = 0; j < KH; ++j) {
      const bf16x8 Lh = *reinterpret_cast<const bf16x8*>(opl + (3 * j + 0) * 512);
      const bf16x8 Lm = *reinterpret_cast<const bf16x8*>(opl + (3 * j + 1) * 512);
      const bf16x8 Ll = *reinterpret_cast<const bf16x8*>(opl + (3 * j + 2) * 512);
      f32x16 c;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const f32x4 q = *reinterpret_cast<const f32x4*>(bl + 32 * j + 8 * u);
#pragma unroll
        for (int v = 0; v < 4; ++v) c[4 * u + v] = q[v];
      }
      const float cst = cl[j];
      f32x16 t[kRB];
#pragma unroll
      for (int rb = 0; rb < kRB; ++rb) t[rb] = mfma32(Lh, xh[rb], c);
#pragma unroll
      for (int rb = 0; rb < kRB; ++rb) t[rb] = mfma32(Lh, xm[rb], t[rb]);
#pragma unroll
      for (int rb = 0; rb < kRB; ++rb) t[rb] = mfma32(Lh, xl[rb], t[rb]);
#pragma unroll
      for (int rb = 0; rb < kRB; ++rb) t[rb] = mfma32(Lm, xh[rb], t[rb]);
#pragma unroll
      for (int rb = 0; rb < kRB; ++rb) t[rb] = mfma32(Lm, xm[rb], t[rb]);
#pragma unroll
      for (int rb = 0; rb < kRB; ++rb) t[rb] = mfma32(Ll, xh[rb], t[rb]);
#pragma unroll
      for (int rb = 0; rb < kRB; ++rb) {
        float q0 = t[rb][0] * t[rb][0], q1 = t[rb][8] * t[rb][8];
#pragma unroll
        for (int v = 1; v < 8; ++v) {
          q0 = fmaf(t[rb][v], t[rb][v], q0);
          q1 = fmaf(t[rb][8 + v], t[rb][8 + v], q1);
        }
        float t0, t1;
        swap32(q0, q1, t0, t1);
        l2v[rb][j] = fmaf(-0.5f * kLog2e, t0 + t1, cst);
      }
    }

#pragma unroll
    for (int rb = 0; rb < kRB; ++rb) {
      const int64_t n = base + 32 * rb + lr;
      float m = -INFINITY;
#pragma unroll
      for (int j = 0; j < KH; ++j) m = fmaxf(m, l2v[rb][j]);
      if (a.labels) {
        // First argmax: the first equal to the half's maximum, then the lower half's
        // among equal maxima.
        int at = 0;
#pragma unroll
        for (int j = KH - 1; j >= 0; --j) at = l2v[rb][j] == m ? j : at;
        float lo, up, li, ui;
        swap32(m, m, lo, up);
        swap32(__int_as_float(at), __int_as_float(at), li, ui);
        if (n < N && g == 0) a.labels[(size_t)b * N + n] = up > lo ? KH + __float_as_int(ui) : __float_as_int(li);
      }
      if (!a.scores && !a.proba) continue;   // (uniform; labels alone need no exponentials)
      m = max2(m);
      float s = 0.f;
#pragma unroll
      for (int j = 0; j < KH; ++j) {
        l2v[rb][j] = fast_exp2(l2v[rb][j] - m);
        s += l2v[rb][j];
      }
      s = sum2(s);
      if (n >= N) continue;   // lanes of one row agree
      if (a.scores && g == 0) a.scores[(size_t)b * N + n] = (m + __log2f(s)) * kLn2;
      if (a.proba) {
        const float inv = 1.f / s;
        float* pr = a.proba + ((size_t)b * N + n) * K + g * KH;
        const int left = K - g * KH;   // (odd K: the upper half's run stops at K)
#pragma unroll
        for (int j = 0; j < KH; j += 4) {
          if (j + 4 <= KH && j + 4 <= left) {
            *reinterpret_cast<f32x4_any*>(pr + j) = f32x4_any{l2v[rb][j] * inv, l2v[rb][j + 1 < KH ? j + 1 : 0] * inv,
                                                             l2v[rb][j + 2 < KH ? j + 2 : 0] * inv, l2v[rb][j + 3 < KH ? j + 3 : 0] * inv};
          } else {
#pragma unroll
            for (int u = 0; u < 4; ++u)
              if (j + u < KH && j + u < left) pr[j + u] = l2v[rb][j + u < KH ? j + u : 0] * inv;
          }
        }
      }
    }
  }   // row tiles
}

void launch_full16_pack(const Full16Args& a, hipStream_t s) {
  full16_pack_kernel<<<dim3(a.K, a.B), 64, 0, s>>>(a);
}

// Compute units of the current device (cached per device; concurrent first calls
// store the same value).
static int full16_cus() {
  static std::atomic<int> cache[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) {
    (void)hipGetLastError();
    return 256;
  }
  const int cached = cache[dev].load(std::memory_order_relaxed);
  if (cached > 0) return cached;
  int cus = 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) {
    (void)hipGetLastError();
    return 256;
  }
  cache[dev].store(cus, std::memory_order_relaxed);
  return cus;
}

void launch_full16_infer(const Full16Args& a, hipStream_t s) {
  const int64_t rows = 32 * kRB * kWaves;
  const int64_t ntiles = (a.N + rows - 1) / rows;
  const int64_t per_problem = std::max<int64_t>(1, (full16_cus() * groups_per_cu((a.K + 1) / 2) + a.B - 1) / a.B);
  const unsigned gx = (unsigned)std::min<int64_t>(ntiles, per_problem);
  const dim3 grid(gx, a.B), block(64 * kWaves);
  switch ((a.K + 1) / 2) {
    case 1: full16_infer_kernel<1><<<grid, block, 0, s>>>(a); break;
    case 2: full16_infer_kernel<2><<<grid, block, 0, s>>>(a); break;
    case 3: full16_infer_kernel<3><<<grid, block, 0, s>>>(a); break;
    case 4: full16_infer_kernel<4><<<grid, block, 0, s>>>(a); break;
    case 5: full16_infer_kernel<5><<<grid, block, 0, s>>>(a); break;
    case 6: full16_infer_kernel<6><<<grid, block, 0, s>>>(a); break;
    case 7: full16_infer_kernel<7><<<grid, block, 0, s>>>(a); break;
    case 8: full16_infer_kernel<8><<<grid, block, 0, s>>>(a); break;
    case 9: full16_infer_kernel<9><<<grid, block, 0, s>>>(a); break;
    case 10: full16_infer_kernel<10><<<grid, block, 0, s>>>(a); break;
    case 11: full16_infer_kernel<11><<<grid, block, 0, s>>>(a); break;
    case 12: full16_infer_kernel<12><<<grid, block, 0, s>>>(a); break;
    case 13: full16_infer_kernel<13><<<grid, block, 0, s>>>(a); break;
    case 14: full16_infer_kernel<14><<<grid, block, 0, s>>>(a); break;
    case 15: full16_infer_kernel<15><<<grid, block, 0, s>>>(a); break;
    default: full16_infer_kernel<16><<<grid, block, 0, s>>>(a); break;
  }
}

}  // namespace gx
