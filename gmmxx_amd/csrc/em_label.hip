// Labels (first argmax) of spherical bf16 rows in one pass, K <= 1024, D <= 128: the
// workgroup holds every component, a wave CT tiles of 32, so there are no partials to
// merge in memory.
//
// Logits as in em_one.hip: P = x·μ - ‖x‖²/2 + C' on the 32x32x16 bf16 MFMA from the
// exact bf16 x and means, l2 = (log2(e)/σ²)·P in fp32 (the tile kernel's label pass,
// which this replaces up to K = 1024, multiplies a hi + lo split: twice the MFMAs, and
// covers 256 components per workgroup).  An x operand read from LDS serves all CT tiles;
// the scales stay in LDS.  Per row: the maximum over the lane's 16·CT logits, its first
// place, the partner lane (l ^ 32), then the waves through LDS one block later; equal
// maxima take the lower component.  Padding components and those of weight zero are
// -inf, so no finite row is far enough out to be labelled with one.
//
// Bound: at K <= 64 the latency of the reads of x (1M x 32, K = 64: 2.6 TB/s with the
// labels); with more components the 16·CT multiplies, maxima and compares per row and
// lane beside the MFMA.  Before (tile kernel) -> here: 300000 x 128, K = 1024 255 -> 120
// us, K = 256 72 -> 42, K = 64 66 -> 28; 1M x 96, K = 200 306 -> 105; 1M x 32, K = 64
// 61 -> 28; 3000 x 128, K = 512 20.1 -> 15.0.  More than 1024 components do not fit the
// registers of one workgroup: the tile kernel and its merge stay there.

#include "common.hpp"
#include "engine.hpp"
#include "sph_bf16.hpp"

namespace gx {

namespace {

using namespace sphb;

template <int DP, int NW, int CT, bool EXACT>
__global__ __launch_bounds__(64 * NW, CT == 1 ? 4 : 2) void sph_bf16_label_kernel(CoopArgs a, int64_t* labels) {
  constexpr int XK = DP / 16;                    // 16-deep k-steps
  constexpr int XS = row_stride(DP), CPR = row_lanes(DP);
  constexpr int NCH = kBN * CPR, NTHR = 64 * NW, PF = (NCH + NTHR - 1) / NTHR;
  constexpr int RR = kBN + 1;

  __shared__ __align__(16) __bf16 xs[2 * kBN * XS];
  __shared__ __align__(16) float scs[NW * CT * kCW];
  __shared__ float red_m[2 * NW * RR];           // [parity][wave][row]
  __shared__ int red_i[2 * NW * RR];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64), lane = tid % 64;
  const int lr = lane % 32, hf = lane / 32;
  const int64_t N = a.N;
  const int K = a.K, D = EXACT ? DP : a.D;
  const int kbase = wave * CT * kCW;
  const int b = blockIdx.y;
  const int64_t rbeg = (int64_t)blockIdx.x * a.rows_per_item;
  const int64_t rend = (rbeg + a.rows_per_item < N) ? rbeg + a.rows_per_item : N;
  if (rbeg >= rend) return;
  const int nrows = (int)(rend - rbeg), nblk = (nrows + kBN - 1) / kBN;

  for (int i = tid; i < 2 * kBN * 3; i += NTHR) {     // constant augmented columns 8..31: [1 0 0 ...]
    const int row = i / 3, ch = 1 + i % 3;
    *reinterpret_cast<uint4*>(xs + row * XS + DP + 8 * ch) =
        make_uint4(ch == 1 ? pack2((__bf16)1.f, (__bf16)0.f) : 0u, 0u, 0u, 0u);
  }
  for (int i = tid; i < NW * CT * kCW; i += NTHR) scs[i] = i < K ? a.w_scale[(size_t)b * K + i] : 1.f;
  bf16x8 wmu[CT][XK], waug[CT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    const int kk = kbase + ct * kCW + lr;
    if (kk < K) {
      const size_t bk = (size_t)b * K + kk;
#pragma unroll
      for (int t = 0; t < XK; ++t)
        wmu[ct][t] = ld16<bf16x8>(reinterpret_cast<const __bf16*>(a.w_mu) + bk * a.DL + 16 * t + 8 * hf);
      waug[ct] = ld16<bf16x8>(reinterpret_cast<const __bf16*>(a.w_augs) + bk * 16 + 8 * hf);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
#pragma unroll
        for (int t = 0; t < XK; ++t) wmu[ct][t][e] = (__bf16)0.f;
        waug[ct][e] = (__bf16)((8 * hf + e) == 6 ? -INFINITY : 0.f);   // (below every row's logits)
      }
    }
  }

  const __bf16* xi = reinterpret_cast<const __bf16*>(a.x) + ((size_t)b * N + rbeg) * D;
  uint4 pf[PF];
  auto fetch = [&](int r0) {
#pragma unroll
    for (int i = 0; i < PF; ++i) {
      const int c = tid + i * NTHR;
      if (NCH % NTHR == 0 || c < NCH) {
        const int r = r0 + c / CPR, cc = (c % CPR) * 8;
        pf[i] = load_row_chunk<EXACT>(xi + (r < nrows ? r : nrows - 1) * D, cc, D, a.vec, r < nrows);
      }
    }
  };
  auto stash = [&](int buf) {
#pragma unroll
    for (int i = 0; i < PF; ++i) {
      const int c = tid + i * NTHR;
      if (NCH % NTHR == 0 || c < NCH) {
        const int r = c / CPR, cc = c % CPR;
        const uint4 raw = pf[i];
        __bf16* row = xs + buf * kBN * XS + r * XS;
        if (8 * CPR == DP || 8 * cc < DP) *reinterpret_cast<uint4*>(row + 8 * cc) = raw;
        const uint32_t w4[4] = {raw.x, raw.y, raw.z, raw.w};
        float q = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const bf16x2 p = __builtin_bit_cast(bf16x2, w4[j]);
          q = __builtin_amdgcn_fdot2_f32_bf16(p, p, q, false);
        }
        q = group_sum<CPR>(q);
        if (cc == 0) {
          __bf16 h, m, l;
          split3(q, h, m, l);
          *reinterpret_cast<uint4*>(row + DP) =
              make_uint4(pack2(h, m), pack2(l, h), pack2(m, h), pack2((__bf16)1.f, (__bf16)1.f));
        }
      }
    }
  };
  // Merge of a block's wave partials: lane (row, wave) of the first 32·NW threads.
  auto write_labels = [&](int pb, int r0) {
    if (tid < kBN * NW) {
      const int r = tid / NW, w = tid % NW;
      const float m = red_m[(pb * NW + w) * RR + r];
      const float M = group_max<NW>(m);
      int idx = m == M ? red_i[(pb * NW + w) * RR + r] : 0x7fffffff;
      auto low = [&](int v) { idx = v < idx ? v : idx; };
      if constexpr (NW >= 2) low(__builtin_amdgcn_update_dpp(0, idx, 0xB1, 0xF, 0xF, false));
      if constexpr (NW >= 4) low(__builtin_amdgcn_update_dpp(0, idx, 0x4E, 0xF, 0xF, false));
      if constexpr (NW >= 8) low(__builtin_amdgcn_update_dpp(0, idx, 0x141, 0xF, 0xF, false));
      if (w == 0 && r0 + r < nrows) labels[(size_t)b * N + rbeg + r0 + r] = label_of(idx, K);
    }
  };

  fetch(0);
  stash(0);
  if (nblk > 1) fetch(kBN);
  __syncthreads();
  for (int i = 0; i < nblk; ++i) {
    const int pb = i & 1;
    const __bf16* xr = xs + pb * kBN * XS + lr * XS + 8 * hf;
    auto opnd = [&](int j) { return ld16<bf16x8>(j == 0 ? xr + DP : xr + 16 * (j - 1)); };
    f32x16 T[CT];
    bf16x8 ob[3];
    ob[0] = opnd(0);
    ob[1] = opnd(1);
    ob[2] = opnd(2);
#pragma unroll
    for (int j = 0; j <= XK; ++j) {
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
        T[ct] = mfma32(j == 0 ? waug[ct] : wmu[ct][j - 1 < 0 ? 0 : j - 1], ob[j % 3], j == 0 ? f32x16{} : T[ct]);
      if (j + 3 <= XK) ob[j % 3] = opnd(j + 3);
    }
    if (i > 0) write_labels(pb ^ 1, (i - 1) * kBN);
    float m = -INFINITY;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const f32x4 s4 = ld16<f32x4>(&scs[kbase + ct * kCW + 8 * u + 4 * hf]);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          T[ct][4 * u + v] *= s4[v];
          m = fmaxf(m, T[ct][4 * u + v]);
        }
      }
    int at = 0x7fffffff;      // register place 16 ct + v of the first maximum
#pragma unroll
    for (int p = 16 * CT - 1; p >= 0; --p) at = T[p / 16][p % 16] == m ? p : at;
    // place -> component: tile ct, component 8 (v / 4) + 4 hf + v % 4
    int idx = at == 0x7fffffff ? at : kbase + 2 * (at & ~3) + 4 * hf + (at & 3);
    const float M = lanes_op<32, true>(m);
    idx = m == M ? idx : 0x7fffffff;
    const auto t2 = __builtin_amdgcn_permlane32_swap((unsigned)idx, (unsigned)idx, false, false);
    idx = min((int)t2[0], (int)t2[1]);
    // Both lanes of a row hold the same values: both store (no branch).
    red_m[(pb * NW + wave) * RR + lr] = M;
    red_i[(pb * NW + wave) * RR + lr] = idx;
    if (i + 1 < nblk) stash(pb ^ 1);
    if (i + 2 < nblk) fetch((i + 2) * kBN);
    __syncthreads();
  }
  write_labels((nblk - 1) & 1, (nblk - 1) * kBN);
}

template <int DP, bool EXACT>
void launch_label_dp(const CoopArgs& a, int64_t* labels, dim3 grid, hipStream_t s) {
  if (a.K <= 64) sph_bf16_label_kernel<DP, 2, 1, EXACT><<<grid, 128, 0, s>>>(a, labels);
  else if (a.K <= 128) sph_bf16_label_kernel<DP, 4, 1, EXACT><<<grid, 256, 0, s>>>(a, labels);
  else if (a.K <= 256) sph_bf16_label_kernel<DP, 8, 1, EXACT><<<grid, 512, 0, s>>>(a, labels);
  else if (a.K <= 512) sph_bf16_label_kernel<DP, 8, 2, EXACT><<<grid, 512, 0, s>>>(a, labels);
  else sph_bf16_label_kernel<DP, 8, 4, EXACT><<<grid, 512, 0, s>>>(a, labels);
}

}  // namespace

int launch_sph_bf16_label(int dp, const CoopArgs& a0, int64_t* labels, hipStream_t s) {
  CoopArgs a = a0;
  if (a.D > dp || a.DL < dp || a.K > 1024 || a.B > 65535) return -1;
  // One round of resident waves (four per SIMD with one tile per wave, else two), at
  // least one block per slice, slices under 2^30 bytes.
  const int nw = a.K <= 64 ? 2 : (a.K <= 128 ? 4 : 8);
  int64_t sl = (a.K <= 256 ? 4096 : 2048) / nw / a.B;
  const int64_t blocks = (a.N + kBN - 1) / kBN, least = (a.N * a.D * 2 + (int64_t(1) << 30) - 1) >> 30;
  sl = sl < 1 ? 1 : sl;
  sl = sl > blocks ? blocks : sl;
  sl = sl < least ? least : sl;
  a.rows_per_item = ((a.N + sl - 1) / sl + kBN - 1) / kBN * kBN;
  const dim3 grid((unsigned)((a.N + a.rows_per_item - 1) / a.rows_per_item), a.B);
  switch (dp) {
    case 32: launch_label_dp<32, false>(a, labels, grid, s); return 0;
    case 64: launch_label_dp<64, false>(a, labels, grid, s); return 0;
    case 96: launch_label_dp<96, false>(a, labels, grid, s); return 0;
    case 128:
      if (a.D == 128 && a.vec) launch_label_dp<128, true>(a, labels, grid, s);
      else launch_label_dp<128, false>(a, labels, grid, s);
      return 0;
    default: return -1;
  }
}

}  // namespace gx
