// Single-pass spherical bf16 EM tile when one workgroup holds every component
// (K <= 256, D <= 128): E-GEMM, row log-normalisers, responsibilities and the
// statistics M-GEMM of a 32-row block in one sweep over x.
//
// As em_coop.hip without the exchange: NW waves of 32 components, both GEMMs on
// the 32x32x16 bf16 MFMA.  The logits are formed as in em_fused.hip, one chain
// P = x·μ - ‖x‖²/2 + C' of the exact bf16 x and means and the augmented chunk,
// then l2 = (log2(e)/σ²)·P in fp32 (one accumulator tile instead of the
// exchanging kernel's two: 16 registers).  The waves' per-row (max, sum)
// meet in LDS, so the lag is one block:
//
//   iteration i:  row factors of block i-1 (merge of the NW waves' partials, by
//                 every wave), r = e·2^(m_w - M)/S staged in LDS
//                 E-GEMM of block i
//                 M-GEMM of block i-1 with block i's exponentials between its MFMAs
//                 block i's wave sums to LDS, block i+1 staged, one barrier
//
// so only one block's exponentials stay in registers (the lag of two of the
// exchanging kernel, with K in one workgroup, spilled 74 to 120 VGPRs at NW = 8).
//
// Bound by latency: the chain row factors, staging of r, E-GEMM on one accumulator, row
// maximum, exponentials, barrier at two waves per SIMD (N = 1M, D = 96, K = 200: MFMA busy
// 23 %, VALU busy 44 %, half of the wave cycles waiting; D = 128, K = 256: 22, 34 and 52 %).
// One EM iteration against the two passes of em_sph_bf16.hip (which form every logit twice from a
// hi + lo split, load rows of D != 32, 64, 128 by element, and write and read the
// row log-normalisers): N = 1M: D = 96, K = 200 0.245 against 0.61 ms; D = 96,
// K = 50 0.114 / 0.58; D = 100, K = 256 0.26 / 0.60; D = 128, K = 256 0.27 / 0.39;
// D = 64, K = 128 0.113 / 0.172; N = 50000 x 2, D = 29, K = 100 0.035 / 0.049.

#include "common.hpp"
#include "engine.hpp"
#include "sph_bf16.hpp"

namespace gx {

namespace {

using namespace sphb;

constexpr int kNB = 3;             // staged row blocks: i-1, i, i+1

template <int DP, int NW, bool EXACT>
__global__ __launch_bounds__(64 * NW, 2) void sph_bf16_one_kernel(CoopArgs a) {
  constexpr int XK = DP / 16;                    // 16-deep k-steps over the x columns (E-GEMM)
  constexpr int XT = DP / 32;                    // 32-wide x tiles of ψ (M-GEMM)
  constexpr int XS = row_stride(DP);             // staged row stride (bf16)
  constexpr int CPR = row_lanes(DP);             // loading lanes (16-byte chunks) per row
  static_assert(DP + kAug <= XS && CPR * 8 >= DP, "a row and its augmented chunk fit");
  constexpr int NCH = kBN * CPR;                 // chunk slots per row block (DP = 96 leaves 4 of 16 idle)
  constexpr int NTHR = 64 * NW;
  constexpr int PF = (NCH + NTHR - 1) / NTHR;
  constexpr int PW = NW < 4 ? NW : NW / 2;       // wave partials a lane merges (NW >= 4: half, the other
                                                 // half in lane ^ 32)
  constexpr int RR = 12;                         // partials' row stride: rows 12 banks apart

  __shared__ __align__(16) __bf16 xs[kNB * kBN * XS];
  __shared__ __align__(16) __bf16 rs[NW * kBN * kRS];
  __shared__ __align__(16) float red_m[2 * kBN * RR];    // [parity][row][wave]
  __shared__ __align__(16) float red_s[2 * kBN * RR];
  __shared__ double ll_s[NW];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64), lane = tid % 64;
  const int lr = lane % 32, hf = lane / 32;      // 32x32 MFMA: row / component of a tile, k half
  const int64_t N = a.N;
  const int K = a.K, D = EXACT ? DP : a.D;
  const int kbase = wave * kCW;

  // Staged rows start at zero, with the constant augmented columns 8..31: [1 0 0 ...].
  for (int i = tid; i < kNB * kBN * XS / 8; i += NTHR) *reinterpret_cast<uint4*>(xs + 8 * i) = make_uint4(0, 0, 0, 0);
  __syncthreads();
  for (int i = tid; i < kNB * kBN; i += NTHR) xs[i * XS + DP + 8] = (__bf16)1.f;

  // Transposing-read addresses of the 32x32x16 operands: lane i of 16-lane group
  // G reads rows 8 (G / 2) + i / 4 (+4) of a k-step and columns 16 (G % 2) + 4 (i % 4).
  const int G16 = lane / 16, i16 = lane % 16;
  const int trow = 8 * (G16 >> 1) + (i16 >> 2), tcol = 16 * (G16 & 1) + 4 * (i16 & 3);

  const int items = a.B * a.spb;
  for (int item = blockIdx.x; item < items; item += gridDim.x) {
    const int b = __builtin_amdgcn_readfirstlane(item / a.spb);   // (uniform: keep the slice's bounds in SGPRs)
    const int sl = item - b * a.spb;
    const int64_t rbeg = (int64_t)sl * a.rows_per_item;
    const int64_t rend = (rbeg + a.rows_per_item < N) ? rbeg + a.rows_per_item : N;
    const int nblk = (rend > rbeg) ? (int)((rend - rbeg + kBN - 1) / kBN) : 0;

    // ---- resident component operands (A side of the E-GEMM): lane (lr, hf) holds
    // component kbase + lr, k half hf; padding components get P = -1e30. ----
    bf16x8 wmu[XK], waug;
    float sc[16];            // log2(e)/σ² of the wave's output components (register v)
    {
      const int kk = kbase + lr;
      if (kk < K) {
        const size_t bk = (size_t)b * K + kk;
#pragma unroll
        for (int t = 0; t < XK; ++t)
          wmu[t] = ld16<bf16x8>(reinterpret_cast<const __bf16*>(a.w_mu) + bk * a.DL + 16 * t + 8 * hf);
        waug = ld16<bf16x8>(reinterpret_cast<const __bf16*>(a.w_augs) + bk * 16 + 8 * hf);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
#pragma unroll
          for (int t = 0; t < XK; ++t) wmu[t][e] = (__bf16)0.f;
          waug[e] = (__bf16)((8 * hf + e) == 6 ? -kHuge : 0.f);
        }
      }
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int kv = kbase + 8 * (v / 4) + 4 * hf + (v % 4);
        sc[v] = kv < K ? a.w_scale[(size_t)b * K + kv] : 1.f;
      }
    }
    f32x16 accx[XT], acca = f32x16{};
#pragma unroll
    for (int xt = 0; xt < XT; ++xt) accx[xt] = f32x16{};
    float er[16];            // e = 2^(l2 - m_w) of the last block (register v: component 8(v/4) + 4hf + v%4 of row lr)
#pragma unroll
    for (int v = 0; v < 16; ++v) er[v] = 0.f;
    float mw = 0.f;          // its wave row maximum
    double ll = 0.0;

    // x rows of this item, addressed with 32-bit offsets from a uniform base (an
    // item is under 2^30 bytes).  Rows past its end read the last one and are zeroed.
    const __bf16* xi = reinterpret_cast<const __bf16*>(a.x) + ((size_t)b * N + rbeg) * D;
    const int nrows = (int)(rend - rbeg);
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
    // Stages the prefetched block into buffer `buf`: x, and columns 0..7 of the
    // augmented chunk [q_h q_m q_l q_h q_m q_h 1 1] with q = ‖x‖².
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

    __syncthreads();         // (the previous item's last reads of the staged rows)
    if (nblk > 0) { fetch(0); stash(0); }
    if (nblk > 1) fetch(kBN);
    __syncthreads();

    // i = 0 .. nblk: the E-GEMM of block i (i = nblk: a stale buffer, discarded)
    // and the M-GEMM of block i-1.  i = 0 multiplies r = 0 by the item's own first
    // block: another buffer may hold rows of the previous item, and 0 · NaN of one that
    // is not finite would reach this problem's sums.
    int bufE = 0, bufM = 0;
    for (int i = 0; i <= nblk; ++i) {
      const int pb = i & 1;
      const int bufN = bufE + 1 == kNB ? 0 : bufE + 1;     // buffer of block i+1 (== of block i-2)
      // ---- row factors and responsibilities of block i-1 ----
      {
        const int row = i * kBN - kBN + lr;                // its row in the item
        const bool valid = row >= 0 && row < nrows;
        const int o = ((pb ^ 1) * kBN + lr) * RR + (NW >= 4 ? PW * hf : 0);
        float pm[PW], ps[PW];
#pragma unroll
        for (int w = 0; w < PW; ++w) { pm[w] = red_m[o + w]; ps[w] = red_s[o + w]; }
        float M = pm[0];
#pragma unroll
        for (int w = 1; w < PW; ++w) M = fmaxf(M, pm[w]);
        if constexpr (NW >= 4) M = lanes_op<32, true>(M);
        float S = 0.f;
#pragma unroll
        for (int w = 0; w < PW; ++w) S = fmaf(ps[w], fast_exp2(pm[w] - M), S);
        if constexpr (NW >= 4) S = lanes_op<32, false>(S);
        if (wave == (i & (NW - 1)) && valid && hf == 0) ll += (double)(M + __log2f(S));   // one wave per block
        const float f = valid ? fast_exp2(mw - M) * __builtin_amdgcn_rcpf(S) : 0.f;
        __bf16* rrow = rs + wave * kBN * kRS + lr * kRS;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const float* e4 = er + 4 * u;
          const uint2 pk = make_uint2(cvt2(e4[0] * f, e4[1] * f), cvt2(e4[2] * f, e4[3] * f));
          *reinterpret_cast<uint2*>(rrow + rswz(lr, 8 * u + 4 * hf)) = pk;
        }
      }
      // ---- E-GEMM of block i: operand j of the XK + 1 MFMAs (0: augmented chunk,
      // 1 + t: k-step t) from a rotating three-register-set pipeline ----
      f32x16 T = f32x16{};
      {
        const __bf16* xr = xs + bufE * kBN * XS + lr * XS + 8 * hf;
        auto opnd = [&](int j) { return ld16<bf16x8>(j == 0 ? xr + DP : xr + 16 * (j - 1)); };
        bf16x8 ob[3];
        ob[0] = opnd(0);
        ob[1] = opnd(1);
        ob[2] = opnd(2);
        __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
#pragma unroll
        for (int j = 0; j <= XK; ++j) {
          T = mfma32(j == 0 ? waug : wmu[j - 1 < 0 ? 0 : j - 1], ob[j % 3], T);
          if (j + 3 <= XK) ob[j % 3] = opnd(j + 3);
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          if (j + 3 <= XK) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
#pragma unroll
        for (int v = 0; v < 16; ++v) T[v] *= sc[v];
      }
      // The staging writes above and the transposing reads below are LDS
      // operations of this wave only, executed in order; keep the compiler
      // from reordering them.
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      // ---- M-GEMM of block i-1 with the exponentials of block i between its MFMAs ----
      float m = T[0];
#pragma unroll
      for (int v = 1; v < 16; ++v) m = fmaxf(m, T[v]);
      m = lanes_op<32, true>(m);
      {
        const __bf16* rw = rs + wave * kBN * kRS;
        const __bf16* xw = xs + bufM * kBN * XS;
        constexpr int HK = 2 * (XT + 1) < 8 ? 2 * (XT + 1) : 8, PH = (16 + HK - 1) / HK;   // MFMAs with, exps per MFMA
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
          const int r0 = 16 * s2 + trow;
          const bf16x8 ar = cat(tr16(rw + r0 * kRS + rswz(r0, tcol)), tr16(rw + (r0 + 4) * kRS + rswz(r0 + 4, tcol)));
          bf16x8 bn = cat(tr16(xw + r0 * XS + tcol), tr16(xw + (r0 + 4) * XS + tcol));
#pragma unroll
          for (int xt = 0; xt <= XT; ++xt) {
            const bf16x8 bq = bn;
            if (xt + 1 <= XT) bn = cat(tr16(xw + r0 * XS + 32 * (xt + 1) + tcol), tr16(xw + (r0 + 4) * XS + 32 * (xt + 1) + tcol));
            if (xt < XT) accx[xt] = mfma32(ar, bq, accx[xt]);
            else acca = mfma32(ar, bq, acca);
            const int k = s2 * (XT + 1) + xt;
#pragma unroll
            for (int u = 0; u < PH; ++u)
              if (PH * k + u < 16) er[PH * k + u] = fast_exp2(T[PH * k + u] - m);
          }
        }
      }
      {
        float ps[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) ps[u] = (er[4 * u] + er[4 * u + 1]) + (er[4 * u + 2] + er[4 * u + 3]);
        const float sum = lanes_op<32, false>((ps[0] + ps[1]) + (ps[2] + ps[3]));
        mw = m;
        // Both lanes of a row hold the same values: both store (no branch).
        red_m[(pb * kBN + lr) * RR + wave] = m;
        red_s[(pb * kBN + lr) * RR + wave] = sum;
      }
      if (i + 1 < nblk) stash(bufN);
      if (i + 2 < nblk) fetch((i + 2) * kBN);
      __syncthreads();
      bufM = bufE;
      bufE = bufN;
    }

    // ---- the item's partial statistics (lane (lr, hf), register v: component
    // 8(v/4) + 4hf + v%4 of the wave, feature 32xt + lr) and log-likelihood ----
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int kk = kbase + 8 * (v / 4) + 4 * hf + (v % 4);
      if (kk < K) {
        // statistics row of width DL + 16: x | augmented 0..15 (DL > DP: zeros between)
        float* dst = a.part_stats + (((size_t)sl * a.B + b) * K + kk) * (a.DL + 16);
#pragma unroll
        for (int xt = 0; xt < XT; ++xt) dst[32 * xt + lr] = accx[xt][v];
        if (!EXACT && DP == 96) dst[DP + lr] = 0.f;
        if (lr < 16) dst[a.DL + lr] = acca[v];
      }
    }
    for (int off = 32; off >= 1; off /= 2) ll += __shfl_xor(ll, off);
    if (lane == 0) ll_s[wave] = ll;
    __syncthreads();
    if (tid == 0) {
      double t = ll_s[0];
      for (int w = 1; w < NW; ++w) t += ll_s[w];
      a.ll_part[(size_t)b * a.spb + sl] = t * (double)kLn2;
    }
  }
}

template <int DP, bool EXACT>
int launch_one_dp(int nw, const CoopArgs& a, hipStream_t s) {
  switch (nw) {
    case 2:
      if constexpr (DP <= 96) { sph_bf16_one_kernel<DP, 2, EXACT><<<a.NG, 128, 0, s>>>(a); return 0; }
      return -1;
    case 4: sph_bf16_one_kernel<DP, 4, EXACT><<<a.NG, 256, 0, s>>>(a); return 0;
    case 8: sph_bf16_one_kernel<DP, 8, EXACT><<<a.NG, 512, 0, s>>>(a); return 0;
    default: return -1;
  }
}

}  // namespace

int launch_sph_bf16_one(int dp, int nw, const CoopArgs& a, hipStream_t s) {
  if (a.D > dp || a.DL < dp || nw * kCW < a.K) return -1;
  switch (dp) {
    case 32: return launch_one_dp<32, false>(nw, a, s);
    case 64: return launch_one_dp<64, false>(nw, a, s);
    case 96: return launch_one_dp<96, false>(nw, a, s);
    case 128: return a.D == 128 && a.vec ? launch_one_dp<128, true>(nw, a, s) : launch_one_dp<128, false>(nw, a, s);
    default: return -1;
  }
}

}  // namespace gx
