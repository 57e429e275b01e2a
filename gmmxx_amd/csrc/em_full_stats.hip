// Full covariance at 16 < D <= 128, M-step statistics for many components:
// N_k, Σ r x and Σ r x xᵀ of 16 components per workgroup from rows staged once.
//
// For every column i the A operand is r_k·x_i (16 components x 32 rows, formed and
// split into three bf16 parts in registers), the B operand the rows' split columns
// 16J .. 16J+15 (J >= i / 16, so only the upper triangle's 16-column blocks run),
// each product as the six bf16 MFMAs of em_full_wide.hip.  One split of r_k·x_i
// serves every block J, and the split of x every component: fw_stats_kernel (one
// wave per component) re-reads x from L2 and splits √r·x for each component,
// 130 VALU instructions and 16 loads beside 18 MFMAs of 32x32x16 at D = 64, and is
// bound by those.  Here 36 VALU instructions go with (NJ - i / 16) · 6 MFMAs.
//
// A workgroup of eight waves takes a row slice; wave w owns columns 16g + 2w and
// 16g + 2w + 1 of every column group g (D <= 64), or of the group pair
// {Q, NJ - 1 - Q} (D > 64: ceil(NJ / 2) workgroups per 16 components, each pair with
// the same number of tiles), so the waves' MFMA counts are equal.  Rows pass
// through LDS in blocks of 32, twice buffered, one barrier per block: transposed
// fp32 columns (the x_i broadcast) and their three bf16 parts (the B operand),
// staged with the responsibilities 2^(l2 - lse2), one per thread (lse2 with the remainder of
// its last rounding: of a row that one component dominates the others' share is below half
// a unit of lse2, and without it every such r is too large, N_k by up to 3e-7).
//
// Bound by MFMA and VALU issue, which barely overlap (N = 262144, D = 64, K = 32: busy 44
// and 46 %; per wave and block 126 MFMAs, 2016 cycles, beside about 370 VALU instructions;
// 0.117 ms of MFMA).  Statistics launch, fw_stats_kernel -> here: D = 64, K = 32
// 0.390 -> 0.254 ms; D = 32, K = 32 0.181 -> 0.112; D = 33, K = 32 0.38 -> 0.164;
// N = 130000: D = 128, K = 16 0.389 -> 0.237; D = 80, K = 24 0.80 -> 0.27.  Error of
// Σ r x xᵀ against float64 at N = 262144, D = 64, K = 32: 2.6e-7 -> 1.9e-7.
//
// 16x16x32 bf16 MFMA operand layout: lane l supplies A[i = l % 16][k = 8 (l / 16) .. +7]
// and B[k = 8 (l / 16) .. +7][j = l % 16]; accumulator register v of lane l holds
// C[4 (l / 16) + v][l % 16].

#include "common.hpp"
#include "engine.hpp"

namespace gx {

namespace {

typedef float f32x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

constexpr int kSW = 8;              // waves per workgroup
constexpr int kXS = kBN + 4;        // row stride of the transposed fp32 columns and of r (floats)
constexpr int kPS = kBN + 8;        // column stride of the bf16 parts: 16 columns on distinct banks

// v = p1 + p2 + p3 exactly, two values (em_full_wide.hip's split3v, whose comment
// explains the constants).
__device__ __forceinline__ void split_pair(float v0, float v1, bf16x2 nlo, bf16x2 nhi, bf16x2& p1, bf16x2& p2,
                                           bf16x2& p3) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  p1 = __builtin_convertvector(f32x2{v0, v1}, bf16x2);
  const float r0 = __builtin_amdgcn_fdot2_f32_bf16(p1, nlo, v0, false);
  const float r1 = __builtin_amdgcn_fdot2_f32_bf16(p1, nhi, v1, false);
  p2 = __builtin_convertvector(f32x2{r0, r1}, bf16x2);
  p3 = __builtin_convertvector(f32x2{__builtin_amdgcn_fdot2_f32_bf16(p2, nlo, r0, false),
                                     __builtin_amdgcn_fdot2_f32_bf16(p2, nhi, r1, false)}, bf16x2);
}

template <int NJ>
struct StatsLds {
  float xt[2][16 * NJ][kXS];                 // [buffer][column][row]
  __bf16 xp[2][3][16 * NJ][kPS];             // [buffer][part][column][row]
};

// Column groups of part Q: all of them up to NJ = 4, else the pair {Q, NJ - 1 - Q}.
template <int NJ, int Q>
struct Groups {
  static constexpr bool kAll = NJ <= 4;
  static constexpr int n = kAll ? NJ : (Q == NJ - 1 - Q ? 1 : 2);
  static constexpr int at(int i) { return kAll ? i : (i == 0 ? Q : NJ - 1 - Q); }
  static constexpr int lowest = kAll ? 0 : Q;
};

template <int NJ, int CT, int Q>
__device__ __forceinline__ void stats_part(const FwArgs& a, int ctile, StatsLds<NJ>& S, float (&rs)[2][CT][16][kXS]) {
  using G = Groups<NJ, Q>;
  constexpr int JW = 16 * NJ;                // staged columns
  constexpr int UP = (JW * 8 + 64 * kSW - 1) / (64 * kSW);   // (column, four rows) units per thread
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, g = lane >> 4;
  const int b = blockIdx.z;
  const int64_t N = a.N;
  const int D = a.D, K = a.K;
  const int64_t r0 = (int64_t)blockIdx.x * a.rows_per_slice;
  const int64_t r1 = (r0 + a.rows_per_slice < N) ? r0 + a.rows_per_slice : N;
  const float* xb = a.x + (size_t)b * N * D;
  const float* lse2 = a.lse2 + (size_t)b * N;
  const int k0 = ctile * CT * 16;
  const int rc = tid / kBN, rr = tid % kBN;  // this thread's responsibility: component, row

  uint32_t clo = 0x0000BF80u, chi = 0xBF800000u;
  asm("" : "+v"(clo), "+v"(chi));
  const bf16x2 nlo = __builtin_bit_cast(bf16x2, clo), nhi = __builtin_bit_cast(bf16x2, chi);

  // ---- loader: raw values of a block, then (one block later) its staged form ----
  float px[UP][4], pl[CT], pn = 0.f, pn_lo = 0.f;
  auto fetch = [&](int64_t n0) {
    const int left = r1 - n0 < kBN ? (int)(r1 - n0) : kBN;
    const float* blk = xb + (size_t)n0 * D;
#pragma unroll
    for (int u = 0; u < UP; ++u) {
      const int e = tid + u * 64 * kSW;
      if (JW * 8 % (64 * kSW) == 0 || e < JW * 8) {
        const int j = e % JW, q = e / JW, jc = j < D ? j : D - 1;
#pragma unroll
        for (int v = 0; v < 4; ++v) px[u][v] = blk[(4 * q + v < left ? 4 * q + v : left - 1) * D + jc];
      }
    }
    const int64_t n = n0 + (rr < left ? rr : left - 1);
    pn = lse2[n];
    if (a.lse_lo) pn_lo = a.lse_lo[(size_t)b * N + n];
    if (!a.hard) {
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        const int k = k0 + 16 * ct + rc;
        pl[ct] = a.l2[((size_t)b * K + (k < K ? k : K - 1)) * N + n];
      }
    }
  };
  auto stash = [&](int buf, int64_t n0) {
    const int left = r1 - n0 < kBN ? (int)(r1 - n0) : kBN;
#pragma unroll
    for (int u = 0; u < UP; ++u) {
      const int e = tid + u * 64 * kSW;
      if (JW * 8 % (64 * kSW) == 0 || e < JW * 8) {
        const int j = e % JW, q = e / JW;
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = (j < D && 4 * q + i < left) ? px[u][i] : 0.f;
        bf16x2 p[3][2];
#pragma unroll
        for (int i = 0; i < 2; ++i) split_pair(v[2 * i], v[2 * i + 1], nlo, nhi, p[0][i], p[1][i], p[2][i]);
        *reinterpret_cast<f32x4*>(&S.xt[buf][j][4 * q]) = f32x4{v[0], v[1], v[2], v[3]};
#pragma unroll
        for (int i = 0; i < 3; ++i)
          *reinterpret_cast<bf16x4*>(&S.xp[buf][i][j][4 * q]) = bf16x4{p[i][0][0], p[i][0][1], p[i][1][0], p[i][1][1]};
      }
    }
    const int64_t n = n0 + (rr < left ? rr : left - 1);
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      const int k = k0 + 16 * ct + rc;
      float r;
      if (a.hard) {
        r = a.hard_idx[(size_t)b * N + n] == k ? 1.f : 0.f;
      } else {
        r = fast_exp2((pl[ct] - pn) - pn_lo);
        if (a.thr2) {      // top-k mode: only the row's kept components
          const float t = a.thr2[(size_t)b * N + n];
          if (!(pl[ct] > t || (pl[ct] == t && k <= a.thr_idx[(size_t)b * N + n]))) r = 0.f;
        }
      }
      rs[buf][ct][rc][rr] = (k < K && rr < left) ? r : 0.f;
    }
  };

  f32x4 acc[CT][G::n][2][NJ], asx[CT];       // (blocks below a group's first are never touched)
  double nk[CT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
#pragma unroll
    for (int gi = 0; gi < G::n; ++gi)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int jb = 0; jb < NJ; ++jb) acc[ct][gi][h][jb] = f32x4{0.f, 0.f, 0.f, 0.f};
    asx[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
    nk[ct] = 0.0;
  }

  fetch(r0);
  stash(0, r0);
  if (r0 + kBN < r1) fetch(r0 + kBN);
  __syncthreads();
  int buf = 0;
  for (int64_t n0 = r0; n0 < r1; n0 += kBN, buf ^= 1) {
    float rv[CT][8];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      const f32x4 lo = *reinterpret_cast<const f32x4*>(&rs[buf][ct][li][8 * g]);
      const f32x4 hi = *reinterpret_cast<const f32x4*>(&rs[buf][ct][li][8 * g + 4]);
#pragma unroll
      for (int u = 0; u < 4; ++u) { rv[ct][u] = lo[u]; rv[ct][4 + u] = hi[u]; }
    }
    bf16x8 bq[NJ][3];
#pragma unroll
    for (int jb = G::lowest; jb < NJ; ++jb)
#pragma unroll
      for (int p = 0; p < 3; ++p) bq[jb][p] = *reinterpret_cast<const bf16x8*>(&S.xp[buf][p][16 * jb + li][8 * g]);

    // A operand from eight fp32 values; the products of blocks jb0 .. NJ-1 smallest
    // first, consecutive MFMAs into different accumulators.
    auto split8 = [&](const float (&v)[8], bf16x8 (&ap)[3]) {
#pragma unroll
      for (int u = 0; u < 8; u += 2) {
        bf16x2 p1, p2, p3;
        split_pair(v[u], v[u + 1], nlo, nhi, p1, p2, p3);
        ap[0][u] = p1[0]; ap[0][u + 1] = p1[1];
        ap[1][u] = p2[0]; ap[1][u + 1] = p2[1];
        ap[2][u] = p3[0]; ap[2][u + 1] = p3[1];
      }
    };
#pragma unroll
    for (int gi = 0; gi < G::n; ++gi) {
      const int jb0 = G::at(gi);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        // (columns D .. 16 NJ - 1 are staged as zeros: no branch, so one column's
        // split can run beside the previous one's MFMAs)
        const int i = 16 * jb0 + 2 * w + h;
        const f32x4 xl = *reinterpret_cast<const f32x4*>(&S.xt[buf][i][8 * g]);
        const f32x4 xh = *reinterpret_cast<const f32x4*>(&S.xt[buf][i][8 * g + 4]);
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
          float v[8];
#pragma unroll
          for (int u = 0; u < 4; ++u) { v[u] = rv[ct][u] * xl[u]; v[4 + u] = rv[ct][4 + u] * xh[u]; }
          bf16x8 ap[3];
          split8(v, ap);
          constexpr int PA[6] = {0, 2, 1, 0, 1, 0}, PB[6] = {2, 0, 1, 1, 0, 0};
#pragma unroll
          for (int p = 0; p < 6; ++p)
#pragma unroll
            for (int jb = 0; jb < NJ; ++jb)
              if (jb >= jb0) acc[ct][gi][h][jb] = mfma_bf16(ap[PA[p]], bq[jb][PB[p]], acc[ct][gi][h][jb]);
        }
      }
    }
    if (Q == 0 && w < NJ) {                    // Σ r x of column block w, Σ r (wave 0)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        bf16x8 ap[3], bw[3];
        split8(rv[ct], ap);
#pragma unroll
        for (int p = 0; p < 3; ++p) bw[p] = *reinterpret_cast<const bf16x8*>(&S.xp[buf][p][16 * w + li][8 * g]);
        constexpr int PA[6] = {0, 2, 1, 0, 1, 0}, PB[6] = {2, 0, 1, 1, 0, 0};
#pragma unroll
        for (int p = 0; p < 6; ++p) asx[ct] = mfma_bf16(ap[PA[p]], bw[PB[p]], asx[ct]);
        if (w == 0)
          nk[ct] += (double)(((rv[ct][0] + rv[ct][1]) + (rv[ct][2] + rv[ct][3])) +
                             ((rv[ct][4] + rv[ct][5]) + (rv[ct][6] + rv[ct][7])));
      }
    }
    if (n0 + kBN < r1) stash(buf ^ 1, n0 + kBN);
    if (n0 + 2 * kBN < r1) fetch(n0 + 2 * kBN);
    __syncthreads();
  }

  // Statistics row: [Σ r x (DP) | Σ r x xᵀ packed (d <= e < DP, row by row) | N_k | 0 ...]
  const int DP = a.nk_dp;
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    double t = nk[ct];
    t += __shfl_xor(t, 16);
    t += __shfl_xor(t, 32);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int k = k0 + 16 * ct + 4 * g + v;
      const float nkv = (float)__shfl(t, 4 * g + v);
      if (k < K) {
        float* out = a.part_stats + (((size_t)blockIdx.x * a.B + b) * K + k) * a.JP;
#pragma unroll
        for (int gi = 0; gi < G::n; ++gi)
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int i = 16 * G::at(gi) + 2 * w + h;
            if (i < D) {
#pragma unroll
              for (int jb = 0; jb < NJ; ++jb)
                if (jb >= G::at(gi) && 16 * jb + li >= i)
                  out[DP + fw_tri(DP, i, 16 * jb + li)] = acc[ct][gi][h][jb][v];
            }
          }
        if (Q == 0 && w < NJ) out[16 * w + li] = asx[ct][v];
        if (Q == 0 && w == 0 && a.nk_col + li < a.JP) out[a.nk_col + li] = li == 0 ? nkv : 0.f;
      }
    }
  }
}

template <int NJ, int CT>
__global__ __launch_bounds__(64 * kSW) void fw_stats_tile_kernel(FwArgs a) {
  __shared__ __align__(16) StatsLds<NJ> S;
  __shared__ __align__(16) float rs[2][CT][16][kXS];
  if constexpr (NJ <= 4) {
    stats_part<NJ, CT, 0>(a, blockIdx.y, S, rs);
  } else {
    constexpr int NP = (NJ + 1) / 2;
    const int ctile = blockIdx.y / NP;
    switch (blockIdx.y % NP) {
      case 0: stats_part<NJ, CT, 0>(a, ctile, S, rs); break;
      case 1: stats_part<NJ, CT, 1>(a, ctile, S, rs); break;
      case 2: if constexpr (NP > 2) stats_part<NJ, CT, 2>(a, ctile, S, rs); break;
      default: if constexpr (NP > 3) stats_part<NJ, CT, 3>(a, ctile, S, rs); break;
    }
  }
}

// Components per workgroup: two tiles of 16 share the staged rows at D <= 32, where the
// accumulators leave the registers for it (K = 32: 0.112 ms, 3.5 µs per component
// slot; three workgroups of one tile at K = 40: 5.5).
int comp_tiles(int D, int K) { return D <= 32 && K > 16 ? 2 : 1; }
int parts_of(int D) { return D <= 64 ? 1 : ((D + 15) / 16 + 1) / 2; }

template <int NJ, int CT = 1>
void launch_tile(const FwArgs& a, int slices, hipStream_t s) {
  fw_stats_tile_kernel<NJ, CT><<<dim3(slices, fw_stats_tile_groups(a.D, a.K), a.B), 64 * kSW, 0, s>>>(a);
}

}  // namespace

int fw_stats_tile_groups(int D, int K) {
  const int per = 16 * comp_tiles(D, K);
  return (K + per - 1) / per * parts_of(D);
}

int launch_fw_stats_tile(const FwArgs& a, int slices, hipStream_t s) {
  switch ((a.D + 15) / 16) {
    case 2:
      if (comp_tiles(a.D, a.K) == 2) launch_tile<2, 2>(a, slices, s);
      else launch_tile<2>(a, slices, s);
      return 0;
    case 3: launch_tile<3>(a, slices, s); return 0;
    case 4: launch_tile<4>(a, slices, s); return 0;
    case 5: launch_tile<5>(a, slices, s); return 0;
    case 6: launch_tile<6>(a, slices, s); return 0;
    case 7: launch_tile<7>(a, slices, s); return 0;
    case 8: launch_tile<8>(a, slices, s); return 0;
    default: return -1;
  }
}

}  // namespace gx
