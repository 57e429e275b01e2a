// Greedy k-means++ seeding on a row sample (initialisation of the EM fit).
//
// Restates _kmeans_plus_plus_init_means (gmmxx/torch_fallback.py:1390-1451):
// the first centre is a given row; every later centre is the best of T
// candidates drawn with probability proportional to the squared distance to the
// nearest centre so far (D² sampling through the running cumulative sum), "best"
// meaning the smallest potential Σ_i min(closest_i, ‖s_i - c‖²).  The random
// numbers (first row, uniform draws) are inputs, so the result is a pure
// function of them.
//
// Per step two launches: kpp_trial_kernel (many workgroups over the rows:
// candidate distances and per-block partial potentials) and kpp_pick_kernel
// (one workgroup per batch: pick the candidate, update the closest distances,
// then scan them and draw the next step's candidates).  The row sample is read
// once per step (T distances per row from one read); everything else is
// O(S) per step.

#include "common.hpp"
#include "engine.hpp"
#include "params.hpp"

namespace gx {

namespace {

constexpr int kTrialThreads = 256;   // rows of one block of the potential sums
constexpr int kBlockWaves = kTrialThreads / 64;
constexpr int kPickThreads = 1024;

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int off = 32; off >= 1; off /= 2) v += __shfl_xor(v, off);
  return v;
}

// Squared Euclidean distances of one row to `t_count` LDS-resident candidates
// (direct differences, as the reference computes them).
template <bool VEC, int TT>
__device__ __forceinline__ void row_dists(const float* __restrict__ row, const float* cand, int D, int t_count,
                                          float (&acc)[TT]) {
#pragma unroll
  for (int t = 0; t < TT; ++t) acc[t] = 0.f;
  if constexpr (VEC) {
#pragma unroll 2
    for (int d = 0; d < D; d += 4) {
      const float4 v = *reinterpret_cast<const float4*>(row + d);
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        if (t < t_count) {
          const float4 c = *reinterpret_cast<const float4*>(cand + t * D + d);
          const float a = v.x - c.x, b = v.y - c.y, e = v.z - c.z, f = v.w - c.w;
          acc[t] = fmaf(a, a, acc[t]);
          acc[t] = fmaf(b, b, acc[t]);
          acc[t] = fmaf(e, e, acc[t]);
          acc[t] = fmaf(f, f, acc[t]);
        }
      }
    }
  } else {
    for (int d = 0; d < D; ++d) {
      const float v = row[d];
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        if (t < t_count) {
          const float a = v - cand[t * D + d];
          acc[t] = fmaf(a, a, acc[t]);
        }
      }
    }
  }
}

// closest_i = ‖s_i - s_first‖²; workgroup (0, b) also writes centre 0.
__global__ __launch_bounds__(kTrialThreads) void kpp_first_kernel(KppArgs a) {
  extern __shared__ float cand[];
  const int b = blockIdx.y;
  const float* sample = a.sample + (size_t)b * a.S * a.D;
  const int64_t f = min<int64_t>(max<int64_t>(a.first[b], 0), a.S - 1);
  for (int d = threadIdx.x; d < a.D; d += blockDim.x) {
    const float v = sample[(size_t)f * a.D + d];
    cand[d] = v;
    if (blockIdx.x == 0) a.centers[(size_t)b * a.K * a.D + d] = v;
  }
  __syncthreads();
  const int i = blockIdx.x * kTrialThreads + threadIdx.x;
  if (i < a.S) {
    float acc[1];
    if (a.vec) row_dists<true, 1>(sample + (size_t)i * a.D, cand, a.D, 1, acc);
    else row_dists<false, 1>(sample + (size_t)i * a.D, cand, a.D, 1, acc);
    a.closest[(size_t)b * a.S + i] = acc[0];
  }
}

// Distances of every row to the step's T candidates (kept for the pick) and the
// wave's partial potentials Σ min(closest, dist) per candidate.  One wave per
// workgroup: a sample of 4096 rows then covers 64 CUs instead of 16.  TT: an upper
// bound of T (the per-candidate code is unrolled TT times).
template <int TT>
__global__ __launch_bounds__(64) void kpp_trial_kernel(KppArgs a) {
  extern __shared__ float cand[];
  const int b = blockIdx.y, T = a.T;
  const float* sample = a.sample + (size_t)b * a.S * a.D;
  for (int t = 0; t < T; ++t) {
    const float* row = sample + (size_t)a.cand[b * kKppMaxTrials + t] * a.D;
    for (int d = threadIdx.x; d < a.D; d += 64) cand[t * a.D + d] = row[d];
  }
  __syncthreads();
  const int i = blockIdx.x * 64 + threadIdx.x;
  float acc[TT];
  if (i < a.S) {
    const float cl = a.closest[(size_t)b * a.S + i];
    if (a.vec) row_dists<true, TT>(sample + (size_t)i * a.D, cand, a.D, T, acc);
    else row_dists<false, TT>(sample + (size_t)i * a.D, cand, a.D, T, acc);
#pragma unroll
    for (int t = 0; t < TT; ++t) {
      if (t < T) {
        a.dist[((size_t)b * kKppMaxTrials + t) * a.S + i] = acc[t];
        acc[t] = fminf(cl, acc[t]);
      }
    }
  } else {
#pragma unroll
    for (int t = 0; t < TT; ++t) acc[t] = 0.f;
  }
#pragma unroll
  for (int t = 0; t < TT; ++t) {
    if (t < T) {
      const float s = wave_sum(acc[t]);
      if (threadIdx.x == 0) a.pot_part[((size_t)b * a.nblk * kBlockWaves + blockIdx.x) * kKppMaxTrials + t] = s;
    }
  }
}

// Inclusive scan of one value per thread over 1024 threads, bit for bit the
// Hillis-Steele scan (step off = 1, 2, 4 .. 512: v[i] += v[i - off]).  The first six
// steps read at most 63 places back, so a wave takes them in registers on its own
// 64 values and the previous wave's (whose left end, wrong after a few steps, is
// out of that reach); only the last four go through LDS, one barrier each (the
// plain form's twenty took most of 2 µs).
__device__ __forceinline__ float scan1024(float v, float (&buf)[2][kPickThreads]) {
  const int tid = threadIdx.x, lane = tid & 63;
  buf[0][tid] = v;
  __syncthreads();
  float prev = tid >= 64 ? buf[0][tid - 64] : 0.f;
#pragma unroll
  for (int off = 1; off < 64; off *= 2) {
    const float own = __shfl_up(v, off), left = __shfl_up(prev, off);
    const float wrap = __shfl(prev, (lane - off) & 63);
    v += lane >= off ? own : wrap;
    prev += lane >= off ? left : 0.f;
  }
  int cur = 1;
#pragma unroll
  for (int off = 64; off < kPickThreads; off *= 2) {
    buf[cur][tid] = v;
    __syncthreads();
    v += tid >= off ? buf[cur][tid - off] : 0.f;
    cur ^= 1;
  }
  return v;
}

// Step `step` (>= 1): the candidate of least potential (first on ties) becomes
// centre `step` and the closest distances take its column.  Then, when
// step + 1 < K, the next step's candidates: thread j owns rows [jR, jR + R),
// the chunk sums are scanned across the workgroup, and draw u·total lands on
// the first row whose running sum reaches it (searchsorted, left side), the
// last row when it exceeds the total, row 0 when the total is 0.
// One workgroup, bound by latency: the potentials' partials are brought to LDS
// together and summed by one thread per candidate in block order (one thread
// reading them all one by one from memory kept the launch at 14.4 µs at S = 4096,
// T = 6; now 7.8).
__global__ __launch_bounds__(kPickThreads) void kpp_pick_kernel(KppArgs a, int step) {
  __shared__ float buf[2][kPickThreads];
  __shared__ float pots[kKppMaxRows / kTrialThreads * kKppMaxTrials];
  __shared__ double pot_s[kKppMaxTrials];
  const int b = blockIdx.x, tid = threadIdx.x, T = a.T;
  const float* sample = a.sample + (size_t)b * a.S * a.D;
  float* closest = a.closest + (size_t)b * a.S;
  int* cand = a.cand + b * kKppMaxTrials;
  const int R = (a.S + kPickThreads - 1) / kPickThreads;
  const int i0 = min(a.S, tid * R), i1 = min(a.S, i0 + R);
  const float* u = a.draws + ((size_t)b * (a.K - 1) + step) * T;
  const bool more = step + 1 < a.K;

  float cs = 0.f;
  if (step >= 1) {
    // a block's potential: its waves' sums in wave order (waves past S wrote none)
    const float* pp = a.pot_part + (size_t)b * a.nblk * kBlockWaves * kKppMaxTrials;
    const int nw = (a.S + 63) / 64;
    for (int e = tid; e < a.nblk * kKppMaxTrials; e += kPickThreads) {
      const int k = e / kKppMaxTrials, t = e % kKppMaxTrials;
      float s = 0.f;
#pragma unroll
      for (int w = 0; w < kBlockWaves; ++w)
        s += k * kBlockWaves + w < nw ? pp[(size_t)(k * kBlockWaves + w) * kKppMaxTrials + t] : 0.f;
      pots[e] = s;
    }
    __syncthreads();
    if (tid < T) {
      double p = 0.0;
#pragma unroll 8
      for (int k = 0; k < a.nblk; ++k) p += (double)pots[k * kKppMaxTrials + tid];
      pot_s[tid] = p;
    }
    __syncthreads();
    int best = 0;
    double best_v = pot_s[0];
    for (int t = 1; t < T; ++t) {
      const double p = pot_s[t];
      if (p < best_v) { best_v = p; best = t; }
    }
    const int64_t row = cand[best];
    for (int d = tid; d < a.D; d += kPickThreads)
      a.centers[((size_t)b * a.K + step) * a.D + d] = sample[(size_t)row * a.D + d];
    if (!more) return;                     // (uniform) nothing reads the closest distances again
    const float* db = a.dist + ((size_t)b * kKppMaxTrials + best) * a.S;
#pragma unroll 4
    for (int i = i0; i < i1; ++i) {
      const float c = fminf(closest[i], db[i]);
      closest[i] = c;
      cs += c;
    }
  } else {
    if (!more) return;
#pragma unroll 4
    for (int i = i0; i < i1; ++i) cs += closest[i];
  }
  // (the scan's barriers also keep every read of cand[] above its rewrite below)
  const float incl = scan1024(cs, buf);
  __syncthreads();
  buf[0][tid] = incl;
  __syncthreads();
  const float prev = (tid == 0) ? 0.f : buf[0][tid - 1];
  const float total = buf[0][kPickThreads - 1];
  for (int t = 0; t < T; ++t) {
    if (!(total > 0.f)) {
      if (tid == 0) cand[t] = 0;
      continue;
    }
    const float target = u[t] * total;
    if (!(target <= total)) {   // beyond the total (or NaN): clamp to the last row
      if (tid == 0) cand[t] = a.S - 1;
      continue;
    }
    if (incl >= target && (tid == 0 || prev < target) && i1 > i0) {
      float run = prev;
      int idx = i1 - 1;
      for (int i = i0; i < i1; ++i) {
        run += closest[i];
        if (run >= target) { idx = i; break; }
      }
      cand[t] = idx;
    }
  }
}

// ---------------------------------------------------------------------------
// Lloyd centre update: centre = mean of its rows (an empty cluster keeps its
// centre) and the largest Euclidean move of any centre, one wave per centre
// (3.8 µs in place of seven elementwise and reduction launches of 3 to 5 µs each).
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(256) void lloyd_update_kernel(const float* nk, const float* sum_x, float* means, int64_t M,
                                                           int D, unsigned* shift) {
  const int64_t k = (int64_t)blockIdx.x * 4 + threadIdx.x / 64;
  const int lane = threadIdx.x & 63;
  if (k >= M) return;
  const float n = nk[k];
  const float den = n < 1.f ? 1.f : n;     // (a NaN count passes through, as torch's clamp_min)
  float q = 0.f;
  for (int d = lane; d < D; d += 64) {
    const float old = means[k * D + d];
    const float v = n > 0.f ? sum_x[k * D + d] / den : old;
    means[k * D + d] = v;
    q = fmaf(v - old, v - old, q);
  }
  q = sqrtf(wave_sum(q));
  // Non-negative floats order as their bits (a NaN above all): the maximum does not
  // depend on the order of the updates.
  if (lane == 0) atomicMax(shift, __float_as_uint(q) & 0x7fffffffu);
}

}  // namespace

int64_t kpp_workspace_bytes(int B, int S, int K, int T) {
  (void)K;
  (void)T;
  const int64_t nblk = (S + kTrialThreads - 1) / kTrialThreads;
  auto up = [](int64_t v) { return (v + 255) / 256 * 256; };
  return up((int64_t)B * S * 4) + up((int64_t)B * kKppMaxTrials * S * 4) +
         up((int64_t)B * nblk * kBlockWaves * kKppMaxTrials * 4) + up((int64_t)B * kKppMaxTrials * 4);
}

void kpp_bind_workspace(KppArgs& a, void* ws) {
  a.nblk = (a.S + kTrialThreads - 1) / kTrialThreads;
  auto up = [](int64_t v) { return (v + 255) / 256 * 256; };
  char* p = static_cast<char*>(ws);
  a.closest = reinterpret_cast<float*>(p);
  p += up((int64_t)a.B * a.S * 4);
  a.dist = reinterpret_cast<float*>(p);
  p += up((int64_t)a.B * kKppMaxTrials * a.S * 4);
  a.pot_part = reinterpret_cast<float*>(p);
  p += up((int64_t)a.B * a.nblk * kBlockWaves * kKppMaxTrials * 4);
  a.cand = reinterpret_cast<int*>(p);
}

void launch_kpp(const KppArgs& a, hipStream_t s) {
  const dim3 rows(a.nblk, a.B);
  kpp_first_kernel<<<rows, kTrialThreads, a.D * sizeof(float), s>>>(a);
  kpp_pick_kernel<<<a.B, kPickThreads, 0, s>>>(a, 0);
  for (int step = 1; step < a.K; ++step) {
    const dim3 waves((a.S + 63) / 64, a.B);
    const size_t lds = (size_t)a.T * a.D * sizeof(float);
    if (a.T <= 4) kpp_trial_kernel<4><<<waves, 64, lds, s>>>(a);
    else if (a.T <= 6) kpp_trial_kernel<6><<<waves, 64, lds, s>>>(a);
    else if (a.T <= 8) kpp_trial_kernel<8><<<waves, 64, lds, s>>>(a);
    else kpp_trial_kernel<kKppMaxTrials><<<waves, 64, lds, s>>>(a);
    kpp_pick_kernel<<<a.B, kPickThreads, 0, s>>>(a, step);
  }
}

void launch_lloyd_update(const float* nk, const float* sum_x, float* means, int64_t M, int D, float* shift,
                         hipStream_t s) {
  launch_zero_words(reinterpret_cast<unsigned*>(shift), 1, s);
  lloyd_update_kernel<<<(unsigned)((M + 3) / 4), 256, 0, s>>>(nk, sum_x, means, M, D, reinterpret_cast<unsigned*>(shift));
}

}  // namespace gx
