// Computational-basis shot sampling: replaces the reference's measure()
// (torchquantum/measurement/measurements.py:37-74), which copies |psi| to the
// host and draws n_shots outcomes per batch row with random.choices over all
// 2^n bitstrings.  Here the state never leaves HBM:
//   1. k_block_probs: p_j = |a_j|^2 summed over blocks of SB = 4096
//      amplitudes (float64 partials), one workgroup per block, and over the
//      block's 64 segments, with their prefix;
//   2. k_block_scan: per row, an inclusive prefix of the block sums;
//   3. k_draw: one thread per shot draws u in [0, 1) from a counter-based
//      generator (splitmix64 of seed, row, shot), finds the block and the
//      segment by binary searches over the prefixes, then walks the segment's
//      amplitudes.
// Only indices with p_j > 0 can be drawn.  The output is the flat in-row
// index (wire 0 = most significant bit, the reference's bitstring order).
#include "tqsv_common.h"

namespace tqsv {

constexpr int SB = 4096;            // amplitudes per block
constexpr int SB_THREADS = 256;     // block-sum workgroup (16 amplitudes per thread)
constexpr int SEGS = 64;            // segments per block, one per lane of a wavefront
constexpr int AHEAD = 8;            // amplitudes a drawing thread loads at once

// One segment: its sum (float64, in index order) and the inclusive prefix of
// the sums over its block.
struct Seg {
  double sum, inc;
};

__device__ __forceinline__ float prob(const float2 a) { return a.x * a.x + a.y * a.y; }

// Amplitudes per segment of a block of blen amplitudes: segment l holds
// [l * per, (l + 1) * per), the last ones cut at blen (or empty).
__device__ __forceinline__ uint32_t seg_len(uint32_t blen) { return (blen + SEGS - 1) / SEGS; }

// sums[row * nb + b] = sum_{j in block b} |a_j|^2 and segs[(row * nb + b) *
// SEGS + l] = segment l; grid = (nb, bsz).  One pass over the state for both:
// the block's probabilities stay in LDS (one spare float after every 64, so
// that the 64 segments' walkers read different banks) while a wavefront's
// lanes add up a segment each.  Bound by the state's read: 28 us for 16 rows
// of 2^20 (21 us before it also wrote the segments).
__global__ __launch_bounds__(SB_THREADS) void k_block_probs(const float2* __restrict__ st, int n, int64_t nb,
                                                            double* __restrict__ sums, Seg* __restrict__ segs) {
  __shared__ float pr[SB + SB / 64];
  const uint64_t row = blockIdx.y;
  const uint64_t b = blockIdx.x;
  const uint64_t N = 1ull << n;
  const uint64_t base = (row << n) + b * SB;
  const uint32_t end = (b * SB + SB < N) ? SB : (uint32_t)(N - b * SB);
  double acc = 0.0;
  for (uint32_t j = threadIdx.x; j < end; j += SB_THREADS) {
    const float p = prob(st[base + j]);
    pr[j + (j >> 6)] = p;
    acc += (double)p;
  }
  for (int o = 32; o >= 1; o >>= 1) acc += __shfl_xor(acc, o, 64);
  __shared__ double part[SB_THREADS / 64];
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x < SEGS) {
    const uint32_t per = seg_len(end);
    uint32_t j = threadIdx.x * per < end ? threadIdx.x * per : end;
    const uint32_t last = j + per < end ? j + per : end;
    double s = 0.0;
    for (; j < last; ++j) s += (double)pr[j + (j >> 6)];
    double inc = s;
    for (int o = 1; o < 64; o <<= 1) {
      const double v = __shfl_up(inc, o, 64);
      if ((int)threadIdx.x >= o) inc += v;
    }
    segs[(row * nb + b) * SEGS + threadIdx.x] = Seg{s, inc};
  } else if (threadIdx.x == SEGS) {
    double s = 0.0;
    for (int w = 0; w < SB_THREADS / 64; ++w) s += part[w];
    sums[row * nb + b] = s;
  }
}

// inclusive prefix of sums over each row, in place; one workgroup per row
__global__ __launch_bounds__(256) void k_block_scan(double* __restrict__ sums, int64_t nb) {
  double* p = sums + (uint64_t)blockIdx.x * nb;
  const int64_t per = (nb + 255) / 256;
  const int64_t lo = threadIdx.x * per;
  const int64_t hi = lo + per < nb ? lo + per : nb;
  double s = 0.0;
  for (int64_t i = lo; i < hi; ++i) s += p[i];
  __shared__ double tot[256];
  tot[threadIdx.x] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double run = 0.0;
    for (int t = 0; t < 256; ++t) {
      const double v = tot[t];
      tot[t] = run;
      run += v;
    }
  }
  __syncthreads();
  double run = tot[threadIdx.x];
  for (int64_t i = lo; i < hi; ++i) {
    run += p[i];
    p[i] = run;
  }
}

__device__ __forceinline__ uint64_t splitmix64(uint64_t x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}

// one thread per (row, shot), 64 threads per workgroup so that few shots still
// spread over the chip.  A shot reads O(log) prefix entries and at most one
// segment (64 amplitudes, AHEAD loads in flight); with a wavefront per shot
// that summed its block's 4096 amplitudes, 131072 shots from 16 rows of 2^20
// took 2082 us, with one that added a segment's amplitudes lane by lane 160 us
// (issue-bound on one live lane), this way 30 us (latency of the searches).
__global__ __launch_bounds__(64) void k_draw(const float2* __restrict__ st, int n, int64_t nb,
                                             const double* __restrict__ prefix, const Seg* __restrict__ segs,
                                             int64_t n_shots, uint64_t seed, int64_t bsz,
                                             int64_t* __restrict__ out) {
  const uint64_t id = (uint64_t)blockIdx.x * 64 + threadIdx.x;
  if (id >= (uint64_t)bsz * (uint64_t)n_shots) return;
  const uint64_t row = id / (uint64_t)n_shots;
  const double* P = prefix + row * nb;
  const double total = P[nb - 1];
  const uint64_t r = splitmix64(seed ^ splitmix64(id));
  const double u = (double)(r >> 11) * (1.0 / 9007199254740992.0);  // [0, 1)
  double t = u * total;
  // first block with prefix > t
  int64_t lo = 0, hi = nb - 1;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (P[mid] > t) hi = mid; else lo = mid + 1;
  }
  const int64_t b = lo;
  t -= (b > 0 ? P[b - 1] : 0.0);
  const uint64_t N = 1ull << n;
  const uint64_t bstart = (uint64_t)b * SB;
  const uint32_t blen = (bstart + SB < N) ? SB : (uint32_t)(N - bstart);
  const uint32_t per = seg_len(blen);
  // first segment with mass whose prefix passes t
  const Seg* S = segs + (row * nb + b) * SEGS;
  int sel = 0;
  for (int step = SEGS / 2; step >= 1; step >>= 1)
    if (!(S[sel + step - 1].inc > t)) sel += step;
  while (sel < SEGS && !(S[sel].inc > t && S[sel].sum > 0.0)) ++sel;
  const bool exact = sel < SEGS;
  if (!exact) {   // rounding pushed t past the block's total: the last segment with mass
    sel = SEGS - 1;
    while (sel > 0 && !(S[sel].sum > 0.0)) --sel;
  }
  const uint32_t lbeg = sel * per < blen ? sel * per : blen;
  const uint32_t len = lbeg + per < blen ? per : blen - lbeg;
  const float2* a = st + (row << n) + bstart + lbeg;
  // the element where the running sum passes t; without an exact hit, the
  // segment's last element with nonzero probability
  uint32_t pick = 0;
  double acc = S[sel].inc - S[sel].sum;
  bool found = false;
  for (uint32_t j0 = 0; j0 < len && !found; j0 += AHEAD) {
    float p[AHEAD];
#pragma unroll
    for (int k = 0; k < AHEAD; ++k) p[k] = j0 + k < len ? prob(a[j0 + k]) : 0.f;
#pragma unroll
    for (int k = 0; k < AHEAD; ++k) {
      if (!found && p[k] > 0.f) {
        pick = j0 + k;
        acc += (double)p[k];
        found = exact && acc > t;
      }
    }
  }
  out[id] = (int64_t)(bstart + lbeg + pick);
}

}  // namespace tqsv

using namespace tqsv;

TQSV_API int64_t tqsv_sample_workspace_bytes(int64_t bsz, int n) {
  if (bsz < 1 || n < 0 || n > 32) return -1;
  const int64_t N = 1ll << n;
  const int64_t nb = (N + SB - 1) / SB;
  return bsz * nb * (int64_t)(sizeof(double) + SEGS * sizeof(Seg));
}

TQSV_API int tqsv_sample(hipStream_t s, const void* state, int64_t bsz, int n, int64_t n_shots, uint64_t seed,
                         int64_t* out, void* workspace, int64_t ws_bytes) {
  if (!state || !out || !workspace) { set_error("tqsv_sample: null pointer"); return E_ARG; }
  if (bsz < 1 || bsz > 65535 || n < 0 || n > 32) { set_error("tqsv_sample: bad bsz/n (bsz <= 65535, n <= 32)"); return E_ARG; }
  if (n_shots < 1) { set_error("tqsv_sample: n_shots must be >= 1"); return E_ARG; }
  const int64_t need = tqsv_sample_workspace_bytes(bsz, n);
  if (ws_bytes < need) { set_error("tqsv_sample: workspace %lld bytes < %lld", (long long)ws_bytes, (long long)need); return E_ARG; }
  const int64_t N = 1ll << n;
  const int64_t nb = (N + SB - 1) / SB;
  const uint64_t shots = (uint64_t)bsz * (uint64_t)n_shots;
  if (shots > (1ull << 26)) { set_error("tqsv_sample: bsz * n_shots exceeds 2^26"); return E_LIMIT; }
  double* sums = (double*)workspace;
  Seg* segs = (Seg*)(sums + bsz * nb);
  k_block_probs<<<dim3((unsigned)nb, (unsigned)bsz), SB_THREADS, 0, s>>>((const float2*)state, n, nb, sums, segs);
  k_block_scan<<<(unsigned)bsz, 256, 0, s>>>(sums, nb);
  k_draw<<<(unsigned)((shots + 63) / 64), 64, 0, s>>>((const float2*)state, n, nb, sums, segs, n_shots, seed, bsz, out);
  return check_launch("tqsv_sample");
}
