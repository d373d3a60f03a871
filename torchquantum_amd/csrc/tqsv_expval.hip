// Pauli expectation kernels (one read pass of the state per distinct flip mask).
//
// Replaces:
//   * expval / MeasureAll (torchquantum/measurement/measurements.py:282-343):
//     |psi|^2 then one full reduction per wire -> here one pass computes
//     <Z_w> for every wire: <Z_w> = sum_j p_j - 2 * sum_{j: bit(w)=1} p_j;
//   * expval_joint_analytical (measurements.py:232-279), which builds a dense
//     2^n x 2^n Kronecker Hamiltonian (O(4^n) memory) -> here a Pauli string
//     P = i^{nY} X^x Z^z is applied through its flip mask x and phase mask z:
//     <psi|P|psi> = i^{nY} sum_j (-1)^{popcount(j & z)} conj(psi_{j^x}) psi_j.
// Reductions: per-thread partial sums -> 64-lane shuffle tree -> LDS across
// waves -> one partial per (row, chunk, term) -> a second tiny kernel sums
// the chunks in float64.  No float atomics, so results are deterministic.
#include <algorithm>
#include <memory>
#include <mutex>
#include <type_traits>
#include <vector>

#include "tqsv_common.h"

namespace tqsv {
int num_cu();
}

namespace tqsv {

constexpr int EV_THREADS = 256;
constexpr int EV_MAXQ = 32;      // wires per <Z_w> launch (n <= 32)
constexpr int EV_MAXT = 16;      // terms per diagonal-term launch

// grid of 256-thread blocks for one wavefront per output
static unsigned sum_grid(int64_t outputs) { return (unsigned)((outputs * 64 + 255) / 256); }

// chunks per row so that the grid has enough blocks; chunk = power of two amps
static int ev_chunk_log2(int64_t bsz, int n) {
  // at least 2 amps per thread per chunk, at most the whole row
  int lg = n;
  const int min_lg = 9 + 2;  // 256 threads * 2 amps * 4 iterations
  const int64_t want_blocks = (int64_t)num_cu() * 8;
  while (lg > min_lg && (bsz << (n - lg)) < want_blocks) --lg;
  if (lg > n) lg = n;
  return lg;
}

__device__ __forceinline__ float block_sum(float v, float* red) {
  // red: >= EV_THREADS / 64 floats of LDS
  v = wave_sum(v, 64);
  const int w = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[w] = v;
  __syncthreads();
  float s = 0.f;
  if (threadIdx.x == 0)
    for (int i = 0; i < (int)(blockDim.x >> 6); ++i) s += red[i];
  return s;  // valid in thread 0
}

__device__ __forceinline__ double wave_sum_d(double v) {
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// The workgroup's sum in float64; red: a double of LDS per wavefront.
__device__ __forceinline__ double block_sum_d(double v, double* red) {
  v = wave_sum_d(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x == 0)
    for (int i = 0; i < (int)(blockDim.x >> 6); ++i) s += red[i];
  return s;  // valid in thread 0
}

// Loads in flight per thread in the chunk walks below: one 16-byte load per
// trip leaves too few bytes in flight to cover HBM latency.
constexpr int EV_UNROLL = 4;
static_assert(EV_UNROLL == 4 && EV_THREADS == 256, "k_ez_part maps amplitude bits 9, 10 to the unroll slot");

// <Z_w> partials: part[(row * nchunks + chunk) * (n + 1) + q], q < n: sum of p
// over amplitudes with bit q set; q = n: total probability.
__global__ __launch_bounds__(EV_THREADS) void k_ez_part(const float4* __restrict__ st, int n, int lg_chunk,
                                                        float* __restrict__ part) {
  __shared__ float red[EV_THREADS / 64];
  const int nchunks = 1 << (n - lg_chunk);
  const uint64_t row = blockIdx.x >> (n - lg_chunk);
  const uint64_t chunk = blockIdx.x & (nchunks - 1);
  const uint64_t first = (row << n) + (chunk << lg_chunk);  // amplitude index
  const uint64_t npairs = (1ull << lg_chunk) >> 1;
  // Thread t reads float4 i = t + 256 k, i.e. amplitudes j = chunk_base +
  // 2 t + 512 k (+1), all parts on disjoint bits: bit 0 of j is the float4
  // half; bits 1..8 are bits of t (fixed per thread: those sums follow from
  // the thread's total at the end); bits 9, 10 are bits of the unroll slot u
  // (k = trip * 4 + u); bits 11 .. lg_chunk - 1 are bits of the trip
  // (wave-uniform, one add per trip); bits >= lg_chunk are bits of the
  // chunk (constant per block: taken from the total at the end).  A chunk
  // shorter than 512 amplitudes is a whole row (n <= 11), where k = 0 and
  // threads past its end read nothing.
  float S[EV_MAXQ];
#pragma unroll
  for (int q = 0; q < EV_MAXQ; ++q) S[q] = 0.f;
  float tot = 0.f, s0 = 0.f;
  for (uint64_t b = threadIdx.x, k = 0; b < npairs; b += EV_UNROLL * EV_THREADS, k += EV_UNROLL) {
    float4 v[EV_UNROLL];
#pragma unroll
    for (int u = 0; u < EV_UNROLL; ++u) {
      const uint64_t i = b + (uint64_t)u * EV_THREADS;
      v[u] = i < npairs ? st[(first >> 1) + i] : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    float ts = 0.f;
#pragma unroll
    for (int u = 0; u < EV_UNROLL; ++u) {
      const float p0 = v[u].x * v[u].x + v[u].y * v[u].y;
      const float p1 = v[u].z * v[u].z + v[u].w * v[u].w;
      const float pp = p0 + p1;
      ts += pp;
      s0 += p1;
      if (u & 1) S[9] += pp;
      if (u & 2) S[10] += pp;
    }
    tot += ts;
    const uint32_t kk = (uint32_t)k;   // wave-uniform, a multiple of 4
#pragma unroll
    for (int q = 11; q < EV_MAXQ; ++q)
      if (q < lg_chunk && ((kk >> (q - 9)) & 1u)) S[q] += ts;
  }
  const uint64_t cb = chunk << lg_chunk;
#pragma unroll
  for (int q = 9; q < EV_MAXQ; ++q)
    if (q >= lg_chunk) S[q] = ((cb >> q) & 1u) ? tot : 0.f;
  S[0] = s0;
#pragma unroll
  for (int q = 1; q <= 8; ++q)
    if (q < n) S[q] = ((threadIdx.x >> (q - 1)) & 1u) ? tot : 0.f;
  float* out = part + (uint64_t)blockIdx.x * (n + 1);
#pragma unroll
  for (int q = 0; q < EV_MAXQ; ++q) {
    if (q < n) {
      const float s = block_sum(S[q], red);
      if (threadIdx.x == 0) out[q] = s;
    }
  }
  const float s = block_sum(tot, red);
  if (threadIdx.x == 0) out[n] = s;
}

// out[row * n + w] = total - 2 * S[n - 1 - w]; one wavefront per output, its
// lanes striding over the row's chunk partials.
__global__ __launch_bounds__(256) void k_ez_final(const float* __restrict__ part, int n, int nchunks, int64_t bsz,
                                                  float* __restrict__ out) {
  const int64_t idx = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 6;   // wave-uniform
  const int lane = threadIdx.x & 63;
  if (idx >= bsz * n) return;
  const int64_t row = idx / n;
  const int q = n - 1 - (int)(idx % n);
  double s = 0.0, t = 0.0;
  for (int c = lane; c < nchunks; c += 64) {
    const float* p = part + (row * nchunks + c) * (n + 1);
    s += p[q];
    t += p[n];
  }
  s = wave_sum_d(s);
  t = wave_sum_d(t);
  if (lane == 0) out[idx] = (float)(t - 2.0 * s);
}

// Diagonal Pauli strings (x = 0): sum_j p_j (-1)^{popcount(j & z_t)}, up to
// EV_MAXT terms per launch.  part[(row*nchunks+chunk)*nt + t].
struct ZMasks {
  int nt;
  uint32_t z[EV_MAXT];
};

// Amplitude j = chunk_base + 512 k + 2 t + h (disjoint bits, as in
// k_ez_part), so parity(j & z) = parity(h & z) ^ parity(2 t & z) ^
// parity((chunk_base + 512 k) & z): the h part picks p0 + p1 or p0 - p1 per
// term, the uniform part is a sign per trip, the thread part one sign at the
// end -- one multiply-add per term per float4.
__global__ __launch_bounds__(EV_THREADS) void k_ediag_part(const float4* __restrict__ st, int n, int lg_chunk,
                                                           ZMasks zm, float* __restrict__ part) {
  __shared__ float red[EV_THREADS / 64];
  const int nchunks = 1 << (n - lg_chunk);
  const uint64_t row = blockIdx.x >> (n - lg_chunk);
  const uint64_t chunk = blockIdx.x & (nchunks - 1);
  const uint64_t first = (row << n) + (chunk << lg_chunk);
  const uint64_t npairs = (1ull << lg_chunk) >> 1;
  float acc[EV_MAXT];
#pragma unroll
  for (int t = 0; t < EV_MAXT; ++t) acc[t] = 0.f;
  for (uint64_t b = threadIdx.x, k = 0; b < npairs; b += EV_UNROLL * EV_THREADS, k += EV_UNROLL) {
    float4 v[EV_UNROLL];
#pragma unroll
    for (int u = 0; u < EV_UNROLL; ++u) {
      const uint64_t i = b + (uint64_t)u * EV_THREADS;
      v[u] = i < npairs ? st[(first >> 1) + i] : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int u = 0; u < EV_UNROLL; ++u) {
      const float p0 = v[u].x * v[u].x + v[u].y * v[u].y;
      const float p1 = v[u].z * v[u].z + v[u].w * v[u].w;
      const float ps = p0 + p1, pd = p0 - p1;
      const uint32_t jhi = (uint32_t)((chunk << lg_chunk) + 512ull * (k + u));   // wave-uniform
#pragma unroll
      for (int t = 0; t < EV_MAXT; ++t) {
        if (t < zm.nt) {
          const float sg = (__popc(jhi & zm.z[t]) & 1) ? -1.f : 1.f;
          acc[t] = fmaf(sg, (zm.z[t] & 1u) ? pd : ps, acc[t]);
        }
      }
    }
  }
  float* out = part + (uint64_t)blockIdx.x * zm.nt;
#pragma unroll
  for (int t = 0; t < EV_MAXT; ++t) {
    if (t < zm.nt) {
      const float tsg = (__popc((2u * threadIdx.x) & zm.z[t]) & 1) ? -1.f : 1.f;
      const float s = block_sum(tsg * acc[t], red);
      if (threadIdx.x == 0) out[t] = s;
    }
  }
}

// One off-diagonal string (x != 0): pairs (j, j ^ x) with j's top x-bit clear.
// Partial of sum_j s_j conj(psi_{j^x}) psi_j (complex; times i^{nY} on host).
__global__ __launch_bounds__(EV_THREADS) void k_ex_part(const float2* __restrict__ st, int n, int lg_chunk,
                                                        uint32_t x, uint32_t z, int top, float* __restrict__ part) {
  __shared__ float red[EV_THREADS / 64];
  // items: in-row indices with bit `top` clear; chunk over items
  const int lg_items = n - 1;
  const int lgc = lg_chunk > lg_items ? lg_items : lg_chunk;
  const int nchunks = 1 << (lg_items - lgc);
  const uint64_t row = blockIdx.x >> (lg_items - lgc);
  const uint64_t chunk = blockIdx.x & (nchunks - 1);
  const uint64_t cnt = 1ull << lgc;
  const float2* r = st + (row << n);
  float ar = 0.f, ai = 0.f;
  for (uint64_t i = threadIdx.x; i < cnt; i += blockDim.x) {
    const uint32_t it = (uint32_t)((chunk << lgc) + i);
    const uint32_t lo = it & ((1u << top) - 1u);
    const uint32_t j = ((it >> top) << (top + 1)) | lo;
    const uint32_t k = j ^ x;
    const float2 a = r[j], b = r[k];
    const float sj = (__popc(j & z) & 1) ? -1.f : 1.f;
    const float sk = (__popc(k & z) & 1) ? -1.f : 1.f;
    // sj * conj(b) * a + sk * conj(a) * b
    const float2 c1 = cmulc(b, a);
    const float2 c2 = cmulc(a, b);
    ar += sj * c1.x + sk * c2.x;
    ai += sj * c1.y + sk * c2.y;
  }
  float* out = part + (uint64_t)blockIdx.x * 2;
  const float sr = block_sum(ar, red);
  if (threadIdx.x == 0) out[0] = sr;
  const float si = block_sum(ai, red);
  if (threadIdx.x == 0) out[1] = si;
}

// Partials of Re <a_row|b_row>: block = (row, chunk of 2^lg amplitudes),
// part[row * nchunks + chunk].
__global__ __launch_bounds__(EV_THREADS) void k_rowdot_part(const float2* __restrict__ a,
                                                            const float2* __restrict__ b, int n, int lg_chunk,
                                                            float* __restrict__ part) {
  __shared__ float red[EV_THREADS / 64];
  const uint64_t row = blockIdx.x >> (n - lg_chunk);
  const uint64_t chunk = blockIdx.x & ((1u << (n - lg_chunk)) - 1u);
  const uint64_t base = (row << n) + (chunk << lg_chunk);
  float d = 0.f;
  for (uint64_t i = threadIdx.x; i < (1ull << lg_chunk); i += blockDim.x) {
    const float2 x = a[base + i], y = b[base + i];
    d = fmaf(x.x, y.x, fmaf(x.y, y.y, d));
  }
  const float t = block_sum(d, red);
  if (threadIdx.x == 0) part[blockIdx.x] = t;
}

// Sum per-chunk partials of one term: partial of (row, chunk) sits at
// part[(row * nchunks + chunk) * cstride] (complex: two floats re, im).
// out[row * ostride + ooff] = scale_re * Re(sum) - scale_im * Im(sum).
// One wavefront per row, its lanes striding over the chunks.
__global__ __launch_bounds__(256) void k_sum_chunks(const float* __restrict__ part, int nchunks, int cstride,
                                                    int is_complex, int64_t bsz, float scale_re, float scale_im,
                                                    float* __restrict__ out, int64_t ostride, int ooff) {
  const int64_t row = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 6;   // wave-uniform
  const int lane = threadIdx.x & 63;
  if (row >= bsz) return;
  double sr = 0.0, si = 0.0;
  for (int c = lane; c < nchunks; c += 64) {
    const float* p = part + (row * nchunks + c) * cstride;
    sr += p[0];
    if (is_complex) si += p[1];
  }
  sr = wave_sum_d(sr);
  si = wave_sum_d(si);
  if (lane == 0) out[row * ostride + ooff] = (float)(scale_re * sr - scale_im * si);
}

// out_j (+)= sum_t coef[row, t] * (-1)^{popcount((j^x_t) & z_t)} * psi_{j ^ x_t}
struct PTerms {
  int nt;
  uint32_t x[EV_MAXT];
  uint32_t z[EV_MAXT];
  int col[EV_MAXT];   // term column in coef
};

__global__ __launch_bounds__(EV_THREADS) void k_pauli_apply(float2* __restrict__ out, const float2* __restrict__ in,
                                                            int n, uint64_t total, PTerms pt,
                                                            const float2* __restrict__ coef, int64_t coef_stride,
                                                            int accumulate) {
  for (uint64_t g = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; g < total;
       g += (uint64_t)gridDim.x * blockDim.x) {
    const uint64_t row = g >> n;
    const uint32_t j = (uint32_t)(g & ((1ull << n) - 1ull));
    const float2* r = in + (row << n);
    const float2* cf = coef + row * coef_stride;
    float2 acc = accumulate ? out[g] : make_float2(0.f, 0.f);
    for (int t = 0; t < pt.nt; ++t) {
      const uint32_t k = j ^ pt.x[t];
      const float2 v = r[k];
      const float2 c = cf[pt.col[t]];
      const float2 cv = cmul(c, v);
      const bool neg = __popc(k & pt.z[t]) & 1;
      acc.x += neg ? -cv.x : cv.x;
      acc.y += neg ? -cv.y : cv.y;
    }
    out[g] = acc;
  }
}


// ---- terms grouped by a local bit set --------------------------------------
// A "local set" L of m <= 13 bit positions (the 4 lowest always among them, so
// that 16 lanes cover a whole 128-byte line) splits each row into groups of
// 2^m amplitudes that differ only in L.  Every term whose flip mask x lies
// inside L maps a group onto itself, so one pass that stages each group in LDS
// serves all of them: one pass over the state per set instead of one per term
// (expectations) or one uncached gather per term (their backward).
//
// A workgroup of NT threads holds a group, NR = 2^m / NT amplitudes per
// thread: local index l = tid | r << log2(NT), r the register slot.  The sign
// of a term splits over the three disjoint fields of the row index (group
// bits: wave-uniform; thread bits: one parity per lane; slot bits: known per
// r), and terms that share the flip mask, the phase mask of the slot bits and
// the parity of their Y count form one "entry": per lane a single factor, per
// amplitude one LDS read and two multiply-adds for all of them.
constexpr int PG_MAXM = 13;
constexpr int PG_MAXT = 96;     // terms per local set
constexpr int PG_LO = 4;        // lowest positions, local in every set

struct PGroup {
  int m, nnl, nt, ne, flips;  // local bits, non-local bits, terms, entries, whether any entry flips bits
  int lpos[PG_MAXM];          // local bit i -> bit position, ascending
  int nlpos[32];              // non-local positions, ascending
  uint32_t ex[PG_MAXT];       // entry: flip mask in local numbering
  uint32_t epm[PG_MAXT];      // entry: bit r = parity of slot r under the phase mask; bit 16: nY odd
  int ebeg[PG_MAXT + 1];      // entry e holds the terms [ebeg[e], ebeg[e + 1])
  uint32_t zt[PG_MAXT];       // term: phase mask of the thread bits; bit 16: parity of x & z
  uint32_t zg[PG_MAXT];       // term: phase mask, non-local part (bit positions)
  int col[PG_MAXT];           // term: column in coef / out
};

// Bit positions of the local indices of a set of M bits: of one, and of the
// slots' parts r * 2^LNT.  M and LNT are the kernel's own (threads, slots), so
// the positions come in a few wide scalar loads: looping over a set's m bits
// for every slot, a load waited for each time, took 9 us a launch (one string,
// 20 qubits bsz 3: 18.9 us, 8.2 this way; 13 qubits bsz 500 17.0 and 8.0).
template <int M>
__device__ __forceinline__ uint32_t pg_scatter(const PGroup& g, uint32_t l) {
  uint32_t o = l & ((1u << PG_LO) - 1u);
#pragma unroll
  for (int i = PG_LO; i < M; ++i) o |= ((l >> i) & 1u) << g.lpos[i];
  return o;
}

template <int LNT, int NR>
__device__ __forceinline__ void pg_slots(const PGroup& g, uint32_t (&rsc)[NR]) {
#pragma unroll
  for (int r = 0; r < NR; ++r) rsc[r] = r ? rsc[r & (r - 1)] | 1u << g.lpos[LNT + __builtin_ctz(r)] : 0u;
}

__device__ __forceinline__ uint32_t pg_group_offset(const PGroup& g, uint64_t rest) {
  uint32_t o = 0;
  for (int i = 0; i < g.nnl; ++i) o |= (uint32_t)((rest >> i) & 1ull) << g.nlpos[i];
  return o;
}

// A group's amplitudes (tsc: the lane's part of the in-group offset, rsc: the
// slots' parts, wave-uniform).  Buffer instructions: a scalar resource, the
// lane's byte offset and a scalar per slot, so no vector registers hold
// addresses; they reach positions up to 27.  BIG: pointers, for states with
// local positions above that.
template <int NR, bool BIG>
__device__ __forceinline__ void pg_load(const float2* __restrict__ p, uint32_t tsc, const uint32_t (&rsc)[NR],
                                        float2 (&v)[NR]) {
  if constexpr (BIG) {
    p += tsc;
    asm volatile("" : "+v"(p));
#pragma unroll
    for (int r = 0; r < NR; ++r) v[r] = p[rsc[r]];
  } else {
    const __amdgpu_buffer_rsrc_t b = __builtin_amdgcn_make_buffer_rsrc(const_cast<float2*>(p), (short)0, -1, 0x00020000);
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const auto q = __builtin_amdgcn_raw_buffer_load_b64(b, tsc * 8u, rsc[r] * 8u, 0);
      v[r] = make_float2(__uint_as_float(q[0]), __uint_as_float(q[1]));
    }
  }
}
template <int NR, bool BIG>
__device__ __forceinline__ void pg_store(float2* __restrict__ p, uint32_t tsc, const uint32_t (&rsc)[NR],
                                         const float2 (&v)[NR]) {
  if constexpr (BIG) {
    p += tsc;
    asm volatile("" : "+v"(p));
#pragma unroll
    for (int r = 0; r < NR; ++r) p[rsc[r]] = v[r];
  } else {
    typedef unsigned v2u __attribute__((__vector_size__(8)));
    const __amdgpu_buffer_rsrc_t b = __builtin_amdgcn_make_buffer_rsrc(p, (short)0, -1, 0x00020000);
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const v2u q = {__float_as_uint(v[r].x), __float_as_uint(v[r].y)};
      __builtin_amdgcn_raw_buffer_store_b64(q, b, tsc * 8u, rsc[r] * 8u, 0);
    }
  }
}

__device__ __forceinline__ float flip_sign(float v, uint32_t neg) {   // neg: 0 or 1
  return __uint_as_float(__float_as_uint(v) ^ (neg << 31));
}

// Bit 31 - (t & 31) of word t >> 5: the sign a term has for thread-field tid
// (its parity under the term's thread mask).  The same for every group, and
// walked by shifting left as the terms go by.  Three scalars, not an array:
// an array indexed by a word number goes to LDS, at an address for which every
// wavefront reads the dispatch packet in host memory (14 us a launch: one
// string, 20 qubits bsz 3: 27.2 us, 18.9 without; 8 qubits bsz 500: 17.5, 4.2).
static_assert(PG_MAXT == 96, "three words of signs");
struct LaneSigns {
  uint32_t a, b, c;
};

__device__ __forceinline__ uint32_t pg_lane_word(const PGroup& g, uint32_t tid, int first) {
  uint32_t w = 0;
  for (int t = first; t < g.nt && t < first + 32; ++t) w |= (__popc(tid & g.zt[t]) & 1u) << (31 - (t & 31));
  return w;
}

__device__ __forceinline__ LaneSigns pg_lane_signs(const PGroup& g, uint32_t tid) {
  return {pg_lane_word(g, tid, 0), pg_lane_word(g, tid, 32), pg_lane_word(g, tid, 64)};
}

__device__ __forceinline__ uint32_t pg_word(const LaneSigns& s, int k) {   // k wave-uniform
  return k == 0 ? s.a : k == 1 ? s.b : s.c;
}

// acc[r] += (+-c) v_r, or (+-i c) v_r with IM, the sign from bit r of pm with
// SIGN; v_r from LDS, at constant offsets where no slot bit is flipped (NEAR).
template <int NT, int NR, bool NEAR, bool SIGN, bool IM>
__device__ __forceinline__ void pg_fma(float2 (&acc)[NR], float c, const char* b8, uint32_t src, uint32_t pm) {
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const float2 v = NEAR ? *(const float2*)(b8 + src + (uint32_t)(r * NT * 8))
                          : *(const float2*)(b8 + (src ^ (uint32_t)(r * NT * 8)));
    const float cr = SIGN ? flip_sign(c, (pm >> r) & 1u) : c;
    if (IM) {
      acc[r].x = fmaf(-cr, v.y, acc[r].x);
      acc[r].y = fmaf(cr, v.x, acc[r].y);
    } else {
      acc[r].x = fmaf(cr, v.x, acc[r].x);
      acc[r].y = fmaf(cr, v.y, acc[r].y);
    }
  }
}

// sum_r (+-) of |a_r|^2 (FROM 0), or of Re conj(b_r) a_r / Im with IM, b_r from LDS.
template <int NT, int NR, int FROM, bool IM>
__device__ __forceinline__ float pg_dot(const float2 (&a)[NR], const char* b8, uint32_t src, uint32_t pm) {
  float F = 0.f;
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const float2 b = FROM == 0   ? a[r]
                     : FROM == 1 ? *(const float2*)(b8 + src + (uint32_t)(r * NT * 8))
                                 : *(const float2*)(b8 + (src ^ (uint32_t)(r * NT * 8)));
    const float d = IM ? fmaf(b.x, a[r].y, -b.y * a[r].x) : fmaf(b.x, a[r].x, b.y * a[r].y);
    F += flip_sign(d, (pm >> r) & 1u);
  }
  return F;
}

// Totals of 8 values over a wavefront, value l >> 3 in lane l (v_permlane
// swaps and DPP: no LDS traffic, 21 instructions).
__device__ __forceinline__ float pg_sum32(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float pg_sum16(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// v of the lane that DPP control C names
template <int C>
__device__ __forceinline__ double pg_dpp(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), C, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), C, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}
// The two steps that halve the values run in float32, the others in float64:
// a sum over all lanes of same-signed slots (a Z string outside the lanes'
// bits) is 64 times a lane's, and so would be the rounding of the last steps.
__device__ __forceinline__ double pg_sum8(const float (&v)[8], int lane) {
  float w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = pg_sum32(v[i], v[i + 4]);
  const double u0 = pg_sum16(w[0], w[2]), u1 = pg_sum16(w[1], w[3]);
  const double s0 = u0 + pg_dpp<0x128>(u0), s1 = u1 + pg_dpp<0x128>(u1);   // row_ror:8
  double z = (lane & 8) ? s1 : s0;
  z += pg_dpp<0x141>(z);   // row_half_mirror
  z += pg_dpp<0x4E>(z);    // quad_perm: l ^ 2
  z += pg_dpp<0xB1>(z);    // quad_perm: l ^ 1
  return z;
}

// out (+)= sum_t coef[row, col_t] (-1)^{popcount((j^x_t) & z_t)} psi_{j ^ x_t}
// for the terms of one local set; one workgroup walks gpw consecutive groups.
// A real or imaginary coefficient -- the usual case, i^{nY} times a real
// weight -- costs two FMA per amplitude and entry.  The next group's psi is
// loaded while this one's entries run.
//
// Bound by memory with few entries and by LDS reads (8 bytes per amplitude and
// entry) with many.  13-bit sets of 4 low and 9 high bits against 12-bit ones
// of 6 and 6, chosen by what they bring in: 22 qubits bsz 8 with 80 strings, 9
// passes of 209 us -> 4 of 213 us (12 bits with 4 low ones: 5 of 189 us; 14
// bits, one workgroup of 1024 threads per CU: 3 of 490 us); 24 qubits bsz 64
// with 48 strings, 3 passes of 6.7 -> 5.0 ms (203 us and 4.8 ms since a launch
// needs less beside its groups).  Held to 128 registers (four
// wavefronts per SIMD): with addresses in registers and the group's psi kept
// beside the next one's the compiler took 218, and a pass 330 us.
//
// dotpart != null: the workgroup also adds Re conj(psi_l) out_l over its
// groups (all in one row) and writes the sum to dotpart[blockIdx.x]; on the
// last pass over out this is the workgroup's part of Re <psi|out>.
template <int NT, int NR, bool BIG>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4))) void k_pauli_group_apply(float2* __restrict__ out, const float2* __restrict__ in,
                                                          int n, PGroup g, const float2* __restrict__ coef,
                                                          int64_t coef_stride, int accumulate, int64_t n_groups,
                                                          int64_t gpw, float* __restrict__ dotpart) {
  __shared__ float2 buf[NR * NT];
  __shared__ float2 cg[PG_MAXT];        // the group's coefficients, signs of the group bits folded in
  __shared__ double red[NT / 64];
  double dsum = 0.0;
  const int tid = threadIdx.x;
  constexpr int LNT = __builtin_ctz(NT);
  const uint32_t tsc = pg_scatter<LNT>(g, (uint32_t)tid);
  uint32_t rsc[NR];
  pg_slots<LNT>(g, rsc);
  // this thread's own term, whose coefficient it puts into cg, and its signs of all terms
  const uint32_t my_zg = tid < g.nt ? g.zg[tid] : 0u;
  const int my_col = tid < g.nt ? g.col[tid] : 0;
  const LaneSigns lw = pg_lane_signs(g, (uint32_t)tid | 0x10000u);
  const int64_t g0 = (int64_t)blockIdx.x * gpw;
  const int64_t g1 = g0 + gpw < n_groups ? g0 + gpw : n_groups;
  const uint64_t rmask = (1ull << g.nnl) - 1ull;
  const char* b8 = (const char*)buf;
  float2 a[NR];        // the coming group's psi: on its way while this group's entries run from LDS
  if (g0 < g1)
    pg_load<NR, BIG>(in + (((uint64_t)g0 >> g.nnl) << n) + pg_group_offset(g, (uint64_t)g0 & rmask), tsc, rsc, a);
  for (int64_t grp = g0; grp < g1; ++grp) {
    const uint64_t row = (uint64_t)grp >> g.nnl;
    const uint32_t goff = pg_group_offset(g, (uint64_t)grp & rmask);
    float2* rout = out + (row << n) + goff;
    float2 acc[NR];
    if (accumulate) {
      pg_load<NR, BIG>(rout, tsc, rsc, acc);
    } else {
#pragma unroll
      for (int r = 0; r < NR; ++r) acc[r] = make_float2(0.f, 0.f);
    }
    __syncthreads();   // the previous group's LDS reads are done
#pragma unroll
    for (int r = 0; r < NR; ++r) buf[tid + r * NT] = a[r];
    if (tid < g.nt) {
      const float2 c = coef[row * coef_stride + my_col];
      const uint32_t neg = __popc(goff & my_zg) & 1u;
      cg[tid] = make_float2(flip_sign(c.x, neg), flip_sign(c.y, neg));
    }
    __syncthreads();
    if (grp + 1 < g1) {
      const uint64_t gn = (uint64_t)grp + 1;
      pg_load<NR, BIG>(in + ((gn >> g.nnl) << n) + pg_group_offset(g, gn & rmask), tsc, rsc, a);
    }
    uint32_t w = lw.a;
    uint32_t x = g.ex[0], pm = g.epm[0];
    int t = 0, tend = g.ebeg[1];
    for (int e = 0; e < g.ne; ++e) {
      const int en = e + 1 < g.ne ? e + 1 : e;           // the next entry's words, ahead of their use
      const uint32_t xn = g.ex[en], pmn = g.epm[en];
      const int tn = g.ebeg[en + 1];
      // this lane's factor: the sum of the entry's coefficients under the
      // signs of the group and thread bits of the source j ^ x
      float2 c = make_float2(0.f, 0.f);
      for (; t < tend; ++t) {
        const float2 ct = cg[t];
        if ((t & 31) == 0 && t) w = pg_word(lw, t >> 5);
        const uint32_t sb = w & 0x80000000u;
        w <<= 1;
        c.x += __uint_as_float(__float_as_uint(ct.x) ^ sb);
        c.y += __uint_as_float(__float_as_uint(ct.y) ^ sb);
      }
      const uint32_t src = ((uint32_t)tid ^ x) * 8u;      // slot r reads local index (tid | r * NT) ^ x
      const bool near = x < (uint32_t)NT;                 // slot bits not flipped: constant offsets
      if (c.y == 0.f) {                                   // real
        if (!near) pg_fma<NT, NR, false, true, false>(acc, c.x, b8, src, pm);
        else if (pm & 0xffffu) pg_fma<NT, NR, true, true, false>(acc, c.x, b8, src, pm);
        else pg_fma<NT, NR, true, false, false>(acc, c.x, b8, src, pm);
      } else if (c.x == 0.f) {                            // imaginary
        if (near) pg_fma<NT, NR, true, true, true>(acc, c.y, b8, src, pm);
        else pg_fma<NT, NR, false, true, true>(acc, c.y, b8, src, pm);
      } else {
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          const float2 v = *(const float2*)(b8 + (src ^ (uint32_t)(r * NT * 8)));
          const uint32_t neg = (pm >> r) & 1u;
          acc[r] = cfma(make_float2(flip_sign(c.x, neg), flip_sign(c.y, neg)), v, acc[r]);
        }
      }
      x = xn;
      pm = pmn;
      tend = tn;
    }
    pg_store<NR, BIG>(rout, tsc, rsc, acc);
    if (dotpart) {
      float d = 0.f;
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        const float2 v = buf[tid + r * NT];
        d = fmaf(v.x, acc[r].x, fmaf(v.y, acc[r].y, d));
      }
      dsum += d;
    }
  }
  if (dotpart) {
    const double t = block_sum_d(dsum, red);
    if (tid == 0) dotpart[blockIdx.x] = (float)t;
  }
}

// Partials of the terms of one local set over the gpw groups of one
// workgroup (all in one row).  With a = psi_j, b = psi_{j^x}:
// <P> = Re(i^{nY} S), S = sum_j (-1)^{popcount(j & z)} conj(b) a, so only
// Re S (nY even) or Im S (nY odd) is accumulated.  Per entry one sum over the
// slots; per term the lane's sign of it, eight terms reduced over the
// wavefront at a time into the wave's row of gacc, in float64: a wave's sum
// runs over many groups, and in float32 its rounding was the largest error of
// the value (24 qubits bsz 4: 4e-6 of the values' norm, now 2e-7).  Bound by the entries' LDS
// reads and multiply-adds: 24 qubits bsz 4 with 60 strings, 5 passes of 198 us
// and one launch for a pass's sums (16 terms at most per set and a launch per
// term before).
// part[(blockIdx.x * nt + t) * 2] = the partial of term t, and what float32
// leaves off it.
// ONE: one group per workgroup (gpw 1), so nothing is loaded ahead (22 qubits
// bsz 1 with 60 strings 77 -> 70 us, 20 qubits bsz 4 with 40 45 -> 42 us).
template <int NT, int NR, bool BIG, bool ONE>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4))) void k_pauli_group_expval(const float2* __restrict__ in, int n, PGroup g,
                                                           int64_t gpw, float* __restrict__ part) {
  __shared__ float2 buf[NR * NT];
  __shared__ double gacc[NT / 64][PG_MAXT];
  __shared__ uint32_t zgs[PG_MAXT];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  double* wacc = gacc[tid >> 6];
  constexpr int LNT = __builtin_ctz(NT);
  const uint32_t tsc = pg_scatter<LNT>(g, (uint32_t)tid);
  uint32_t rsc[NR];
  pg_slots<LNT>(g, rsc);
  for (int t = tid; t < (NT / 64) * PG_MAXT; t += NT) gacc[0][t] = 0.0;
  if (tid < g.nt) zgs[tid] = g.zg[tid];
  const LaneSigns lw = pg_lane_signs(g, (uint32_t)tid);
  const int64_t g0 = (int64_t)blockIdx.x * gpw;
  const uint64_t rmask = (1ull << g.nnl) - 1ull;
  const char* b8 = (const char*)buf;
  float2 a[NR];
  pg_load<NR, BIG>(in + (((uint64_t)g0 >> g.nnl) << n) + pg_group_offset(g, (uint64_t)g0 & rmask), tsc, rsc, a);
  for (int64_t grp = g0; grp < g0 + gpw; ++grp) {
    const uint32_t goff = pg_group_offset(g, (uint64_t)grp & rmask);
    __syncthreads();     // the previous group's LDS reads (and the setting up above) are done
    if (g.flips) {
#pragma unroll
      for (int r = 0; r < NR; ++r) buf[tid + r * NT] = a[r];
      __syncthreads();
    }
    float2 an[NR];
    if constexpr (!ONE) {   // the last group once more at the end: behind a branch 24 qubits bsz 4 took 671 instead of 655 us
      const uint64_t gn = (uint64_t)(grp + 1 < g0 + gpw ? grp + 1 : grp);
      pg_load<NR, BIG>(in + ((gn >> g.nnl) << n) + pg_group_offset(g, gn & rmask), tsc, rsc, an);
    }
    int e = 0, tnext = 0;
    float F = 0.f;
    uint32_t x = g.ex[0], pm = g.epm[0], w = 0;
    for (int t0 = 0; t0 < g.nt; t0 += 8) {
      float v[8];
      if ((t0 & 31) == 0) w = pg_word(lw, t0 >> 5);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int t = t0 + k;
        if (t == tnext && t < g.nt) {      // the next entry's sum over the slots
          const uint32_t src = ((uint32_t)tid ^ x) * 8u;
          if (x == 0u) F = pg_dot<NT, NR, 0, false>(a, b8, src, pm);
          else if (pm >> 16) F = x < (uint32_t)NT ? pg_dot<NT, NR, 1, true>(a, b8, src, pm)
                                                  : pg_dot<NT, NR, 2, true>(a, b8, src, pm);
          else F = x < (uint32_t)NT ? pg_dot<NT, NR, 1, false>(a, b8, src, pm)
                                    : pg_dot<NT, NR, 2, false>(a, b8, src, pm);
          ++e;
          tnext = g.ebeg[e];
          const int en = e < g.ne ? e : e - 1;
          x = g.ex[en];
          pm = g.epm[en];
        }
        v[k] = __uint_as_float(__float_as_uint(F) ^ (w & 0x80000000u));
        w <<= 1;
      }
      const double c = pg_sum8(v, lane);
      const int t = t0 + (lane >> 3);
      if ((lane & 7) == 0 && t < g.nt) wacc[t] += (__popc(goff & zgs[t]) & 1u) ? -c : c;
    }
    if constexpr (!ONE) {
#pragma unroll
      for (int r = 0; r < NR; ++r) a[r] = an[r];
    }
  }
  __syncthreads();
  for (int t = tid; t < g.nt; t += NT) {
    double s = 0.0;
    for (int w = 0; w < NT / 64; ++w) s += gacc[w][t];
    float* o = part + ((uint64_t)blockIdx.x * g.nt + t) * 2;
    const float f = (float)s;
    o[0] = f;
    o[1] = (float)(s - (double)f);
  }
}

// out[row * ostride + col[t]] = the sum of the W floats at
// part[((row * nchunks + c) * nt + t) * W] over the chunks, in float64, negated where bit t of neg is set; one
// wavefront per (row, t).
struct TermSums {
  int nt;
  int col[PG_MAXT];
  uint32_t neg[(PG_MAXT + 31) / 32];
};

template <int W>
__global__ __launch_bounds__(256) void k_sum_terms(const float* __restrict__ part, int nchunks, int64_t bsz,
                                                   TermSums ts, float* __restrict__ out, int64_t ostride) {
  const int64_t i = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 6;   // wave-uniform
  const int lane = threadIdx.x & 63;
  if (i >= bsz * ts.nt) return;
  const int64_t row = i / ts.nt;
  const int t = (int)(i - row * ts.nt);
  double s = 0.0;
  for (int c = lane; c < nchunks; c += 64) {
    const float* p = part + ((row * nchunks + c) * ts.nt + t) * W;
#pragma unroll
    for (int k = 0; k < W; ++k) s += p[k];
  }
  s = wave_sum_d(s);
  if (lane == 0) out[row * ostride + ts.col[t]] = (float)((ts.neg[t >> 5] >> (t & 31)) & 1u ? -s : s);
}

// Workgroups per row of the grouped-term launches: a power of two dividing
// the 2^nnl groups of a row, about as many over the batch as are resident at
// once (4 per CU of 256 threads, 2 of 512).
static int64_t pg_wg_per_row(int64_t bsz, int nnl, int m) {
  const int64_t per_row = 1ll << nnl;
  int64_t wpr = (int64_t)num_cu() * (m == 13 ? 2 : 4) / bsz;
  if (wpr < 1) wpr = 1;
  if (wpr > per_row) wpr = per_row;
  while (per_row % wpr) --wpr;        // per_row is a power of two: wpr becomes one too
  return wpr;
}

// f with the threads and slots of a set's width -- m = 8 + log2(NR) with 256
// threads up to 12 bits, 512 threads for 13 -- and whether buffer
// instructions do not reach its positions.  (Below 13 bits a set is the whole
// row of m wires.)
template <class F>
static int pg_dispatch(const PGroup& g, F f) {
  using std::integral_constant;
  const integral_constant<int, 256> t256;
  const integral_constant<int, 512> t512;
  const integral_constant<int, 16> n16;
  const std::false_type buf;
  const std::true_type big;
  switch (g.m) {
    case 8: return f(t256, integral_constant<int, 1>(), buf);
    case 9: return f(t256, integral_constant<int, 2>(), buf);
    case 10: return f(t256, integral_constant<int, 4>(), buf);
    case 11: return f(t256, integral_constant<int, 8>(), buf);
    case 12: return f(t256, n16, buf);
    default: return g.lpos[g.m - 1] > 27 ? f(t512, n16, big) : f(t512, n16, buf);
  }
}

// One pass over the terms of a local set; every workgroup stays in one row
// (wpr workgroups per row), so with dotpart each writes one row partial:
// dotpart[row * wpr + k].
static int pg_apply_launch(hipStream_t s, float2* out, const float2* in, int n, const PGroup& g, const float2* coef,
                           int64_t coef_stride, int acc, int64_t bsz, float* dotpart) {
  const int64_t wpr = pg_wg_per_row(bsz, g.nnl, g.m);
  const int64_t gpw = (1ll << g.nnl) / wpr;
  const int64_t grid = bsz * wpr;
  if (grid > 0x7fffffffll) { set_error("tqsv_pauli_apply: batch too large"); return E_LIMIT; }
  return pg_dispatch(g, [&](auto nt, auto nr, auto big) {
    k_pauli_group_apply<nt(), nr(), big()><<<(unsigned)grid, nt(), 0, s>>>(out, in, n, g, coef, coef_stride, acc,
                                                                    bsz << g.nnl, gpw, dotpart);
    return check_launch("tqsv_pauli_apply/group");
  });
}

static int pg_expval_launch(hipStream_t s, const float2* in, int n, const PGroup& g, int64_t bsz, void* ws,
                            int64_t ws_bytes, int64_t& wpr) {
  const int64_t per_row = 1ll << g.nnl;
  wpr = pg_wg_per_row(bsz, g.nnl, g.m);
  const int64_t gpw = per_row / wpr;
  const int64_t grid = bsz * wpr;
  if (grid > 0x7fffffffll || ws_bytes < grid * 2 * g.nt * (int64_t)sizeof(float)) return 1;   // caller falls back
  return pg_dispatch(g, [&](auto nt, auto nr, auto big) {
    auto launch = [&](auto one) {
      k_pauli_group_expval<nt(), nr(), big(), one()><<<(unsigned)grid, nt(), 0, s>>>(in, n, g, gpw, (float*)ws);
    };
    if constexpr (decltype(nt)::value == 512) {      // narrower sets are whole rows: one group
      if (gpw > 1) launch(std::false_type());
      else launch(std::true_type());
    } else {
      launch(std::true_type());
    }
    return check_launch("tqsv_expval_pauli/group");
  });
}

// Host side: the local sets of a list of terms.  Each set keeps the lowest
// PG_LO bits plus up to m - PG_LO higher bits that its terms flip; it is filled
// up to m bits with the lowest unused positions (n >= 8, so m >= 8).  Terms
// that flip more than m - PG_LO bits above PG_LO are left for the per-term
// kernels.  A set starts from the flip mask with the most bits and grows:
//   * with up to PG_EXACT different masks left, by the mask that brings in the
//     most terms per added bit (masks x masks per step);
//   * with more, by the bit that the most masks still lack, each weighted by
//     8^-(bits it lacks) (masks per step).  Trying every mask for all of 8000
//     strings of up to 4 letters on 22 wires took 0.32 s and left 90 sets,
//     this way takes 7 ms and leaves 91; 1000 strings 3.1 and 0.5 ms, 18 sets.
constexpr size_t PG_EXACT = 128;

struct PGPlan {
  std::vector<PGroup> sets;
  std::vector<int> rest;          // terms in no set, ascending
};

struct PGMask {
  uint32_t bits;     // high bits flipped
  int terms;         // terms of the list that flip them
};

// The high bits of the next set.
static uint32_t pg_grow(const std::vector<PGMask>& masks, int room) {
  uint32_t H = 0;
  for (const PGMask& k : masks)
    if (__builtin_popcount(k.bits) > __builtin_popcount(H)) H = k.bits;
  for (;;) {
    uint32_t best = 0;
    if (masks.size() <= PG_EXACT) {
      int best_gain = 0, best_bits = 1;
      for (const PGMask& h : masks) {
        if (!(h.bits & ~H) || __builtin_popcount(H | h.bits) > room) continue;
        const int bits = __builtin_popcount(h.bits & ~H);
        int gain = 0;
        for (const PGMask& k : masks)
          if ((k.bits & ~H) && !(k.bits & ~(H | h.bits))) gain += k.terms;
        if (gain * best_bits > best_gain * bits) { best = h.bits; best_gain = gain; best_bits = bits; }
      }
    } else {
      float weight[32] = {};
      for (const PGMask& k : masks) {
        const uint32_t lacks = k.bits & ~H;
        if (!lacks || __builtin_popcount(H | k.bits) > room) continue;
        const float w = (float)k.terms / (float)(1ull << 3 * __builtin_popcount(lacks));   // at most 9 bits
        for (uint32_t b = lacks; b; b &= b - 1) weight[__builtin_ctz(b)] += w;
      }
      int top = 0;
      for (int b = 1; b < 32; ++b)
        if (weight[b] > weight[top]) top = b;
      if (weight[top] > 0.f) best = 1u << top;
    }
    if (!best) return H;
    H |= best;
  }
}

static PGPlan pg_build(int n, int m, const std::vector<uint32_t>& x, const std::vector<uint32_t>& z) {
  PGPlan P;
  const int nterms = (int)x.size();
  const int room = m - PG_LO;
  const int tb = m == 13 ? 9 : 8;        // thread bits
  const uint32_t hi_mask = ~((1u << PG_LO) - 1u);
  std::vector<int> todo;
  for (int t = 0; t < nterms; ++t) {
    if (__builtin_popcount(x[t] & hi_mask) <= room) todo.push_back(t);
    else P.rest.push_back(t);
  }
  // the different masks, in the order of their first terms
  std::vector<PGMask> masks;
  std::vector<int> mask_of(nterms);
  {
    std::vector<int> by(todo);
    std::stable_sort(by.begin(), by.end(), [&](int p, int q) { return (x[p] & hi_mask) < (x[q] & hi_mask); });
    std::vector<int> first(nterms, -1);        // first term of the same mask
    for (size_t i = 0; i < by.size(); ++i)
      first[by[i]] = i && (x[by[i]] & hi_mask) == (x[by[i - 1]] & hi_mask) ? first[by[i - 1]] : by[i];
    for (int t : todo) {
      if (first[t] == t) {
        mask_of[t] = (int)masks.size();
        masks.push_back({x[t] & hi_mask, 0});
      } else {
        mask_of[t] = mask_of[first[t]];
      }
      ++masks[mask_of[t]].terms;
    }
  }
  while (!todo.empty()) {
    const uint32_t H = pg_grow(masks, room);
    std::vector<int> members, left;
    for (int t : todo) {
      if (!(x[t] & hi_mask & ~H) && (int)members.size() < PG_MAXT) {
        members.push_back(t);
        --masks[mask_of[t]].terms;
      } else {
        left.push_back(t);
      }
    }
    {   // the masks that still have terms
      std::vector<int> at(masks.size());
      size_t kept = 0;
      for (size_t i = 0; i < masks.size(); ++i) {
        at[i] = (int)kept;
        if (masks[i].terms) masks[kept++] = masks[i];
      }
      masks.resize(kept);
      for (int t : left) mask_of[t] = at[mask_of[t]];
    }
    PGroup g{};
    g.m = m;
    uint32_t L = ((1u << PG_LO) - 1u) | H;
    for (int b = PG_LO; b < n && __builtin_popcount(L) < m; ++b) L |= 1u << b;
    int nl = 0;
    for (int b = 0; b < n; ++b) {
      if ((L >> b) & 1u) g.lpos[nl++] = b;
      else g.nlpos[g.nnl++] = b;
    }
    auto to_local = [&](uint32_t mask) {
      uint32_t v = 0;
      for (int i = 0; i < m; ++i) v |= ((mask >> g.lpos[i]) & 1u) << i;
      return v;
    };
    struct Term { uint32_t x, zh, odd; int t; };
    std::vector<Term> ts;
    for (int t : members)
      ts.push_back({to_local(x[t]), to_local(z[t]) >> tb, (uint32_t)__builtin_popcount(x[t] & z[t]) & 1u, t});
    std::stable_sort(ts.begin(), ts.end(), [](const Term& p, const Term& q) {
      return p.x != q.x ? p.x < q.x : p.zh != q.zh ? p.zh < q.zh : p.odd < q.odd;
    });
    g.nt = (int)ts.size();
    for (int q = 0; q < g.nt; ++q) {
      const Term& T = ts[q];
      if (q == 0 || T.x != ts[q - 1].x || T.zh != ts[q - 1].zh || T.odd != ts[q - 1].odd) {
        g.ex[g.ne] = T.x;
        for (uint32_t r = 0; r < 16; ++r) g.epm[g.ne] |= ((uint32_t)__builtin_popcount(r & T.zh) & 1u) << r;
        g.epm[g.ne] |= T.odd << 16;
        g.ebeg[g.ne++] = q;
      }
      const uint32_t zl = to_local(z[T.t]);
      g.flips |= T.x != 0;
      g.zt[q] = (zl & ((1u << tb) - 1u)) | ((uint32_t)__builtin_popcount(x[T.t] & z[T.t]) & 1u) << 16;
      g.zg[q] = z[T.t] & ~L;
      g.col[q] = T.t;
    }
    g.ebeg[g.ne] = g.nt;
    P.sets.push_back(g);
    todo.swap(left);
  }
  return P;
}

// The sets of a list of terms, kept for the next call with the same list (a
// loop over one observable): planning 80 terms takes about 0.05 ms.  At most
// 64 lists; holds masks only, nothing of a state or a stream.
static std::shared_ptr<const PGPlan> pg_plan(int n, int nterms, const uint64_t* xmask, const uint64_t* zmask) {
  struct Entry {
    int n;
    std::vector<uint32_t> x, z;
    std::shared_ptr<const PGPlan> plan;
  };
  static std::mutex mu;
  static std::vector<Entry> kept;
  static size_t next = 0;
  std::vector<uint32_t> x(xmask, xmask + nterms), z(zmask, zmask + nterms);
  {
    std::lock_guard<std::mutex> lock(mu);
    for (const Entry& e : kept)
      if (e.n == n && e.x == x && e.z == z) return e.plan;
  }
  auto plan = std::make_shared<const PGPlan>(pg_build(n, n < PG_MAXM ? n : PG_MAXM, x, z));
  std::lock_guard<std::mutex> lock(mu);
  Entry e{n, std::move(x), std::move(z), plan};
  if (kept.size() < 64) kept.push_back(std::move(e));
  else kept[next++ % 64] = std::move(e);
  return plan;
}

}  // namespace tqsv

using namespace tqsv;

static unsigned grid_cap(uint64_t work) {
  uint64_t b = (work + EV_THREADS - 1) / EV_THREADS;
  uint64_t cap = (uint64_t)num_cu() * 16;
  if (b > cap) b = cap;
  return b ? (unsigned)b : 1u;
}

// A launch takes 2^32 threads at most (more are cut off without an error), and
// the kernels here use up to 512 a row and 64 a (row, term): the entry points
// go over larger batches in slabs of rows.  2^19 rows of 96 terms are 2^31.6.
constexpr int64_t ROW_SLAB = 1ll << 19;

// f(first row, rows) for each slab until one fails
template <class F>
static int row_slabs(int64_t bsz, F f) {
  for (int64_t r0 = 0; r0 < bsz; r0 += ROW_SLAB) {
    const int rc = f(r0, bsz - r0 < ROW_SLAB ? bsz - r0 : ROW_SLAB);
    if (rc) return rc;
  }
  return OK;
}

// Bytes of float workspace the expectation entry points need.
// ---- allocation-free <Z_w> -------------------------------------------------
// tqsv_expval_z_all_noalloc runs the same two kernels as tqsv_expval_z_all,
// with the chunk partials in a fixed device array instead of a caller
// workspace, for callers that cannot allocate device memory.  Each GPU holds
// its own copy of the array until the process ends.  Every partial that
// k_ez_final reads is written by k_ez_part in the same call, so nothing needs
// clearing between calls.  Calls that overlap on one GPU share the array and
// race; callers serialise them (one stream, or their own ordering).
constexpr int64_t NOALLOC_SCRATCH_FLOATS = 1ll << 20;   // 4 MiB
constexpr int NOALLOC_MAX_DEVICES = 64;
static __device__ __align__(256) float scratch[NOALLOC_SCRATCH_FLOATS];
static std::mutex g_scratch_mu;
static float* g_scratch_dev[NOALLOC_MAX_DEVICES];      // device address of `scratch`, per device

// Device address of this GPU's `scratch`, looked up once per device (with
// that device current); host code uses only this address, never the symbol.
static int scratch_address(float** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= NOALLOC_MAX_DEVICES) {
    set_error("tqsv_expval_z_all_noalloc: no current HIP device (or device index >= %d)", NOALLOC_MAX_DEVICES);
    return E_LAUNCH;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_dev[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      set_error("tqsv_expval_z_all_noalloc: hipGetSymbolAddress failed on device %d: %s", dev, hipGetErrorString(e));
      return E_LAUNCH;
    }
    g_scratch_dev[dev] = (float*)p;
  }
  *out = g_scratch_dev[dev];
  return OK;
}

TQSV_API int64_t tqsv_expval_workspace_bytes(int64_t bsz, int n, int nterms) {
  if (bsz < 1 || n < 1 || n > 32) return -1;
  const int lg = ev_chunk_log2(bsz, n);
  const int64_t blocks = bsz << (n - lg);
  int64_t per = (int64_t)(n + 1);
  if (nterms * 2 > per) per = nterms * 2;
  if (EV_MAXT * 2 > per) per = EV_MAXT * 2;
  return blocks * per * (int64_t)sizeof(float) * 2;
}

// <Z_w> for all wires w: out[bsz, n] (wire order as in the reference: out[:, w]).
TQSV_API int tqsv_expval_z_all(hipStream_t s, const void* state, int64_t bsz, int n, float* out, void* workspace,
                               int64_t ws_bytes) {
  if (!state || !out || !workspace) { set_error("tqsv_expval_z_all: null pointer"); return E_ARG; }
  if (bsz < 1 || n < 1 || n > EV_MAXQ) { set_error("tqsv_expval_z_all: need 1 <= n <= %d", EV_MAXQ); return E_ARG; }
  if ((uintptr_t)state & 15) { set_error("tqsv_expval_z_all: state must be 16-byte aligned"); return E_ARG; }
  const int lg = ev_chunk_log2(bsz, n);
  const int64_t blocks = bsz << (n - lg);
  if (ws_bytes < blocks * (n + 1) * (int64_t)sizeof(float)) { set_error("tqsv_expval_z_all: workspace too small"); return E_ARG; }
  return row_slabs(bsz, [&](int64_t r0, int64_t rows) {
    const int lg = ev_chunk_log2(rows, n);
    k_ez_part<<<(unsigned)(rows << (n - lg)), EV_THREADS, 0, s>>>((const float4*)((const float2*)state + (r0 << n)), n, lg,
                                                                  (float*)workspace);
    const int rc = check_launch("tqsv_expval_z_all/part");
    if (rc) return rc;
    k_ez_final<<<sum_grid(rows * n), 256, 0, s>>>((const float*)workspace, n, 1 << (n - lg), rows, out + r0 * n);
    return check_launch("tqsv_expval_z_all/final");
  });
}

// <Z_w> for every wire, as tqsv_expval_z_all, with no workspace argument and
// no allocation: the partials go to this GPU's fixed scratch array
// (NOALLOC_SCRATCH_FLOATS floats; larger shapes are rejected).
TQSV_API int tqsv_expval_z_all_noalloc(hipStream_t s, const void* state, int64_t bsz, int n, float* out) {
  if (!state || !out) { set_error("tqsv_expval_z_all_noalloc: null pointer"); return E_ARG; }
  if (bsz < 1 || n < 1 || n > EV_MAXQ) { set_error("tqsv_expval_z_all_noalloc: need 1 <= n <= %d", EV_MAXQ); return E_ARG; }
  if ((uintptr_t)state & 15) { set_error("tqsv_expval_z_all_noalloc: state must be 16-byte aligned"); return E_ARG; }
  const int lg = ev_chunk_log2(bsz, n);
  const int64_t blocks = bsz << (n - lg);
  const int64_t need = blocks * (n + 1);
  if (need > NOALLOC_SCRATCH_FLOATS) {
    set_error("tqsv_expval_z_all_noalloc: bsz %lld x %d qubits needs %lld floats of scratch, the maximum is %lld "
              "(use tqsv_expval_z_all with a workspace)", (long long)bsz, n, (long long)need,
              (long long)NOALLOC_SCRATCH_FLOATS);
    return E_LIMIT;
  }
  float* ws = nullptr;
  int rc = scratch_address(&ws);
  if (rc) return rc;
  k_ez_part<<<(unsigned)blocks, EV_THREADS, 0, s>>>((const float4*)state, n, lg, ws);
  if ((rc = check_launch("tqsv_expval_z_all_noalloc/part"))) return rc;
  k_ez_final<<<sum_grid(bsz * n), 256, 0, s>>>(ws, n, 1 << (n - lg), bsz, out);
  return check_launch("tqsv_expval_z_all_noalloc/final");
}

// The terms' values of one slab of rows.
static int expval_pauli_rows(hipStream_t s, const void* state, int64_t bsz, int n, int nterms, const uint64_t* xmask,
                             const uint64_t* zmask, float* out, int64_t out_stride, void* workspace,
                             int64_t ws_bytes) {
  const int lg = ev_chunk_log2(bsz, n);
  const int64_t nchunks = 1ll << (n - lg);
  const int64_t blocks = bsz * nchunks;
  bool flips = false;
  for (int t = 0; t < nterms; ++t) flips |= xmask[t] != 0;
  // terms grouped by local set, one pass per set; what fits no set, and terms
  // that all are diagonal and few, go on below
  std::vector<char> done(nterms, 0);
  if (n >= 8 && (flips || nterms > EV_MAXT)) {
    const std::shared_ptr<const PGPlan> P = pg_plan(n, nterms, xmask, zmask);
    for (const PGroup& g : P->sets) {
      int64_t wpr = 0;
      int rc = pg_expval_launch(s, (const float2*)state, n, g, bsz, workspace, ws_bytes, wpr);
      if (rc == 1) continue;   // workspace too small: these terms take the per-term path
      if (rc) return rc;
      TermSums ts{};
      ts.nt = g.nt;
      for (int q = 0; q < g.nt; ++q) {
        // partial = Re S (nY even) or Im S (nY odd); <P> = Re(i^{nY} S)
        const int t = g.col[q];
        const int ny = __builtin_popcountll(xmask[t] & zmask[t]);
        ts.col[q] = t;
        if ((ny & 3) == 1 || (ny & 3) == 2) ts.neg[q >> 5] |= 1u << (q & 31);
        done[t] = 1;
      }
      k_sum_terms<2><<<sum_grid(bsz * g.nt), 256, 0, s>>>((const float*)workspace, (int)wpr, bsz, ts, out, out_stride);
      if ((rc = check_launch("tqsv_expval_pauli/groupsum"))) return rc;
    }
  }
  // diagonal terms, EV_MAXT at a time
  for (int t = 0; t < nterms;) {
    ZMasks zm;
    TermSums ts{};
    for (zm.nt = 0; t < nterms && zm.nt < EV_MAXT; ++t) {
      if (xmask[t] || done[t]) continue;
      zm.z[zm.nt] = (uint32_t)zmask[t];
      ts.col[zm.nt++] = t;
    }
    if (zm.nt == 0) break;
    if (ws_bytes < blocks * zm.nt * (int64_t)sizeof(float)) { set_error("tqsv_expval_pauli: workspace too small"); return E_ARG; }
    k_ediag_part<<<(unsigned)blocks, EV_THREADS, 0, s>>>((const float4*)state, n, lg, zm, (float*)workspace);
    int rc = check_launch("tqsv_expval_pauli/diag");
    if (rc) return rc;
    ts.nt = zm.nt;
    k_sum_terms<1><<<sum_grid(bsz * ts.nt), 256, 0, s>>>((const float*)workspace, (int)nchunks, bsz, ts, out, out_stride);
    if ((rc = check_launch("tqsv_expval_pauli/sum"))) return rc;
  }
  for (int t = 0; t < nterms; ++t) {
    if (xmask[t] == 0 || done[t]) continue;
    const uint32_t x = (uint32_t)xmask[t], z = (uint32_t)zmask[t];
    const int top = 31 - __builtin_clz(x);
    const int ny = __builtin_popcount(x & z);
    // i^{ny}: (re, im) scale
    float sre = 0.f, sim = 0.f;
    switch (ny & 3) { case 0: sre = 1.f; break; case 1: sim = 1.f; break; case 2: sre = -1.f; break; default: sim = -1.f; }
    const int lgi = n - 1;
    const int lgc = lg > lgi ? lgi : lg;
    const int64_t nch = 1ll << (lgi - lgc);
    const int64_t blk = bsz * nch;
    if (ws_bytes < blk * 2 * (int64_t)sizeof(float)) { set_error("tqsv_expval_pauli: workspace too small"); return E_ARG; }
    k_ex_part<<<(unsigned)blk, EV_THREADS, 0, s>>>((const float2*)state, n, lg, x, z, top, (float*)workspace);
    int rc = check_launch("tqsv_expval_pauli/x");
    if (rc) return rc;
    // Re(i^ny * S) = sre*Re(S) - sim*Im(S)
    k_sum_chunks<<<sum_grid(bsz), 256, 0, s>>>((const float*)workspace, (int)nch, 2, 1, bsz, sre,
                                                               sim, out, out_stride, t);
    if ((rc = check_launch("tqsv_expval_pauli/xsum"))) return rc;
  }
  return OK;
}

// Re <psi|P_t|psi> for nterms Pauli strings given by bit masks (in-row bit
// positions; host arrays).  out[row * out_stride + t].
TQSV_API int tqsv_expval_pauli(hipStream_t s, const void* state, int64_t bsz, int n, int nterms,
                               const uint64_t* xmask, const uint64_t* zmask, float* out, int64_t out_stride,
                               void* workspace, int64_t ws_bytes) {
  if (!state || !out || !workspace || (nterms > 0 && (!xmask || !zmask))) {
    set_error("tqsv_expval_pauli: null pointer");
    return E_ARG;
  }
  if (bsz < 1 || n < 1 || n > 32 || nterms < 0) { set_error("tqsv_expval_pauli: need 1 <= n <= 32"); return E_ARG; }
  if ((uintptr_t)state & 15) { set_error("tqsv_expval_pauli: state must be 16-byte aligned"); return E_ARG; }
  for (int t = 0; t < nterms; ++t)
    if ((xmask[t] | zmask[t]) >> n) { set_error("tqsv_expval_pauli: mask beyond n bits"); return E_ARG; }
  return row_slabs(bsz, [&](int64_t r0, int64_t rows) {
    return expval_pauli_rows(s, (const float2*)state + (r0 << n), rows, n, nterms, xmask, zmask, out + r0 * out_stride,
                             out_stride, workspace, ws_bytes);
  });
}

// out (+)= sum_t coef[row * coef_stride + t] P_t psi.  dotpart != null: the
// last pass also leaves the row partials of Re <psi|out> there and sets
// *dot_wpr to their count per row (dotpart[row * wpr + k]); 0 when the last
// pass was a per-term launch, which computes no partials.
static int pauli_apply_impl(hipStream_t s, void* out, const void* in, int64_t bsz, int n, int nterms,
                            const uint64_t* xmask, const uint64_t* zmask, const void* coef, int64_t coef_stride,
                            int accumulate, float* dotpart, int64_t* dot_wpr) {
  const uint64_t total = (uint64_t)bsz << n;
  int acc = accumulate ? 1 : 0;
  if (dot_wpr) *dot_wpr = 0;
  // terms grouped by local set: one LDS-staged pass per set
  std::shared_ptr<const PGPlan> P;
  if (n >= 8) P = pg_plan(n, nterms, xmask, zmask);
  std::vector<int> rest;
  if (P) {
    rest = P->rest;
    for (size_t i = 0; i < P->sets.size(); ++i) {
      const PGroup& g = P->sets[i];
      float* dp = (dotpart && rest.empty() && i + 1 == P->sets.size()) ? dotpart : nullptr;
      const int rc = pg_apply_launch(s, (float2*)out, (const float2*)in, n, g, (const float2*)coef, coef_stride, acc,
                                     bsz, dp);
      if (rc) return rc;
      if (dp) *dot_wpr = pg_wg_per_row(bsz, g.nnl, g.m);
      acc = 1;
    }
  } else {
    for (int t = 0; t < nterms; ++t) rest.push_back(t);
  }
  // the rest: gathered per amplitude, EV_MAXT terms per launch
  for (size_t t0 = 0; t0 < rest.size(); t0 += EV_MAXT) {
    PTerms pt;
    pt.nt = (int)(rest.size() - t0 < (size_t)EV_MAXT ? rest.size() - t0 : (size_t)EV_MAXT);
    for (int q = 0; q < pt.nt; ++q) {
      pt.x[q] = (uint32_t)xmask[rest[t0 + q]];
      pt.z[q] = (uint32_t)zmask[rest[t0 + q]];
      pt.col[q] = rest[t0 + q];
    }
    k_pauli_apply<<<grid_cap(total), EV_THREADS, 0, s>>>((float2*)out, (const float2*)in, n, total, pt,
                                                         (const float2*)coef, coef_stride, acc);
    int rc = check_launch("tqsv_pauli_apply");
    if (rc) return rc;
    acc = 1;
  }
  return OK;
}

static int pauli_args_ok(const char* who, const void* out, const void* in, int64_t bsz, int n, int nterms,
                         const uint64_t* xmask, const uint64_t* zmask, const void* coef) {
  if (!out || !in || !coef || (nterms > 0 && (!xmask || !zmask))) { set_error("%s: null pointer", who); return E_ARG; }
  if (out == in) { set_error("%s: out must not alias in", who); return E_ARG; }
  if (bsz < 1 || n < 1 || n > 32 || nterms < 1) { set_error("%s: bad sizes", who); return E_ARG; }
  for (int t = 0; t < nterms; ++t)
    if ((xmask[t] | zmask[t]) >> n) { set_error("%s: mask beyond n bits", who); return E_ARG; }
  return OK;
}

// out (+)= sum_t coef[row, t] P_t psi   (coef: device complex64 [bsz, nterms],
// already including i^{nY}); used for d/d psi of Pauli expectations.
TQSV_API int tqsv_pauli_apply(hipStream_t s, void* out, const void* in, int64_t bsz, int n, int nterms,
                              const uint64_t* xmask, const uint64_t* zmask, const void* coef, int accumulate) {
  int rc = pauli_args_ok("tqsv_pauli_apply", out, in, bsz, n, nterms, xmask, zmask, coef);
  if (rc) return rc;
  return row_slabs(bsz, [&](int64_t r0, int64_t rows) {
    return pauli_apply_impl(s, (float2*)out + (r0 << n), (const float2*)in + (r0 << n), rows, n, nterms, xmask, zmask,
                            (const float2*)coef + r0 * nterms, nterms, accumulate, nullptr, nullptr);
  });
}

// Floats of workspace tqsv_pauli_sum_grad needs (row partials of the dot).
TQSV_API int64_t tqsv_pauli_sum_grad_workspace_floats(int64_t bsz, int n) {
  if (bsz < 1 || n < 1 || n > 32) return -1;
  const int64_t fused = n >= 8 ? bsz * pg_wg_per_row(bsz, n - 8, 8) : 0;       // no set has more workgroups
  const int64_t plain = bsz << (n - ev_chunk_log2(bsz, n));
  return fused > plain ? fused : plain;
}

// Passes over the state that a list of strings takes (its sets; strings that
// fit none one each), planned anew.  Host work only.
TQSV_API int tqsv_pauli_passes(int n, int nterms, const uint64_t* xmask, const uint64_t* zmask) {
  if (n < 1 || n > 32 || nterms < 0 || (nterms > 0 && (!xmask || !zmask))) { set_error("tqsv_pauli_passes: bad arguments"); return E_ARG; }
  for (int t = 0; t < nterms; ++t)
    if ((xmask[t] | zmask[t]) >> n) { set_error("tqsv_pauli_passes: mask beyond n bits"); return E_ARG; }
  if (n < 8) return nterms;
  const std::vector<uint32_t> x(xmask, xmask + nterms), z(zmask, zmask + nterms);
  const PGPlan P = pg_build(n, n < PG_MAXM ? n : PG_MAXM, x, z);
  return (int)(P.sets.size() + P.rest.size());
}

// A Pauli sum and its state gradient in one go: out = sum_t coef[t] P_t psi
// (coef: device complex64 [nterms], the same for every row, including
// i^{nY}) and dot[row] = Re <psi_row|out_row> (device float [bsz]).  With
// coef = 2 c_t i^{nY_t}, dot / 2 is the row's sum_t c_t <P_t> and
// g_row * out is d(sum_row g_row value_row) / d conj(psi) -- what a
// differentiated Pauli-sum loss needs, for the cost of the backward's passes
// alone.  workspace: tqsv_pauli_sum_grad_workspace_floats floats.
TQSV_API int tqsv_pauli_sum_grad(hipStream_t s, void* out, const void* in, int64_t bsz, int n, int nterms,
                                 const uint64_t* xmask, const uint64_t* zmask, const void* coef, float* dot,
                                 float* workspace, int64_t workspace_floats) {
  int rc = pauli_args_ok("tqsv_pauli_sum_grad", out, in, bsz, n, nterms, xmask, zmask, coef);
  if (rc) return rc;
  if (!dot || !workspace) { set_error("tqsv_pauli_sum_grad: null pointer"); return E_ARG; }
  if ((uintptr_t)in & 15) { set_error("tqsv_pauli_sum_grad: state must be 16-byte aligned"); return E_ARG; }
  const int64_t need = tqsv_pauli_sum_grad_workspace_floats(bsz, n);
  if (workspace_floats < need) {
    set_error("tqsv_pauli_sum_grad: workspace of %lld floats, need %lld", (long long)workspace_floats,
              (long long)need);
    return E_ARG;
  }
  return row_slabs(bsz, [&](int64_t r0, int64_t rows) {
    float2* o = (float2*)out + (r0 << n);
    const float2* x = (const float2*)in + (r0 << n);
    int64_t wpr = 0;
    int rc = pauli_apply_impl(s, o, x, rows, n, nterms, xmask, zmask, coef, 0, 0, workspace, &wpr);
    if (rc) return rc;
    if (wpr == 0) {      // the last pass computed no partials: one read of psi and out
      const int lg = ev_chunk_log2(rows, n);
      k_rowdot_part<<<(unsigned)(rows << (n - lg)), EV_THREADS, 0, s>>>(x, o, n, lg, workspace);
      if ((rc = check_launch("tqsv_pauli_sum_grad/dot"))) return rc;
      wpr = 1ll << (n - lg);
    }
    k_sum_chunks<<<sum_grid(rows), 256, 0, s>>>(workspace, (int)wpr, 1, 0, rows, 1.f, 0.f, dot + r0, 1, 0);
    return check_launch("tqsv_pauli_sum_grad/sum");
  });
}
