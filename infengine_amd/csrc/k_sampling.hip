// Token selection over fp32 logits.
//
// argmax — reference sample_token_amax (kernels/sampling.cu:28-58) is a single
// 1024-thread block whose tie rule depends on thread layout.  Here the rule is
// torch.argmax's: the largest value wins, ties go to the smallest index, NaN
// counts as larger than everything, -0.0 equals +0.0.  Each (value, index) is
// packed into one 64-bit key whose unsigned order is exactly that rule, so the
// reduction is a plain max: per-workgroup max, then a device-scope atomicMax
// into a slot; the last workgroup of a row (counter) reads and clears the slot.
//
// top-p — no reference counterpart (the reference samples greedily).  The kept
// set follows HF TopPLogitsWarper (logits/T, drop the ascending-cumulative mass
// <= 1-p, keep >= 1 token): token i is kept iff the probability mass of tokens
// with a strictly larger scaled logit is < p.  Masses are exp(l/T - max) in
// fixed point (2^-40 units, uint64), so every sum is exact and order-free:
//   1. max of l/T; e_i = expf(l_i/T - max); Z = sum q_i
//   2. the cut key kappa with mass(key > kappa) < target <= mass(key >= kappa): the positive
//      masses binned by distance to the max locate its bin, then a radix select (4 x 8-bit
//      digits of the order-preserving key of l_i/T) over that bin's tokens
//   3. Z_kept = mass(key >= kappa); t = floor(Z_kept * u), u a 24-bit counter-RNG
//      uniform of (seed, row, step)
//   4. the sampled token is the smallest id whose kept prefix mass exceeds t
//      (inverse CDF in token-id order), found with a block-wide exclusive scan.
#include <cmath>
#include <mutex>

#include "ie_kernels.h"

namespace ie {

namespace {

__device__ __forceinline__ uint32_t order_key(float v) {
  if (v != v) return 0xFFFFFFFFu;
  if (v == 0.f) v = 0.f;
  const uint32_t u = __float_as_uint(v);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ __forceinline__ unsigned long long argmax_key(float v, unsigned idx) {
  return ((unsigned long long)order_key(v) << 32) | (unsigned long long)(0xFFFFFFFFu - idx);
}

__device__ __forceinline__ unsigned long long wave_max_u64(unsigned long long v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const unsigned long long w = __shfl_xor(v, o, 64);
    v = w > v ? w : v;
  }
  return v;
}

constexpr int kArgmaxBlocks = 64;

__global__ __launch_bounds__(256) void argmax_kernel(const float* logits, int vocab, int* out,
                                                     unsigned long long* slots,
                                                     unsigned int* counters, ArgmaxTail tail) {
  __shared__ unsigned long long red[4];
  const int row = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const float* L = logits + (size_t)row * vocab;
  const int chunk = (vocab + gridDim.x - 1) / gridDim.x;
  const int beg = blockIdx.x * chunk;
  const int end = min(vocab, beg + chunk);
  unsigned long long best = 0ull;
  // 8 loads in flight per thread per round (a chunk of the 128256-entry vocabulary is one
  // round): indices past the chunk load its last element and count as key 0
  for (int i0 = beg + tid; i0 < end; i0 += 8 * 256) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = L[min(i0 + u * 256, end - 1)];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int i = i0 + u * 256;
      // (masked arithmetically: a select let the compiler move a load under a branch)
      const unsigned long long k =
          argmax_key(v[u], (unsigned)i) & (0ull - (unsigned long long)(i < end));
      best = k > best ? k : best;
    }
  }
  best = wave_max_u64(best);
  if (lane == 0) red[wave] = best;
  __syncthreads();
  if (tid == 0) {
    unsigned long long b = red[0];
    for (int w = 1; w < 4; ++w) b = red[w] > b ? red[w] : b;
    // Device-scope atomics on one address are coherent across the XCDs; waiting for the max
    // to be performed before counting in orders the two, so the workgroup that counts last
    // exchanges out the final max.  (No __threadfence: on this part it writes back the L2.)
    unsigned long long* slot = slots + row * kSlotStride;
    unsigned int* counter = counters + row * kCntStride;
    atomicMax(slot, b);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (atomicAdd(counter, 1u) == gridDim.x - 1) {
      const unsigned long long fin = atomicExch(slot, 0ull);
      const int tok = (int)(0xFFFFFFFFu - (unsigned)(fin & 0xFFFFFFFFull));
      out[row] = tok;
      atomicExch(counter, 0u);
      if (row == 0) {
        if (tail.host_tok)
          __hip_atomic_store(tail.host_tok, tok, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        if (tail.seq) {
          const int s = *tail.seq;
          if (tail.tok_buf) tail.tok_buf[s] = tok;
          *tail.seq = s + 1;
        }
      }
    }
  }
}

// ---------------------------------------------------------------- top-p
constexpr int kTopPThreads = 1024;
constexpr float kFix = 1099511627776.0f;  // 2^40

__device__ __forceinline__ unsigned long long fix_mass(float e) {
  return (unsigned long long)(e * kFix);
}

template <typename T>
__device__ __forceinline__ T wave_sum_u64(T v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Inclusive scan over the wave's lanes.
template <typename T>
__device__ __forceinline__ T wave_scan(T v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const T w = __shfl_up(v, o, 64);
    if (lane >= o) v += w;
  }
  return v;
}

// Tokens with a positive fixed-point mass lie within 28 nats of the largest scaled logit
// (exp(-27.8) * 2^40 < 1), and only they can be kept (the cut token has positive mass, and every
// zero-mass token's key is below its key).  They are binned by their distance d = max - l/T into
// kTopPBins bins: bin(d) is non-decreasing in d, so every key of a lower bin is strictly larger
// than every key of a higher one and equal keys share a bin.  The bin where the cumulative mass
// from the top reaches the target holds the cut; the radix select runs over its tokens only.
// Tokens of lower bins are kept whole.
//
// Each row is split into kTopPChunks chunks, one workgroup each (a chunk of the 128256-entry
// vocabulary is one round of 8 loads in flight a thread), over four launches; the row's state is
// a TopPRow in the workspace, the masses are recomputed from the logits (a division and an expf a
// token, cheaper than caching them in memory):
//   tp_max     chunk maxima of l (the max of l/T is fl(max l / T): division by T > 0 is
//              monotone); the row's histogram and candidate count are cleared
//   tp_hist    chunk mass; the chunk's masses up to the last bin that can hold the cut, binned in
//              LDS and added to the row's histogram
//   tp_gather  every workgroup scans the histogram for the cut bin (identical results), then
//              appends its chunk's tokens of that bin to the candidates and sums the mass of its
//              tokens in lower bins
//   tp_finish  one workgroup per row: radix select of the cut key over the candidates (over the
//              row's tokens of the cut bin when there are more than kTopPCandMax), the chunks' kept
//              masses, t, the chunk holding t, then its token by a scan in token-id order
// 16 rows of the 128256-entry vocabulary: 30 us, 1 row 23; the six launches that cached
// the exponentials, used 2048 bins and summed the kept masses over all tokens took 53-57 and 37.
// 512 bins in place of 2048: the device-scope additions of the histograms (the largest part, 700
// thousand a call at 16 rows) fall to a quarter.
// The bins are octaves of 1.08 d + 2 in 128 steps each, 0.0145 nats wide at the top, 0.029 past 1.9 and
// 0.058 past 5.6: a row's cut lies at a few times the spread of its scaled logits, so that a flatter
// row has its cut where the bins are finer.  The cut bin of N(0, s) logits holds up to about 128256 x
// width / (2.5 s) tokens: the candidate list takes them from s = 0.09 on.  512 even bins took them from
// 0.27 on; 16 rows at p = 0.5, us, even bins / these: s = 0.1 275 / 46, 0.3 46 / 34, 0.8 34.5 / 32, 2.0
// 29.5 / 29.7 (p = 0.9: 31.2 / 31.7).  (576 bins, even past 1.2 nats: 30.3 and 32.9 at s = 2.0.)
constexpr int kTopPBins = 512;
constexpr int kTopPChunks = 64;
constexpr int kTopPChunkThreads = 256;
constexpr int kTopPCandMax = 9214;
constexpr int kTopPCandLds = 4096;  // candidates that tp_finish keeps in LDS

struct TopPRow {
  unsigned long long hist[kTopPBins];
  unsigned long long zpart[kTopPChunks];
  unsigned long long klow[kTopPChunks];  // mass of the chunk's tokens in bins below the cut bin
  float pmax[kTopPChunks];
  unsigned int ncand;
  int bcut;
  unsigned long long above, target;
  uint32_t cand_key[kTopPCandMax];
  unsigned long long cand_q[kTopPCandMax];  // mass (41 bits) | chunk << 48
};
// (rows that share cache lines make the histograms' additions slower: 16 rows 30.2 us, 29.1 so)
static_assert(sizeof(TopPRow) <= kTopPRowBytes && sizeof(TopPRow) % 256 == 0,
              "within the row of a caller's workspace, whole cache lines");

// The octaves 2-4, 4-8, 8-16 and 16-32 of 1.08 d + 2 (from 32 on, and NaN: any bin, without mass).
__host__ __device__ __forceinline__ int top_p_bin(float d) {
  return (int)(__builtin_bit_cast(uint32_t, fmaf(d, 1.08f, 2.0f)) >> 16 & (uint32_t)(kTopPBins - 1));
}
static_assert(kTopPBins == 512 && 1.08 * 27.73 + 2 < 32, "128 bins an octave; exp(-27.73) * 2^40 < 1");

__device__ __forceinline__ int tp_chunk_len(int vocab) {
  return (vocab + kTopPChunks - 1) / kTopPChunks;
}

// 8 logits of chunk [beg, end) from i on, 256 apart (past the end: the chunk's last one).
__device__ __forceinline__ void tp_load8(const float* L, int i, int end, float (&v)[8]) {
#pragma unroll
  for (int u = 0; u < 8; ++u) v[u] = L[min(i + u * kTopPChunkThreads, end - 1)];
}

// One 256-bin digit step of the radix select (wave 0): the highest digit whose cumulative mass
// from the top reaches t_rem; sets *bin and *above (the mass of the digits above it).
__device__ __forceinline__ void top_p_digit(const unsigned long long* hist, unsigned long long t_rem,
                                            int* s_bin, unsigned long long* s_above) {
  const int lane = threadIdx.x & 63;
  // lane l owns bins 255-4l .. 252-4l (descending digit order)
  unsigned long long hb[4], loc = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    hb[j] = hist[255 - 4 * lane - j];
    loc += hb[j];
  }
  const unsigned long long inc = wave_scan(loc);
  const unsigned long long exc = inc - loc;
  const unsigned long long hit = __ballot(inc >= t_rem);
  const int first = hit ? __ffsll((long long)hit) - 1 : 63;
  if (lane == first) {
    unsigned long long cum = exc;
    int bin = 252 - 4 * lane;
    unsigned long long above = cum;
    for (int j = 0; j < 4; ++j) {
      if (cum + hb[j] >= t_rem || j == 3) {
        bin = 255 - 4 * lane - j;
        above = cum;
        break;
      }
      cum += hb[j];
    }
    *s_bin = bin;
    *s_above = above;
  }
}

__global__ __launch_bounds__(kTopPChunkThreads) void tp_max_kernel(const float* logits, int vocab,
                                                                   TopPRow* rows) {
  __shared__ float redf[4];
  const int c = blockIdx.x, row = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  TopPRow& R = rows[row];
  const float* L = logits + (size_t)row * vocab;
  const int cl = tp_chunk_len(vocab), beg = c * cl, end = min(vocab, beg + cl);
  if (tid < kTopPBins / kTopPChunks) R.hist[c * (kTopPBins / kTopPChunks) + tid] = 0;
  if (c == 0 && tid == 0) R.ncand = 0;
  float m = -INFINITY;
  for (int i = beg + tid; i < end; i += 8 * kTopPChunkThreads) {
    float v[8];
    tp_load8(L, i, end, v);
#pragma unroll
    for (int u = 0; u < 8; ++u) m = fmaxf(m, v[u]);
  }
  m = wave_max(m);
  if (lane == 0) redf[wave] = m;
  __syncthreads();
  if (tid == 0) R.pmax[c] = fmaxf(fmaxf(redf[0], redf[1]), fmaxf(redf[2], redf[3]));
}

static_assert(kTopPChunks == 64, "one chunk a lane");

__device__ __forceinline__ float tp_row_max(const TopPRow& R, float temperature) {
  return wave_max(R.pmax[threadIdx.x & 63]) / temperature;
}

__global__ __launch_bounds__(kTopPChunkThreads) void tp_hist_kernel(const float* logits, int vocab,
                                                                    float temperature, int last_bin,
                                                                    TopPRow* rows) {
  __shared__ unsigned long long hist[kTopPBins];
  __shared__ unsigned long long red[4];
  const int c = blockIdx.x, row = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  TopPRow& R = rows[row];
  const float* L = logits + (size_t)row * vocab;
  const int cl = tp_chunk_len(vocab), beg = c * cl, end = min(vocab, beg + cl);
  for (int b = tid; b < kTopPBins; b += kTopPChunkThreads) hist[b] = 0;
  const float mx = tp_row_max(R, temperature);
  __syncthreads();
  unsigned long long z = 0;
  for (int i = beg + tid; i < end; i += 8 * kTopPChunkThreads) {
    float v[8];
    tp_load8(L, i, end, v);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      if (i + u * kTopPChunkThreads >= end) continue;
      const float sv = v[u] / temperature;
      const unsigned long long q = fix_mass(expf(sv - mx));
      z += q;
      const int b = top_p_bin(mx - sv);
      if (q && b <= last_bin) atomicAdd(&hist[b], q);
    }
  }
  z = wave_sum_u64(z);
  if (lane == 0) red[wave] = z;
  __syncthreads();
  if (tid == 0) R.zpart[c] = (red[0] + red[1]) + (red[2] + red[3]);
  for (int b = tid; b <= last_bin; b += kTopPChunkThreads)
    if (hist[b]) atomicAdd(&R.hist[b], hist[b]);
}

__global__ __launch_bounds__(kTopPChunkThreads) void tp_gather_kernel(const float* logits, int vocab,
                                                                      float temperature, float top_p,
                                                                      TopPRow* rows) {
  static_assert(kTopPBins == 2 * kTopPChunkThreads, "two bins a thread");
  __shared__ unsigned long long red[4];
  __shared__ unsigned int cnt[4], s_base;
  __shared__ int s_bin;
  __shared__ unsigned long long s_above;
  const int c = blockIdx.x, row = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  TopPRow& R = rows[row];
  const float* L = logits + (size_t)row * vocab;
  const int cl = tp_chunk_len(vocab), beg = c * cl, end = min(vocab, beg + cl);
  const unsigned long long z = wave_sum_u64(R.zpart[lane]);
  const float mx = tp_row_max(R, temperature);
  // (held to z: past 2^53 units, a row whose exp(l/T - max) sum to over 8192, (double)z may round
  // up, and at top_p = 1 no bin would reach a target past the row's mass)
  unsigned long long target = (unsigned long long)((double)z * (double)top_p);
  if (target > z) target = z;
  if (target < 1) target = 1;
  // the cut bin: thread t owns bins 2t, 2t + 1 (ascending distance), block inclusive scan
  const unsigned long long h0 = R.hist[2 * tid], h1 = R.hist[2 * tid + 1];
  unsigned long long inc = wave_scan(h0 + h1);
  if (lane == 63) red[wave] = inc;
  if (tid == 0) s_bin = -1, s_above = 0;
  __syncthreads();
  for (int w = 0; w < wave; ++w) inc += red[w];
  const unsigned long long exc = inc - (h0 + h1);
  if (exc < target && inc >= target) {  // exactly one thread
    const bool first = exc + h0 >= target;
    s_bin = first ? 2 * tid : 2 * tid + 1;
    s_above = first ? exc : exc + h0;
  }
  __syncthreads();
  const int bcut = s_bin;
  if (c == 0 && tid == 0) {
    R.bcut = bcut;
    R.above = s_above;
    R.target = target;
  }
  unsigned long long low = 0;
  // (beg and end are the workgroup's: every thread runs every round and its barriers)
  for (int i0 = beg; i0 < end; i0 += 8 * kTopPChunkThreads) {
    const int i = i0 + tid;
    float v[8];
    tp_load8(L, i, end, v);
    unsigned int hits = 0;
    unsigned long long q[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const float sv = v[u] / temperature;
      const int b = top_p_bin(mx - sv);
      const bool in = i + u * kTopPChunkThreads < end;
      q[u] = fix_mass(expf(sv - mx));
      if (in && b < bcut) low += q[u];
      if (in && b == bcut && q[u]) hits |= 1u << u;
    }
    // this round's candidates take consecutive slots: one device-scope addition a workgroup
    const unsigned int n = __popc(hits), ninc = wave_scan(n);
    if (lane == 63) cnt[wave] = ninc;
    __syncthreads();
    if (tid == 0) {
      const unsigned int all = (cnt[0] + cnt[1]) + (cnt[2] + cnt[3]);
      s_base = all ? atomicAdd(&R.ncand, all) : 0;
    }
    __syncthreads();
    unsigned int slot = s_base + ninc - n;
    for (int w = 0; w < wave; ++w) slot += cnt[w];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      if (!(hits >> u & 1)) continue;
      if (slot < (unsigned)kTopPCandMax) {
        R.cand_key[slot] = order_key(v[u] / temperature);
        R.cand_q[slot] = q[u] | (unsigned long long)c << 48;
      }
      ++slot;
    }
    __syncthreads();  // cnt and s_base are reused
  }
  low = wave_sum_u64(low);
  if (lane == 0) red[wave] = low;
  __syncthreads();
  if (tid == 0) R.klow[c] = (red[0] + red[1]) + (red[2] + red[3]);
}

__global__ __launch_bounds__(kTopPThreads) void tp_finish_kernel(const float* logits, int vocab,
                                                                 float temperature, uint64_t seed,
                                                                 uint64_t step, TopPRow* rows,
                                                                 int* out) {
  __shared__ unsigned long long hist[256];
  __shared__ uint32_t ck[kTopPCandLds];
  __shared__ unsigned long long cq[kTopPCandLds];
  __shared__ unsigned long long kpart[kTopPChunks];
  __shared__ unsigned long long red[kTopPThreads / 64];
  __shared__ int s_bin, s_chunk, s_tok;
  __shared__ unsigned long long s_above, s_t;
  const int row = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  TopPRow& R = rows[row];
  const float* L = logits + (size_t)row * vocab;
  const int cl = tp_chunk_len(vocab);
  const int ncand = (int)R.ncand, bcut = R.bcut;
  const bool listed = ncand <= kTopPCandMax, in_lds = ncand <= kTopPCandLds;
  const float mx = tp_row_max(R, temperature);
  unsigned long long t_rem = R.target - R.above;
  if (tid < kTopPChunks) kpart[tid] = R.klow[tid];
  if (tid == 0) s_tok = -1;
  if (in_lds)
    for (int j = tid; j < ncand; j += kTopPThreads) ck[j] = R.cand_key[j], cq[j] = R.cand_q[j];
  // f(key, mass, chunk) over the tokens of the cut bin (chunk 0 for those of a row that is not listed)
  const auto each = [&](auto f) {
    if (listed) {
      for (int j = tid; j < ncand; j += kTopPThreads) {
        const uint32_t k = in_lds ? ck[j] : R.cand_key[j];
        const unsigned long long q = in_lds ? cq[j] : R.cand_q[j];
        f(k, q & 0xFFFFFFFFFFFFull, (int)(q >> 48));
      }
    } else {
      for (int i = tid; i < vocab; i += kTopPThreads) {
        const float sv = L[i] / temperature;
        if (top_p_bin(mx - sv) != bcut) continue;
        const unsigned long long q = fix_mass(expf(sv - mx));
        if (q) f(order_key(sv), q, 0);
      }
    }
  };
  uint32_t prefix = 0, mask = 0;
  for (int shift = 24; shift >= 0; shift -= 8) {
    if (tid < 256) hist[tid] = 0;
    __syncthreads();
    each([&](uint32_t k, unsigned long long q, int) {
      if ((k & mask) == prefix) atomicAdd(&hist[(k >> shift) & 255u], q);
    });
    __syncthreads();
    if (wave == 0) top_p_digit(hist, t_rem, &s_bin, &s_above);
    __syncthreads();
    prefix |= (uint32_t)s_bin << shift;
    mask |= 255u << shift;
    t_rem -= s_above;
    __syncthreads();
  }
  const uint32_t kappa = prefix;
  // the chunks' kept masses: lower bins whole, the cut bin's keys from kappa up
  if (listed) {
    each([&](uint32_t k, unsigned long long q, int c) {
      if (k >= kappa) atomicAdd(&kpart[c], q);
    });
  } else {
    // a wave per chunk (adding token by token to 64 sums took 50 us of a row of equal logits; rolled
    // up: more code for these rows cost the listed ones 0.3 us)
    for (int c = wave; c < kTopPChunks; c += kTopPThreads / 64) {
      const int end = min(vocab, c * cl + cl);
      unsigned long long kept = 0;
#pragma unroll 1
      for (int i = c * cl + lane; i < end; i += 64) {
        const float sv = L[i] / temperature;
        if (top_p_bin(mx - sv) == bcut && order_key(sv) >= kappa) kept += fix_mass(expf(sv - mx));
      }
      kept = wave_sum_u64(kept);
      if (lane == 0) kpart[c] += kept;
    }
  }
  __syncthreads();
  // t, and the chunk holding it (kept masses in chunk order = token-id order)
  if (wave == 0) {
    const unsigned long long kp = kpart[lane], inc = wave_scan(kp);
    const unsigned long long zk = __shfl(inc, 63, 64);
    const uint64_t bits = splitmix64(synth_base(seed, 0x70707070ull + (uint64_t)row) + step) >> 40;
    const unsigned long long t = (zk >> 24) * bits + (((zk & 0xFFFFFFull) * bits) >> 24);
    const unsigned long long hit = __ballot(inc > t);
    const int c = hit ? __ffsll((long long)hit) - 1 : kTopPChunks - 1;
    if (lane == c) {
      s_chunk = c;
      s_t = t - (inc - kp);  // within the chunk
    }
  }
  __syncthreads();
  // the chunk's tokens in token-id order, kTopPThreads at a time
  const int cbeg = min(vocab, s_chunk * cl), cend = min(vocab, cbeg + cl);
  unsigned long long base = 0;
  for (int i0 = cbeg; i0 < cend; i0 += kTopPThreads) {
    const int i = i0 + tid;
    unsigned long long q = 0;
    if (i < cend) {
      const float sv = L[i] / temperature;
      if (order_key(sv) >= kappa) q = fix_mass(expf(sv - mx));
    }
    unsigned long long inc = wave_scan(q);
    if (lane == 63) red[wave] = inc;
    __syncthreads();
    unsigned long long all = 0;
#pragma unroll
    for (int w = 0; w < kTopPThreads / 64; ++w) {
      if (w < wave) inc += red[w];
      all += red[w];
    }
    inc += base;
    if (q && inc - q <= s_t && s_t < inc) s_tok = i;  // exactly one token
    base += all;
    __syncthreads();
  }
  if (tid == 0) out[row] = s_tok;
}

}  // namespace

static_assert(kTopPScratchBytes >= kTopPNoallocRows * sizeof(TopPRow),
              "the static scratch holds the largest no-allocation workspace");

// ---------------------------------------------------------------- no-allocation scratch
// The top-p sampler's workspace (a TopPRow per row) for the entry point that takes none: a
// file-scope device array of kTopPScratchBytes (kTopPNoallocRows TopPRows), one copy per GPU
// for the life of the process.  Host code never passes `scratch` itself to a kernel (on the
// host the name is only a stand-in, not the device address): top_p_scratch_init looks up each
// device's address once with hipGetSymbolAddress and the launcher passes that.
static __device__ __align__(256) float scratch[kTopPScratchBytes / sizeof(float)];

namespace {
constexpr int kMaxDevices = 64;
float* g_scratch_addr[kMaxDevices] = {};
std::mutex g_scratch_mu;
}  // namespace

int top_p_scratch_init(int device) {
  IE_REQUIRE(device >= 0 && device < kMaxDevices, "top_p scratch: device %d out of [0, %d)",
             device, kMaxDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_addr[device]) return IE_OK;
  int cur = -1;
  IE_CHECK_HIP(hipGetDevice(&cur));
  IE_REQUIRE(cur == device, "top_p scratch: device %d is not current (%d is)", device, cur);
  void* addr = nullptr;
  IE_CHECK_HIP(hipGetSymbolAddress(&addr, HIP_SYMBOL(scratch)));
  IE_REQUIRE(addr != nullptr, "top_p scratch: no device address for device %d", device);
  g_scratch_addr[device] = static_cast<float*>(addr);
  return IE_OK;
}

float* top_p_scratch(int device) {
  if (device < 0 || device >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  return g_scratch_addr[device];
}

int launch_argmax_rows(int rows, int vocab, const float* logits, int* out,
                       unsigned long long* slots, unsigned int* counters, hipStream_t st,
                       ArgmaxTail tail) {
  IE_REQUIRE(rows >= 1 && rows <= kNumSlots, "argmax: rows=%d out of range [1,%d]", rows,
             kNumSlots);
  IE_REQUIRE(vocab >= 1, "argmax: vocab=%d", vocab);
  int blocks = kArgmaxBlocks;
  if (vocab < blocks * 256) blocks = (vocab + 255) / 256;
  hipLaunchKernelGGL(argmax_kernel, dim3(blocks, rows), dim3(256), 0, st, logits, vocab, out,
                     slots, counters, tail);
  IE_CHECK_LAUNCH();
  return IE_OK;
}

size_t top_p_workspace_bytes(int rows) { return (size_t)rows * kTopPRowBytes; }

int launch_top_p(int rows, int vocab, const float* logits, float temperature, float top_p,
                 uint64_t seed, uint64_t step, int* out, float* ws, hipStream_t st) {
  IE_REQUIRE(rows >= 1 && rows <= 65535, "top_p: rows=%d", rows);
  IE_REQUIRE(vocab >= 1, "top_p: vocab=%d", vocab);
  IE_REQUIRE(temperature > 0.f, "top_p: temperature must be > 0 (got %g)", (double)temperature);
  IE_REQUIRE(top_p > 0.f && top_p <= 1.f, "top_p: top_p must be in (0, 1] (got %g)",
             (double)top_p);
  TopPRow* R = reinterpret_cast<TopPRow*>(ws);
  // The last bin that can hold the cut: the largest token alone has mass 1, the tokens past d
  // nats at most vocab exp(-d), and the cut lies before the point where what is past it falls
  // below the (1 - p) Z left out (half of it, for the roundings).
  const double left = 1.0 - (double)top_p;
  const double d0 = left > 1e-9 ? std::log(2.0 * vocab / left) : 28.0;
  const int last_bin = d0 < 27.0 ? top_p_bin((float)d0) + 1 : kTopPBins - 1;
  const dim3 chunks(kTopPChunks, rows);
  hipLaunchKernelGGL(tp_max_kernel, chunks, dim3(kTopPChunkThreads), 0, st, logits, vocab, R);
  hipLaunchKernelGGL(tp_hist_kernel, chunks, dim3(kTopPChunkThreads), 0, st, logits, vocab,
                     temperature, last_bin, R);
  hipLaunchKernelGGL(tp_gather_kernel, chunks, dim3(kTopPChunkThreads), 0, st, logits, vocab,
                     temperature, top_p, R);
  hipLaunchKernelGGL(tp_finish_kernel, dim3(rows), dim3(kTopPThreads), 0, st, logits, vocab,
                     temperature, seed, step, R, out);
  IE_CHECK_LAUNCH();
  return IE_OK;
}

}  // namespace ie
