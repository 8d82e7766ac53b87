// Stochastic token sampling on the device: the steps of the reference's
// sampler_sample (source/sampler.c:234-337) on logits already in HBM.
//
//   presence penalty (source/sampler.c:238-248): logits of tokens seen
//     (the previous token is marked first) lower by the penalty;
//   greedy (temperature 0): the first index of the maximum (argmax kernels);
//   else: logits / temperature, softmax (max, expf(x - max), divide by the
//     sum), one xorshift64* coin, top-k (the k most likely), top-p (the
//     shortest descending prefix whose running sum reaches top_p),
//     renormalisation (double sum), and the first index whose running sum
//     of probabilities in index order exceeds the coin.
//
// Differences from the sequential host code are in summation order only:
// the softmax sum and the renormalisation's double sum, and without a top-k of
// at most 1024 the top-p and the index-order running sums too, are formed from
// fixed-order partial sums (deterministic, but rounded differently), so a
// draw can differ from the reference's only when the coin or top_p lies within
// that rounding of a boundary. (A top-k of at most 1024 adds both running sums
// one probability after the other, as the reference does.) Equal probabilities
// rank by index, as a stable sort of the reference's index-ordered array ranks
// them. The coin stream, the
// penalty and every per-element operation (division by the temperature,
// expf, division by the sum, multiplication by the float inverse of the
// double sum) are the reference's.
#include <limits.h>

#include "device_common.h"
#include "hip_check.h"
#include "kernels.h"

namespace sg {
namespace {

constexpr int kSB = 256;    // blocks of the element-wise passes
constexpr int kST = 256;    // their threads
constexpr int kPick = 1024; // threads of the single-block passes
static_assert(kSB == kST, "the per-block partials are reduced by one block of kST threads");

__device__ __forceinline__ float block_max256(float v, float* red) {
  v = wave_peak(v);
  const int w = threadIdx.x / WAVE, l = threadIdx.x % WAVE;
  if (l == 0) red[w] = v;
  __syncthreads();
  float m = -INFINITY;
#pragma unroll
  for (int i = 0; i < kST / WAVE; i++) m = fmaxf(m, red[i]);
  __syncthreads();
  return m;
}

// Penalty, temperature, per-block maxima. Marks the previous token present;
// clears the candidate count of the small top-k draw, if given.
__global__ __launch_bounds__(kST) void sample_scale_kernel(SampleParams p, unsigned* count) {
  if (count && blockIdx.x == 0 && threadIdx.x == 0) *count = 0u;
  __shared__ float red[kST / WAVE];
  const int prev = p.prev ? *p.prev : p.prev_value;
  float m = -INFINITY;
  for (int i = blockIdx.x * kST + threadIdx.x; i < p.V; i += kSB * kST) {
    float x = p.logits[i];
    if (p.penalty != 0.0f && (p.presence[i] || i == prev)) x -= p.penalty;
    if (p.temperature != 0.0f) x = x / p.temperature;
    p.y[i] = x;
    m = fmaxf(m, x);
  }
  m = block_max256(m, red);
  if (threadIdx.x == 0) p.part[blockIdx.x] = m;
  if (blockIdx.x == 0 && threadIdx.x == 0 && prev >= 0 && prev < p.V) p.presence[prev] = 1;
}

// expf(x - max) in place, per-block sums.
__global__ __launch_bounds__(kST) void sample_exp_kernel(SampleParams p) {
  __shared__ float red[kST / WAVE];
  const float mx = block_max256(p.part[threadIdx.x], red);  // the same in every block
  float s = 0.0f;
  for (int i = blockIdx.x * kST + threadIdx.x; i < p.V; i += kSB * kST) {
    const float e = expf(p.y[i] - mx);
    p.y[i] = e;
    s += e;
  }
  s = block_sum<kST>(s, red);
  if (threadIdx.x == 0) p.part[kSB + blockIdx.x] = s;
}

// Probabilities, the sort keys, cleared keep marks, and the coin.
__global__ __launch_bounds__(kST) void sample_norm_kernel(SampleParams p) {
  __shared__ float red[kST / WAVE];
  const float sum = block_sum<kST>(p.part[kSB + threadIdx.x], red);  // the same in every block
  for (int i = blockIdx.x * kST + threadIdx.x; i < p.V; i += kSB * kST) {
    const float q = p.y[i] / sum;
    p.y[i] = q;
    if (p.keys) {
      p.keys[i] = __float_as_uint(q);  // q >= 0: the bit patterns order like the values
      p.vals[i] = i;
      p.keep[i] = 0;
    }
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    unsigned long long s = *p.rng;  // xorshift64* (source/sampler.c:79-90)
    s ^= s >> 12;
    s ^= s << 25;
    s ^= s >> 27;
    *p.rng = s;
    const unsigned u = (unsigned)((s * 0x2545F4914F6CDD1Dull) >> 32);
    p.scal[0] = (float)(u >> 8) / 16777216.0f;
  }
}

__device__ __forceinline__ double block_sum_d(double v, double* red) {
  red[threadIdx.x] = v;
  __syncthreads();
  for (int st = kPick / 2; st > 0; st >>= 1) {
    if (threadIdx.x < st) red[threadIdx.x] += red[threadIdx.x + st];
    __syncthreads();
  }
  const double s = red[0];
  __syncthreads();
  return s;
}

// Top-k / top-p cut over the descending order, the renormalisation factor,
// and the kept tokens' marks.
__global__ __launch_bounds__(kPick) void sample_select_kernel(SampleParams p) {
  __shared__ float scan[2][kPick];
  __shared__ double dred[kPick];
  __shared__ int found;
  const int tid = threadIdx.x, V = p.V;
  const bool sorted = p.keys != nullptr;
  int n = V;
  if (sorted) {
    const int kact = p.top_k > 0 && p.top_k < V ? p.top_k : V;
    n = kact;
    if (p.top_p > 0.0f && p.top_p <= 1.0f) {
      if (tid == 0) found = INT_MAX;
      float carry = 0.0f;
      __syncthreads();
      for (int base = 0; base < kact; base += kPick) {
        const int i = base + tid;
        float v = i < kact ? __uint_as_float(p.keys_sorted[i]) : 0.0f;
        int cur = 0;
        scan[0][tid] = v;
        __syncthreads();
        for (int off = 1; off < kPick; off <<= 1) {  // inclusive scan, fixed order
          const float add = tid >= off ? scan[cur][tid - off] : 0.0f;
          scan[cur ^ 1][tid] = scan[cur][tid] + add;
          cur ^= 1;
          __syncthreads();
        }
        const float cum = carry + scan[cur][tid];
        if (i < kact && cum >= p.top_p) atomicMin(&found, i);  // the first index reaching top_p
        __syncthreads();
        carry += scan[cur][kPick - 1];
        __syncthreads();
        if (found != INT_MAX) break;
      }
      if (found != INT_MAX) n = found + 1 < kact ? found + 1 : kact;
    }
  }
  double s = 0.0;
  if (sorted) {
    for (int r = tid; r < n; r += kPick) s += (double)__uint_as_float(p.keys_sorted[r]);
  } else {
    for (int i = tid; i < V; i += kPick) s += (double)p.y[i];
  }
  s = block_sum_d(s, dred);
  if (sorted)
    for (int r = tid; r < n; r += kPick) p.keep[p.vals_sorted[r]] = 1;
  if (tid == 0) {
    p.scal[1] = s > 0.0 ? (float)(1.0 / s) : 0.0f;
    p.scal[2] = s > 0.0 ? 0.0f : 1.0f;  // nothing left: uniform over every token
    *p.nkeep = n;
  }
}

// The first index of nonzero weight whose running sum of renormalised
// probabilities (index order) exceeds the coin; then the token bookkeeping
// of the decode loop.
__global__ __launch_bounds__(kPick) void sample_pick_kernel(SampleParams p) {
  __shared__ float pre[kPick];
  __shared__ int best;
  const int tid = threadIdx.x, V = p.V;
  const float coin = p.scal[0], inv = p.scal[1];
  const bool uniform = p.scal[2] != 0.0f, all = p.keys == nullptr;
  const float u = 1.0f / (float)V;
  const int R = (V + kPick - 1) / kPick, lo = min(V, tid * R), hi = min(V, lo + R);
  auto w = [&](int i) -> float {
    return uniform ? u : (all || p.keep[i]) ? p.y[i] * inv : 0.0f;
  };
  float s = 0.0f;
  for (int i = lo; i < hi; i++) s += w(i);
  pre[tid] = s;
  if (tid == 0) best = V;
  __syncthreads();
  if (tid == 0) {  // exclusive prefix in thread order, sequential
    float c = 0.0f;
    for (int t = 0; t < kPick; t++) {
      const float x = pre[t];
      pre[t] = c;
      c += x;
    }
  }
  __syncthreads();
  // A thread's start (the prefix of separately summed partials) can round
  // above the previous thread's last running sum; only an index of nonzero
  // weight is taken, so a coin in that gap never picks a token that top-k or
  // top-p removed (the reference's loop never returns one either).
  float cdf = pre[tid];
  for (int i = lo; i < hi; i++) {
    const float wi = w(i);
    cdf += wi;
    if (wi > 0.0f && coin < cdf) {
      atomicMin(&best, i);
      break;
    }
  }
  __syncthreads();
  if (tid == 0) {
    const int tok = best < V ? best : V - 1;  // rounding fallback, as the reference's
    *p.out = tok;
    if (p.seq) p.seq[(*p.seq_len)++] = tok;
    if (p.pos_inc) (*p.pos_inc)++;
  }
}

// ----------------------------------------------------------- small top-k --
// top_k of at most kTopMax (the usual case) needs no sort of the
// vocabulary: three launches instead of seventeen. Bound by their launches and
// chains of barriers, not by bytes (V floats read and written twice):
// V = 128256, k = 50, 225 -> 29 us a draw, of which the full sort's picking
// kernel took 121 (one block walking the whole vocabulary) and the sort 81;
// k = 1024 with a top-p 235 -> 122, at V = 32000 107 -> 78. The worst case is a
// vocabulary of equal probabilities, all of them candidates of the one drawing
// block: 233 us, the full sort 207 and 14 launches more.
// * scale (above): penalty, temperature, block maxima;
// * exp: expf, block sums, and each block's candidates: the elements in the
//   eighth-octave bins of expf down to the bin that holds the block's k-th
//   largest, and one bin more, so that a value which the division by the sum
//   rounds onto a larger one across a bin's edge is there too (every element
//   where that division can leave the normal range);
// * draw: one block divides the candidates by the sum, finds the k largest
//   by radix selection on (probability bits, lower index first), sorts them
//   and applies top-p, the renormalisation and the pick in the reference's
//   sequential orders.
// Results are those of the full sort below: the same probabilities bit for
// bit, the same order, ties by index.
constexpr int kTopMax = 1024;
constexpr int kTopCap = 2048;   // elements the draw sorts in LDS
constexpr int kTopBins = 4096;  // 12-bit digits of the radix selection
constexpr int kExpBins = 1024;  // bits >> 20 of expf(x - max) <= 1 (NaNs in the last bin)
constexpr int kExpLow = 264;    // 2^-94: below it a value over a sum < 2^31 can be subnormal

__device__ __forceinline__ int exp_bin(float e) { return (int)min(__float_as_uint(e) >> 20, (unsigned)(kExpBins - 1)); }

__global__ __launch_bounds__(kST) void sample_exp_top_kernel(SampleParams p, unsigned* count) {
  constexpr int PER = kExpBins / kST;
  __shared__ float red[kST / WAVE];
  __shared__ unsigned hist[kExpBins];
  __shared__ unsigned above[kST + 1];  // elements in the bins of threads >= t
  __shared__ int cut;
  __shared__ unsigned base, next;
  const int tid = threadIdx.x;
  for (int b = tid; b < kExpBins; b += kST) hist[b] = 0u;
  if (tid == 0) {
    cut = 0;
    next = 0u;
    above[kST] = 0u;
  }
  const float mx = block_max256(p.part[tid], red);  // the same in every block (its barriers order hist)
  float s = 0.0f;
  for (int i = blockIdx.x * kST + tid; i < p.V; i += kSB * kST) {
    const float e = expf(p.y[i] - mx);
    p.y[i] = e;
    s += e;
    atomicAdd(&hist[exp_bin(e)], 1u);
  }
  s = block_sum<kST>(s, red);
  if (tid == 0) p.part[kSB + blockIdx.x] = s;
  // suffix counts, PER bins a thread
  unsigned mine = 0u;
#pragma unroll
  for (int b = 0; b < PER; b++) mine += hist[tid * PER + b];
  above[tid] = mine;
  __syncthreads();
  for (int off = 1; off < kST; off <<= 1) {
    const unsigned add = tid + off < kST ? above[tid + off] : 0u;
    __syncthreads();
    above[tid] += add;
    __syncthreads();
  }
  // the largest bin with at least k elements at or above it (bin 0 if the
  // block holds fewer)
  const unsigned k = (unsigned)p.top_k;
  if (above[tid] >= k && above[tid + 1] < k) {
    unsigned c = above[tid + 1];
    int b = PER;
    while (c < k) c += hist[tid * PER + --b];
    b += tid * PER - 1;
    cut = b >= kExpLow ? b : 0;
  }
  __syncthreads();
  if (tid == 0) {
    const int t = cut / PER;
    unsigned n = above[t + 1];
    for (int b = cut % PER; b < PER; b++) n += hist[t * PER + b];
    base = n ? atomicAdd(count, n) : 0u;
  }
  __syncthreads();
  for (int i = blockIdx.x * kST + tid; i < p.V; i += kSB * kST) {
    const float e = p.y[i];  // written by this thread above
    if (exp_bin(e) < cut) continue;
    const unsigned at = base + atomicAdd(&next, 1u);
    p.keys_sorted[at] = __float_as_uint(e);
    p.vals_sorted[at] = i;
  }
}

// Sorts key[0..n) descending into out (n <= kTopCap, distinct keys): by
// counting the larger keys up to 256, else a bitonic network in place (the
// result is copied to out). All kPick threads call it.
__device__ void sort_desc_lds(unsigned long long* key, unsigned long long* out, int n) {
  const int tid = threadIdx.x;
  if (n <= 256) {
    if (tid < n) {
      const unsigned long long x = key[tid];
      int rank = 0;
      for (int j = 0; j < n; j++) rank += key[j] > x;
      out[rank] = x;
    }
    __syncthreads();
    return;
  }
  int m = 512;
  while (m < n) m <<= 1;
  for (int i = n + tid; i < m; i += kPick) key[i] = 0ull;
  __syncthreads();
  for (int size = 2; size <= m; size <<= 1) {
    for (int st = size >> 1; st > 0; st >>= 1) {
      for (int q = tid; q < m / 2; q += kPick) {
        const int i = 2 * q - (q & (st - 1)), j = i + st;
        const unsigned long long a = key[i], b = key[j];
        if ((a < b) == ((i & size) == 0)) {
          key[i] = b;
          key[j] = a;
        }
      }
      __syncthreads();
    }
  }
  for (int i = tid; i < n; i += kPick) out[i] = key[i];
  __syncthreads();
}

__global__ __launch_bounds__(kPick) void sample_draw_kernel(SampleParams p, const unsigned* count) {
  __shared__ unsigned hist[kTopBins];
  __shared__ unsigned above[kPick + 1];
  __shared__ unsigned long long key[kTopCap], sorted[kTopCap];
  __shared__ double dred[kPick];
  __shared__ float red[kST / WAVE];
  __shared__ unsigned long long prefix_s;
  __shared__ unsigned above_s, bin_s, got;
  __shared__ int kept_s, best;
  const int tid = threadIdx.x, lane = tid % WAVE, V = p.V;
  const unsigned total = *count;
  // the sum of sample_exp_top_kernel's block sums, in block_sum<kST>'s order
  float sum = 0.0f;
  if (tid < kST) {
    const float v = wave_sum(p.part[kSB + tid]);
    if (lane == 0) red[tid / WAVE] = v;
  }
  if (tid == 0) {
    got = 0u;
    best = V;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kST / WAVE; i++) sum += red[i];
  // Every candidate's key (larger probability first, then the lower index:
  // distinct) to f(valid, key), by all lanes of a wavefront together, kU
  // candidates a thread in flight: near-uniform distributions make candidates
  // of the whole vocabulary, and one at a time each pass over 128256 of them
  // waited 125 latencies.
  auto each = [&](auto f) {
    constexpr int kU = 8;
    auto keyed = [&](unsigned c, unsigned e, int index) {
      const float q = __uint_as_float(e) / sum;
      f(c < total, ((unsigned long long)__float_as_uint(q) << 32) | (unsigned)~index);
    };
    if (total <= (unsigned)kPick) {
      const unsigned c = min((unsigned)tid, total - 1);
      keyed(tid, p.keys_sorted[c], p.vals_sorted[c]);
      return;
    }
    for (unsigned c0 = 0; c0 < total; c0 += kU * kPick) {
      unsigned kb[kU];
      int vi[kU];
#pragma unroll
      for (int u = 0; u < kU; u++) {
        const unsigned c = min(c0 + u * kPick + tid, total - 1);
        kb[u] = p.keys_sorted[c];
        vi[u] = p.vals_sorted[c];
      }
#pragma unroll
      for (int u = 0; u < kU; u++) {
        if (c0 + u * kPick >= total) break;
        keyed(c0 + u * kPick + tid, kb[u], vi[u]);
      }
    }
  };

  // Radix selection: 12-bit digits from the top until what lies at or above
  // the k-th key's digits fits the LDS sort (the first digit nearly always;
  // all of them for a vocabulary of equal probabilities).
  const unsigned k = (unsigned)p.top_k;
  unsigned long long prefix = 0ull;
  unsigned over = 0u;  // elements above the prefix
  int shift = 64;
  for (;;) {
    const int low = max(shift - 12, 0), bits = shift - low;
    for (int b = tid; b < kTopBins; b += kPick) hist[b] = 0u;
    if (tid == 0) above[kPick] = 0u;
    __syncthreads();
    each([&](bool valid, unsigned long long x) {
      const bool in = valid && (shift == 64 || (x >> shift) == prefix);
      const unsigned b = (unsigned)(x >> low) & ((1u << bits) - 1u);
      const unsigned long long m = __ballot(in);
      if (!m) return;
      const int first = __ffsll((long long)m) - 1;
      // one addition where the wavefront's digits agree (ties: 64 additions
      // to one address are done one after the other)
      if (__ballot(in && b == (unsigned)__builtin_amdgcn_readlane((int)b, first)) == m) {
        if (lane == first) atomicAdd(&hist[b], (unsigned)__popcll(m));
      } else if (in) {
        atomicAdd(&hist[b], 1u);
      }
    });
    __syncthreads();
    constexpr int PER = kTopBins / kPick;
    unsigned mine = 0u;
#pragma unroll
    for (int b = 0; b < PER; b++) mine += hist[tid * PER + b];
    // inclusive suffix sums: within the wavefront, then over the wavefronts
    unsigned run = mine;
#pragma unroll
    for (int off = 1; off < WAVE; off <<= 1) {
      const unsigned add = __shfl_down(run, off, WAVE);
      if (lane + off < WAVE) run += add;
    }
    __shared__ unsigned wtot[kPick / WAVE];
    if (lane == 0) wtot[tid / WAVE] = run;
    __syncthreads();
    for (int w = tid / WAVE + 1; w < kPick / WAVE; w++) run += wtot[w];
    above[tid] = run;
    __syncthreads();
    if (over + above[tid] >= k && over + above[tid + 1] < k) {
      unsigned c = over + above[tid + 1];
      int b = PER;
      unsigned h = 0u;
      while (c < k) {
        h = hist[tid * PER + --b];
        c += h;
      }
      prefix_s = (shift == 64 ? 0ull : prefix << bits) | (unsigned)(tid * PER + b);
      above_s = c - h;
      bin_s = h;
    }
    __syncthreads();
    prefix = prefix_s;
    over = above_s;
    shift = low;
    if (over + bin_s <= (unsigned)kTopCap || shift == 0) break;
    __syncthreads();  // prefix_s, above_s and bin_s are read before the next digit's
  }
  each([&](bool valid, unsigned long long x) {
    if (valid && (x >> shift) >= prefix) {
      const unsigned at = atomicAdd(&got, 1u);
      if (at < (unsigned)kTopCap) key[at] = x;
    }
  });
  __syncthreads();
  const int n0 = (int)min(got, (unsigned)kTopCap);
  sort_desc_lds(key, sorted, n0);

  // Running sums of value[0 .. n) one after the other (the reference's
  // order), by one thread: 16 values requested while 16 are added, up to the
  // 16 that hold the first sum that ends the walk (later ones are not written:
  // whatever is there comes after it). (A wavefront that took its lanes' values
  // in turn and tested each sum needed 50 ns for each: 1024 kept tokens of
  // 32000 130 us a draw, now 78.)
  float *value = (float*)hist, *cum = value + kTopMax;
  auto running_sums = [&](int n, auto ends) {
    __syncthreads();
    if (tid == 0) {
      constexpr int B = 16;
      float x[B], c = 0.0f;
#pragma unroll
      for (int u = 0; u < B; u++) x[u] = value[u];
      for (int at = 0; at < n; at += B) {  // (past n: values never looked at)
        float y[B];
#pragma unroll
        for (int u = 0; u < B; u++) y[u] = value[min(at + B, kTopMax - B) + u];
#pragma unroll
        for (int u = 0; u < B; u++) {
          c += x[u];
          cum[at + u] = c;
        }
        if (ends(c)) break;
#pragma unroll
        for (int u = 0; u < B; u++) x[u] = y[u];
      }
    }
    __syncthreads();
  };

  // The cut: the first k, or fewer where the running sum reaches top_p.
  const int kact = min((int)k, n0);
  if (tid == 0) kept_s = kact;
  if (p.top_p > 0.0f && p.top_p <= 1.0f) {
    if (tid < kact) value[tid] = __uint_as_float((unsigned)(sorted[tid] >> 32));
    running_sums(kact, [&](float c) { return c >= p.top_p; });
    if (tid < kact && cum[tid] >= p.top_p) atomicMin(&kept_s, tid + 1);
  }
  __syncthreads();
  const int n = kept_s;
  double ds = 0.0;
  for (int r = tid; r < n; r += kPick) ds += (double)__uint_as_float((unsigned)(sorted[r] >> 32));
  ds = block_sum_d(ds, dred);
  const bool uniform = !(ds > 0.0);  // nothing left: uniform over every token
  const float inv = uniform ? 0.0f : (float)(1.0 / ds);

  unsigned long long st = *p.rng;  // xorshift64* (source/sampler.c:79-90)
  st ^= st >> 12;
  st ^= st << 25;
  st ^= st >> 27;
  const float coin = (float)((unsigned)((st * 0x2545F4914F6CDD1Dull) >> 32) >> 8) / 16777216.0f;
  __syncthreads();  // every read of the state comes before its update
  if (tid == 0) *p.rng = st;

  if (uniform) {  // the running sums of sample_pick_kernel over equal weights
    float* pre = (float*)dred;
    const float u = 1.0f / (float)V;
    const int R = (V + kPick - 1) / kPick, lo = min(V, tid * R), hi = min(V, lo + R);
    float s = 0.0f;
    for (int i = lo; i < hi; i++) s += u;
    pre[tid] = s;
    __syncthreads();
    if (tid == 0) {
      float c = 0.0f;
      for (int t = 0; t < kPick; t++) {
        const float x = pre[t];
        pre[t] = c;
        c += x;
      }
    }
    __syncthreads();
    float cdf = pre[tid];
    for (int i = lo; i < hi; i++) {
      cdf += u;
      if (coin < cdf) {
        atomicMin(&best, i);
        break;
      }
    }
    __syncthreads();
  } else {
    // the kept tokens in index order: their keys with the halves exchanged
    for (int r = tid; r < n; r += kPick) key[r] = (sorted[r] << 32) | (sorted[r] >> 32);
    __syncthreads();
    sort_desc_lds(key, sorted, n);
    const float w = tid < n ? __uint_as_float((unsigned)sorted[tid]) * inv : 0.0f;
    if (tid < n) value[tid] = w;
    if (tid == 0) kept_s = n;  // (its value is in n)
    running_sums(n, [&](float c) { return coin < c; });
    if (tid < n && w > 0.0f && coin < cum[tid]) atomicMin(&kept_s, tid);
    __syncthreads();
    if (tid == 0 && kept_s < n) best = (int)~(unsigned)(sorted[kept_s] >> 32);
  }
  if (tid == 0) {
    const int tok = best < V ? best : V - 1;  // rounding fallback, as the reference's
    *p.out = tok;
    if (p.seq) p.seq[(*p.seq_len)++] = tok;
    if (p.pos_inc) (*p.pos_inc)++;
  }
}

// ------------------------------------------------------------ radix sort --
// Stable descending sort of (key, value) pairs: a least-significant-digit
// radix sort of the inverted keys (ascending on ~key is descending on key),
// four passes of 8-bit digits. A pass is three launches over kRsBlocks
// contiguous chunks of the input:
// * histogram: the digit counts of each chunk, stored bin-major
//   (hist[digit][chunk]);
// * scan: one block turns them into exclusive offsets in that order, so a
//   digit's elements of chunk c land after those of chunks < c;
// * scatter: each chunk, in tiles of kRsThreads elements in input order,
//   ranks every element among the equal digits of its tile (within a
//   wavefront by ballots over the digit's bits, across wavefronts by
//   per-wavefront counts) and writes it at its digit's running offset.
// Every step keeps input order among equal digits, hence the stability.
constexpr int kRsThreads = 256;
constexpr int kRsWaves = kRsThreads / WAVE;
constexpr int kRsBlocks = 64;
constexpr int kRsBins = 256;
constexpr int kRsScan = 1024;  // threads of the scan: kRsBins * kRsBlocks / kRsScan entries each
static_assert(kRsBins * kRsBlocks % kRsScan == 0, "scan partition");

__device__ __forceinline__ int rs_chunk(int n) { return (n + kRsBlocks - 1) / kRsBlocks; }
__device__ __forceinline__ unsigned rs_digit(unsigned key, int shift) { return (~key >> shift) & (kRsBins - 1); }

__global__ __launch_bounds__(kRsThreads) void rs_hist_kernel(const unsigned* keys, int n, int shift,
                                                           unsigned* hist) {
  __shared__ unsigned h[kRsBins];
  for (int i = threadIdx.x; i < kRsBins; i += kRsThreads) h[i] = 0u;
  __syncthreads();
  const int ch = rs_chunk(n), lo = min(n, (int)blockIdx.x * ch), hi = min(n, lo + ch);
  for (int i = lo + threadIdx.x; i < hi; i += kRsThreads) atomicAdd(&h[rs_digit(keys[i], shift)], 1u);
  __syncthreads();
  for (int d = threadIdx.x; d < kRsBins; d += kRsThreads) hist[d * kRsBlocks + blockIdx.x] = h[d];
}

// Exclusive scan of the kRsBins * kRsBlocks counts in place: each thread a
// run of consecutive entries, then a scan of the runs' sums in thread order.
__global__ __launch_bounds__(kRsScan) void rs_scan_kernel(unsigned* hist) {
  constexpr int PER = kRsBins * kRsBlocks / kRsScan;
  __shared__ unsigned run[2][kRsScan];
  const int t = threadIdx.x;
  unsigned v[PER], sum = 0u;
#pragma unroll
  for (int i = 0; i < PER; i++) {
    v[i] = hist[t * PER + i];
    sum += v[i];
  }
  int cur = 0;
  run[0][t] = sum;
  __syncthreads();
  for (int off = 1; off < kRsScan; off <<= 1) {  // inclusive scan of the run sums
    const unsigned add = t >= off ? run[cur][t - off] : 0u;
    run[cur ^ 1][t] = run[cur][t] + add;
    cur ^= 1;
    __syncthreads();
  }
  unsigned base = run[cur][t] - sum;
#pragma unroll
  for (int i = 0; i < PER; i++) {
    hist[t * PER + i] = base;
    base += v[i];
  }
}

__global__ __launch_bounds__(kRsThreads) void rs_scatter_kernel(const unsigned* kin, const int* vin, int n,
                                                              int shift, const unsigned* offs, unsigned* kout,
                                                              int* vout) {
  __shared__ unsigned base[kRsBins];           // the digits' running output offsets
  __shared__ unsigned cnt[kRsWaves][kRsBins];  // a tile's digit counts per wavefront, then their prefixes
  __shared__ unsigned tot[kRsBins];            // a tile's digit counts
  const int tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE;
  for (int e = tid; e < kRsBins; e += kRsThreads) base[e] = offs[e * kRsBlocks + blockIdx.x];
  const int ch = rs_chunk(n), lo = min(n, (int)blockIdx.x * ch), hi = min(n, lo + ch);
  const unsigned long long below = (1ull << lane) - 1ull;  // the lanes before this one
  for (int t0 = lo; t0 < hi; t0 += kRsThreads) {
    for (int e = tid; e < kRsWaves * kRsBins; e += kRsThreads) cnt[e / kRsBins][e % kRsBins] = 0u;
    __syncthreads();
    const int i = t0 + tid;
    const bool valid = i < hi;  // the invalid lanes are the tile's last ones
    const unsigned key = valid ? kin[i] : 0u;
    const int val = valid ? (vin ? vin[i] : i) : 0;
    const unsigned d = rs_digit(key, shift);
    // the lanes of this wavefront holding the same digit
    unsigned long long same = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; b++) {
      const unsigned long long ones = __ballot((d >> b) & 1u);
      same &= ((d >> b) & 1u) ? ones : ~ones;
    }
    const unsigned rank = (unsigned)__popcll(same & below), group = (unsigned)__popcll(same);
    if (valid && rank == group - 1u) cnt[wave][d] = group;  // the group's last lane
    __syncthreads();
    for (int e = tid; e < kRsBins; e += kRsThreads) {  // prefixes over the wavefronts in order
      unsigned r = 0u;
#pragma unroll
      for (int w = 0; w < kRsWaves; w++) {
        const unsigned c = cnt[w][e];
        cnt[w][e] = r;
        r += c;
      }
      tot[e] = r;
    }
    __syncthreads();
    if (valid) {
      const unsigned pos = base[d] + cnt[wave][d] + rank;
      kout[pos] = key;
      vout[pos] = val;
    }
    __syncthreads();  // every read of base and cnt for this tile is done
    for (int e = tid; e < kRsBins; e += kRsThreads) base[e] += tot[e];
  }
}

}  // namespace

size_t sample_sort_temp_bytes(int V) {
  // a key and a value buffer for the passes between the input and the
  // output, and the digit counts
  return (size_t)V * (sizeof(unsigned) + sizeof(int)) + (size_t)kRsBins * kRsBlocks * sizeof(unsigned) + 256;
}

void sort_pairs_desc(const unsigned* keys, const int* vals, int n, unsigned* keys_out, int* vals_out, void* temp,
                     hipStream_t s) {
  if (n < 0 || n > kSortMax) ST_DIE("sort_pairs_desc: n out of range");
  if (n == 0) return;
  unsigned* tk = (unsigned*)temp;
  int* tv = (int*)(tk + n);
  unsigned* hist = (unsigned*)(((uintptr_t)(tv + n) + 255) & ~(uintptr_t)255);
  // passes 0..3: input -> temp -> output -> temp -> output
  const unsigned* kin = keys;
  const int* vin = vals;
  for (int pass = 0; pass < 4; pass++) {
    unsigned* ko = pass % 2 ? keys_out : tk;
    int* vo = pass % 2 ? vals_out : tv;
    const int shift = 8 * pass;
    hipLaunchKernelGGL(rs_hist_kernel, dim3(kRsBlocks), dim3(kRsThreads), 0, s, kin, n, shift, hist);
    hipLaunchKernelGGL(rs_scan_kernel, dim3(1), dim3(kRsScan), 0, s, hist);
    hipLaunchKernelGGL(rs_scatter_kernel, dim3(kRsBlocks), dim3(kRsThreads), 0, s, kin, vin, n, shift, hist, ko,
                       vo);
    kin = ko;
    vin = vo;
  }
  HIP_CHECK(hipGetLastError());
}

void sample(const SampleParams& p, hipStream_t s) {
  if (p.V <= 0) ST_DIE("sample needs a vocabulary");
  if (!(p.temperature >= 0.0f)) ST_DIE("sampling temperature must be >= 0");
  if (p.top_k < 0) ST_DIE("sampling top_k must be >= 0");
  const bool greedy = p.temperature == 0.0f;
  const bool top = !greedy && p.top_k > 0 && p.top_k <= kTopMax && p.top_k < p.V;
  // (the sort's scratch holds the candidate count)
  if (!greedy && (p.top_k > 0 || (p.top_p > 0.0f && p.top_p <= 1.0f)) &&
      p.sort_temp_bytes < sample_sort_temp_bytes(p.V))
    ST_DIE("sample: sort scratch too small");
  unsigned* count = top ? (unsigned*)p.sort_temp : nullptr;
  hipLaunchKernelGGL(sample_scale_kernel, dim3(kSB), dim3(kST), 0, s, p, count);
  if (top) {
    hipLaunchKernelGGL(sample_exp_top_kernel, dim3(kSB), dim3(kST), 0, s, p, count);
    hipLaunchKernelGGL(sample_draw_kernel, dim3(1), dim3(kPick), 0, s, p, count);
    HIP_CHECK(hipGetLastError());
    return;
  }
  if (greedy) {
    ArgmaxParams a{};
    a.x = p.y;
    a.n = p.V;
    a.part_v = p.argmax_v;
    a.part_i = p.argmax_i;
    a.out = p.out;
    a.seq = p.seq;
    a.seq_len = p.seq_len;
    a.pos_inc = p.pos_inc;
    argmax(a, s);
    return;
  }
  const bool filter = p.top_k > 0 || (p.top_p > 0.0f && p.top_p <= 1.0f);
  SampleParams q = p;
  if (!filter) q.keys = nullptr;  // keep every token: no sort
  hipLaunchKernelGGL(sample_exp_kernel, dim3(kSB), dim3(kST), 0, s, q);
  hipLaunchKernelGGL(sample_norm_kernel, dim3(kSB), dim3(kST), 0, s, q);
  if (filter) {
    sort_pairs_desc(p.keys, p.vals, p.V, p.keys_sorted, p.vals_sorted, p.sort_temp, s);
  }
  hipLaunchKernelGGL(sample_select_kernel, dim3(1), dim3(kPick), 0, s, q);
  hipLaunchKernelGGL(sample_pick_kernel, dim3(1), dim3(kPick), 0, s, q);
  HIP_CHECK(hipGetLastError());
}

}  // namespace sg
