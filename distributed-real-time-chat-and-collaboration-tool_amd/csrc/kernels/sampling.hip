// Fused token sampler (gfx950): one 1024-thread workgroup (16 waves) per row.
//
//  * temperature <= 0 : greedy argmax (ties -> lowest index), one row pass.
//  * 0 < top_k <= 1024: exact top-k, then temperature softmax + top-p over the
//    k candidates.  Selection without a histogram in the common case: every
//    thread keeps the max key of the elements it streams; a threshold tau0 that
//    k of those 1024 thread maxima reach, and few more, is a lower bound on the
//    k-th largest logit, so gathering `key >= tau0` yields all top-k plus a few
//    extra, and such an element can only sit in a thread whose own max is
//    >= tau0: only those ~k threads' elements are read again, eight lanes to a
//    thread (many threads: each its own).  One row pass.  If ties push the gather
//    past 1024 slots, the row falls back to a 16-bit radix select (two histogram
//    passes) and a ballot-compacted full gather.
//    What bounds a row is the chain of its stages, and fetching code that runs
//    once a step: tau0 by one wave's ballots instead of the workgroup's
//    histograms, and a gather in a few instructions instead of one unrolled over
//    32 elements.  A row of up to 32,768 is held in registers, asked for when it
//    is known to need them: the other modes read as ever (greedy, exact top-p).
//    V 32000, top-k 64, top-p 0.95, before / now: 1 row 11.4 / 6.9 us, 256 12.0 /
//    8.2, 1024 31.4 / 22.2; V 128256, 1 row 19.7 / 13.0, 256 26.2 / 21.4, 1024
//    72.2 / 63.5.
//    Up to 128 candidates find their places by counting and are drawn from by one wave;
//    more are bitonic-sorted.  All tokens tied with the k-th value stay.
//  * top_k == 0       : temperature sampling with EXACT top-p over the whole
//    vocabulary (no candidate cap).  With p_i ~ exp(x_i / T) and
//    P = top_p * sum(p), token i is in the nucleus iff the mass of tokens
//    strictly more probable than i is < P (ties are in or out together).
//    Pivot rejection: draw j from the tokens above a pivot L (inverse CDF:
//    per-thread masses, block scan, the owning thread re-walks its own
//    elements), then one row pass computes mass(key > key_j); accept if < P,
//    else every token up to key_j is outside and L = key_j.  The same pass
//    evaluates a bisection key between L and a known-inside bound H, so the
//    pivot range halves every pass: <= ~17 passes worst case, 1-2 on real
//    distributions.  Accepted draws follow p restricted to the nucleus
//    exactly (the eligible set always contains the nucleus).
// Rows are streamed with 16-byte loads (8 bf16 per lane) when 16-B aligned.
// The random draws are counter-based hashes of (seed, step, row, round);
// `step` lives in device memory so the kernel replays inside a hipGraph.
// Keys: bf16 bit patterns mapped to unsigned 16-bit keys ordered like the
// float values, so comparisons on keys are exact comparisons on logits.
// A NaN or -inf is never drawn; a row of nothing else gets the token -1.
#include "common.h"
#include "launchers.h"

#include <type_traits>

namespace drtc {

constexpr int kSampThreads = 1024;
constexpr int kSampWaves = kSampThreads / 64;
constexpr int kCand = 1024;
constexpr int kMaxRounds = 40;

DRTC_DEVICE unsigned ord16(unsigned short b) {
  return (b & 0x8000u) ? (unsigned)(~b & 0xFFFFu) : (unsigned)(b | 0x8000u);
}
constexpr unsigned kLowKey = 0x80u, kTopKey = 0xff80u;  // keys of the numbers above -inf; NaNs lie on both sides
DRTC_DEVICE float bits2f(unsigned short b) { return __uint_as_float((unsigned)b << 16); }

DRTC_DEVICE uint64_t mix64(uint64_t x) {
  x ^= x >> 33; x *= 0xff51afd7ed558ccdULL;
  x ^= x >> 33; x *= 0xc4ceb9fe1a85ec53ULL;
  x ^= x >> 33;
  return x;
}
// uniform in (0, 1) for draw `round` of (seed, step, row)
DRTC_DEVICE float uniform(uint64_t seed, uint64_t st, int row, int round) {
  const uint64_t h = mix64(seed ^ mix64(st * 0x9E3779B97F4A7C15ULL + (uint64_t)row) +
                           (uint64_t)round * 0xD1B54A32D192ED03ULL);
  return (float)((h >> 40) + 0.5) * (1.0f / 16777216.0f);
}

// Visit this thread's elements of the row, in a fixed order: f(index, raw bf16).
// kUnroll 16-byte loads are issued before any is consumed (a lane streams
// ~16 vectors of a 128k row: one load in flight would leave the pass
// latency-bound at about half the HBM rate).
constexpr int kUnroll = 4;  // default U (one workgroup per CU)
template <int U, class F>
DRTC_DEVICE void for_row(const unsigned short* lr, int V, bool vec, F&& f) {
  const int tid = threadIdx.x;
  if (vec) {
    const int nv = V >> 3;
    for (int v = tid; v < nv; v += U * kSampThreads) {
      u16x8 x[U];
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (v + u * kSampThreads < nv)
          x[u] = *reinterpret_cast<const u16x8*>(lr + 8 * (v + u * kSampThreads));
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (v + u * kSampThreads < nv) {
#pragma unroll
          for (int j = 0; j < 8; ++j) f(8 * (v + u * kSampThreads) + j, x[u][j]);
        }
      }
    }
    for (int i = (nv << 3) + tid; i < V; i += kSampThreads) f(i, lr[i]);
  } else {
    for (int i = tid; i < V; i += kSampThreads) f(i, lr[i]);
  }
}

// A row that fits the workgroup's registers, read once: vectors of a thread in for_row's order, -inf behind the end.
constexpr int kHeld = 4, kHeldRow = 8 * kHeld * kSampThreads;
struct HeldRow {
  u16x8 x[kHeld];
  DRTC_DEVICE void load(const unsigned short* lr, int V) {
    const u16x8 none = {0xff80, 0xff80, 0xff80, 0xff80, 0xff80, 0xff80, 0xff80, 0xff80};
#pragma unroll
    for (int u = 0; u < kHeld; ++u) {
      const int v = threadIdx.x + u * kSampThreads;
      x[u] = v < V >> 3 ? *reinterpret_cast<const u16x8*>(lr + 8 * v) : none;
    }
  }
  template <class F>
  DRTC_DEVICE void operator()(F&& f) const {
#pragma unroll
    for (int u = 0; u < kHeld; ++u)
#pragma unroll
      for (int j = 0; j < 8; ++j) f(8 * ((int)threadIdx.x + u * kSampThreads) + j, x[u][j]);
  }
};
template <int U>
struct ReadRow {
  const unsigned short* lr;
  int V;
  bool vec;
  template <class F>
  DRTC_DEVICE void operator()(F&& f) const { for_row<U>(lr, V, vec, f); }
};

DRTC_DEVICE float wave_sum(float x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
  return x;
}
DRTC_DEVICE float wave_max(float x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x = fmaxf(x, __shfl_xor(x, o, 64));
  return x;
}

// Where a row's token goes: device memory, and for a step's graph the host's buffer of the staging set that it read, which
// waits for the step anyway (a copy behind the step is 4 us more).
struct TokenOut {
  int *tokens, *host;
  DRTC_DEVICE void put(int row, int token) const {
    tokens[row] = token;
    if (host) __hip_atomic_store(host + row, token, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
};

struct SampShared {
  float val[kCand];
  int idx[kCand];
  unsigned hist[kSampWaves][256];
  float wred[4][kSampWaves];
  int misc[8];
};

// Sum over the block of two values (fixed order: deterministic).
DRTC_DEVICE void block_sum2(SampShared& s, float a, float b, float& ra, float& rb) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  a = wave_sum(a);
  b = wave_sum(b);
  if (lane == 0) { s.wred[0][wid] = a; s.wred[1][wid] = b; }
  __syncthreads();
  float x = 0.f, y = 0.f;
#pragma unroll
  for (int w = 0; w < kSampWaves; ++w) { x += s.wred[0][w]; y += s.wred[1][w]; }
  __syncthreads();
  ra = x; rb = y;
}

// Exclusive block scan of v (thread order); also returns the block total and
// the highest thread index with v > 0 (-1 if none).
DRTC_DEVICE float block_excl_scan(SampShared& s, float v, float& total, int& last_pos) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  float x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const float y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  const uint64_t pos = __ballot(v > 0.f);
  if (lane == 63) {
    s.wred[2][wid] = x;
    s.wred[3][wid] = pos ? __int_as_float(wid * 64 + 63 - __clzll(pos)) : __int_as_float(-1);
  }
  __syncthreads();
  float off = 0.f, tot = 0.f;
  int lp = -1;
#pragma unroll
  for (int w = 0; w < kSampWaves; ++w) {
    const float t = s.wred[2][w];
    if (w < wid) off += t;
    tot += t;
    lp = max(lp, __float_as_int(s.wred[3][w]));
  }
  __syncthreads();
  total = tot;
  last_pos = lp;
  return off + x - v;
}

// Among 256 bins (hist[d], d = 0..255), walking from the top bin down, the bin
// where the running count reaches `remaining`: returns it in misc[0] and the
// count still needed inside it in misc[1].  Threads 0..255 take part.
DRTC_DEVICE void select_bin(SampShared& s, const unsigned* hist, int remaining) {
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  int c = 0, x = 0;
  if (tid < 256) {
    c = (int)hist[255 - tid];
    x = c;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(x, o, 64);
      if (lane >= o) x += y;
    }
    if (lane == 63) s.misc[4 + wid] = x;  // misc[4..7]: 4 wave totals
  }
  __syncthreads();
  if (tid < 256) {
    int off = 0;
    for (int w = 0; w < wid; ++w) off += s.misc[4 + w];
    const int incl = off + x, excl = incl - c;
    if (incl >= remaining && excl < remaining) { s.misc[0] = 255 - tid; s.misc[1] = remaining - excl; }
    if (tid == 255 && incl < remaining) { s.misc[0] = 0; s.misc[1] = remaining - excl; }
  }
  __syncthreads();
}

// Exact key of the k-th largest number by a 16-bit radix select (two
// histogram passes over the row; per-wave histograms).
template <int U>
DRTC_DEVICE unsigned radix_kth(SampShared& s, const unsigned short* lr, int V, bool vec, int k) {
  const int tid = threadIdx.x, wid = tid >> 6;
  unsigned prefix = 0, mask = 0;
  int remaining = k;
  for (int pass = 8; pass >= 0; pass -= 8) {
    for (int i = tid; i < kSampWaves * 256; i += kSampThreads) (&s.hist[0][0])[i] = 0;
    __syncthreads();
    unsigned* h = s.hist[wid];
    for_row<U>(lr, V, vec, [&](int, unsigned short b) {
      const unsigned key = ord16(b);
      if ((key & mask) == prefix && key <= kTopKey) atomicAdd(&h[(key >> pass) & 255u], 1u);
    });
    __syncthreads();
    if (tid < 256) {
      unsigned t = 0;
#pragma unroll
      for (int w = 1; w < kSampWaves; ++w) t += s.hist[w][tid];
      s.hist[0][tid] += t;
    }
    __syncthreads();
    select_bin(s, s.hist[0], remaining);
    prefix |= (unsigned)s.misc[0] << pass;
    mask |= 255u << pass;
    remaining = s.misc[1];
    __syncthreads();
  }
  return prefix;
}

// Gather every number with key >= thr into s.val / s.idx (ballot-compacted);
// returns the number found (may exceed kCand: only the first kCand are kept).
template <int U>
DRTC_DEVICE int gather_ge(SampShared& s, const unsigned short* lr, int V, bool vec, unsigned thr) {
  const int tid = threadIdx.x, lane = tid & 63;
  if (tid == 0) s.misc[2] = 0;
  s.val[tid] = -INFINITY;
  s.idx[tid] = 0x7fffffff;
  __syncthreads();
  auto put = [&](bool pred, int i, unsigned short b) {
    const uint64_t m = __ballot(pred);
    if (m == 0) return;
    const int leader = __ffsll((long long)m) - 1;
    int base = 0;
    if (lane == leader) base = atomicAdd(&s.misc[2], __popcll(m));
    base = __shfl(base, leader, 64);
    if (pred) {
      const int slot = base + __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                                        __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
      if (slot < kCand) { s.val[slot] = bits2f(b); s.idx[slot] = i; }
    }
  };
  auto in = [&](unsigned short b) { return ord16(b) - thr <= kTopKey - thr; };
  // wave-uniform trip counts (the ballots need every lane): pad to whole waves
  const int w0 = tid & ~63;
  if (vec) {
    const int nv = V >> 3;
    for (int v0 = w0; v0 < nv; v0 += U * kSampThreads) {
      u16x8 x[U];
      bool any[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int v = v0 + u * kSampThreads + lane;
        x[u] = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
        if (v < nv) x[u] = *reinterpret_cast<const u16x8*>(lr + 8 * v);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int v = v0 + u * kSampThreads + lane;
        any[u] = false;
        if (v < nv) {
#pragma unroll
          for (int j = 0; j < 8; ++j) any[u] |= in(x[u][j]);
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (__ballot(any[u]) == 0) continue;  // wave-uniform
        const int v = v0 + u * kSampThreads + lane;
#pragma unroll
        for (int j = 0; j < 8; ++j) put(v < nv && in(x[u][j]), 8 * v + j, x[u][j]);
      }
    }
    for (int i0 = (nv << 3) + w0; i0 < V; i0 += kSampThreads) {
      const int i = i0 + lane;
      const unsigned short b = i < V ? lr[i] : (unsigned short)0;
      put(i < V && in(b), i, b);
    }
  } else {
    for (int i0 = w0; i0 < V; i0 += kSampThreads) {
      const int i = i0 + lane;
      const unsigned short b = i < V ? lr[i] : (unsigned short)0;
      put(i < V && in(b), i, b);
    }
  }
  __syncthreads();
  return s.misc[2];
}

// The wave's largest in lane 63: shifts within rows of 16, then a row's last lane to the next row and the next two.
template <int... Ctrl>
DRTC_DEVICE unsigned last_max(unsigned x) {
  ((x = max(x, (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, Ctrl, 0xf, 0xf, false))), ...);
  return x;
}

// A threshold that at least k of 1024 keys reach, found by one wave that holds 16 to a lane: down from the largest in
// doubled steps, then halved, until no more than `enough` reach it or no higher one does.
DRTC_DEVICE unsigned few_above(const unsigned short* keys, int k, int enough) {
  const int lane = threadIdx.x & 63;
  u32x4 x[2];
  unsigned top = 0;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    x[i] = *reinterpret_cast<const u32x4*>(keys + 512 * i + 8 * lane);
#pragma unroll
    for (int j = 0; j < 4; ++j) top = max(top, max(x[i][j] >> 16, x[i][j] & 0xffffu));
  }
  top = last_max<0x111, 0x112, 0x114, 0x118, 0x142, 0x143>(top);
  auto reach = [&](unsigned t) {
    int n = 0;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        n += __popcll(__ballot(x[i][j] >= t << 16)) + __popcll(__ballot((unsigned short)x[i][j] >= (unsigned short)t));
    return n;
  };
  unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)top, 63) + 1, lo = hi;
  int n = 0;
  for (unsigned d = 32; n < k; d *= 2) {  // (0 is reached by all)
    hi = lo;
    lo = lo > d ? lo - d : 0;
    n = reach(lo);
  }
  while (n > enough && hi - lo > 1) {
    const unsigned mid = (lo + hi) / 2;
    const int m = reach(mid);
    if (m >= k) {
      lo = mid;
      n = m;
    } else {
      hi = mid;
    }
  }
  return lo;
}

// The rest of sample_topk for up to 128 gathered candidates, n: each finds its place by counting those
// ahead of it (8 threads to a candidate; sort: their places' keys, of rows whose indexes have 16 bits), then one wave does what
// is left, two candidates to a lane - the same sums in the same order as the form below with two barriers instead of some fifty.
constexpr int kFew = 128;
// an order of all bit patterns, zeros alike
DRTC_DEVICE unsigned place_key(float v) { return v == 0.f ? 0x8000u : ord16((unsigned short)(__float_as_uint(v) >> 16)); }
// against the largest: 1 for itself, at +inf too
DRTC_DEVICE float weight(float v, float top, float inv_t) { return v == top ? 1.f : __expf((v - top) * inv_t); }
DRTC_DEVICE void sample_few(SampShared& s, const unsigned* sort, const TokenOut& out, int row, float temp, int k, int n,
                            float pp) {
  const int tid = threadIdx.x, lane = tid & 63, own = tid >> 3;
  float* const sv = reinterpret_cast<float*>(&s.hist[8][0]);
  int* const si = reinterpret_cast<int*>(&s.hist[9][0]);
  // every candidate gets a place of its own
  if (own < n) {
    const float v = s.val[own];
    const int id = s.idx[own];
    int ahead = 0;
    if (sort) {  // (0 behind the last)
      const unsigned mine = sort[own];
#pragma unroll
      for (int i = 0; i < kFew / 32; ++i) {
        const u32x4 q = *reinterpret_cast<const u32x4*>(sort + 32 * i + 4 * (tid & 7));
        ahead += (q[0] > mine) + (q[1] > mine) + (q[2] > mine) + (q[3] > mine);
      }
    } else {
      const unsigned key = place_key(v);
      for (int j = tid & 7; j < n; j += 8) {
        const unsigned kj = place_key(s.val[j]);
        ahead += kj > key || (kj == key && s.idx[j] < id);
      }
    }
    ahead += __shfl_xor(ahead, 1, 64);
    ahead += __shfl_xor(ahead, 2, 64);
    ahead += __shfl_xor(ahead, 4, 64);
    if ((tid & 7) == 0) {
      sv[ahead] = v;
      si[ahead] = id;
    }
  }
  __syncthreads();
  if (tid >= 64) return;
  const unsigned kth = place_key(sv[min(k, n) - 1]);
  float x[2], lo[2];
  int total_n = 0;
#pragma unroll
  for (int z = 0; z < 2; ++z)  // ties with the k-th value stay
    total_n += __popcll(__ballot(lane + 64 * z < n && place_key(sv[min(lane + 64 * z, n - 1)]) >= kth));
  n = total_n;
  const float top = sv[0], inv_t = 1.f / temp;
#pragma unroll
  for (int z = 0; z < 2; ++z) x[z] = lane + 64 * z < n ? weight(sv[min(lane + 64 * z, n - 1)], top, inv_t) : 0.f;
  // inclusive scan over the next power of two
  for (int off = 1; off < n; off <<= 1) {
    const float a = off < 64 ? __shfl_up(x[0], off, 64) : 0.f, b = off < 64 ? __shfl_up(x[1], off, 64) : 0.f;
    const float c = __shfl(x[0], (lane + 64 - off) & 63, 64);  // for the second half
    x[1] += off < 64 && lane >= off ? b : c;
    x[0] += off < 64 && lane >= off ? a : 0.f;
  }
  lo[0] = __shfl_up(x[0], 1, 64);
  lo[1] = __shfl_up(x[1], 1, 64);
  const float mid = __shfl(x[0], 63, 64);
  if (lane == 0) {
    lo[0] = 0.f;
    lo[1] = mid;
  }
  const float total = __shfl(n > 64 ? x[1] : x[0], (n - 1) & 63, 64), need = pp * total;
  int cut = n - 1;
#pragma unroll
  for (int z = 1; z >= 0; --z) {
    const int i = lane + 64 * z;
    const uint64_t hit = __ballot(i < n && x[z] >= need && (i == 0 || lo[z] < need));
    if (hit) cut = 64 * z + __ffsll((unsigned long long)hit) - 1;
  }
  const float target = s.wred[0][0] * __shfl(cut >= 64 ? x[1] : x[0], cut & 63, 64);  // (the draw)
  int at = 0;  // (the first, where a temperature that is no number leaves no weights)
#pragma unroll
  for (int z = 0; z < 2; ++z) {
    const int i = lane + 64 * z;
    const uint64_t hit = __ballot(i <= cut && target >= lo[z] && (target < x[z] || i == cut));
    if (hit) at = 64 * z + 63 - __clzll((long long)hit);
  }
  if (lane == 0) out.put(row, si[at]);
}

constexpr int kAlike = 112;  // thresholds of any k up to this one let as many threads through
// each: visits the thread's elements of the row
template <int U, class Row>
DRTC_DEVICE void sample_topk(SampShared& s, const TokenOut& out, const Row& each, const unsigned short* lr, int V,
                             bool vec, int row, float temp, int k, float pp, uint64_t seed,
                             uint64_t st) {
  const int tid = threadIdx.x, lane = tid & 63;
  // ---- pass 1: per-thread max key; tau0: reached by k of the thread maxima, by few more where it can be
  float most = -INFINITY;  // (of floats: NaNs drop out, and +0 is above -0 as in the keys)
  each([&](int, unsigned short b) { most = fmaxf(most, bits2f(b)); });
  const unsigned tm = ord16((unsigned short)(__float_as_uint(most) >> 16));
  // hist doubles as a buffer of 1024 keys, of the threads that are looked at again, and of the candidates' sort keys
  int* const again = reinterpret_cast<int*>(&s.hist[4][0]);
  unsigned* const sort = V <= 0x10000 ? &s.hist[12][0] : nullptr;
  s.hist[12 + tid / 256][tid & 255] = 0;
  if (tid == 64) s.wred[0][0] = uniform(seed, st, row, 0);
  if (tid == 0) s.misc[2] = s.misc[3] = 0;
  const bool many = k > kAlike && (k > 224 || V <= 16384);
  if (many) {
    s.val[tid] = -INFINITY;
    s.idx[tid] = 0x7fffffff;
  }
  unsigned short* const h = reinterpret_cast<unsigned short*>(&s.hist[0][0]);
  h[tid] = (unsigned short)tm;
  __syncthreads();
  if (tid < 64) {
    // c of 1024 threads reach a threshold by about -1024 log(1 - c / 1024) elements: as many as are likely to fit 128 candidates
    // (sample_few), 256 or 512 (powers of two, the sort).  No more than k threads with elements: all of them are looked at.
    const int full = vec ? V >> 3 : V;
    const int enough = full < 768 ? k : k <= kAlike ? kAlike : k <= 214 ? 214 : k <= 384 ? 384 : k;
    const unsigned t = full <= k ? 0 : few_above(h, k, enough);
    if (tid == 0) s.misc[0] = (int)t;
  }
  __syncthreads();
  const unsigned prefix = max((unsigned)s.misc[0], kLowKey);
  // places in a list for the lanes of m, counted by one atomic for the wave
  auto places = [&](int* count, int n) {
    int base = 0;
    if (lane == 0) base = atomicAdd(count, n);
    return __builtin_amdgcn_readfirstlane(base);
  };
  auto below = [](uint64_t m) { return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u)); };
  // ---- gather key >= tau0 (>= k elements by construction, or all numbers).  Such an element can only sit in a thread
  // whose own max is >= tau0.  Few threads: of their elements (about k of the 1024) every lane takes a few of one's, eight
  // lanes to a thread, 128 threads at a time.  Many: each looks through its own, which is one turn, where the lanes would
  // wait for the memory several times, or be idle where a thread has a vector or two.  256 rows, us by lanes / by threads: V
  // 8000, k 200 15.5 / 14.8, k 300 19.2 / 17.1; V 16000, k 250 19.2 / 18.0; V 32000, k 200 16.2 / 18.8, k 1000 53.7 / 51.7; V
  // 50304, k 250 23.2 / 22.3; V 128256, k 200 29.2 / 33.0, k 500 46.7 / 42.3, k 1000 139 / 130.
  if (many) {
    if (tm >= prefix) for_row<U>(lr, V, vec, [&](int i, unsigned short b) {
      if (ord16(b) - prefix <= kTopKey - prefix) {  // key in [prefix, kTopKey]
        const int slot = atomicAdd(&s.misc[2], 1);
        if (slot < kCand) { s.val[slot] = bits2f(b); s.idx[slot] = i; }
      }
    });
  } else {
    if (const uint64_t m = __ballot(tm >= prefix)) {
      const int at = places(&s.misc[3], __popcll(m)) + below(m);
      if (tm >= prefix) again[at] = tid;
    }
    __syncthreads();
    const int threads = s.misc[3], nv = vec ? V >> 3 : 0;
    // N elements from index i on, those that are `in` the row
    auto take = [&](auto count, int i, bool in) {
      constexpr int N = decltype(count)::value;
      typedef unsigned short Some __attribute__((ext_vector_type(N)));
      Some x = {};
      if (in) x = *reinterpret_cast<const Some*>(lr + i);
      uint64_t m[N];
      int n = 0;
#pragma unroll
      for (int j = 0; j < N; ++j) {
        m[j] = __ballot(in && ord16(x[j]) - prefix <= kTopKey - prefix);  // key in [prefix, kTopKey]
        n += __popcll(m[j]);
      }
      if (n == 0) return;
      int base = places(&s.misc[2], n);
#pragma unroll
      for (int j = 0; j < N; ++j) {
        const int slot = base + below(m[j]);
        if ((m[j] >> lane & 1) && slot < kCand) {
          const float v = bits2f(x[j]);
          s.val[slot] = v;
          s.idx[slot] = i + j;
          if (sort) sort[slot] = place_key(v) << 16 | (0xffffu - (unsigned)(i + j));
        }
        base += __popcll(m[j]);
      }
    };
#pragma unroll 1
    for (int g = 0; g < threads; g += kSampThreads / 8) {
      const bool on = g + (tid >> 3) < threads;
      const int t = on ? again[g + (tid >> 3)] : 0;
#pragma unroll 1
      for (int v = 0; v < nv; v += 4 * kSampThreads) {
        const int at = v + t + (tid >> 1 & 3) * kSampThreads;
        take(std::integral_constant<int, 4>{}, 8 * at + 4 * (tid & 1), on && at < nv);
      }
#pragma unroll 1
      for (int e = 8 * nv; e < V; e += 8 * kSampThreads) {
        const int at = e + t + (tid & 7) * kSampThreads;
        take(std::integral_constant<int, 1>{}, at, on && at < V);
      }
    }
  }
  __syncthreads();
  int n = s.misc[2];
  const unsigned* gathered = many ? nullptr : sort;  // (nor by gather_ge)
  if (n > kCand) {  // heavy ties: exact k-th key by radix select, gather again
    const unsigned thr = radix_kth<U>(s, lr, V, vec, k);
    n = min(gather_ge<U>(s, lr, V, vec, thr), kCand);
    gathered = nullptr;
  }
  if (n == 0) {
    if (tid == 0) out.put(row, -1);
    return;
  }
  if (n <= kFew) {
    sample_few(s, gathered, out, row, temp, k, n, pp);
    return;
  }
  int np2 = 1;
  while (np2 < n) np2 <<= 1;
  if (!many) {
    if (tid >= n) {
      s.val[tid] = -INFINITY;
      s.idx[tid] = 0x7fffffff;
    }
    __syncthreads();
  }
  // ---- bitonic sort, descending (ties -> lower index first)
  for (int size = 2; size <= np2; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      const int j = tid ^ stride;
      if (tid < np2 && j > tid) {
        const bool desc = ((tid & size) == 0);
        const float a = s.val[tid], b = s.val[j];
        const int ia = s.idx[tid], ib = s.idx[j];
        const bool a_first = (a > b) || (a == b && ia < ib);
        if (desc != a_first) {
          s.val[tid] = b; s.val[j] = a;
          s.idx[tid] = ib; s.idx[j] = ia;
        }
      }
      __syncthreads();
    }
  }
  // keep exactly the elements >= the k-th value (ties with it included)
  const float kth = s.val[min(k, n) - 1];
  {
    const bool edge = tid < n && s.val[tid] >= kth && (tid + 1 == n || s.val[tid + 1] < kth);
    if (edge) s.misc[3] = tid + 1;
  }
  __syncthreads();
  n = s.misc[3];
  np2 = 1;
  while (np2 < n) np2 <<= 1;
  // ---- softmax + top-p + draw over the n candidates
  const float top = s.val[0];
  const float inv_t = 1.f / temp;
  const float pv = (tid < n) ? weight(s.val[tid], top, inv_t) : 0.f;
  __syncthreads();
  s.val[tid] = pv;
  __syncthreads();
  for (int off = 1; off < np2; off <<= 1) {  // inclusive Hillis-Steele scan
    const float add = (tid >= off && tid < np2) ? s.val[tid - off] : 0.f;
    __syncthreads();
    s.val[tid] += add;
    __syncthreads();
  }
  const float total = s.val[n - 1];
  if (tid == 0) {
    s.misc[3] = n - 1;
    s.misc[0] = 0;  // (the first, where a temperature that is no number leaves no weights)
  }
  __syncthreads();
  {
    const float need = pp * total;
    const bool hit = tid < n && s.val[tid] >= need && (tid == 0 || s.val[tid - 1] < need);
    if (hit) s.misc[3] = tid;
  }
  __syncthreads();
  const int cut = s.misc[3];
  const float target = uniform(seed, st, row, 0) * s.val[cut];
  if (tid <= cut) {
    const float lo = (tid == 0) ? 0.f : s.val[tid - 1];
    if (target >= lo && (target < s.val[tid] || tid == cut)) s.misc[0] = tid;
  }
  __syncthreads();
  if (tid == 0) out.put(row, s.idx[s.misc[0]]);
}

template <int U>
DRTC_DEVICE void sample_topp_full(SampShared& s, const TokenOut& out, const unsigned short* lr, int V,
                                  bool vec, int row, float temp, float pp, uint64_t seed,
                                  uint64_t st) {
  const int tid = threadIdx.x;
  const float inv_t = 1.f / temp;
  // ---- pass 1: row max and per-thread softmax mass (online, 8 at a time)
  float m_t = -INFINITY, s_t = 0.f;
  for_row<U>(lr, V, vec, [&](int, unsigned short b) {
    const float x = bits2f(b);
    if (!(x > -INFINITY)) return;  // -inf (masked) or NaN: zero mass
    if (x > m_t) {
      s_t = s_t * __expf((m_t - x) * inv_t) + 1.f;
      m_t = x;
    } else {
      s_t += __expf((x - m_t) * inv_t);
    }
  });
  const int lane = tid & 63, wid = tid >> 6;
  float wm = wave_max(m_t);
  if (lane == 0) s.wred[0][wid] = wm;
  __syncthreads();
  float m = -INFINITY;
#pragma unroll
  for (int w = 0; w < kSampWaves; ++w) m = fmaxf(m, s.wred[0][w]);
  __syncthreads();
  float e = (s_t > 0.f) ? s_t * __expf((m_t - m) * inv_t) : 0.f;  // eligible mass, this thread
  float Z, dummy;
  block_sum2(s, e, 0.f, Z, dummy);
  const float P = pp * Z;
  unsigned L = 0;                                     // eligible: key > L (0 = every finite key)
  unsigned H = ord16(__float_as_uint(m) >> 16);       // keys >= H are inside the nucleus
  bool l_open = true;                                 // L not yet set: everything eligible
  for (int round = 0; round < kMaxRounds; ++round) {
    // ---- draw j from the eligible set
    float E;
    int last_pos;
    if (tid == 0) s.misc[0] = -1;
    const float excl = block_excl_scan(s, e, E, last_pos);  // (barriers inside)
    const float target = uniform(seed, st, row, round) * E;
    // the owning thread re-walks its own elements in the pass order
    auto walk = [&](float tgt) {
      float acc = excl;
      int pick = -1, last = -1;
      unsigned pk = 0, lk = 0;
      for_row<U>(lr, V, vec, [&](int i, unsigned short b) {
        const unsigned key = ord16(b);
        const float x = bits2f(b);
        if (pick < 0 && (l_open || key > L) && x > -INFINITY) {
          acc += __expf((x - m) * inv_t);
          last = i; lk = key;
          if (acc > tgt) { pick = i; pk = key; }
        }
      });
      if (pick < 0) { pick = last; pk = lk; }
      s.misc[0] = pick;
      s.misc[1] = (int)pk;
    };
    if (e > 0.f && target >= excl && target < excl + e) walk(target);
    __syncthreads();
    if (s.misc[0] < 0 && tid == last_pos) walk(INFINITY);  // rounding at the scan edges
    __syncthreads();
    const int j = s.misc[0];
    const unsigned kj = (unsigned)s.misc[1];
    __syncthreads();
    if (pp >= 1.f || kj >= H || round == kMaxRounds - 1) {
      if (tid == 0) out.put(row, j);
      return;
    }
    // ---- verify: mass above key_j, plus the bisection key between L and H
    const unsigned lo = l_open ? 0u : L;
    const unsigned t = lo + ((H - lo) >> 1);
    const bool bis = t > lo && t < H && t != kj;
    float a_t = 0.f, f_t = 0.f;
    for_row<U>(lr, V, vec, [&](int, unsigned short b) {
      const unsigned key = ord16(b);
      const float w = __expf((bits2f(b) - m) * inv_t);
      a_t += key > kj ? w : 0.f;
      f_t += key > t ? w : 0.f;
    });
    float A, F;
    block_sum2(s, a_t, f_t, A, F);
    if (A != A || F != F) {  // NaNs among the logits: once more without them
      a_t = f_t = 0.f;
      for_row<U>(lr, V, vec, [&](int, unsigned short b) {
        const unsigned key = ord16(b);
        const float w = bits2f(b) > -INFINITY ? __expf((bits2f(b) - m) * inv_t) : 0.f;
        a_t += key > kj ? w : 0.f;
        f_t += key > t ? w : 0.f;
      });
      block_sum2(s, a_t, f_t, A, F);
    }
    if (A < P) {  // token j is inside the nucleus
      if (tid == 0) out.put(row, j);
      return;
    }
    // key_j and everything below it is outside
    L = kj; l_open = false; e = a_t;
    if (bis) {
      if (F >= P) {
        if (t > L) { L = t; e = f_t; }
      } else {
        H = min(H, t);
      }
    }
  }
}

// OCC = 1: one 1024-thread workgroup per CU (91 VGPRs, 4-deep load unroll); OCC = 2: two
// (<= 64 VGPRs, 2-deep unroll), so one row's selection tail (scans, block reductions,
// barriers) overlaps another row's stream on the same CU.
template <int OCC, bool HELD>
__global__ __launch_bounds__(kSampThreads, 4 * OCC) void sample_kernel(
    int* __restrict__ out_tokens, const bf16_t* __restrict__ logits, int V,
    int ld, const float* __restrict__ temperature, const int* __restrict__ top_k,
    const float* __restrict__ top_p, uint64_t seed,
    const int64_t* __restrict__ step, SampleMirror mirror) {
  constexpr int U = OCC == 1 ? kUnroll : 2;
  const int row = blockIdx.x;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wid = tid >> 6;
  const unsigned short* lr = (const unsigned short*)(logits + (int64_t)row * ld);
  const bool vec = ((reinterpret_cast<uintptr_t>(lr) & 15) == 0);
  const float temp = temperature ? temperature[row] : 0.f;
  const TokenOut out{out_tokens, mirror.turn ? mirror.host[~*mirror.turn & 1] : nullptr};  // (the turn is the next step's)
  __shared__ SampShared s;

  if (temp <= 0.f) {  // ---------------------------------- greedy argmax
    float best = -INFINITY;
    int bi = 0x7fffffff;
    for_row<U>(lr, V, vec, [&](int i, unsigned short b) {
      const float v = bits2f(b);
      if (v > best || (v == best && i < bi)) { best = v; bi = i; }
    });
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float ov = __shfl_xor(best, o, 64);
      const int oi = __shfl_xor(bi, o, 64);
      if (ov > best || (ov == best && oi < bi)) { best = ov; bi = oi; }
    }
    if (lane == 0) { s.val[wid] = best; s.idx[wid] = bi; }
    __syncthreads();
    if (tid == 0) {
      for (int w = 1; w < kSampWaves; ++w)
        if (s.val[w] > best || (s.val[w] == best && s.idx[w] < bi)) { best = s.val[w]; bi = s.idx[w]; }
      out.put(row, bi < V ? bi : -1);
    }
    return;
  }
  // Nothing of a row is asked for ahead of these two: held for a row that turned out greedy or of exact top-p, 64 registers
  // spilled (1024 rows of 32,000 with top-p alone 62 -> 77 us, of 512 22 -> 33, greedy 8.4 -> 15.7), and the round trip that
  // it saves is 0.4 us of a row.  k behind the greedy rows, which would wait for it (1024 x 32000 18.6 / 19.0).
  int k = top_k ? top_k[row] : 0;
  if (k >= V) k = 0;
  const uint64_t st = step ? (uint64_t)step[0] : 0ull;
  const float asked = top_p ? top_p[row] : 1.f, pp = asked > 0.f && asked < 1.f ? asked : 1.f;
  if (k > 0) {
    using Row = std::conditional_t<HELD, HeldRow, ReadRow<U>>;
    Row each;
    if constexpr (HELD) each.load(lr, V);
    else each = {lr, V, vec};
    sample_topk<U>(s, out, each, lr, V, vec, row, temp, min(k, kCand), pp, seed, st);
  } else {
    sample_topp_full<U>(s, out, lr, V, vec, row, temp, pp, seed, st);
  }
}

// The start of a decode step: each row's token, from the last step's samples (src >= 0) or from the host,
// and the step's position in the random stream, which the next step's start finds advanced.  One launch
// in place of compare, clamp, index_select, where and add, 3 to 5 us each between two kernels of a graph.
__global__ __launch_bounds__(256) void step_begin_kernel(int* __restrict__ ids, const int64_t* __restrict__ src,
                                                         const int* __restrict__ sampled,
                                                         const int* __restrict__ host, int B,
                                                         int64_t* __restrict__ counter,
                                                         int64_t* __restrict__ position) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < B) {
    const int64_t s = src[i];
    ids[i] = s < 0 ? host[i] : s < B ? sampled[s] : -1;  // -1: no such row, and no such token
  }
  if (i == 0) {
    const int64_t c = *counter;
    *position = c;
    *counter = c + 1;
  }
}

// A step's inputs from pinned host memory: the words of a few ranges, as far as the batch uses them, read over the bus by
// the chip itself, at system scope (nothing of the step before stays in a cache).  A copy of the whole staging buffer is
// handed to the copy engines from some ten kilobytes on, which the chain of a step waits for.
DRTC_DEVICE unsigned host_word(const unsigned* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
DRTC_DEVICE void stage_words(unsigned* dst, const unsigned* host, unsigned first, unsigned words, unsigned blk) {
  const unsigned i = blk * kStageWords + threadIdx.x;
  unsigned v[4];
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (i + 256 * j < words) v[j] = host_word(host + first + i + 256 * j);
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (i + 256 * j < words) dst[first + i + 256 * j] = v[j];
}
// The table's first `ahead` columns, of all rows, which wait for no length.
DRTC_DEVICE void stage_ahead(unsigned* dst, const unsigned* host, const StageTable& t, unsigned blk) {
  const unsigned e = blk * kStageWords + threadIdx.x, words = t.rows * t.ahead;
  if (t.ahead == t.columns) {
    stage_words(dst, host, t.first, words, blk);
    return;
  }
  unsigned at[4], v[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const unsigned row = (e + 256 * j) / t.ahead;
    at[j] = t.first + row * t.columns + (e + 256 * j - row * t.ahead);
    if (e + 256 * j < words) v[j] = host_word(host + at[j]);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (e + 256 * j < words) dst[at[j]] = v[j];
}
// The others as far as the rows' lengths say, 16 rows to a workgroup: 16 lanes a row take every chunks-th kStageChunk columns
// from `chunk` on.  The lengths are one request of the workgroup: many workgroups ask for the same ones, and the bus
// serves requests for a line one after the other.
DRTC_DEVICE void stage_rest(unsigned* dst, const unsigned* host, const StageTable& t, unsigned row, unsigned chunk) {
  __shared__ unsigned needs[16];
  if (threadIdx.x < 16) {
    const unsigned length = row + threadIdx.x < t.rows ? host_word(host + t.lengths + row + threadIdx.x) : 0;
    needs[threadIdx.x] = min(length / t.per + (length % t.per != 0), t.columns);
  }
  __syncthreads();
  const unsigned need = needs[threadIdx.x >> 4], at = t.first + (row + (threadIdx.x >> 4)) * t.columns;
  for (unsigned c = t.ahead + kStageChunk * chunk + (threadIdx.x & 15); c < need; c += kStageChunk * t.chunks) {
    unsigned v[kStageChunk / 16];
#pragma unroll
    for (unsigned j = 0; j < kStageChunk / 16; ++j)
      if (c + 16 * j < need) v[j] = host_word(host + at + c + 16 * j);
#pragma unroll
    for (unsigned j = 0; j < kStageChunk / 16; ++j)
      if (c + 16 * j < need) dst[at + c + 16 * j] = v[j];
  }
}
DRTC_DEVICE void stage_part(unsigned* dst, const unsigned* host, const StageRanges& r, unsigned blk) {
  if (blk < r.rest) {
    stage_ahead(dst, host, r.table, blk);
  } else if (blk < r.start[0]) {
    const unsigned group = (blk - r.rest) / r.table.chunks;
    stage_rest(dst, host, r.table, 16 * group, blk - r.rest - group * r.table.chunks);
  } else {
    int i = 0;
    while (blk >= r.start[i + 1]) ++i;
    stage_words(dst, host, r.first[i], r.words[i], blk - r.start[i]);
  }
}
__global__ __launch_bounds__(256) void stage_rows_kernel(unsigned* __restrict__ dst, const unsigned* host, StageRanges r) {
  stage_part(dst, host, r, blockIdx.x);
}

// The same along with the start of the step, the first node of its graph: the two staging sets take turns, and the last
// workgroup to have looked whose turn it is gives it to the other (turn: set, workgroups that have looked).  Steps, us, with the
// copies and step_begin / with this and the sampler's own writes to the host: one row 190.1 / 187.6, alone on the chip 211 /
// 204; 224 of 256 rows 627 / 612, 64 of 64 597 / 582.
__global__ __launch_bounds__(256) void step_stage_kernel(unsigned* __restrict__ dst, const unsigned* host0, const unsigned* host1,
                                                         StageRanges r, StepTokens t, int* turn) {
  // One wave reads the turn for its workgroup, and counts it when it has it: no read is left that the next turn could
  // overtake.  (Read by every wave, a barrier behind the read and a count behind that do not make the other waves' reads
  // complete: a barrier waits for no load from memory.)
  __shared__ int whose;
  int turn_now = 0;
  if (threadIdx.x < 64) turn_now = __hip_atomic_load(turn, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  // the tokens, the first workgroups', are what a step waits for: both sets' are on their way with the turn, one trip
  const int tokens = (t.B + 255) / 256, i = blockIdx.x * 256 + threadIdx.x;
  unsigned ahead[6];
  if (i < t.B) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const unsigned* h = k ? host1 : host0;
      ahead[3 * k] = host_word(h + t.src + 2 * i);
      ahead[3 * k + 1] = host_word(h + t.src + 2 * i + 1);
      ahead[3 * k + 2] = host_word(h + t.host + i);
    }
  }
  if (threadIdx.x == 0) whose = turn_now;
  __syncthreads();
  const int set = whose;
  if (threadIdx.x == 0 &&
      __hip_atomic_fetch_add(turn + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (int)gridDim.x - 1) {
    __hip_atomic_store(turn + 1, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(turn, set ^ 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if ((int)blockIdx.x >= tokens) {
    stage_part(dst, set & 1 ? host1 : host0, r, blockIdx.x - tokens);
    return;
  }
  if (i < t.B) {
    const unsigned lo = set & 1 ? ahead[3] : ahead[0], hi = set & 1 ? ahead[4] : ahead[1], id = set & 1 ? ahead[5] : ahead[2];
    const int64_t s = (int64_t)((uint64_t)hi << 32 | lo);
    t.ids[i] = s < 0 ? (int)id : s < t.B ? t.sampled[s] : -1;
  }
  if (i == 0) {
    const int64_t c = *t.counter;
    *t.position = c;
    *t.counter = c + 1;
  }
}

// Cuts the ranges and the table into workgroups; false: out of what the kernels take.
static bool stage_cut(const void* dst, StageRanges& r) {
  StageTable& t = r.table;
  if (r.n < 0 || r.n > kStageRanges || (uintptr_t)dst % 4 || (t.rows && (!t.per || (uint64_t)t.rows * t.columns >= 1u << 31)))
    return false;
  if (t.columns == 0) t.rows = 0;
  // ahead of the lengths: 16 KB of all rows, a fraction of a trip over the bus.  Of the rest at most 512 workgroups, or eight to
  // 16 rows, as each counts itself; more columns than they have lanes for are taken in turn.  Steps of four layers of 2048, us,
  // tables of 512 / 5120 / 32,768 tokens: 1024 rows of contexts of 150, whole rows by the copy engines 1003 / 1009 / 1071, by this
  // kernel's ranges 971 / 988 / 1418, this 968 / 969 / 973; 64 rows of 1500 413 / 415 (5120 / 32,768), 398 / 403, 396 / 396
  t.ahead = t.rows ? std::min(t.columns, std::max(16u, 4096u / t.rows)) : 1;
  const unsigned groups = t.rows && t.columns > t.ahead ? (t.rows + 15) / 16 : 0;
  t.chunks = groups ? std::min((t.columns - t.ahead + kStageChunk - 1) / kStageChunk, std::max(8u, 512u / groups)) : 1;
  r.rest = (t.rows * t.ahead + kStageWords - 1) / kStageWords;
  r.start[0] = r.rest + groups * t.chunks;
  for (int i = 0; i < r.n; ++i) r.start[i + 1] = r.start[i] + (r.words[i] + kStageWords - 1) / kStageWords;
  return true;
}

int launch_stage_rows(void* dst, const void* host, StageRanges r, hipStream_t st) {
  if (!stage_cut(dst, r) || (uintptr_t)host % 4) return -1;
  const unsigned grid = r.start[r.n];
  if (grid == 0) return 0;
  stage_rows_kernel<<<grid, 256, 0, st>>>((unsigned*)dst, (const unsigned*)host, r);
  return (int)hipGetLastError();
}

int launch_step_stage(void* dst, const void* host0, const void* host1, StageRanges r, const StepTokens& t, int* turn,
                      hipStream_t st) {
  if (!stage_cut(dst, r) || (uintptr_t)host0 % 4 || (uintptr_t)host1 % 4 || t.B <= 0) return -1;
  step_stage_kernel<<<(t.B + 255) / 256 + r.start[r.n], 256, 0, st>>>(
      (unsigned*)dst, (const unsigned*)host0, (const unsigned*)host1, r, t, turn);
  return (int)hipGetLastError();
}

int launch_step_begin(int* ids, const int64_t* src, const int* sampled, const int* host, int B, int64_t* counter,
                      int64_t* position, hipStream_t st) {
  if (B <= 0) return B == 0 ? 0 : -1;
  step_begin_kernel<<<(B + 255) / 256, 256, 0, st>>>(ids, src, sampled, host, B, counter, position);
  return (int)hipGetLastError();
}

int launch_sample(int* out_tokens, const void* logits, int B, int V, int ld,
                  const float* temperature, const int* top_k, const float* top_p,
                  uint64_t seed, const int64_t* step, const SampleMirror& mirror, hipStream_t st) {
  if (B == 0) return 0;
  if (mirror.turn && (!mirror.host[0] || !mirror.host[1])) return -1;
  // two workgroups per CU by default: B = 1024, V = 128k, top-k 64 / top-p 0.95 in 76.5 vs
  // 106.0 us, greedy 44.8 vs 58.1, full-vocabulary top-p 179 vs 237 (profiles/r3v);
  // DRTC_SAMPLER_OCC=1 restores one per CU
  static const int occ = [] {
    const char* e = getenv("DRTC_SAMPLER_OCC");
    return e && e[0] == '1' ? 1 : 2;
  }();
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(B), dim3(kSampThreads), 0, st, out_tokens, (const bf16_t*)logits, V, ld, temperature,
                       top_k, top_p, seed, step, mirror);
  };
  const bool held = V <= kHeldRow && V % 8 == 0 && ld % 8 == 0 && (uintptr_t)logits % 16 == 0;
  if (occ == 2) held ? go(sample_kernel<2, true>) : go(sample_kernel<2, false>);
  else held ? go(sample_kernel<1, true>) : go(sample_kernel<1, false>);
  return (int)hipGetLastError();
}

}  // namespace drtc
