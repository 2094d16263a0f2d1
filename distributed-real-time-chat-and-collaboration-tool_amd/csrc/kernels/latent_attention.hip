// Latent attention (gfx950): per-token key/value latents in a paged cache, a rotated key part
// shared by all heads, sliding window, softmax sinks, sigmoid gates per head.
//
// Cache row of a token (LW elements, a multiple of 32):  [ latent R | rotated key r | 0 ... ]
// 32 rows to a block.  A step runs
//   latent_prep      RMS norm of the latent, rotary on its key part and on the queries, cache
//                    write - one workgroup per token
//   prompt portions  per-head keys / values are projected up from the latents of the portion
//                    and of the window ahead of it (latent_gather + a GEMM), then varlen flash
//                    attention on MFMA (latent_prefill_kernel)
//   decode           the query is projected down into the latent space instead (head_gemm), so
//                    all heads attend to the SAME cached rows, which are both keys (all LW
//                    columns) and values (the first R): latent_decode_kernel stages each
//                    32-token block in LDS once for up to 64 heads; the result goes back up
//                    per head (head_gemm)
// bf16 runs on MFMA with the operand maps of attention_prefill.hip; sizes those do not cover,
// and fp32, run the *_any kernels.
#include "attend_any.h"
#include "hybrid_launchers.h"
#include "lds_dma.h"

#include <algorithm>

namespace drtc {

constexpr int kLB = 32;  // tokens per cache block

typedef short lat_s16x4 __attribute__((ext_vector_type(4)));
DRTC_DEVICE bf16x4 lat_read_tr16(const bf16_t* p) {
  lat_s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) lat_s16x4*)(p));
  return __builtin_bit_cast(bf16x4, v);
}
// Factor of a head's output: 1, or the sigmoid of its gate input.
template <class T>
DRTC_DEVICE float head_gate(const void* gate, int64_t at) {
  return gate ? 1.f / (1.f + expf(-to_f32(((const T*)gate)[at]))) : 1.f;
}
DRTC_DEVICE bf16x8 zero8() {
  bf16x8 z;
#pragma unroll
  for (int j = 0; j < 8; ++j) z[j] = f2bf(0.f);
  return z;
}

// ------------------------------------------------------------------ per-token preparation
// One workgroup per token.  V: elements a thread moves at once (8, or 2 where the sizes or the
// rows do not align); pairs never straddle a vector.
template <class T, int V>
DRTC_DEVICE void lat_load(float (&v)[V], const T* p) {
  if constexpr (V == 8) load8(v, p);
  else {
#pragma unroll
    for (int j = 0; j < V; ++j) v[j] = to_f32(p[j]);
  }
}
template <class T, int V>
DRTC_DEVICE void lat_store(T* p, const float (&v)[V]) {
  if constexpr (V == 8) store8(p, v);
  else {
#pragma unroll
    for (int j = 0; j < V; ++j) p[j] = from_f32<T>(v[j]);
  }
}

template <class T, int V>
DRTC_DEVICE void latent_prep_row(const LatentPrepArgs& a, int row) {
  __shared__ float red[16];
  const int tid = threadIdx.x;
  T* pr = (T*)a.proj + (int64_t)row * a.ldp;
  const T* kv = pr + a.off_kv;
  const int half = a.rot_dims >> 1;
  const float* cs = a.cos_sin + (int64_t)a.positions[row] * a.rot_dims;
  // V elements of a rotated part from element i on
  auto turn = [&](const T* src, T* dst, int i) {
    float x[V];
    lat_load<T, V>(x, src + i);
#pragma unroll
    for (int j = 0; j < V; j += 2) {
      const int k = (i + j) >> 1;
      if (k < half) {
        const float u = x[j], v = x[j + 1], c = cs[k], s = cs[half + k];
        x[j] = u * c - v * s;
        x[j + 1] = v * c + u * s;
      }
    }
    lat_store<T, V>(dst + i, x);
  };
  // queries: in place, or into the latent-space query rows
  const int dq = a.dim + a.rot;
  if (a.qa) {
    const int tail = (a.LW - a.R) / V, own = a.rot / V;
    for (int k = tid; k < a.H * tail; k += 256) {
      const int h = k / tail, i = k - h * tail;
      T* d = (T*)a.qa + ((int64_t)row * a.H + h) * a.LW + a.R;
      if (i < own) turn(pr + h * dq + a.dim, d, i * V);
      else {
#pragma unroll
        for (int j = 0; j < V; ++j) d[i * V + j] = from_f32<T>(0.f);
      }
    }
  } else {
    const int per = (a.rot_dims + V - 1) / V;
    for (int k = tid; k < a.H * per; k += 256) {
      const int h = k / per;
      T* q = pr + h * dq + a.dim;
      turn(q, q, (k - h * per) * V);
    }
  }
  if (a.off_kv < 0) return;  // the latents are another layer's
  const int64_t slot = a.slots ? a.slots[row] : -1;
  T* lat = a.lat ? (T*)a.lat + (int64_t)row * a.LW : nullptr;
  T* cache = a.cache && slot >= 0 ? (T*)a.cache + slot * a.LW : nullptr;
  float ss = 0.f;
  for (int i = tid * V; i < a.R; i += 256 * V) {
    float x[V];
    lat_load<T, V>(x, kv + i);
#pragma unroll
    for (int j = 0; j < V; ++j) ss += x[j] * x[j];
  }
  const float rinv = 1.f / sqrtf(block_sum(ss, red) / (float)a.R + a.eps);
  for (int i = tid * V; i < a.LW; i += 256 * V) {
    float x[V];
    if (i < a.R) {
      lat_load<T, V>(x, kv + i);
#pragma unroll
      for (int j = 0; j < V; ++j) x[j] *= rinv * a.norm_w[i + j];
    } else if (i < a.R + a.rot) {
      lat_load<T, V>(x, kv + i);
#pragma unroll
      for (int j = 0; j < V; j += 2) {
        const int k = (i + j - a.R) >> 1;
        if (k < half) {
          const float u = x[j], v = x[j + 1], c = cs[k], s = cs[half + k];
          x[j] = u * c - v * s;
          x[j + 1] = v * c + u * s;
        }
      }
    } else {
#pragma unroll
      for (int j = 0; j < V; ++j) x[j] = 0.f;
    }
    if (lat) lat_store<T, V>(lat + i, x);
    if (cache) lat_store<T, V>(cache + i, x);
  }
}

template <class T, int V>
__global__ __launch_bounds__(256) void latent_prep_kernel(LatentPrepArgs a) {
  latent_prep_row<T, V>(a, blockIdx.x);
}

static bool lat_prep_whole(const LatentPrepArgs& a) {  // vectors of 8
  return a.R % 8 == 0 && a.rot % 8 == 0 && a.dim % 8 == 0 && a.ldp % 8 == 0 && (a.off_kv < 0 || a.off_kv % 8 == 0) &&
         a.LW % 8 == 0;
}
static bool lat_prep_takes(const LatentPrepArgs& a) {
  return a.rot_dims <= a.rot && a.rot_dims % 2 == 0 && a.R + a.rot <= a.LW && a.R % 2 == 0 && a.rot % 2 == 0 && a.LW % 2 == 0;
}

template <class T>
static void lat_prep_t(const LatentPrepArgs& a, hipStream_t st) {
  if (lat_prep_whole(a))
    latent_prep_kernel<T, 8><<<dim3(a.rows), dim3(256), 0, st>>>(a);
  else
    latent_prep_kernel<T, 2><<<dim3(a.rows), dim3(256), 0, st>>>(a);
}

int launch_latent_prep(int f32, const LatentPrepArgs& a, hipStream_t st) {
  if (a.rows == 0) return 0;
  if (!lat_prep_takes(a)) return -1;
  if (f32) lat_prep_t<float>(a, st);
  else lat_prep_t<bf16_t>(a, st);
  return (int)hipGetLastError();
}

__global__ __launch_bounds__(256) void latent_gather_kernel(u32x4* __restrict__ out,
                                                            const u32x4* __restrict__ cache,
                                                            const int64_t* __restrict__ slots,
                                                            int64_t nvec, int vpr) {
  const int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (v >= nvec) return;
  const int64_t row = v / vpr;
  const int64_t slot = slots[row];
  u32x4 x = {0u, 0u, 0u, 0u};
  if (slot >= 0) x = cache[slot * vpr + (v - row * vpr)];
  out[v] = x;
}

int launch_latent_gather(void* out, const void* cache, const int64_t* slots, int rows,
                         int row_bytes, hipStream_t st) {
  if (rows == 0) return 0;
  if (row_bytes % 16) return -1;
  const int vpr = row_bytes / 16;
  const int64_t n = (int64_t)rows * vpr;
  latent_gather_kernel<<<dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st>>>(
      (u32x4*)out, (const u32x4*)cache, slots, n, vpr);
  return (int)hipGetLastError();
}

// ------------------------------------------------------------------ attention, any size
template <class T>
__global__ __launch_bounds__(256) void latent_prefill_any_kernel(LatentPrefillArgs a) {
  const int row = blockIdx.x, h = blockIdx.y;
  // portion of this query row (binary search over the cumulative starts)
  int lo = 0, hi = a.nseq;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (a.q_cu[mid] <= row) lo = mid; else hi = mid;
  }
  const int k0 = a.k_cu[lo];
  const int last = a.ctx[lo] + row - a.q_cu[lo];
  const int first = a.window > 0 ? max(0, last - a.window + 1) : 0;
  const T* q = (const T*)a.q + (int64_t)row * a.ldq + h * (a.dim + a.rot);
  const T* kv = (const T*)a.kv + (int64_t)k0 * a.ldkv;
  const T* lat = (const T*)a.lat + (int64_t)k0 * a.LW + a.R;
  attend_any<T>(first, last + 1, a.vdim, a.sink != nullptr, a.sink ? a.sink[h] : 0.f,
                head_gate<T>(a.gate, (int64_t)row * a.ldg + h),
                (T*)a.out + (int64_t)row * a.ldo + h * a.vdim,
                [&](int j) {
                  const T* k = kv + (int64_t)j * a.ldkv + h * a.dim;
                  float s = 0.f;
                  for (int i = 0; i < a.dim; ++i) s += to_f32(q[i]) * to_f32(k[i]);
                  const T* r = lat + (int64_t)j * a.LW;
                  for (int i = 0; i < a.rot; ++i) s += to_f32(q[a.dim + i]) * to_f32(r[i]);
                  return s * a.scale;
                },
                [&](int j, int d) {
                  return to_f32(kv[(int64_t)j * a.ldkv + a.voff + h * a.vdim + d]);
                });
}

template <class T>
__global__ __launch_bounds__(256) void latent_decode_any_kernel(LatentDecodeArgs a) {
  const int b = blockIdx.x, h = blockIdx.y;
  const int ctx = a.context_lens[b];
  T* out = (T*)a.out + ((int64_t)b * a.H + h) * a.R;
  if (ctx <= 0) {
    for (int i = threadIdx.x; i < a.R; i += 256) out[i] = from_f32<T>(0.f);
    return;
  }
  const int first = a.window > 0 ? max(0, ctx - a.window) : 0;
  const int* bt = a.block_tables + (int64_t)b * a.bt_stride;
  const T* q = (const T*)a.qa + ((int64_t)b * a.H + h) * a.LW;
  const T* cache = (const T*)a.cache;
  auto row = [&](int j) { return cache + ((int64_t)bt[j / kLB] * kLB + j % kLB) * a.LW; };
  attend_any<T>(first, ctx, a.R, a.sink != nullptr, a.sink ? a.sink[h] : 0.f,
                head_gate<T>(a.gate, (int64_t)b * a.ldg + h), out,
                [&](int j) {
                  const T* k = row(j);
                  float s = 0.f;
                  for (int i = 0; i < a.LW; ++i) s += to_f32(q[i]) * to_f32(k[i]);
                  return s * a.scale;
                },
                [&](int j, int d) { return to_f32(row(j)[d]); });
}

// ------------------------------------------------------------------ prompt portions on MFMA
// Workgroup: NW waves, QF x 16 query rows each, one head.  K tile [64 keys][DKP] (per-head part,
// then the shared rotated part) and V tile [64][DVP] in LDS, NB buffers; the next tile's global
// loads are in flight during this tile's MFMAs.  S^T = K Q^T, so its accumulators are the P^T
// operand of O^T = V^T P^T without lane movement.  QF = 2 halves the LDS reads per MFMA; NB = 1
// then leaves room for a second workgroup per CU, whose MFMAs run under this one's softmax.
constexpr int kLK = 64;

template <int DKP, int DVP, int NB>
struct LatLds {
  static constexpr int KROW = DKP + 8;
  static constexpr int VROW = DVP + 16;
  static constexpr int K_ELEMS = kLK * KROW;
  static constexpr int BUF = K_ELEMS + kLK * VROW;
  static constexpr size_t BYTES = (size_t)NB * BUF * 2;
};

template <int DKP, int DVP, int QF, int NW, int NB>
__global__ __launch_bounds__(64 * NW, NB == 1 ? 2 : 1) void latent_prefill_kernel(
    LatentPrefillArgs a) {
  using L = LatLds<DKP, DVP, NB>;
  constexpr int NTHR = 64 * NW;
  constexpr int KS = DKP / 32, NT = DVP / 16;
  constexpr int NK = kLK * (DKP / 8) / NTHR, NV = kLK * (DVP / 8) / NTHR;
  constexpr int QT = 16 * NW * QF;
  // LDS reads in flight ahead of the MFMAs, in pinned order: left alone the compiler reads two operands and waits for
  // them (192 / 128, window 1024, 256 rows: 4 x 3500 tokens of 16 heads 234 -> 220 us, 15 x 1000 of 32 386 -> 362, 8 x 300
  // of 16 21.9 -> 21.2).  128 rows have no registers for it (64 x 150 of 16 heads 73.8 -> 76.3).
  constexpr int AHEAD = NW == 8 ? 4 : 0;
  static_assert(NK * NTHR == kLK * (DKP / 8) && NV * NTHR == kLK * (DVP / 8), "staging split");
  extern __shared__ __attribute__((aligned(16))) bf16_t lat_lds[];

  const int seq = a.tile_seq[blockIdx.x], q0 = a.tile_q0[blockIdx.x], h = blockIdx.y;
  const int qb = a.q_cu[seq], n = a.q_cu[seq + 1] - qb;
  const int kb0 = a.k_cu[seq], nk = a.k_cu[seq + 1] - kb0;
  const int ctx = a.ctx[seq];
  const int w = wave_id_uniform(), lane = threadIdx.x & 63;
  const int col = lane & 15, g = lane >> 4;
  const int dq = a.dim + a.rot;
  const bf16_t* kvp = (const bf16_t*)a.kv + (int64_t)kb0 * a.ldkv;
  const bf16_t* latp = (const bf16_t*)a.lat + (int64_t)kb0 * a.LW + a.R;
  const int win = a.window > 0 ? a.window : 0x3fffffff;
  const int k_lo = max(0, ctx + q0 - win + 1);
  const int k_hi = min(nk, ctx + min(n, q0 + QT));
  const int t_lo = k_lo / kLK, t_hi = (k_hi + kLK - 1) / kLK;

  bf16x8 kr[NK], vr[NV];
  auto issue = [&](int k0) {
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      const int v = threadIdx.x + i * NTHR;
      const int key = v / (DKP / 8), c = (v % (DKP / 8)) * 8;
      bf16x8 x = zero8();
      if (k0 + key < k_hi) {
        if (c < a.dim) x = load_bf16x8(kvp + (int64_t)(k0 + key) * a.ldkv + h * a.dim + c);
        else if (c < dq) x = load_bf16x8(latp + (int64_t)(k0 + key) * a.LW + (c - a.dim));
      }
      kr[i] = x;
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int v = threadIdx.x + i * NTHR;
      const int key = v / (DVP / 8), c = (v % (DVP / 8)) * 8;
      bf16x8 x = zero8();
      if (k0 + key < k_hi && c < a.vdim)
        x = load_bf16x8(kvp + (int64_t)(k0 + key) * a.ldkv + a.voff + h * a.vdim + c);
      vr[i] = x;
    }
  };
  auto commit = [&](bf16_t* kb) {
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      const int v = threadIdx.x + i * NTHR;
      store_bf16x8(kb + (v / (DKP / 8)) * L::KROW + (v % (DKP / 8)) * 8, kr[i]);
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int v = threadIdx.x + i * NTHR;
      store_bf16x8(kb + L::K_ELEMS + (v / (DVP / 8)) * L::VROW + (v % (DVP / 8)) * 8, vr[i]);
    }
  };

  if (t_lo < t_hi) issue(t_lo * kLK);
  const int qw = q0 + 16 * QF * w;  // this wave's first query row
  bf16x8 qf[QF][KS];
#pragma unroll
  for (int f = 0; f < QF; ++f) {
    const int qr = qw + 16 * f + col;
    const bf16_t* qp = (const bf16_t*)a.q + (int64_t)(qb + qr) * a.ldq + h * dq;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int c = 32 * s + 8 * g;
      qf[f][s] = qr < n && c < dq ? load_bf16x8(qp + c) : zero8();
    }
  }
  f32x4 o[QF][NT];
  float m[QF], lsum[QF];  // m: running maximum of the unscaled scores
#pragma unroll
  for (int f = 0; f < QF; ++f) {
    m[f] = kNegBig;
    lsum[f] = 0.f;
#pragma unroll
    for (int i = 0; i < NT; ++i) o[f][i] = (f32x4){0.f, 0.f, 0.f, 0.f};
  }
  const float sl2 = a.scale * kLog2e;
  const int tr_off = ((col >> 2) + 4 * g) * L::VROW + 4 * (col & 3);

  int buf = 0;
  for (int kt = t_lo; kt < t_hi; ++kt) {
    bf16_t* kb = lat_lds + buf * L::BUF;
    const bf16_t* vb = kb + L::K_ELEMS;
    if constexpr (NB == 1) __syncthreads();
    else buf ^= 1;
    commit(kb);
    __syncthreads();
    if (kt + 1 < t_hi) issue((kt + 1) * kLK);
    const int k0 = kt * kLK;
    // nothing of this tile for this wave's queries (causal / window): skip its products
    const int q_first = ctx + qw, q_last = ctx + qw + 16 * QF - 1;
    if (k0 > q_last || k0 + kLK - 1 <= q_first - win) continue;
    const bool whole = k0 + kLK - 1 <= q_first && k0 > q_last - win;

    f32x4 sc[QF][4];
    bf16x8 kf[4 * KS];
    auto read_k = [&](int n) { kf[n] = load_bf16x8(kb + (16 * (n / KS) + col) * L::KROW + 32 * (n % KS) + 8 * g); };
#pragma unroll
    for (int n = 0; n < AHEAD; ++n) read_k(n);
#pragma unroll
    for (int n = 0; n < 4 * KS; ++n) {
      if constexpr (AHEAD > 0) __builtin_amdgcn_sched_barrier(0);
      if (n + AHEAD < 4 * KS) read_k(n + AHEAD);
      const int st = n / KS, s = n % KS;
#pragma unroll
      for (int f = 0; f < QF; ++f) {
        if (s == 0) sc[f][st] = (f32x4){0.f, 0.f, 0.f, 0.f};
        sc[f][st] = mfma16(kf[n], qf[f][s], sc[f][st]);
      }
    }
    if (!whole) {
#pragma unroll
      for (int f = 0; f < QF; ++f) {
        const int qpos = ctx + qw + 16 * f + col;
#pragma unroll
        for (int st = 0; st < 4; ++st)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int key = k0 + 16 * st + 4 * g + r;
            if (key > qpos || key <= qpos - win) sc[f][st][r] = kNegBig;
          }
      }
    }
    bf16x8 pf[QF][2];
    float alpha[QF];
    bool moved = false;
#pragma unroll
    for (int f = 0; f < QF; ++f) {
      float bmax = kNegBig;
#pragma unroll
      for (int st = 0; st < 4; ++st)
#pragma unroll
        for (int r = 0; r < 4; ++r) bmax = fmaxf(bmax, sc[f][st][r]);
      bmax = fmaxf(bmax, __shfl_xor(bmax, 16, 64));
      bmax = fmaxf(bmax, __shfl_xor(bmax, 32, 64));
      const float m_new = fmaxf(m[f], bmax);
      alpha[f] = fast_exp2((m[f] - m_new) * sl2);
      moved |= m_new > m[f];
      m[f] = m_new;
      // a row with no key in any tile so far: offset 0, so that its p are 0 (kNegBig minus a
      // rounded product of itself would not be)
      const float off = m_new > 0.5f * kNegBig ? m_new * sl2 : 0.f;
      float psum = 0.f;
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float pa = fast_exp2(sc[f][2 * ks][r] * sl2 - off);
          const float pb = fast_exp2(sc[f][2 * ks + 1][r] * sl2 - off);
          psum += pa + pb;
          pf[f][ks][r] = f2bf(pa);
          pf[f][ks][4 + r] = f2bf(pb);
        }
      lsum[f] = lsum[f] * alpha[f] + psum;
    }
    if (__any(moved)) {
#pragma unroll
      for (int f = 0; f < QF; ++f)
#pragma unroll
        for (int i = 0; i < NT; ++i) o[f][i] *= alpha[f];
    }
    bf16x8 vf[2 * NT];
    auto read_v = [&](int n) {
      const bf16_t* p = vb + tr_off + 32 * (n % 2) * L::VROW + 16 * (n / 2);
      const bf16x4 lo = lat_read_tr16(p), hi = lat_read_tr16(p + 16 * L::VROW);
#pragma unroll
      for (int j = 0; j < 4; ++j) { vf[n][j] = lo[j]; vf[n][4 + j] = hi[j]; }
    };
#pragma unroll
    for (int n = 0; n < AHEAD; ++n) read_v(n);
#pragma unroll
    for (int n = 0; n < 2 * NT; ++n) {
      if constexpr (AHEAD > 0) __builtin_amdgcn_sched_barrier(0);
      if (n + AHEAD < 2 * NT) read_v(n + AHEAD);
#pragma unroll
      for (int f = 0; f < QF; ++f) o[f][n / 2] = mfma16(vf[n], pf[f][n % 2], o[f][n / 2]);
    }
  }
#pragma unroll
  for (int f = 0; f < QF; ++f) {
    float l = lsum[f];
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    if (a.sink) l += fast_exp2(a.sink[h] * kLog2e - m[f] * sl2);
    const int qr = qw + 16 * f + col;
    if (qr < n) {
      const float inv = head_gate<bf16_t>(a.gate, (int64_t)(qb + qr) * a.ldg + h) / l;
      bf16_t* op = (bf16_t*)a.out + (int64_t)(qb + qr) * a.ldo + h * a.vdim;
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        const int d = 16 * i + 4 * g;
        if (d < a.vdim) {
          bf16x4 v;
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = f2bf(o[f][i][r] * inv);
          *reinterpret_cast<bf16x4*>(op + d) = v;
        }
      }
    }
  }
}

template <int DKP, int DVP, int QF, int NW, int NB>
static int lat_prefill_go(const LatentPrefillArgs& a, hipStream_t st) {
  latent_prefill_kernel<DKP, DVP, QF, NW, NB>
      <<<dim3(a.ntiles, a.H), dim3(64 * NW), LatLds<DKP, DVP, NB>::BYTES, st>>>(a);
  return 0;
}
template <int DKP, int DVP>
static int lat_prefill_q(const LatentPrefillArgs& a, hipStream_t st) {
  if constexpr (DKP <= 192 && DVP <= 128) {
    if (a.qtile == 256) return lat_prefill_go<DKP, DVP, 2, 8, 2>(a, st);
    if (a.qtile == 128) return lat_prefill_go<DKP, DVP, 2, 4, 1>(a, st);
  }
  return a.qtile == 64 ? lat_prefill_go<DKP, DVP, 1, 4, 2>(a, st) : -1;
}
template <int DKP>
static int lat_prefill_v(const LatentPrefillArgs& a, hipStream_t st) {
  if (a.vdim <= 64) return lat_prefill_q<DKP, 64>(a, st);
  if (a.vdim <= 128) return lat_prefill_q<DKP, 128>(a, st);
  return lat_prefill_q<DKP, 256>(a, st);
}

int launch_latent_prefill(int f32, const LatentPrefillArgs& a, hipStream_t st) {
  if (a.nseq == 0 || a.nq == 0) return 0;
  const int dq = a.dim + a.rot;
  const bool mfma = !f32 && a.dim % 8 == 0 && a.rot % 8 == 0 && a.vdim % 8 == 0 && dq <= 256 &&
                    a.vdim <= 256 && a.ldq % 8 == 0 && a.ldkv % 8 == 0 && a.voff % 8 == 0 &&
                    a.R % 8 == 0 && a.LW % 8 == 0 && a.ldo % 4 == 0;
  int rc = 0;
  if (mfma) {
    if (dq <= 64) rc = lat_prefill_v<64>(a, st);
    else if (dq <= 128) rc = lat_prefill_v<128>(a, st);
    else if (dq <= 192) rc = lat_prefill_v<192>(a, st);
    else rc = lat_prefill_v<256>(a, st);
  } else {
    if (a.vdim > 1024) return -1;
    if (f32) latent_prefill_any_kernel<float><<<dim3(a.nq, a.H), dim3(256), 0, st>>>(a);
    else latent_prefill_any_kernel<bf16_t><<<dim3(a.nq, a.H), dim3(256), 0, st>>>(a);
  }
  return rc ? rc : (int)hipGetLastError();
}

// ------------------------------------------------------------------ decode on MFMA
// Workgroup: NH head tiles of 16 x ND slices of the output dims, one wave each; grid
// (sequence, group of 16 NH heads, split of the window).  Every wave of a head tile computes
// the tile's scores (they are cheap beside the block's HBM time) and accumulates its slice of
// O^T = C^T P^T.  RT: the latent size in units of 64 (rounded up to 1, 2, 4, 8).  KSX: the
// exact number of 32-column steps of a cache row with R = 64 RT (branch-free products, loads
// batched ahead of them); 0: both at run time.
constexpr int kLatPad = 8;  // row padding: 16 rows of one b128 column start on distinct banks

// A wave's 16 heads x 64 RT / ND dims: the output, or the split's part of it.
template <int RT, int ND>
DRTC_DEVICE void lat_decode_out(const LatentDecodeArgs& a, int b, int h, int sp, int nparts, int dw, int g, int R,
                                const f32x4 (&o)[4 * RT / ND], float m, float lsum) {
  constexpr int NTW = 4 * RT / ND;
  lsum += __shfl_xor(lsum, 16, 64);
  lsum += __shfl_xor(lsum, 32, 64);
  if (h >= a.H) return;
  if (nparts == 1) {
    if (a.sink) lsum += fast_exp2(a.sink[h] * kLog2e - m);
    const float inv = head_gate<bf16_t>(a.gate, (int64_t)b * a.ldg + h) / lsum;
    bf16_t* op = (bf16_t*)a.out + ((int64_t)b * a.H + h) * R;
#pragma unroll
    for (int i = 0; i < NTW; ++i) {
      const int d = 16 * (NTW * dw + i) + 4 * g;
      if (d < R) {
        bf16x4 v;
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = f2bf(o[i][r] * inv);
        *reinterpret_cast<bf16x4*>(op + d) = v;
      }
    }
    return;
  }
  const int64_t pi = ((int64_t)b * a.H + h) * a.nsplits + sp;
#pragma unroll
  for (int i = 0; i < NTW; ++i) {
    const int d = 16 * (NTW * dw + i) + 4 * g;
    if (d < R) *reinterpret_cast<f32x4*>(a.part_o + pi * R + d) = o[i];
  }
  if (dw == 0 && g == 0) {
    a.part_ml[2 * pi] = m;
    a.part_ml[2 * pi + 1] = lsum;
  }
}

template <int RT, int NH, int ND, int KSX>
__global__ __launch_bounds__(64 * NH * ND, 2) void latent_decode_kernel(LatentDecodeArgs a) {
  constexpr int NTHR = 64 * NH * ND;
  constexpr int KSM = KSX ? KSX : 2 * RT + 2;  // 32-column steps of a cache row, at most
  constexpr int NTW = 4 * RT / ND;            // output tiles of 16 dims per wave
  constexpr int NVM = (4 * 32 * KSM + NTHR - 1) / NTHR;
  extern __shared__ __attribute__((aligned(16))) bf16_t lat_lds[];
  const int b = blockIdx.x, sp = blockIdx.z;
  const int w = wave_id_uniform(), lane = threadIdx.x & 63;
  const int hw = w / ND, dw = w % ND;
  const int col = lane & 15, g = lane >> 4;
  const int h = (blockIdx.y * NH + hw) * 16 + col;
  const int LW = KSX ? 32 * KSX : a.LW, R = KSX ? 64 * RT : a.R, ks = LW / 32, row_l = LW + kLatPad, tile_l = kLB * row_l;
  const int ctx = a.context_lens[b];
  if (ctx <= 0) {
    if (sp == 0 && h < a.H)
      for (int i = dw * 4 + g; i < R; i += 4 * ND)
        ((bf16_t*)a.out)[((int64_t)b * a.H + h) * R + i] = f2bf(0.f);
    return;
  }
  const int lo = a.window > 0 ? max(0, ctx - a.window) : 0;
  const int t0 = lo / kLB, t1 = (ctx + kLB - 1) / kLB;
  const int nparts = (t1 - t0 + a.tiles_per_split - 1) / a.tiles_per_split;
  const int tb = t0 + sp * a.tiles_per_split, te = min(t1, tb + a.tiles_per_split);
  if (tb >= te) return;
  const int* bt = a.block_tables + (int64_t)b * a.bt_stride;

  // staging: a block is kLB * LW contiguous elements; vector v goes to its padded LDS row
  const int nv = 4 * LW;
  int dst[NVM];
#pragma unroll
  for (int i = 0; i < NVM; ++i) {
    const int v = threadIdx.x + i * NTHR;
    const int r = v * 8 / LW;
    dst[i] = v * 8 + r * (row_l - LW);
  }
  bf16x8 st[NVM];
  auto issue = [&](int t) {
    const bf16_t* p = (const bf16_t*)a.cache + (int64_t)bt[t] * kLB * LW;
#pragma unroll
    for (int i = 0; i < NVM; ++i) {
      const int v = threadIdx.x + i * NTHR;
      if (v < nv) st[i] = load_bf16x8(p + v * 8);
    }
  };
  auto commit = [&](bf16_t* d) {
#pragma unroll
    for (int i = 0; i < NVM; ++i) {
      const int v = threadIdx.x + i * NTHR;
      if (v < nv) store_bf16x8(d + dst[i], st[i]);
    }
  };
  issue(tb);
  bf16x8 qf[KSM];
  const bf16_t* qp = (const bf16_t*)a.qa + ((int64_t)b * a.H + min(h, a.H - 1)) * LW;
#pragma unroll
  for (int s = 0; s < KSM; ++s)
    qf[s] = h < a.H && s < ks ? load_bf16x8(qp + 32 * s + 8 * g) : zero8();
  f32x4 o[NTW];
#pragma unroll
  for (int i = 0; i < NTW; ++i) o[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
  float m = kNegBig, lsum = 0.f;
  const float sl2 = a.scale * kLog2e;
  const int tr_off = ((col >> 2) + 4 * g) * row_l + 4 * (col & 3) + 16 * NTW * dw;

  int buf = 0;
  for (int t = tb; t < te; ++t) {
    bf16_t* kb = lat_lds + buf * tile_l;
    buf ^= 1;
    commit(kb);
    __syncthreads();
    if (t + 1 < te) issue(t + 1);
    // four chains (token half x step parity) hide the MFMA latency
    f32x4 part[2][2];
#pragma unroll
    for (int i = 0; i < 4; ++i) part[i >> 1][i & 1] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KSM; ++s)
      if (KSX || s < ks) {
#pragma unroll
        for (int h2 = 0; h2 < 2; ++h2)
          part[h2][s & 1] = mfma16(load_bf16x8(kb + (16 * h2 + col) * row_l + 32 * s + 8 * g),
                                   qf[s], part[h2][s & 1]);
      }
    f32x4 sc[2];
#pragma unroll
    for (int h2 = 0; h2 < 2; ++h2) sc[h2] = part[h2][0] + part[h2][1];
    float bmax = kNegBig;
#pragma unroll
    for (int h2 = 0; h2 < 2; ++h2)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int pos = t * kLB + 16 * h2 + 4 * g + r;
        sc[h2][r] = pos >= lo && pos < ctx ? sc[h2][r] * sl2 : kNegBig;
        bmax = fmaxf(bmax, sc[h2][r]);
      }
    bmax = fmaxf(bmax, __shfl_xor(bmax, 16, 64));
    bmax = fmaxf(bmax, __shfl_xor(bmax, 32, 64));
    const float m_new = fmaxf(m, bmax);  // every tile of a split holds a visible token
    const float alpha = fast_exp2(m - m_new);
    const bool moved = __any(m_new > m);
    m = m_new;
    bf16x8 pf;
    float psum = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float pa = fast_exp2(sc[0][r] - m_new), pb = fast_exp2(sc[1][r] - m_new);
      psum += pa + pb;
      pf[r] = f2bf(pa);
      pf[4 + r] = f2bf(pb);
    }
    lsum = lsum * alpha + psum;
    if (moved) {
#pragma unroll
      for (int i = 0; i < NTW; ++i) o[i] *= alpha;
    }
#pragma unroll
    for (int i = 0; i < NTW; ++i) {
      if (KSX || 16 * (NTW * dw + i) < R) {
        const bf16x4 x = lat_read_tr16(kb + tr_off + 16 * i);
        const bf16x4 y = lat_read_tr16(kb + tr_off + 16 * row_l + 16 * i);
        bf16x8 vf;
#pragma unroll
        for (int j = 0; j < 4; ++j) { vf[j] = x[j]; vf[4 + j] = y[j]; }
        o[i] = mfma16(vf, pf, o[i]);
      }
    }
  }
  lat_decode_out<RT, ND>(a, b, h, sp, nparts, dw, g, R, o, m, lsum);
}

// The same for rows of R = 64 RT and 64 rotated or padding columns, whole cache lines.  Two blocks at a time go
// straight into LDS, by loads that the waves wait for by count, while the two before them are worked on; each of a head
// tile's ND waves takes 64 / ND of the 64 tokens' scores and hands them to the others through LDS, where the form above
// has every wave compute them all.  Chunk c (16 bytes) of row t lies at c ^ (t / 2 % 8).  That form was bound
// by each block's chain - the scores' LDS reads fourfold, one wave a SIMD, two barriers for 64 tokens in both: 64
// sequences of 1500 tokens, 32 heads of 512 + 64, four splits: 28.4 -> 26.6 us.
template <int RT, int NH, int ND>
struct LatPair {
  static constexpr int KS = 2 * RT + 2, LW = 32 * KS, CPR = LW / 8, NW = NH * ND;
  static constexpr int TILE = kLB * LW;                                   // elements of a block
  static constexpr size_t BYTES = (size_t)4 * TILE * 2 + 4096 * NH;       // two pairs, [NH][4][64] f32x4 of scores
};
template <int RT, int NH, int ND>
__global__ __launch_bounds__(64 * NH * ND, 1) void latent_decode_pair_kernel(LatentDecodeArgs a) {
  using L = LatPair<RT, NH, ND>;
  constexpr int KS = L::KS, LW = L::LW, R = 64 * RT, NTW = 4 * RT / ND, QT = 4 / ND;
  constexpr int DP = KS * 4 / L::NW;  // loads of 1 KiB to a wave and pair of blocks
  static_assert(KS * 4 % L::NW == 0, "loads to a wave");
  extern __shared__ __attribute__((aligned(16))) bf16_t lat_lds[];
  f32x4* const scores = reinterpret_cast<f32x4*>(lat_lds + 4 * L::TILE);
  const int b = blockIdx.x, sp = blockIdx.z;
  const int w = wave_id_uniform(), lane = threadIdx.x & 63;
  const int hw = w / ND, dw = w % ND;
  const int col = lane & 15, g = lane >> 4;
  const int h = (blockIdx.y * NH + hw) * 16 + col;
  bf16x8 qf[KS];
  const bf16_t* qp = (const bf16_t*)a.qa + ((int64_t)b * a.H + min(h, a.H - 1)) * LW;
#pragma unroll
  for (int s = 0; s < KS; ++s) qf[s] = load_bf16x8(qp + 32 * s + 8 * g);  // (rows past the heads: not stored)
  const int ctx = a.context_lens[b];
  if (ctx <= 0) {
    if (sp == 0 && h < a.H)
      for (int i = dw * 4 + g; i < R; i += 4 * ND)
        ((bf16_t*)a.out)[((int64_t)b * a.H + h) * R + i] = f2bf(0.f);
    return;
  }
  const int lo = a.window > 0 ? max(0, ctx - a.window) : 0;
  const int t0 = lo / kLB, t1 = (ctx + kLB - 1) / kLB;
  const int nparts = (t1 - t0 + a.tiles_per_split - 1) / a.tiles_per_split;
  const int tb = t0 + sp * a.tiles_per_split, te = min(t1, tb + a.tiles_per_split);
  if (tb >= te) return;
  const int* bt = a.block_tables + (int64_t)b * a.bt_stride;
  // the table, 64 entries ahead, a lane each; waited for here, not where it is read among the ring's loads
  int table = 0, table_at = tb;
  auto next_table = [&](int t) {
    table_at = t;
    table = t + lane < te ? bt[t + lane] : 0;
    asm volatile("" : "+v"(table)::"memory");
  };
  next_table(tb);
#pragma unroll
  for (int s = 0; s < KS; ++s) asm volatile("" : "+v"(qf[s])::"memory");
  // load j of a pair, of 1 KiB: block j / (2 KS), its j % (2 KS)-th; wave w takes j = w, w + NW, ...
  unsigned voff[DP];
#pragma unroll
  for (int i = 0; i < DP; ++i) {
    const int c = 64 * ((i * L::NW + w) % (2 * KS)) + lane, t = c / L::CPR, p = c - t * L::CPR;
    voff[i] = (unsigned)(t * L::CPR + (p ^ (t / 2 % 8))) * 16u;
  }
  const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)(lds_ptr)lat_lds);
  auto fetch = [&](int t, int stage) {  // blocks t and t + 1 (a split's last one: itself again)
    if (t - table_at >= 64) next_table(t);
    const bf16_t* const cache = (const bf16_t*)a.cache;
    const int p0 = __builtin_amdgcn_readlane(table, t - table_at);
    const int p1 = __builtin_amdgcn_readlane(table, min(t + 1, te - 1) - table_at);
    const __amdgpu_buffer_rsrc_t r0 = dma_rsrc(cache + (int64_t)p0 * L::TILE), r1 = dma_rsrc(cache + (int64_t)p1 * L::TILE);
#pragma unroll
    for (int i = 0; i < DP; ++i) {
      const int j = i * L::NW + w;
      dma16<true>(lds0 + (unsigned)stage * (2 * L::TILE * 2) + 1024u * j, voff[i], j < 2 * KS ? r0 : r1, 0u);
    }
  };
  fetch(tb, 0);
  f32x4 o[NTW];
#pragma unroll
  for (int i = 0; i < NTW; ++i) o[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
  float m = kNegBig, lsum = 0.f;
  const float sl2 = a.scale * kLog2e;
  const int tr_row = (col >> 2) + 4 * g, tr_x = tr_row / 2 % 8, key_x = col / 2 % 8;
  int stage = 0;
  for (int t = tb; t < te; t += 2, stage ^= 1) {
    const bf16_t* kb = lat_lds + stage * 2 * L::TILE;
    wait_vm<0>();
    lds_barrier();  // the pair has landed, and everyone is through with the pair before and its scores
    if (t + 2 < te) fetch(t + 2, stage ^ 1);
#pragma unroll
    for (int q = 0; q < QT; ++q) {  // tokens 16 (dw QT + q) .. of the pair
      const int grp = dw * QT + q;
      f32x4 part[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
      const bf16_t* row = kb + (16 * grp + col) * LW;
#pragma unroll
      for (int s = 0; s < KS; ++s)
        part[s & 1] = mfma16(load_bf16x8(row + ((4 * s + g) ^ key_x) * 8), qf[s], part[s & 1]);
      f32x4 sc = part[0] + part[1];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int pos = t * kLB + 16 * grp + 4 * g + r;
        sc[r] = pos >= lo && pos < min(ctx, te * kLB) ? sc[r] * sl2 : kNegBig;
      }
      scores[(hw * 4 + grp) * 64 + lane] = sc;
    }
    lds_barrier();
    f32x4 sc[4];
    float bmax = kNegBig;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      sc[q] = scores[(hw * 4 + q) * 64 + lane];
#pragma unroll
      for (int r = 0; r < 4; ++r) bmax = fmaxf(bmax, sc[q][r]);
    }
    bmax = fmaxf(bmax, __shfl_xor(bmax, 16, 64));
    bmax = fmaxf(bmax, __shfl_xor(bmax, 32, 64));
    const float m_new = fmaxf(m, bmax);  // every tile of a split holds a visible token
    const float alpha = fast_exp2(m - m_new);
    const bool moved = __any(m_new > m);
    m = m_new;
    bf16x8 pf[2];
    float psum = 0.f;
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float p = fast_exp2(sc[q][r] - m_new);
        psum += p;
        pf[q >> 1][(q & 1) * 4 + r] = f2bf(p);
      }
    lsum = lsum * alpha + psum;
    if (moved) {
#pragma unroll
      for (int i = 0; i < NTW; ++i) o[i] *= alpha;
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (u == 1 && t + 1 >= te) break;  // (a lone last block is there twice, its second scores masked)
#pragma unroll
      for (int i = 0; i < NTW; ++i) {
        const int c = (2 * (NTW * dw + i) + ((col & 3) >> 1)) ^ tr_x;
        const bf16_t* at = kb + (32 * u + tr_row) * LW + c * 8 + 4 * (col & 1);
        const bf16x4 x = lat_read_tr16(at), y = lat_read_tr16(at + 16 * LW);
        bf16x8 vf;
#pragma unroll
        for (int j = 0; j < 4; ++j) { vf[j] = x[j]; vf[4 + j] = y[j]; }
        o[i] = mfma16(vf, pf[u], o[i]);
      }
    }
  }
  lat_decode_out<RT, ND>(a, b, h, sp, nparts, dw, g, R, o, m, lsum);
}

// The same for latents of 512 and up to 16 heads, and for up to 32 where a split has few blocks (lat_ring_takes): a block at a
// time, three more on their way, so that what a CU takes in never waits for a barrier.  A wave's scores are 16 of the block's
// tokens over one half of the columns; V's operands are read during the softmax, K's ahead of their products, and blocks inside
// the context are not masked.  16 heads, pairs -> this: 200 sequences of 500 tokens 33 -> 29 us in the pass (5.1 TB/s behind 6.5
// us of launch and first loads, which a context of one block takes), alone 25.6 -> 23.4, 256 x 400 25.2 -> 22.7, 64 x 1500 27.3 ->
// 25.2.  Slower than pairs for latents of 256 (16 heads 200 x 500 16.6 / 17.8, 32 18.8 / 22.6: two barriers for half the tokens) and
// for more heads (64 x 1500 of 48 38.6 / 40.5: registers for fewer reads ahead), which keep them.
template <int NH>
struct LatRing {
  static constexpr int RT = 8, ND = 4, KS = 2 * RT + 2, LW = 32 * KS, CPR = LW / 8, NW = NH * ND, ST = 4;
  static constexpr int TILE = kLB * LW;                                // elements of a block
  static constexpr size_t BYTES = (size_t)ST * TILE * 2 + 1024 * NW;   // and [NW][64] f32x4 of scores
};
// the largest of the lanes 16 apart
DRTC_DEVICE float rows_max(float v) {
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

template <int NH>
__global__ __launch_bounds__(256 * NH, 2) void latent_decode_ring_kernel(LatentDecodeArgs a) {
  using L = LatRing<NH>;
  constexpr int LW = L::LW, RT = L::RT, ND = L::ND, R = 64 * RT, NTW = 4 * RT / ND, ST = L::ST, KS = L::KS / 2;
  constexpr int LOADS = 2 * L::KS, DP = LOADS / L::NW;   // loads of 1 KiB to a block, and to a wave (the first ones one more)
  constexpr int MORE = LOADS % L::NW, DM = DP + (MORE > 0);
  extern __shared__ __attribute__((aligned(16))) bf16_t lat_lds[];
  f32x4* const scores = reinterpret_cast<f32x4*>(lat_lds + ST * L::TILE);
  const int b = blockIdx.x, sp = blockIdx.z;
  const int w = wave_id_uniform(), lane = threadIdx.x & 63;
  const int hw = w / ND, dw = w % ND, grp = dw & 1, s0 = (dw >> 1) * KS;
  const int col = lane & 15, g = lane >> 4;
  const int h = (blockIdx.y * NH + hw) * 16 + col;
  bf16x8 qf[KS];
  const bf16_t* qp = (const bf16_t*)a.qa + ((int64_t)b * a.H + min(h, a.H - 1)) * LW;
#pragma unroll
  for (int s = 0; s < KS; ++s) qf[s] = load_bf16x8(qp + 32 * (s0 + s) + 8 * g);  // (rows past the heads: not stored)
  // without a window the first blocks' table entries need not wait for the context's length (those behind it are not used)
  const int* bt = a.block_tables + (int64_t)b * a.bt_stride;
  int table = a.window > 0 || a.bt_cols < 1 ? 0 : bt[min(sp * a.tiles_per_split + lane, a.bt_cols - 1)];
  const int ctx = a.context_lens[b];
  if (ctx <= 0) {
    if (sp == 0 && h < a.H)
      for (int i = dw * 4 + g; i < R; i += 4 * ND)
        ((bf16_t*)a.out)[((int64_t)b * a.H + h) * R + i] = f2bf(0.f);
    return;
  }
  const int lo = a.window > 0 ? max(0, ctx - a.window) : 0;
  const int t0 = lo / kLB, t1 = (ctx + kLB - 1) / kLB;
  const int nparts = (t1 - t0 + a.tiles_per_split - 1) / a.tiles_per_split;
  const int tb = t0 + sp * a.tiles_per_split, te = min(t1, tb + a.tiles_per_split);
  if (tb >= te) return;
  // the table, 64 entries ahead, a lane each; waited for here, not where it is read among the ring's loads
  int table_at = tb;
  auto next_table = [&](int t) {
    table_at = t;
    table = t + lane < te ? bt[t + lane] : 0;
    asm volatile("" : "+v"(table)::"memory");
  };
  if (a.window > 0) next_table(tb);
  else asm volatile("" : "+v"(table)::"memory");
#pragma unroll
  for (int s = 0; s < KS; ++s) asm volatile("" : "+v"(qf[s])::"memory");
  // load j of a block, of 1 KiB; wave w takes j = w, w + NW, ...
  unsigned voff[DM];
#pragma unroll
  for (int i = 0; i < DM; ++i) {
    const int c = 64 * (i * L::NW + w) + lane, t = c / L::CPR, p = c - t * L::CPR;
    voff[i] = (unsigned)(t * L::CPR + (p ^ (t / 2 % 8))) * 16u;
  }
  const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)(lds_ptr)lat_lds);
  auto fetch = [&](int t) {
    if (t - table_at >= 64) next_table(t);
    const __amdgpu_buffer_rsrc_t rows =
        dma_rsrc((const bf16_t*)a.cache + (int64_t)__builtin_amdgcn_readlane(table, t - table_at) * L::TILE);
    const unsigned to = lds0 + (unsigned)((t - tb) % ST) * (L::TILE * 2) + 1024u * w;
#pragma unroll
    for (int i = 0; i < DM; ++i)
      if (i < DP || w < MORE) dma16<true>(to + 1024u * (i * L::NW), voff[i], rows, 0u);
  };
#pragma unroll 1
  for (int t = tb; t < min(tb + ST - 1, te); ++t) fetch(t);
  f32x4 o[NTW];
#pragma unroll
  for (int i = 0; i < NTW; ++i) o[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
  float m = kNegBig, lsum = 0.f;
  const float sl2 = a.scale * kLog2e;
  const int tr_row = (col >> 2) + 4 * g, tr_x = tr_row / 2 % 8, key_x = col / 2 % 8;
  for (int t = tb; t < te; ++t) {
    const bf16_t* kb = lat_lds + (t - tb) % ST * L::TILE;
    const int younger = min(ST - 2, te - 1 - t);
    if (w < MORE) wait_groups<DM, ST - 2>(younger);
    else wait_groups<DP, ST - 2>(younger);
    lds_barrier();  // the block has landed, and everyone is through with the block before and its scores
    if (t + ST - 1 < te) fetch(t + ST - 1);
    {  // tokens 16 grp .. of the block
      f32x4 part[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
      const bf16_t* row = kb + (16 * grp + col) * LW;
      bf16x8 kf[KS];
#pragma unroll
      for (int s = 0; s < KS; ++s) kf[s] = load_bf16x8(row + ((4 * (s0 + s) + g) ^ key_x) * 8);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < KS; ++s) part[s & 1] = mfma16(kf[s], qf[s], part[s & 1]);
      scores[w * 64 + lane] = part[0] + part[1];
    }
    lds_barrier();
    f32x4 sc[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) sc[q] = scores[(hw * ND + q) * 64 + lane] + scores[(hw * ND + 2 + q) * 64 + lane];
    __builtin_amdgcn_sched_barrier(0);
    bf16x8 vf[NTW];
#pragma unroll
    for (int i = 0; i < NTW; ++i) {
      const int c = (2 * (NTW * dw + i) + ((col & 3) >> 1)) ^ tr_x;
      const bf16_t* at = kb + tr_row * LW + c * 8 + 4 * (col & 1);
      const bf16x4 x = lat_read_tr16(at), y = lat_read_tr16(at + 16 * LW);
#pragma unroll
      for (int j = 0; j < 4; ++j) { vf[i][j] = x[j]; vf[i][4 + j] = y[j]; }
    }
    __builtin_amdgcn_sched_barrier(0);
    const bool whole = t * kLB >= lo && (t + 1) * kLB <= ctx;
    float bmax = kNegBig;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      if (!whole) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int pos = t * kLB + 16 * q + 4 * g + r;
          sc[q][r] = pos >= lo && pos < ctx ? sc[q][r] * sl2 : kNegBig;
        }
      } else {
        sc[q] *= sl2;
      }
      bmax = fmaxf(bmax, fmaxf(fmaxf(sc[q][0], sc[q][1]), fmaxf(sc[q][2], sc[q][3])));
    }
    bmax = rows_max(bmax);
    const float m_new = fmaxf(m, bmax);  // every block of a split holds a visible token
    const float alpha = fast_exp2(m - m_new);
    const bool moved = __any(m_new > m);
    m = m_new;
    bf16x8 pf;
    float psum = 0.f;
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float p = fast_exp2(sc[q][r] - m_new);
        psum += p;
        pf[4 * q + r] = f2bf(p);
      }
    lsum = lsum * alpha + psum;
    if (moved) {
#pragma unroll
      for (int i = 0; i < NTW; ++i) o[i] *= alpha;
    }
#pragma unroll
    for (int i = 0; i < NTW; ++i) o[i] = mfma16(vf[i], pf, o[i]);
  }
  lat_decode_out<RT, ND>(a, b, h, sp, nparts, dw, g, R, o, m, lsum);
}

// Merge of the window splits (and the sink): one workgroup per (sequence, head).
__global__ __launch_bounds__(128) void latent_merge_kernel(LatentDecodeArgs a) {
  const int b = blockIdx.x, h = blockIdx.y;
  const int ctx = a.context_lens[b];
  if (ctx <= 0) return;
  const int lo = a.window > 0 ? max(0, ctx - a.window) : 0;
  const int nt = (ctx + kLB - 1) / kLB - lo / kLB;
  const int nparts = (nt + a.tiles_per_split - 1) / a.tiles_per_split;
  if (nparts == 1) return;
  const int64_t pi = ((int64_t)b * a.H + h) * a.nsplits;
  float m = kNegBig;
  for (int p = 0; p < nparts; ++p) m = fmaxf(m, a.part_ml[2 * (pi + p)]);
  float l = a.sink ? fast_exp2(a.sink[h] * kLog2e - m) : 0.f;
  for (int p = 0; p < nparts; ++p)
    l += a.part_ml[2 * (pi + p) + 1] * fast_exp2(a.part_ml[2 * (pi + p)] - m);
  const float inv = head_gate<bf16_t>(a.gate, (int64_t)b * a.ldg + h) / l;
  for (int d = threadIdx.x * 4; d < a.R; d += 512) {
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
    for (int p = 0; p < nparts; ++p)
      s += *reinterpret_cast<const f32x4*>(a.part_o + (pi + p) * a.R + d) *
           fast_exp2(a.part_ml[2 * (pi + p)] - m);
    bf16x4 v;
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = f2bf(s[r] * inv);
    *reinterpret_cast<bf16x4*>((bf16_t*)a.out + ((int64_t)b * a.H + h) * a.R + d) = v;
  }
}

template <int RT, int NH>
constexpr bool lat_ring = RT == 8 && NH <= 2;
template <int RT, int NH>
constexpr bool lat_pair = RT != 8 || NH != 1;  // (up to 16 heads of 512 all go by single blocks)
// Whether 17 to 32 heads go by single blocks, by the blocks of a split (a table wider than the contexts counts as long ones).  The
// ring starts 1 - 2 us sooner and reads no lone last block twice; pairs have one barrier a block less, and few heads beyond the
// first 16 need little of what the ring gives.  us, pairs / ring, of rows of 576 that no cache holds:
//   odd, up to 11: 17 heads 0.99 - 1.04 times as fast, 24 1.00 - 1.06, 32 1.01 - 1.08 (64 x 1500 of 32, a window of 1024, splits of
//     nine: 29.8 / 29.2)
//   even, more than 24 heads: up to 12 without a window 0.98 - 1.28 (64 x 400 of 32 21.1 / 20.1, 200 x 200 20.2 / 19.7), with
//     one, whose start waits for the context anyway, four (0.98 - 1.04; six: 40 x 1500 24.0 / 24.5)
//   even, 20 to 24 heads: four without a window 0.99 - 1.26, with one 0.95 - 1.02; eight 0.98 - 1.00
//   even, 17 to 19: 0.92 - 0.98 (40 x 1500 24.6 / 25.8), but for contexts of a block
//   more: 32 heads 64 x 1000 in one split of 40 55.0 / 58.5, 40 x 3000 in splits of 20 40.0 / 41.7; short contexts in such a table
//     give up what the ring's start saves (64 x 20 12.0 / 9.9, 100 x 100 15.7 / 14.8).
static bool lat_ring_takes(const LatentDecodeArgs& a) {
  const int n = a.tiles_per_split, even = a.H > 24 ? (a.window > 0 ? 4 : 12) : a.H >= 20 && a.window <= 0 ? 4 : 0;
  return a.H <= 16 || n <= (n % 2 ? 11 : even);
}
template <int RT, int NH, int ND>
static void lat_decode_go(const LatentDecodeArgs& a, hipStream_t st) {
  const size_t lds = (size_t)2 * kLB * (a.LW + kLatPad) * 2;
  const dim3 grid(a.B, (a.H + 16 * NH - 1) / (16 * NH), a.nsplits), block(64 * NH * ND);
  if constexpr (RT >= 4) {
    // (into LDS by whole 16-byte pieces)
    if (a.R == 64 * RT && a.LW == 32 * (2 * RT + 2) && (uintptr_t)a.cache % 16 == 0) {
      constexpr int NP = NH == 2 ? 4 : ND;  // eight waves where the heads fill two tiles
      if constexpr (lat_ring<RT, NH>)
        if (lat_ring_takes(a)) {
          latent_decode_ring_kernel<NH><<<grid, dim3(256 * NH), LatRing<NH>::BYTES, st>>>(a);
          return;
        }
      if constexpr (lat_pair<RT, NH>) {
        latent_decode_pair_kernel<RT, NH, NP><<<grid, dim3(64 * NH * NP), LatPair<RT, NH, NP>::BYTES, st>>>(a);
        return;
      }
    }
    if (a.R == 64 * RT && a.LW == 32 * (2 * RT + 1)) {
      latent_decode_kernel<RT, NH, ND, 2 * RT + 1><<<grid, block, lds, st>>>(a);
      return;
    }
  }
  latent_decode_kernel<RT, NH, ND, 0><<<grid, block, lds, st>>>(a);
}
template <int RT>
static void lat_decode_h(const LatentDecodeArgs& a, hipStream_t st) {
  if (a.H <= 16) lat_decode_go<RT, 1, 4>(a, st);
  else if (a.H <= 32) lat_decode_go<RT, 2, 2>(a, st);
  else lat_decode_go<RT, 4, 2>(a, st);
}

static int lat_decode_need(const LatentDecodeArgs& a) { return std::max((a.R + 63) / 64, (a.LW / 32 - 1) / 2); }
static bool lat_decode_mfma(int f32, const LatentDecodeArgs& a) {
  return !f32 && a.R % 8 == 0 && a.LW % 32 == 0 && lat_decode_need(a) <= 8 && a.R <= 512;
}
static bool lat_decode_split(int f32, const LatentDecodeArgs& a) { return lat_decode_mfma(f32, a) && a.nsplits > 1; }
static void lat_decode_parts(const LatentDecodeArgs& a, hipStream_t st) {
  const int need = lat_decode_need(a);
  if (need <= 1) lat_decode_h<1>(a, st);
  else if (need <= 2) lat_decode_h<2>(a, st);
  else if (need <= 4) lat_decode_h<4>(a, st);
  else lat_decode_h<8>(a, st);
}

int launch_latent_decode(int f32, const LatentDecodeArgs& a, hipStream_t st) {
  if (a.B == 0) return 0;
  if (lat_decode_mfma(f32, a)) {
    lat_decode_parts(a, st);
    if (a.nsplits > 1) latent_merge_kernel<<<dim3(a.B, a.H), dim3(128), 0, st>>>(a);
  } else {
    if (a.R > 1024) return -1;
    if (f32) latent_decode_any_kernel<float><<<dim3(a.B, a.H), dim3(256), 0, st>>>(a);
    else latent_decode_any_kernel<bf16_t><<<dim3(a.B, a.H), dim3(256), 0, st>>>(a);
  }
  return (int)hipGetLastError();
}

// ------------------------------------------------------------------ per-head projections
// y[b, h, :] = W[h] x[b, h, :], W [H, N, K].  MFMA: 16 output dims per wave, 64 batch rows per
// workgroup sharing each weight fragment; operands straight from global memory (the weights
// are read once per 64 rows and stay in L2).
// WHOLE: K % 128 == 0 - four steps' loads ahead of their products.
struct HeadGemm {
  bf16_t* y;
  const bf16_t *x, *w;
  int B, N, K;
  int64_t yb, yh, xb, xh;
};
template <int NBT, bool WHOLE>
DRTC_DEVICE void head_gemm_tile(const HeadGemm& q, int tile, int rows, int h) {
  const auto [y, x, w, B, N, K, yb, yh, xb, xh] = q;
  const int b0 = rows * 16 * NBT;
  const int wv = wave_id_uniform(), lane = threadIdx.x & 63;
  const int col = lane & 15, g = lane >> 4;
  const int n0 = (tile * 4 + wv) * 16;
  if (n0 >= N) return;
  const bf16_t* wr = w + ((int64_t)h * N + min(n0 + col, N - 1)) * K;
  const bf16_t* xr[NBT];
#pragma unroll
  for (int i = 0; i < NBT; ++i) xr[i] = x + (int64_t)min(b0 + 16 * i + col, B - 1) * xb + h * xh;
  f32x4 acc[NBT];
#pragma unroll
  for (int i = 0; i < NBT; ++i) acc[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
  if constexpr (WHOLE) {
    for (int k = 0; k < K; k += 128) {
      bf16x8 wf[4], xf[4][NBT];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        wf[s] = load_bf16x8(wr + k + 32 * s + 8 * g);
#pragma unroll
        for (int i = 0; i < NBT; ++i) xf[s][i] = load_bf16x8(xr[i] + k + 32 * s + 8 * g);
      }
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < NBT; ++i) acc[i] = mfma16(wf[s], xf[s][i], acc[i]);
    }
  } else {
    for (int k = 0; k < K; k += 32) {
      const int c = k + 8 * g;
      const bool in = c < K;
      const bf16x8 wf = in ? load_bf16x8(wr + c) : zero8();
#pragma unroll
      for (int i = 0; i < NBT; ++i)
        acc[i] = mfma16(wf, in ? load_bf16x8(xr[i] + c) : zero8(), acc[i]);
    }
  }
#pragma unroll
  for (int i = 0; i < NBT; ++i) {
    const int b = b0 + 16 * i + col, n = n0 + 4 * g;
    if (b < B && n < N) {
      bf16x4 v;
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = f2bf(acc[i][r]);
      *reinterpret_cast<bf16x4*>(y + b * yb + h * yh + n) = v;
    }
  }
}

// The same for long K on a chip with room: a workgroup's waves share its 16 output dims and take every fourth
// 128 of K, their sums meet in LDS: one round trip to memory where a wave alone makes K / 128.  128 dims from 512, us:
// 200 rows of 16 heads 11.3 -> 7.2, 64 of 32 11.2 -> 4.8.
template <int NBT>
__global__ __launch_bounds__(256) void head_gemm_shared_kernel(HeadGemm q) {
  const auto [y, x, w, B, N, K, yb, yh, xb, xh] = q;
  __shared__ f32x4 sums[4][NBT][64];
  const int h = blockIdx.z, b0 = blockIdx.y * 16 * NBT, n0 = blockIdx.x * 16;
  const int wv = wave_id_uniform(), lane = threadIdx.x & 63;
  const int col = lane & 15, g = lane >> 4;
  const bf16_t* wr = w + ((int64_t)h * N + min(n0 + col, N - 1)) * K;
  const bf16_t* xr[NBT];
#pragma unroll
  for (int i = 0; i < NBT; ++i) xr[i] = x + (int64_t)min(b0 + 16 * i + col, B - 1) * xb + h * xh;
  f32x4 acc[NBT];
#pragma unroll
  for (int i = 0; i < NBT; ++i) acc[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
  for (int k = 128 * wv; k < K; k += 512) {
    bf16x8 wf[4], xf[4][NBT];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      wf[s] = load_bf16x8(wr + k + 32 * s + 8 * g);
#pragma unroll
      for (int i = 0; i < NBT; ++i) xf[s][i] = load_bf16x8(xr[i] + k + 32 * s + 8 * g);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int i = 0; i < NBT; ++i) acc[i] = mfma16(wf[s], xf[s][i], acc[i]);
  }
#pragma unroll
  for (int i = 0; i < NBT; ++i) sums[wv][i][lane] = acc[i];
  __syncthreads();
  for (int i = wv; i < NBT; i += 4) {
    const f32x4 s = (sums[0][i][lane] + sums[1][i][lane]) + (sums[2][i][lane] + sums[3][i][lane]);
    const int b = b0 + 16 * i + col, n = n0 + 4 * g;
    if (b < B && n < N) {
      bf16x4 v;
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = f2bf(s[r]);
      *reinterpret_cast<bf16x4*>(y + b * yb + h * yh + n) = v;
    }
  }
}

// The shared form for up to 16 rows behind a split window (LatentDecodeArgs a), K = a.R: each workgroup adds the
// splits up itself, into LDS, while its weights are on their way.
constexpr int kUpParts = 1024;  // rows times splits
template <int KMAX>
__global__ __launch_bounds__(256) void latent_up_kernel(LatentDecodeArgs a, HeadGemm q) {
  __shared__ f32x4 sums[4][64];
  __shared__ float factor[kUpParts];
  __shared__ int count[16];
  __shared__ __attribute__((aligned(16))) bf16_t xs[16][KMAX + 8];
  const int h = blockIdx.y, n0 = blockIdx.x * 16, K = q.K, N = q.N, B = q.B;
  const int wv = wave_id_uniform(), lane = threadIdx.x & 63;
  const int col = lane & 15, g = lane >> 4;
  const bf16_t* wr = q.w + ((int64_t)h * N + min(n0 + col, N - 1)) * K + 128 * wv + 8 * g;
  bf16x8 wf[KMAX / 512][4];
#pragma unroll
  for (int j = 0; j < KMAX / 512; ++j)
#pragma unroll
    for (int s = 0; s < 4; ++s) wf[j][s] = 128 * wv + 512 * j < K ? load_bf16x8(wr + 512 * j + 32 * s) : zero8();
  for (int b = wv; b < B; b += 4) {
    const int ctx = a.context_lens[b], lo = a.window > 0 ? max(0, ctx - a.window) : 0;
    const int n = ctx <= 0 ? 0 : ((ctx + kLB - 1) / kLB - lo / kLB + a.tiles_per_split - 1) / a.tiles_per_split;
    const float* ml = a.part_ml + ((int64_t)b * a.H + h) * a.nsplits * 2;
    if (lane == 0) count[b] = n;
    if (n < 2) continue;
    float top = kNegBig, l = 0.f;
    for (int p = lane; p < n; p += 64) top = fmaxf(top, ml[2 * p]);
    top = wave_max(top);
    for (int p = lane; p < n; p += 64) l += ml[2 * p + 1] * fast_exp2(ml[2 * p] - top);
    l = wave_sum(l) + (a.sink ? fast_exp2(a.sink[h] * kLog2e - top) : 0.f);
    const float inv = head_gate<bf16_t>(a.gate, (int64_t)b * a.ldg + h) / l;
    for (int p = lane; p < n; p += 64) factor[b * a.nsplits + p] = fast_exp2(ml[2 * p] - top) * inv;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < B * (K / 4); i += 256) {
    const int b = i / (K / 4), d = 4 * (i - b * (K / 4)), n = count[b];
    const int64_t row = (int64_t)b * a.H + h;
    bf16x4 v;
    if (n == 1) {  // (written as it is)
      v = load_bf16x4((const bf16_t*)a.out + row * K + d);
    } else {
      const float* po = a.part_o + row * a.nsplits * K + d;
      f32x4 s = {0.f, 0.f, 0.f, 0.f};
      for (int p0 = 0; p0 < n; p0 += 8) {  // eight on their way
        f32x4 t[8];
#pragma unroll
        for (int p = 0; p < 8; ++p) t[p] = *reinterpret_cast<const f32x4*>(po + (int64_t)min(p0 + p, n - 1) * K);
#pragma unroll
        for (int p = 0; p < 8; ++p) s += t[p] * (p0 + p < n ? factor[b * a.nsplits + p0 + p] : 0.f);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = f2bf(s[r]);
    }
    *reinterpret_cast<bf16x4*>(&xs[b][d]) = v;
  }
  __syncthreads();
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < KMAX / 512; ++j) {
    if (128 * wv + 512 * j >= K) continue;
#pragma unroll
    for (int s = 0; s < 4; ++s)
      acc = mfma16(wf[j][s], load_bf16x8(&xs[min(col, B - 1)][128 * wv + 512 * j + 32 * s + 8 * g]), acc);
  }
  sums[wv][lane] = acc;
  __syncthreads();
  if (wv) return;
  const f32x4 s = (sums[0][lane] + sums[1][lane]) + (sums[2][lane] + sums[3][lane]);
  const int n = n0 + 4 * g;
  if (col < B && n < N) {
    bf16x4 v;
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = f2bf(s[r]);
    *reinterpret_cast<bf16x4*>(q.y + col * q.yb + h * q.yh + n) = v;
  }
}
template <int NBT, bool WHOLE>
__global__ __launch_bounds__(256) void head_gemm_kernel(HeadGemm q) {
  head_gemm_tile<NBT, WHOLE>(q, blockIdx.x, blockIdx.y, blockIdx.z);
}

// A decode step's preparation and its queries' way down into the latent space, which read and write other columns: the
// rows' workgroups, then the product's.  Both are a round trip to memory and their launch, and one of them is saved: 2.2 us
// a layer at 1 to 200 rows.
template <int NBT>
__global__ __launch_bounds__(256) void latent_front_kernel(LatentPrepArgs a, HeadGemm q) {
  if ((int)blockIdx.x < a.rows) {
    latent_prep_row<bf16_t, 8>(a, blockIdx.x);
    return;
  }
  const int i = blockIdx.x - a.rows, gx = (q.N + 63) / 64, t = i / gx, gy = (q.B + 16 * NBT - 1) / (16 * NBT);
  head_gemm_tile<NBT, true>(q, i - t * gx, t % gy, t / gy);
}

static bool head_gemm_shares(const HeadGemm& q, int H, int nbt) {
  // shared where a CU would have half a workgroup: 128 dims from 512 of 32 heads, 128 rows 11.4 / 8.4 us, 200 (one a
  // CU) 12.4 / 13.7; with fewer rows to a workgroup up to one a CU: 256 dims of 64 heads, 32 rows 8.8 / 8.3
  return q.K % 128 == 0 && q.K >= 256 &&
         (int64_t)((q.N + 63) / 64) * ((q.B + 16 * nbt - 1) / (16 * nbt)) * H <= (nbt == 4 ? 128 : 256);
}
template <int NBT>
static void head_gemm_go(const HeadGemm& q, int H, hipStream_t st) {
  const dim3 grid((q.N + 63) / 64, (q.B + 16 * NBT - 1) / (16 * NBT), H);
  if (head_gemm_shares(q, H, NBT))
    head_gemm_shared_kernel<NBT><<<dim3((q.N + 15) / 16, grid.y, H), dim3(256), 0, st>>>(q);
  else if (q.K % 128 == 0)
    head_gemm_kernel<NBT, true><<<grid, dim3(256), 0, st>>>(q);
  else
    head_gemm_kernel<NBT, false><<<grid, dim3(256), 0, st>>>(q);
}

template <class T>
__global__ __launch_bounds__(256) void head_gemm_any_kernel(
    T* __restrict__ y, const T* __restrict__ x, const T* __restrict__ w, int N, int K, int64_t yb,
    int64_t yh, int64_t xb, int64_t xh) {
  const int b = blockIdx.x, h = blockIdx.y, n = blockIdx.z * 256 + threadIdx.x;
  if (n >= N) return;
  const T* xr = x + b * xb + h * xh;
  const T* wr = w + ((int64_t)h * N + n) * K;
  float s = 0.f;
  for (int k = 0; k < K; ++k) s += to_f32(xr[k]) * to_f32(wr[k]);
  y[b * yb + h * yh + n] = from_f32<T>(s);
}

static bool head_gemm_whole(int N, int K, int64_t yb, int64_t yh, int64_t xb, int64_t xh) {
  return K % 8 == 0 && N % 4 == 0 && yb % 4 == 0 && yh % 4 == 0 && xb % 8 == 0 && xh % 8 == 0;
}
int launch_head_gemm(int f32, void* y, const void* x, const void* w, int B, int H, int N, int K,
                     int64_t yb, int64_t yh, int64_t xb, int64_t xh, hipStream_t st) {
  if (B == 0) return 0;
  if (!f32 && head_gemm_whole(N, K, yb, yh, xb, xh)) {
    const HeadGemm q{(bf16_t*)y, (const bf16_t*)x, (const bf16_t*)w, B, N, K, yb, yh, xb, xh};
    if (B <= 16) head_gemm_go<1>(q, H, st);
    else if (B <= 32) head_gemm_go<2>(q, H, st);
    else head_gemm_go<4>(q, H, st);
  } else {
    const dim3 grid(B, H, (N + 255) / 256);
    if (f32)
      head_gemm_any_kernel<float><<<grid, dim3(256), 0, st>>>(
          (float*)y, (const float*)x, (const float*)w, N, K, yb, yh, xb, xh);
    else
      head_gemm_any_kernel<bf16_t><<<grid, dim3(256), 0, st>>>(
          (bf16_t*)y, (const bf16_t*)x, (const bf16_t*)w, N, K, yb, yh, xb, xh);
  }
  return (int)hipGetLastError();
}

// Decode: launch_latent_prep, and qa[b, h, :R] = w[h] proj[b, h, :dim] for w [H, R, dim].
int launch_latent_front(int f32, const LatentPrepArgs& a, const void* w, hipStream_t st) {
  if (a.rows == 0) return 0;
  if (!a.qa || !lat_prep_takes(a)) return -1;
  const int dq = a.dim + a.rot;
  const HeadGemm q{(bf16_t*)a.qa, (const bf16_t*)a.proj, (const bf16_t*)w, a.rows, a.R, a.dim,
                   (int64_t)a.H * a.LW, a.LW, a.ldp, dq};
  const int nbt = a.rows <= 16 ? 1 : a.rows <= 32 ? 2 : 4;
  if (f32 || !lat_prep_whole(a) || !head_gemm_whole(q.N, q.K, q.yb, q.yh, q.xb, q.xh) || a.dim % 128 ||
      head_gemm_shares(q, a.H, nbt)) {
    const int e = launch_latent_prep(f32, a, st);
    return e ? e : launch_head_gemm(f32, a.qa, a.proj, w, a.rows, a.H, a.R, a.dim, q.yb, q.yh, q.xb, q.xh, st);
  }
  const int grid = a.rows + (a.R + 63) / 64 * ((a.rows + 16 * nbt - 1) / (16 * nbt)) * a.H;
  (nbt == 1 ? latent_front_kernel<1> : nbt == 2 ? latent_front_kernel<2> : latent_front_kernel<4>)<<<dim3(grid), dim3(256), 0, st>>>(a, q);
  return (int)hipGetLastError();
}

// Whether the way up adds up the splits itself, in each of its workgroups again: where a thread has up to two vectors of the
// rows, B R <= 2048 (965 sizes of 4 to 64 heads, behind each other in a graph: one vector 1.12, of more than 16 splits 1.37, two 1.00
// and in decode steps of three and four rows 1.00 to 1.01, three 0.92, eight 0.77: 16 rows of 16 heads, two splits of 512 dims
// 14.6 / 21.8 us), and up to 64 KB of them.
// A step of one row at 3500, two such layers, 381 -> 364 us with the launch below.
bool latent_up_merges(int B, int R, int nsplits) {
  return B <= 16 && B * R <= 2048 && B * nsplits <= kUpParts && (int64_t)B * nsplits * R <= 16384;
}

// Decode: launch_latent_decode, and y[b, h, :] = w[h] out[b, h, :] for w [H, N, R].
int launch_latent_decode_up(int f32, const LatentDecodeArgs& a, void* y, const void* w, int N, int64_t yb, int64_t yh,
                            hipStream_t st) {
  if (a.B == 0) return 0;
  const HeadGemm q{(bf16_t*)y, (const bf16_t*)a.out, (const bf16_t*)w, a.B, N, a.R, yb, yh, (int64_t)a.H * a.R, a.R};
  if (!lat_decode_split(f32, a) || !head_gemm_whole(N, a.R, yb, yh, q.xb, q.xh) || a.R % 128 ||
      !latent_up_merges(a.B, a.R, a.nsplits)) {
    const int e = launch_latent_decode(f32, a, st);
    return e ? e : launch_head_gemm(f32, y, a.out, w, a.B, a.H, N, a.R, yb, yh, q.xb, q.xh, st);
  }
  lat_decode_parts(a, st);
  latent_up_kernel<512><<<dim3((N + 15) / 16, a.H), dim3(256), 0, st>>>(a, q);
  return (int)hipGetLastError();
}

// dynamic LDS above 64 KB
template <int DKP, int DVP, int QF, int NW, int NB>
static int lat_prefill_attr() {
  return (int)hipFuncSetAttribute((const void*)latent_prefill_kernel<DKP, DVP, QF, NW, NB>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)LatLds<DKP, DVP, NB>::BYTES);
}
template <int DKP, int DVP>
static int lat_prefill_lds() {
  int e = lat_prefill_attr<DKP, DVP, 1, 4, 2>();
  if constexpr (DKP <= 192 && DVP <= 128) {
    if (!e) e = lat_prefill_attr<DKP, DVP, 2, 8, 2>();
    if (!e) e = lat_prefill_attr<DKP, DVP, 2, 4, 1>();
  }
  return e;
}
template <int DKP>
static int lat_prefill_lds_v() {
  int e = lat_prefill_lds<DKP, 64>();
  if (!e) e = lat_prefill_lds<DKP, 128>();
  if (!e) e = lat_prefill_lds<DKP, 256>();
  return e;
}
template <int NH, int ND, int KSX>
static int lat_decode_attr() {
  return (int)hipFuncSetAttribute((const void*)latent_decode_kernel<8, NH, ND, KSX>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize,
                                  2 * kLB * (18 * 32 + kLatPad) * 2);
}
template <int RT, int NH, int ND>
static int lat_pair_attr() {
  int e = 0;
  if constexpr (lat_ring<RT, NH>)
    e = (int)hipFuncSetAttribute((const void*)latent_decode_ring_kernel<NH>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                 (int)LatRing<NH>::BYTES);
  if constexpr (lat_pair<RT, NH>)
    if (!e)
      e = (int)hipFuncSetAttribute((const void*)latent_decode_pair_kernel<RT, NH, ND>,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)LatPair<RT, NH, ND>::BYTES);
  return e;
}
template <int NH, int ND>
static int lat_decode_lds() {
  constexpr int NP = NH == 2 ? 4 : ND;
  int e = lat_decode_attr<NH, ND, 0>();
  if (!e) e = lat_decode_attr<NH, ND, 17>();
  if (!e) e = lat_pair_attr<8, NH, NP>();
  if (!e) e = lat_pair_attr<4, NH, NP>();
  return e;
}
int configure_latent() {
  int e = lat_prefill_lds_v<64>();
  if (!e) e = lat_prefill_lds_v<128>();
  if (!e) e = lat_prefill_lds_v<192>();
  if (!e) e = lat_prefill_lds_v<256>();
  if (!e) e = lat_decode_lds<1, 4>();
  if (!e) e = lat_decode_lds<2, 2>();
  if (!e) e = lat_decode_lds<4, 2>();
  return e;
}

}  // namespace drtc
