// Memory-bound fused elementwise kernels for the decoder layer (gfx950).
//
//  * RMSNorm, optionally fused with the residual add that precedes it
//    (residual += x; out = norm(residual) * w), Llama (w) and Gemma (1 + w)
//    weight conventions.  One 256-thread workgroup per row, 16-byte bf16
//    vectors held in registers between the sum-of-squares and the scale pass,
//    so every row is read from HBM exactly once.
//  * Gated activations act(gate) * up (SiLU for Llama/Mixtral, tanh-GELU for
//    Gemma) over the fused [gate | up] GEMM output.
//  * RoPE applied in place on the fused QKV GEMM output, fused with the
//    paged KV-cache write (K token-major [blk][h][tok][d], V dim-major
//    [blk][h][d][tok], the layout the paged decode kernel reads with MFMA).
//    cos/sin come from a host-precomputed fp32 table (no device trig).
#include "common.h"
#include "launchers.h"
#include "router.h"

namespace drtc {

// --------------------------------------------------------------- embedding
// out[row] = table[ids[row]]; a workgroup per row.  A launch and two round trips at decode sizes, where the
// library's form for few rows walks them one after the other: 16 rows of 4096 in 2.2 us (6.7 of the
// library, 12 between two kernels of a step); equal from 200 rows, 16384 in 40 us (6.7 TB/s).  A row of
// a token outside of the vocabulary is NaN.
template <typename I>
__global__ __launch_bounds__(256) void embed_kernel(bf16_t* __restrict__ out, const I* __restrict__ ids,
                                                    const bf16_t* __restrict__ table, int V, int H) {
  const int64_t id = ids[blockIdx.x];
  const bf16_t* from = table + id * H;
  bf16_t* to = out + (int64_t)blockIdx.x * H;
  bf16x8 none;
#pragma unroll
  for (int j = 0; j < 8; ++j) none[j] = f2bf(__builtin_nanf(""));
  const bool there = id >= 0 && id < V;
  for (int i = threadIdx.x * 8; i < H; i += 256 * 8) store_bf16x8(to + i, there ? load_bf16x8(from + i) : none);
}

int launch_embed(void* out, const void* ids, int wide, const void* table, int rows, int V, int H, hipStream_t st) {
  if (rows == 0) return 0;
  if (rows < 0 || V <= 0 || H <= 0 || H % 8) return -1;
  if (wide)
    embed_kernel<<<rows, 256, 0, st>>>((bf16_t*)out, (const int64_t*)ids, (const bf16_t*)table, V, H);
  else
    embed_kernel<<<rows, 256, 0, st>>>((bf16_t*)out, (const int*)ids, (const bf16_t*)table, V, H);
  return (int)hipGetLastError();
}

// ----------------------------------------------------------------- RMSNorm
// PARTS: x is the S fp32 partial sums [S][rows][H] of the product ahead, added up here instead of in a pass of
// its own (4096 columns: 16 rows of 4 parts 4.8 us against 4.7 from bf16 rows, 160 rows of 8 6.5 against 4.9; the pass takes 3 - 8).
// ROUTER: and the logits of the E <= kRouterFuse experts of a mixture, logits[row] = router [E][H] . out[row] in
// fp32 from the rounded row.  A router of its own reads as few bytes, but waits for the norm, its
// launch and two round trips: 13 rows of 4096, 16 experts 4.8 + 13.7 us, now 7.9; 224 of 2048 5.0 + 10.0, now 7.6.  The
// router's rows are asked for ahead of everything, by every row's workgroup: for decode batches only.
template <int VPT, bool GEMMA, bool RESID, bool PARTS = false, bool ROUTER = false>
__global__ __launch_bounds__(256) void rmsnorm_kernel(
    bf16_t* __restrict__ out, bf16_t* __restrict__ residual,
    const void* __restrict__ xv, const bf16_t* __restrict__ w, int H,
    float eps, int x_stride, int out_stride, int res_stride, int S, const bf16_t* __restrict__ router = nullptr,
    float* __restrict__ logits = nullptr, int E = 0) {
  const int row = blockIdx.x;
  const int tid = threadIdx.x;
  [[maybe_unused]] RouterDots<ROUTER ? VPT : 1> dots;
  if constexpr (ROUTER) dots.start(router, H, H, E);
  const bf16_t* xr = (const bf16_t*)xv + (int64_t)row * x_stride;
  float v[VPT][8];
  float ss = 0.f;
  // the weight row is loaded with the activations, not after the reduction: a decode-sized
  // norm (one short workgroup per row) then pays one memory latency, not two
  bf16x8 wv[VPT];
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int idx = (tid + i * 256) * 8;
    if (idx < H) wv[i] = load_bf16x8(w + idx);
  }
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int idx = (tid + i * 256) * 8;
    if (idx < H) {
      bf16x8 a;
      if constexpr (!PARTS) a = load_bf16x8(xr + idx);
      if constexpr (PARTS) {
        bf16_t* rr = residual + (int64_t)row * res_stride + idx;
        const bf16x8 r = load_bf16x8(rr);
        float s[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) s[j] = 0.f;
        add_parts(s, (const float*)xv + (int64_t)row * H + idx, (int64_t)gridDim.x * H, S);
#pragma unroll
        for (int j = 0; j < 8; ++j) a[j] = f2bf(s[j] + bf2f(r[j]));
        store_bf16x8(rr, a);
      } else if constexpr (RESID) {
        bf16_t* rr = residual + (int64_t)row * res_stride + idx;
        bf16x8 r = load_bf16x8(rr);
        bf16x8 s;
#pragma unroll
        for (int j = 0; j < 8; ++j) s[j] = f2bf(bf2f(a[j]) + bf2f(r[j]));
        store_bf16x8(rr, s);
        a = s;
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        v[i][j] = bf2f(a[j]);
        ss += v[i][j] * v[i][j];
      }
    }
  }
  __shared__ float red[4];
  ss = wave_sum(ss);
  if ((tid & 63) == 0) red[tid >> 6] = ss;
  __syncthreads();
  const float tot = red[0] + red[1] + red[2] + red[3];
  const float rstd = rsqrtf(tot / (float)H + eps);
  bf16_t* orow = out + (int64_t)row * out_stride;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int idx = (tid + i * 256) * 8;
    if (idx < H) {
      bf16x8 o;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float ww = bf2f(wv[i][j]);
        if constexpr (GEMMA) ww += 1.f;
        o[j] = f2bf(v[i][j] * rstd * ww);
        if constexpr (ROUTER) v[i][j] = bf2f(o[j]);
      }
      store_bf16x8(orow + idx, o);
    }
  }
  if constexpr (ROUTER) dots.finish(v, logits + (int64_t)row * E);
}

template <bool GEMMA, bool RESID, bool PARTS = false>
static void launch_rmsnorm_t(bf16_t* out, bf16_t* residual, const void* x,
                             const bf16_t* w, int rows, int H, float eps,
                             int x_stride, int out_stride, int res_stride, int S,
                             hipStream_t st) {
  const int vpt = (H / 8 + 255) / 256;
  dim3 grid(rows), block(256);
#define DRTC_RMS_CASE(N)                                                      \
  case N:                                                                    \
    hipLaunchKernelGGL((rmsnorm_kernel<N, GEMMA, RESID, PARTS>), grid, block, \
                       0, st, out, residual, x, w, H, eps, x_stride,          \
                       out_stride, res_stride, S, nullptr, nullptr, 0);       \
    break;
  switch (vpt) {
    DRTC_RMS_CASE(1)
    DRTC_RMS_CASE(2)
    DRTC_RMS_CASE(3)
    DRTC_RMS_CASE(4)
    DRTC_RMS_CASE(8)
    default:
      break;
  }
#undef DRTC_RMS_CASE
}

int launch_rmsnorm(void* out, void* residual, const void* x, const void* w,
                   int rows, int H, float eps, int x_stride, int out_stride,
                   int res_stride, bool gemma, hipStream_t st) {
  const int vpt = (H / 8 + 255) / 256;
  if (H % 8 != 0 || vpt < 1 || (vpt > 4 && vpt != 8)) return -1;
  if (rows == 0) return 0;
  auto o = (bf16_t*)out;
  auto r = (bf16_t*)residual;
  auto ww = (const bf16_t*)w;
  if (residual) {
    if (gemma) launch_rmsnorm_t<true, true>(o, r, x, ww, rows, H, eps, x_stride, out_stride, res_stride, 0, st);
    else launch_rmsnorm_t<false, true>(o, r, x, ww, rows, H, eps, x_stride, out_stride, res_stride, 0, st);
  } else {
    if (gemma) launch_rmsnorm_t<true, false>(o, r, x, ww, rows, H, eps, x_stride, out_stride, res_stride, 0, st);
    else launch_rmsnorm_t<false, false>(o, r, x, ww, rows, H, eps, x_stride, out_stride, res_stride, 0, st);
  }
  return (int)hipGetLastError();
}

// residual += x [rows][H] (or S > 0: the sum of the fp32 parts x [S][rows][H]); out = norm(residual) * w;
// logits [rows][E] = out . router
int launch_rmsnorm_router(void* out, void* residual, const void* x, int S, const void* w, const void* router, float* logits,
                          int E, int rows, int H, float eps, int x_stride, int out_stride, int res_stride,
                          hipStream_t st) {
  const int vpt = (H / 8 + 255) / 256;
  if (H % 8 || vpt < 1 || vpt > 2 || S < 0 || S > kMaxParts || !residual || E < 1 || E > kRouterFuse) return -1;
  if (rows == 0) return 0;
#define DRTC_NORM_ROUTER(V, P)                                                                                    \
  if (vpt == V && (S > 0) == P)                                                                                   \
    rmsnorm_kernel<V, false, true, P, true><<<dim3(rows), dim3(256), 0, st>>>(                                    \
        (bf16_t*)out, (bf16_t*)residual, x, (const bf16_t*)w, H, eps, x_stride, out_stride, res_stride, S,        \
        (const bf16_t*)router, logits, E);
  DRTC_NORM_ROUTER(1, false) DRTC_NORM_ROUTER(1, true) DRTC_NORM_ROUTER(2, false) DRTC_NORM_ROUTER(2, true)
#undef DRTC_NORM_ROUTER
  return (int)hipGetLastError();
}

// residual += the sum of the parts fp32 [S][rows][H]; out = norm(residual) * w
int launch_rmsnorm_parts(void* out, void* residual, const float* parts, int S, const void* w, int rows, int H, float eps,
                         int out_stride, int res_stride, bool gemma, hipStream_t st) {
  const int vpt = (H / 8 + 255) / 256;
  if (H % 8 != 0 || vpt < 1 || (vpt > 4 && vpt != 8) || S < 1 || S > kMaxParts || !residual) return -1;
  if (rows == 0) return 0;
  auto go = gemma ? launch_rmsnorm_t<true, true, true> : launch_rmsnorm_t<false, true, true>;
  go((bf16_t*)out, (bf16_t*)residual, parts, (const bf16_t*)w, rows, H, eps, 0, out_stride, res_stride, S, st);
  return (int)hipGetLastError();
}

// ------------------------------------------------------- gated activations
template <int ACT>  // 0 = SiLU, 1 = tanh-GELU, 2 = clamped
__global__ __launch_bounds__(256) void act_glu_kernel(
    bf16_t* __restrict__ out, const bf16_t* __restrict__ gu, int64_t T, int I,
    int gu_stride, float limit) {
  const int vpr = I / 8;
  const int64_t total = T * vpr;
  for (int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x; v < total;
       v += (int64_t)gridDim.x * 256) {
    const int64_t t = v / vpr;
    const int c = (int)(v - t * vpr) * 8;
    const bf16_t* row = gu + t * gu_stride;
    bf16x8 g = load_bf16x8(row + c);
    bf16x8 u = load_bf16x8(row + I + c);
    bf16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      o[j] = f2bf(glu_value<ACT>(bf2f(g[j]), bf2f(u[j]), limit));
    }
    store_bf16x8(out + t * I + c, o);
  }
}

int launch_act_glu(void* out, const void* gu, int64_t T, int I, int gu_stride,
                   int act, float limit, hipStream_t st) {
  if (I % 8 != 0) return -1;
  const int64_t total = T * (I / 8);
  if (total == 0) return 0;
  int64_t blocks = (total + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  if (act == 0)
    hipLaunchKernelGGL(act_glu_kernel<0>, dim3((unsigned)blocks), dim3(256), 0, st,
                       (bf16_t*)out, (const bf16_t*)gu, T, I, gu_stride, limit);
  else if (act == 1)
    hipLaunchKernelGGL(act_glu_kernel<1>, dim3((unsigned)blocks), dim3(256), 0, st,
                       (bf16_t*)out, (const bf16_t*)gu, T, I, gu_stride, limit);
  else
    hipLaunchKernelGGL(act_glu_kernel<2>, dim3((unsigned)blocks), dim3(256), 0, st,
                       (bf16_t*)out, (const bf16_t*)gu, T, I, gu_stride, limit);
  return (int)hipGetLastError();
}

// ------------------------------------------------------ RoPE + KV write
// qkv: [T][qkv_stride] with heads laid out q(Hq) | k(Hkv) | v(Hkv), each D.
// cos_sin: [max_pos][D] fp32, first D/2 = cos, last D/2 = sin (NeoX halves).
//
// Blocks [0, nseg Hkv): V of a prompt's cache blocks (write_v_block).  Then one a token: a single pass over rope
// items + V items where those are written by the token (threads = their count rounded up to whole waves, looping
// only past 1024), cos/sin read as 16-B vectors, and the V scatter mapped one cache dim per lane: a wave's
// stores then hit 64 consecutive 8-B slots of the dim-major V group (4 cache lines) instead of 8 dims per lane
// (every store instruction spread over 32 lines).  Then one for each row of `pad` to clear.  All three in a
// launch, since each of them is mostly launch where a prompt is short (160 rows, 32 + 8 heads of 128: 4.8 + 3.9
// + 1.8 us in three, now 4.8).
template <int D>
DRTC_DEVICE void write_v_block(const RopeArgs& a, int seg, int h, bf16_t* tile);

template <int D>
__global__ __launch_bounds__(1024) void rope_kv_kernel(RopeArgs a) {
  constexpr int HV = D / 16;
  __shared__ bf16_t tile[32 * (D + 2)];
  int t = blockIdx.x;
  const int Hq = a.Hq, Hkv = a.Hkv, nv = a.nseg * Hkv;
  if (t < nv) {
    write_v_block<D>(a, t / Hkv, t % Hkv, tile);
    return;
  }
  t -= nv;
  if (t >= a.T) {
    bf16_t* row = (bf16_t*)a.pad + (int64_t)(t - a.T) * a.pad_stride;
    for (int i = threadIdx.x; i < a.pad_cols; i += blockDim.x) row[i] = f2bf(0.f);
    return;
  }
  const int n_rope = (Hq + Hkv) * HV;
  const int pos = a.positions[t];
  const int64_t slot = a.slots ? a.slots[t] : -1;
  const int n_items = n_rope + ((slot >= 0 && a.write_v) ? Hkv * (D / 2) : 0);
  bf16_t* row = (bf16_t*)a.qkv + (int64_t)t * a.qkv_stride;
  int64_t blk = 0, off = 0;
  if (slot >= 0) {
    blk = slot / a.block_size;
    off = slot - blk * a.block_size;
  }
  for (int item = threadIdx.x; item < n_items; item += blockDim.x) {
    if (item < n_rope) {
      const int head = item / HV;
      const int vi = item - head * HV;
      const float* cs = a.cos_sin + (int64_t)pos * D + vi * 8;
      const f32x4 ca = *reinterpret_cast<const f32x4*>(cs);
      const f32x4 cb = *reinterpret_cast<const f32x4*>(cs + 4);
      const f32x4 sa = *reinterpret_cast<const f32x4*>(cs + D / 2);
      const f32x4 sb = *reinterpret_cast<const f32x4*>(cs + D / 2 + 4);
      bf16_t* base = row + head * D + vi * 8;
      const bf16x8 x1 = load_bf16x8(base);
      const bf16x8 x2 = load_bf16x8(base + D / 2);
      bf16x8 o1, o2;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float c = j < 4 ? ca[j] : cb[j - 4];
        const float sn = j < 4 ? sa[j] : sb[j - 4];
        const float p = bf2f(x1[j]), q = bf2f(x2[j]);
        o1[j] = f2bf(p * c - q * sn);
        o2[j] = f2bf(q * c + p * sn);
      }
      store_bf16x8(base, o1);
      store_bf16x8(base + D / 2, o2);
      if (head >= Hq && slot >= 0) {
        bf16_t* kd = (bf16_t*)a.k_cache + ((blk * Hkv + (head - Hq)) * a.block_size + off) * D + vi * 8;
        store_bf16x8(kd, o1);
        store_bf16x8(kd + D / 2, o2);
      }
    } else {
      // V block layout: [block_size/4 groups][D][4 tokens] (see write_v_block)
      const int vitem = item - n_rope;
      const int h = vitem / (D / 2);
      const int d = vitem - h * (D / 2);
      const bf16_t* src = row + (Hq + Hkv + h) * D + d;
      bf16_t* vd = (bf16_t*)a.v_cache + (blk * Hkv + h) * D * a.block_size + (off >> 2) * (4 * D) + d * 4 +
                   (off & 3);
      const bf16_t v0 = src[0], v1 = src[D / 2];
      vd[0] = v0;
      vd[2 * D] = v1;  // dim d + D/2: 4 * (D/2) elements further
    }
  }
}

// V of a prompt's cache block, transposed.  V cache block layout (per kv head): 8 groups of 4 tokens, each
// group dim-major [D][4] - the decode kernel's P.V operand wants 4 consecutive
// tokens of one dim in 8 contiguous bytes, and a decode-time write of ONE
// token then touches D 8-byte slots inside a 2*D-byte span (a plain [D][32]
// dim-major block scatters it over D separate 64-B rows: ~8x the HBM write
// traffic).  In prefill a whole block's tokens are contiguous rows of the
// QKV buffer, so one workgroup per (block segment, kv head) stages the
// [32][D] tile in LDS and writes the block with 16-byte stores (two dims x
// 4 tokens each).
template <int D>
DRTC_DEVICE void write_v_block(const RopeArgs& a, int seg, int h, bf16_t* tile) {
  constexpr int BS = 32;
  constexpr int ROW = D + 2;  // padded LDS row (elements)
  const int t0 = a.seg_tok[seg], n = a.seg_len[seg];
  const int64_t blk = a.seg_blk[seg];
  const int voff = (a.Hq + a.Hkv + h) * D;
  for (int v = threadIdx.x; v < BS * (D / 8); v += blockDim.x) {
    const int t = v / (D / 8), c = (v - t * (D / 8)) * 8;
    bf16x8 x;
    if (t < n) x = load_bf16x8((const bf16_t*)a.qkv + (int64_t)(t0 + t) * a.qkv_stride + voff + c);
    else for (int j = 0; j < 8; ++j) x[j] = f2bf(0.f);
#pragma unroll
    for (int j = 0; j < 8; ++j) tile[t * ROW + c + j] = x[j];
  }
  __syncthreads();
  bf16_t* dst = (bf16_t*)a.v_cache + (blk * a.Hkv + h) * (int64_t)D * BS;
  for (int v = threadIdx.x; v < (BS / 4) * (D / 2); v += blockDim.x) {
    const int q4 = v / (D / 2), d = (v - q4 * (D / 2)) * 2;
    bf16x8 y;
#pragma unroll
    for (int j = 0; j < 8; ++j) y[j] = tile[(4 * q4 + (j & 3)) * ROW + d + (j >> 2)];
    store_bf16x8(dst + q4 * (4 * D) + d * 4, y);
  }
}

int launch_rope_kv(const RopeArgs& a, hipStream_t st) {
  if (a.nseg && a.block_size != 32) return -1;
  const int pad = a.pad ? a.pad_rows : 0, grid = a.nseg * a.Hkv + a.T + pad;
  if (grid == 0) return 0;
  const int items = a.T == 0 ? 256 : (a.Hq + a.Hkv) * (a.D / 16) + (a.slots && a.write_v ? a.Hkv * (a.D / 2) : 0);
  const int threads = std::max(a.nseg ? 256 : 64, std::min(1024, (items + 63) / 64 * 64));
  switch (a.D) {
    case 64: rope_kv_kernel<64><<<grid, threads, 0, st>>>(a); break;
    case 128: rope_kv_kernel<128><<<grid, threads, 0, st>>>(a); break;
    case 256: rope_kv_kernel<256><<<grid, threads, 0, st>>>(a); break;
    default: return -1;
  }
  return (int)hipGetLastError();
}

}  // namespace drtc
