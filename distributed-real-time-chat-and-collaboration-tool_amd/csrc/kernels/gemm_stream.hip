// Weight-streaming GEMM of decode batches (gfx950): y[M, N] = epi(x[M, K] @ W[N, K]^T), 1 <= M <= 64,
// bf16 in and out, fp32 accumulation; optionally x = norm(x + residual) (RMSNorm) on the way in.
//
// The bound is one pass over W.  A persistent workgroup of 8 waves divides K: a wave keeps its
// K / (8 slices) columns of all x rows in registers as MFMA operands, for as long as it lives, and
// streams 16-row tiles of W past them, straight into registers with non-temporal 16-byte loads.  The
// fragment that an MFMA has read is loaded again at once for the next tile, so KS KB per wave - 64 to
// 128 KB per CU - are in flight across the tiles' ends, and no x is read twice.  The 8 partial sums of a
// tile meet in LDS, behind a barrier that waits for LDS only; a wave adds them, another one for each
// tile.
// Non-temporal loads want whole 128-byte lines: 16 rows x 64 bytes to an instruction read 5.6 TB/s here,
// 8 rows x 128 bytes 6.4 (28672 x 4096).  So two loads take a line of the rows 0 .. 7 and one of the rows
// 8 .. 15, and two selects sort their halves into two operands, the second with the rows r ^ 8.
// W of 28672 x 4096, gated, 16 rows of x: 41.8 us (5.6 TB/s) against 58 for the library's GEMM and the
// activation behind it; 32000 x 4096: 46 against 65 us; 64128 x 4096: 90 against 104.
//   x:      lane (r = l & 15, g = l >> 4) holds k = 32 s + 8 g .. of token r; MT tiles of 16 tokens
//   gated:  a gate tile and the up tile at the same rows, one after the other, then act(gate) * up
//   slices: K too long for the registers is cut over workgroups; a wave that has summed its
//           workgroup's part of a tile leaves it in the workspace (write-through), draws a ticket,
//           and the last one adds the parts in the order of the slices.  No wave waits for another.
// Which shapes take it: ops/gemm.py stream_ok.
#include "common.h"
#include "launchers.h"
#include "typed.h"

#include <algorithm>

namespace drtc {
namespace {

struct StreamArgs {
  bf16_t* y;
  const bf16_t* x;
  const bf16_t* w;
  int M, N, K, ldx, ldy;  // N: rows of W, gated: half of them
  int act;                // gated: 0 SiLU, 1 tanh-GELU, 2 clamped at limit; else 0 store, 1 squared relu
  float limit;
  int slices;
  float* slab;
  int* tickets;
};

DRTC_DEVICE void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}
DRTC_DEVICE bf16x8 load_once(const bf16_t* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(p));
}

template <int KS, int MT, bool GLU>
__global__ __launch_bounds__(512, KS * (1 + MT) <= 16 ? 4 : 2) void stream_gemm_kernel(StreamArgs a) {
  static_assert(KS % 2 == 0, "loads come in pairs");
  constexpr int TP = GLU ? 2 : 1, NW = 8;
  __shared__ __attribute__((aligned(16))) f32x4 red[2][NW][TP][MT][64];
  const int wv = wave_id_uniform(), lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int slice = blockIdx.x % a.slices, b = blockIdx.x / a.slices, G = gridDim.x / a.slices;
  const int tiles = a.N / 16, k0 = (slice * NW + wv) * (32 * KS);
  // a pair of loads: 128 bytes of rows 0 .. 7, then of rows 8 .. 15
  const bool low = r < 8;
  const bf16_t* wa = a.w + (int64_t)(r & 7) * a.K + k0 + (low ? 8 * g : 32 + 8 * g);
  const bf16_t* wb = a.w + (int64_t)(8 + (r & 7)) * a.K + k0 + (low ? 32 + 8 * g : 8 * g);
  auto rows = [&](int t, int p) { return ((int64_t)p * a.N + 16 * t) * a.K; };
  bf16x8 wr[KS], xb[MT][KS];
  {
    const int64_t at = rows(b, 0);
#pragma unroll
    for (int s = 0; s < KS; s += 2) {
      wr[s] = load_once(wa + at + 32 * s);
      wr[s + 1] = load_once(wb + at + 32 * s);
    }
  }
  const bf16x8 zero = {};
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int m = 16 * mt + r;
    const bf16_t* xp = a.x + (int64_t)min(m, a.M - 1) * a.ldx + k0 + 8 * g;
#pragma unroll
    for (int s = 0; s < KS; ++s) xb[mt][s] = load_bf16x8(xp + 32 * s);
#pragma unroll
    for (int s = 0; s < KS; ++s)
      if (m >= a.M) xb[mt][s] = zero;
  }
  // products of a tile: [0] with W row r in row r, [1] in row r ^ 8
  f32x4 acc[MT][2];
  auto pass = [&](bool more, int64_t next) {  // next: the rows after these
    // behind the last tile: one line of W for all (two forms of the loop would share the selects, all of
    // them ahead of the first load)
    const bf16_t* na = more ? wa + next : a.w;
    const bf16_t* nb = more ? wb + next : a.w;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt][0] = acc[mt][1] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; s += 2) {
      const u32x4 x = *(const u32x4*)&wr[s], z = *(const u32x4*)&wr[s + 1];
      u32x4 f0, f1;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        f0[i] = low ? x[i] : z[i];
        f1[i] = low ? z[i] : x[i];
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        acc[mt][0] = mfma16(*(const bf16x8*)&f0, xb[mt][s], acc[mt][0]);
        acc[mt][1] = mfma16(*(const bf16x8*)&f1, xb[mt][s + 1], acc[mt][1]);
      }
      wr[s] = load_once(na + 32 * s);
      wr[s + 1] = load_once(nb + 32 * s);
      __builtin_amdgcn_sched_barrier(0);  // a load goes to the registers just read, no others
    }
  };
  auto finish = [&](int t, int mt, const f32x4 (&v)[TP]) {
    if (16 * mt + r >= a.M) return;
    bf16x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float f;
      if constexpr (GLU)
        f = a.act == 0 ? glu_value<0>(v[0][i], v[1][i], 0.f) : a.act == 1 ? glu_value<1>(v[0][i], v[1][i], 0.f)
                                                             : glu_value<2>(v[0][i], v[1][i], a.limit);
      else
        f = a.act == 1 ? fmaxf(v[0][i], 0.f) * fmaxf(v[0][i], 0.f) : v[0][i];
      o[i] = f2bf(f);
    }
    *reinterpret_cast<bf16x4*>(a.y + (int64_t)(16 * mt + r) * a.ldy + 16 * t + 4 * g) = o;
  };
  // slices: this wave's part of token tile mt of tile t to the workspace; the last one adds them
  const int64_t part = (int64_t)tiles * MT * TP * 256;
  auto publish = [&](int t, int mt, f32x4 (&v)[TP]) {
    float* at = a.slab + (((int64_t)t * MT + mt) * TP) * 256 + 4 * lane;
#pragma unroll
    for (int p = 0; p < TP; ++p)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        __hip_atomic_store(at + slice * part + p * 256 + i, v[p][i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    int n = 0;
    int* ticket = a.tickets + t * MT + mt;
    if (lane == 0) n = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (__builtin_amdgcn_readfirstlane(n) != a.slices - 1) return;
    if (lane == 0) __hip_atomic_store(ticket, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int p = 0; p < TP; ++p) v[p] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int z = 0; z < a.slices; ++z)
#pragma unroll
      for (int p = 0; p < TP; ++p)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          v[p][i] += __hip_atomic_load(at + z * part + p * 256 + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    finish(t, mt, v);
  };
  // slices: a wave's sum waits here for the end (one at most, see go): publishing drains its loads
  f32x4 held[TP];
  int held_t = -1, held_mt = 0, buf = 0;
  for (int u = 0;; ++u) {  // gated: u counts gate and up tiles
    const int i = u / TP, t = b + i * G, p = u % TP, p1 = (u + 1) % TP, t1 = b + (u + 1) / TP * G;
    if (t >= tiles) break;
    pass(t1 < tiles, rows(t1, p1));
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      // rows r ^ 8 of the second sum lie 32 lanes away
      f32x4 v = acc[mt][0];
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] += __shfl_xor(acc[mt][1][j], 32, 64);
      red[buf][wv][p][mt][lane] = v;
    }
    if (p1 != 0) continue;
    lds_barrier();
    // lane l: y[16 mt + (l & 15)][16 t + 4 (l >> 4) ..]; the buffer is written again only behind the
    // next barrier, which this wave reaches after it has read
    const int mt = (wv - MT * i) & (NW - 1);  // MT of the waves, others for the next tile
    if (mt < MT) {
      f32x4 v[TP];
#pragma unroll
      for (int q = 0; q < TP; ++q) {
        v[q] = red[buf][0][q][mt][lane];
#pragma unroll
        for (int j = 1; j < NW; ++j) v[q] += red[buf][j][q][mt][lane];
      }
      if (a.slices == 1) {
        finish(t, mt, v);
      } else {
        held_t = t;
        held_mt = mt;
#pragma unroll
        for (int q = 0; q < TP; ++q) held[q] = v[q];
      }
    }
    buf ^= 1;
  }
  if (held_t >= 0) publish(held_t, held_mt, held);
}

template <int KS, int MT, bool GLU>
int go(const StreamArgs& a, hipStream_t st) {
  // one round of workgroups, two to a CU where the registers allow it
  const int cap = (KS * (1 + MT) <= 16 ? 512 : 256) / a.slices, tiles = a.N / 16;
  int rounds = (tiles + cap - 1) / cap;
  if (a.slices > 1) rounds = std::min(rounds, 8 / MT);  // a wave sums one tile at most
  const int G = (tiles + rounds - 1) / rounds;
  stream_gemm_kernel<KS, MT, GLU><<<dim3(G * a.slices), dim3(512), 0, st>>>(a);
  return (int)hipGetLastError();
}
template <int KS, int MT>
int form(const StreamArgs& a, bool glu, hipStream_t st) {
  return glu ? go<KS, MT, true>(a, st) : go<KS, MT, false>(a, st);
}

}  // namespace

// glu 0: act 0 store, 1 squared relu; glu 1: W holds N gate rows, then N up rows.  slices > 1: slab of
// slices * N / 16 * tiles of M * (1 + glu) KB and N / 16 * tiles of M tickets, zero (they are left zero).
int launch_stream_gemm(void* y, const void* x, const void* w, int M, int N, int K, int ldx, int ldy, int glu, int act,
                       float limit, int slices, void* slab, int64_t slab_bytes, void* tickets, int n_tickets,
                       hipStream_t st) {
  const int mt = M <= 16 ? 1 : M <= 32 ? 2 : 4;
  if (M < 1 || M > 64 || N < 16 || N % 16 || slices < 1 || slices > 16 || K % (256 * slices) || ldx % 8 || ldy % 4 ||
      act < 0 || act > (glu ? 2 : 1))
    return -1;
  const int64_t parts = (int64_t)(N / 16) * mt;
  if (slices > 1 && (!slab || !tickets || slab_bytes < slices * parts * (1 + (glu != 0)) * 1024 || n_tickets <= parts))
    return -2;
  const StreamArgs a{(bf16_t*)y, (const bf16_t*)x, (const bf16_t*)w, M, N, K, ldx, ldy, act, limit, slices,
                     (float*)slab, (int*)tickets};
  const int ks = K / (256 * slices);
#define DRTC_STREAM(KS, MT) \
  if (ks == KS && mt == MT) return form<KS, MT>(a, glu != 0, st);
  DRTC_STREAM(8, 1) DRTC_STREAM(14, 1) DRTC_STREAM(16, 1)
  DRTC_STREAM(8, 2) DRTC_STREAM(14, 2) DRTC_STREAM(16, 2)
  DRTC_STREAM(8, 4)
#undef DRTC_STREAM
  return -1;
}

}  // namespace drtc
