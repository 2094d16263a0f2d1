// Weight-streaming GEMM of decode batches (gfx950): y[M, N] = epi(x[M, K] @ W[N, K]^T), 1 <= M <= 64,
// bf16 in and out, fp32 accumulation.
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
//   slices: K too long for the registers is cut over up to four workgroups (plain products, M <= 32); a
//           wave that has summed its workgroup's part of a tile leaves it in the workspace (write-through),
//           draws a ticket, and the last one adds the parts in the order of the slices.  No wave waits for
//           another.
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

DRTC_DEVICE bf16x8 load_once(const bf16_t* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(p));
}

// A tile of W past the x in registers, its fragments loaded again from na and nb as they are read.  The sums
// of the wave go to red: products with W row r in row r, plus those in row r ^ 8, which lie 32 lanes away.
template <int KS, int MT>
DRTC_DEVICE void stream_tile(f32x4 (&red)[MT][64], bf16x8 (&wr)[KS], const bf16x8 (&xb)[MT][KS], bool low, int lane,
                             const bf16_t* na, const bf16_t* nb) {
  f32x4 acc[MT][2];
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
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    f32x4 v = acc[mt][0];
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] += __shfl_xor(acc[mt][1][j], 32, 64);
    red[mt][lane] = v;
  }
}

// The waves' sums of token tile mt (gated: of gate and up), in the order of the waves.
template <int NW, int TP, int MT>
DRTC_DEVICE void stream_sum(f32x4 (&v)[TP], const f32x4 (&red)[NW][TP][MT][64], int mt, int lane) {
#pragma unroll
  for (int q = 0; q < TP; ++q) {
    v[q] = red[0][q][mt][lane];
#pragma unroll
    for (int j = 1; j < NW; ++j) v[q] += red[j][q][mt][lane];
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Four values of y.  gated: act 0 SiLU, 1 tanh-GELU, 2 clamped at limit; else squared relu or the sums.
template <int TP>
DRTC_DEVICE bf16x4 stream_value(const f32x4 (&v)[TP], int act, bool relu2, float limit) {
  bf16x4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float f;
    if constexpr (TP == 2)
      f = act == 0 ? glu_value<0>(v[0][i], v[1][i], 0.f) : act == 1 ? glu_value<1>(v[0][i], v[1][i], 0.f)
                                                         : glu_value<2>(v[0][i], v[1][i], limit);
    else
      f = relu2 ? fmaxf(v[0][i], 0.f) * fmaxf(v[0][i], 0.f) : v[0][i];
    o[i] = f2bf(f);
  }
  return o;
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
  auto finish = [&](int t, int mt, const f32x4 (&v)[TP]) {
    if (16 * mt + r >= a.M) return;
    *reinterpret_cast<bf16x4*>(a.y + (int64_t)(16 * mt + r) * a.ldy + 16 * t + 4 * g) =
        stream_value<TP>(v, a.act, a.act == 1, a.limit);
  };
  // slices: this wave's part of token tile mt of tile t to the workspace; the last one adds them
  auto publish = [&](int t, int mt, f32x4 (&v)[TP]) {
    const int64_t part = (int64_t)tiles * MT * 256;
    float* at = a.slab + ((int64_t)t * MT + mt) * 256 + 4 * lane;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      __hip_atomic_store(at + slice * part + i, v[0][i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    int n = 0;
    int* ticket = a.tickets + t * MT + mt;
    if (lane == 0) n = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (__builtin_amdgcn_readfirstlane(n) != a.slices - 1) return;
    if (lane == 0) __hip_atomic_store(ticket, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    v[0] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int z = 0; z < a.slices; ++z)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        v[0][i] += __hip_atomic_load(at + z * part + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    finish(t, mt, v);
  };
  // slices: a wave's sum waits here for the end (one at most, see go): publishing drains its loads.  The
  // branch stays in instances that are never cut: without it the gated ones came out 9 % slower (7168 x 2048,
  // 8 rows 16.4 -> 17.9 us)
  f32x4 held[TP];
  int held_t = -1, held_mt = 0, buf = 0;
#pragma unroll 1
  for (int u = 0;; ++u) {  // gated: u counts gate and up tiles
    const int i = u / TP, t = b + i * G, p = u % TP, p1 = (u + 1) % TP, t1 = b + (u + 1) / TP * G;
    if (t >= tiles) break;
    // behind the last tile: one line of W for all (two forms of the loop would share the selects, all of
    // them ahead of the first load)
    const int64_t next = rows(t1, p1);
    const bool more = t1 < tiles;
    stream_tile<KS, MT>(red[buf][wv][p], wr, xb, low, lane, more ? wa + next : a.w, more ? wb + next : a.w);
    if (p1 != 0) continue;
    lds_barrier();
    // lane l: y[16 mt + (l & 15)][16 t + 4 (l >> 4) ..]; the buffer is written again only behind the
    // next barrier, which this wave reaches after it has read
    const int mt = (wv - MT * i) & (NW - 1);  // MT of the waves, others for the next tile
    if (mt < MT) {
      f32x4 v[TP];
      stream_sum<NW, TP, MT>(v, red[buf], mt, lane);
      if (a.slices == 1) {
        finish(t, mt, v);
      } else {
        held_t = t;
        held_mt = mt;
        held[0] = v[0];
      }
    }
    buf ^= 1;
  }
  if (held_t >= 0) publish(held_t, held_mt, held);
}

// The same over the experts of a mixture: entry i of the device's table is up to 16 MT rows of x for one
// expert's matrix.  The (entry, tile) pairs in order are dealt to the workgroups in equal runs, so a run
// seldom changes its expert; the stream of W goes on while x is read again.  GATHER: rows of x by token.
struct StreamMoe {
  bf16_t* y;
  const bf16_t* x;
  const bf16_t* w;
  int N, K, ldx, ldy, act;  // N: rows of an expert's matrix, gated: half of them
  float limit;
  int64_t w_stride;         // elements of an expert's matrix
  const int *tok, *expert, *row0, *rows, *n;
};
template <int KS, int MT, bool GLU, bool GATHER, int NW>
__global__ __launch_bounds__(64 * NW, KS * (1 + MT) <= 16 && !GLU ? 4 : 2) void stream_moe_kernel(StreamMoe a) {
  static_assert(KS % 2 == 0, "loads come in pairs");
  constexpr int TP = GLU ? 2 : 1;
  __shared__ __attribute__((aligned(16))) f32x4 red[2][NW][TP][MT][64];
  const int wv = wave_id_uniform(), lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int tiles = a.N / 16, units = a.n[0] * tiles, k0 = wv * (32 * KS);
  const int q0 = (int)((int64_t)blockIdx.x * units / gridDim.x), q1 = (int)((int64_t)(blockIdx.x + 1) * units / gridDim.x);
  if (q0 >= q1) return;
  const bool low = r < 8;
  const bf16_t* wa = a.w + (int64_t)(r & 7) * a.K + k0 + (low ? 8 * g : 32 + 8 * g);
  const bf16_t* wb = a.w + (int64_t)(8 + (r & 7)) * a.K + k0 + (low ? 32 + 8 * g : 8 * g);
  int ei = q0 / tiles, t = q0 - ei * tiles;
  auto rows = [&](int64_t base, int t, int p) { return base + ((int64_t)p * a.N + 16 * t) * a.K; };
  int64_t base = a.expert[ei] * a.w_stride;  // this entry's matrix
  bf16x8 wr[KS], xb[MT][KS];
  {
    const int64_t at = rows(base, t, 0);
#pragma unroll
    for (int s = 0; s < KS; s += 2) {
      wr[s] = load_once(wa + at + 32 * s);
      wr[s + 1] = load_once(wb + at + 32 * s);
    }
  }
  const bf16x8 zero = {};
  int row0 = 0, nr = 0, buf = 0, first = 0;
  bool fresh = true;
#pragma unroll 1
  for (int u = q0 * TP; u < q1 * TP; ++u) {
    const int p = u % TP;
    if (fresh) {  // x of this entry
      row0 = a.row0[ei];
      nr = a.rows[ei];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const int m = min(16 * mt + r, nr - 1);
        const bf16_t* xp = a.x + (int64_t)(GATHER ? a.tok[row0 + m] : row0 + m) * a.ldx + k0 + 8 * g;
#pragma unroll
        for (int s = 0; s < KS; ++s) xb[mt][s] = load_bf16x8(xp + 32 * s);
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int s = 0; s < KS; ++s)
          if (16 * mt + r >= nr) xb[mt][s] = zero;
      fresh = false;
    }
    // the tile after this one
    const int e0 = ei, t0 = t;
    const int64_t b0 = base;
    if (p == TP - 1 && ++t == tiles) {
      t = 0;
      ++ei;
      if (u + 1 < q1 * TP) base = a.expert[ei] * a.w_stride;
      fresh = true;
    }
    const bool more = u + 1 < q1 * TP;
    const int64_t next = p == TP - 1 ? rows(base, t, 0) : rows(b0, t0, 1);
    stream_tile<KS, MT>(red[buf][wv][p], wr, xb, low, lane, more ? wa + next : a.w, more ? wb + next : a.w);
    if (p != TP - 1) continue;
    lds_barrier();
    int mt = wv - first;  // MT of the waves from ``first`` on, the next ones for the next tile
    mt += mt < 0 ? NW : 0;
    first = (first + MT) % NW;
    if (mt < MT) {
      f32x4 v[TP];
      stream_sum<NW, TP, MT>(v, red[buf], mt, lane);
      if (16 * mt + r < nr)
        *reinterpret_cast<bf16x4*>(a.y + (int64_t)(row0 + 16 * mt + r) * a.ldy + 16 * t0 + 4 * g) =
            stream_value<TP>(v, a.act, a.act == 3, a.limit);
    }
    buf ^= 1;
  }
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

// K steps and waves of stream_moe for K columns, {0, 0}: none
struct MoeCut { int ks, nw; };
MoeCut moe_cut(int K, int mt) {
  for (const MoeCut c : {MoeCut{8, 8}, MoeCut{8, 7}, MoeCut{16, 8}, MoeCut{14, 8}})
    if (K == 32 * c.ks * c.nw && (mt <= 2 || c.ks == 8)) return c;
  return {0, 0};
}
template <int MT, bool GLU, bool GATHER>
int moe_go(const StreamMoe& a, hipStream_t st) {
  const MoeCut c = moe_cut(a.K, MT);
#define DRTC_MOE_CUT(KS, NW)                                                                                        \
  if (c.ks == KS && c.nw == NW) {                                                                                   \
    stream_moe_kernel<KS, MT, GLU, GATHER, NW>                                                                      \
        <<<dim3(KS * (1 + MT) <= 16 && !GLU ? 512 : 256), dim3(64 * NW), 0, st>>>(a);                               \
    return (int)hipGetLastError();                                                                                  \
  }
  DRTC_MOE_CUT(8, 8)
  DRTC_MOE_CUT(8, 7)
  if constexpr (MT == 1 || (MT == 2 && !GLU)) {  // (stream_moe_tiles)
    DRTC_MOE_CUT(16, 8)
    DRTC_MOE_CUT(14, 8)
  }
#undef DRTC_MOE_CUT
  return -1;
}
template <int MT>
int moe_form(const StreamMoe& a, bool glu, bool gather, hipStream_t st) {
  if (glu) return gather ? moe_go<MT, true, true>(a, st) : -1;
  return gather ? moe_go<MT, false, true>(a, st) : moe_go<MT, false, false>(a, st);
}

}  // namespace

// glu 0: act 0 store, 1 squared relu; glu 1: W holds N gate rows, then N up rows.  slices > 1 (glu 0, M <= 32):
// slab of slices * N / 16 * tiles of M KB and N / 16 * tiles of M tickets, zero (they are left zero).
int launch_stream_gemm(void* y, const void* x, const void* w, int M, int N, int K, int ldx, int ldy, int glu, int act,
                       float limit, int slices, void* slab, int64_t slab_bytes, void* tickets, int n_tickets,
                       hipStream_t st) {
  const int mt = M <= 16 ? 1 : M <= 32 ? 2 : 4;
  if (M < 1 || M > 64 || N < 16 || N % 16 || slices < 1 || slices > 4 || K % (256 * slices) || ldx % 8 || ldy % 4 ||
      act < 0 || act > (glu ? 2 : 1) || (slices > 1 && (glu || mt > 2)))
    return -1;
  const int64_t parts = (int64_t)(N / 16) * mt;
  if (slices > 1 && (!slab || !tickets || slab_bytes < slices * parts * 1024 || n_tickets <= parts))
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

// Tiles of 16 rows that a table entry of the streamed experts holds where they hold ``rows_e`` rows on
// average (1, 2, 4), 0: not taken.  H and I: the columns of the experts' matrices.  An expert with more
// rows than an entry is streamed again, so entries hold half as many more than the average.  us of a whole
// layer against variants 1 and 3, rows: 2048 x 1792, 16 gated experts, 3: 75 / 97, 103; 24: 83 / 100, 105;
// 40: 88 / 101, 106; 50: 105 / 104, 108.  20 squared-relu ones, 40: 89 / 112, 112; 60: 104 / 118, 118.
// 4096 x 3584, gated, 3: 226 / 283, 244; 12: 266 / 296, 259; squared relu, 2: 209 / 293, 255; 19: 221 / 290,
// 259.
int stream_moe_tiles(int rows_e, int H, int I, bool glu) {
  if (H % 16 || I % 16 || H > 16384 || I > 16384) return 0;
  const bool wide = H > 2048 || I > 2048;  // registers for 32 rows at most
  const int mt = rows_e <= 10 ? 1 : rows_e <= 22 && !(wide && glu) ? 2 : rows_e <= (glu ? 44 : 60) && !wide ? 4 : 0;
  return mt && moe_cut(H, mt).ks && moe_cut(I, mt).ks ? mt : 0;
}

// act: of launch_moe (3: squared relu without a gate, 4: none); tok: rows of x by token, or null.
int launch_stream_moe(void* y, const void* x, const void* w, int N, int K, int ldx, int ldy, int mt, int act,
                      float limit, int64_t w_stride, const int* tok, const int* expert, const int* row0,
                      const int* rows, const int* n, hipStream_t st) {
  const bool glu = act < 3;
  if (N % 16 || ldx % 8 || ldy % 4 || act < 0 || act > 4 || (glu && !tok)) return -1;
  const StreamMoe a{(bf16_t*)y, (const bf16_t*)x, (const bf16_t*)w, N, K, ldx, ldy, act, limit, w_stride, tok,
                    expert, row0, rows, n};
  if (mt == 1) return moe_form<1>(a, glu, tok != nullptr, st);
  if (mt == 2) return moe_form<2>(a, glu, tok != nullptr, st);
  if (mt == 4) return moe_form<4>(a, glu, tok != nullptr, st);
  return -1;
}

}  // namespace drtc
