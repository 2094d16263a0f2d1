// Experts of decode batches with up to a hundred rows or so each (gfx950): W past up to 128 rows of x, both
// through a ring of 64-deep K tiles in LDS.
//
// Bound by one pass over the experts' matrices, 5.2 - 5.5 TB/s here.  What it takes:
//   * Neighbouring rows of W lie 2 K bytes apart.  Where that is a multiple of 4 KB, workgroups that walk K in
//     step ask few of the memory channels at a time: 20 matrices of 1792 x 2048, 200 tokens, 36.9 us (4.0
//     TB/s).  So workgroup b starts its K tiles at b: 28.0 us, and 16 of 3584 x 2048, gated, 58.5 -> 44.
//   * The loads never stop: a table entry's columns are cut evenly over 256 / entries workgroups, one per CU,
//     and what a workgroup has is the tiles - up to 4 NF units of 16 columns, gated 2 NF - of one stream of
//     K tiles.  The ring is ST - 1 K tiles ahead of the products, across the tiles' ends.  (Equal runs over
//     all columns, as gemm_stream.hip deals them, end in the middle of an entry, and the second tile of such a run costs
//     as many steps as the first: 36 against 32 us.)
//   * Rows past an entry's and columns past the tile's are out of the descriptors' range: no memory access, and
//     waves without a row or a column of their own skip the products.  Entries of 64 rows were no faster for a
//     few rows per expert, and read W again above them.
//   * 8 waves, 2 x 4 over rows and columns, 64 x 16 NF outputs each: no exchange at a tile's end.
// A layer with routing, both products and combine, us before and now: 16 x 2048 x 1792, gated, 4 per token: 24 tokens
// 69 -> 67, 128 80 -> 73, 224 101 -> 80, 448 121 -> 92; 20 x 2048 x 1792, squared relu: 48 tokens 65 -> 60, 200 84 -> 68,
// 500 146 -> 86; 16 x 4096 x 3584, gated: 64 247 -> 234, 256 278 -> 254; 8 x 4096 x 14336, 2 per token: 16 467 ->
// 417, 256 522 -> 482; 64 x 2048 x 1408, 6 per token: 256 256 -> 210; 128 x 2048 x 768, 8 per token: 256 302 -> 233.
// Operands: MFMA A = W rows, B = x rows, so lane l holds 4 consecutive columns 4 (l >> 4) .. of row l & 15; gated:
// fragments 2 j and 2 j + 1 are the gate and up rows of the same columns.  LDS rows are 128 bytes,
// 16-byte chunk c of row r at c ^ ((r >> 1) & 7): no bank conflicts.
#include "lds_dma.h"
#include "launchers.h"
#include "typed.h"
#include <algorithm>
#include <initializer_list>

namespace drtc {
namespace {

constexpr int kRingGroups = 256;  // a workgroup to a CU

struct RingMoe {
  bf16_t* y;
  const bf16_t* x;
  const bf16_t* w;
  int N, K, ldx, ldy, act;  // N: output columns; act as launch_moe's, 4: none
  float limit;
  int64_t w_stride;         // elements of an expert's matrix
  const int *tok, *expert, *row0, *rows, *n;
};

template <int NF_>
struct RingCfg {
  static constexpr int FA = kRingRows / 32, NF = NF_;  // 16-row and 16-column fragments of a wave
  static constexpr int BOFF = kRingRows * 128, STAGE = BOFF + 64 * NF * 128;
  static constexpr int DA = FA / 2, DB = NF, D = DA + DB;  // loads per wave and K tile
  static constexpr int ST = 160 * 1024 / STAGE;
  static_assert(FA % 2 == 0 && ST >= 3, "whole loads, and a ring");
};

template <class C, bool GLU, bool GATHER>
__global__ __launch_bounds__(512, 1) void moe_ring_kernel(RingMoe a) {
  constexpr int FA = C::FA, NF = C::NF;
  constexpr int PU = GLU ? 2 * NF : 4 * NF;  // units of 16 output columns to a tile
  extern __shared__ __attribute__((aligned(16))) char ring[];
  const int lane = threadIdx.x & 63, wv = wave_id_uniform(), wm = wv >> 2, wn = wv & 3, r = lane & 15, g = lane >> 4;
  const int units = a.N / 16, n = a.n[0], G = gridDim.x, b = blockIdx.x;
  int q0, q1;
  if (n < 1) return;
  if (n <= G) {
    const int per = G / n, e = b / per, i = b - e * per;
    q0 = e * units + i * units / per;
    q1 = e < n ? e * units + (i + 1) * units / per : q0;
  } else {
    q0 = (int)((int64_t)b * n * units / G);
    q1 = (int)((int64_t)(b + 1) * n * units / G);
  }
  if (q0 >= q1) return;
  const int nk = a.K >> 6;
  // the tile from unit q on: its entry, first unit, units
  auto tile = [&](int q, int& e, int& t, int& u) {
    e = q / units;
    t = q - e * units;
    const int len = min(q1 - q, units - t), parts = (len + PU - 1) / PU;
    u = (len + parts - 1) / parts;
  };

  // ---- loads: an instruction fills 8 rows of 128 bytes; wave wv takes the groups wv, wv + 8, ..
  const unsigned lds0 = (unsigned)(uintptr_t)(lds_ptr)ring;
  const int lr = lane >> 3;
  unsigned va[C::DA], vb[C::DB], off_b[C::DB];
  int unit_b[C::DB];
#pragma unroll
  for (int i = 0; i < C::DB; ++i) {
    const int R = 8 * (wv + 8 * i) + lr, c = (lane & 7) ^ ((R >> 1) & 7);
    const int w = R / (16 * NF), j = R % (16 * NF) / 16;  // wave and fragment of the row
    unit_b[i] = GLU ? w * (NF / 2) + j / 2 : w * NF + j;
    const int src = 16 * unit_b[i] + (R & 15) + (GLU && j & 1 ? a.N : 0);
    off_b[i] = (unsigned)src * (unsigned)(a.K * 2) + c * 16;
  }
  // The first two entries of the run, mostly all, are asked for ahead of everything: a wait for an ordinary
  // load would also wait for the ring.
  struct Entry {
    int expert, row0, rows;
    unsigned va[C::DA];
  };
  auto entry = [&](int e) {
    Entry n;
    n.expert = __builtin_amdgcn_readfirstlane(a.expert[e]);
    n.row0 = __builtin_amdgcn_readfirstlane(a.row0[e]);
    n.rows = __builtin_amdgcn_readfirstlane(a.rows[e]);
#pragma unroll
    for (int i = 0; i < C::DA; ++i) {
      const int R = 8 * (wv + 8 * i) + lr, c = (lane & 7) ^ ((R >> 1) & 7);
      const int src = GATHER ? a.tok[n.row0 + min(R, n.rows - 1)] : n.row0 + R;
      n.va[i] = R < n.rows ? (unsigned)(src * a.ldx * 2 + c * 16) : kNoRow;
    }
    return n;
  };
  const int e0 = q0 / units;
  const Entry first = entry(e0), second = entry(min(e0 + 1, (q1 - 1) / units));
  auto find = [&](int e) { return e == e0 ? first : e == e0 + 1 ? second : entry(e); };
  const __amdgpu_buffer_rsrc_t ra = dma_rsrc(a.x);
  const bf16_t* wt = a.w;
  auto aim = [&](int q) {  // the loads at the tile of unit q; -> the unit behind it
    int e, t, u;
    tile(q, e, t, u);
    const Entry n = find(e);
    wt = a.w + n.expert * a.w_stride + (int64_t)16 * t * a.K;
#pragma unroll
    for (int i = 0; i < C::DA; ++i) va[i] = n.va[i];
#pragma unroll
    for (int i = 0; i < C::DB; ++i) vb[i] = unit_b[i] < u ? off_b[i] : kNoRow;
    return q + u;
  };
  int ahead = aim(q0), lk = 0, fill = 0;  // the unit behind the tile that is loaded, its next K tile, its stage
  unsigned kt = b % nk;
  auto load = [&] {
    const unsigned at = lds0 + fill * C::STAGE;
    const __amdgpu_buffer_rsrc_t rb = dma_rsrc(wt);
#pragma unroll
    for (int i = 0; i < C::DB; ++i) dma16<true>(at + C::BOFF + 1024 * (wv + 8 * i), vb[i], rb, kt * 128u);
#pragma unroll
    for (int i = 0; i < C::DA; ++i) dma16<false>(at + 1024 * (wv + 8 * i), va[i], ra, kt * 128u);
    kt = kt + 1 == nk ? 0 : kt + 1;
    fill = fill + 1 == C::ST ? 0 : fill + 1;
    if (++lk == nk) {
      lk = 0;
      ahead = ahead < q1 ? aim(ahead) : q1 + 1;  // q1 + 1: nothing left
    }
  };
  int flying = 0;
#pragma unroll 1
  for (; flying < C::ST - 1 && ahead <= q1; ++flying) load();

  const int fx = (r >> 1) & 7;
  const char* xa = ring + (16 * FA * wm + r) * 128;
  const char* wa = ring + C::BOFF + (16 * NF * wn + r) * 128;
  int at = 0;
#pragma unroll 1
  for (int q = q0; q < q1;) {
    int e, t, u;
    tile(q, e, t, u);
    q += u;
    const Entry here = find(e);
    const int row0 = here.row0, rows = here.rows, mine = wn * (GLU ? NF / 2 : NF);  // the wave's first unit
    const bool busy = 16 * FA * wm < rows && mine < u;
    f32x4 acc[FA][NF];
#pragma unroll
    for (int i = 0; i < FA; ++i)
#pragma unroll
      for (int j = 0; j < NF; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int k = 0; k < nk; ++k) {
      --flying;
      wait_groups<C::D, C::ST - 2>(flying);
      // everyone's part of the K tile is there, and everyone has read the one before, whose stage is filled next
      lds_barrier();
      if (ahead <= q1) {
        load();
        ++flying;
      }
      if (busy) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int ch = ((4 * h + g) ^ fx) * 16;
          bf16x8 fb[NF], fa[FA];
#pragma unroll
          for (int j = 0; j < NF; ++j) fb[j] = *reinterpret_cast<const bf16x8*>(wa + at + ch + 2048 * j);
#pragma unroll
          for (int i = 0; i < FA; ++i) fa[i] = *reinterpret_cast<const bf16x8*>(xa + at + ch + 2048 * i);
#pragma unroll
          for (int i = 0; i < FA; ++i)
#pragma unroll
            for (int j = 0; j < NF; ++j) acc[i][j] = mfma16(fb[j], fa[i], acc[i][j]);
        }
      }
      at = at + C::STAGE == C::ST * C::STAGE ? 0 : at + C::STAGE;
    }
    if (!busy) continue;
#pragma unroll
    for (int i = 0; i < FA; ++i) {
      const int m = 16 * (FA * wm + i) + r;
      if (m >= rows) continue;
      bf16_t* y = a.y + (int64_t)(row0 + m) * a.ldy + 16 * (t + mine) + 4 * g;
      if constexpr (GLU) {
#pragma unroll
        for (int j = 0; j < NF / 2; ++j) {
          if (mine + j >= u) continue;
          bf16x4 o;
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const float gv = acc[i][2 * j][c], uv = acc[i][2 * j + 1][c];
            o[c] = f2bf(a.act == 0 ? glu_value<0>(gv, uv, 0.f) : a.act == 1 ? glu_value<1>(gv, uv, 0.f)
                                                              : glu_value<2>(gv, uv, a.limit));
          }
          *reinterpret_cast<bf16x4*>(y + 16 * j) = o;
        }
      } else {
#pragma unroll
        for (int j = 0; j < NF; ++j) {
          if (mine + j >= u) continue;
          bf16x4 o;
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const float v = a.act == 3 ? fmaxf(acc[i][j][c], 0.f) : acc[i][j][c];
            o[c] = f2bf(a.act == 3 ? v * v : v);
          }
          *reinterpret_cast<bf16x4*>(y + 16 * j) = o;
        }
      }
    }
  }
}

template <class C, bool GLU, bool GATHER>
int ring_go(const RingMoe& a, hipStream_t st) {
  moe_ring_kernel<C, GLU, GATHER><<<dim3(kRingGroups), dim3(512), C::ST * C::STAGE, st>>>(a);
  return (int)hipGetLastError();
}
template <int NF>
int ring_form(const RingMoe& a, bool glu, hipStream_t st) {
  using C = RingCfg<NF>;
  if constexpr (NF % 2 == 0)
    if (glu) return a.tok ? ring_go<C, true, true>(a, st) : -1;
  return a.tok ? ring_go<C, false, true>(a, st) : ring_go<C, false, false>(a, st);
}
template <int NF>
int ring_cfg() {
  using C = RingCfg<NF>;
  int e = 0;
  for (const void* f : {(const void*)moe_ring_kernel<C, NF % 2 == 0, true>, (const void*)moe_ring_kernel<C, false, true>,
                        (const void*)moe_ring_kernel<C, false, false>})
    e |= (int)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, C::ST * C::STAGE);
  return e;
}
// 32-bit offsets of the rows of x and of an expert's matrix
bool ring_fits(int64_t x_rows, int64_t ldx, int64_t N, int64_t K, bool glu) {
  return x_rows * ldx * 2 < (1ll << 31) && ((glu ? N : 0) + 256) * K * 2 < (1ll << 31);
}

}  // namespace

// Whether both products of a layer of T tokens and P pairs take the form.
bool ring_moe_ok(int T, int P, int H, int I, bool glu) {
  return H % 64 == 0 && I % 64 == 0 && ring_fits(T, H, I, H, glu) && ring_fits(P, I, H, I, false);
}

// Table entries of up to kRingRows rows; x_rows: rows of x (gathered) or pairs; act: of launch_moe, 4: none; tok: rows of
// x by token, or null; entries: about how many there are.
int launch_ring_moe(void* y, const void* x, const void* w, int x_rows, int N, int K, int ldx, int ldy, int act, float limit,
                    int64_t w_stride, const int* tok, const int* expert, const int* row0, const int* rows, const int* n,
                    int entries, hipStream_t st) {
  const bool glu = act < 3;
  if (N < 16 || N % 16 || K < 64 || K % 64 || ldx % 8 || ldy % 4 || act < 0 || act > 4 || w_stride % 8 ||
      !ring_fits(x_rows, ldx, N, K, glu))
    return -1;
  if ((uintptr_t)x % 16 || (uintptr_t)w % 16 || (uintptr_t)y % 8) return -1;
  const RingMoe a{(bf16_t*)y, (const bf16_t*)x, (const bf16_t*)w, N, K, ldx, ldy, act, limit, w_stride, tok, expert, row0,
                  rows, n};
  // the narrowest tile with the fewest parts to a workgroup: narrow ones leave more K tiles in flight
  const int per = std::max(1, kRingGroups / std::max(1, entries)), run = (N / 16 + per - 1) / per;
  int nf = 0, parts = 0;
  for (int f = 2; f <= 4; f += glu ? 2 : 1) {
    const int wide = (glu ? 2 : 4) * f, p = (run + wide - 1) / wide;
    if (!nf || p < parts) nf = f, parts = p;
  }
  return nf == 2 ? ring_form<2>(a, glu, st) : nf == 3 ? ring_form<3>(a, glu, st) : ring_form<4>(a, glu, st);
}

int configure_ring_moe() { return ring_cfg<2>() | ring_cfg<3>() | ring_cfg<4>(); }

}  // namespace drtc
