// Medium-M projection GEMM (gfx950): y[M, N] = epi(x[M, K] @ W[N, K]^T) for up to 256 rows, bf16 in and out,
// fp32 accumulation, 16x16x32 MFMA.
//
// What bounds it: W is read once (5.3 - 6 TB/s), and a CU takes in 50 - 70 GB/s of operands, from L2 as from
// HBM, however many loads are in flight; less where both mix.  A tile of all M rows and TN columns over a K
// slice costs its CU (M + TN) x slice x 2 bytes, so:
//   * a tile holds all rows, in steps of 32 (rows past M are out of the descriptor's range: no memory access),
//     and 64 or 128 columns of W;
//   * K is cut into slices until the tiles fill the CUs (ops/gemm.py parts_form); the slices' fp32 tiles go
//     to a slab, and the sum is taken by the kernel that reads y next - a residual add and norm - or by
//     midm_reduce_kernel.  The kernel boundary orders them: no atomics, no waiting.  A 32-bit part is written and
//     read instead of a bf16 row: 1 - 2 us against 3 - 8 for a pass, and one rounding less;
//   * x and W pass through LDS (LDS-DMA, a ring of 64-deep K tiles, W non-temporal: every byte enters one CU
//     once).  XCD x takes a contiguous range of the slice-major tile order, so its part of x stays in its L2, and
//     its workgroups start their K walk at different tiles (rows of W a multiple of 4 KB apart, walked in step, ask few
//     memory channels at a time: 32000 x 2048, 64 rows 30.6 -> 24.9 us);
//   * 8 waves: 2 x 2 over the tile, times the two 32-deep halves of a K tile - a wave's fragments are read
//     once for 16 FA x 16 NF outputs, and 8 waves issue loads.  The halves meet in LDS at the end.
// us of the table's kernel / of the slices' sums: 4096 x 4096, 16 rows 11.1 / 8.5, 64 14.1 / 9.9, 160 19.5 / 15.0; 4096 x 14336
// 24.2 / 19.8, 28.3 / 22.7, 39.0 / 30.8; 2048 x 7168 12.3 / 7.6, 22.0 / 9.1, 24.2 / 14.1.
// Operands: MFMA A = W rows, B = x rows, so lane l holds 4 consecutive columns n = 4 (l >> 4) .. of the row
// m = l & 15.  LDS rows are 128 bytes, 16-byte chunk c of row r at c ^ ((r >> 1) & 7): no bank conflicts.
#include "lds_dma.h"
#include "launchers.h"

namespace drtc {
namespace {

constexpr int kMidThreads = 512;
enum { MID_STORE = 0, MID_RESIDUAL = 1, MID_SILU = 2, MID_GELU = 3, MID_SLAB = 4 };

struct MidArgs {
  bf16_t* y;
  float* slab;
  const bf16_t* x;
  const bf16_t* w;
  const bf16_t* res;
  int M, N, K, ldx, ldy, ldr;  // N: rows of W
  int out;
  int tiles, slices, per_xcd;
};

template <int FA_, int NF_>
struct MidCfg {
  static constexpr int FA = FA_, NF = NF_;     // 16-row and 16-column fragments of a wave
  static constexpr int TM = 32 * FA, TN = 32 * NF;
  static constexpr int BOFF = TM * 128, STAGE = BOFF + TN * 128;
  static constexpr int ODD = FA % 2;           // waves 4 .. 7 have one load of x less: one out of range instead
  static constexpr int DA = (FA + 1) / 2, DB = NF / 2, D = DA + DB;  // LDS-DMA per wave and K tile
  static constexpr int FIT = (160 * 1024 - 1024 * ODD) / STAGE;
  static constexpr int ST = FIT < 6 ? FIT : 6;
  static constexpr int LDS = ST * STAGE + 1024 * ODD;
  static_assert(FA * NF * 4096 <= LDS && ST >= 3, "the halves' exchange fits the ring");
};

template <class C, bool GLU>
__global__ __launch_bounds__(kMidThreads, 1) void midm_kernel(MidArgs a) {
  constexpr int FA = C::FA, NF = C::NF;
  extern __shared__ __attribute__((aligned(16))) char mid_lds[];
  const int b = blockIdx.x, item = (b & 7) * a.per_xcd + (b >> 3);
  if (item >= a.tiles * a.slices) return;
  const int slice = item / a.tiles, tile = item - slice * a.tiles;
  const int nkt = a.K >> 6, kt0 = slice * nkt / a.slices, nk = (slice + 1) * nkt / a.slices - kt0;
  constexpr int TNO = GLU ? C::TN / 2 : C::TN;  // output columns of a tile
  const int n0 = tile * TNO, up = a.N / 2;
  const int lane = threadIdx.x & 63, wv = wave_id_uniform();
  const int kg = wv >> 2, wm = (wv >> 1) & 1, wn = wv & 1, r = lane & 15, g = lane >> 4;

  // ---- loads: an instruction fills 8 rows of 128 bytes; wave wv takes the groups wv, wv + 8, ..
  const __amdgpu_buffer_rsrc_t ra = dma_rsrc(a.x + (int64_t)kt0 * 64);
  const __amdgpu_buffer_rsrc_t rb = dma_rsrc(a.w + (int64_t)n0 * a.K + (int64_t)kt0 * 64);
  const unsigned lds0 = (unsigned)(uintptr_t)(lds_ptr)mid_lds;
  unsigned va[C::DA], vb[C::DB];
#pragma unroll
  for (int i = 0; i < C::DA; ++i) {
    const int R = 8 * (wv + 8 * i) + (lane >> 3), c = (lane & 7) ^ ((R >> 1) & 7);
    va[i] = R < C::TM && R < a.M ? (unsigned)(R * a.ldx * 2 + c * 16) : kNoRow;
  }
#pragma unroll
  for (int i = 0; i < C::DB; ++i) {
    const int R = 8 * (wv + 8 * i) + (lane >> 3), c = (lane & 7) ^ ((R >> 1) & 7);
    int src = R;
    if constexpr (GLU) {  // fragments 2 j and 2 j + 1 of a wave: gate and up rows of the same columns
      const int w = R / (16 * NF), j = R % (16 * NF) / 16;
      src = w * 8 * NF + j / 2 * 16 + (R & 15) + (j & 1 ? up : 0);
    }
    vb[i] = (unsigned)src * (unsigned)(a.K * 2) + c * 16;
  }
  const int turn = (b >> 3) % nk;
  auto load = [&](int t, int slot) {
    const int kt = t + turn;
    const unsigned at = lds0 + slot * C::STAGE, k = (unsigned)(kt < nk ? kt : kt - nk) * 128u;
#pragma unroll
    for (int i = 0; i < C::DB; ++i) dma16<true>(at + C::BOFF + 1024 * (wv + 8 * i), vb[i], rb, k);
#pragma unroll
    for (int i = 0; i < C::DA; ++i) {
      unsigned dst = at + 1024 * (wv + 8 * i);
      if (C::ODD && i == C::DA - 1 && wv >= 4) dst = lds0 + C::ST * C::STAGE;
      dma16<false>(dst, va[i], ra, k);
    }
  };
  int issued = 0, fill = 0;
#pragma unroll 1
  for (; issued < min(C::ST - 1, nk); ++issued, ++fill) load(issued, fill);

  const int fx = (r >> 1) & 7, ch = ((4 * kg + g) ^ fx) * 16;
  const char* xa = mid_lds + (16 * FA * wm + r) * 128 + ch;
  const char* wa = mid_lds + C::BOFF + (16 * NF * wn + r) * 128 + ch;
  f32x4 acc[FA][NF];
#pragma unroll
  for (int i = 0; i < FA; ++i)
#pragma unroll
    for (int j = 0; j < NF; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
  int at = 0;
#pragma unroll 1
  for (int t = 0; t < nk; ++t) {
    wait_groups<C::D, C::ST - 2>(issued - t - 1);
    // everyone's part of tile t is there, and everyone has read tile t - 1, whose stage is filled next
    lds_barrier();
    if (issued < nk) {
      load(issued, fill);
      ++issued;
      fill = fill + 1 == C::ST ? 0 : fill + 1;
    }
    bf16x8 fb[NF], fa[FA];
#pragma unroll
    for (int j = 0; j < NF; ++j) fb[j] = *reinterpret_cast<const bf16x8*>(wa + at + 2048 * j);
#pragma unroll
    for (int i = 0; i < FA; ++i) fa[i] = *reinterpret_cast<const bf16x8*>(xa + at + 2048 * i);
#pragma unroll
    for (int i = 0; i < FA; ++i)
#pragma unroll
      for (int j = 0; j < NF; ++j) acc[i][j] = mfma16(fb[j], fa[i], acc[i][j]);
    at = at + C::STAGE == C::ST * C::STAGE ? 0 : at + C::STAGE;
  }

  // ---- the two halves of K: wave kg 0 gets the sums of the row fragments below FI, kg 1 the others
  constexpr int FI = (FA + 1) / 2;
  lds_barrier();  // everyone has read the last tile
  {
    f32x4* to = reinterpret_cast<f32x4*>(mid_lds) + (wv & 3) * (FA * NF * 64) + lane;
#pragma unroll
    for (int i = 0; i < FA; ++i)
      if ((i < FI) == (kg == 1))
#pragma unroll
        for (int j = 0; j < NF; ++j) to[(i * NF + j) * 64] = acc[i][j];
    lds_barrier();
#pragma unroll
    for (int i = 0; i < FA; ++i)
      if ((i < FI) == (kg == 0))
#pragma unroll
        for (int j = 0; j < NF; ++j) acc[i][j] += to[(i * NF + j) * 64];
  }

#pragma unroll
  for (int i = 0; i < FA; ++i) {
    const int m = 16 * (FA * wm + i) + r;
    if ((i < FI) != (kg == 0) || m >= a.M) continue;
    if (a.out == MID_SLAB) {
#pragma unroll
      for (int j = 0; j < NF; ++j) {
        const int n = GLU ? n0 + 8 * NF * wn + j / 2 * 16 + (j & 1 ? up : 0) : n0 + 16 * (NF * wn + j);
        *reinterpret_cast<f32x4*>(a.slab + ((int64_t)slice * a.M + m) * a.N + n + 4 * g) = acc[i][j];
      }
    } else if constexpr (GLU) {
#pragma unroll
      for (int j = 0; j < NF; j += 2) {
        bf16x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          o[e] = f2bf(a.out == MID_SILU ? glu_value<0>(acc[i][j][e], acc[i][j + 1][e], 0.f)
                                        : glu_value<1>(acc[i][j][e], acc[i][j + 1][e], 0.f));
        *reinterpret_cast<bf16x4*>(a.y + (int64_t)m * a.ldy + n0 + 8 * NF * wn + 8 * j + 4 * g) = o;
      }
    } else {
#pragma unroll
      for (int j = 0; j < NF; ++j) {
        const int n = n0 + 16 * (NF * wn + j) + 4 * g;
        f32x4 v = acc[i][j];
        if (a.out == MID_RESIDUAL) {
          const bf16x4 rv = *reinterpret_cast<const bf16x4*>(a.res + (int64_t)m * a.ldr + n);
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] += bf2f(rv[e]);
        }
        bf16x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = f2bf(v[e]);
        *reinterpret_cast<bf16x4*>(a.y + (int64_t)m * a.ldy + n) = o;
      }
    }
  }
}

// Sum the S fp32 partial slabs (fixed order) and apply the epilogue.
//   EPI 0: y = sum;  1: y = bf16(sum + res);  2 / 3: y[:, j] = act(sum[:, j]) *
//   sum[:, j + N/2] with SiLU / GELU-tanh (N = 2 I, the fused [gate | up] rows).
template <int EPI>
__global__ __launch_bounds__(256) void midm_reduce_kernel(bf16_t* __restrict__ y,
                                                          const float* __restrict__ slab,
                                                          const bf16_t* __restrict__ res, int M,
                                                          int N, int S, int ldy, int ldr) {
  const int NO = (EPI >= 2) ? N / 2 : N;  // output columns
  const int per_row = NO / 4;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)M * per_row) return;
  const int m = (int)(i / per_row);
  const int n = (int)(i - (int64_t)m * per_row) * 4;
  f32x4 a = {0.f, 0.f, 0.f, 0.f}, b = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int s = 0; s < S; ++s) {
    const float* row = slab + ((int64_t)s * M + m) * N;
    a += *reinterpret_cast<const f32x4*>(row + n);
    if constexpr (EPI >= 2) b += *reinterpret_cast<const f32x4*>(row + n + NO);
  }
  bf16x4 o;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float v = a[j];
    if constexpr (EPI == 1) v += bf2f(res[(int64_t)m * ldr + n + j]);
    if constexpr (EPI == 2) v = act_value<0>(a[j]) * b[j];
    if constexpr (EPI == 3) v = act_value<1>(a[j]) * b[j];
    o[j] = f2bf(v);
  }
  *reinterpret_cast<bf16x4*>(y + (int64_t)m * ldy + n) = o;
}

template <class C>
int mid_launch(const MidArgs& a, bool glu, hipStream_t st) {
  const dim3 grid(8 * a.per_xcd), block(kMidThreads);
  if (glu) midm_kernel<C, true><<<grid, block, C::LDS, st>>>(a);
  else midm_kernel<C, false><<<grid, block, C::LDS, st>>>(a);
  return (int)hipGetLastError();
}
template <class C>
int mid_cfg() {
  return (int)hipFuncSetAttribute((const void*)midm_kernel<C, true>, hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS) |
         (int)hipFuncSetAttribute((const void*)midm_kernel<C, false>, hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS);
}
#define DRTC_MID_ROWS(X, NF) X(1, NF) X(2, NF) X(3, NF) X(4, NF) X(5, NF) X(6, NF) X(7, NF) X(8, NF)

}  // namespace

int64_t midm_slab_bytes(int M, int N, int S) { return (int64_t)S * M * N * 4; }

// epi: 0 store, 1 residual add (res may alias y), 2 SiLU-GLU, 3 GELU-GLU (N = 2 I, y has N / 2 columns),
// 4: the slices' fp32 sums stay in the slab [S][M][N], y is not written.  nf: 16-column fragments of a
// wave, 2 or 4.  S K slices (at most K / 64); S > 1 or epi 4 needs `slab` (midm_slab_bytes).
int launch_midm_gemm(void* y, const void* x, const void* w, const void* res, int M, int N,
                     int K, int ldx, int ldy, int ldr, int epi, int S, int nf, void* slab,
                     int64_t slab_bytes, hipStream_t st) {
  const bool glu = epi == MID_SILU || epi == MID_GELU;
  if (M < 1 || M > 256 || (nf != 2 && nf != 4) || N < 1 || N % (32 * nf) || K < 64 || K % 64 || S < 1 ||
      S > K / 64 || ldx % 8 || ldy % 4 || epi < 0 || epi > MID_SLAB ||
      (epi == MID_RESIDUAL && (res == nullptr || ldr % 4)))
    return -1;
  if ((uintptr_t)x % 16 || (uintptr_t)w % 16 || (uintptr_t)y % 8 || (uintptr_t)res % 8) return -1;
  // 32-bit offsets from the tile's first row
  if ((int64_t)M * ldx * 2 >= (1ll << 31) || ((int64_t)(glu ? N / 2 : 0) + 32 * nf) * K * 2 >= (1ll << 31)) return -1;
  const bool use_slab = S > 1 || epi == MID_SLAB;
  if (use_slab && (slab == nullptr || slab_bytes < midm_slab_bytes(M, N, S))) return -2;
  const int tiles = N / (32 * nf);
  if ((int64_t)tiles * S >= (1 << 24)) return -1;
  const MidArgs a{(bf16_t*)y, (float*)slab, (const bf16_t*)x, (const bf16_t*)w, (const bf16_t*)res,
                  M, N, K, ldx, ldy, ldr, use_slab ? (int)MID_SLAB : epi, tiles, S, (tiles * S + 7) / 8};
  int e = -1;
#define DRTC_MID(FA, NF) \
  if ((M + 31) / 32 == FA && nf == NF) e = mid_launch<MidCfg<FA, NF>>(a, glu, st);
  DRTC_MID_ROWS(DRTC_MID, 2)
  DRTC_MID_ROWS(DRTC_MID, 4)
#undef DRTC_MID
  if (e || !use_slab || epi == MID_SLAB) return e;
  const int NO = glu ? N / 2 : N;
  const int64_t items = (int64_t)M * (NO / 4);
  const dim3 rgrid((unsigned)((items + 255) / 256)), rblock(256);
  bf16_t* yy = (bf16_t*)y;
  const float* sl = (const float*)slab;
  const bf16_t* rr = (const bf16_t*)res;
  switch (epi) {
    case MID_STORE: midm_reduce_kernel<0><<<rgrid, rblock, 0, st>>>(yy, sl, rr, M, N, S, ldy, ldr); break;
    case MID_RESIDUAL: midm_reduce_kernel<1><<<rgrid, rblock, 0, st>>>(yy, sl, rr, M, N, S, ldy, ldr); break;
    case MID_SILU: midm_reduce_kernel<2><<<rgrid, rblock, 0, st>>>(yy, sl, rr, M, N, S, ldy, ldr); break;
    default: midm_reduce_kernel<3><<<rgrid, rblock, 0, st>>>(yy, sl, rr, M, N, S, ldy, ldr); break;
  }
  return (int)hipGetLastError();
}

int configure_gemm_midm() {
  int e = 0;
#define DRTC_MID(FA, NF) e |= mid_cfg<MidCfg<FA, NF>>();
  DRTC_MID_ROWS(DRTC_MID, 2)
  DRTC_MID_ROWS(DRTC_MID, 4)
#undef DRTC_MID
  return e;
}

}  // namespace drtc
