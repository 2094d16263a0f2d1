// Varlen causal flash-attention forward on MFMA (gfx950), GQA/MQA-aware.
//
// Inputs are read straight out of the fused QKV GEMM output (after the
// in-place RoPE kernel), so no Q/K/V copies are made: sequence s occupies
// rows cu_seqlens[s] .. cu_seqlens[s+1] of the packed [T, qkv_stride] buffer.
//
// Work decomposition: a workgroup owns a 64-row query tile of GH query heads
// sharing one KV head.  Head sizes 64 and 128 run prefill_attn32_kernel (32
// rows per wave, at the end), 256 and single heads of 128 the two kernels of
// 16 rows per wave.
//
// MFMA formulation (16x16x32 bf16): the scores are computed transposed,
//   S^T[key, q] = K[key, :] . Q[q, :]   (A = K from LDS, B = Q^T in registers)
// so that the accumulator tiles of two 16-key halves become the P^T
// B-operand of O^T[d, q] += V^T[d, key] . P^T[key, q] without any lane
// movement (same token permutation trick as the decode kernel).  The online
// softmax per query column needs only two cross-lane xor-shuffles.
#include "common.h"
#include "launchers.h"

#include <type_traits>

namespace drtc {

constexpr int kQT = 64;   // query rows per workgroup
constexpr int kKT = 64;   // keys per LDS tile

// One workgroup = one 64-row query tile x GH query heads that share a KV head
// (4 waves per head, 16 rows per wave): each K/V tile is fetched from HBM and
// staged in LDS ONCE for the GH heads instead of once per head.  Staging is
// split issue-early / write-late (the next tile's global loads are in flight
// during this tile's MFMAs; double-buffered LDS, one barrier per tile).  V is
// staged row-major exactly as loaded (16-B ds_write) and read as the P.V
// A-operand with ds_read_b64_tr_b16 (CDNA4 hardware transpose: lanes 4q+p of a
// 16-lane group address row q / columns 4p..4p+3, lane i receives column i).
// Row paddings: K rows D+8 (conflict-free ds_read_b128), V rows D+16 (the 8
// rows of one tr-read half land on distinct bank octets).
template <int D, int GH>
struct PrefillLds {
  static constexpr int KROW = D + 8;
  static constexpr int VROW = D + 16;
  static constexpr int K_ELEMS = kKT * KROW;
  static constexpr int V_ELEMS = kKT * VROW;
  static constexpr int BUF = K_ELEMS + V_ELEMS;  // one stage
  static constexpr size_t BYTES = (size_t)2 * BUF * 2;
};

typedef short s16x4 __attribute__((ext_vector_type(4)));

DRTC_DEVICE bf16x4 lds_read_tr16(const bf16_t* p) {
  s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) s16x4*)(p));
  return __builtin_bit_cast(bf16x4, v);
}

template <int D, int GH>
__global__ __launch_bounds__(256 * GH) void prefill_attn_kernel(
    bf16_t* __restrict__ out, int out_stride, const bf16_t* __restrict__ qkv,
    int qkv_stride, int Hq, int Hkv, const int* __restrict__ cu_seqlens,
    const int* __restrict__ tile_seq, const int* __restrict__ tile_q0,
    float scale_log2e, int causal) {
  using L = PrefillLds<D, GH>;
  constexpr int NTHR = 256 * GH;
  constexpr int KS = D / 32;
  constexpr int NT = D / 16;
  constexpr int VPR = D / 8;                 // 16-B vectors per K/V row
  constexpr int NV = kKT * VPR / NTHR;       // vectors per thread per operand
  static_assert(NV >= 1 && (kKT * VPR) % NTHR == 0, "staging split");
  extern __shared__ __attribute__((aligned(16))) bf16_t lds[];

  const int tile = blockIdx.x;
  const int G = Hq / Hkv;
  const int groups = G / GH;
  const int hk = blockIdx.y / groups;
  const int hq0 = hk * G + (blockIdx.y - hk * groups) * GH;
  const int w = wave_id_uniform();
  const int hq = hq0 + (w >> 2);
  const int seq = tile_seq[tile];
  const int q0 = tile_q0[tile];
  const int s_begin = cu_seqlens[seq];
  const int seqlen = cu_seqlens[seq + 1] - s_begin;
  const int lane = threadIdx.x & 63;
  const int col = lane & 15, g = lane >> 4;
  const int qrow = q0 + 16 * (w & 3) + col;
  const int k_off = (Hq + hk) * D;
  const int v_off = (Hq + Hkv + hk) * D;
  const int kv_end = causal ? min(seqlen, q0 + kQT) : seqlen;
  const int ntiles = (kv_end + kKT - 1) / kKT;

  bf16x8 kr[NV], vr[NV];
  auto issue = [&](int k0) {
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      const int v = threadIdx.x + n * NTHR;
      const int key = v / VPR;
      const int c = (v - key * VPR) * 8;
      if (k0 + key < seqlen) {
        const bf16_t* rp = qkv + (int64_t)(s_begin + k0 + key) * qkv_stride;
        kr[n] = load_bf16x8(rp + k_off + c);
        vr[n] = load_bf16x8(rp + v_off + c);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) { kr[n][j] = f2bf(0.f); vr[n][j] = f2bf(0.f); }
      }
    }
  };
  auto commit = [&](bf16_t* kb) {
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      const int v = threadIdx.x + n * NTHR;
      const int key = v / VPR;
      const int c = (v - key * VPR) * 8;
      store_bf16x8(kb + key * L::KROW + c, kr[n]);
      store_bf16x8(kb + L::K_ELEMS + key * L::VROW + c, vr[n]);
    }
  };

  issue(0);
  bf16x8 qf[KS];
  {
    const bf16_t* qp = qkv + (int64_t)(s_begin + qrow) * qkv_stride + hq * D;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      if (qrow < seqlen) qf[s] = load_bf16x8(qp + 32 * s + 8 * g);
      else for (int j = 0; j < 8; ++j) qf[s][j] = f2bf(0.f);
    }
  }
  f32x4 o[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i) o[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
  float m = kNegBig, lsum = 0.f;
  // tr-read lane address within a 16-lane group: row q = (lane&15)>>2, cols 4p
  const int tr_off = ((col >> 2) + 4 * g) * L::VROW + 4 * (col & 3);

  for (int kt = 0; kt < ntiles; ++kt) {
    bf16_t* kb = lds + (kt & 1) * L::BUF;
    const bf16_t* vb = kb + L::K_ELEMS;
    commit(kb);
    __syncthreads();
    if (kt + 1 < ntiles) issue((kt + 1) * kKT);
    const int k0 = kt * kKT;

    f32x4 sc[4];
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      sc[st] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        bf16x8 a = load_bf16x8(kb + (16 * st + col) * L::KROW + 32 * s + 8 * g);
        sc[st] = mfma16(a, qf[s], sc[st]);
      }
    }
    float bmax = kNegBig;
#pragma unroll
    for (int st = 0; st < 4; ++st)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int key = k0 + 16 * st + 4 * g + r;
        const bool ok = key < seqlen && (!causal || key <= qrow);
        sc[st][r] = ok ? sc[st][r] * scale_log2e : kNegBig;
        bmax = fmaxf(bmax, sc[st][r]);
      }
    bmax = fmaxf(bmax, __shfl_xor(bmax, 16, 64));
    bmax = fmaxf(bmax, __shfl_xor(bmax, 32, 64));
    const float m_new = fmaxf(m, bmax);
    const float alpha = fast_exp2(m - m_new);
    m = m_new;
    bf16x8 pf[2];
    float psum = 0.f;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float pa = fast_exp2(sc[2 * ks][r] - m_new);
        const float pb = fast_exp2(sc[2 * ks + 1][r] - m_new);
        psum += pa + pb;
        pf[ks][r] = f2bf(pa);
        pf[ks][4 + r] = f2bf(pb);
      }
    lsum = lsum * alpha + psum;
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      o[i] *= alpha;
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const bf16x4 lo = lds_read_tr16(vb + tr_off + 32 * ks * L::VROW + 16 * i);
        const bf16x4 hi = lds_read_tr16(vb + tr_off + (32 * ks + 16) * L::VROW + 16 * i);
        bf16x8 a;
#pragma unroll
        for (int j = 0; j < 4; ++j) { a[j] = lo[j]; a[4 + j] = hi[j]; }
        o[i] = mfma16(a, pf[ks], o[i]);
      }
    }
  }
  lsum += __shfl_xor(lsum, 16, 64);
  lsum += __shfl_xor(lsum, 32, 64);
  if (qrow < seqlen) {
    const float inv = 1.f / lsum;
    bf16_t* op = out + (int64_t)(s_begin + qrow) * out_stride + hq * D + 4 * g;
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      bf16x4 v;
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = f2bf(o[i][r] * inv);
      *reinterpret_cast<bf16x4*>(op + 16 * i) = v;
    }
  }
}

// Persistent variant: resident workgroups loop over the work items (query
// tile, head group), tile-major in the longest-first order of prefill_tiles,
// one item per round of gridDim.x items in snake order.  Chat
// prompts give ~24k items of 1-3 K/V tiles each: with one 1024-thread
// workgroup resident per CU, the non-persistent kernel spends most of its
// time launching and draining workgroups (r1j PMC: waves alive ~20 % of the
// kernel).  Here the waves stay resident; the next item's first K/V tile and
// its Q fragments are loaded while the current item's last tile is computed,
// and the LDS double buffer keeps alternating across items (the barrier of
// each step orders the reuse exactly as inside one item).  Per-tile math is
// identical to prefill_attn_kernel.
template <int D, int GH>
__global__ __launch_bounds__(256 * GH) void prefill_attn_persist_kernel(
    bf16_t* __restrict__ out, int out_stride, const bf16_t* __restrict__ qkv,
    int qkv_stride, int Hq, int Hkv, const int* __restrict__ cu_seqlens,
    const int* __restrict__ tile_seq, const int* __restrict__ tile_q0, int n_tiles,
    float scale_log2e, int causal) {
  using L = PrefillLds<D, GH>;
  constexpr int NTHR = 256 * GH;
  constexpr int KS = D / 32;
  constexpr int NT = D / 16;
  constexpr int VPR = D / 8;
  constexpr int NV = kKT * VPR / NTHR;
  static_assert(NV >= 1 && (kKT * VPR) % NTHR == 0, "staging split");
  extern __shared__ __attribute__((aligned(16))) bf16_t lds[];

  const int G = Hq / Hkv;
  const int groups = G / GH;
  const int n_hg = Hq / GH;
  const int n_work = n_tiles * n_hg;
  const int w = wave_id_uniform();
  const int lane = threadIdx.x & 63;
  const int col = lane & 15, g = lane >> 4;

  struct Item {
    int item, s_begin, seqlen, q0, hq, hk, ntiles;
  };
  auto info = [&](int item) -> Item {
    const int tile = item / n_hg;
    const int hg = item - tile * n_hg;
    const int hk = hg / groups;
    const int hq = hk * G + (hg - hk * groups) * GH + (w >> 2);
    const int seq = tile_seq[tile];
    const int q0 = tile_q0[tile];
    const int s_begin = cu_seqlens[seq];
    const int seqlen = cu_seqlens[seq + 1] - s_begin;
    const int kv_end = causal ? min(seqlen, q0 + kQT) : seqlen;
    return Item{item, s_begin, seqlen, q0, hq, hk, (kv_end + kKT - 1) / kKT};
  };
  bf16x8 kr[NV], vr[NV];
  auto issue = [&](const Item& it, int k0) {
    const int k_off = (Hq + it.hk) * D;
    const int v_off = (Hq + Hkv + it.hk) * D;
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      const int v = threadIdx.x + n * NTHR;
      const int key = v / VPR;
      const int c = (v - key * VPR) * 8;
      if (k0 + key < it.seqlen) {
        const bf16_t* rp = qkv + (int64_t)(it.s_begin + k0 + key) * qkv_stride;
        kr[n] = load_bf16x8(rp + k_off + c);
        vr[n] = load_bf16x8(rp + v_off + c);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) { kr[n][j] = f2bf(0.f); vr[n][j] = f2bf(0.f); }
      }
    }
  };
  auto commit = [&](bf16_t* kb) {
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      const int v = threadIdx.x + n * NTHR;
      const int key = v / VPR;
      const int c = (v - key * VPR) * 8;
      store_bf16x8(kb + key * L::KROW + c, kr[n]);
      store_bf16x8(kb + L::K_ELEMS + key * L::VROW + c, vr[n]);
    }
  };
  auto load_q = [&](bf16x8* qf, const Item& it) {
    const int qrow = it.q0 + 16 * (w & 3) + col;
    const bf16_t* qp = qkv + (int64_t)(it.s_begin + qrow) * qkv_stride + it.hq * D;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      if (qrow < it.seqlen) qf[s] = load_bf16x8(qp + 32 * s + 8 * g);
      else for (int j = 0; j < 8; ++j) qf[s][j] = f2bf(0.f);
    }
  };
  const int tr_off = ((col >> 2) + 4 * g) * L::VROW + 4 * (col & 3);

  // Items are sorted longest-first; a workgroup takes one item per round of
  // gridDim.x items, in snake order (round r even: slot blockIdx.x, odd: the
  // mirrored slot), so every workgroup gets a balanced mix of long and short
  // items instead of the longest of every round.
  const int nwg = gridDim.x;
  auto item_of = [&](int round) -> int {
    const int slot = (round & 1) ? nwg - 1 - (int)blockIdx.x : (int)blockIdx.x;
    return round * nwg + slot;
  };
  int round = 0;
  if (item_of(0) >= n_work) return;
  Item cur = info(item_of(0));
  issue(cur, 0);
  bf16x8 qf[KS], qn[KS];
  load_q(qf, cur);
  int buf = 0;
  while (true) {
    const int qrow = cur.q0 + 16 * (w & 3) + col;
    f32x4 o[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) o[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
    float m = kNegBig, lsum = 0.f;
    const int nxt_item = item_of(round + 1);
    const bool have_next = nxt_item < n_work;
    Item nxt = cur;
    for (int kt = 0; kt < cur.ntiles; ++kt) {
      bf16_t* kb = lds + buf * L::BUF;
      const bf16_t* vb = kb + L::K_ELEMS;
      buf ^= 1;
      commit(kb);
      __syncthreads();
      if (kt + 1 < cur.ntiles) {
        issue(cur, (kt + 1) * kKT);
      } else if (have_next) {
        nxt = info(nxt_item);
        issue(nxt, 0);
        load_q(qn, nxt);
      }
      const int k0 = kt * kKT;
      f32x4 sc[4];
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        sc[st] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          bf16x8 a = load_bf16x8(kb + (16 * st + col) * L::KROW + 32 * s + 8 * g);
          sc[st] = mfma16(a, qf[s], sc[st]);
        }
      }
      float bmax = kNegBig;
#pragma unroll
      for (int st = 0; st < 4; ++st)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int key = k0 + 16 * st + 4 * g + r;
          const bool ok = key < cur.seqlen && (!causal || key <= qrow);
          sc[st][r] = ok ? sc[st][r] * scale_log2e : kNegBig;
          bmax = fmaxf(bmax, sc[st][r]);
        }
      bmax = fmaxf(bmax, __shfl_xor(bmax, 16, 64));
      bmax = fmaxf(bmax, __shfl_xor(bmax, 32, 64));
      const float m_new = fmaxf(m, bmax);
      const float alpha = fast_exp2(m - m_new);
      m = m_new;
      bf16x8 pf[2];
      float psum = 0.f;
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float pa = fast_exp2(sc[2 * ks][r] - m_new);
          const float pb = fast_exp2(sc[2 * ks + 1][r] - m_new);
          psum += pa + pb;
          pf[ks][r] = f2bf(pa);
          pf[ks][4 + r] = f2bf(pb);
        }
      lsum = lsum * alpha + psum;
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        o[i] *= alpha;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          const bf16x4 lo = lds_read_tr16(vb + tr_off + 32 * ks * L::VROW + 16 * i);
          const bf16x4 hi = lds_read_tr16(vb + tr_off + (32 * ks + 16) * L::VROW + 16 * i);
          bf16x8 a;
#pragma unroll
          for (int j = 0; j < 4; ++j) { a[j] = lo[j]; a[4 + j] = hi[j]; }
          o[i] = mfma16(a, pf[ks], o[i]);
        }
      }
    }
    lsum += __shfl_xor(lsum, 16, 64);
    lsum += __shfl_xor(lsum, 32, 64);
    if (qrow < cur.seqlen) {
      const float inv = 1.f / lsum;
      bf16_t* op = out + (int64_t)(cur.s_begin + qrow) * out_stride + cur.hq * D + 4 * g;
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        bf16x4 v;
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = f2bf(o[i][r] * inv);
        *reinterpret_cast<bf16x4*>(op + 16 * i) = v;
      }
    }
    if (!have_next) break;
    cur = nxt;
    ++round;
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[s] = qn[s];
  }
}

// Head sizes 64 and 128: 32 query rows per wave.  What bounds a wave of 16 rows is the LDS: it reads each
// tile's K and V (32 KiB at D = 128) for 512 cycles of MFMA, and 16 waves of a CU take 4096 LDS cycles
// for 2048 of the matrix cores.  Two 32-row column blocks halve that: S^T[key, q] and O^T[d, q] are 32x32x16 MFMAs
// (A = K rows / V columns, B = Q^T / P^T), lane l holds query l % 32 and, of 32 keys, those of its
// half h = l / 32: accumulator word i is key 8 (i / 4) + 4 h + i % 4, so words 8t..8t+7 are the P^T operand of
// the t-th 16 keys as they stand and the V operand is read in the same order of keys.
// A workgroup is the 64-row query tile of GH heads as above, 2 waves per head.  The mask runs on tiles
// that reach past the first query row or the sequence only, the rescaling of O where a maximum grew.
// V rows are padded to 16 banks more than whole turns (the four rows and two column halves of a tr read).
// PERSIST: resident workgroups loop over the items (see prefill_attn_persist_kernel).
// 16 rows per wave -> this, us (TF/s of the causal half): 4 x 4000 tokens of 16 heads over 4 444 -> 331
// (773), 4 x 4096 of 32 over 8 880 -> 636 (865), 15 x 1000 persistent 228 -> 188, 300 x 148 301 -> 292,
// 8 x 2000 of 16 heads of 64 138 -> 101.  What bounds it now is each wave's own chain of scores, softmax
// and output with only two waves to a SIMD (matrix cores busy for about 36 %).
// One head of 128 per workgroup (2 waves, 64 staging registers each) stays with the 16-row waves above:
// 16 x 1000 tokens 172 us there, 173 here, 64 x 150 45 and 53.
template <int D, int GH>
constexpr bool prefill32 = D == 64 || (D == 128 && GH >= 2);

template <int D, int GH>
struct Prefill32 {
  static constexpr int KROW = D + 8;
  static constexpr int VROW = D == 64 ? 96 : D + 32;
  static constexpr int K_ELEMS = kKT * KROW;
  static constexpr int BUF = K_ELEMS + kKT * VROW;
  static constexpr size_t BYTES = (size_t)2 * BUF * 2;
  static constexpr int NTHR = 128 * GH;
};

typedef float f32x16 __attribute__((ext_vector_type(16)));

DRTC_DEVICE f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }

// the other half's value: lanes l and l ^ 32
DRTC_DEVICE float half_max(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

template <int D, int GH, bool PERSIST>
__global__ __launch_bounds__(128 * GH, 2) void prefill_attn32_kernel(
    bf16_t* __restrict__ out, int out_stride, const bf16_t* __restrict__ qkv, int qkv_stride, int Hq, int Hkv,
    const int* __restrict__ cu_seqlens, const int* __restrict__ tile_seq, const int* __restrict__ tile_q0, int n_tiles,
    float scale, float to_q, int causal) {
  using L = Prefill32<D, GH>;
  constexpr int KS = D / 16, NT = D / 32, VPR = D / 8, NV = kKT * VPR / L::NTHR;
  // LDS reads in flight ahead of the MFMAs, in pinned order: left alone the compiler reads an operand or two ahead, and
  // each MFMA waits for most of the LDS's latency (128: 15 x 1000 of 16 heads over 4 108 -> 102 us, 148 of 32 11.2 ->
  // 10.6, 8 x 2000 of 16 over 8 181 -> 176; 64 loses, 8 x 2000 of 16 over 8 112 -> 119)
  constexpr int AHEAD = D == 128 ? 4 : 0;
  static_assert(NV >= 1 && (kKT * VPR) % L::NTHR == 0, "staging split");
  extern __shared__ __attribute__((aligned(16))) bf16_t lds[];
  const int G = Hq / Hkv, groups = G / GH, n_hg = Hq / GH, n_work = n_tiles * n_hg;
  const int w = wave_id_uniform(), lane = threadIdx.x & 63;
  const int col = lane & 31, h = lane >> 5;

  struct Item {
    int s_begin, seqlen, q0, hq, hk, ntiles;
  };
  auto info = [&](int item) -> Item {
    const int tile = item / n_hg, hg = item - tile * n_hg, hk = hg / groups;
    const int seq = tile_seq[tile], q0 = tile_q0[tile], s_begin = cu_seqlens[seq];
    const int seqlen = cu_seqlens[seq + 1] - s_begin;
    const int kv_end = causal ? min(seqlen, q0 + kQT) : seqlen;
    return Item{s_begin, seqlen, q0, hk * G + (hg - hk * groups) * GH + (w >> 1), hk, (kv_end + kKT - 1) / kKT};
  };
  bf16x8 kr[NV], vr[NV];
  auto issue = [&](const Item& it, int k0) {
    const bf16_t* base = qkv + (int64_t)(it.s_begin + k0) * qkv_stride + (Hq + it.hk) * D;
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      const int v = threadIdx.x + n * L::NTHR, key = v / VPR, c = (v - key * VPR) * 8;
      if (k0 + key < it.seqlen) {
        const bf16_t* rp = base + key * qkv_stride + c;
        kr[n] = load_bf16x8(rp);
        vr[n] = load_bf16x8(rp + Hkv * D);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) kr[n][j] = vr[n][j] = f2bf(0.f);
      }
    }
  };
  auto commit = [&](bf16_t* kb) {
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      const int v = threadIdx.x + n * L::NTHR, key = v / VPR, c = (v - key * VPR) * 8;
      store_bf16x8(kb + key * L::KROW + c, kr[n]);
      store_bf16x8(kb + L::K_ELEMS + key * L::VROW + c, vr[n]);
    }
  };
  auto load_q = [&](bf16x8* qf, const Item& it) {
    const int qrow = it.q0 + 32 * (w & 1) + col;
    const bf16_t* qp = qkv + (int64_t)(it.s_begin + qrow) * qkv_stride + it.hq * D + 8 * h;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      if (qrow < it.seqlen) qf[s] = load_bf16x8(qp + 16 * s);
      else for (int j = 0; j < 8; ++j) qf[s][j] = f2bf(0.f);
    }
  };
  auto turn = [&](bf16x8* qf) {
    if (to_q == 1.f) return;
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int j = 0; j < 8; ++j) qf[s][j] = f2bf(bf2f(qf[s][j]) * to_q);
  };
  const int k_at = col * L::KROW + 8 * h;
  const int v_at = (4 * h + ((lane & 15) >> 2)) * L::VROW + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);

  const int nwg = gridDim.x;
  auto item_of = [&](int round) -> int {
    const int slot = (round & 1) ? nwg - 1 - (int)blockIdx.x : (int)blockIdx.x;
    return round * nwg + slot;
  };
  int round = 0, buf = 0;
  if (item_of(0) >= n_work) return;
  Item cur = info(item_of(0));
  issue(cur, 0);
  bf16x8 qf[KS], qn[PERSIST ? KS : 1];
  load_q(qf, cur);
  while (true) {
    turn(qf);
    const int qrow = cur.q0 + 32 * (w & 1) + col;
    // keys below `open` need no mask for any row of the workgroup
    const int open = causal ? min(cur.seqlen, cur.q0 + 1) : cur.seqlen;
    const int last = causal ? min(cur.seqlen - 1, qrow) : cur.seqlen - 1;  // last key of this row
    f32x16 o[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[i][r] = 0.f;
    float m = kNegBig, lsum = 0.f;
    const bool have_next = PERSIST && item_of(round + 1) < n_work;
    Item nxt = cur;
    for (int kt = 0; kt < cur.ntiles; ++kt) {
      bf16_t* kb = lds + buf * L::BUF;
      const bf16_t* vb = kb + L::K_ELEMS + v_at;
      buf ^= 1;
      commit(kb);
      __syncthreads();
      if (kt + 1 < cur.ntiles) {
        issue(cur, (kt + 1) * kKT);
      } else if (have_next) {
        nxt = info(item_of(round + 1));
        issue(nxt, 0);
        if constexpr (PERSIST) load_q(qn, nxt);
      }
      f32x16 sc[2];
      bf16x8 kf[2 * KS], vf[4 * NT];
      auto read_k = [&](int n) { kf[n] = load_bf16x8(kb + 32 * (n / KS) * L::KROW + k_at + 16 * (n % KS)); };
      auto read_v = [&](int n) {
        const bf16_t* p = vb + 16 * (n % 4) * L::VROW + 32 * (n / 4);
        const bf16x4 lo = lds_read_tr16(p), hi = lds_read_tr16(p + 8 * L::VROW);
#pragma unroll
        for (int j = 0; j < 4; ++j) { vf[n][j] = lo[j]; vf[n][4 + j] = hi[j]; }
      };
#pragma unroll
      for (int n = 0; n < AHEAD; ++n) read_k(n);
#pragma unroll
      for (int n = 0; n < 2 * KS; ++n) {
        if constexpr (AHEAD > 0) __builtin_amdgcn_sched_barrier(0);
        if (n + AHEAD < 2 * KS) read_k(n + AHEAD);
        if (n % KS == 0)
#pragma unroll
          for (int r = 0; r < 16; ++r) sc[n / KS][r] = 0.f;
        sc[n / KS] = mfma32(kf[n], qf[n % KS], sc[n / KS]);
      }
      const int k0 = kt * kKT;
      if (k0 + kKT > open) {
        const int past = last - k0 - 4 * h;
#pragma unroll
        for (int st = 0; st < 2; ++st)
#pragma unroll
          for (int r = 0; r < 16; ++r) sc[st][r] = 32 * st + 8 * (r / 4) + r % 4 <= past ? sc[st][r] : kNegBig;
      }
      float top = kNegBig;
#pragma unroll
      for (int st = 0; st < 2; ++st)
#pragma unroll
        for (int r = 0; r < 16; ++r) top = fmaxf(top, sc[st][r]);
      const float m_new = fmaxf(m, half_max(top) * scale);
      const float alpha = fast_exp2(m - m_new);
      if (__any(m != m_new)) {
        lsum *= alpha;
#pragma unroll
        for (int i = 0; i < NT; ++i) o[i] *= alpha;
      }
      m = m_new;
      float psum[4] = {0.f, 0.f, 0.f, 0.f};
      bf16x8 pf[4];
#pragma unroll
      for (int st = 0; st < 2; ++st)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float p = fast_exp2(__builtin_fmaf(sc[st][r], scale, -m));
          psum[r & 3] += p;
          pf[2 * st + r / 8][r % 8] = f2bf(p);
        }
      lsum += (psum[0] + psum[1]) + (psum[2] + psum[3]);
#pragma unroll
      for (int n = 0; n < AHEAD; ++n) read_v(n);
#pragma unroll
      for (int n = 0; n < 4 * NT; ++n) {
        if constexpr (AHEAD > 0) __builtin_amdgcn_sched_barrier(0);
        if (n + AHEAD < 4 * NT) read_v(n + AHEAD);
        o[n / 4] = mfma32(vf[n], pf[n % 4], o[n / 4]);
      }
    }
    lsum += __shfl_xor(lsum, 32, 64);
    if (qrow < cur.seqlen) {
      const float inv = 1.f / lsum;
      bf16_t* op = out + (int64_t)(cur.s_begin + qrow) * out_stride + cur.hq * D + 4 * h;
#pragma unroll
      for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          bf16x4 v;
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = f2bf(o[i][4 * q + r] * inv);
          *reinterpret_cast<bf16x4*>(op + 32 * i + 8 * q) = v;
        }
    }
    if (!have_next) break;
    if constexpr (PERSIST) {
      cur = nxt;
      ++round;
#pragma unroll
      for (int s = 0; s < KS; ++s) qf[s] = qn[s];
    }
  }
}

// every wave's reads and writes of the LDS are done; loads from memory stay in flight
DRTC_DEVICE void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Four heads of 128 and sequences of some length: the scores of the next tile are computed between the exponentials and
// the outputs of this one.  What bounds a wave above is that its matrix instructions and its softmax follow one
// another, and the barrier of each tile keeps the two waves of a SIMD in step.  (4 x 4000 tokens of
// 16 heads over 4: 633,000 -> 587,000 cycles, matrix cores busy 41 -> 44 % of them, waits for an instruction to issue
// 104 -> 77 M of 288 -> 268 M wave cycles; the clock 2.16 -> 2.10 GHz.)
// us, above / this: 4 x 4000 of 16 heads over 4 293 / 280, 4 x 3000 of 32 over 8 324 / 316, one of 700 26.4 / 25.7, of 2000
// 64 / 58 (above without its pinned reads).  Few tiles do not pay for the first one's scores by themselves (one of 256
// 14.2 / 14.7, 16 x 512 90 / 94), two heads not for the registers (8 x 2000 180 / 258), persistent workgroups not for
// theirs (8 x 1000 50.3 / 52.3, 16 x 512 of 32 82.5 / 85.4): the caller picks by the longest sequence.  Every sum is the
// one above's, in its order.
__global__ __launch_bounds__(512, 2) void prefill_ahead_kernel(
    bf16_t* __restrict__ out, int out_stride, const bf16_t* __restrict__ qkv, int qkv_stride, int Hq, int Hkv,
    const int* __restrict__ cu_seqlens, const int* __restrict__ tile_seq, const int* __restrict__ tile_q0,
    float scale, float to_q, int causal) {
  constexpr int D = 128, GH = 4;
  using L = Prefill32<D, GH>;
  constexpr int KS = D / 16, NT = D / 32, VPR = D / 8, NV = kKT * VPR / L::NTHR;
  extern __shared__ __attribute__((aligned(16))) bf16_t lds[];
  const int G = Hq / Hkv, groups = G / GH, n_hg = Hq / GH;
  const int w = wave_id_uniform(), lane = threadIdx.x & 63;
  const int col = lane & 31, h = lane >> 5;

  const int tile = blockIdx.x / n_hg, hg = blockIdx.x - tile * n_hg, hk = hg / groups;
  const int hq = hk * G + (hg - hk * groups) * GH + (w >> 1);
  const int seq = tile_seq[tile], q0 = tile_q0[tile], s_begin = cu_seqlens[seq];
  const int seqlen = cu_seqlens[seq + 1] - s_begin;
  const int ntiles = ((causal ? min(seqlen, q0 + kQT) : seqlen) + kKT - 1) / kKT;
  const int qrow = q0 + 32 * (w & 1) + col;
  // tile kt of K (at = Hq + hk) or V (Hkv further), kept in registers until its place in the LDS is free
  auto issue = [&](bf16x8 (&x)[NV], int at, int kt) {
    const bf16_t* base = qkv + (int64_t)(s_begin + kt * kKT) * qkv_stride + at * D;
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      const int v = threadIdx.x + n * L::NTHR, key = v / VPR, c = (v - key * VPR) * 8;
      if (kt * kKT + key < seqlen) {
        x[n] = load_bf16x8(base + key * qkv_stride + c);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) x[n][j] = f2bf(0.f);
      }
    }
  };
  auto commit = [&](const bf16x8 (&x)[NV], bf16_t* to, int row) {
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      const int v = threadIdx.x + n * L::NTHR, key = v / VPR, c = (v - key * VPR) * 8;
      store_bf16x8(to + key * row + c, x[n]);
    }
  };
  auto ks = [&](int kt) { return lds + (kt & 1) * L::BUF; };
  auto vs = [&](int kt) { return lds + (kt & 1) * L::BUF + L::K_ELEMS; };
  const int k_at = col * L::KROW + 8 * h;
  const int v_at = (4 * h + ((lane & 15) >> 2)) * L::VROW + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);

  bf16x8 kr[NV], k2[NV], vr[NV], qf[KS];
  issue(kr, Hq + hk, 0);
  issue(vr, Hq + Hkv + hk, 0);
  if (ntiles > 1) issue(k2, Hq + hk, 1);
  const bf16_t* qp = qkv + (int64_t)(s_begin + qrow) * qkv_stride + hq * D + 8 * h;
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    if (qrow < seqlen) qf[s] = load_bf16x8(qp + 16 * s);
    else for (int j = 0; j < 8; ++j) qf[s][j] = f2bf(0.f);
  }
  if (to_q != 1.f) {
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int j = 0; j < 8; ++j) qf[s][j] = f2bf(bf2f(qf[s][j]) * to_q);
  }
  // keys below `open` need no mask for any row of the workgroup
  const int open = causal ? min(seqlen, q0 + 1) : seqlen;
  const int last = causal ? min(seqlen - 1, qrow) : seqlen - 1;  // last key of this row
  f32x16 o[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[i][r] = 0.f;
  float m = kNegBig, lsum = 0.f;

  // Tile kt: the softmax and the output of its scores `sc`, and (NEXT) the scores of tile kt + 1 into `sn`.  A slot of
  // the stream holds a score MFMA, an output MFMA of the 16 keys before and the exponentials of 2 keys a
  // lane between them; operands are read two slots ahead.
  auto step = [&](auto next, f32x16 (&sc)[2], f32x16 (&sn)[2], int kt) {
    constexpr bool NEXT = decltype(next)::value;
    constexpr int U = KS / 2, E = 8 / U;  // slots to 16 keys, scores a lane to a slot
    static_assert(NT == U, "an output MFMA to a score MFMA");
    const bf16_t* kb = ks(kt + 1) + k_at;
    const bf16_t* vb = vs(kt) + v_at;
    bf16x8 kf[2 * KS], vf[4 * NT];
    auto read_k = [&](int n) { kf[n] = load_bf16x8(kb + 32 * (n / KS) * L::KROW + 16 * (n % KS)); };
    auto read_v = [&](int n) {  // keys 16 (n / NT).., columns 32 (n % NT)..
      const bf16_t* p = vb + 16 * (n / NT) * L::VROW + 32 * (n % NT);
      const bf16x4 lo = lds_read_tr16(p), hi = lds_read_tr16(p + 8 * L::VROW);
#pragma unroll
      for (int j = 0; j < 4; ++j) { vf[n][j] = lo[j]; vf[n][4 + j] = hi[j]; }
    };
    if constexpr (NEXT) { read_k(0); read_k(1); }
    const int k0 = kt * kKT;
    if (k0 + kKT > open) {
      const int past = last - k0 - 4 * h;
#pragma unroll
      for (int st = 0; st < 2; ++st)
#pragma unroll
        for (int r = 0; r < 16; ++r) sc[st][r] = 32 * st + 8 * (r / 4) + r % 4 <= past ? sc[st][r] : kNegBig;
    }
    float top = kNegBig;
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int r = 0; r < 16; ++r) top = fmaxf(top, sc[st][r]);
    const float m_new = fmaxf(m, half_max(top) * scale);
    if (__any(m != m_new)) {
      const float alpha = fast_exp2(m - m_new);
      lsum *= alpha;
#pragma unroll
      for (int i = 0; i < NT; ++i) o[i] *= alpha;
    }
    m = m_new;
    __builtin_amdgcn_sched_barrier(0);
    float psum[4] = {0.f, 0.f, 0.f, 0.f};
    bf16x8 pf[4];
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int n = U * c + u;
        if constexpr (NEXT) {
          if (n + 2 < 2 * KS) read_k(n + 2);
        }
        if (n + 2 >= U) read_v(n + 2 - U);
        if constexpr (NEXT) {
          if (n % KS == 0)
#pragma unroll
            for (int r = 0; r < 16; ++r) sn[n / KS][r] = 0.f;
          sn[n / KS] = mfma32(kf[n], qf[n % KS], sn[n / KS]);
        }
#pragma unroll
        for (int e = 0; e < E; ++e) {
          if (e == E / 2) {
            __builtin_amdgcn_sched_barrier(0);
            if (c > 0) o[u] = mfma32(vf[n - U], pf[c - 1], o[u]);
          }
          const int r = 8 * (c & 1) + E * u + e;
          const float p = fast_exp2(__builtin_fmaf(sc[c >> 1][r], scale, -m));
          psum[r & 3] += p;
          pf[c][r & 7] = f2bf(p);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    lsum += (psum[0] + psum[1]) + (psum[2] + psum[3]);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (u + 2 < U) read_v(3 * U + u + 2);
      o[u] = mfma32(vf[3 * U + u], pf[3], o[u]);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // what the LDS holds is read and written a tile apart: K a tile ahead of V
  auto turnover = [&](int kt) {
    lds_barrier();
    if (kt + 2 < ntiles) commit(kr, ks(kt), L::KROW);
    commit(vr, vs(kt + 1), L::VROW);
    if (kt + 3 < ntiles) issue(kr, Hq + hk, kt + 3);
    if (kt + 2 < ntiles) issue(vr, Hq + Hkv + hk, kt + 2);
  };
  commit(kr, ks(0), L::KROW);
  commit(vr, vs(0), L::VROW);
  if (ntiles > 1) {
    commit(k2, ks(1), L::KROW);
    issue(vr, Hq + Hkv + hk, 1);
    if (ntiles > 2) issue(kr, Hq + hk, 2);
  }
  lds_barrier();
  f32x16 sa[2], sb[2];
#pragma unroll
  for (int st = 0; st < 2; ++st) {
#pragma unroll
    for (int r = 0; r < 16; ++r) sa[st][r] = 0.f;
#pragma unroll
    for (int s = 0; s < KS; ++s)
      sa[st] = mfma32(load_bf16x8(ks(0) + 32 * st * L::KROW + k_at + 16 * s), qf[s], sa[st]);
  }
  int kt = 0;
  for (; kt + 2 < ntiles; kt += 2) {
    turnover(kt);
    step(std::true_type{}, sa, sb, kt);
    turnover(kt + 1);
    step(std::true_type{}, sb, sa, kt + 1);
  }
  if (kt + 1 < ntiles) {
    turnover(kt);
    step(std::true_type{}, sa, sb, kt);
    sa[0] = sb[0];
    sa[1] = sb[1];
    ++kt;
  }
  lds_barrier();
  step(std::false_type{}, sa, sb, kt);
  lsum += __shfl_xor(lsum, 32, 64);
  if (qrow < seqlen) {
    const float inv = 1.f / lsum;
    bf16_t* op = out + (int64_t)(s_begin + qrow) * out_stride + hq * D + 4 * h;
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        bf16x4 v;
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = f2bf(o[i][4 * q + r] * inv);
        *reinterpret_cast<bf16x4*>(op + 32 * i + 8 * q) = v;
      }
  }
}

// prefill_attn32_kernel's scale and factor of Q for scores scaled by ``s``.  The kernel masks scores ahead
// of the scale, which must keep a masked one (kNegBig) out of reach, and takes the largest one ahead of it
// too: the sign goes to Q, and of scales below 2^-40 (0 as well) the power of two (exact where an element
// of Q stays above 2^-126).
static void split_scale(float s, float& scale, float& to_q) {
  scale = fabsf(s);
  to_q = 1.f;
  if (scale < 0x1p-40f) {
    to_q = scale < 0x1p-126f ? 0.f : ldexpf(1.f, ilogbf(scale));
    scale = to_q > 0.f ? scale / to_q : 1.f;
  }
  if (s < 0.f) to_q = -to_q;
}

static int prefill_persist_grid(int n_work) {
  static int n_cu = 0;
  if (n_cu == 0) {
    int dev = 0;
    (void)hipGetDevice(&dev);
    if (hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        n_cu <= 0)
      n_cu = 256;
  }
  return std::max(1, std::min(n_work, n_cu));
}

template <int D, int GH>
static void launch_tile(dim3 grid, hipStream_t st, bf16_t* out, int out_stride, const bf16_t* qkv,
                      int qkv_stride, int Hq, int Hkv, const int* cu, const int* ts,
                      const int* tq, float sl2, int causal, int persist) {
  const int n_work = (int)(grid.x * grid.y);
  if constexpr (prefill32<D, GH>) {
    using L = Prefill32<D, GH>;
    float scale, to_q;
    split_scale(sl2, scale, to_q);
    if constexpr (GH == 4) {  // with fewer waves to a workgroup the others of its CU fill its gaps
      if (persist == 1) {
        static int per_cu = 0;
        if (per_cu == 0 && (hipOccupancyMaxActiveBlocksPerMultiprocessor(
                                &per_cu, prefill_attn32_kernel<D, GH, true>, L::NTHR, L::BYTES) != hipSuccess ||
                            per_cu <= 0))
          per_cu = 1;
        const int n_wg = std::min(n_work, prefill_persist_grid(n_work * per_cu) * per_cu);
        prefill_attn32_kernel<D, GH, true><<<std::max(1, n_wg), L::NTHR, L::BYTES, st>>>(
            out, out_stride, qkv, qkv_stride, Hq, Hkv, cu, ts, tq, (int)grid.x, scale, to_q, causal);
        return;
      }
    }
    if constexpr (GH == 4) {
      if (persist == 2) {
        prefill_ahead_kernel<<<n_work, L::NTHR, L::BYTES, st>>>(out, out_stride, qkv, qkv_stride, Hq, Hkv, cu, ts, tq, scale,
                                                                to_q, causal);
        return;
      }
    }
    prefill_attn32_kernel<D, GH, false><<<n_work, L::NTHR, L::BYTES, st>>>(
        out, out_stride, qkv, qkv_stride, Hq, Hkv, cu, ts, tq, (int)grid.x, scale, to_q, causal);
  } else {
    constexpr size_t lds_bytes = PrefillLds<D, GH>::BYTES;
    if (persist == 1) {
      // resident workgroups per CU for this instantiation (VGPRs / LDS / waves)
      static int per_cu = 0;
      if (per_cu == 0) {
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &per_cu, prefill_attn_persist_kernel<D, GH>, 256 * GH, lds_bytes) != hipSuccess ||
            per_cu <= 0)
          per_cu = 1;
      }
      const int n_wg = std::min(n_work, prefill_persist_grid(n_work * per_cu) * per_cu);
      prefill_attn_persist_kernel<D, GH><<<dim3(std::max(1, n_wg)), dim3(256 * GH),
                                            lds_bytes, st>>>(
          out, out_stride, qkv, qkv_stride, Hq, Hkv, cu, ts, tq, (int)grid.x, sl2, causal);
      return;
    }
    prefill_attn_kernel<D, GH><<<grid, dim3(256 * GH), lds_bytes, st>>>(
        out, out_stride, qkv, qkv_stride, Hq, Hkv, cu, ts, tq, sl2, causal);
  }
}

template <int D>
static int launch_gh(int GH, int ntiles, int Hq, int Hkv, hipStream_t st, bf16_t* out,
                        int out_stride, const bf16_t* qkv, int qkv_stride, const int* cu,
                        const int* ts, const int* tq, float sl2, int causal, int persist) {
  dim3 grid(ntiles, Hq / GH);
  switch (GH) {
    case 1: launch_tile<D, 1>(grid, st, out, out_stride, qkv, qkv_stride, Hq, Hkv, cu, ts, tq, sl2, causal, persist); break;
    case 2: launch_tile<D, 2>(grid, st, out, out_stride, qkv, qkv_stride, Hq, Hkv, cu, ts, tq, sl2, causal, persist); break;
    case 4:
      if constexpr (D == 128) {
        launch_tile<D, 4>(grid, st, out, out_stride, qkv, qkv_stride, Hq, Hkv, cu, ts, tq, sl2, causal, persist);
        break;
      }
      return -1;
    default: return -1;
  }
  return 0;
}

int launch_prefill_attn(void* out, int out_stride, const void* qkv,
                        int qkv_stride, int Hq, int Hkv, int D,
                        const int* cu_seqlens, const int* tile_seq,
                        const int* tile_q0, int ntiles, float scale, int causal,
                        int persist, hipStream_t st) {
  if (ntiles == 0) return 0;
  if (Hkv <= 0 || Hq % Hkv != 0) return -1;
  const float sl2 = scale * kLog2e;
  const int G = Hq / Hkv;
  // heads per workgroup: 4 for D=128 (1024 threads), 2 for D=64 (one
  // 16-B K and V vector per thread) and D=256 (VGPR budget)
  const int gh_max = D == 128 ? 4 : 2;
  const int GH = gh_max <= G ? gh_max : (G >= 2 ? 2 : 1);
  if (G % GH != 0) return -1;
  const bf16_t* q = (const bf16_t*)qkv;
  bf16_t* o = (bf16_t*)out;
  int rc;
  switch (D) {
    case 64: rc = launch_gh<64>(GH, ntiles, Hq, Hkv, st, o, out_stride, q, qkv_stride, cu_seqlens, tile_seq, tile_q0, sl2, causal, persist); break;
    case 128: rc = launch_gh<128>(GH, ntiles, Hq, Hkv, st, o, out_stride, q, qkv_stride, cu_seqlens, tile_seq, tile_q0, sl2, causal, persist); break;
    case 256: rc = launch_gh<256>(GH, ntiles, Hq, Hkv, st, o, out_stride, q, qkv_stride, cu_seqlens, tile_seq, tile_q0, sl2, causal, persist); break;
    default: return -1;
  }
  if (rc) return rc;
  return (int)hipGetLastError();
}

template <int D, int GH>
static int set_lds() {
  auto set = [](auto* kernel, size_t bytes) {
    return (int)hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  };
  int e;
  if constexpr (prefill32<D, GH>) {
    e = set(prefill_attn32_kernel<D, GH, false>, Prefill32<D, GH>::BYTES);
    if constexpr (GH == 4) {
      if (!e) e = set(prefill_attn32_kernel<D, GH, true>, Prefill32<D, GH>::BYTES);
      if (!e) e = set(prefill_ahead_kernel, Prefill32<D, GH>::BYTES);
    }
  } else {
    e = set(prefill_attn_kernel<D, GH>, PrefillLds<D, GH>::BYTES);
    if (!e) e = set(prefill_attn_persist_kernel<D, GH>, PrefillLds<D, GH>::BYTES);
  }
  return e;
}

int configure_prefill() {
  int e = set_lds<64, 1>();
  if (!e) e = set_lds<64, 2>();
  if (!e) e = set_lds<128, 1>();
  if (!e) e = set_lds<128, 2>();
  if (!e) e = set_lds<128, 4>();
  if (!e) e = set_lds<256, 1>();
  if (!e) e = set_lds<256, 2>();
  return e;
}

}  // namespace drtc
