// Gated delta rule with per-channel decay (gfx950): short causal convolutions, the recurrence,
// and the gated output norm.
//
// Per head, with the 32-bit state S [dim, vdim] of a sequence:
//   S <- g * S (rows),  u = beta (v - S^T k),  S <- S + k u^T,  o = S^T q
//   out = o / rms(o) * w * sigmoid(gate)
// The columns of S are independent, so a column lives in the registers of 8 lanes: lane 8 c + p
// of a wave holds rows {32 m + 4 p .. + 3} of CPL columns, both products with the decayed state
// are taken in one pass (S^T q = (gS)^T q + u (k.q)) and reduced with three DPP adds.  CPL
// columns share each LDS read of k, q, g.
//   short_conv_kernel    prompt portions: convolution + SiLU of the packed rows; inputs ahead
//                        of a portion come from the sequence's ring of the last `taps` inputs
//   delta_chunk_kernel   one workgroup per (portion, head): 8 tokens at a time in matrix form on
//                        the fp32 MFMA (derivation at the kernel)
//   delta_prep / chain / read_kernel  the same in three launches with chunks of 16 tokens, for a few
//                        long portions (ops/delta.py _chain_ok)
//   delta_scan_kernel    the same token by token, for sizes the chunk form does not take
//   delta_decode_kernel  one workgroup per (sequence, head): all of it for one token; the
//                        state streams through registers once
// A ring entry is position % taps: the entry a token writes is the one its own convolution no
// longer reads, so heads sharing a key never race on it.
#include "hybrid_launchers.h"
#include "typed.h"

#include <algorithm>

namespace drtc {

DRTC_DEVICE float silu_f(float x) { return x / (1.f + expf(-x)); }
// result rounded to bf16: hardware exp and reciprocal
template <class T>
DRTC_DEVICE float silu_as(float x) { return silu_f(x); }
template <>
DRTC_DEVICE float silu_as<bf16_t>(float x) {
  return x * __builtin_amdgcn_rcpf(1.f + fast_exp2(-kLog2e * x));
}
DRTC_DEVICE float sigmoid_f(float x) { return 1.f / (1.f + expf(-x)); }
DRTC_DEVICE float softplus_f(float x) { return x > 20.f ? x : log1pf(expf(x)); }

// ------------------------------------------------------------------ convolution
// VEC channels per thread, 16 consecutive rows per workgroup (the rows behind a row stay in
// the L1).  TAPS 0: any number of taps.
constexpr int kConvRows = 16;

template <class T, int VEC, int TAPS>
__global__ __launch_bounds__(256) void short_conv_kernel(
    T* __restrict__ out, const T* __restrict__ proj, int ldp, const float* __restrict__ w,
    const T* __restrict__ ring, const int* __restrict__ positions,
    const int* __restrict__ row_off, const int* __restrict__ row_state, int rows, int C,
    int taps_rt) {
  const int taps = TAPS ? TAPS : taps_rt;
  const int c = (blockIdx.y * 256 + threadIdx.x) * VEC;
  if (c >= C) return;
  float wr[TAPS ? TAPS : 1][VEC];
  auto loadw = [&](float (&d)[VEC], int j) {
#pragma unroll
    for (int i = 0; i < VEC; ++i) d[i] = w[(int64_t)j * C + c + i];
  };
  if constexpr (TAPS != 0) {
#pragma unroll
    for (int j = 0; j < TAPS; ++j) loadw(wr[j], j);
  }
  auto loadx = [&](float (&d)[VEC], const T* p) {
    if constexpr (VEC == 8) load8(d, p);
    else d[0] = to_f32(*p);
  };
  const int r1 = min(rows, (int)(blockIdx.x + 1) * kConvRows);
  // the inputs of the rows behind: hist[j] belongs to row - 1 - j while ``have`` > j
  float hist[TAPS > 1 ? TAPS - 1 : 1][VEC];
  int have = 0;
  for (int row = blockIdx.x * kConvRows; row < r1; ++row) {
    const int slot = row_state[row];
    float acc[VEC], x0[VEC];
#pragma unroll
    for (int i = 0; i < VEC; ++i) acc[i] = 0.f;
    if (slot >= 0) {
      const int off = row_off[row], pos = positions[row];
      loadx(x0, proj + (int64_t)row * ldp + c);
      auto add = [&](const float (&x)[VEC], const float (&wj)[VEC]) {
#pragma unroll
        for (int i = 0; i < VEC; ++i) acc[i] += x[i] * wj[i];
      };
      auto fetch = [&](float (&x)[VEC], int j) {  // j tokens back; false: before the start
        if (j <= off) loadx(x, proj + (int64_t)(row - j) * ldp + c);
        else if (j <= pos) loadx(x, ring + ((int64_t)slot * taps + (pos - j) % taps) * C + c);
        else return false;
        return true;
      };
      if constexpr (TAPS != 0) {
        add(x0, wr[TAPS - 1]);
#pragma unroll
        for (int j = 1; j < TAPS; ++j) {
          if (j <= have && j <= off) add(hist[j - 1], wr[TAPS - 1 - j]);
          else {
            float x[VEC];
            if (fetch(x, j)) add(x, wr[TAPS - 1 - j]);
          }
        }
      } else {
        loadw(wr[0], taps - 1);
        add(x0, wr[0]);
        for (int j = 1; j < taps; ++j) {
          float x[VEC];
          loadw(wr[0], taps - 1 - j);
          if (fetch(x, j)) add(x, wr[0]);
        }
      }
#pragma unroll
      for (int i = 0; i < VEC; ++i) acc[i] = silu_as<T>(acc[i]);
      if constexpr (TAPS > 1) {
#pragma unroll
        for (int j = TAPS - 2; j > 0; --j)
#pragma unroll
          for (int i = 0; i < VEC; ++i) hist[j][i] = hist[j - 1][i];
#pragma unroll
        for (int i = 0; i < VEC; ++i) hist[0][i] = x0[i];
        ++have;
      }
    } else {
      have = 0;
    }
    T* op = out + (int64_t)row * C + c;
    if constexpr (VEC == 8) store8(op, acc);
    else *op = from_f32<T>(acc[0]);
  }
}

template <class T>
static void conv_t(void* out, const void* proj, int ldp, const float* w, const void* ring,
                   const int* positions, const int* row_off, const int* row_state, int rows,
                   int C, int taps, hipStream_t st) {
  const bool vec = C % 8 == 0 && ldp % 8 == 0;
  const int per = 256 * (vec ? 8 : 1);
  const dim3 grid((rows + kConvRows - 1) / kConvRows, (C + per - 1) / per);
#define DRTC_CONV(V, N)                                                                       \
  short_conv_kernel<T, V, N><<<grid, dim3(256), 0, st>>>((T*)out, (const T*)proj, ldp, w,     \
                                                         (const T*)ring, positions, row_off,  \
                                                         row_state, rows, C, taps)
  if (vec && taps == 4) DRTC_CONV(8, 4);
  else if (vec) DRTC_CONV(8, 0);
  else DRTC_CONV(1, 0);
#undef DRTC_CONV
}

int launch_short_conv(int f32, void* out, const void* proj, int ldp, const float* w,
                      const void* ring, const int* positions, const int* row_off,
                      const int* row_state, int rows, int C, int taps, hipStream_t st) {
  if (rows == 0) return 0;
  if (taps < 1) return -1;
  if (f32) conv_t<float>(out, proj, ldp, w, ring, positions, row_off, row_state, rows, C, taps, st);
  else conv_t<bf16_t>(out, proj, ldp, w, ring, positions, row_off, row_state, rows, C, taps, st);
  return (int)hipGetLastError();
}

// ------------------------------------------------------------------ the recurrence
// This lane's rows of CPL consecutive columns, from / to S [dim, vdim].
template <int DPL, int CPL>
struct StateTile {
  float s[DPL][CPL];
  DRTC_DEVICE void zero() {
#pragma unroll
    for (int i = 0; i < DPL; ++i)
#pragma unroll
      for (int c = 0; c < CPL; ++c) s[i][c] = 0.f;
  }
  DRTC_DEVICE static int row_of(int i, int p) { return 32 * (i >> 2) + 4 * p + (i & 3); }
  DRTC_DEVICE void load(const float* S, int col, int p, int dim, int vdim) {
    if constexpr (CPL % 4 == 0) {
      if ((vdim & 3) == 0) {
#pragma unroll
        for (int i = 0; i < DPL; ++i) {
          const int r = row_of(i, p);
#pragma unroll
          for (int c = 0; c < CPL; c += 4) {
            f32x4 v = {0.f, 0.f, 0.f, 0.f};
            if (r < dim && col + c < vdim)
              v = *reinterpret_cast<const f32x4*>(S + (int64_t)r * vdim + col + c);
#pragma unroll
            for (int j = 0; j < 4; ++j) s[i][c + j] = v[j];
          }
        }
        return;
      }
    }
#pragma unroll
    for (int i = 0; i < DPL; ++i) {
      const int r = row_of(i, p);
#pragma unroll
      for (int c = 0; c < CPL; ++c)
        s[i][c] = r < dim && col + c < vdim ? S[(int64_t)r * vdim + col + c] : 0.f;
    }
  }
  // of a state that fills the tiles: one register of addresses.  NT: non-temporal
  template <bool STORE, bool NT = false>
  DRTC_DEVICE void move_all(float* S, int col, int p, int vdim) {
    static_assert(CPL % 4 == 0, "16-byte pieces");
    const __amdgpu_buffer_rsrc_t at =
        __builtin_amdgcn_make_buffer_rsrc((void*)S, (short)0, 8 * DPL * vdim * 4, 0x00020000);
    const int off = (4 * p * vdim + col) * 4;
#pragma unroll
    for (int i = 0; i < DPL; ++i)
#pragma unroll
      for (int c = 0; c < CPL; c += 4) {
        const int so = row_of(i, 0) * vdim * 4;
        f32x4 v;
        if constexpr (STORE) {
#pragma unroll
          for (int j = 0; j < 4; ++j) v[j] = s[i][c + j];
          // the whole offset in a register of the lanes: behind a 16-byte store whose scalar offset is a register
          // the compiler writes the data's registers again at once, and the store, read late on a busy chip,
          // took lanes 12 - 15 of each 16 from there
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), at, off + 4 * c + so, 0, NT ? 2 : 0);
        } else {
          v = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(at, off + 4 * c, so, NT ? 2 : 0));
#pragma unroll
          for (int j = 0; j < 4; ++j) s[i][c + j] = v[j];
        }
      }
  }
  DRTC_DEVICE void store(float* S, int col, int p, int dim, int vdim) const {
    if constexpr (CPL % 4 == 0) {
      if ((vdim & 3) == 0) {
#pragma unroll
        for (int i = 0; i < DPL; ++i) {
          const int r = row_of(i, p);
#pragma unroll
          for (int c = 0; c < CPL; c += 4) {
            f32x4 v;
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = s[i][c + j];
            if (r < dim && col + c < vdim)
              *reinterpret_cast<f32x4*>(S + (int64_t)r * vdim + col + c) = v;
          }
        }
        return;
      }
    }
#pragma unroll
    for (int i = 0; i < DPL; ++i) {
      const int r = row_of(i, p);
#pragma unroll
      for (int c = 0; c < CPL; ++c)
        if (r < dim && col + c < vdim) S[(int64_t)r * vdim + col + c] = s[i][c];
    }
  }
  // One token: k, q, g rows in LDS (padded to 8 DPL), qk = k.q; o[c] = the read-out.
  DRTC_DEVICE void token(const float* k, const float* q, const float* g, int p, float beta,
                         float qk, const float (&v)[CPL], float (&o)[CPL]) {
    float kk[DPL], ks[CPL], qs[CPL];
#pragma unroll
    for (int c = 0; c < CPL; ++c) ks[c] = qs[c] = 0.f;
#pragma unroll
    for (int m = 0; m < DPL / 4; ++m) {
      const int at = 32 * m + 4 * p;
      const f32x4 k4 = *reinterpret_cast<const f32x4*>(k + at);
      const f32x4 q4 = *reinterpret_cast<const f32x4*>(q + at);
      const f32x4 g4 = *reinterpret_cast<const f32x4*>(g + at);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        kk[4 * m + j] = k4[j];
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
          const float x = s[4 * m + j][c] * g4[j];
          s[4 * m + j][c] = x;
          ks[c] += k4[j] * x;
          qs[c] += q4[j] * x;
        }
      }
    }
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
      const float u = beta * (v[c] - sum8(ks[c]));
      o[c] = sum8(qs[c]) + u * qk;
#pragma unroll
      for (int i = 0; i < DPL; ++i) s[i][c] += kk[i] * u;
    }
  }
};

// Convolution inputs of a portion's last `taps` tokens into the ring, by the workgroup of head h
// (its values; the group's first head also its queries and keys).
template <class T>
DRTC_DEVICE void keep_ring(const DeltaArgs& a, int slot, int h, int n, int row0, int pos0) {
  const int grp = a.H / a.Hk, hk = h / grp;
  const int cq = hk * a.dim, ck = (a.Hk + hk) * a.dim, cv = 2 * a.Hk * a.dim + h * a.vdim;
  const T* proj = (const T*)a.proj;
  T* ring = (T*)a.ring + (int64_t)slot * a.taps * a.C;
  const int nr = min(n, a.taps), own = h % grp == 0 ? 2 * a.dim : 0;
  for (int k = threadIdx.x; k < nr * (own + a.vdim); k += blockDim.x) {
    const int j = k / (own + a.vdim), i = k % (own + a.vdim);
    const int c = i < own ? (i < a.dim ? cq + i : ck + i - a.dim) : cv + i - own;
    const int t = n - nr + j;
    ring[(int64_t)((pos0 + t) % a.taps) * a.C + c] = proj[(int64_t)(row0 + t) * a.ldp + c];
  }
}

template <int DPL>
struct ScanShape {
  static constexpr int DP = 8 * DPL;             // padded key size
  static constexpr int CT = DPL <= 16 ? 16 : 8;  // tokens staged at a time
};

template <class T, int DPL, int CPL>
__global__ __launch_bounds__(512) void delta_scan_kernel(DeltaArgs a) {
  constexpr int DP = ScanShape<DPL>::DP, CT = ScanShape<DPL>::CT;
  extern __shared__ __attribute__((aligned(16))) float sm[];
  const int seg = blockIdx.x, h = blockIdx.y;
  const int slot = a.seg_state[seg];
  const int n = a.seg_len[seg], row0 = a.seg_row[seg], pos0 = a.seg_pos[seg];
  const int tid = threadIdx.x, nthr = blockDim.x;
  T* out = (T*)a.out;
  const int ldo = a.H * a.vdim;
  if (slot < 0) {  // padding row of a decode bucket
    for (int i = tid; i < n * a.vdim; i += nthr)
      out[(int64_t)(row0 + i / a.vdim) * ldo + h * a.vdim + i % a.vdim] = from_f32<T>(0.f);
    return;
  }
  const int dvp = (a.vdim + 3) & ~3;
  float* ks = sm;
  float* qs = ks + CT * DP;
  float* gs = qs + CT * DP;
  float* vs = gs + CT * DP;
  float* os = vs + CT * dvp;
  float* qk = os + CT * dvp;
  float* bs = qk + CT;

  const int lane = tid & 63, p = lane & 7;
  const int col = ((tid >> 6) * 8 + (lane >> 3)) * CPL;
  const int grp = a.H / a.Hk, hk = h / grp;
  const int cq = hk * a.dim, ck = (a.Hk + hk) * a.dim, cv = 2 * a.Hk * a.dim + h * a.vdim;
  const float aexp = a.a_exp[h], qscale = rsqrtf((float)a.dim);
  float* S = a.state + ((int64_t)slot * a.H + h) * a.dim * a.vdim;
  StateTile<DPL, CPL> st;
  if (pos0 > 0) st.load(S, col, p, a.dim, a.vdim);
  else st.zero();
  const int l16 = tid & 15, g16 = tid >> 4, n16 = nthr >> 4;
  const T* conv = (const T*)a.conv;
  const T* proj = (const T*)a.proj;
  const T* dec = (const T*)a.decay;
  const T* gate = (const T*)a.gate;

  for (int t0 = 0; t0 < n; t0 += CT) {
    const int nt = min(CT, n - t0);
    for (int t = g16; t < nt; t += n16) {  // 16 lanes per token
      const int64_t row = row0 + t0 + t;
      const T* cr = conv + row * a.C;
      float sq = 0.f, sk = 0.f, dot = 0.f;
      for (int i = l16; i < DP; i += 16) {
        const float q = i < a.dim ? to_f32(cr[cq + i]) : 0.f;
        const float k = i < a.dim ? to_f32(cr[ck + i]) : 0.f;
        sq += q * q;
        sk += k * k;
        dot += q * k;
        gs[t * DP + i] = i < a.dim
            ? expf(-aexp * softplus_f(to_f32(dec[row * a.ld_decay + h * a.dim + i]) +
                                      a.dt_bias[h * a.dim + i]))
            : 1.f;
        qs[t * DP + i] = q;
        ks[t * DP + i] = k;
      }
      const float rq = qscale / sqrtf(sum16(sq) + 1e-6f), rk = 1.f / sqrtf(sum16(sk) + 1e-6f);
      dot = sum16(dot);
      for (int i = l16; i < DP; i += 16) {
        qs[t * DP + i] *= rq;
        ks[t * DP + i] *= rk;
      }
      for (int i = l16; i < a.vdim; i += 16) vs[t * dvp + i] = to_f32(cr[cv + i]);
      if (l16 == 0) {
        qk[t] = dot * rq * rk;
        bs[t] = sigmoid_f(to_f32(proj[row * a.ldp + a.off_b + h]));
      }
    }
    __syncthreads();
    if (col < a.vdim) {
      for (int t = 0; t < nt; ++t) {
        float v[CPL], o[CPL];
#pragma unroll
        for (int c = 0; c < CPL; ++c) v[c] = col + c < a.vdim ? vs[t * dvp + col + c] : 0.f;
        st.token(ks + t * DP, qs + t * DP, gs + t * DP, p, bs[t], qk[t], v, o);
        if (p == 0) {
#pragma unroll
          for (int c = 0; c < CPL; ++c)
            if (col + c < a.vdim) os[t * dvp + col + c] = o[c];
        }
      }
    }
    __syncthreads();
    for (int t = g16; t < nt; t += n16) {
      const int64_t row = row0 + t0 + t;
      float so = 0.f;
      for (int i = l16; i < a.vdim; i += 16) {
        const float o = os[t * dvp + i];
        so += o * o;
      }
      const float r = 1.f / sqrtf(sum16(so) / (float)a.vdim + a.eps);
      for (int i = l16; i < a.vdim; i += 16)
        out[row * ldo + h * a.vdim + i] =
            from_f32<T>(os[t * dvp + i] * r * a.norm_w[i] *
                        sigmoid_f(to_f32(gate[row * a.ld_gate + h * a.vdim + i])));
    }
    // the next chunk's staging writes ks / qs / gs / vs, last read before the barrier above;
    // os is written again only after the next barrier
  }
  if (col < a.vdim) st.store(S, col, p, a.dim, a.vdim);
  keep_ring<T>(a, slot, h, n, row0, pos0);
}


// ------------------------------------------------------------------ chunks on the fp32 MFMA
// For the tokens 1..8 of a chunk let c_i be the running sum of log2 g (per key channel),
// S the state ahead of the chunk, E_i = 2^{c_i}.  Unrolling the recurrence,
//   S_i = E_i * S + sum_{j <= i} (2^{c_i - c_j} * k_j) u_j^T
//   u_i = beta_i (v_i - (E_i * k_i)^T S - sum_{j < i} A_ij u_j),  A_ij = k_i . (2^{c_i - c_j} * k_j)
//   o_i = (E_i * q_i)^T S + sum_{j <= i} B_ij u_j,                B_ij = q_i . (2^{c_i - c_j} * k_j)
// (exponents of differences are never positive: no decay is divided by).  With R = V - (E*K)^T S,
//   U = (I + diag(beta) A)^{-1} diag(beta) R = M_U R,   O = (E*Q)^T S + B U = (E*Q)^T S + M_O R.
// All products with S are 16-row MFMAs - 8 key rows and 8 query rows of a chunk - and so are
// the products with [M_U; M_O]; the 8 x 8 inverse is a forward substitution shared by all
// columns.  A wave keeps 32 columns of S as accumulator tiles: their layout (row 4 g + r of
// lane group g) is also a B operand with k-step r taking dim 4 g + r, so S feeds its own
// products without lane movement.
// 16 tokens (two chunks) are staged at a time; their global loads are in flight while the
// previous 16 are computed.
DRTC_DEVICE f32x4 mfma_f32(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
DRTC_DEVICE float log2_fast(float x) { return __builtin_amdgcn_logf(x); }
// softplus by hardware exp2 / log2; for large -x its series, where 1 + e^x would round
DRTC_DEVICE float softplus_hw(float x) {
  const float e = fast_exp2(x * kLog2e);
  const float l = log2_fast(1.f + e) * (1.f / kLog2e);
  return x > 20.f ? x : x < -6.f ? e * (1.f - e * (0.5f - e * (1.f / 3.f))) : l;
}
DRTC_DEVICE float sigmoid_hw(float x) {
  return 1.f / (1.f + fast_exp2(-kLog2e * x));
}

template <int DT, int NTHR>
struct ChunkLds {
  static constexpr int DP = 16 * DT, DS = DP + 4, KD = DP + 16;
  static constexpr int NW = NTHR / 64, VS = 32 * NW + 4, UB = 36;
  static constexpr int k = 0, q = k + 16 * DS, c = q + 16 * DS, kd = c + 16 * DS;
  static constexpr int gt = kd + 16 * KD, v = gt + 2 * DP, mm = v + 16 * VS, beta = mm + 256;
  static constexpr int tmp = beta + 16;  // pair sums [2][2][2][64], then each wave's U [8][UB]
  static constexpr int tmp_n = NW * 8 * UB > 512 ? NW * 8 * UB : 512;
  static constexpr size_t BYTES = sizeof(float) * (size_t)(tmp + tmp_n);
};

template <class T, int DT, int NTHR>
__global__ __launch_bounds__(NTHR, 2) void delta_chunk_kernel(DeltaArgs a) {
  using L = ChunkLds<DT, NTHR>;
  constexpr int NVV = NTHR / 256;  // 8-column vectors of v per lane of a token's 16
  extern __shared__ __attribute__((aligned(16))) float sm[];
  const int seg = blockIdx.x, h = blockIdx.y;
  const int slot = a.seg_state[seg];
  const int n = a.seg_len[seg], row0 = a.seg_row[seg], pos0 = a.seg_pos[seg];
  const int tid = threadIdx.x;
  T* out = (T*)a.out;
  const int ldo = a.H * a.vdim;
  if (slot < 0) {  // padding row of a decode bucket
    for (int i = tid; i < n * a.vdim; i += NTHR)
      out[(int64_t)(row0 + i / a.vdim) * ldo + h * a.vdim + i % a.vdim] = from_f32<T>(0.f);
    return;
  }
  const int w = wave_id_uniform(), lane = tid & 63, col = lane & 15, g = lane >> 4;
  const int grp = a.H / a.Hk, hk = h / grp;
  const int cq = hk * a.dim, ck = (a.Hk + hk) * a.dim, cv = 2 * a.Hk * a.dim + h * a.vdim;
  const float decay_scale = -a.a_exp[h] * kLog2e, qscale = rsqrtf((float)a.dim);
  float* S = a.state + ((int64_t)slot * a.H + h) * a.dim * a.vdim;
  const bool owner = 32 * w < a.vdim;  // this wave has columns

  f32x4 st[DT][2];
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int ct = 0; ct < 2; ++ct)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = 16 * t + 4 * g + r, x = 32 * w + 16 * ct + col;
        st[t][ct][r] = pos0 > 0 && d < a.dim && x < a.vdim ? S[(int64_t)d * a.vdim + x] : 0.f;
      }

  // staging: 16 lanes per token, 8 elements each
  const int tok = tid >> 4, e8 = (tid & 15) * 8;
  const bool stager = tok < 16;
  float dtb[8], nw[NVV][8];
#pragma unroll
  for (int j = 0; j < 8; ++j) dtb[j] = e8 + j < a.dim ? a.dt_bias[h * a.dim + e8 + j] : 0.f;
#pragma unroll
  for (int i = 0; i < NVV; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int x = 128 * i + e8 + j;
      nw[i][j] = x < a.vdim ? a.norm_w[x] : 0.f;
    }
  struct alignas(16) Vec { T x[8]; };
  Vec pq, pk, pd, pv[NVV], pg[NVV], ng[NVV];
  T pb = from_f32<T>(0.f);
  auto get = [](float (&d)[8], const Vec& s) {
#pragma unroll
    for (int j = 0; j < 8; ++j) d[j] = to_f32(s.x[j]);
  };
  auto prefetch = [&](int t0) {
    if (!stager || t0 + tok >= n) return;
    const int64_t row = row0 + t0 + tok;
    const T* cr = (const T*)a.conv + row * a.C;
    if (e8 < a.dim) {
      pq = *(const Vec*)(cr + cq + e8);
      pk = *(const Vec*)(cr + ck + e8);
      pd = *(const Vec*)((const T*)a.decay + row * a.ld_decay + h * a.dim + e8);
    }
#pragma unroll
    for (int i = 0; i < NVV; ++i)
      if (128 * i + e8 < a.vdim) {
        pv[i] = *(const Vec*)(cr + cv + 128 * i + e8);
        ng[i] = *(const Vec*)((const T*)a.gate + row * a.ld_gate + h * a.vdim + 128 * i + e8);
      }
    pb = ((const T*)a.proj)[row * a.ldp + a.off_b + h];
  };
  prefetch(0);

  for (int t0 = 0; t0 < n; t0 += 16) {
    const bool live = stager && t0 + tok < n;
    if (stager) {
      float q[8], k[8], l[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) q[j] = k[j] = l[j] = 0.f;
      if (live && e8 < a.dim) {
        get(q, pq);
        get(k, pk);
        get(l, pd);
#pragma unroll
        for (int j = 0; j < 8; ++j) l[j] = decay_scale * softplus_hw(l[j] + dtb[j]);
      }
      float sq = 0.f, sk = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        sq += q[j] * q[j];
        sk += k[j] * k[j];
      }
      const float rq = qscale / sqrtf(sum16(sq) + 1e-6f), rk = 1.f / sqrtf(sum16(sk) + 1e-6f);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        q[j] *= rq;
        k[j] *= rk;
      }
      if (e8 < L::DP) {
        store8(sm + L::q + tok * L::DS + e8, q);
        store8(sm + L::k + tok * L::DS + e8, k);
        store8(sm + L::c + tok * L::DS + e8, l);
      }
#pragma unroll
      for (int i = 0; i < NVV; ++i)
        if (128 * i + e8 < L::VS - 4) {
          float v[8];
#pragma unroll
          for (int j = 0; j < 8; ++j) v[j] = 0.f;
          if (live && 128 * i + e8 < a.vdim) get(v, pv[i]);
          store8(sm + L::v + tok * L::VS + 128 * i + e8, v);
          pg[i] = ng[i];
        }
      if ((tid & 15) == 0) sm[L::beta + tok] = live ? sigmoid_hw(to_f32(pb)) : 0.f;
    }
    prefetch(t0 + 16);
    __syncthreads();
    // running decays of the two chunks; keys decayed to the chunk's end
    if (tid < 2 * L::DP) {
      const int ch = tid / L::DP, d = tid % L::DP;
      float* c = sm + L::c + 8 * ch * L::DS + d;
      float run[8], acc = 0.f;
#pragma unroll
      for (int t = 0; t < 8; ++t) run[t] = acc += c[t * L::DS];
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        c[t * L::DS] = run[t];
        sm[L::kd + (8 * ch + t) * L::KD + d] =
            sm[L::k + (8 * ch + t) * L::DS + d] * fast_exp2(acc - run[t]);
      }
      sm[L::gt + ch * L::DP + d] = fast_exp2(acc);
    }
    __syncthreads();
    // A and B: one (i, j) pair per lane, two halves of the channels
    if (tid < 256) {
      const int ch = tid >> 7, half = (tid >> 6) & 1, i = (tid >> 3) & 7, j = tid & 7;
      const float* ki = sm + L::k + (8 * ch + i) * L::DS + half * (L::DP / 2);
      const float* kj = sm + L::k + (8 * ch + j) * L::DS + half * (L::DP / 2);
      const float* qi = ki + (L::q - L::k);
      const float* ci = ki + (L::c - L::k);
      const float* cj = kj + (L::c - L::k);
      float A = 0.f, B = 0.f;
#pragma unroll 2
      for (int d = 0; d < L::DP / 2; d += 4) {
        const f32x4 k4 = *(const f32x4*)(ki + d), q4 = *(const f32x4*)(qi + d);
        const f32x4 x4 = *(const f32x4*)(kj + d);
        const f32x4 c4 = *(const f32x4*)(ci + d), z4 = *(const f32x4*)(cj + d);
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          const float y = x4[m] * fast_exp2(fminf(c4[m] - z4[m], 0.f));
          A += k4[m] * y;
          B += q4[m] * y;
        }
      }
      float* pr = sm + L::tmp + ch * 256 + half * 64 + i * 8 + j;
      pr[0] = A;
      pr[128] = B;
    }
    __syncthreads();
    if (w < 2) {  // [M_U; M_O] of chunk w, column lane & 7
      const float* pr = sm + L::tmp + w * 256;
      const float* be = sm + L::beta + 8 * w;
      const int c = lane & 7;
      float m[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        float x = 0.f;
#pragma unroll
        for (int j = 0; j < i; ++j) x += (pr[i * 8 + j] + pr[64 + i * 8 + j]) * m[j];
        m[i] = (i == c ? be[c] : 0.f) - be[i] * x;
      }
      if (lane < 8) {
        float* mm = sm + L::mm + w * 128 + c;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          float x = 0.f;
#pragma unroll
          for (int j = 0; j <= i; ++j) x += (pr[128 + i * 8 + j] + pr[192 + i * 8 + j]) * m[j];
          mm[i * 8] = m[i];
          mm[(8 + i) * 8] = x;
        }
      }
    }
    // decay keys and queries from the chunk's start
    if (stager && e8 < L::DP) {
      float* k = sm + L::k + tok * L::DS + e8;
      float c[8], x[8];
      load8(c, sm + L::c + tok * L::DS + e8);
#pragma unroll
      for (int j = 0; j < 8; ++j) c[j] = fast_exp2(c[j]);
      load8(x, k);
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] *= c[j];
      store8(k, x);
      load8(x, k + (L::q - L::k));
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] *= c[j];
      store8(k + (L::q - L::k), x);
    }
    __syncthreads();
    if (owner) {
#pragma unroll
      for (int ch = 0; ch < 2; ++ch) {
        if (t0 + 8 * ch >= n) break;
        const float* row = sm + (col < 8 ? L::k + (8 * ch + col) * L::DS
                                         : L::q + (8 * ch + col - 8) * L::DS) + 4 * g;
        f32x4 acc[2];
        acc[0] = acc[1] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < DT; ++t) {
          const f32x4 x = *(const f32x4*)(row + 16 * t);
#pragma unroll
          for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int ct = 0; ct < 2; ++ct) acc[ct] = mfma_f32(x[r], st[t][ct][r], acc[ct]);
        }
        // lane groups 0, 1: R of tokens 4 g + r; groups 2, 3: the queries' part of O
        float* vo = sm + L::v + (8 * ch + 4 * (g & 1)) * L::VS + 32 * w + col;
        f32x4 m4 = {0.f, 0.f, 0.f, 0.f};
        if (g < 2) m4 = *(const f32x4*)(sm + L::mm + ch * 128 + col * 8 + 4 * g);
        float* ub = sm + L::tmp + w * 8 * L::UB;
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) {
          f32x4 res;
#pragma unroll
          for (int r = 0; r < 4; ++r)
            res[r] = g < 2 ? vo[r * L::VS + 16 * ct] - acc[ct][r] : 0.f;
          f32x4 y = acc[ct];
          if (g < 2) y = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int r = 0; r < 4; ++r) y = mfma_f32(m4[r], res[r], y);
          if (g < 2) {
#pragma unroll
            for (int r = 0; r < 4; ++r) ub[(4 * g + r) * L::UB + 16 * ct + col] = y[r];
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) vo[r * L::VS + 16 * ct] = y[r];
          }
        }
        float u[2][2];
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
          for (int ct = 0; ct < 2; ++ct) u[s][ct] = ub[(4 * s + g) * L::UB + 16 * ct + col];
        const float* gt = sm + L::gt + ch * L::DP + 4 * g;
        const float* kd = sm + L::kd + (8 * ch + g) * L::KD + col;
#pragma unroll
        for (int t = 0; t < DT; ++t) {
          const f32x4 g4 = *(const f32x4*)(gt + 16 * t);
          const float k0 = kd[16 * t], k1 = kd[4 * L::KD + 16 * t];
#pragma unroll
          for (int ct = 0; ct < 2; ++ct) {
            f32x4 x = st[t][ct] * g4;
            x = mfma_f32(k0, u[0][ct], x);
            st[t][ct] = mfma_f32(k1, u[1][ct], x);
          }
        }
      }
    }
    __syncthreads();
    if (stager) {
      float o[NVV][8], so = 0.f;
#pragma unroll
      for (int i = 0; i < NVV; ++i)
        if (128 * i + e8 < a.vdim) {
          load8(o[i], sm + L::v + tok * L::VS + 128 * i + e8);
#pragma unroll
          for (int j = 0; j < 8; ++j) so += o[i][j] * o[i][j];
        }
      const float r = 1.f / sqrtf(sum16(so) / (float)a.vdim + a.eps);
      if (live) {
#pragma unroll
        for (int i = 0; i < NVV; ++i)
          if (128 * i + e8 < a.vdim) {
            float gg[8];
            get(gg, pg[i]);
#pragma unroll
            for (int j = 0; j < 8; ++j) o[i][j] *= r * nw[i][j] * sigmoid_hw(gg[j]);
            store8(out + (int64_t)(row0 + t0 + tok) * ldo + h * a.vdim + 128 * i + e8, o[i]);
          }
      }
      // the next staging overwrites o only with this lane's own v
    }
  }
  if (owner) {
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int ct = 0; ct < 2; ++ct)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int d = 16 * t + 4 * g + r, x = 32 * w + 16 * ct + col;
          if (d < a.dim && x < a.vdim) S[(int64_t)d * a.vdim + x] = st[t][ct][r];
        }
  }
  keep_ring<T>(a, slot, h, n, row0, pos0);
}

// The same in three launches, for a few long portions: what a chunk needs besides the state does not
// wait for it.  Chunks of 16 tokens:
//   delta_prep   a workgroup per (chunk, head): unit keys and queries, decays, A, B, [M_U; M_O] -
//                written as MFMA operands, 16 bytes per lane (ChainEntry)
//   delta_chain  a workgroup per (portion, head, 16 CT value columns): its waves divide the key
//                channels of S, kept as accumulator tiles; the partial products meet in LDS, wave ct
//                forms R, U and O of column tile ct (CT = 1: delta_chain_narrow).  R and U of 16
//                tokens are one tile each, whose layout is also a B operand
//   delta_read   output norm and gate, rings
// The chain is bound by the fp32 MFMA (32 cycles each, 64 + 32 of them per chunk and column tile, over
// NW waves) and by two exchanges through LDS.  Only the keys' products are ahead of the first: the queries' run while
// the parts come back.  The operands of two chunks are under way at any time, which the compiler's waits count only
// since nothing older than they is pending in the loop (S is waited for ahead of it, pointers are uniform): before, every
// second chunk waited for all loads, 1.6 us per 16 tokens, now 1.4 at CT = 2 (0.8 in delta_chain_narrow), 10.3 in
// delta_chunk, whose five barriers also wait for the staging.  Heads of 128, 4 x 3,500 tokens, 16 heads: 605 us (prep 173,
// chain 365, read 64), delta_chunk 2,244; one portion of 4,000: 290 (chain 205) against 2,492.  With portions and heads enough
// for every CU delta_chunk keeps the fp32 units as busy without
// operands in memory (64 x 250, 32 heads: 959 against 1,249).
// Chunks are numbered through the portions in their order: at most rows / 16 + nseg of them.
template <int DT>
struct ChainEntry {  // floats of a (chunk, head)
  static constexpr int ek = 0, eq = 256 * DT, kd = 512 * DT;  // [DT][64 lanes][4]
  static constexpr int gt = 768 * DT;                         // [16 DT] decay over the chunk
  static constexpr int mu = gt + 16 * DT, mo = mu + 256;      // [64 lanes][4]
  static constexpr int N = mo + 256;
};
struct ChunkAt {
  int seg, slot, n, row0, pos0, t0;  // portion, its state, tokens, first row and position; first token
};

// The portion of chunk blockIdx.x, by a scan of the portions' chunk counts in every wave (no
// barrier, no LDS); false: none.
DRTC_DEVICE bool find_chunk(const DeltaArgs& a, ChunkAt& at) {
  const int e = blockIdx.x, lane = threadIdx.x & 63;
  int base = 0;  // chunks of the portions ahead of s0
  for (int s0 = 0; s0 < a.nseg; s0 += 64) {
    const int s = s0 + lane, c = s < a.nseg ? (a.seg_len[s] + 15) / 16 : 0;
    int x = c;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(x, o, 64);
      x += lane >= o ? y : 0;
    }
    const int first = base + x - c;
    const uint64_t hit = __ballot(e >= first && e < first + c);
    if (hit) {
      const int l = __builtin_ctzll(hit), f = __builtin_amdgcn_readlane(first, l), i = s0 + l;
      at = {i, a.seg_state[i], a.seg_len[i], a.seg_row[i], a.seg_pos[i], 16 * (e - f)};
      return true;
    }
    base += __builtin_amdgcn_readlane(x, 63);
  }
  return false;
}

template <class T, int DT>
__global__ __launch_bounds__(256, 5) void delta_prep_kernel(DeltaArgs a, int h0) {
  using E = ChainEntry<DT>;
  constexpr int DP = 16 * DT, DS = DP + 4;
  __shared__ __attribute__((aligned(16))) float ks[16 * DS], qs[16 * DS], cs[16 * DS];
  __shared__ float am[16][17], bm[16][17], mu[16][17], mo[16][17], be[16];
  ChunkAt at;
  if (!find_chunk(a, at) || at.slot < 0) return;
  const int tid = threadIdx.x, h = h0 + blockIdx.y;
  float* w = a.ws + ((int64_t)blockIdx.x * gridDim.y + blockIdx.y) * E::N;
  const int hk = h / (a.H / a.Hk), cq = hk * a.dim, ck = (a.Hk + hk) * a.dim;
  {
    const int tok = tid >> 4, e8 = (tid & 15) * 8;
    const bool live = at.t0 + tok < at.n && e8 < a.dim;
    float q[8], k[8], l[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) q[j] = k[j] = l[j] = 0.f;
    const int64_t row = at.row0 + at.t0 + tok;
    if (live) {
      const float decay_scale = -a.a_exp[h] * kLog2e;
      load8(q, (const T*)a.conv + row * a.C + cq + e8);
      load8(k, (const T*)a.conv + row * a.C + ck + e8);
      load8(l, (const T*)a.decay + row * a.ld_decay + h * a.dim + e8);
#pragma unroll
      for (int j = 0; j < 8; ++j) l[j] = decay_scale * softplus_hw(l[j] + a.dt_bias[h * a.dim + e8 + j]);
    }
    float sq = 0.f, sk = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      sq += q[j] * q[j];
      sk += k[j] * k[j];
    }
    const float rq = rsqrtf((float)a.dim) / sqrtf(sum16(sq) + 1e-6f), rk = 1.f / sqrtf(sum16(sk) + 1e-6f);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      q[j] *= rq;
      k[j] *= rk;
    }
    if (e8 < DP) {
      store8(qs + tok * DS + e8, q);
      store8(ks + tok * DS + e8, k);
      store8(cs + tok * DS + e8, l);
    }
    if ((tid & 15) == 0)
      be[tok] = at.t0 + tok < at.n ? sigmoid_hw(to_f32(((const T*)a.proj)[row * a.ldp + a.off_b + h])) : 0.f;
  }
  __syncthreads();
  if (tid < DP) {  // running decays; keys decayed to the chunk's end
    float run[16], acc = 0.f;
#pragma unroll
    for (int t = 0; t < 16; ++t) run[t] = acc += cs[t * DS + tid];
    w[E::gt + tid] = fast_exp2(acc);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      f32x4 x;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        cs[(4 * g + r) * DS + tid] = run[4 * g + r];
        x[r] = ks[(4 * g + r) * DS + tid] * fast_exp2(acc - run[4 * g + r]);
      }
      *(f32x4*)(w + E::kd + ((tid >> 4) * 64 + 16 * g + (tid & 15)) * 4) = x;
    }
  }
  __syncthreads();
  // A and B: 32 lanes to a block of 4 x 4 pairs, a lane four channels.  Of two blocks apart the decay is cut at the later one's
  // first token, 2^{c_i - c_r} 2^{c_r - c_j}: 8 exponentials for 16 pairs, none of them above 1.  Waves 0 .. 2 take these, wave 3
  // the four blocks of neighbours.  (16 lanes to a block and an exponential a pair, on two waves and a half, left the last
  // SIMD idle.  Heads of 128, 16 heads, 4 x 3,500 tokens 194 -> 173 us, 2.2 TB/s of operands written, 4,000 61 -> 52, 868 x 2 33 -> 29;
  // two or four heads to a workgroup, each head's rows asked for ahead of the one before, are no faster: 174, 177.)
  {
    const int wv = tid >> 6, half = (tid >> 5) & 1, d = 4 * (tid & 31), l16 = tid & 15;
    auto at4 = [&](const float* m, int t) { return d < DP ? *(const f32x4*)(m + t * DS + d) : (f32x4){0.f, 0.f, 0.f, 0.f}; };
    auto exp4 = [](f32x4 x) {
#pragma unroll
      for (int m = 0; m < 4; ++m) x[m] = fast_exp2(x[m]);
      return x;
    };
    auto dot4 = [](f32x4 x, f32x4 y) { return x[0] * y[0] + x[1] * y[1] + x[2] * y[2] + x[3] * y[3]; };
    // lanes of 16: sums of A, the next 16 lanes of B; then a pair to a lane
    auto put = [&](const float (&A)[16], const float (&B)[16], int bi, int bj) {
      float x = 0.f;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(A[e]), __float_as_uint(B[e]), false, false);
        const float v = sum_lanes<16>(__uint_as_float(r[0]) + __uint_as_float(r[1]));
        x = l16 == e ? v : x;
      }
      (tid & 16 ? bm : am)[4 * bi + (l16 >> 2)][4 * bj + (l16 & 3)] = x;
    };
    float A[16], B[16];
    if (wv < 3) {
      const int blk = 2 * wv + half, bi = blk < 1 ? 1 : blk < 3 ? 2 : 3, bj = blk - (blk < 1 ? 0 : blk < 3 ? 1 : 3);
      const f32x4 cr = at4(cs, 4 * bi);
      f32x4 y[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) y[j] = at4(ks, 4 * bj + j) * exp4(cr - at4(cs, 4 * bj + j));
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        f32x4 k4 = at4(ks, 4 * bi + i), q4 = at4(qs, 4 * bi + i);
        if (i > 0) {
          const f32x4 e = exp4(at4(cs, 4 * bi + i) - cr);
          k4 *= e;
          q4 *= e;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          A[4 * i + j] = dot4(k4, y[j]);
          B[4 * i + j] = dot4(q4, y[j]);
        }
      }
      put(A, B, bi, bj);
    } else {
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        const int bi = 2 * n + half;
        f32x4 x[4], z[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          x[j] = at4(ks, 4 * bi + j);
          z[j] = at4(cs, 4 * bi + j);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const f32x4 q4 = at4(qs, 4 * bi + i);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const f32x4 y = j < i ? x[j] * exp4(z[i] - z[j]) : x[j];
            A[4 * i + j] = j < i ? dot4(x[i], y) : 0.f;
            B[4 * i + j] = j <= i ? dot4(q4, y) : 0.f;
          }
        }
        put(A, B, bi, bi);
      }
    }
  }
  __syncthreads();
  if (tid < 64) {  // column tid & 15 of M_U by forward substitution; four rows of it of M_O = B M_U
    const int c = tid & 15, g = tid >> 4;
    float m[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float x = 0.f;
#pragma unroll
      for (int j = 0; j < i; ++j) x += am[i][j] * m[j];
      m[i] = (i == c ? be[i] : 0.f) - be[i] * x;
      if (g == 0) mu[i][c] = m[i];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float x = 0.f;
#pragma unroll
      for (int j = 0; j < 16; ++j) x += j <= 4 * g + i ? bm[4 * g + i][j] * m[j] : 0.f;
      mo[4 * g + i][c] = x;
    }
  }
  // keys and queries decayed from the chunk's start, in lane order
#pragma unroll
  for (int i = 0; i < DT / 4 + (DT < 4); ++i) {
    const int v = 256 * i + tid, d = 16 * (v >> 6) + 4 * ((v >> 4) & 3), t = v & 15;
    if (DT >= 4 || v < 64 * DT) {
      const f32x4 c4 = *(const f32x4*)(cs + t * DS + d);
      f32x4 k4 = *(const f32x4*)(ks + t * DS + d), q4 = *(const f32x4*)(qs + t * DS + d);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float e = fast_exp2(c4[r]);
        k4[r] *= -e;  // R = V - (E*K)^T S is a sum
        q4[r] *= e;
      }
      *(f32x4*)(w + E::ek + v * 4) = k4;
      *(f32x4*)(w + E::eq + v * 4) = q4;
    }
  }
  __syncthreads();
  if (tid < 64) {
    f32x4 x, y;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      x[r] = mu[tid & 15][4 * (tid >> 4) + r];
      y[r] = mo[tid & 15][4 * (tid >> 4) + r];
    }
    *(f32x4*)(w + E::mu + tid * 4) = x;
    *(f32x4*)(w + E::mo + tid * 4) = y;
  }
}

// Waves of a workgroup divide the key channels; all of them hold the same CT column tiles of S.
constexpr int chain_waves(int dt) { return dt < 4 ? dt : 4; }
template <class T, int DT, int CT>
__global__ __launch_bounds__(64 * chain_waves(DT), 2) void delta_chain_kernel(DeltaArgs a, int h0, int nh) {
  using E = ChainEntry<DT>;
  constexpr int NW = chain_waves(DT), TW = DT / NW;
  static_assert(CT > 1 && CT <= NW, "a wave to a column tile");
  __shared__ __attribute__((aligned(16))) float part[NW * 2 * CT * 256], us[CT * 256];
  const int seg = blockIdx.x / nh, hh = blockIdx.x % nh, h = h0 + hh;
  // uniform, and in scalar registers: the loads of a chunk advance a scalar pointer past fixed lane offsets
  auto uniform = [](int x) { return __builtin_amdgcn_readfirstlane(x); };
  const int slot = uniform(a.seg_state[seg]);
  if (slot < 0) return;
  const int n = uniform(a.seg_len[seg]), row0 = uniform(a.seg_row[seg]), pos0 = uniform(a.seg_pos[seg]);
  const int nch = (n + 15) / 16;
  const int w = wave_id_uniform(), lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4;
  const int x0 = 16 * CT * blockIdx.y;
  int entry = 0;
  for (int s = lane; s < seg; s += 64) entry += (a.seg_len[s] + 15) / 16;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) entry += __shfl_xor(entry, o, 64);
  float* S = a.state + ((int64_t)slot * a.H + h) * a.dim * a.vdim;
  auto state = [&](auto&& f) {
#pragma unroll
    for (int t = 0; t < TW; ++t)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int d = 16 * (TW * w + t) + 4 * g + r, x = x0 + 16 * ct + col;
          f(t, ct, r, d < a.dim && x < a.vdim, S + (int64_t)d * a.vdim + x);
        }
  };
  f32x4 st[TW][CT];
  state([&](int t, int ct, int r, bool in, float* at) { st[t][ct][r] = pos0 > 0 && in ? *at : 0.f; });
  // S is there before the loop: else its first use in there waits for all loads, those of the chunks ahead too
#pragma unroll
  for (int t = 0; t < TW; ++t)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) asm volatile("" : "+v"(st[t][ct]));
  entry = uniform(entry);
  const float* p = a.ws + ((int64_t)entry * nh + hh) * E::N;
  const bool lead = w < CT;  // wave ct forms R, U and O of column tile ct
  const int xo = x0 + 16 * min(w, CT - 1) + col;
  const T* v = (const T*)a.conv + (int64_t)row0 * a.C + 2 * a.Hk * a.dim + h * a.vdim;
  unsigned vrow[4], vlast[4];  // of a lane's rows of a chunk; of the last one, where rows behind the end are the last row
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    vrow[r] = (4 * g + r) * a.C + min(xo, a.vdim - 1);
    vlast[r] = min(4 * g + r, (n - 1) & 15) * a.C + min(xo, a.vdim - 1);
  }
  const int64_t ldo = (int64_t)a.H * a.vdim16;
  float* o = a.ws_o + (int64_t)entry * 16 * ldo + h * a.vdim16;
  const unsigned orow = 4 * g * (unsigned)ldo + xo;
  const bool mine = lead && xo < a.vdim16;
  // operands of two chunks: each part is loaded again, two chunks ahead, where it has been read
  // (one chunk is shorter than a load from HBM takes)
  struct Ops {
    f32x4 ek[TW], eq[TW], kd[TW], gt[TW], mu, mo;
    T v[4];
  };
  auto load_k = [&](Ops& x, const float* p) {
#pragma unroll
    for (int t = 0; t < TW; ++t) {
      x.ek[t] = *(const f32x4*)(p + E::ek + 256 * (TW * w + t) + 4u * lane);
      x.eq[t] = *(const f32x4*)(p + E::eq + 256 * (TW * w + t) + 4u * lane);
    }
  };
  auto load_u = [&](Ops& x, const float* p) {
#pragma unroll
    for (int t = 0; t < TW; ++t) {
      x.kd[t] = *(const f32x4*)(p + E::kd + 256 * (TW * w + t) + 4u * lane);
      x.gt[t] = *(const f32x4*)(p + E::gt + 16 * (TW * w + t) + 4u * g);
    }
  };
  auto load_m = [&](Ops& x, const float* p, int c) {
    x.mu = *(const f32x4*)(p + E::mu + 4u * lane);
    x.mo = *(const f32x4*)(p + E::mo + 4u * lane);
    const bool last = c >= nch - 1;
    const T* at = v + (int64_t)(16 * min(c, nch - 1)) * a.C;
#pragma unroll
    for (int r = 0; r < 4; ++r) x.v[r] = at[last ? vlast[r] : vrow[r]];
  };
  Ops even, odd;
  auto chunk = [&](int c) { return p + (int64_t)min(c, nch - 1) * nh * E::N; };
  if (nch > 0) {
    load_k(even, chunk(0));
    load_m(even, chunk(0), 0);
    load_u(even, chunk(0));
    load_k(odd, chunk(1));
    load_m(odd, chunk(1), 1);
    load_u(odd, chunk(1));
  }
  float* mypart = part + w * 2 * CT * 256 + 4 * lane;
  const float* sums = part + 256 * min(w, CT - 1) + 4 * lane;
  auto compute = [&](int c, Ops& x) {
    const float* ahead = chunk(c + 2);
    f32x4 rk[CT], ok[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) rk[ct] = ok[ct] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < TW; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) rk[ct] = mfma_f32(x.ek[t][r], st[t][ct][r], rk[ct]);
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) *(f32x4*)(mypart + 256 * ct) = rk[ct];
    lds_barrier();
    // the queries' products run while the keys' parts come back from LDS
    f32x4 rs[NW];
    if (lead) {
#pragma unroll
      for (int i = 0; i < NW; ++i) rs[i] = *(const f32x4*)(sums + i * 2 * CT * 256);
    }
#pragma unroll
    for (int t = 0; t < TW; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) ok[ct] = mfma_f32(x.eq[t][r], st[t][ct][r], ok[ct]);
    load_k(x, ahead);
    f32x4 res;
    if (lead) {
#pragma unroll
      for (int i = 1; i < NW; ++i) rs[0] += rs[i];
      f32x4 u = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int r = 0; r < 4; ++r) res[r] = 16 * c + 4 * g + r < n ? to_f32(x.v[r]) + rs[0][r] : 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r) u = mfma_f32(x.mu[r], res[r], u);
      *(f32x4*)(us + 256 * w + 4 * lane) = u;
    }
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) *(f32x4*)(mypart + 256 * (CT + ct)) = ok[ct];
    lds_barrier();
    f32x4 u[CT], ys[NW];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) u[ct] = *(const f32x4*)(us + 256 * ct + 4 * lane);
    if (lead) {
#pragma unroll
      for (int i = 0; i < NW; ++i) ys[i] = *(const f32x4*)(sums + i * 2 * CT * 256 + 256 * CT);
    }
#pragma unroll
    for (int t = 0; t < TW; ++t)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) st[t][ct] *= x.gt[t];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int t = 0; t < TW; ++t)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) st[t][ct] = mfma_f32(x.kd[t][r], u[ct][r], st[t][ct]);
    load_u(x, ahead);
    if (lead) {
      f32x4 y = ys[0];
#pragma unroll
      for (int i = 1; i < NW; ++i) y += ys[i];
#pragma unroll
      for (int r = 0; r < 4; ++r) y = mfma_f32(x.mo[r], res[r], y);
      if (mine)
#pragma unroll
        for (int r = 0; r < 4; ++r) (o + (16 * c + r) * ldo)[orow] = y[r];
    }
    load_m(x, ahead, c + 2);
  };
#pragma unroll 1
  for (int c = 0; c + 1 < nch; c += 2) {
    compute(c, even);
    compute(c + 1, odd);
  }
  if (nch & 1) compute(nch - 1, even);
  state([&](int t, int ct, int r, bool in, float* at) {
    if (in) *at = st[t][ct][r];
  });
}

// The same with one column tile to a workgroup, for few chains: a chunk's serial path sets the time, so every wave forms R
// and U itself (four MFMAs more, an exchange through LDS less), M_O R and the outputs are divided over the waves, a chunk's
// outputs are summed beside the next one's products, and operands come through buffer descriptors that scalar adds move on
// (with addresses in vector registers a chunk was 250 instructions of a wave that is alone on its SIMD, now 130).  One
// workgroup to a CU: 16 chains of 4,000 tokens 253 -> 205 us, the MFMAs half of it, 32 262 -> 245; more to a CU:
// 64 chains of 3,500 392 -> 365, 96 of 2,000 308 -> 277.  Two tiles in one workgroup, which reads the operands once: 315, 202,
// 379, 354; operands four chunks ahead spill.
template <class T, int DT>
__global__ __launch_bounds__(64 * chain_waves(DT), 2) void delta_chain_narrow_kernel(DeltaArgs a, int h0, int nh) {
  using E = ChainEntry<DT>;
  constexpr int NW = chain_waves(DT), TW = DT / NW, RW = 4 / NW;
  static_assert(NW * RW == 4, "the four rows of a lane to the waves");
  // parts of the keys' and of the queries' products by chunk parity: one barrier a chunk
  __shared__ __attribute__((aligned(16))) float part[2][2][NW * 256];
  const int seg = blockIdx.x / nh, hh = blockIdx.x % nh, h = h0 + hh;
  auto uniform = [](int x) { return __builtin_amdgcn_readfirstlane(x); };
  const int slot = uniform(a.seg_state[seg]);
  if (slot < 0) return;
  const int n = uniform(a.seg_len[seg]), row0 = uniform(a.seg_row[seg]), pos0 = uniform(a.seg_pos[seg]);
  const int nch = (n + 15) / 16;
  const int w = wave_id_uniform(), lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4;
  const int x0 = 16 * blockIdx.y;
  int entry = 0;
  for (int s = lane; s < seg; s += 64) entry += (a.seg_len[s] + 15) / 16;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) entry += __shfl_xor(entry, o, 64);
  float* S = a.state + ((int64_t)slot * a.H + h) * a.dim * a.vdim;
  auto state = [&](auto&& f) {
#pragma unroll
    for (int t = 0; t < TW; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = 16 * (TW * w + t) + 4 * g + r, x = x0 + col;
        f(t, r, d < a.dim && x < a.vdim, S + (int64_t)d * a.vdim + x);
      }
  };
  f32x4 st[TW];
  state([&](int t, int r, bool in, float* at) { st[t][r] = pos0 > 0 && in ? *at : 0.f; });
  // S is there before the loop: else its first use in there waits for all loads, those of the chunks ahead too
#pragma unroll
  for (int t = 0; t < TW; ++t) asm volatile("" : "+v"(st[t]));
  entry = uniform(entry);
  const char* ahead = (const char*)(a.ws + ((int64_t)entry * nh + hh) * E::N);  // chunk to load next, or the last one
  const int64_t stride = (int64_t)nh * E::N * 4;
  const unsigned vk = 1024 * TW * w + 16 * lane, vg = 64 * TW * w + 16 * g, vm = 16 * lane;
  // Wave 0 starts the keys' sums with V: rows behind the portion's end, and all rows in the other waves, load as 0
  const T* v = (const T*)a.conv + (int64_t)row0 * a.C + 2 * a.Hk * a.dim + h * a.vdim;
  const unsigned vfull = uniform(w == 0 ? 16 * a.C * (int)sizeof(T) : 0);
  const unsigned vtail = uniform(w == 0 ? (n - 16 * (nch - 1)) * a.C * (int)sizeof(T) : 0);
  unsigned vv[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) vv[r] = ((4 * g + r) * a.C + min(x0 + col, a.vdim - 1)) * (unsigned)sizeof(T);
  auto rsrc = [](const void* at, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)at, (short)0, (int)bytes, 0x00020000);
  };
  auto ld = [](__amdgpu_buffer_rsrc_t b, unsigned off, unsigned soff) {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(b, off, soff, 0));
  };
  // operands of two chunks: each part is loaded again, two chunks ahead, where it has been read
  struct Ops {
    f32x4 ek[TW], eq[TW], kd[TW], gt[TW], mu;
    float mo[RW];
    unsigned v[4];  // a word each: packed in pairs, they would be waited for where they are loaded
  };
  auto load_k = [&](Ops& x) {
    const auto b = rsrc(ahead, E::N * 4);
#pragma unroll
    for (int t = 0; t < TW; ++t) {
      x.ek[t] = ld(b, vk + 1024 * t, 4 * E::ek);
      x.eq[t] = ld(b, vk + 1024 * t, 4 * E::eq);
    }
  };
  auto load_rest = [&](Ops& x, int c) {  // in the order of the chunks
    const auto b = rsrc(ahead, E::N * 4);
    x.mu = ld(b, vm, 4 * E::mu);
#pragma unroll
    for (int j = 0; j < RW; ++j)
      x.mo[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(b, vm + 4 * (RW * w + j), 4 * E::mo, 0));
    const auto bv = rsrc(v, c < nch - 1 ? vfull : c == nch - 1 ? vtail : 0);
    v += 16 * a.C;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if constexpr (sizeof(T) == 2) x.v[r] = __builtin_amdgcn_raw_buffer_load_b16(bv, vv[r], 0, 0);
      else x.v[r] = __builtin_amdgcn_raw_buffer_load_b32(bv, vv[r], 0, 0);
    }
#pragma unroll
    for (int t = 0; t < TW; ++t) {
      x.kd[t] = ld(b, vk + 1024 * t, 4 * E::kd);
      x.gt[t] = ld(b, vg + 64 * t, 4 * E::gt);
    }
    ahead += c + 1 < nch ? stride : 0;
  };
  Ops even, odd;
  if (nch > 0) {
    load_k(even);
    load_rest(even, 0);
    load_k(odd);
    load_rest(odd, 1);
  }
  // Outputs: rows 4 g + RW w + j are this wave's
  const int64_t ldo = (int64_t)a.H * a.vdim16;
  float* o = a.ws_o + (int64_t)(entry - 1) * 16 * ldo + h * a.vdim16;  // of the chunk ahead of the next one
  unsigned orow[RW];
#pragma unroll
  for (int j = 0; j < RW; ++j) orow[j] = 4 * ((4 * g + RW * w + j) * (unsigned)ldo + x0 + col);
  auto read_out = [&](float (&ys)[RW][NW], const int par) {
#pragma unroll
    for (int j = 0; j < RW; ++j)
#pragma unroll
      for (int i = 0; i < NW; ++i) ys[j][i] = part[1][par][i * 256 + 4 * lane + RW * w + j];
  };
  auto write_out = [&](const float (&ys)[RW][NW], bool any) {
    const auto b = rsrc(o, any ? 64 * (unsigned)ldo : 0);
    o += 16 * ldo;
#pragma unroll
    for (int j = 0; j < RW; ++j) {
      float y = ys[j][0];
#pragma unroll
      for (int i = 1; i < NW; ++i) y += ys[j][i];
      // (no scalar offset: it is taken off the descriptor's size, and off a size of 0 it would leave everything in range)
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, y), b, orow[j], 0, 0);
    }
  };
  auto compute = [&](int c, Ops& x, const int par) {
    f32x4 rk, ok, u;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      rk[r] = __builtin_bit_cast(float, sizeof(T) == 2 ? x.v[r] << 16 : x.v[r]);
      ok[r] = u[r] = 0.f;
    }
    // the queries' products fill the waits for the keys' parts and for U
    auto queries = [&](int lo, int hi) {
#pragma unroll
      for (int i = lo; i < hi; ++i) ok = mfma_f32(x.eq[i >> 2][i & 3], st[i >> 2][i & 3], ok);
    };
#pragma unroll
    for (int t = 0; t < TW; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) rk = mfma_f32(x.ek[t][r], st[t][r], rk);
    *(f32x4*)(part[0][par] + w * 256 + 4 * lane) = rk;
    lds_barrier();
    f32x4 rs[NW];
#pragma unroll
    for (int i = 0; i < NW; ++i) rs[i] = *(const f32x4*)(part[0][par] + i * 256 + 4 * lane);
    float ys[RW][NW];
    read_out(ys, 1 - par);  // of the chunk before; of none ahead of the first, whose store is out of range
    __builtin_amdgcn_sched_barrier(0);
    queries(0, 3 * TW);
#pragma unroll
    for (int i = 1; i < NW; ++i) rs[0] += rs[i];
    if (16 * c + 16 > n)
#pragma unroll
      for (int r = 0; r < 4; ++r) rs[0][r] = 16 * c + 4 * g + r < n ? rs[0][r] : 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) u = mfma_f32(x.mu[r], rs[0][r], u);
    queries(3 * TW, 4 * TW);
    load_k(x);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < TW; ++t) st[t] *= x.gt[t];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int t = 0; t < TW; ++t) st[t] = mfma_f32(x.kd[t][r], u[r], st[t]);
#pragma unroll
    for (int j = 0; j < RW; ++j) {  // M_O R: a k-step to each wave
      const f32x4 y = rs[0];
      ok = mfma_f32(x.mo[j], RW == 1 ? w & 2 ? w & 1 ? y[3] : y[2] : w & 1 ? y[1] : y[0] : w ? y[2 + j] : y[j], ok);
    }
    *(f32x4*)(part[1][par] + w * 256 + 4 * lane) = ok;
    load_rest(x, c + 2);
    write_out(ys, c > 0);
  };
#pragma unroll 1
  for (int c = 0; c + 1 < nch; c += 2) {
    compute(c, even, 0);
    compute(c + 1, odd, 1);
  }
  if (nch & 1) compute(nch - 1, even, 0);
  lds_barrier();
  if (nch > 0) {
    float ys[RW][NW];
    read_out(ys, (nch - 1) & 1);
    write_out(ys, true);
  }
  state([&](int t, int r, bool in, float* at) {
    if (in) *at = st[t][r];
  });
}

// Four heads of a chunk, NV times 8 columns per lane.
template <class T, int NV>
__global__ __launch_bounds__(256) void delta_read_kernel(DeltaArgs a) {
  constexpr int NH = 4;
  ChunkAt at;
  if (!find_chunk(a, at)) return;
  const int tok = threadIdx.x >> 4, l16 = threadIdx.x & 15, h0 = NH * blockIdx.y;
  const int64_t row = at.row0 + at.t0 + tok;
  const bool live = at.t0 + tok < at.n;
  if (live && at.slot < 0) {  // padding row of a decode bucket
    T* out = (T*)a.out + (row * a.H + h0) * a.vdim;
    for (int i = l16; i < min(NH, a.H - h0) * a.vdim; i += 16) out[i] = from_f32<T>(0.f);
  } else if (live) {
    const float* o = a.ws_o + (((int64_t)blockIdx.x * 16 + tok) * a.H + h0) * a.vdim16;
    const T* gate = (const T*)a.gate + row * a.ld_gate + h0 * a.vdim;
    T* out = (T*)a.out + (row * a.H + h0) * a.vdim;
    float x[NH][NV][8], z[NH][NV][8];
#pragma unroll
    for (int k = 0; k < NH; ++k)
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int e = 128 * i + 8 * l16;
#pragma unroll
        for (int j = 0; j < 8; ++j) x[k][i][j] = 0.f;
        if (h0 + k < a.H && e < a.vdim) {
          load8(x[k][i], o + k * a.vdim16 + e);
          load8(z[k][i], gate + k * a.vdim + e);
        }
      }
    float w[NV][8];
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) w[i][j] = 128 * i + 8 * l16 < a.vdim ? a.norm_w[128 * i + 8 * l16 + j] : 0.f;
#pragma unroll
    for (int k = 0; k < NH; ++k) {
      float so = 0.f;
#pragma unroll
      for (int i = 0; i < NV; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) so += x[k][i][j] * x[k][i][j];
      const float r = 1.f / sqrtf(sum_lanes<16>(so) / (float)a.vdim + a.eps);
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int e = 128 * i + 8 * l16;
#pragma unroll
        for (int j = 0; j < 8; ++j) x[k][i][j] *= r * w[i][j] * sigmoid_hw(z[k][i][j]);
        if (h0 + k < a.H && e < a.vdim) store8(out + k * a.vdim + e, x[k][i]);
      }
    }
  }
  if (at.slot >= 0 && at.t0 + 16 >= at.n)
    for (int h = h0; h < min(a.H, h0 + NH); ++h) keep_ring<T>(a, at.slot, h, at.n, at.row0, at.pos0);
}

// Bound by the state, read and written once; everything a token needs besides it is asked for ahead of
// it, so that the token is prepared while it arrives (memory answers in order).  EXACT: the state fills
// the lanes' tiles, so no load of it stands behind a condition and the waits can count them.  64 sequences x 32 heads of
// 128 x 128 58.7 -> 53.7 us (5.0 TB/s), 256 x 32 284 -> 223 (4.8).  NT: the states past the caches, which hold a step's
// weights instead; in the pass of 64 x 32 heads 60.5 -> 54 and the kernels around it 2 % (the rule: kStatesPastCaches).
constexpr int kDecodeTaps = 4;  // taps whose inputs are fetched ahead; more are read where they are used
template <class T, int DPL, int CPL, bool EXACT, bool NT = false>
__global__ __launch_bounds__(512) void delta_decode_kernel(DeltaArgs a) {
  constexpr int DP = 8 * DPL;
  extern __shared__ __attribute__((aligned(16))) float sm[];
  __shared__ float red[16];
  const int row = blockIdx.x, h = blockIdx.y;
  const int slot = a.row_state[row];
  const int tid = threadIdx.x, nthr = blockDim.x;
  T* out = (T*)a.out + ((int64_t)row * a.H + h) * a.vdim;
  if (slot < 0) {
    for (int i = tid; i < a.vdim; i += nthr) out[i] = from_f32<T>(0.f);
    return;
  }
  float* ks = sm;
  float* qs = ks + DP;
  float* gs = qs + DP;
  float* vs = gs + DP;
  const int pos = a.positions[row];
  const int lane = tid & 63, p = lane & 7;
  const int col = ((tid >> 6) * 8 + (lane >> 3)) * CPL;
  const int grp = a.H / a.Hk, hk = h / grp;
  const int cq = hk * a.dim, ck = (a.Hk + hk) * a.dim, cv = 2 * a.Hk * a.dim + h * a.vdim;
  float* S = a.state + ((int64_t)slot * a.H + h) * a.dim * a.vdim;
  const T* pr = (const T*)a.proj + (int64_t)row * a.ldp;
  T* ring = (T*)a.ring + (int64_t)slot * a.taps * a.C;
  const bool own = h % grp == 0;
  const int back = min(pos, a.taps - 1);
  struct Taps {
    T x[kDecodeTaps];
    float w[kDecodeTaps];
  };
  auto fetch = [&](Taps& t, int c) {
#pragma unroll
    for (int j = 0; j < kDecodeTaps; ++j) {
      t.x[j] = from_f32<T>(0.f);
      t.w[j] = 0.f;
      if (j <= back) {
        t.x[j] = j ? ring[(int64_t)((pos - j) % a.taps) * a.C + c] : pr[c];
        t.w[j] = a.conv_w[(int64_t)(a.taps - 1 - j) * a.C + c];
      }
    }
  };
  auto conv = [&](const Taps& t, int c, bool keep) {
    float acc = to_f32(t.x[0]) * t.w[0];
#pragma unroll
    for (int j = 1; j < kDecodeTaps; ++j) acc += to_f32(t.x[j]) * t.w[j];
    for (int j = kDecodeTaps; j <= back; ++j)
      acc += to_f32(ring[(int64_t)((pos - j) % a.taps) * a.C + c]) *
             a.conv_w[(int64_t)(a.taps - 1 - j) * a.C + c];
    if (keep) ring[(int64_t)(pos % a.taps) * a.C + c] = t.x[0];
    return to_f32(from_f32<T>(silu_as<T>(acc)));
  };
  // this thread's first channels: q, k, the decay, v; threads past them take the last
  const T* dec = (const T*)a.decay + (int64_t)row * a.ld_decay + h * a.dim;
  const int i0 = min(tid, a.dim - 1), e0 = min(tid, a.vdim - 1);
  Taps tq, tk, tv;
  fetch(tq, cq + i0);
  fetch(tk, ck + i0);
  fetch(tv, cv + e0);
  T d0 = dec[i0];
  const float dt0 = a.dt_bias[h * a.dim + i0];
  __builtin_amdgcn_sched_barrier(0);
  StateTile<DPL, CPL> st;
  if constexpr (EXACT) st.template move_all<false, NT>(S, col, p, a.vdim);
  else if (pos > 0) st.load(S, col, p, a.dim, a.vdim);
  __builtin_amdgcn_sched_barrier(0);
  float sq = 0.f, sk = 0.f, dot = 0.f;
  const float aexp = a.a_exp[h];
  for (int i = tid; i < DP; i += nthr) {
    float q = 0.f, k = 0.f, g = 1.f;
    if (i < a.dim) {
      if (i != tid) {
        fetch(tq, cq + i);
        fetch(tk, ck + i);
        d0 = dec[i];
      }
      q = conv(tq, cq + i, own);
      k = conv(tk, ck + i, own);
      g = expf(-aexp * softplus_f(to_f32(d0) + (i == tid ? dt0 : a.dt_bias[h * a.dim + i])));
    }
    qs[i] = q;
    ks[i] = k;
    gs[i] = g;
    sq += q * q;
    sk += k * k;
    dot += q * k;
  }
  for (int i = tid; i < a.vdim; i += nthr) {
    if (i != tid) fetch(tv, cv + i);
    vs[i] = conv(tv, cv + i, true);
  }
  const float beta = sigmoid_f(to_f32(pr[a.off_b + h]));
  const float rq = rsqrtf((float)a.dim) / sqrtf(block_sum(sq, red) + 1e-6f);
  const float rk = 1.f / sqrtf(block_sum(sk, red) + 1e-6f);
  const float qk = block_sum(dot, red) * rq * rk;
  for (int i = tid; i < DP; i += nthr) {
    qs[i] *= rq;
    ks[i] *= rk;
  }
  __syncthreads();
  if (pos == 0) st.zero();
  float o[CPL], so = 0.f;
#pragma unroll
  for (int c = 0; c < CPL; ++c) o[c] = 0.f;
  if (col < a.vdim) {
    float v[CPL];
#pragma unroll
    for (int c = 0; c < CPL; ++c) v[c] = col + c < a.vdim ? vs[col + c] : 0.f;
    st.token(ks, qs, gs, p, beta, qk, v, o);
    if constexpr (EXACT) st.template move_all<true, NT>(S, col, p, a.vdim);
    else st.store(S, col, p, a.dim, a.vdim);
#pragma unroll
    for (int c = 0; c < CPL; ++c)
      if (col + c < a.vdim && p == 0) so += o[c] * o[c];
  }
  const float r = 1.f / sqrtf(block_sum(so, red) / (float)a.vdim + a.eps);
  const T* gate = (const T*)a.gate + (int64_t)row * a.ld_gate + h * a.vdim;
  if (p == 0) {
#pragma unroll
    for (int c = 0; c < CPL; ++c)
      if (col + c < a.vdim)
        out[col + c] = from_f32<T>(o[c] * r * a.norm_w[col + c] * sigmoid_f(to_f32(gate[col + c])));
  }
}

template <class T, int DPL, int CPL>
static int scan_go(const DeltaArgs& a, hipStream_t st) {
  using S = ScanShape<DPL>;
  const int waves = (a.vdim + 8 * CPL - 1) / (8 * CPL);
  const int dvp = (a.vdim + 3) & ~3;
  const size_t lds = sizeof(float) * (size_t)(S::CT * (3 * S::DP + 2 * dvp) + 2 * S::CT);
  if (waves > 8 || lds > 65536) return -1;
  delta_scan_kernel<T, DPL, CPL><<<dim3(a.nseg, a.H), dim3(64 * waves), lds, st>>>(a);
  return 0;
}
template <class T, int DPL>
static int scan_c(const DeltaArgs& a, int cpl, hipStream_t st) {
  // columns per lane: at most 8 waves to a workgroup
  if (a.vdim > 256) return scan_go<T, DPL, 8>(a, st);
  if (cpl >= 4 || a.vdim > 128) return scan_go<T, DPL, 4>(a, st);
  return scan_go<T, DPL, 2>(a, st);
}
template <class T>
static int scan_t(const DeltaArgs& a, int cpl, hipStream_t st) {
  const bool big = a.vdim > 256;  // fewer staged tokens
  if (a.dim > 256 || a.vdim > 512) return -1;
  if (a.dim > 128 || big) return scan_c<T, 32>(a, cpl, st);
  if (a.dim > 64) return scan_c<T, 16>(a, cpl, st);
  if (a.dim > 32) return scan_c<T, 8>(a, cpl, st);
  return scan_c<T, 4>(a, cpl, st);
}

template <class T, int DT>
static int chunk_go(const DeltaArgs& a, hipStream_t st) {
  const dim3 grid(a.nseg, a.H);
  if (a.vdim <= 128)
    delta_chunk_kernel<T, DT, 256><<<grid, dim3(256), ChunkLds<DT, 256>::BYTES, st>>>(a);
  else
    delta_chunk_kernel<T, DT, 512><<<grid, dim3(512), ChunkLds<DT, 512>::BYTES, st>>>(a);
  static_assert(ChunkLds<DT, 512>::BYTES <= 65536, "LDS without an attribute");
  return 0;
}
template <class T>
static int chunk_t(const DeltaArgs& a, hipStream_t st) {
  if (a.dim <= 32) return chunk_go<T, 2>(a, st);
  if (a.dim <= 64) return chunk_go<T, 4>(a, st);
  return chunk_go<T, 8>(a, st);
}

template <class T, int DT>
static int chain_go(const DeltaArgs& a, hipStream_t st) {
  const int64_t entries = a.rows / 16 + a.nseg;
  const int nh = (int)std::min<int64_t>(a.H, a.ws_floats / (entries * ChainEntry<DT>::N));
  if (nh < 1) return -1;
  for (int h0 = 0; h0 < a.H; h0 += nh) {
    const int m = std::min(nh, a.H - h0);
    delta_prep_kernel<T, DT><<<dim3(entries, m), dim3(256), 0, st>>>(a, h0);
    constexpr int NW = chain_waves(DT);
    auto go = [&](auto kernel, int columns) {
      kernel<<<dim3(a.nseg * m, (a.vdim16 + columns - 1) / columns), dim3(64 * NW), 0, st>>>(a, h0, m);
    };
    // The fewest columns to a workgroup wait least between its products and overlap with a CU's other ones; more
    // read the operands less often.  Heads of 128, us with 16 / 32 columns: 16 chains of 4,000 tokens 205 / 371, 32 of 868
    // 50 / 86, 64 of 3,500 365 / 390, 96 of 2,000 277 / 358; with 16 / 64 columns 144 of 1,000 234 / 213.
    const int64_t chains = (int64_t)a.nseg * m;
    if (chains * ((a.vdim16 + 15) / 16) <= 768) go(delta_chain_narrow_kernel<T, DT>, 16);
    else if (NW == 4 && chains * ((a.vdim16 + 63) / 64) >= 512) go(delta_chain_kernel<T, DT, NW>, 16 * NW);
    else go(delta_chain_kernel<T, DT, 2>, 32);
  }
  if (a.vdim <= 128) delta_read_kernel<T, 1><<<dim3(entries, (a.H + 3) / 4), dim3(256), 0, st>>>(a);
  else delta_read_kernel<T, 2><<<dim3(entries, (a.H + 3) / 4), dim3(256), 0, st>>>(a);
  return 0;
}
template <class T>
static int chain_t(const DeltaArgs& a, hipStream_t st) {
  if (a.dim <= 32) return chain_go<T, 2>(a, st);
  if (a.dim <= 64) return chain_go<T, 4>(a, st);
  return chain_go<T, 8>(a, st);
}

// cpl 0: the chunk form where the sizes allow it
int launch_delta_scan(int f32, const DeltaArgs& a, int cpl, hipStream_t st) {
  if (a.nseg == 0) return 0;
  if (a.Hk < 1 || a.H % a.Hk) return -1;
  if (cpl == 0 && a.ws) {
    if (a.dim % 8 || a.vdim % 8 || a.dim > 128 || a.vdim > 256 || a.ld_decay % 8 || a.ld_gate % 8 ||
        a.vdim16 % 16 || a.vdim16 < a.vdim || !a.ws_o)
      return -1;
    const int rc = f32 ? chain_t<float>(a, st) : chain_t<bf16_t>(a, st);
    return rc ? rc : (int)hipGetLastError();
  }
  if (cpl == 0) {
    if (a.dim % 8 == 0 && a.vdim % 8 == 0 && a.dim <= 128 && a.vdim <= 256 &&
        a.ld_decay % 8 == 0 && a.ld_gate % 8 == 0) {
      const int rc = f32 ? chunk_t<float>(a, st) : chunk_t<bf16_t>(a, st);
      return rc ? rc : (int)hipGetLastError();
    }
    cpl = 4;
  }
  const int rc = f32 ? scan_t<float>(a, cpl, st) : scan_t<bf16_t>(a, cpl, st);
  return rc ? rc : (int)hipGetLastError();
}

// Bytes of a step's states from which on they go past the caches.  us a step of four layers, two of them these, through /
// past: 128 MiB (64 sequences, 32 heads, width 4096) 617 / 597, 96 547 / 541, 80 528 / 538, 64 486 / 498; on width 2048, whose
// weights a cache holds, 128 MiB 496 / 462, 64 366 / 335.
constexpr int64_t kStatesPastCaches = 96ll << 20;
template <class T, int DPL, int CPL>
static int decode_go(const DeltaArgs& a, hipStream_t st) {
  const int waves = (a.vdim + 8 * CPL - 1) / (8 * CPL);
  const size_t lds = sizeof(float) * (size_t)(3 * 8 * DPL + a.vdim);
  if (waves > 8) return -1;
  if constexpr (DPL <= 16) {
    if (a.dim == 8 * DPL && a.vdim == 8 * CPL * waves) {
      const bool past = (int64_t)a.rows * a.H * a.dim * a.vdim * 4 >= kStatesPastCaches;
      (past ? delta_decode_kernel<T, DPL, CPL, true, true> : delta_decode_kernel<T, DPL, CPL, true>)
          <<<dim3(a.rows, a.H), dim3(64 * waves), lds, st>>>(a);
      return 0;
    }
  }
  delta_decode_kernel<T, DPL, CPL, false><<<dim3(a.rows, a.H), dim3(64 * waves), lds, st>>>(a);
  return 0;
}
template <class T, int DPL>
static int decode_c(const DeltaArgs& a, hipStream_t st) {
  return a.vdim > 256 ? decode_go<T, DPL, 8>(a, st) : decode_go<T, DPL, 4>(a, st);
}
template <class T>
static int decode_t(const DeltaArgs& a, hipStream_t st) {
  if (a.dim > 256 || a.vdim > 512) return -1;
  if (a.dim > 128) return decode_c<T, 32>(a, st);
  if (a.dim > 64) return decode_c<T, 16>(a, st);
  if (a.dim > 32) return decode_c<T, 8>(a, st);
  return decode_c<T, 4>(a, st);
}

int launch_delta_decode(int f32, const DeltaArgs& a, hipStream_t st) {
  if (a.rows == 0) return 0;
  if (a.Hk < 1 || a.H % a.Hk) return -1;
  const int rc = f32 ? decode_t<float>(a, st) : decode_t<bf16_t>(a, st);
  return rc ? rc : (int)hipGetLastError();
}

}  // namespace drtc
