// Router logits of a row that a workgroup holds, for the norms ahead of mixtures.
#pragma once
#include "common.h"

namespace drtc {

constexpr int kRouterFuse = 32;  // experts at most

// logits[e] = router[e] . x over the E experts, in fp32.  256 threads, thread t holds x[i] = columns (t + 256 i) * 8 ..
// < H.  ``start`` asks for the first rows and comes ahead of whatever makes x; the reads of x's row need not wait.
template <int VPT>
struct RouterDots {
  static constexpr int RE = 8;  // experts at a time
  bf16x8 rw[2][RE][VPT];
  const bf16_t* router;
  int64_t ld;
  int H, E;

  DRTC_DEVICE void load(bf16x8 (&d)[RE][VPT], int e0) {
#pragma unroll
    for (int e = 0; e < RE; ++e)
#pragma unroll
      for (int i = 0; i < VPT; ++i) {
        const int idx = (threadIdx.x + i * 256) * 8;
        if (idx < H) d[e][i] = load_bf16x8(router + min(e0 + e, E - 1) * ld + idx);
      }
  }
  DRTC_DEVICE void start(const bf16_t* r, int64_t ld_, int H_, int E_) {
    router = r;
    ld = ld_;
    H = H_;
    E = E_;
    load(rw[0], 0);
    load(rw[1], RE);
  }
  DRTC_DEVICE void finish(const float (&x)[VPT][8], float* __restrict__ logits) {
    __shared__ float dots[4][kRouterFuse + RE];
    const int tid = threadIdx.x, lane = tid & 63;
    for (int e0 = 0; e0 < E; e0 += 2 * RE) {
#pragma unroll
      for (int z = 0; z < 2; ++z) {
        if (e0 + z * RE >= E) break;
        float p[RE];
#pragma unroll
        for (int e = 0; e < RE; ++e) {
          p[e] = 0.f;
#pragma unroll
          for (int i = 0; i < VPT; ++i)
            if ((tid + i * 256) * 8 < H)
#pragma unroll
              for (int j = 0; j < 8; ++j) p[e] += x[i][j] * bf2f(rw[z][e][i][j]);
        }
        if (e0 + (z + 2) * RE < E) load(rw[z], e0 + (z + 2) * RE);
        // sums over the wave: each step halves the experts of a lane, lanes 8 e .. end with expert e
#pragma unroll
        for (int n = RE / 2, o = 32; n > 0; n >>= 1, o >>= 1)
#pragma unroll
          for (int e = 0; e < n; ++e) {
            const bool hi = lane & o;
            const float keep = hi ? p[e + n] : p[e], give = hi ? p[e] : p[e + n];
            p[e] = keep + __shfl_xor(give, o, 64);
          }
        float s = p[0];
        s += __shfl_xor(s, 4, 64);
        s += __shfl_xor(s, 2, 64);
        s += __shfl_xor(s, 1, 64);
        if ((lane & 7) == 0) dots[tid >> 6][e0 + z * RE + (lane >> 3)] = s;
      }
    }
    __syncthreads();
    if (tid < E) logits[tid] = dots[0][tid] + dots[1][tid] + dots[2][tid] + dots[3][tid];
  }
};

}  // namespace drtc
