// fft_wgrad.hip -- gradient of the spectral weights of y = W . F x over a batch:
//   gw[i] = sum_b Re(conj(g[b][i]) f[b][i]),  f = F x.
//
// HBM bound: g and f are read once (16 bytes a point) and gw written once; as
// separate conjugate, product and sum kernels the same took 48 bytes a point
// (25.7 us for 9 x (32 x 64 x 128), 7.7 us here; 5.4-5.6 TB/s from 2 GB down to
// 0.5).  A thread owns two adjacent points (16-byte loads); the TB threads of
// one pair take every TB-th batch member and meet in LDS, so that a few points
// over a large batch still fill the device.
// Products of FP32 values are exact in FP64 and are summed there: the result
// is rounded once, whatever the batch.
#include <hip/hip_runtime.h>

#include "launch.h"

#include "fft_plane.h"

namespace fftamd {

constexpr int WG_NT = 256;
// The batch is split until the launch has two workgroups per CU: 9 x 2^18
// points (512 workgroups) take 7.7 us unsplit and 8.2 split four ways, 9 x 2^15
// (64) 3.6 and 2.9, 1000 x 2^15 522 and 150, 93 split sixteen ways.
constexpr unsigned long long WG_MIN_BLOCKS = 512;

template <int TB, int V>
__global__ void __launch_bounds__(WG_NT) k_weight_grad(const float* __restrict__ g, const float* __restrict__ f,
                                                       float* __restrict__ gw, unsigned long long points,
                                                       unsigned batch) {
  constexpr int TP = WG_NT / TB;  // threads side by side along the points
  typedef float vf __attribute__((ext_vector_type(2 * V)));
  const int tp = threadIdx.x % TP, tb = threadIdx.x / TP;
  const unsigned long long i = ((unsigned long long)blockIdx.x * TP + tp) * V;
  double acc[V];
#pragma unroll
  for (int v = 0; v < V; ++v) acc[v] = 0.0;
  if (i < points) {
#pragma unroll 4
    for (unsigned b = (unsigned)tb; b < batch; b += TB) {
      const unsigned long long o = 2ull * ((unsigned long long)b * points + i);
      const vf a = *reinterpret_cast<const vf*>(g + o), c = *reinterpret_cast<const vf*>(f + o);
#pragma unroll
      for (int v = 0; v < V; ++v) {
        acc[v] += (double)a[2 * v] * (double)c[2 * v];
        acc[v] += (double)a[2 * v + 1] * (double)c[2 * v + 1];
      }
    }
  }
  if constexpr (TB > 1) {
    __shared__ double s[TB][TP * V];
#pragma unroll
    for (int v = 0; v < V; ++v) s[tb][tp * V + v] = acc[v];
    __syncthreads();
    if (tb == 0) {
#pragma unroll
      for (int v = 0; v < V; ++v)
        for (int t = 1; t < TB; ++t) acc[v] += s[t][tp * V + v];
    }
  }
  if (tb == 0 && i < points) {
#pragma unroll
    for (int v = 0; v < V; ++v) gw[i + v] = (float)acc[v];
  }
}

template <int TB, int V>
static bool launch_wg(const float* g, const float* f, float* gw, unsigned long long points, unsigned batch,
                      hipStream_t s) {
  const unsigned long long per = (unsigned long long)(WG_NT / TB) * V;
  const unsigned long long blocks = (points + per - 1) / per;
  if (blocks > 0xFFFFFFFFull / WG_NT) return false;  // grid size in work-items is 32-bit
  FFTAMD_LAUNCH((k_weight_grad<TB, V>), dim3((unsigned)blocks), dim3(WG_NT), 0, s, g, f, gw, points, batch);
  return true;
}

void preload_wgrad() { preload_kernel(reinterpret_cast<const void*>(&k_weight_grad<1, 2>)); }

int launch_weight_grad(const void* g, const void* f, void* gw, unsigned long long points, unsigned batch,
                       void* stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const float *pg = static_cast<const float*>(g), *pf = static_cast<const float*>(f);
  float* pw = static_cast<float*>(gw);
  bool ok;
  // 16-byte loads need an even number of points (every member then starts on
  // a 16-byte boundary if the first does)
  const bool wide = points % 2 == 0 && (((uintptr_t)g | (uintptr_t)f) & 15) == 0;
  if (!wide) {
    ok = launch_wg<1, 1>(pg, pf, pw, points, batch, s);
  } else {
    const unsigned long long blocks = (points + 2 * WG_NT - 1) / (2 * WG_NT);
    if (blocks >= WG_MIN_BLOCKS || batch < 4) ok = launch_wg<1, 2>(pg, pf, pw, points, batch, s);
    else if (4 * blocks >= WG_MIN_BLOCKS || batch < 16) ok = launch_wg<4, 2>(pg, pf, pw, points, batch, s);
    else if (16 * blocks >= WG_MIN_BLOCKS || batch < 64) ok = launch_wg<16, 2>(pg, pf, pw, points, batch, s);
    else ok = launch_wg<64, 2>(pg, pf, pw, points, batch, s);
  }
  if (!ok) return -1;
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace fftamd
