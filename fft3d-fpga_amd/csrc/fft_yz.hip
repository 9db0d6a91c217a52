// fft_yz.hip -- second pass of NZ x LY R x LX boxes whose planes are too large
// for one workgroup: the y axis is split R x LY between the two passes, as in the
// cubes' pairs (fft_cube.hip).
//
// y = a + R b (a < R, b < LY), ky = k + LY d (k < LY, d < R):
//   X[k + LY d] = sum_a W_R^{a d} W_{R LY}^{a k} T_a[k],  T_a[k] = sum_b x[a + R b] W_LY^{b k}.
//
// The first pass is the plane pass (fft_plane.hip) over the LY x LX planes of
// every R-th row, x and T_a[k], written to row LY a + k, out of place.  Here one
// workgroup takes rows LY a + k, a < R, of 16 adjacent columns in all NZ planes
// (16 R NZ points, R NZ threads, up to 133 KiB of LDS): a thread holds the R rows
// of one column in 16 / R planes, does the R-point DFT over a in registers, and
// the 16 R lines along z go through LDS with the line passes' strided stages.
// In place.
//
// HBM bound: two reads and writes of the array instead of the three of x, y and z
// line passes (what it gains is at yz_split in fft_plane.h; with non-temporal stores
// past the caches 2 x (128 x 512 x 256) 218 -> 200 us).
#include <hip/hip_runtime.h>

#include "launch.h"

#include "fft_pass_dev.h"
#include "fft_plane.h"

namespace fftamd {

constexpr int YZ_C = 16;  // columns: 128-byte row segments

template <int NZ, int R>
struct YzGeom {
  using G = Geom<NZ, MODE_STRIDED, YZ_C * R>;
  static constexpr int NT = NZ * R;
  static_assert(G::NT == NT, "16 points per thread in both phases");
};

template <int NZ, int R, bool INV, bool WS>
__global__ void __launch_bounds__(NZ* R) k_fft_yz(const YzArgs a) {
  using G = typename YzGeom<NZ, R>::G;
  constexpr int CC = YZ_C * R, J = 16 / R, ZT = NZ * R / 16;  // planes per thread, z step
  __shared__ cpx<float> lds[G::LDS_ELEMS];
  // the row k varies fastest over blockIdx, so the tiles in flight together cover
  // whole planes' rows (as in the cubes' second pass)
  const unsigned b = blockIdx.x;
  const unsigned k = b & (a.ly - 1u);
  const unsigned ngroups = a.lx / YZ_C;
  const unsigned xg = (b / a.ly) & (ngroups - 1u);
  const unsigned long long blk = b / a.ly / ngroups;
  const long long plane = (long long)a.ly * R * a.lx;
  const long long base = (long long)blk * NZ * plane + (long long)k * a.lx + YZ_C * xg;
  const cpx<float>* in = reinterpret_cast<const cpx<float>*>(a.in) + base;
  cpx<float>* out = reinterpret_cast<cpx<float>*>(a.out) + base;
  const int tid = threadIdx.x;
  const int x = tid & (YZ_C - 1), zz = tid / YZ_C;
  const long long arow = (long long)a.ly * a.lx;  // between rows LY a + k
  cpx<float> v[16];
#pragma unroll
  for (int j = 0; j < J; ++j)
#pragma unroll
    for (int r = 0; r < R; ++r) v[j * R + r] = in[(zz + ZT * j) * plane + r * arow + x];
  // T_a[k] times W_{R LY}^{a k} (k is uniform over the workgroup)
  const cpx<float>* __restrict__ w512 = reinterpret_cast<const cpx<float>*>(a.w512);
  cpx<float> w[R];
#pragma unroll
  for (int r = 1; r < R; ++r) w[r] = w512[r * k * a.wstep];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    cpx<float>* t = v + j * R;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (INV) t[r] = cswap(t[r]);
      if (r) t[r] = cmul(t[r], w[r]);
    }
    dft<float, R>(t);
#pragma unroll
    for (int d = 0; d < R; ++d) lds[G::idx(YZ_C * d + x, zz + ZT * j)] = t[d];
  }
  __syncthreads();
  // z: thread (line c = 16 d + x, tau)
  const int c = tid % CC, tau = tid / CC;
  stage_load_lds<float, NZ, MODE_STRIDED, 0, CC>(v, lds, c, tau);
  __syncthreads();  // every thread holds its stage-0 inputs before stage 0 stores
  run_stages<float, NZ, MODE_STRIDED, 0, false, CC>(v, lds, c, tau, reinterpret_cast<const cpx<float>*>(a.tw));
  constexpr int NP = G::NP;
  constexpr int RL = sched_radix(NZ, NP - 1), NSL = sched_ns(NZ, NP - 1), NBL = 16 / RL;
  const long long row = (c / YZ_C) * arow + (c & (YZ_C - 1));  // row k + LY d
#pragma unroll
  for (int q = 0; q < NBL; ++q) {
    const int j = tau + q * G::TPL;
#pragma unroll
    for (int r = 0; r < RL; ++r) {
      const long long e = (j + r * NSL) * plane + row;
      cpx<float> s = v[q * RL + r];
      if (INV) s = cswap(s);
      if (WS) s = cscale(s, a.w_store[(unsigned long long)(base + e) & a.w_mask]);
      if (a.stream) __builtin_nontemporal_store(__builtin_bit_cast(long long, s), reinterpret_cast<long long*>(out + e));
      else out[e] = s;
    }
  }
}

template <int NZ, int R>
static bool launch_yz(const YzArgs& a, unsigned blocks, hipStream_t s) {
  if constexpr (!yz_tile_ok(NZ, R)) {
    return false;
  } else {
    const dim3 g(blocks), t(YzGeom<NZ, R>::NT);
    if (a.inverse) {
      if (a.w_store) FFTAMD_LAUNCH((k_fft_yz<NZ, R, true, true>), g, t, 0, s, a);
      else FFTAMD_LAUNCH((k_fft_yz<NZ, R, true, false>), g, t, 0, s, a);
    } else {
      if (a.w_store) FFTAMD_LAUNCH((k_fft_yz<NZ, R, false, true>), g, t, 0, s, a);
      else FFTAMD_LAUNCH((k_fft_yz<NZ, R, false, false>), g, t, 0, s, a);
    }
    return true;
  }
}

template <int R>
static bool dispatch_yz(const YzArgs& a, unsigned blocks, hipStream_t s) {
  switch (a.nz) {
    case 16: return launch_yz<16, R>(a, blocks, s);
    case 32: return launch_yz<32, R>(a, blocks, s);
    case 64: return launch_yz<64, R>(a, blocks, s);
    case 128: return launch_yz<128, R>(a, blocks, s);
    case 256: return launch_yz<256, R>(a, blocks, s);
    default: return false;
  }
}

void preload_yz() { preload_kernel(reinterpret_cast<const void*>(&k_fft_yz<16, 4, false, false>)); }

int launch_fft_yz(const YzArgs& a, void* stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (yz_split(a.nz, (long long)a.ly * a.r, a.lx) != a.r || !a.w512 || a.wstep * a.ly * a.r != 512 || a.nblocks == 0)
    return -1;
  const unsigned long long blocks = a.nblocks * a.ly * (a.lx / YZ_C);
  if (blocks > 0xFFFFFFFFull / 1024) return -1;  // grid size in work-items is 32-bit
  const bool ok = a.r == 4    ? dispatch_yz<4>(a, (unsigned)blocks, s)
                  : a.r == 8  ? dispatch_yz<8>(a, (unsigned)blocks, s)
                  : a.r == 16 ? dispatch_yz<16>(a, (unsigned)blocks, s)
                              : false;
  if (!ok) return -1;
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace fftamd
