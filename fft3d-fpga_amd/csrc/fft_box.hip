// fft_box.hip -- the 3D transform of small boxes in one pass over HBM, one
// workgroup per box of LZ x LY x LX = 4096 to 16384 points (FP64: 8192), sides
// from 16.
//
// LZ * LY * LX / 16 threads hold the box in registers, 16 points each, and in
// LDS (34 to 136 KiB) between the axes.  z first: adjacent threads load adjacent
// (y, x) columns, whole 128-byte segments and more; then the rows along x, then
// y, whose last stage stores adjacent x.  The stages are the line passes'
// (fft_pass_dev.h), two LDS exchanges between the three axes.
//
// HBM bound: one read and one write, instead of the three line passes of 16^3
// boxes (whose 256-column tiles held 16 columns of each box) or a plane and a z
// pass.  1000 x 16^3 67.7 -> 12.1 us (5.4 TB/s), 1000 x (16 x 16 x 32) 85.4 -> 31.4,
// 1000 x (16 x 32 x 32) 103.5 -> 72.9 (one workgroup per CU), FP64 1000 x 16^3 106.7
// -> 28.1.  In place allowed: a workgroup holds its whole box before it stores.
#include <hip/hip_runtime.h>

#include "launch.h"

#include "fft_pass_dev.h"
#include "fft_plane.h"

namespace fftamd {

constexpr int max3(int a, int b, int c) { return a > b ? (a > c ? a : c) : (b > c ? b : c); }

template <int LZ, int LY, int LX>
struct BoxGeom {
  static constexpr int N = LZ * LY * LX, NT = N / 16, S = LY * LX;
  using GZ = Geom<LZ, MODE_STRIDED, S>;        // columns (y, x) along z
  using GX = Geom<LX, MODE_CONTIG, LZ * LY>;   // rows (z, y)
  using GY = Geom<LY, MODE_STRIDED, LX>;       // columns x along y, one set per z
  static_assert(LZ >= 16 && LY >= 16 && LX >= 16 && GZ::NT == NT && GX::NT == NT && LZ * GY::NT == NT,
                "16 points per thread for every axis");
  static constexpr int LDS = max3(GZ::LDS_ELEMS, GX::LDS_ELEMS, LZ * GY::LDS_ELEMS);
};

template <int LZ, int LY, int LX, bool INV, typename R>
__global__ void __launch_bounds__(LZ * LY * LX / 16) k_fft_box(const BoxArgs a) {
  using BG = BoxGeom<LZ, LY, LX>;
  using GZ = typename BG::GZ;
  using GX = typename BG::GX;
  using GY = typename BG::GY;
  constexpr int S = BG::S;
  __shared__ cpx<R> lds[BG::LDS];
  const unsigned long long base = (unsigned long long)blockIdx.x * BG::N;
  const cpx<R>* in = reinterpret_cast<const cpx<R>*>(a.in) + base;
  cpx<R>* out = reinterpret_cast<cpx<R>*>(a.out) + base;
  const int tid = threadIdx.x;
  cpx<R> v[16];

  // ---- z: thread (column c, tau); stage 0 reads its butterfly inputs from HBM
  {
    constexpr int RAD = sched_radix(LZ, 0), NB = 16 / RAD;
    const int c = tid % S, tau = tid / S;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < RAD; ++r) {
        const int e = (tau + b * GZ::TPL + r * (LZ / RAD)) * S + c;
        cpx<R> x = in[e];
        if (a.w_load) x = cscale(x, (R)a.w_load[(base + e) & a.w_mask]);
        v[b * RAD + r] = INV ? cswap(x) : x;
      }
    run_stages<R, LZ, MODE_STRIDED, 0, false, S>(v, lds, c, tau, reinterpret_cast<const cpx<R>*>(a.tw_z));
    constexpr int NP = GZ::NP, RL = sched_radix(LZ, NP - 1), NSL = sched_ns(LZ, NP - 1);
    if constexpr (NP > 1) __syncthreads();  // the last stage has read its inputs
#pragma unroll
    for (int b = 0; b < 16 / RL; ++b)
#pragma unroll
      for (int r = 0; r < RL; ++r)
        lds[GX::idx((tau + b * GZ::TPL + r * NSL) * LY + c / LX, c % LX)] = v[b * RL + r];
  }
  __syncthreads();

  // ---- x: thread (row c = (z, y), tau)
  {
    const int c = tid / GX::TPL, tau = tid % GX::TPL;
    stage_load_lds<R, LX, MODE_CONTIG, 0, LZ * LY>(v, lds, c, tau);
    if constexpr (GX::NP > 1) __syncthreads();  // every thread holds its stage-0 inputs before stage 0 stores
    run_stages<R, LX, MODE_CONTIG, 0, false, LZ * LY>(v, lds, c, tau, reinterpret_cast<const cpx<R>*>(a.tw_x));
    constexpr int NP = GX::NP, RL = sched_radix(LX, NP - 1), NSL = sched_ns(LX, NP - 1);
    __syncthreads();  // every thread has read its last row inputs
    cpx<R>* plane = lds + (c / LY) * GY::LDS_ELEMS;
#pragma unroll
    for (int b = 0; b < 16 / RL; ++b)
#pragma unroll
      for (int r = 0; r < RL; ++r) plane[GY::idx(tau + b * GX::TPL + r * NSL, c % LY)] = v[b * RL + r];
  }
  __syncthreads();

  // ---- y: thread (z, column c = x, tau), adjacent threads on adjacent columns
  {
    const int z = tid / GY::NT, t = tid % GY::NT;
    const int c = t % LX, tau = t / LX;
    cpx<R>* plane = lds + z * GY::LDS_ELEMS;
    stage_load_lds<R, LY, MODE_STRIDED, 0, LX>(v, plane, c, tau);
    if constexpr (GY::NP > 1) __syncthreads();
    run_stages<R, LY, MODE_STRIDED, 0, false, LX>(v, plane, c, tau, reinterpret_cast<const cpx<R>*>(a.tw_y));
    constexpr int NP = GY::NP, RL = sched_radix(LY, NP - 1), NSL = sched_ns(LY, NP - 1);
#pragma unroll
    for (int b = 0; b < 16 / RL; ++b)
#pragma unroll
      for (int r = 0; r < RL; ++r) {
        const int e = z * S + (tau + b * GY::TPL + r * NSL) * LX + c;
        cpx<R> x = v[b * RL + r];
        if (INV) x = cswap(x);
        if (a.w_store) x = cscale(x, (R)a.w_store[(base + e) & a.w_mask]);
        out[e] = x;
      }
  }
}

constexpr bool box_ok(long long lz, long long ly, long long lx, int prec) {
  const long long m = prec == PREC_F32 ? BOX_F32_MAX : BOX_F64_MAX;
  auto side = [](long long v) { return v >= 16 && v <= 64 && (v & (v - 1)) == 0; };
  return side(lz) && side(ly) && side(lx) && lz * ly * lx <= m;
}
bool box_supported(long long lz, long long ly, long long lx, int prec) { return box_ok(lz, ly, lx, prec); }

template <typename R, int LZ, int LY, int LX>
static bool launch_shape(const BoxArgs& a, hipStream_t s) {
  if constexpr (!box_ok(LZ, LY, LX, sizeof(R) == 4 ? PREC_F32 : PREC_F64)) {
    return false;
  } else {
    const dim3 g((unsigned)a.nboxes), t(BoxGeom<LZ, LY, LX>::NT);
    if (a.inverse) FFTAMD_LAUNCH((k_fft_box<LZ, LY, LX, true, R>), g, t, 0, s, a);
    else FFTAMD_LAUNCH((k_fft_box<LZ, LY, LX, false, R>), g, t, 0, s, a);
    return true;
  }
}

template <typename R, int LZ, int LY>
static bool dispatch_x(int lx, const BoxArgs& a, hipStream_t s) {
  return lx == 16 ? launch_shape<R, LZ, LY, 16>(a, s)
         : lx == 32 ? launch_shape<R, LZ, LY, 32>(a, s)
                    : lx == 64 && launch_shape<R, LZ, LY, 64>(a, s);
}
template <typename R, int LZ>
static bool dispatch_y(int ly, int lx, const BoxArgs& a, hipStream_t s) {
  return ly == 16 ? dispatch_x<R, LZ, 16>(lx, a, s)
         : ly == 32 ? dispatch_x<R, LZ, 32>(lx, a, s)
                    : ly == 64 && dispatch_x<R, LZ, 64>(lx, a, s);
}
template <typename R>
static bool dispatch_z(int lz, int ly, int lx, const BoxArgs& a, hipStream_t s) {
  return lz == 16 ? dispatch_y<R, 16>(ly, lx, a, s)
         : lz == 32 ? dispatch_y<R, 32>(ly, lx, a, s)
                    : lz == 64 && dispatch_y<R, 64>(ly, lx, a, s);
}

void preload_box() { preload_kernel(reinterpret_cast<const void*>(&k_fft_box<16, 16, 16, false, float>)); }

int launch_fft_box(int lz, int ly, int lx, const BoxArgs& a, void* stream, int prec) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (!box_ok(lz, ly, lx, prec) || a.nboxes == 0 || a.nboxes > BOX_MAX_COUNT ||
      (prec == PREC_F64 && (a.w_load || a.w_store)))
    return -1;
  const bool ok = prec == PREC_F32 ? dispatch_z<float>(lz, ly, lx, a, s) : dispatch_z<double>(lz, ly, lx, a, s);
  if (!ok) return -1;
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace fftamd
