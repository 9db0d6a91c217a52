// fft_plane.hip -- the 2D transform of every LY x LX plane of an array in one
// pass over HBM, for planes of 1024 to 32768 points with sides 16 to 512: up to
// 8192 points the plane sits in one workgroup's LDS, above that in its registers.
//
// One workgroup per plane, LY * LX / 16 threads, 16 points per thread in both
// phases.  Rows: each thread loads its first-stage butterfly inputs of one row
// straight from HBM (coalesced along the row), runs the Stockham stages with
// LDS exchanges ([row][x + x/16] layout), and writes the row's results into
// the column layout ([y][col], one pad column).  Columns: the same stages
// along y, and the last stage writes natural-order rows to HBM (coalesced
// along x).  A 3D transform of 128^3-sized planes then takes two passes over
// HBM instead of three, and the plane is read and written exactly once.
//
// The radix stages are the line passes' (fft_pass_dev.h), instantiated with a
// whole plane's rows or columns per workgroup.  FP32 planes of 16384 points and
// more use k_fft_plane_halves below.
//
// HBM bound: one read and one write instead of the two of separate x and y line
// passes.  1024 planes of 16 x 256 24.1 -> 12.8 us, of 512 x 16 103.6 -> 48.0, of
// 32 x 256 52.7 -> 31.6, of 64 x 256 96.2 -> 60.5, of 512 x 32 133.0 -> 67.6; of 128 x
// 256 (one workgroup per CU, 256 KiB planes) 197.4 -> 129.5.
#include <hip/hip_runtime.h>

#include "launch.h"

#include "fft_pass_dev.h"
#include "fft_plane.h"
#include "fft_plane_dev.h"

namespace fftamd {

// SPLIT: radix-16 stages on FP16 matrix cores with hi+lo operands (fft_split.h).
// FP64 planes of up to 8192 points (139 KiB of LDS; up to 4096 points two
// workgroups per CU): a 3D array of such planes takes two passes over HBM
// instead of three line passes.  30 x 64^3 129.8 -> 92.4 us, 200 x 32^3 128.5
// -> 78.6 us; 8192 points, one workgroup per CU: 500 planes of 64 x 128 46.6 ->
// 30.5 us, 13 x (64 x 128 x 64) 117.7 -> 97.5 us.
template <int LY, int LX, bool INV, bool SPLIT, typename R = float>
__global__ void __launch_bounds__(LY * LX / 16) k_fft_plane(const PlaneArgs a) {
  __shared__ cpx<R> lds[PlaneGeom<LY, LX, SPLIT>::LDS];
  plane_tile<LY, LX, INV, SPLIT, R>(a, blockIdx.x, lds, (int)threadIdx.x);
}

// Planes of 16384 points (128 KiB) and 32768 points (256 KiB) in two halves:
// 512 or 1024 threads hold the plane in registers (32 points each) and LDS
// stages half of it at a time (rows 0..LY/2-1, then the others; then columns
// 0..LX/2-1, then the others).  At 16384 points LDS is then 68 KiB, so two
// workgroups share a CU and one loads or stores while the other computes; the
// whole-plane kernel above needs 136 KiB and runs one workgroup per CU.  At 32768
// points (1024 threads, at most 139 KiB) it is one workgroup per CU.
template <int LY, int LX>
struct HalfGeom {
  using GX = Geom<LX, MODE_CONTIG, LY / 2>;   // rows: LY/2 lines of LX points
  using GY = Geom<LY, MODE_STRIDED, LX / 2>;  // columns: LX/2 lines of LY points
  static constexpr int NT = LY * LX / 32;
  static_assert(GX::NT == NT && GY::NT == NT, "16 points per thread per half");
  static constexpr int LDS = GX::LDS_ELEMS > GY::LDS_ELEMS ? GX::LDS_ELEMS : GY::LDS_ELEMS;
  // last row stage: radix 16, one butterfly per thread, so point k = tau + TPL r
  static_assert(sched_radix(LX, GX::NP - 1) == 16 && sched_ns(LX, GX::NP - 1) == GX::TPL,
                "points tau + TPL r: r < 8 are columns 0 .. LX/2 - 1");
};

// WL, WS: the launch carries load or store weights.  RS: planes of every rsplit-th
// row (see PlaneArgs), the first pass of a box with larger planes.
template <int LY, int LX, bool INV, bool WL, bool WS, bool RS = false>
__global__ void __launch_bounds__(LY * LX / 32, 4) k_fft_plane_halves(const PlaneArgs a) {
  using HG = HalfGeom<LY, LX>;
  using GX = typename HG::GX;
  using GY = typename HG::GY;
  constexpr int HY = LY / 2, HX = LX / 2;
  __shared__ cpx<float> lds[HG::LDS];
  const unsigned long long plane = blockIdx.x;
  long long base = (long long)plane * a.plane_stride, obase = base;
  if (a.tab) {  // planes of a batch of transforms placed anywhere
    const unsigned t = (unsigned)(plane / a.ppt), z = (unsigned)(plane % a.ppt);
    base = (long long)a.tab[2 * t] + (long long)z * (LY * LX);
    obase = (long long)a.tab[2 * t + 1] + (long long)z * (LY * LX);
  }
  const int rstride = RS ? a.rsplit * LX : LX;  // between the plane's rows
  if (RS) {
    const long long res = (long long)(plane & (unsigned)(a.rsplit - 1));
    base = ((long long)plane - res) * (LY * LX) + res * LX;
  }
  const cpx<float>* __restrict__ in = reinterpret_cast<const cpx<float>*>(a.in) + base;
  cpx<float>* __restrict__ out = reinterpret_cast<cpx<float>*>(a.out) + obase;
  const int tid = threadIdx.x;
  cpx<float> rr[2][16];  // row results of row halves 0 and 1: point tau + TPL r of row c + HY h

  // ---- rows, in two halves: thread (row c, tau); stage 0 reads from HBM
  const int rc = tid / GX::TPL, rtau = tid % GX::TPL;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    using D = RowDeal<LX, HY>;
    constexpr int RAD = D::RAD, NB = 16 / RAD;
    cpx<float>* v = rr[h];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
#pragma unroll
      for (int r = 0; r < RAD; ++r) {
        const int e = (D::row(tid, b) + HY * h) * rstride + D::j(tid, b) + r * D::J;
        cpx<float> x = in[e];
        if (WL) x = cscale(x, a.w_load[(unsigned long long)(base + e) & a.w_mask]);
        v[b * RAD + r] = INV ? cswap(x) : x;
      }
    }
    if (h) __syncthreads();  // the first half's last stage has read the buffer
    run_rows<float, LX, false, HY, false>(v, lds, tid, reinterpret_cast<const cpx<float>*>(a.tw_x));
  }

  // ---- columns, in two halves: thread (column c, tau), adjacent threads on adjacent columns
  const int cc = tid % HX, ctau = tid / HX;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    __syncthreads();  // the previous stage has read the buffer
    // points tau + TPL r with r in [8h, 8h + 8) are the columns of half h
#pragma unroll
    for (int rh = 0; rh < 2; ++rh)
#pragma unroll
      for (int r = 0; r < 8; ++r) lds[GY::idx(rtau + GX::TPL * r, rc + HY * rh)] = rr[rh][8 * h + r];
    __syncthreads();
    cpx<float> v[16];
    stage_load_lds<float, LY, MODE_STRIDED, 0, HX>(v, lds, cc, ctau);
    __syncthreads();  // every thread holds its stage-0 inputs before stage 0 stores
    run_stages<float, LY, MODE_STRIDED, 0, false, HX, false>(v, lds, cc, ctau, reinterpret_cast<const cpx<float>*>(a.tw_y));
    constexpr int NPY = GY::NP;
    constexpr int RL = sched_radix(LY, NPY - 1), NSL = sched_ns(LY, NPY - 1), NBL = 16 / RL;
#pragma unroll
    for (int b = 0; b < NBL; ++b) {
      const int j = ctau + b * GY::TPL;
#pragma unroll
      for (int r = 0; r < RL; ++r) {
        const int e = (j + r * NSL) * LX + HX * h + cc;
        cpx<float> x = v[b * RL + r];
        if (INV) x = cswap(x);
        if (WS) x = cscale(x, a.w_store[(unsigned long long)(obase + e) & a.w_mask]);
        out[e] = x;
      }
    }
  }
}

// shapes that yz_split leaves the first pass
constexpr bool rsplit_shape(int ly, int lx) { return lx >= 128 && ly * lx == 16384; }

template <int LY, int LX, bool INV>
static void launch_halves(const PlaneArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)a.nplanes), block(HalfGeom<LY, LX>::NT);
  if constexpr (rsplit_shape(LY, LX)) {
    if (a.rsplit) {
      if (a.w_load) FFTAMD_LAUNCH((k_fft_plane_halves<LY, LX, INV, true, false, true>), grid, block, 0, s, a);
      else FFTAMD_LAUNCH((k_fft_plane_halves<LY, LX, INV, false, false, true>), grid, block, 0, s, a);
      return;
    }
  }
  if (a.w_load) {
    if (a.w_store) FFTAMD_LAUNCH((k_fft_plane_halves<LY, LX, INV, true, true>), grid, block, 0, s, a);
    else FFTAMD_LAUNCH((k_fft_plane_halves<LY, LX, INV, true, false>), grid, block, 0, s, a);
  } else {
    if (a.w_store) FFTAMD_LAUNCH((k_fft_plane_halves<LY, LX, INV, false, true>), grid, block, 0, s, a);
    else FFTAMD_LAUNCH((k_fft_plane_halves<LY, LX, INV, false, false>), grid, block, 0, s, a);
  }
}

template <int LY, int LX, bool SPLIT>
static void launch_shape_f32(const PlaneArgs& a, hipStream_t s) {
  if constexpr (LY * LX >= 16384 && !SPLIT) {
    if (a.inverse) launch_halves<LY, LX, true>(a, s);
    else launch_halves<LY, LX, false>(a, s);
  } else {
    // split-precision stages would spill registers in the halves kernel and
    // keep the whole plane in LDS (up to 16384 points)
    constexpr int NT = PlaneGeom<LY, LX, SPLIT>::NT;
    if (a.inverse)
      FFTAMD_LAUNCH((k_fft_plane<LY, LX, true, SPLIT>), dim3((unsigned)a.nplanes), dim3(NT), 0, s, a);
    else
      FFTAMD_LAUNCH((k_fft_plane<LY, LX, false, SPLIT>), dim3((unsigned)a.nplanes), dim3(NT), 0, s, a);
  }
}

constexpr bool plane_shape_ok(long long ly, long long lx, int kind) {
  return ly >= 16 && ly <= 512 && lx >= 16 && lx <= 512 && (ly & (ly - 1)) == 0 && (lx & (lx - 1)) == 0 &&
         ly * lx >= 1024 && ly * lx <= (kind == KIND_F32 ? PLANE_F32_MAX : kind == KIND_SPLIT ? PLANE_SPLIT_MAX : PLANE_F64_MAX);
}

bool plane_shape_supported(long long ly, long long lx, int kind) { return plane_shape_ok(ly, lx, kind); }

template <int LY, int LX, bool SPLIT, typename R>
static bool launch_shape(const PlaneArgs& a, hipStream_t s) {
  constexpr int kind = sizeof(R) == 8 ? KIND_F64 : SPLIT ? KIND_SPLIT : KIND_F32;
  if constexpr (!plane_shape_ok(LY, LX, kind)) {
    return false;
  } else if constexpr (kind == KIND_F64) {
    const dim3 g((unsigned)a.nplanes), t(PlaneGeom<LY, LX, false>::NT);
    if (a.inverse) FFTAMD_LAUNCH((k_fft_plane<LY, LX, true, false, double>), g, t, 0, s, a);
    else FFTAMD_LAUNCH((k_fft_plane<LY, LX, false, false, double>), g, t, 0, s, a);
    return true;
  } else {
    launch_shape_f32<LY, LX, SPLIT>(a, s);
    return true;
  }
}

template <int LY, bool SPLIT, typename R>
static bool dispatch_lx(int lx, const PlaneArgs& a, hipStream_t s) {
  switch (lx) {
    case 16: return launch_shape<LY, 16, SPLIT, R>(a, s);
    case 32: return launch_shape<LY, 32, SPLIT, R>(a, s);
    case 64: return launch_shape<LY, 64, SPLIT, R>(a, s);
    case 128: return launch_shape<LY, 128, SPLIT, R>(a, s);
    case 256: return launch_shape<LY, 256, SPLIT, R>(a, s);
    case 512: return launch_shape<LY, 512, SPLIT, R>(a, s);
    default: return false;
  }
}

template <bool SPLIT, typename R = float>
static bool dispatch_ly(int ly, int lx, const PlaneArgs& a, hipStream_t s) {
  switch (ly) {
    case 16: return dispatch_lx<16, SPLIT, R>(lx, a, s);
    case 32: return dispatch_lx<32, SPLIT, R>(lx, a, s);
    case 64: return dispatch_lx<64, SPLIT, R>(lx, a, s);
    case 128: return dispatch_lx<128, SPLIT, R>(lx, a, s);
    case 256: return dispatch_lx<256, SPLIT, R>(lx, a, s);
    case 512: return dispatch_lx<512, SPLIT, R>(lx, a, s);
    default: return false;
  }
}

void preload_plane() { preload_kernel(reinterpret_cast<const void*>(&k_fft_plane<64, 64, false, false>)); }

int launch_fft_plane(int ly, int lx, const PlaneArgs& a, void* stream, bool split, int prec) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (!plane_shape_ok(ly, lx, pass_kind(split, prec)) || (prec == PREC_F64 && (split || a.w_load || a.w_store)) || a.nplanes == 0 || a.nplanes > 0xFFFFFFFFull / 1024 ||
      (a.tab && a.ppt == 0))
    return -1;
  if (a.rsplit && (!rsplit_shape(ly, lx) || prec != PREC_F32 || split || a.tab || a.w_store || a.plane_stride != (long long)ly * lx ||
                   (a.rsplit != 4 && a.rsplit != 8 && a.rsplit != 16) || a.nplanes % (unsigned)a.rsplit))
    return -1;
  const bool ok = prec == PREC_F64 ? dispatch_ly<false, double>(ly, lx, a, s)
                  : split           ? dispatch_ly<true>(ly, lx, a, s)
                                    : dispatch_ly<false>(ly, lx, a, s);
  if (!ok) return -1;
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace fftamd
