// fft_plane.h -- arguments of the plane passes: the 2D transform of every
// (LY x LX) plane of an array, both axes in one pass over HBM.
#pragma once

namespace fftamd {

struct PlaneArgs {
  const void* in;
  void* out;
  unsigned long long nplanes;    // planes in the array
  long long plane_stride;        // complex elements between planes
  const void* tw_x;              // Stockham twiddles of the LX-point rows
  const void* tw_y;              // Stockham twiddles of the LY-point columns
  const float* w_load;           // optional real weights (see PassArgs)
  const float* w_store;
  unsigned long long w_mask;
  int inverse;
  // optional transform table (planes up to 128 x 128 only): plane b belongs
  // to transform b / ppt, whose first input and output elements are
  // tab[2 t] and tab[2 t + 1] (complex elements from in / out); NULL: plane b
  // starts at b * plane_stride in both
  const unsigned long long* tab;
  unsigned ppt;
  // 4, 8 or 16: plane b is made of the rows a + rsplit y, a = b mod rsplit, of
  // plane b / rsplit of the array (rsplit LY rows), read there and written as a
  // plane of its own, rows LY a + k; out of place, LX >= 128, FP32 planes of 16384
  // points and more.  0: plain planes
  int rsplit;
};

// 256 x 256 planes, four workgroups per plane (fft_xy.hip).  0 on success, -1
// when the grid does not fit, -2 on a launch error.  Out of place only: in
// and out must not overlap.
int launch_fft_xy256(const PlaneArgs& a, void* stream);

// LY x LX planes with 16 <= LY, LX <= 512 and 1024 <= LY * LX <= the kind's
// maximum below, one workgroup per plane (fft_plane.hip).  split: radix-16
// stages on FP16 matrix cores with hi+lo operands.  FP64: no weights.  0 on success, -1 for an unsupported shape or grid, -2 on a launch
// error.  In place allowed.
constexpr long long PLANE_F32_MAX = 32768, PLANE_SPLIT_MAX = 16384, PLANE_F64_MAX = 8192;
int launch_fft_plane(int ly, int lx, const PlaneArgs& a, void* stream, bool split = false, int prec = 0);
bool plane_shape_supported(long long ly, long long lx, int kind);  // kind: PassKind

// The 3D transform of every lz x ly x lx box of an array of boxes, sides 16 to
// 64, up to BOX_F32_MAX or BOX_F64_MAX points, one workgroup per box
// (fft_box.hip).  FP64: no weights.  0 on success, -1 for an unsupported shape
// or grid, -2 on a launch error.  In place allowed.
struct BoxArgs {
  const void* in;
  void* out;
  unsigned long long nboxes;
  const void* tw_z;              // Stockham twiddles of each axis
  const void* tw_y;
  const void* tw_x;
  const float* w_load;           // optional real weights (see PassArgs)
  const float* w_store;
  unsigned long long w_mask;
  int inverse;
};
constexpr long long BOX_F32_MAX = 16384, BOX_F64_MAX = 8192;
constexpr unsigned long long BOX_MAX_COUNT = 0xFFFFFFFFull / 1024;  // grid size in work-items is 32-bit
int launch_fft_box(int lz, int ly, int lx, const BoxArgs& a, void* stream, int prec);
bool box_supported(long long lz, long long ly, long long lx, int prec);

// The l-point transform (l = 4096 or 2048) along the second-fastest axis of
// blocks of l rows of lx elements (fft_col.hip): element (o, row, x) at o * in_o
// + row * lx + x.  l / 2048 workgroups per group of 16 adjacent columns.
struct ColArgs {
  const void* in;
  void* out;
  int l;
  long long lx;                  // row length in complex elements (multiple of 16)
  long long in_o;                // elements between blocks (l * lx)
  unsigned long long nitems;     // blocks x column groups
  unsigned ngroups;              // column groups per block (lx / 16)
  const void* w256;              // W256^m, m = 0..255
  const void* ptw_lo;            // W_l^t = ptw_hi[t >> ptw_hb] * ptw_lo[t & (2^ptw_hb - 1)]
  const void* ptw_hi;
  unsigned ptw_hb;
  const float* w_load;           // optional real weights (see PassArgs)
  const float* w_store;
  unsigned long long w_mask;
  int inverse;
};

// 0 on success, -1 for an unsupported shape or grid, -2 on a launch error.
// Out of place only: in and out must not overlap.
int launch_fft_col(const ColArgs& a, void* stream);
bool col_supported(int l, long long lx, unsigned long long nouter);

// Arrays of n x n x n blocks (n = 512, 256 or 128) in two passes with the y
// axis split between them: (n/4) x 4 for n = 256 and 128 (fft_cube.hip),
// 64 x 8 for n = 512 (fft_cube512.hip).  Pass A: x and the larger y stage of
// every plane, out of place only.  Pass B: the smaller y stage and z of every
// block, in place allowed.  Pass A takes load weights only, pass B store
// weights only (see PassArgs).  0 on success, -1 for an unsupported shape or
// grid, -2 on a launch error.
struct CubeArgs {
  const void* in;
  void* out;
  int n;                         // block side: 512, 256 or 128
  unsigned long long nplanes;    // n x n planes in the array (a multiple of n for pass B)
  const void* tw;                // Stockham twiddles of n-point lines (not read for n = 512)
  const void* w256;              // W256^m, m = 0..255 (in the values' precision)
  const void* w512;              // W512^m, m = 0..511 (n = 512)
  const float* w_load;
  const float* w_store;
  unsigned long long w_mask;
  int inverse;
  int split;                     // radix-16 stages on FP16 MFMA with hi + lo operands (no weights)
  int f64;                       // FP64 values and tables (n = 128, no weights)
  // optional transform table (n = 128 only, no weights): block t starts at
  // tab[2 t] in `in` and tab[2 t + 1] in `out` (complex elements); NULL:
  // block t at t n^3 in both
  const unsigned long long* tab;
};
int launch_fft_cube_a(const CubeArgs& a, void* stream);
int launch_fft_cube_b(const CubeArgs& a, void* stream);
int launch_fft_c512_a(const CubeArgs& a, void* stream);  // n = 512 (fft_cube512.hip)
int launch_fft_c512_b(const CubeArgs& a, void* stream);

// Boxes of nz x (ly r) x lx whose y axis is split r x ly: the second pass, after
// a plane pass with rsplit = r (fft_yz.hip).  In place allowed.  0 on success, -1
// for an unsupported shape or grid, -2 on a launch error.
struct YzArgs {
  const void* in;
  void* out;
  int nz, r;
  unsigned ly, lx;
  unsigned long long nblocks;
  const void* tw;                // Stockham twiddles of nz-point lines
  const void* w512;              // W512^m, m = 0..511; W_{ly r}^t = W512^{wstep t}
  unsigned wstep;
  const float* w_store;          // optional real weights (see PassArgs)
  unsigned long long w_mask;
  int inverse;
  int stream;                    // non-temporal stores: for arrays that outgrow the caches
};
constexpr bool yz_tile_ok(int nz, int r) { return nz >= 16 && nz <= 256 && nz * r <= 1024; }
// How many ways the y axis of an nz x ny x nx box is split: so that the first
// pass has planes of 16384 points (two workgroups per CU); 0 where there is no
// such pair.  Planes of up to 32768 points have a plane pass of their own, 256 x
// 256 ones the four-workgroup one.  Against three line passes, at any batch (the
// smallest, one box of 16 x 128 x 512, 23.4 -> 21.5 us): 4 x (64 x 512 x 128) 151 ->
// 100 us, 2 x (128 x 512 x 256) 289 -> 218, 4 x (64 x 128 x 512) 141 -> 109, 64 x 512 x
// 512 142 -> 118.  First-pass planes of 32768 points, which would take deeper
// boxes, gained nothing: 256 x 256 x 512 278 and 284, 128 x 512 x 512 287 and 288.
constexpr int yz_split(long long nz, long long ny, long long nx) {
  if (nx < 128 || nx > 512 || ny < 128 || ny > 512 || (nx & (nx - 1)) || (ny & (ny - 1)) || (nz & (nz - 1)) || nz < 16 ||
      nz > 256 || ny * nx < 65536 || (ny == 256 && nx == 256))
    return 0;
  const int r = (int)(ny * nx / 16384);
  return yz_tile_ok((int)nz, r) ? r : 0;
}
int launch_fft_yz(const YzArgs& a, void* stream);

// gw[i] = sum_b Re(conj(g[b][i]) f[b][i]) for FP32 complex g, f of batch x
// points values (fft_wgrad.hip).  0 on success, -1 when the grid does not fit,
// -2 on a launch error.
int launch_weight_grad(const void* g, const void* f, void* gw, unsigned long long points, unsigned batch,
                       void* stream);

}  // namespace fftamd
