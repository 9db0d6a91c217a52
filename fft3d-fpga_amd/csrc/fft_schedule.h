// fft_schedule.h -- compile-time radix schedule and launch geometry of the
// Stockham line-FFT pass kernels.  Shared by the device kernels and by the
// host code that builds twiddle tables and launch grids, so both always agree.
//
// A "line" is one 1D transform of L = 2^lg points.  A pass kernel holds C
// lines per workgroup, PPT points of each line per thread (TPL threads per
// line), and runs NP radix stages: the first of radix 2^(lg - 4(NP-1)), the
// rest radix 16.  Stage s sees sub-transforms of span NS(s) = prod of the
// radices before it (Stockham autosort: natural order in, natural order out).
#pragma once

namespace fftamd {

// MODE_PLANE: fused x+y pass over whole planes (fft_xy.hip for 256 x 256,
// fft_plane.hip for smaller ones); MODE_COL: a 4096- or 2048-point second-fastest
// axis in one pass (fft_col.hip); MODE_CUBE_A / MODE_CUBE_B: the two passes of
// 256 x 256 x 256 blocks with the y axis split 64 x 4 (fft_cube.hip); MODE_BOX:
// all three axes of small boxes in one pass (fft_box.hip)
enum PassMode { MODE_CONTIG = 0, MODE_STRIDED = 1, MODE_PLANE = 2, MODE_COL = 3, MODE_CUBE_A = 4,
                MODE_CUBE_B = 5, MODE_BOX = 6, MODE_YA = 7, MODE_YB = 8 };
// EPI_TWIDDLE multiplies point k of column c by W_M^{(c >> cshift) * k}
// (four-step split of a long axis); EPI_BITREV stores point k at bitrev(k).
// EPI_TWIDDLE_T is EPI_TWIDDLE of a strided pass whose output lines are
// contiguous (out_p == 1): the launcher picks it, a plan says EPI_TWIDDLE.
enum PassEpilogue { EPI_NONE = 0, EPI_TWIDDLE = 1, EPI_BITREV = 2, EPI_TWIDDLE_T = 3 };
enum Precision { PREC_F32 = 0, PREC_F64 = 1 };

constexpr int ilog2c(long long x) { return x <= 1 ? 0 : 1 + ilog2c(x >> 1); }

// ---- radix schedule ------------------------------------------------------
constexpr int sched_np(int L) { return L <= 16 ? 1 : (ilog2c(L) + 3) / 4; }
constexpr int sched_radix(int L, int s) {
  return s == 0 ? (1 << (ilog2c(L) - 4 * (sched_np(L) - 1))) : 16;
}
constexpr int sched_ns(int L, int s) {
  int n = 1;
  for (int i = 0; i < s; ++i) n *= sched_radix(L, i);
  return n;
}
// Stages s >= 1 are radix 16.  Their twiddles sit at [twoff(s) + 4k + q],
// k < NS(s), holding W_{16 NS}^{k * 2^q} for q = 0..3; the other powers
// W^{k r} (r = 1..15) are formed by at most three complex products.
constexpr int TW_PER_K = 4;
constexpr int sched_twoff(int L, int s) {
  int o = 0;
  for (int i = 1; i < s; ++i) o += sched_ns(L, i) * TW_PER_K;
  return o;
}
constexpr int sched_twsize(int L) { return sched_twoff(L, sched_np(L)); }

// ---- geometry -------------------------------------------------------------
constexpr int geom_ppt(int L) { return L < 16 ? L : 16; }
constexpr int geom_tpl(int L) { return L / geom_ppt(L); }
// Lines per workgroup.  Contiguous lines: 256 threads per workgroup (one line
// per workgroup from L = 4096 up).  Strided lines: at least 16 adjacent
// columns (128-byte row segments; narrower segments measured far slower) and
// 256 threads up to L = 256; at L = 512 32 columns (256-byte segments, 1024
// threads; measured 7-18% faster than 16 on the y and z passes of a 512^3 array,
// slower at L = 256) for large launches, see geom_cols_launch; 16 columns
// (1024 threads) at L = 1024, the four-step passes of long 1D axes.
constexpr int geom_cols(int L, int mode) {
  return mode == MODE_CONTIG ? (geom_tpl(L) >= 256 ? 1 : 256 / geom_tpl(L))
                             : (L >= 1024 ? 16 : L >= 512 ? 32 : L >= 256 ? 16 : 256 / geom_tpl(L));
}
constexpr int geom_threads(int L, int mode) { return geom_cols(L, mode) * geom_tpl(L); }
// Lines per workgroup of a line pass by the kind of its stages.  Strided lines
// of 512 points and more: split precision keeps 16 columns (two workgroups per
// CU; with the FP32 layout's 32 columns, one, the split 512^3 line passes took
// 1.80 against 1.59 ms), FP64 8 (128-byte segments; 1024 points are 144 KiB of
// LDS).
enum PassKind { KIND_F32 = 0, KIND_SPLIT = 1, KIND_F64 = 2 };
constexpr int pass_kind(bool split, int prec) { return split ? KIND_SPLIT : prec == PREC_F64 ? KIND_F64 : KIND_F32; }
constexpr int geom_cols_for(int L, int mode, int kind) {
  return mode == MODE_STRIDED && L >= 512 && kind != KIND_F32 ? (kind == KIND_SPLIT ? 16 : 8) : geom_cols(L, mode);
}
// Smaller tiles for a launch whose usual ones would leave CUs idle: `mid`, one
// wave or 16 strided columns, and `tiny`, 8 strided columns (64-byte segments),
// 0 where the kind of line has none.
constexpr int geom_wave_lines(int L) { return geom_tpl(L) >= 64 ? 1 : 64 / geom_tpl(L); }
constexpr int geom_cols_mid(int L, int mode, int kind) {
  const int c = mode == MODE_CONTIG || geom_wave_lines(L) > 16 ? geom_wave_lines(L) : 16;
  return kind != KIND_SPLIT && c < geom_cols_for(L, mode, kind) ? c : 0;
}
constexpr int geom_cols_tiny(int L, int mode, int kind) {
  return kind != KIND_SPLIT && mode == MODE_STRIDED && geom_wave_lines(L) <= 8 && geom_cols_for(L, mode, kind) > 8 ? 8
                                                                                                                  : 0;
}
// Lines per workgroup of a launch of `lines` lines: `mid` where the usual tile
// gives at most half of the 256 CUs a workgroup, then `tiny` below 64 workgroups.
// Measured for both passes of natural-order 1D transforms: 2^18 points (16
// workgroups of 32 columns) 20.9 us, of 8 columns 14.2; 2^21 (128 of 32 in its
// first pass) 37.3 us, of 16 columns 35.2; 12 x 2^18 of 16 columns 29.1 us, of 8
// 36.0; 2^20 (64 of 16) 25.0 us, of 8 24.6; 3 x 2^20 (192 of 16) 29.1 us, of 8
// 36.8.  Contiguous 1024-point lines, 100 of them (25 workgroups of four): 10.9
// us, one per workgroup 9.8.
// FP32 strided lines of 512 points take 16 columns, two workgroups per CU instead
// of one of 1024 threads, up to 512 MiB: 60 x 2^18 points 120.4 -> 103.8 us, 8 x (512 x
// 256 x 16) 99.9 -> 92.3, 8 x (512 x 4096) 102.5 -> 93.2, 256 MiB 2 x (512 x 256 x 128)
// 248.5 -> 246.4; past the caches 1000 x (512 x 256), 1 GiB, 797 -> 831.
constexpr int geom_cols_launch(int L, int mode, int kind, unsigned long long lines) {
  int c = geom_cols_for(L, mode, kind);
  const int mid = geom_cols_mid(L, mode, kind), tiny = geom_cols_tiny(L, mode, kind);
  const bool l512 = L == 512 && mode == MODE_STRIDED && kind == KIND_F32;
  if (mid && lines <= (l512 ? 131072ull : 128ull * (unsigned)c)) c = mid;
  if (tiny && lines < 64ull * (unsigned)c) c = tiny;
  return c;
}

// Largest line held by one workgroup (LDS budget).  Longer axes are split
// four-step into two passes.
constexpr int lmax_contig(int prec) { return prec == PREC_F32 ? 8192 : 4096; }
constexpr int lmax_strided(int prec) { return prec == PREC_F32 ? 512 : 256; }
// The strided passes of a four-step split of a long contiguous axis may hold
// 1024 points (16 columns FP32, 8 FP64, 139-144 KiB of LDS): 2^22 points as
// 1024 x 4096 measured 38.1 against 41.4 us for 512 x 8192.
constexpr int lmax_strided_fourstep(int) { return 1024; }

}  // namespace fftamd
