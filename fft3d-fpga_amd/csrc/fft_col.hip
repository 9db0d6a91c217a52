// fft_col.hip -- the 4096- or 2048-point transform along the second-fastest
// axis of an array (the columns of an R x L x LX block, LX >= 16) in one pass
// over HBM.
//
// A line pass holds whole lines in LDS, and the narrowest coalesced group, 16
// adjacent columns (128-byte row segments), is 512 KiB at 4096 points, so
// otherwise the axis is split four-step into two passes.  Here a workgroup of
// 1024 threads holds 32768 points in registers: the 16 columns of 2048 points
// whole, of 4096 points half of the output rows.  L = N1 x 16, n = n1 + N1 n2,
// k = k1 + 16 k2; at 4096 points part q of two owns the rows with k1 = q mod 2,
// reads all rows of the group and evaluates its eight outputs of each
// first-stage 16-point DFT over n2 (one butterfly step, then an 8-point DFT),
// so no arithmetic is repeated; at 2048 points the one part takes all sixteen.
// Each line (k1, column) is multiplied by W_L^{n1 k1} and transformed over n1
// with the line passes' strided stages, half of the lines at a time through
// LDS (at most 134 KiB, one workgroup per CU).
//
// HBM bound.  The two parts of a group are consecutive blocks of one XCD, so
// the group comes from HBM once and from that XCD's L2 for the other part; they
// read the row groups in different orders, so that what one misses the other
// finds.  Two parts instead of four of 512 threads (which kept the L2 busy with
// four reads of every row, and as much of the data in flight was the same
// data): 4096 x 4096 on inputs not in the caches 97 -> 71 us, with the row pass
// 139.5 -> 114.7 us.  One part of 8 columns (64-byte segments, nothing read
// twice) took 125.6 us with the row pass.
//
// Rows are addressed through buffer resources with one VGPR offset per lane
// and scalar row offsets.  Out of place only.
#include <hip/hip_runtime.h>

#include "launch.h"

#include "fft_pass_dev.h"
#include "fft_plane.h"

namespace fftamd {

constexpr int CL_C = 16;             // columns per group
constexpr int CL_NT = 1024;          // threads per workgroup
constexpr int CL_NG = CL_NT / CL_C;  // first-stage row groups: thread (column, gi) takes n1 = gi + 64 i

template <int L>
struct ColK {
  static_assert(L == 4096 || L == 2048, "32768 points per workgroup");
  static constexpr int Q = L / 2048;        // workgroups per group
  static constexpr int N1 = L / 16;         // n = n1 + N1 n2
  static constexpr int PER = N1 / CL_NG;    // n1 per thread
  static constexpr int LH = 8 / Q;          // k1 per half of the lines
  using G = Geom<N1, MODE_STRIDED, LH * CL_C>;
  static_assert(G::NT == CL_NT, "16 points per thread per half");
};

// x * (-i)^M
template <int M>
__device__ __forceinline__ cpx<float> col_rot(cpx<float> x) {
  constexpr int m = M & 3;
  if constexpr (m == 0) return x;
  else if constexpr (m == 1) return {x.y, -x.x};
  else if constexpr (m == 2) return {-x.x, -x.y};
  else return {-x.y, x.x};
}

// x * W16^P
template <int P>
__device__ __forceinline__ cpx<float> col_w16(cpx<float> x) {
  constexpr int p = P & 15;
  if constexpr ((p & 3) == 0) return col_rot<p / 4>(x);
  else if constexpr (p == 2) return mul_w8_1(x);
  else if constexpr (p == 6) return mul_w8_3(x);
  else if constexpr (p == 10) return col_rot<2>(mul_w8_1(x));
  else if constexpr (p == 14) return col_rot<2>(mul_w8_3(x));
  else {  // odd p: cos(pi p / 8) - i sin(pi p / 8)
    constexpr float c = (p == 1 || p == 15) ? K<float>::C16 : (p == 3 || p == 13) ? K<float>::S16
                        : (p == 5 || p == 11) ? -K<float>::S16 : -K<float>::C16;
    constexpr float sn = (p == 1 || p == 7) ? K<float>::S16 : (p == 3 || p == 5) ? K<float>::C16
                         : (p == 9 || p == 15) ? -K<float>::S16 : -K<float>::C16;
    return cmul(x, cpx<float>{c, -sn});
  }
}

// Outputs k1 = G + Q u, u < 16 / Q, of the 16-point DFT of v[].  Q = 2:
// X[G + 2u] = sum_{a < 8} W8^{a u} W16^{a G} (v[a] + (-1)^G v[a + 8]).
template <int Q, int G>
__device__ __forceinline__ void col_residue(cpx<float>* v) {
  if constexpr (Q == 1) {
    dft16(v);
  } else {
#pragma unroll
    for (int a = 0; a < 8; ++a) v[a] = G ? csub(v[a], v[a + 8]) : cadd(v[a], v[a + 8]);
    if constexpr (G == 1) {
      v[1] = col_w16<1>(v[1]);
      v[2] = col_w16<2>(v[2]);
      v[3] = col_w16<3>(v[3]);
      v[4] = col_w16<4>(v[4]);
      v[5] = col_w16<5>(v[5]);
      v[6] = col_w16<6>(v[6]);
      v[7] = col_w16<7>(v[7]);
    }
    dft8(v);
  }
}

typedef unsigned col_u2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ __amdgpu_buffer_rsrc_t col_rsrc(const void* base, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}

// Stage 2 of the lines (k1 = P + Q (LH h + l), column c16), l < LH, held in
// LDS: the twiddle W_L^{n1 k1}, the N1-point transform over n1 and the stores of
// rows k = k1 + 16 k2.  Thread (line c = 16 l + c16, tau).
template <int L, int P, bool INV, bool WS>
__device__ __forceinline__ void col_stage2(const ColArgs& a, __amdgpu_buffer_rsrc_t rout,
                                           __amdgpu_buffer_rsrc_t rws, int h, cpx<float>* lds,
                                           const cpx<float>* tws) {
  using CK = ColK<L>;
  using G = typename CK::G;
  constexpr int N1 = CK::N1, TPL = G::TPL;
  static_assert(sched_np(N1) == 2 && sched_ns(N1, 1) == TPL, "two stages, the second radix 16 over span TPL");
  const int tid = threadIdx.x;
  const int c = tid % G::C, tau = tid / G::C;
  const int k1 = P + CK::Q * (CK::LH * h + (c >> 4));
  cpx<float> v[16];
  stage_load_lds<float, N1, MODE_STRIDED, 0, G::C>(v, lds, c, tau);
  // point n1 = tau + TPL m: W_L^{n1 k1} = W_L^{tau k1} W256^{m k1} (L / TPL = 256);
  // m of the butterfly inputs v[b RAD + r], n1 = tau + b TPL + r N1 / RAD
  {
    constexpr int RAD = sched_radix(N1, 0), NB = 16 / RAD;
    const cpx<float>* lo = reinterpret_cast<const cpx<float>*>(a.ptw_lo);
    const cpx<float>* hi = reinterpret_cast<const cpx<float>*>(a.ptw_hi);
    const unsigned t = (unsigned)(tau * k1);  // < 256
    const cpx<float> base = cmul(hi[t >> a.ptw_hb], lo[t & ((1u << a.ptw_hb) - 1u)]);
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < RAD; ++r) {
        const int m = b + r * (N1 / RAD / TPL);
        cpx<float> x = cmul(v[b * RAD + r], base);
        if (m) x = cmul(x, tws[15 * k1 + m - 1]);  // W256^{m k1} from the LDS table (k1 < 16)
        v[b * RAD + r] = x;
      }
  }
  __syncthreads();  // every thread holds its stage-0 inputs before stage 0 stores
  stage_compute<float, N1, MODE_STRIDED, 0, false, G::C>(v, tau, nullptr);  // no twiddles
  stage_store_lds<float, N1, MODE_STRIDED, 0, G::C>(v, lds, c, tau);
  __syncthreads();
  stage_load_lds<float, N1, MODE_STRIDED, 1, G::C>(v, lds, c, tau);
  // radix-16 stage over sub-transforms of span TPL: twiddles W_N1^{tau r} = W256^{(256 / N1) tau r}
#pragma unroll
  for (int r = 1; r < 16; ++r) v[r] = cmul(v[r], tws[15 * (256 / N1) * tau + r - 1]);
  dft16(v);
  // point k2 = tau + TPL r of the line: row k1 + 16 k2, 16 lanes on 16 adjacent
  // columns (128 contiguous bytes)
  const unsigned lx8 = (unsigned)a.lx * 8u;
  const unsigned voff = (unsigned)(k1 + 16 * tau) * lx8 + (unsigned)(c & 15) * 8u;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    cpx<float> x = INV ? cswap(v[r]) : v[r];
    const unsigned soff = (unsigned)(16 * TPL * r) * lx8;
    if (WS) x = cscale(x, __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rws, voff / 2u, soff / 2u, 0)));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(col_u2, x), rout, voff, soff, 0);
  }
}

// Part P of the workgroups of a group.
template <int L, int P, bool INV, bool WL, bool WS>
__device__ __forceinline__ void col_part(const ColArgs& a, unsigned long long o, unsigned grp, cpx<float>* lds,
                                         const cpx<float>* tws) {
  using CK = ColK<L>;
  using G = typename CK::G;
  // keep the first loads inside this part's code: hoisted above the branch
  // over the part, they were spilled across it
  asm volatile("" ::: "memory");
  const int tid = threadIdx.x;
  const int c16 = tid & (CL_C - 1);
  // n1 group: 16 threads per group, four groups per wave (not wave-uniform)
  const int gi = tid >> 4;
  const unsigned lx8 = (unsigned)a.lx * 8u;
  const unsigned long long first = o * (unsigned long long)a.in_o + (unsigned long long)grp * CL_C;
  const unsigned bytes = (unsigned)(L - 1) * lx8 + CL_C * 8u;  // the group's span
  const __amdgpu_buffer_rsrc_t rin = col_rsrc(reinterpret_cast<const cpx<float>*>(a.in) + first, bytes);
  const __amdgpu_buffer_rsrc_t rout = col_rsrc(reinterpret_cast<cpx<float>*>(a.out) + first, bytes);
  // weights of element e of the block are w[(o * in_o) & w_mask + e]: the
  // weight period is a multiple of the block (checked by the launcher)
  const unsigned long long wfirst = ((o * (unsigned long long)a.in_o) & a.w_mask) + (unsigned long long)grp * CL_C;
  const __amdgpu_buffer_rsrc_t rwl = col_rsrc(a.w_load + wfirst, bytes / 2u);
  const __amdgpu_buffer_rsrc_t rws = col_rsrc(a.w_store + wfirst, bytes / 2u);
  const unsigned voff = (unsigned)gi * lx8 + (unsigned)c16 * 8u;

  // ---- first stage: thread (c16, gi) for n1 = gi + 64 i: the 16-point DFT
  // over n2 (rows n1 + N1 n2), outputs k1 = P + Q u; the first LH go to LDS as
  // lines 16 u + c16, the others stay in registers.  The row groups i start at
  // another one for each group of columns, and the two parts of a group swap
  // neighbours
  cpx<float> held[CK::PER][CK::LH];
  const int rot = (int)(grp & (CK::PER - 1));
#pragma unroll
  for (int i = 0; i < CK::PER; ++i) {
    const int ir = ((i ^ P) + rot) & (CK::PER - 1);
    cpx<float> v[16];
#pragma unroll
    for (int n2 = 0; n2 < 16; ++n2) {
      const unsigned soff = (unsigned)(CL_NG * ir + CK::N1 * n2) * lx8;
      cpx<float> s = __builtin_bit_cast(cpx<float>, __builtin_amdgcn_raw_buffer_load_b64(rin, voff, soff, 0));
      if (WL) s = cscale(s, __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rwl, voff / 2u, soff / 2u, 0)));
      v[n2] = INV ? cswap(s) : s;
    }
    col_residue<CK::Q, P>(v);
    const int n1 = gi + CL_NG * ir;
#pragma unroll
    for (int u = 0; u < CK::LH; ++u) {
      lds[G::idx(CL_C * u + c16, n1)] = v[u];
      held[i][u] = v[CK::LH + u];
    }
    // the registers are needed for the values held: keep the next group's
    // loads below this group's arithmetic
    __builtin_amdgcn_sched_barrier(0);
  }
  __syncthreads();
  col_stage2<L, P, INV, WS>(a, rout, rws, 0, lds, tws);
  __syncthreads();  // the last stage has read the buffer
#pragma unroll
  for (int i = 0; i < CK::PER; ++i) {
    const int n1 = gi + CL_NG * (((i ^ P) + rot) & (CK::PER - 1));
#pragma unroll
    for (int u = 0; u < CK::LH; ++u) lds[G::idx(CL_C * u + c16, n1)] = held[i][u];
  }
  __syncthreads();
  col_stage2<L, P, INV, WS>(a, rout, rws, 1, lds, tws);
}

// One workgroup per CU: 128 VGPRs, at most 136 KiB of LDS.
template <int L, bool INV, bool WL, bool WS>
__global__ void __launch_bounds__(CL_NT, 4) k_fft_col(const ColArgs a) {
  using CK = ColK<L>;
  __shared__ cpx<float> lds[CK::G::LDS_ELEMS];
  __shared__ cpx<float> tws[16 * 15];  // W256^{k r} at [15 k + r - 1]: stage-2 twiddles (read after barriers)
  if (threadIdx.x < 16 * 15)
    tws[threadIdx.x] = reinterpret_cast<const cpx<float>*>(a.w256)[(threadIdx.x / 15) * (threadIdx.x % 15 + 1)];
  // XCD-aware mapping: block b runs on XCD b % 8; the k-th block of an XCD takes
  // part k % Q of item (k / Q) * 8 + XCD, so the parts of a column group are
  // consecutive blocks of one XCD
  const unsigned b = blockIdx.x;
  const unsigned xcd = b & 7u, k = b >> 3;
  const unsigned long long item = (unsigned long long)(k / CK::Q) * 8ull + xcd;
  if (item >= a.nitems) return;  // uniform over the workgroup
  const unsigned grp = (unsigned)(item % a.ngroups);
  const unsigned long long o = item / a.ngroups;
  if constexpr (CK::Q == 2) {  // uniform: the part is a compile-time constant inside
    if (k & 1u) {
      col_part<L, 1, INV, WL, WS>(a, o, grp, lds, tws);
      return;
    }
  }
  col_part<L, 0, INV, WL, WS>(a, o, grp, lds, tws);
}

template <int L, bool INV, bool WL, bool WS>
static void launch_colw(const ColArgs& a, hipStream_t s, unsigned blocks) {
  FFTAMD_LAUNCH((k_fft_col<L, INV, WL, WS>), dim3(blocks), dim3(CL_NT), 0, s, a);
}

template <int L, bool INV>
static void launch_coli(const ColArgs& a, hipStream_t s, unsigned blocks) {
  if (a.w_load) {
    if (a.w_store) launch_colw<L, INV, true, true>(a, s, blocks);
    else launch_colw<L, INV, true, false>(a, s, blocks);
  } else {
    if (a.w_store) launch_colw<L, INV, false, true>(a, s, blocks);
    else launch_colw<L, INV, false, false>(a, s, blocks);
  }
}

bool col_supported(int l, long long lx, unsigned long long nouter) {
  // 16-column groups; the group's span (l - 1 rows + 16 columns) addressed with
  // 32-bit byte offsets
  return (l == 4096 || l == 2048) && lx >= CL_C && lx % CL_C == 0 &&
         (unsigned long long)(l - 1) * (unsigned long long)lx * 8ull + CL_C * 8ull < (1ull << 31) && nouter > 0;
}

void preload_col() { preload_kernel(reinterpret_cast<const void*>(&k_fft_col<4096, false, false, false>)); }

int launch_fft_col(const ColArgs& a, void* stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (!col_supported(a.l, a.lx, a.nitems / (a.ngroups ? a.ngroups : 1)) || a.ngroups != (unsigned)(a.lx / CL_C) ||
      a.in_o != (long long)a.l * a.lx)
    return -1;
  // weights: element e of block o has weight index (o * in_o + e) & w_mask,
  // read as ((o * in_o) & w_mask) + e, which needs a period that is a
  // multiple of the block
  if ((a.w_load || a.w_store) && (a.w_mask + 1ull) % (unsigned long long)a.in_o != 0) return -1;
  const unsigned long long items8 = (a.nitems + 7ull) / 8ull * 8ull;
  const unsigned long long blocks = items8 * (unsigned)(a.l / 2048);
  if (blocks > 0xFFFFFFFFull / CL_NT) return -1;
  if (a.l == 4096) {
    if (a.inverse) launch_coli<4096, true>(a, s, (unsigned)blocks);
    else launch_coli<4096, false>(a, s, (unsigned)blocks);
  } else {
    if (a.inverse) launch_coli<2048, true>(a, s, (unsigned)blocks);
    else launch_coli<2048, false>(a, s, (unsigned)blocks);
  }
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace fftamd
