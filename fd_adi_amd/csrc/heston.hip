// Fused, batched Heston ADI engine.
//
// Replaces the per-step operator-call loops of
// FiniteDifferenceEngineGPU.pyx:379-593 (and the CPU-only Craig-Sneyd loops
// of FiniteDifferenceEngine.pyx:778-898) with one launch per ADI stage for a
// whole batch of options with uneven grids.
//
// Layout.  Option k's state is an (nS, nv) row-major block at d_state+off[k]
// (variance contiguous, as the reference's Grid).  No 2-D operator is stored:
// every band of A0 (spot), A1 (variance) and A01 (cross) is generated in the
// kernels from 1-D tables built on the device from the meshes:
//   A0[i,j] band = P(i) + v_j Q(i)                 (mu_S d/dS + 1/2 v S^2 d2/dS2 - r/2)
//   A1[i,j] band = [S_i != 0] G(j) - r/2 on mid    (kappa(theta-v) d/dv + 1/2 sigma^2 v d2/dv2)
//   A01[i,j]     = rho sigma S_i v_j ws(i) x wv(j) (9-point)
// Boundary rows are those of _TriBandedOperatorGPU.cu:203-362: Dirichlet 0
// at S=0 (and at Smax for a barrier), dU/dS=1 at Smax, one-sided first
// derivative at both variance ends, d2/dv2 Von Neumann 0 at v=0 and the
// second-order backward row (with its -2 band entry, folded) at vmax.
//
// Sweeps.  A spot sweep gives each workgroup (option, tile of NL variance
// columns) pairs, one or, for wide tiles, one after another; a variance sweep
// one workgroup per (option, tile of NL spot rows).  The tile's right-hand side is formed (fusing every explicit term of
// the stage) straight into LDS, the NL tridiagonal lines are solved in LDS,
// and the stage output (fusing the next stage's explicit term) is written
// back: one read of each input vector and one write per stage, no
// transposes.  The line solve uses the time-invariant LU factorisation of
// I - theta dt A (built once per configure): each line is split into chunks
// owned by threads, and both triangular sweeps are first-order linear
// recurrences composed across chunks with a wave-level scan of affine maps.
#include "common.h"

#include <algorithm>
#include <numeric>
#include <vector>

namespace fdadi {
namespace {

enum SpotField {
  SP_PSUB, SP_PMID, SP_PSUP, SP_QSUB, SP_QMID, SP_QSUP, SP_PR, SP_QR,
  SP_WSUB, SP_WMID, SP_WSUP, SP_S, SP_NF
};
enum VarField {
  VT_GSUB, VT_GMID, VT_GSUP, VT_WSUB, VT_WMID, VT_WSUP, VT_V, VT_M, VT_RD, VT_N, VT_NF
};

struct HOpt {
  int64_t nS, nv, off;  // grid and state offset
  int64_t so, vo;       // offsets into the spot / variance tables
  double r, kappa, theta, sigma, rho, dt;
  double tdt;           // weight of the implicit part (theta*dt, or dt for implicit)
  double th;            // the scheme's theta
  double fold_f;        // bottom fold factor of I - tdt A1 (lines with S != 0)
  double rdS0;          // 1 / (1 + tdt r/2): the S = 0 variance line
  double Gz;            // A1[nv-1, nv-3] for S != 0
  int32_t barrier, pad;
};

struct Tile {
  int32_t opt;
  int32_t start;  // first column (spot sweep) / first row (variance sweep)
};

enum StageMode {
  // spot sweeps
  SM_FIRST = 0,  // rhs = U + F U - Le0 U;               out = x - Le1 U
  SM_HV = 1,     // rhs = U + F U + 1/2 F^(Y2-U) - Le0 Y2; out = x - Le1 Y2
  SM_CS = 2,     // rhs = U + F U + dt/2 A01 (Y2-U) - Le0 U; out = x - Le1 U
  SM_MCS = 3,    // rhs = U + F U + th dt A01 D + (1/2-th) F D - Le0 U; out = x - Le1 U
  SM_IMPL = 4,   // rhs = W + dt R0;                     out = x
  // variance sweeps
  VM_PLAIN = 10, // rhs = W;                             out = x
  VM_IMPL = 11   // rhs = U + dt A01 U;                  out = x
};

struct Ctx {
  const HOpt *opts;
  const double *sp;  // spot tables, field-major, stride sp_n
  const double *vt;  // variance tables, field-major, stride vt_n
  int64_t sp_n, vt_n;
  const double *rd0;  // spot-line pivots 1/u, state layout
  const double *spr;  // spot table, one 16-double row per node
};

__device__ __forceinline__ double SP(const Ctx &c, const HOpt &o, int f, int64_t i) {
  return c.sp[f * c.sp_n + o.so + i];
}
__device__ __forceinline__ double VT(const Ctx &c, const HOpt &o, int f, int64_t j) {
  return c.vt[f * c.vt_n + o.vo + j];
}

// A0 band entry p + w2 * c00 as the reference's combined operator holds it:
// the (0,) band (with -r/2 on the diagonal) plus the (0,0) weight scaled by
// c00 = (1/2 v) S^2, one rounding each (no fused multiply-add), so that the
// discrete operator is bit-identical to the reference's.
__device__ __forceinline__ double band_add(double p, double w2, double c00) {
#pragma clang fp contract(off)
  const double t = w2 * c00;
  return p + t;
}

__device__ __forceinline__ double c00_of(double v, double S) {
#pragma clang fp contract(off)
  return (0.5 * v) * (S * S);
}

// (A01 x)(i,j): rho sigma S v times the 9-point central product stencil.
template <class F>
__device__ double a01_dot(const Ctx &c, const HOpt &o, int64_t i, int64_t j, F x) {
  if (o.rho == 0.0 || i == 0 || i == o.nS - 1 || j == 0 || j == o.nv - 1) return 0.0;
  const double ws[3] = {SP(c, o, SP_WSUB, i), SP(c, o, SP_WMID, i), SP(c, o, SP_WSUP, i)};
  const double wv[3] = {VT(c, o, VT_WSUB, j), VT(c, o, VT_WMID, j), VT(c, o, VT_WSUP, j)};
  double acc = 0.0;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    double row = wv[0] * x(i + a - 1, j - 1) + wv[1] * x(i + a - 1, j) + wv[2] * x(i + a - 1, j + 1);
    acc += ws[a] * row;
  }
  const double coef = ((o.rho * o.sigma) * SP(c, o, SP_S, i)) * VT(c, o, VT_V, j);
  return coef * acc;
}

// ---- wave-level scans of affine maps ------------------------------------------
// A map y -> E + M y is the pair (M, E); composing "earlier then later" gives
// (M_l M_e, E_l + M_l E_e).  The scans run on DPP lane moves (no LDS round
// trip): row_shr/row_shl within rows of 16 lanes, row_bcast:15/31 across rows
// for prefixes, wave_shr/wave_shl for the exclusive shift.  Lanes with no
// source keep the identity (M, E) = (1, 0).  Every lane of the wave must be
// active.
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_or(double x, double old) {
  const int lo = __builtin_amdgcn_update_dpp(__double2loint(old), __double2loint(x), CTRL, ROWS,
                                             0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(__double2hiint(old), __double2hiint(x), CTRL, ROWS,
                                             0xF, false);
  return __hiloint2double(hi, lo);
}

// One prefix level: combine with the map of lane ln - D (ln = lane within a
// segment of W lanes); the DPP control already fetches from lane - D.
template <int CTRL, int ROWS, int D, int W>
__device__ __forceinline__ void prefix_level(double &M, double &E, int ln) {
  double Mp = dpp_or<CTRL, ROWS>(M, 1.0), Ep = dpp_or<CTRL, ROWS>(E, 0.0);
  if (W < 16 && ln < D) {
    Mp = 1.0;
    Ep = 0.0;
  }
  E = E + M * Ep;
  M = M * Mp;
}

// Inclusive prefix scan over segments of W lanes (W a power of two <= 64).
template <int W>
__device__ __forceinline__ void wave_prefix_scan(double &M, double &E, int ln) {
  if (W > 1) prefix_level<0x111, 0xF, 1, W>(M, E, ln);
  if (W > 2) prefix_level<0x112, 0xF, 2, W>(M, E, ln);
  if (W > 4) prefix_level<0x114, 0xF, 4, W>(M, E, ln);
  if (W > 8) prefix_level<0x118, 0xF, 8, W>(M, E, ln);
  if (W > 16) prefix_level<0x142, 0xA, 16, W>(M, E, ln);  // row_bcast:15 into rows 1, 3
  if (W > 32) prefix_level<0x143, 0xC, 32, W>(M, E, ln);  // row_bcast:31 into rows 2, 3
}

// Inclusive suffix scan over segments of W lanes: maps of higher lanes are
// applied first.  Within rows by DPP row_shl (after those levels a lane holds
// the maps from itself to the end of its row).  Across rows, mirroring
// row_bcast of the prefix scan: at D = 16 rows 0 and 2 take the first lane of
// the next row (which holds that whole row), at D = 32 rows 0 and 1 take lane
// 32 (which then holds rows 2-3); by ds_bpermute.
template <int CTRL, int D, int W>
__device__ __forceinline__ void suffix_level(double &M, double &E, int ln) {
  double Mn, En;
  bool take;
  if (D < 16) {
    Mn = dpp_or<CTRL, 0xF>(M, 1.0);
    En = dpp_or<CTRL, 0xF>(E, 0.0);
    take = ln + D < W;
  } else {
    const int lane = threadIdx.x % 64;
    const int src = D == 16 ? (lane | 15) + 1 : 32;
    Mn = __shfl(M, src & 63, 64);
    En = __shfl(E, src & 63, 64);
    take = D == 16 ? ((lane >> 4) & 1) == 0 : lane < 32;
  }
  if (!take) {
    Mn = 1.0;
    En = 0.0;
  }
  E = E + M * En;
  M = M * Mn;
}

template <int W>
__device__ __forceinline__ void wave_suffix_scan(double &M, double &E, int ln) {
  if (W > 1) suffix_level<0x101, 1, W>(M, E, ln);
  if (W > 2) suffix_level<0x102, 2, W>(M, E, ln);
  if (W > 4) suffix_level<0x104, 4, W>(M, E, ln);
  if (W > 8) suffix_level<0x108, 8, W>(M, E, ln);
  if (W > 16) suffix_level<0, 16, W>(M, E, ln);
  if (W > 32) suffix_level<0, 32, W>(M, E, ln);
}

// Value of lane ln - 1 of the segment (0 for its first lane).
template <int W>
__device__ __forceinline__ double from_prev_lane(double x, int ln) {
  const double v = dpp_or<0x138, 0xF>(x, 0.0);  // wave_shr:1
  return ln == 0 ? 0.0 : v;
}

// Value of lane ln + 1 of the segment (0 for its last lane).
template <int W>
__device__ __forceinline__ double from_next_lane(double x, int ln) {
  const double v = dpp_or<0x130, 0xF>(x, 0.0);  // wave_shl:1
  return ln == W - 1 ? 0.0 : v;
}

// Exclusive scan of affine maps y -> E + M y along the TPL chunks of each of
// the NL lines of a tile.  Entries live in LDS at [l*(TPL+1) + c] (line by
// line, odd pitch: the lanes of a line read consecutive entries and the
// writers of one chunk hit distinct banks).  Forward
// (REV=false): carry(0)=0, carry(c+1)=E[c]+M[c]*carry(c).  Backward
// (REV=true): the same from the last chunk down.  A line takes W = min(TPL,
// 64) lanes (K = TPL / W entries per lane), so a wave scans 64 / W lines at
// once with segmented scans.
template <int THREADS, int NL, bool REV>
__device__ void affine_scan(const double *cM, const double *cE, double *cIn) {
  constexpr int TPL = THREADS / NL;
  constexpr int TPLP = TPL + 1;
  constexpr int W = TPL < 64 ? TPL : 64;
  constexpr int K = TPL / W;
  constexpr int LPW = 64 / W;
  constexpr int NW = THREADS / 64;
  static_assert(W >= 16 && (W & (W - 1)) == 0, "16 to 64 lanes per line");
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  const int ln = lane % W;
  for (int l0 = wave * LPW; l0 < NL; l0 += NW * LPW) {
    const int l = l0 + lane / W;
    const bool ok = l < NL;
    // Compose this lane's K entries (in scan order).
    double Mloc = 1.0, Eloc = 0.0;
#pragma unroll
    for (int q = 0; q < K; ++q) {
      const int s = ln * K + q;
      const int cidx = REV ? TPL - 1 - s : s;
      const double m = ok ? cM[l * TPLP + cidx] : 1.0, e = ok ? cE[l * TPLP + cidx] : 0.0;
      Eloc = e + m * Eloc;
      Mloc = m * Mloc;
    }
    // Inclusive segmented scan of (M, E) (later maps applied after earlier ones).
    double M = Mloc, E = Eloc;
    wave_prefix_scan<W>(M, E, ln);
    // Exclusive: the carry entering this lane's first entry.
    double carry = from_prev_lane<W>(E, ln);
#pragma unroll
    for (int q = 0; q < K; ++q) {
      const int s = ln * K + q;
      const int cidx = REV ? TPL - 1 - s : s;
      if (ok) {
        cIn[l * TPLP + cidx] = carry;
        carry = cE[l * TPLP + cidx] + cM[l * TPLP + cidx] * carry;
      }
    }
  }
}

// The same for four-column tiles without a scan through LDS: the value entering
// this thread's chunk of its line, given the chunk's map y -> E + M y and 0
// entering the line's first chunk (REV: its last; the maps are applied from
// the last chunk down).  A wave holds 16 chunks of each line, lane = chunk * 4
// + line: it scans them across lanes, leaves the map of all of them in
// tot[waves][4], and after one barrier composes the carry entering the wave
// from the waves before it.  One barrier instead of three: a single option is
// bound by latency, and its solve runs on four-column tiles.  Calls that
// follow one another without a barrier in between use different `tot`s.
template <int CTRL>
__device__ __forceinline__ void map_level(double &M, double &E) {
  const double Mp = dpp_or<CTRL, 0xF>(M, 1.0), Ep = dpp_or<CTRL, 0xF>(E, 0.0);
  E = E + M * Ep;
  M = M * Mp;
}
__device__ __forceinline__ void map_level_from(double &M, double &E, int src, bool take) {
  const double Mp = __shfl(M, src, 64), Ep = __shfl(E, src, 64);
  E = take ? E + M * Ep : E;
  M = take ? M * Mp : M;
}

template <int THREADS, bool REV>
__device__ __forceinline__ double quad_carry(double M, double E, double2 *tot) {
  constexpr int NW = THREADS / 64;
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64, line = lane % 4, row = lane / 16;
  // inclusive scan over the wave's chunks: within rows of 16 lanes by DPP
  // (row_shl / row_shr by 4 and 8 lanes), then across rows from a row's last
  // chunk in scan order
  map_level<REV ? 0x104 : 0x114>(M, E);
  map_level<REV ? 0x108 : 0x118>(M, E);
  const int end = REV ? line : 12 + line;
  map_level_from(M, E, (REV ? row | 1 : row & ~1) * 16 + end, (row & 1) == (REV ? 0 : 1));
  map_level_from(M, E, (REV ? 32 : 16) + end, REV ? row < 2 : row >= 2);
  const bool first = REV ? lane >= 60 : lane < 4;
  if (REV ? lane < 4 : lane >= 60) tot[wave * 4 + line] = make_double2(M, E);
  // the map of the chunks before this one
  const int prev = (REV ? lane + 4 : lane - 4) & 63;
  const double Mp = __shfl(M, prev, 64), Ep = __shfl(E, prev, 64);
  __syncthreads();
  double c = 0.0;
#pragma unroll
  for (int q = 0; q < NW - 1; ++q) {
    const int w = REV ? NW - 1 - q : q;
    if (REV ? w > wave : w < wave) {
      const double2 t = tot[w * 4 + line];
      c = t.y + t.x * c;
    }
  }
  return first ? c : Ep + Mp * c;
}

// ---- spot sweep ---------------------------------------------------------------
// One 128-byte row of per-node spot coefficients, built from the spot table
// with the boundary handling folded in:
// [psub' pmid psup' qsub' | qmid qsup' pr qr | S*wsub S*wmid S*wsup S^2 | (padding)]
// (p*: first-derivative bands scaled by r S, with -r/2 on the diagonal; q*:
// raw second-derivative weights, and qr the raw residual, to be scaled by
// c00 = (1/2 v) S^2 in the kernel) where ' marks band entries zeroed when
// they multiply a Dirichlet neighbour (row 0 for row 1; row nS-1 for row nS-2
// under a barrier) -- the explicit apply forces those neighbours to 0, and in
// the solve the coupling to a Dirichlet row (whose value is 0) contributes
// nothing.  Dirichlet rows have all-zero bands, so row 0 has no use for S^2 and
// holds [S != 0] there (the spot mesh increases strictly from S >= 0, so only
// row 0 can have S = 0; S^2 itself is 0 already for S below 1e-162).
constexpr int kSpRow = 16;
constexpr int kSpFields = 12;

struct SpotRow {
  double psub, pmid, psup, qsub, qmid, qsup, pr, qr, wsub, wmid, wsup, S2;
};

// A1 on one variance column scaled by a step weight c (c = dt for the
// explicit operator dt A1, c = theta dt for theta dt A1): the entries the
// reference's scaled operator holds, fl(c * a), for lines with S != 0 (sub,
// mid, sup and, on the last column, z = the j-2 entry of the second-order
// backward row) and the diagonal c * (-r/2) of the S = 0 line.
struct ColOp {
  double sub, mid, sup, z, s0;
};

struct VarCol {  // variance coefficients of column j (constant along a spot line)
  double wv0, wv1, wv2;
  double c0h;     // v / 2 (c00 = c0h S^2)
  double rsv;     // rho * sigma * v
  ColOp f1, t1;   // dt A1 and theta dt A1 on this column
};

// A0 bands of row i at variance v (Dirichlet handling is in the bands).
struct Bands {
  double sub, mid, sup, r0;
};

// A0 band entry p + w2 * c00 with c00 = (1/2 v) S^2, one rounding each.
__device__ __forceinline__ Bands a0_bands(const SpotRow &R, double c0h) {
#pragma clang fp contract(off)
  const double c00 = c0h * R.S2;
  Bands b;
  b.sub = band_add(R.psub, R.qsub, c00);
  b.mid = band_add(R.pmid, R.qmid, c00);
  b.sup = band_add(R.psup, R.qsup, c00);
  b.r0 = band_add(R.pr, R.qr, c00);  // residual: zero except on the Smax row
  return b;
}

__device__ __forceinline__ ColOp col_op(double c, double gsub, double gmid, double gsup,
                                        double gz, double split) {
  return ColOp{c * gsub, c * gmid, c * gsup, c * gz, c * split};
}

// A state row at this lane's column j: columns j-1, j, j+1 (clamped to the
// grid).
struct Row3 {
  double l, c, r;
};

// This lane's columns of a tile, as byte offsets within a state row.
struct LaneCols {
  unsigned jcb, jxb;  // column j and the edge column, clamped to the grid
  bool last, ok;      // j is the grid's last column (or clamped to it) / inside the grid
};

// A row as loaded for the window: column j and this lane's edge column jx
// (j - 1 on the tile's first lane, j + 1 on its last, j elsewhere).  The
// inner neighbours come from the adjacent lanes, which hold exactly those
// columns (a lane past the grid's last column loads that column, the clamped
// j + 1 of the last one); column j - 2 of the grid's last column comes from
// the lane two before it (the tile list puts the last column on a tile's last
// lane).
struct Raw2 {
  double e, c;
};

// An option's state (or pivots) as a buffer of nS * nv doubles addressed by
// 32-bit byte offsets: a read past it (also at a negative offset, which wraps
// far beyond its end) gives 0 and a store past it is dropped, so rows outside
// the grid need no clamping and no lane masks.
using Buf = __amdgpu_buffer_rsrc_t;
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ Buf buf_of(const double *p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<double *>(p), 0, (int)bytes, 0x00027000);
}
__device__ __forceinline__ double buf_load(Buf b, unsigned off) {
  const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(b, (int)off, 0, 0);
  return __hiloint2double((int)v.y, (int)v.x);
}
__device__ __forceinline__ void buf_store(Buf b, unsigned off, double x) {
  const u32x2 v = {(unsigned)__double2loint(x), (unsigned)__double2hiint(x)};
  __builtin_amdgcn_raw_buffer_store_b64(v, b, (int)off, 0, 0);
}

// The row at byte offset rowb (row * nv * 8).
__device__ __forceinline__ Raw2 load_raw2(Buf f, unsigned rowb, const LaneCols &lc) {
  return Raw2{buf_load(f, rowb + lc.jxb), buf_load(f, rowb + lc.jcb)};
}

// 16 bytes per lane from `src` into LDS at dst + 16 * lane (dst uniform over
// the wave), without passing through registers; lds_loads_done() waits for
// this wave's, a barrier after it for everyone's.
__device__ __forceinline__ void load_lds16(const double *src, double *dst) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)src,
                                   (__attribute__((address_space(3))) void *)dst, 16, 0, 0);
}
__device__ __forceinline__ void lds_loads_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Value of the lane before / after / two before within the tile's lanes
// (quad_perm for four columns; row_shr / row_shl within a DPP row of 16
// lanes for 8 and 16; wave_shr / wave_shl across the two DPP rows of a
// 32-column tile; the tile's first and last lanes use their edge load).  Two
// before serves the last column only, which sits on the tile's last lane
// (lane 31 of a 32-column tile, nv >= 32), so row_shr:2 stays in its row.
template <int CTRL>
__device__ __forceinline__ double dpp_mov(double x) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), CTRL, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}
template <int NL>
__device__ __forceinline__ double from_prev_col(double x) {
  // quad_perm [0,0,1,2] / row_shr:1 / wave_shr:1
  return dpp_mov<NL == 4 ? 0x90 : (NL == 32 ? 0x138 : 0x111)>(x);
}
template <int NL>
__device__ __forceinline__ double from_next_col(double x) {
  // quad_perm [1,2,3,3] / row_shl:1 / wave_shl:1
  return dpp_mov<NL == 4 ? 0xF9 : (NL == 32 ? 0x130 : 0x101)>(x);
}
template <int NL>
__device__ __forceinline__ double from_prev2_col(double x) {
  return dpp_mov<NL == 4 ? 0x40 : 0x112>(x);  // quad_perm [0,0,0,1] / row_shr:2
}

template <int NL>
__device__ __forceinline__ Row3 expand_raw(const Raw2 &w, int jj) {
  if constexpr (NL == 16) {
    // a DPP row of 16 lanes is the tile: its first and last lanes, which have
    // no source lane for row_shr:1 / row_shl:1, keep the edge load
    return Row3{dpp_or<0x111, 0xF>(w.c, w.e), w.c, dpp_or<0x101, 0xF>(w.c, w.e)};
  } else {
    const double l = from_prev_col<NL>(w.c), r = from_next_col<NL>(w.c);
    return Row3{jj == 0 ? w.e : l, w.c, jj == NL - 1 ? w.e : r};
  }
}

// (c A1 f)(i,j) with the scaled entries K of this column over row i of f; on
// the tile with the grid's last column (ends, the same for every lane) that
// column adds its j - 2 entry.
template <int NL>
__device__ __forceinline__ double a1s(const ColOp &K, const Row3 &w, bool ends, bool last) {
  double v = (K.sup * w.r + K.mid * w.c) + K.sub * w.l;
  if (ends) {
    const double m2 = from_prev2_col<NL>(w.c);
    v = last ? v + K.z * m2 : v;
  }
  return v;
}

// What the sliding window keeps of a row once it has entered: the value at
// column j and the row's share of the cross product, wv . (x_{j-1}, x_j,
// x_{j+1}), of U and of D = Y - U, Y at column j, and the A1 products the
// stage takes at this row (dt A1 U, theta dt A1 U, dt A1 D, theta dt A1 Y).
// Each is formed once per row, when the row enters.
struct WinRow {
  double uc, urs, dc, drs, yc;
  double f1u, t1u, f1d, t1y;
};

// (wv . (l, c, r), every operation written out: a rounding that differs here
// differs in every later step, and the trained surrogates and their gate
// thresholds follow the labels' last bits.  For the same reason the two rows
// before a chunk's walk, `first`, keep the order of the fused operations they
// have always had.)
__device__ __forceinline__ double row_share(const VarCol &q, const Row3 &w, bool first) {
  const double t = first ? __builtin_fma(q.wv0, w.l, q.wv1 * w.c) : __builtin_fma(q.wv1, w.c, q.wv0 * w.l);
  return __builtin_fma(q.wv2, w.r, t);
}

template <int MODE, int NL, bool HALF, bool FIRST>
__device__ __forceinline__ void enter_row(const VarCol &q, const Row3 &u, const Row3 &y, bool ends,
                                          bool last, WinRow &w) {
  constexpr bool HAS_Y = MODE == SM_HV || MODE == SM_CS || MODE == SM_MCS;
  w.uc = u.c;
  if constexpr (MODE != SM_IMPL) {
    w.urs = row_share(q, u, FIRST);
    w.f1u = a1s<NL>(q.f1, u, ends, last);
  }
  if constexpr (!HALF && (MODE == SM_FIRST || MODE == SM_CS || MODE == SM_MCS))
    w.t1u = a1s<NL>(q.t1, u, ends, last);
  if constexpr (HAS_Y) {
    const Row3 d{y.l - u.l, y.c - u.c, y.r - u.r};
    w.dc = d.c;
    w.drs = row_share(q, d, FIRST);
    w.yc = y.c;
    if constexpr (MODE == SM_HV || MODE == SM_MCS) w.f1d = a1s<NL>(q.f1, d, ends, last);
    if constexpr (MODE == SM_HV) w.t1y = a1s<NL>(HALF ? q.f1 : q.t1, y, ends, last);
  }
}

// The S = 0 line (row 0 when the spot mesh starts at 0): A1 keeps only the
// -r/2 of the split, c * (-r/2) * f(i, j).
template <int MODE, bool HALF>
__device__ __forceinline__ void zero_line(const VarCol &q, WinRow &w) {
  if constexpr (MODE != SM_IMPL) w.f1u = q.f1.s0 * w.uc;
  if constexpr (!HALF && (MODE == SM_FIRST || MODE == SM_CS || MODE == SM_MCS)) w.t1u = q.t1.s0 * w.uc;
  if constexpr (MODE == SM_HV || MODE == SM_MCS) w.f1d = q.f1.s0 * w.dc;
  if constexpr (MODE == SM_HV) w.t1y = (HALF ? q.f1.s0 : q.t1.s0) * w.yc;
}

// Work-group index -> tile index so that consecutive tiles (which share cache
// lines of the state) run on the same XCD: dispatch places work-group k on
// XCD k mod 8.
__device__ __forceinline__ int xcd_tile(int k, int G) {
  const int q = G / 8, rem = G % 8, x = k % 8, y = k / 8;
  return x * q + (x < rem ? x : rem) + y;
}

// Broadcast lane Q of each group of four lanes (DPP quad_perm [Q,Q,Q,Q]).
template <int Q>
__device__ __forceinline__ double quad_bcast(double x) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), Q * 0x55, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), Q * 0x55, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}

// Four-column tiles: the quad's lanes share a table row; lane jj of the quad
// loads doubles [4jj, 4jj+4) (two 16-byte loads) and the fields are broadcast
// (every lane of the quad must execute quad_row_fields).
__device__ __forceinline__ void quad_row_load(const double *__restrict__ spr, int jj, double2 &a,
                                              double2 &b) {
  const double2 *p = reinterpret_cast<const double2 *>(spr + 4 * jj);
  a = p[0];
  b = p[1];
}

__device__ __forceinline__ SpotRow quad_row_fields(double2 a, double2 b) {
  SpotRow r;
  r.psub = quad_bcast<0>(a.x); r.pmid = quad_bcast<0>(a.y);
  r.psup = quad_bcast<0>(b.x); r.qsub = quad_bcast<0>(b.y);
  r.qmid = quad_bcast<1>(a.x); r.qsup = quad_bcast<1>(a.y);
  r.pr = quad_bcast<1>(b.x);   r.qr = quad_bcast<1>(b.y);
  r.wsub = quad_bcast<2>(a.x); r.wmid = quad_bcast<2>(a.y);
  r.wsup = quad_bcast<2>(b.x); r.S2 = quad_bcast<2>(b.y);
  return r;
}

// Wider tiles (8 to 32 columns): the work-group holds the table rows its chunks
// read in LDS, chunk by chunk (MAXL rows of 12 fields), and each lane reads
// its row with six 16-byte LDS loads (the lanes of a chunk read the same
// address).
__device__ __forceinline__ SpotRow lds_row_fields(const double *__restrict__ p) {
  const double2 *q = reinterpret_cast<const double2 *>(p);
  const double2 a = q[0], b = q[1], c = q[2], d = q[3], e = q[4], f = q[5];
  return SpotRow{a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y, e.x, e.y, f.x, f.y};
}

// An empty asm that reads x: x has to be computed before this point.  The
// row walk keeps its results in registers (no store orders it), so without
// these fences the compiler hoists every row's loads to the top of the
// unrolled walk and runs out of registers.
__device__ __forceinline__ void pin(double x) { asm volatile("" ::"v"(x)); }

// A spot sweep: tiles of (option, NL adjacent variance columns), NL = 4, 8, 16
// or 32; thread (jj, ch) = (tid % NL, tid / NL) owns rows
// [ch*L, ch*L+L) of column j0+jj through every phase.  The NL lanes of a
// chunk work on the same rows, so they share the spot-table rows.  Four
// columns per tile keep a large grid spread over every CU (2048 x 1024: 256
// tiles); wider tiles make each load of a wave touch fewer, longer row
// segments, which pays where the batch has tiles to spare.
//
// Wide tiles: a work-group takes tile after tile of its XCD's share, and all
// that a tile waits for is loaded while the tile before it finishes -- its
// first state rows by the walk's own ring of loads once that tile needs no
// more rows, its other first values after the walk, its table rows from memory
// straight into LDS between the scans, its option's record a tile earlier.
// Before this every tile was a work-group of its own and spent half its life
// (11,400 of 23,800 cycles on a 256 x 128 grid) on that chain of dependent
// loads with the CU's other work-group as its only cover.  Neighbouring tiles
// run side by side on one XCD because each row of a tile also touches the
// lines of the tiles beside it: walking along an option instead (eight tiles
// in a row) tripled the bytes fetched and was slower.  On 4,096 such grids the
// first stage went from 811 to 608 us, the Craig-Sneyd second stage from 973
// to 810 us (one 512-thread work-group per CU on 32 columns).  They move 2.4 and
// 3.7 GB, 4.0 and 4.6 TB/s, in row segments of 128 to 256 bytes; the variance
// stage, whose rows are whole, reaches 5.6 TB/s, and 256 such grids, whose
// vectors the last-level cache nearly holds, take as long for each, so it is
// the access pattern rather than HBM that they wait for.  A variant with 66
// instead of 80 VALU instructions a point gained 3%, more rows in flight
// nothing, and lines touched a tile ahead are evicted from the 4 MB L2 before
// they are used.
// Four-column tiles (few tiles, a work-group each) keep the one-tile form.
//
// With theta = 1/2 every entry of theta dt A is half the entry of dt A, exactly,
// so one set of products serves both (HALF): the same bits, and 1 to 5% less
// time on wide tiles.  Other thetas take the general form.  (Both stand in one
// kernel, chosen by the option's record: a captured graph stays valid when
// theta changes.)
//
// The row walk keeps a window of three rows (i-1, i, i+1) of what the stage
// needs from U and Y2, the loads of rows i+2 and i+3 in flight, and forms the
// fused right-hand side (and the next stage's explicit term) of row i.  Rows
// outside the grid read as 0; rows past the chunk are computed and discarded.
//
// The LU solve is run in scaled form: with pivots rd = 1/u, multipliers
// mu_i = -a_i rd_i and n_i = -c_i rd_i, the forward sweep computes
// y'_i = rd_i d_i + mu_i y'_{i-1} (= rd_i y_i) and the backward sweep
// x_i = y'_i + n_i x_{i+1}, so the pivots are needed only while the
// right-hand side is formed.  The pivots rd_i = 1 / (b_i - (a_i rd_{i-1})
// c_{i-1}) are recomputed down the chunk from the stored pivot of the row
// before it (the recurrence the factorisation ran).  mu, n and y' (then x)
// stay in registers; LDS holds the next stage's explicit term (thread-private
// slots [k*THREADS + tid]), the chunk carries of the scans and, for wide
// tiles, the table rows.
//
// Rows k >= L of a chunk belong to the next chunk: the uniform guard k < L
// keeps them out of both chunk maps.  In the last chunk, rows past the grid
// (i >= nS) have finite values and follow row nS - 1, whose super-diagonal is
// zero (n = 0), so they do not reach any valid row either way.

// An option's record as the lanes of a wave hold it (lane l: its l-th 8-byte
// word), loaded a tile ahead with a vector load -- a scalar load in flight
// would make every LDS read of the walk wait for it -- and read out with
// v_readlane.
static_assert(sizeof(HOpt) == 17 * 8, "OptWords names HOpt's words");
struct OptWords {
  double w;
  __device__ __forceinline__ void load(const HOpt *o) {
    const int l = threadIdx.x % 64;
    w = reinterpret_cast<const double *>(o)[l < 16 ? l : 16];
  }
  __device__ __forceinline__ int lo(int k) const {
    return __builtin_amdgcn_readlane(__double2loint(w), k);
  }
  __device__ __forceinline__ double f(int k) const {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(w), k), lo(k));
  }
  __device__ __forceinline__ int64_t i(int k) const {
    return (int64_t)(((uint64_t)(uint32_t)__builtin_amdgcn_readlane(__double2hiint(w), k) << 32) |
                     (uint32_t)lo(k));
  }
  __device__ __forceinline__ int nS() const { return lo(0); }
  __device__ __forceinline__ int nv() const { return lo(1); }
  __device__ __forceinline__ int64_t off() const { return i(2); }
  __device__ __forceinline__ int64_t so() const { return i(3); }
  __device__ __forceinline__ int64_t vo() const { return i(4); }
  __device__ __forceinline__ double r() const { return f(5); }
  __device__ __forceinline__ double rho_sigma() const { return f(9) * f(8); }
  __device__ __forceinline__ double dt() const { return f(10); }
  __device__ __forceinline__ double tdt() const { return f(11); }
  __device__ __forceinline__ double th() const { return f(12); }
  __device__ __forceinline__ double Gz() const { return f(15); }
  __device__ __forceinline__ bool barrier() const { return lo(16) != 0; }
};

template <int MODE, int THREADS, int NL, int MAXL, bool HALF>
__device__ __forceinline__ void spot_tiles(const Ctx &c, const Tile *__restrict__ tiles,
                                           int ntiles, OptWords ow, int start,
                                           const double *__restrict__ U,
                                           const double *__restrict__ Y,
                                           double *__restrict__ out, double *lds) {
  static_assert(NL == 4 || NL == 8 || NL == 16 || NL == 32,
                "spot tiles are 4, 8, 16 or 32 columns wide");
  constexpr int TPL = THREADS / NL;
  constexpr bool HAS_Y = MODE == SM_HV || MODE == SM_CS || MODE == SM_MCS;
  constexpr bool HAS_EX = MODE != SM_IMPL;
  constexpr bool TAB_LDS = NL != 4;
  constexpr bool RUNS = NL != 4;  // several tiles per work-group
  constexpr int CHP = MAXL * kSpFields;  // LDS table: doubles per chunk
  // state rows in flight (two for the second-stage modes on long chunks,
  // whose window and registers are largest)
  constexpr int PF = HAS_Y && MAXL == 16 ? 2 : 4;
  static_assert(MAXL % PF == 0, "the ring's slots line up from tile to tile");
  // the chunk carries (four-column tiles: the wave totals of the two scans),
  // then the next stage's explicit term, slot [k * THREADS + tid], and the
  // table rows
  double *cM = lds, *cE = cM + NL * (TPL + 1), *cIn = cE + NL * (TPL + 1);
  double2 *tot_f = reinterpret_cast<double2 *>(lds), *tot_b = tot_f + THREADS / 64 * 4;
  double *eb = lds + (NL == 4 ? THREADS / 4 : 3 * NL * (TPL + 1));
  double *tab = eb + (HAS_EX ? MAXL * THREADS : 0);  // 16-byte aligned
  const int tid = threadIdx.x;
  const int jj = tid % NL, ch = tid / NL;

  // A tile's geometry: its option's rows as byte offsets (nS <= 2048 and
  // nv <= 1024 keep them far below 2^31), this lane's columns and its chunk of
  // L rows from s on.  The grid's last tile ends on the last column
  // (build_spot_tiles).
  struct Geom {
    unsigned rstep, nbytes;
    int nS, L, s;
    LaneCols lc;
    bool ends;  // the tile holds the grid's last column
    Buf u, y2;
  };
  auto geom_of = [&](const OptWords &w, int j0) {
    Geom g;
    const int nv = w.nv();
    g.nS = w.nS();
    g.rstep = (unsigned)nv * 8u;
    g.nbytes = (unsigned)g.nS * g.rstep;
    g.L = (g.nS + TPL - 1) / TPL;
    g.s = ch * g.L;
    const int j = j0 + jj;
    const int jc = j < nv ? j : nv - 1;  // clamped column for loads
    const int jm = jc > 0 ? jc - 1 : 0, jp = jc < nv - 1 ? jc + 1 : jc;
    const int jx = jj == 0 ? jm : (jj == NL - 1 ? jp : jc);
    g.lc = LaneCols{(unsigned)jc * 8u, (unsigned)jx * 8u, jc == nv - 1, j < nv};
    g.ends = j0 + NL >= nv;
    g.u = buf_of(U + w.off(), g.nbytes);
    g.y2 = buf_of((HAS_Y ? Y : U) + w.off(), g.nbytes);
    return g;
  };

  // What a tile needs before its walk starts, loaded while the tile before it
  // finishes: rows s-1 and s of the window, rows s+1 .. s+PF in flight (row
  // s+1+m in ring slot m % PF), the pivot of row s-1, the column's variance
  // coefficients and the option's spot-table rows.
  Raw2 ru[PF], ry[PF], ua, ub, ya, yb;
  double rdraw, vtab[7];
  ya = yb = Raw2{0.0, 0.0};
  auto load_head = [&](const Geom &g, const OptWords &w) {
    const unsigned rb = (unsigned)g.s * g.rstep, ra = rb - g.rstep;
    ua = load_raw2(g.u, ra, g.lc);
    ub = load_raw2(g.u, rb, g.lc);
    if constexpr (HAS_Y) {
      ya = load_raw2(g.y2, ra, g.lc);
      yb = load_raw2(g.y2, rb, g.lc);
    }
    rdraw = buf_load(buf_of(c.rd0 + w.off(), g.nbytes), ra + g.lc.jcb);
    const char *vt = reinterpret_cast<const char *>(c.vt + w.vo()) + g.lc.jcb;
#pragma unroll
    for (int f = 0; f < 7; ++f)
      vtab[f] = *reinterpret_cast<const double *>(vt + (int64_t)f * c.vt_n * 8);
  };
  static_assert(VT_GSUB == 0 && VT_V == 6, "vtab holds the first seven variance fields");
  // table rows of every chunk, straight from memory into LDS: 16-byte unit e of
  // the table is fields 2 (e % 6), 2 (e % 6) + 1 of row slot e / 6 (rows past
  // the grid repeat the last one, whose results are discarded)
  constexpr int UNITS = TPL * MAXL * kSpFields / 2;
  static_assert(!TAB_LDS || UNITS % 64 == 0, "whole waves of table units");
  // Left to itself the compiler keeps the units' places (12 on 8-column tiles) in
  // registers throughout the walk, which then spills where chunks are long (up
  // to 70 registers: the second stages of HV and MCS on 512 grids of 512 x 128 in
  // 8-column tiles took 450 us, 341 now; 425 and 420 with one tile per
  // work-group).  There they are formed anew for each tile; where they fit they
  // stay (3 VALU instructions a point less on 32 columns, 0.3% of a solve).
  constexpr bool PLACES_FIT = MAXL == 8 || (NL == 32 ? MODE != SM_HV : NL == 16 && !HAS_Y);
  auto load_table = [&](const Geom &g, const OptWords &w) {
    const double *spr = c.spr + w.so() * kSpRow;
    int tq = tid;
    if constexpr (!PLACES_FIT) asm volatile("" : "+v"(tq));
    const int wave0 = __builtin_amdgcn_readfirstlane(tid / 64 * 64);
#pragma unroll
    for (int e0 = 0; e0 < UNITS; e0 += THREADS) {
      if (UNITS % THREADS == 0 || e0 + wave0 < UNITS) {
        const int e = e0 + tq, slot = e / 6, part = e % 6;
        const int r = (slot / MAXL) * g.L + slot % MAXL;
        load_lds16(spr + (unsigned)((r < g.nS ? r : g.nS - 1) * kSpRow + part * 2),
                   tab + 2 * (e0 + wave0));
      }
    }
  };
  const double *tch = tab + ch * CHP;

  // The work-group's tiles: every `step`-th of its XCD's share of the list
  // (dispatch places work-group b on XCD b mod 8; tiles next to each other
  // share cache lines of the state, so they run side by side on one XCD).
  const int xcd = blockIdx.x % 8, step = ((int)gridDim.x - xcd + 7) / 8;
  const int share = ntiles / 8 + (xcd < ntiles % 8 ? 1 : 0);
  const Tile *mine = tiles + xcd * (ntiles / 8) + (xcd < ntiles % 8 ? xcd : ntiles % 8);
  int at = blockIdx.x / 8;
  int lane_zero = 0;  // makes the address per-lane, so that the load is a vector load
  asm volatile("" : "+v"(lane_zero));
  auto load_tile = [&](int k) { return mine[(k < share ? k : share - 1) + lane_zero]; };
  // the tile after this one and its option; the one after that
  Tile t1{0, 0}, t2{0, 0};
  OptWords on = ow;
  int start_n = start;
  if constexpr (RUNS) {
    t1 = load_tile(at + step);
    t2 = load_tile(at + 2 * step);
  }

  Geom g = geom_of(ow, start);
  if constexpr (TAB_LDS) load_table(g, ow);
  load_head(g, ow);
#pragma unroll
  for (int m = 0; m < PF; ++m) {
    const unsigned rr = (unsigned)(g.s + 1 + m) * g.rstep;
    ru[m] = load_raw2(g.u, rr, g.lc);
    ry[m] = Raw2{0.0, 0.0};
    if constexpr (HAS_Y) ry[m] = load_raw2(g.y2, rr, g.lc);
  }
  if constexpr (RUNS) {
    on.load(c.opts + __builtin_amdgcn_readfirstlane(t1.opt));
    start_n = __builtin_amdgcn_readfirstlane(t1.start);
  }
  if constexpr (TAB_LDS) {
    lds_loads_done();
    __syncthreads();
  }

  for (;;) {
    const bool more = RUNS && at + step < share;
    const int nS = g.nS, L = g.L, s = g.s;
    const unsigned rstep = g.rstep;
    const LaneCols lc = g.lc;
    const Buf u = g.u, y2 = g.y2;
    const double tdt = ow.tdt(), dt = ow.dt();
    const double *spr = c.spr + ow.so() * kSpRow;
    auto clamp_row = [&](int i) { return (unsigned)(i < 0 ? 0 : (i >= nS ? nS - 1 : i)); };
    VarCol q;
    {
      q.wv0 = vtab[VT_WSUB]; q.wv1 = vtab[VT_WMID]; q.wv2 = vtab[VT_WSUP];
      q.c0h = 0.5 * vtab[VT_V];
      q.rsv = ow.rho_sigma() * vtab[VT_V];
      const double gz = lc.last ? ow.Gz() : 0.0, split = -ow.r() / 2.0;
      q.f1 = col_op(dt, vtab[VT_GSUB], vtab[VT_GMID], vtab[VT_GSUP], gz, split);
      if constexpr (!HALF)
        q.t1 = col_op(tdt, vtab[VT_GSUB], vtab[VT_GMID], vtab[VT_GSUP], gz, split);
    }
    // four-column tiles: table rows i and i+1 in flight
    double2 ta0, tb0, ta1, tb1;
    if constexpr (!TAB_LDS) {
      quad_row_load(spr + clamp_row(s) * kSpRow, jj, ta0, tb0);
      quad_row_load(spr + clamp_row(s + 1) * kSpRow, jj, ta1, tb1);
    }
    // Pivot recurrence state from the row before the chunk.
    double rdp = 0.0, cp = 0.0;
    if (s > 0) {
      const double *pr =
          TAB_LDS ? tch - CHP + (L - 1) * kSpFields : spr + clamp_row(s - 1) * kSpRow;
      const double c00 = q.c0h * pr[11];
      rdp = rdraw;
      cp = -tdt * band_add(pr[2], pr[5], c00);
    }
    WinRow wa, wb, wc;
    const bool ends = g.ends;
    enter_row<MODE, NL, HALF, true>(q, expand_raw<NL>(ua, jj), expand_raw<NL>(ya, jj), ends, lc.last, wa);
    enter_row<MODE, NL, HALF, true>(q, expand_raw<NL>(ub, jj), expand_raw<NL>(yb, jj), ends, lc.last, wb);
    // the S = 0 line (row 0 when the mesh starts at 0): A1 keeps only the -r/2
    // of the split
    if (s == 0 && (TAB_LDS ? tch[11] : spr[11]) == 0.0) zero_line<MODE, HALF>(q, wb);  // [S != 0]
    // the next tile (this one again after the last)
    const Geom gn = RUNS ? geom_of(on, start_n) : g;
    // byte offsets of the row the walk loads next (row s + 1 + PF + k at step
    // k), at the column and at the edge column
    unsigned oc = (unsigned)(s + 1 + PF) * rstep + lc.jcb, ox = oc - lc.jcb + lc.jxb;

    double mu[MAXL], nreg[MAXL], dv[MAXL];
#pragma unroll
    for (int k = 0; k < MAXL; ++k) {
      const int slot = k % PF;
      // the table row of row s + k
      SpotRow R;
      double2 ta2, tb2;
      if constexpr (TAB_LDS) {
        R = lds_row_fields(tch + k * kSpFields);
      } else {
        quad_row_load(spr + clamp_row(s + k + 2) * kSpRow, jj, ta2, tb2);
      }
      // row s + k + 1 enters the window; its slot takes the loads of row
      // s + k + 1 + PF, or, where this tile needs no more rows, the next
      // tile's row of that slot
      {
        const Row3 un = expand_raw<NL>(ru[slot], jj);
        Row3 yn{0.0, 0.0, 0.0};
        if constexpr (HAS_Y) yn = expand_raw<NL>(ry[slot], jj);
        enter_row<MODE, NL, HALF, false>(q, un, yn, ends, lc.last, wc);
        if (RUNS && k == MAXL - PF) {
          oc = (unsigned)(gn.s + 1) * gn.rstep + gn.lc.jcb;
          ox = oc - gn.lc.jcb + gn.lc.jxb;
        }
        const bool here = k < MAXL - PF;
        if (RUNS || here) {
          const Buf bu = here ? u : gn.u, by = here ? y2 : gn.y2;
          ru[slot] = Raw2{buf_load(bu, ox), buf_load(bu, oc)};
          if constexpr (HAS_Y) ry[slot] = Raw2{buf_load(by, ox), buf_load(by, oc)};
        }
        oc += here ? rstep : gn.rstep;
        ox += here ? rstep : gn.rstep;
      }
      if constexpr (!TAB_LDS) R = quad_row_fields(ta0, tb0);

      const Bands B = a0_bands(R, q.c0h);
      // the entries of dt A0 and theta dt A0, fl(c * a), as the reference's
      // scaled operators hold them; applied in its band order (super, main,
      // sub).  With theta = 1/2 the latter are half the former, exactly, and so
      // is every product and sum of them.
      const double dsub = dt * B.sub, dmid = dt * B.mid, dsup = dt * B.sup;
      const double tsub = HALF ? 0.5 * dsub : tdt * B.sub, tsup = HALF ? 0.5 * dsup : tdt * B.sup;
      const double tmid = tdt * B.mid;
      double rhs = 0.0, ex = 0.0;
      if constexpr (MODE == SM_IMPL) {
        rhs = wb.uc + dt * B.r0;
      } else {
        auto a0d = [&](double xa, double xb, double xc) {
          return (dsup * xc + dmid * xb) + dsub * xa;
        };
        // d - (theta dt A0 x), given a = dt A0 x
        auto less_a0t = [&](double d, double a, double xa, double xb, double xc) {
          if constexpr (HALF) return __builtin_fma(-0.5, a, d);
          return d - ((tsup * xc + tmid * xb) + tsub * xa);
        };
        // (A01 f)(i, j) from the rows' shares
        auto x01 = [&](double ra, double rb, double rc) {
          return q.rsv * (R.wsub * ra + R.wmid * rb + R.wsup * rc);
        };
        // Y0 = U + dt A0 U + dt R0 + dt A01 U + dt A1 U, in the reference's
        // order of its explicit operators (spot, cross, variance)
        const double a0 = a0d(wa.uc, wb.uc, wc.uc);
        const double y0 =
            ((wb.uc + (a0 + dt * B.r0)) + dt * x01(wa.urs, wb.urs, wc.urs)) + wb.f1u;
        ex = HALF ? wb.f1u : wb.t1u;
        if constexpr (MODE == SM_FIRST) {
          rhs = less_a0t(y0, a0, wa.uc, wb.uc, wc.uc);
        } else if constexpr (MODE == SM_HV) {
          // the second-stage corrections act on the difference of the states
          // (FiniteDifferenceEngine.pyx:744-765, 818-835, 881-894)
          // V = Y0 - 1/2 F (U - Y2) over the explicit operators (no residual)
          const double v1 = ((y0 + 0.5 * a0d(wa.dc, wb.dc, wc.dc)) +
                             0.5 * (dt * x01(wa.drs, wb.drs, wc.drs))) +
                            0.5 * wb.f1d;
          rhs = less_a0t(v1, HALF ? a0d(wa.yc, wb.yc, wc.yc) : 0.0, wa.yc, wb.yc, wc.yc);
          ex = wb.t1y;
        } else if constexpr (MODE == SM_CS) {
          rhs = less_a0t(y0 + (0.5 * dt) * x01(wa.drs, wb.drs, wc.drs), a0, wa.uc, wb.uc, wc.uc);
        } else {  // SM_MCS: (1/2 - theta) F (Y2 - U), residual included
          const double h = 0.5 - ow.th();
          const double xd = x01(wa.drs, wb.drs, wc.drs);
          const double v1 = (((y0 + tdt * xd) + h * (a0d(wa.dc, wb.dc, wc.dc) + dt * B.r0)) +
                             h * (dt * xd)) +
                            h * wb.f1d;
          rhs = less_a0t(v1, a0, wa.uc, wb.uc, wc.uc);
        }
      }
      // the solve forces the Dirichlet row 0 to 0 (a barrier's row below)
      if (k == 0 && s == 0) rhs = 0.0;
      // I - tdt*A0 on this row (identity rows on Dirichlet rows and zero
      // off-diagonals at the line ends come from the bands), scaled by the
      // pivot.  The diagonal 1 - tdt*b is one fused operation, as
      // spot_factor forms it, written out so that the compiler's
      // contraction choices cannot change how the recomputed pivots round.
      const double rd0 = recip(__builtin_fma(-tdt, B.mid, 1.0) - (-tsub * rdp) * cp);
      rdp = rd0;
      cp = -tsup;
      const double dsc = rd0 * rhs;
      mu[k] = tsub * rd0;
      nreg[k] = tsup * rd0;
      dv[k] = dsc;
      if constexpr (HAS_EX) eb[k * THREADS + tid] = ex;
      // slide the window
      wa = wb;
      wb = wc;
      if constexpr (!TAB_LDS) {
        ta0 = ta1; tb0 = tb1; ta1 = ta2; tb1 = tb2;
      }
      // this row's results before the next row's loads (registers)
      pin(dsc);
      pin(rdp);
      if constexpr (HAS_EX) pin(ex);
      __builtin_amdgcn_sched_barrier(0);
    }
    // (also after the last tile, which is then loaded again: a branch would
    // keep this tile's values alive through the walk)
    const bool barrier = ow.barrier();
    const Buf ob = buf_of(out + ow.off(), g.nbytes);
    if constexpr (RUNS) {
      load_head(gn, on);
    }
    // a barrier's Dirichlet row (its bands are zero, its pivot 1)
    if (barrier) {
#pragma unroll
      for (int k = 0; k < MAXL; ++k)
        if (s + k == nS - 1) dv[k] = 0.0;
    }
    // Chunk maps and fix-ups.  Rows k >= L belong to the next chunk; L is
    // uniform, so full chunks (L == MAXL, the common case) take unguarded loops.
    const bool full = L == MAXL;
    const bool active = lc.ok && s < nS;
    double M = 1.0, E = 0.0;
    if (full) {
#pragma unroll
      for (int k = 0; k < MAXL; ++k) {
        E = dv[k] + mu[k] * E;
        M = mu[k] * M;
      }
    } else {
#pragma unroll
      for (int k = 0; k < MAXL; ++k) {
        if (k < L) {
          E = dv[k] + mu[k] * E;
          M = mu[k] * M;
        }
      }
    }
    double yv = 0.0;
    if constexpr (NL == 4) {
      yv = quad_carry<THREADS, false>(active ? M : 1.0, active ? E : 0.0, tot_f);
    } else {
      cM[jj * (TPL + 1) + ch] = active ? M : 1.0;
      cE[jj * (TPL + 1) + ch] = active ? E : 0.0;
      __syncthreads();
      // every wave is past its walk
      // the next tile's table rows, and the records of the tiles after it
      load_table(gn, on);
      ow = on;
      on.load(c.opts + __builtin_amdgcn_readfirstlane(t2.opt));
      start_n = __builtin_amdgcn_readfirstlane(t2.start);
      t2 = load_tile(at + 3 * step);
      affine_scan<THREADS, NL, false>(cM, cE, cIn);
      __syncthreads();
      yv = cIn[jj * (TPL + 1) + ch];
    }
    // Forward fix-up, then the local backward recurrence x = y' + n x'.
#pragma unroll
    for (int k = 0; k < MAXL; ++k) {
      yv = dv[k] + mu[k] * yv;
      dv[k] = yv;
    }
    M = 1.0;
    E = 0.0;
    if (full) {
#pragma unroll
      for (int k = MAXL - 1; k >= 0; --k) {
        E = dv[k] + nreg[k] * E;
        M = nreg[k] * M;
      }
    } else {
#pragma unroll
      for (int k = MAXL - 1; k >= 0; --k) {
        if (k < L) {
          E = dv[k] + nreg[k] * E;
          M = nreg[k] * M;
        }
      }
    }
    double x = 0.0;
    if constexpr (NL == 4) {
      x = quad_carry<THREADS, true>(active ? M : 1.0, active ? E : 0.0, tot_b);
    } else {
      __syncthreads();  // everyone done reading cIn of the forward scan
      cM[jj * (TPL + 1) + ch] = active ? M : 1.0;
      cE[jj * (TPL + 1) + ch] = active ? E : 0.0;
      __syncthreads();
      affine_scan<THREADS, NL, true>(cM, cE, cIn);
      lds_loads_done();
      __syncthreads();  // the carries, and the next tile's table rows
      x = cIn[jj * (TPL + 1) + ch];
    }
    // Backward fix-up; stage output x - tdt*A1(f) written straight from the
    // chunk (rows past the grid and lanes past its columns fall outside the
    // buffer).
    // byte offset of (row s + k, column j), stepped down the chunk
    unsigned sb = lc.ok ? (unsigned)(s + MAXL - 1) * rstep + lc.jcb : 0xfffffff8u;
    auto put = [&](int k) {
      double v = x;
      if constexpr (HAS_EX) {
        const double ex = eb[k * THREADS + tid];
        v = HALF ? __builtin_fma(-0.5, ex, x) : x - ex;
      }
      buf_store(ob, sb, v);
    };
    if (full) {
#pragma unroll
      for (int k = MAXL - 1; k >= 0; --k) {
        x = dv[k] + nreg[k] * x;
        put(k);
        sb -= rstep;
      }
    } else {
#pragma unroll
      for (int k = MAXL - 1; k >= 0; --k) {
        if (k < L) {
          x = dv[k] + nreg[k] * x;
          put(k);
        }
        sb -= rstep;
      }
    }
    if (!more) break;
    at += step;
    g = gn;
  }
}

// Waves per SIMD that a sweep's registers have to leave room for.  Craig-Sneyd's
// second stage on four-column tiles of 8 rows fits three (168 registers; left
// alone it takes 170 and two): 1,024 uneven grids in 658 us instead of 739,
// 512 grids of 512 x 128 in 335 instead of 389.
constexpr int spot_waves(int mode, int threads, int nl, int maxl) {
  return nl == 4 && maxl == 8 && mode == SM_CS ? 3 : threads == 256 ? 2 : 1;
}

template <int MODE, int THREADS, int NL, int MAXL>
__global__ void __launch_bounds__(THREADS, spot_waves(MODE, THREADS, NL, MAXL))
spot_sweep_kernel(Ctx c, const Tile *__restrict__ tiles, int ntiles, const double *__restrict__ U,
                  const double *__restrict__ Y, double *__restrict__ out) {
  extern __shared__ double lds[];
  const Tile t = tiles[xcd_tile(blockIdx.x, ntiles)];
  OptWords o;
  o.load(c.opts + t.opt);
  if (MODE != SM_IMPL && o.th() == 0.5)
    spot_tiles<MODE, THREADS, NL, MAXL, MODE != SM_IMPL>(c, tiles, ntiles, o, t.start, U, Y, out, lds);
  else
    spot_tiles<MODE, THREADS, NL, MAXL, false>(c, tiles, ntiles, o, t.start, U, Y, out, lds);
}

// ---- variance sweep -------------------------------------------------------------
// Lines along the variance axis are contiguous.  A work-group of 256 threads
// handles G = 256/TPL adjacent spot rows of one option; lane ln of a line owns
// positions [ln*L, ln*L + L) with L = ceil(nv / TPL) <= MAXL.  The rows are
// staged in LDS in a slot layout: line g, chunk ln, slot k (k < MAXL) at
// g*LP + ln*(MAXL+1) + k (odd pitch: the TPL lanes reading slot k hit
// distinct banks).  Slots past a chunk's L positions or past the line end
// hold the identity of the two recurrences (right-hand side 0, multipliers
// 1, pivot 0), so every chunk is MAXL slots long and the loops carry no
// guards.  Staging walks the 256*MAXL slots of the tile with shifts only
// (G * TPL * MAXL = 256 * MAXL).  The factorisation tables (M, N, RD, shared
// by every S != 0 line of the option) are staged the same way.  Each lane
// then solves its chunk in registers; the chunk carries of both triangular
// sweeps are combined with segmented wave scans of affine maps, the result
// goes back to LDS and is stored with coalesced writes.  The S = 0 line is
// diagonal.
template <int MODE, int TPL, int MAXL>
__global__ void __launch_bounds__(256)
var_sweep_kernel(Ctx c, const Tile *__restrict__ tiles, const double *__restrict__ W,
                 double *__restrict__ out) {
  static_assert((MAXL & (MAXL - 1)) == 0 && (TPL & (TPL - 1)) == 0, "powers of two");
  extern __shared__ double lds[];
  constexpr int G = 256 / TPL;
  constexpr int P = MAXL + 1;         // slot pitch of a chunk
  constexpr int LP = TPL * P + 1;     // line pitch
  constexpr int SL = TPL * MAXL;      // slots per line
  constexpr int NI = G * SL / 256;    // slots per thread (= MAXL)
  const Tile t = tiles[xcd_tile(blockIdx.x, gridDim.x)];
  const HOpt o = c.opts[t.opt];
  const int nS = (int)o.nS, nv = (int)o.nv, i0 = t.start;
  const int L = (nv + TPL - 1) / TPL;
  double *tM = lds, *tN = tM + LP, *tR = tN + LP, *lines = tR + LP;
  const int tid = threadIdx.x;
  const int rows = nS - i0 < G ? nS - i0 : G;
  const double *w = W + o.off;
  const unsigned unv = (unsigned)nv;

  // Stage the tables (one line of slots) ...
#pragma unroll
  for (int a = 0; a < (SL + 255) / 256; ++a) {
    const int sq = tid + 256 * a;
    if (SL >= 256 || sq < SL) {
      const int ln = sq / MAXL, k = sq % MAXL;
      const int j = ln * L + k;
      const bool valid = k < L && j < nv;
      const int jl = valid ? j : 0;
      const double m = VT(c, o, VT_M, jl), n = VT(c, o, VT_N, jl), r = VT(c, o, VT_RD, jl);
      const int slot = ln * P + k;
      tM[slot] = valid ? m : 1.0;
      tN[slot] = valid ? n : 1.0;
      tR[slot] = valid ? r : 0.0;
    }
  }
  // ... and the rows (all loads first, then the LDS writes).
  {
    double val[NI];
#pragma unroll
    for (int a = 0; a < NI; ++a) {
      const int q = tid + 256 * a;
      const int g = q / SL, sq = q % SL;
      const int ln = sq / MAXL, k = sq % MAXL;
      const int j = ln * L + k;
      const bool valid = g < rows && k < L && j < nv;
      const unsigned ii = (unsigned)(i0 + (g < rows ? g : 0));
      const unsigned jl = valid ? (unsigned)j : 0u;
      double v = w[ii * unv + jl];
      if (MODE == VM_IMPL) {
        auto xw = [&](int64_t x, int64_t y) { return w[x * nv + y]; };
        v += o.dt * a01_dot(c, o, (int64_t)ii, (int64_t)jl, xw);
      }
      val[a] = valid ? v : 0.0;
    }
#pragma unroll
    for (int a = 0; a < NI; ++a) {
      const int q = tid + 256 * a;
      const int g = q / SL, sq = q % SL;
      const int ln = sq / MAXL, k = sq % MAXL;
      lines[g * LP + ln * P + k] = val[a];
    }
  }
  __syncthreads();
  const int ln = tid % TPL, g = tid / TPL;
  const int i = i0 + g;
  const bool row_ok = g < rows;
  const bool diag = row_ok && SP(c, o, SP_S, i) == 0.0;
  const bool fact = row_ok && !diag;
  // Bottom fold of the right-hand side, d[nv-1] += f d[nv-2], by one lane
  // per line (the slots of both positions are staged).
  if (fact && ln == 0) {
    const int j1 = nv - 1, j2 = nv - 2;
    double *ln0 = lines + g * LP;
    ln0[(j1 / L) * P + j1 % L] += o.fold_f * ln0[(j2 / L) * P + j2 % L];
  }
  __syncthreads();
  double *lp = lines + g * LP + ln * P;
  double d[MAXL], mreg[MAXL], nreg[MAXL], rreg[MAXL];
#pragma unroll
  for (int k = 0; k < MAXL; ++k) {
    d[k] = lp[k];
    mreg[k] = tM[ln * P + k];
    nreg[k] = tN[ln * P + k];
    rreg[k] = tR[ln * P + k];
  }
  // Local forward recurrence y = d + m y.
  double M = 1.0, E = 0.0;
#pragma unroll
  for (int k = 0; k < MAXL; ++k) {
    E = d[k] + mreg[k] * E;
    M = mreg[k] * M;
  }
  // Segmented inclusive prefix scan, then the carry entering each chunk.
  wave_prefix_scan<TPL>(M, E, ln);
  const double carry = from_prev_lane<TPL>(E, ln);
  {
    double y = carry;
#pragma unroll
    for (int k = 0; k < MAXL; ++k) {
      y = d[k] + mreg[k] * y;
      d[k] = y;
    }
  }
  // Local backward recurrence x = rd y + n x'.
  M = 1.0;
  E = 0.0;
#pragma unroll
  for (int k = MAXL - 1; k >= 0; --k) {
    E = rreg[k] * d[k] + nreg[k] * E;
    M = nreg[k] * M;
  }
  // Segmented inclusive suffix scan (maps of higher lanes applied first).
  wave_suffix_scan<TPL>(M, E, ln);
  const double after = from_next_lane<TPL>(E, ln);
  {
    double x = after;
#pragma unroll
    for (int k = MAXL - 1; k >= 0; --k) {
      x = rreg[k] * d[k] + nreg[k] * x;
      d[k] = x;
    }
  }
  if (diag) {
    // the S = 0 line is diagonal: x = rdS0 * rhs (slots, not the solve above)
#pragma unroll
    for (int k = 0; k < MAXL; ++k) d[k] = o.rdS0 * lp[k];
  }
#pragma unroll
  for (int k = 0; k < MAXL; ++k) lp[k] = d[k];
  __syncthreads();
  double *ob = out + o.off + (int64_t)i0 * nv;
#pragma unroll
  for (int a = 0; a < NI; ++a) {
    const int q = tid + 256 * a;
    const int gq = q / SL, sq = q % SL;
    const int lq = sq / MAXL, k = sq % MAXL;
    const int j = lq * L + k;
    if (gq < rows && k < L && j < nv) ob[(unsigned)gq * unv + (unsigned)j] = lines[gq * LP + lq * P + k];
  }
}

// ---- set-up kernels ---------------------------------------------------------------
// One thread per spot node of every option: the (0,) and (0,0) template rows
// (with boundary rows) scaled by r*S and 1/2*S^2, and the cross weights.
__global__ void spot_tables_kernel(const HOpt *opts, int nopt, const int64_t *row_opt,
                                   const double *__restrict__ spots, double *sp, int64_t sp_n,
                                   double *spr) {
#pragma clang fp contract(off)
  const int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (g >= sp_n) return;
  const int k = (int)row_opt[g];
  const HOpt o = opts[k];
  const int64_t i = g - o.so, n = o.nS;
  const double *m = spots + o.so;
  double w1[3] = {0, 0, 0}, w2[3] = {0, 0, 0}, ws[3] = {0, 0, 0};
  double R1 = 0.0, R2 = 0.0;
  const bool dir = (i == 0) || (o.barrier && i == n - 1);
  if (i > 0 && i < n - 1) {
    const double hm = m[i] - m[i - 1], hp = m[i + 1] - m[i], x = hm + hp;
    w1[2] = hm / (hp * x);
    w1[1] = (-hm + hp) / (hm * hp);
    w1[0] = -hp / (hm * x);
    w2[2] = 2 / (hp * x);
    w2[1] = -2 / (hm * hp);
    w2[0] = 2 / (hm * x);
    ws[0] = w1[0]; ws[1] = w1[1]; ws[2] = w1[2];
  } else if (i == n - 1 && !o.barrier) {
    const double d = m[n - 1] - m[n - 2];
    R1 = 1.0;                 // dU/dS = 1 (Von Neumann)
    w2[1] = -2 / (d * d);     // second derivative with known first derivative
    w2[0] = 2 / (d * d);
    R2 = 2 / d;
  }
  const double S = m[i];
  const double c0 = o.r * S;
  const double S2h = 0.5 * (S * S);
  double *col = sp + g;
  col[SP_PSUB * sp_n] = dir ? 0.0 : w1[0] * c0;
  col[SP_PMID * sp_n] = dir ? 0.0 : w1[1] * c0 + (-0.5 * o.r);
  col[SP_PSUP * sp_n] = dir ? 0.0 : w1[2] * c0;
  col[SP_QSUB * sp_n] = dir ? 0.0 : w2[0];
  col[SP_QMID * sp_n] = dir ? 0.0 : w2[1];
  col[SP_QSUP * sp_n] = dir ? 0.0 : w2[2];
  col[SP_PR * sp_n] = dir ? 0.0 : R1 * c0;
  col[SP_QR * sp_n] = dir ? 0.0 : R2;
  col[SP_WSUB * sp_n] = ws[0];
  col[SP_WMID * sp_n] = ws[1];
  col[SP_WSUP * sp_n] = ws[2];
  col[SP_S * sp_n] = S;
  // AoS row of the spot sweep (layout at kSpRow): neighbour-of-Dirichlet band
  // entries zeroed, cross weights premultiplied by S, S^2 (row 0: [S != 0]).
  double *row = spr + g * 16;
  const bool zsub = i == 1;                       // row 0 is Dirichlet
  const bool zsup = o.barrier && i == n - 2;      // row n-1 is Dirichlet
  row[0] = zsub ? 0.0 : col[SP_PSUB * sp_n];
  row[1] = col[SP_PMID * sp_n];
  row[2] = zsup ? 0.0 : col[SP_PSUP * sp_n];
  row[3] = zsub ? 0.0 : col[SP_QSUB * sp_n];
  row[4] = col[SP_QMID * sp_n];
  row[5] = zsup ? 0.0 : col[SP_QSUP * sp_n];
  row[6] = col[SP_PR * sp_n];
  row[7] = col[SP_QR * sp_n];
  row[8] = S * ws[0];
  row[9] = S * ws[1];
  row[10] = S * ws[2];
  row[11] = i > 0 ? S * S : (S != 0.0 ? 1.0 : 0.0);
}

// One thread per variance node: A1 rows for S != 0 lines and cross weights.
__global__ void var_tables_kernel(const HOpt *opts, const int64_t *row_opt,
                                  const double *__restrict__ vars, double *vt, int64_t vt_n) {
#pragma clang fp contract(off)
  const int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (g >= vt_n) return;
  const int k = (int)row_opt[g];
  const HOpt o = opts[k];
  const int64_t j = g - o.vo, n = o.nv;
  const double *m = vars + o.vo;
  double u1[3] = {0, 0, 0}, u2[3] = {0, 0, 0}, wv[3] = {0, 0, 0};
  if (j > 0 && j < n - 1) {
    const double hm = m[j] - m[j - 1], hp = m[j + 1] - m[j], x = hm + hp;
    u1[2] = hm / (hp * x);
    u1[1] = (-hm + hp) / (hm * hp);
    u1[0] = -hp / (hm * x);
    u2[2] = 2 / (hp * x);
    u2[1] = -2 / (hm * hp);
    u2[0] = 2 / (hm * x);
    wv[0] = u1[0]; wv[1] = u1[1]; wv[2] = u1[2];
  } else if (j == 0) {
    const double d1 = m[1] - m[0];
    u1[2] = 1 / d1;   // one-sided first derivative; d2/dv2 row is Von Neumann 0
    u1[1] = -1 / d1;
  } else {
    const double d1 = m[n - 1] - m[n - 2], d2 = m[n - 2] - m[n - 3];
    u1[1] = 1.0 / d1;
    u1[0] = -1.0 / d1;
    const double rd = 1.0 / (0.5 * (d2 + d1) * d2 * d1);
    u2[0] = -(d2 + d1) * rd;
    u2[1] = d2 * rd;
  }
  const double v = m[j];
  const double c1 = o.kappa * (o.theta - v);
  const double c11 = (0.5 * (o.sigma * o.sigma)) * v;
  double *col = vt + g;
  col[VT_GSUB * vt_n] = u1[0] * c1 + u2[0] * c11;
  // diagonal of the combined operator for S != 0 lines, in the reference's
  // order: ((1,) band + split) + (1,1) band
  col[VT_GMID * vt_n] = (u1[1] * c1 + (-o.r / 2.0)) + u2[1] * c11;
  col[VT_GSUP * vt_n] = u1[2] * c1 + u2[2] * c11;
  col[VT_WSUB * vt_n] = wv[0];
  col[VT_WMID * vt_n] = wv[1];
  col[VT_WSUP * vt_n] = wv[2];
  col[VT_V * vt_n] = v;
}

// Gz and the folded LU of I - tdt*A1 for S != 0 lines, one wave per option.
// Bound by the pivots' serial chain: 64 rows at a time their band entries are
// formed one row per lane and passed through LDS, every lane runs the chain on
// broadcast reads, and each keeps the pivot of its row for the coalesced
// results.  One thread per option, loading as it went, took 224 us for
// one option of 1,024 rows (57 now) and 33 us for 150 (12 now).
constexpr int kFactorRows = 64;
__device__ __forceinline__ void var_factor(double (*rows)[8], int k, HOpt *opts,
                                           const double *__restrict__ vars, double *vt,
                                           int64_t vt_n) {
  const int lane = threadIdx.x;
  HOpt o = opts[k];
  const int64_t n = o.nv;
  const double *m = vars + o.vo;
  const double *G = vt;
  auto g = [&](int f, int64_t j) { return G[f * vt_n + o.vo + j]; };
  {
    const double d1 = m[n - 1] - m[n - 2], d2 = m[n - 2] - m[n - 3];
    const double rd = 1.0 / (0.5 * (d2 + d1) * d2 * d1);
    o.Gz = (d1 * rd) * ((0.5 * (o.sigma * o.sigma)) * m[n - 1]);
  }
  const double t = o.tdt;
  auto row = [&](int64_t j, double &a, double &b, double &c) {
    a = j > 0 ? -t * g(VT_GSUB, j) : 0.0;
    b = 1.0 - t * g(VT_GMID, j);
    c = j < n - 1 ? -t * g(VT_GSUP, j) : 0.0;
  };
  // Fold of the last row: f = -zL / aL[n-2].
  double a2, b2, c2;
  row(n - 2, a2, b2, c2);
  const double zL = -t * o.Gz;
  const double f = a2 == 0.0 ? 0.0 : -zL / a2;
  o.fold_f = f;
  o.rdS0 = 1.0 / (1.0 - t * (-0.5 * o.r));
  double *M = vt + VT_M * vt_n + o.vo, *RD = vt + VT_RD * vt_n + o.vo,
         *N = vt + VT_N * vt_n + o.vo;
  double rdprev = 0.0, cprev = 0.0;
  for (int64_t j0 = 0; j0 < n; j0 += kFactorRows) {
    const int64_t j = j0 + lane;
    double a = 0.0, b = 1.0, c = 0.0;  // rows beyond the last one
    if (j < n) row(j, a, b, c);
    if (j == n - 1) {
      a += f * b2;
      b += f * c2;
    }
    __syncthreads();
    rows[lane][0] = a;
    rows[lane][1] = b;
    rows[lane][2] = c;
    __syncthreads();
    const double before = rdprev;
    double rd = 0.0;
#pragma unroll 8
    for (int q = 0; q < kFactorRows; ++q) {
      const double l = rows[q][0] * rdprev;
      rdprev = recip(rows[q][1] - l * cprev);
      cprev = rows[q][2];
      if (lane == q) rd = rdprev;
    }
    double rdup = __shfl_up(rd, 1, 64);
    if (lane == 0) rdup = before;
    if (j < n) {
      M[j] = -(a * rdup);
      RD[j] = rd;
      N[j] = -c * rd;
    }
  }
  if (lane == 0) {
    opts[k].Gz = o.Gz;
    opts[k].fold_f = o.fold_f;
    opts[k].rdS0 = o.rdS0;
  }
}

// Pivots 1/b' of I - tdt*A0 on every spot line, one wave per 64 lines of an
// option.  Bound by each line's serial chain (a mesh of 1,024 lines is 16
// waves): the table rows, the same for all lanes, are fetched 64 at a time a
// chunk ahead of the chain and read back from LDS, and the next rows' band
// entries fill the chain's gaps.  Loading each row where it is used took 669
// us on 2,048 x 1,024 nodes (166 now) and 50 us on 150 x 150 (15 now).
__device__ __forceinline__ void spot_factor(double (*rows)[8], const Ctx &c, Tile t,
                                            double *rd0) {
  const HOpt o = c.opts[t.opt];
  const int lane = threadIdx.x;
  const int64_t n = o.nS;
  // lanes past the last column repeat it (no branch around the stores, which
  // would keep a row's arithmetic from filling the gaps of another's)
  const int64_t j = t.start + lane < o.nv ? t.start + lane : o.nv - 1;
  const double v = c.vt[VT_V * c.vt_n + o.vo + j];
  double *rd = rd0 + o.off + j;
  double f[7];
  auto fetch = [&](int64_t i) {  // table row i of this lane's (the last one beyond it)
    const double *col = c.sp + o.so + (i < n ? i : n - 1);
    f[0] = col[SP_PSUB * c.sp_n];
    f[1] = col[SP_QSUB * c.sp_n];
    f[2] = col[SP_PMID * c.sp_n];
    f[3] = col[SP_QMID * c.sp_n];
    f[4] = col[SP_PSUP * c.sp_n];
    f[5] = col[SP_QSUP * c.sp_n];
    f[6] = col[SP_S * c.sp_n];
  };
  // Row 0 is Dirichlet, and the last one of a barrier option: a = c = 0, b = 1.
  double rdprev = 1.0, cprev = 0.0;
  rd[0] = 1.0;
  const int64_t last = o.barrier ? n - 1 : n;
  fetch(1 + lane);
  for (int64_t i0 = 1; i0 < last; i0 += kFactorRows) {
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 7; ++q) rows[lane][q] = f[q];
    __syncthreads();
    fetch(i0 + kFactorRows + lane);
    auto step = [&](int q) {
      const double *w = rows[q];
      const double c00 = c00_of(v, w[6]);
      const double a = -o.tdt * band_add(w[0], w[1], c00);
      const double b = 1.0 - o.tdt * band_add(w[2], w[3], c00);
      rdprev = recip(b - (a * rdprev) * cprev);
      cprev = -o.tdt * band_add(w[4], w[5], c00);
      rd[(i0 + q) * o.nv] = rdprev;
    };
    if (last - i0 >= kFactorRows) {
#pragma unroll 8
      for (int q = 0; q < kFactorRows; ++q) step(q);
    } else {
      for (int q = 0; q < (int)(last - i0); ++q) step(q);
    }
  }
  if (o.barrier) rd[(n - 1) * o.nv] = 1.0 / (1.0 - (0.0 * rdprev) * cprev);
}

// Both factorisations, which are independent, side by side: work-groups
// [0, nopt) the options' variance lines, the rest tiles of spot lines.  (Each
// writes what the other does not read.)
__global__ void __launch_bounds__(64) factor_kernel(Ctx c, HOpt *opts, int nopt,
                                                    const double *__restrict__ vars, double *vt,
                                                    const Tile *__restrict__ tiles, double *rd0) {
  __shared__ __attribute__((aligned(16))) double rows[kFactorRows][8];
  if ((int)blockIdx.x < nopt)
    var_factor(rows, blockIdx.x, opts, vars, vt, c.vt_n);
  else
    spot_factor(rows, c, tiles[(int)blockIdx.x - nopt], rd0);
}

// Step sizes of every option from the scheme's theta and the dt multiplier,
// taken from device scalars (d_theta, d_scale) when given, else from the host
// values; the pair used is kept in `slots` for later refactorisations.
__global__ void step_scalars_kernel(HOpt *opts, int nopt, const double *__restrict__ base_dt,
                                    const double *d_theta, const double *d_scale, double theta,
                                    double scale, int implicit, double *slots) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nopt) return;
  const double th = d_theta ? *d_theta : theta;
  const double sc = d_scale ? *d_scale : scale;
  HOpt &o = opts[k];
  o.dt = base_dt[k] * sc;
  o.tdt = implicit ? o.dt : th * o.dt;
  o.th = implicit ? 1.0 : th;
  if (k == 0 && slots) {
    slots[0] = th;
    slots[1] = sc;
  }
}

// Parameters of every option from a device array of rows (r, kappa, theta,
// sigma, rho, dt); the shapes and offsets stay.
__global__ void set_params_kernel(HOpt *opts, int nopt, const double *__restrict__ rows,
                                  double *base_dt) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nopt) return;
  const double *q = rows + 6 * (int64_t)k;
  HOpt &o = opts[k];
  o.r = q[0];
  o.kappa = q[1];
  o.theta = q[2];
  o.sigma = q[3];
  o.rho = q[4];
  o.dt = q[5];
  o.barrier = 0;
  base_dt[k] = q[5];
}

// One work-group per spot row of every option: V(i, j) = max(S_i - K_k, 0).
__global__ void call_payoff_kernel(const HOpt *opts, const int64_t *row_opt,
                                   const double *__restrict__ spots, int64_t sp_n,
                                   const double *__restrict__ strikes, double *state) {
  const int64_t g = blockIdx.x;
  if (g >= sp_n) return;
  const int k = (int)row_opt[g];
  const HOpt o = opts[k];
  const int64_t i = g - o.so;
  const double v = fmax(spots[g] - strikes[k], 0.0);
  double *row = state + o.off + i * o.nv;
  for (int64_t j = threadIdx.x; j < o.nv; j += blockDim.x) row[j] = v;
}

// First node of the 4-point stencil around x on mesh m[0..n): nodes
// i-2 .. i+1 with i the first node >= x, shifted to stay inside the mesh.
__device__ __forceinline__ int64_t stencil4(const double *m, int64_t n, double x) {
  int64_t lo = 0, hi = n;  // lower bound: first index with m[i] >= x
  while (lo < hi) {
    const int64_t mid = (lo + hi) / 2;
    if (m[mid] < x) lo = mid + 1; else hi = mid;
  }
  int64_t s = lo - 2;
  if (s > n - 4) s = n - 4;
  if (s < 0) s = 0;
  return s;
}

__device__ __forceinline__ void lagrange4w(double x, const double *nd, double w[4]) {
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    double p = 1.0;
#pragma unroll
    for (int b = 0; b < 4; ++b)
      if (a != b) p *= (x - nd[b]) / (nd[a] - nd[b]);
    w[a] = p;
  }
}

// One thread per option: the state read at (S0_k, v0_k) by tensor-product
// cubic Lagrange interpolation on the 4 x 4 nodes around the point.
__global__ void read_bicubic_kernel(const HOpt *opts, int nopt, const double *__restrict__ spots,
                                    const double *__restrict__ vars,
                                    const double *__restrict__ state, const double *S0,
                                    const double *v0, double *out) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nopt) return;
  const HOpt o = opts[k];
  const double *ms = spots + o.so, *mv = vars + o.vo;
  const int64_t i = stencil4(ms, o.nS, S0[k]), j = stencil4(mv, o.nv, v0[k]);
  double ws[4], wv[4];
  lagrange4w(S0[k], ms + i, ws);
  lagrange4w(v0[k], mv + j, wv);
  const double *V = state + o.off;
  double acc = 0.0;
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    const double *row = V + (i + a) * o.nv + j;
    acc += ws[a] * (((row[0] * wv[0] + row[1] * wv[1]) + row[2] * wv[2]) + row[3] * wv[3]);
  }
  out[k] = acc;
}

}  // namespace
}  // namespace fdadi

using namespace fdadi;

struct fdadi_hb {
  int nopt = 0;
  std::vector<HOpt> h_opts;  // host copy (dt of each option before dt_scale)
  std::vector<double> base_dt;
  HOpt *d_opts = nullptr;
  double *d_spots = nullptr, *d_vars = nullptr;
  double *d_sp = nullptr, *d_vt = nullptr, *d_spr = nullptr;
  int64_t sp_n = 0, vt_n = 0, total = 0;
  int64_t nSmax = 0, nvmax = 0;
  double *d_state = nullptr, *d_w1 = nullptr, *d_y2 = nullptr, *d_rd0 = nullptr;
  int64_t *d_sp_row = nullptr, *d_vt_row = nullptr;
  Tile *d_stiles = nullptr, *d_vtiles = nullptr, *d_ftiles = nullptr;
  int nstiles = 0, nvtiles = 0, nftiles = 0;
  int64_t cap_stiles = 0, cap_vtiles = 0;  // tile-list capacity (every launch shape fits)
  fdadi_arena *arena = nullptr;            // the one device allocation behind every buffer
  int spot_threads = 0;
  int var_tpl = 1, var_rows = 256;  // variance sweep: lanes per line, rows per 256-thread tile
  std::vector<int> order;           // options, largest first
  int spot_maxl = 8;  // rows per thread in the spot sweep (8, or 16 for long lines)
  int spot_nl = 4;    // columns per spot-sweep tile (4, 8, 16 or 32)
  // Launch groups of each sweep: a shape and a range of its tile list.  One
  // group, unless the shape is chosen per option from its line length
  // (fdadi_hb_set_shape with threads = -1): then options of one shape share
  // a group, and a stage launches once per group.
  struct SweepGroup {
    int threads, maxl;  // spot: threads and rows per thread; variance: lanes per line, -
    int first, ntiles;
  };
  std::vector<SweepGroup> sgroups, vgroups;
  bool spot_split = false, var_split = false;
  int scheme = -1;
  double theta = 0.5, dt_scale = 1.0;
  bool dev_scalars = false;        // last configure took theta and dt from device memory
  bool opts_on_device = false;     // parameters last set by fdadi_hb_update_dev (the host
                                   // copy keeps only the shapes and offsets current)
  double *d_base_dt = nullptr;     // each option's step before the multiplier
  double *d_slots = nullptr;       // [theta, dt multiplier] of the configured scheme
  hipGraph_t graph = nullptr;
  hipGraphExec_t gexec = nullptr;
  std::vector<hipEvent_t> events;  // pool for fdadi_hb_step_timed
};

namespace fdadi {
namespace {

constexpr int kMAXL = 16;  // variance sweep: positions per thread
constexpr int kMAXLs = 8;  // spot sweep: rows per thread
constexpr int kMAXLs3 = 12;  // spot sweep, 16-column tiles chosen per option: rows per thread

Ctx ctx_of(const fdadi_hb *hb) {
  Ctx c;
  c.opts = hb->d_opts;
  c.sp = hb->d_sp;
  c.vt = hb->d_vt;
  c.sp_n = hb->sp_n;
  c.vt_n = hb->vt_n;
  c.rd0 = hb->d_rd0;
  c.spr = hb->d_spr;
  return c;
}

#define FDADI_RET(x)         \
  do {                       \
    int _st = (x);           \
    if (_st) return _st;     \
  } while (0)

// Spot-sweep shape for lines of length n: `threads` per work-group (0 =
// default), `nl` columns per tile (4, 8, 16 or 32), and the rows per thread
// (8, or 16 for long lines).  A thread keeps four values per row in
// registers, so a work-group has at most 512 threads (two waves per SIMD).
int spot_shape(int64_t n, int threads, int nl, int *t_out, int *maxl_out) {
  if (nl != 4 && nl != 8 && nl != 16 && nl != 32) {
    set_error("fdadi_hb_set_shape: spot tiles are 4, 8, 16 or 32 columns wide");
    return FDADI_ERR_ARG;
  }
  if (threads == 0) {
    if (nl == 4 && n <= 512) {
      const int64_t need = (n + kMAXLs - 1) / kMAXLs * 4;
      int t = 64;
      while (t < need) t *= 2;
      *t_out = t;
      *maxl_out = kMAXLs;
      return FDADI_OK;
    }
    threads = 512;
  }
  const int tpl = threads / nl;
  const bool t_ok = threads >= 64 && threads <= 512 && (threads & (threads - 1)) == 0 &&
                    tpl >= 1 && (nl == 4 || threads >= 256) && (nl != 32 || threads == 512);
  if (t_ok && (int64_t)tpl * kMAXLs >= n) {
    *t_out = threads;
    *maxl_out = kMAXLs;
  } else if (t_ok && (int64_t)tpl * 2 * kMAXLs >= n && (threads == 256 || threads == 512)) {
    *t_out = threads;
    *maxl_out = 2 * kMAXLs;
  } else {
    set_error("fdadi_hb_set_shape: too few threads for the longest spot line");
    return FDADI_ERR_ARG;
  }
  return FDADI_OK;
}

// Spot shapes (threads, rows per thread) for nl-column tiles, by the spot
// lines they cover ((threads / nl) * rows), smallest first.
std::vector<std::pair<int, int>> spot_candidates(int nl) {
  std::vector<std::pair<int, int>> c;
  for (int t : {64, 128, 256, 512})
    for (int ml : {kMAXLs, kMAXLs3, 2 * kMAXLs}) {
      // the launch shapes spot_shape accepts, and 12 rows per thread for
      // 16-column tiles (the per-option groups' in-between size)
      if (t / nl < 1 || (nl != 4 && t < 256) || (nl == 32 && t != 512)) continue;
      if (ml != kMAXLs && t != 256 && t != 512) continue;
      if (ml == kMAXLs3 && nl != 16) continue;
      c.push_back({t, ml});
    }
  std::stable_sort(c.begin(), c.end(), [nl](const std::pair<int, int> &a, const std::pair<int, int> &b) {
    return a.first / nl * a.second < b.first / nl * b.second;
  });
  return c;
}

// The shape a split spot sweep gives option o: the smallest candidate whose
// lines cover its nS (-1 if none does).
int spot_group_of(const std::vector<std::pair<int, int>> &c, int nl, int64_t nS) {
  for (size_t g = 0; g < c.size(); ++g)
    if ((int64_t)(c[g].first / nl) * c[g].second >= nS) return (int)g;
  return -1;
}

// (Re)build the spot-sweep tile list (spot_nl columns per tile) and its
// launch groups.
int build_spot_tiles(fdadi_hb *hb) {
  std::vector<Tile> st;
  hb->sgroups.clear();
  const int nl = hb->spot_nl;
  auto add_group = [&](int threads, int maxl, const std::vector<int> &opts) {
    const int first = (int)st.size();
    for (int k : opts) {
      const HOpt &o = hb->h_opts[k];
      // the last tile ends on the last column (it may overlap the one before,
      // whose shared columns both compute identically): the kernel takes
      // column nv - 3 of the last column from the lane two before it
      for (int64_t j0 = 0; j0 < o.nv; j0 += nl)
        st.push_back(Tile{k, (int32_t)(j0 + nl > o.nv && o.nv >= nl ? o.nv - nl : j0)});
    }
    hb->sgroups.push_back({threads, maxl, first, (int)st.size() - first});
  };
  if (!hb->spot_split) {
    add_group(hb->spot_threads, hb->spot_maxl, hb->order);
  } else {
    const auto c = spot_candidates(nl);
    for (size_t g = 0; g < c.size(); ++g) {
      std::vector<int> opts;
      for (int k : hb->order)  // largest first within a group
        if (spot_group_of(c, nl, hb->h_opts[k].nS) == (int)g) opts.push_back(k);
      if (!opts.empty()) add_group(c[g].first, c[g].second, opts);
    }
  }
  FDADI_REQUIRE((int64_t)st.size() <= hb->cap_stiles, FDADI_ERR_STATE,
                "spot tile list exceeds its capacity");
  FDADI_TRY_HIP(hipMemcpy(hb->d_stiles, st.data(), sizeof(Tile) * st.size(),
                          hipMemcpyHostToDevice));
  hb->nstiles = (int)st.size();
  return FDADI_OK;
}

constexpr size_t kCuLds = 160 * 1024;

// Kernels using more than 64 KB of dynamic LDS must say so once.
int allow_lds(const void *fn, size_t bytes) {
  if (bytes <= 65536) return FDADI_OK;
  FDADI_REQUIRE(bytes <= kCuLds, FDADI_ERR_UNSUPPORTED,
                "sweep tile needs " + std::to_string(bytes) + " bytes of LDS (> 160 KB)");
  FDADI_TRY_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
  return FDADI_OK;
}

// Lanes per variance line so that each lane's chunk fits kMAXL registers.
int var_tpl_for(int64_t nv) {
  int t = 1;
  while ((int64_t)t * kMAXL < nv && t < 64) t *= 2;
  return t;
}

// (Re)build the variance-sweep tile list (256 / lanes-per-line spot rows per
// tile) and its launch groups; split: each option gets the fewest lanes
// whose chunks of kMAXL positions cover its variance line.
int build_var_tiles(fdadi_hb *hb) {
  std::vector<Tile> vtl;
  hb->vgroups.clear();
  auto add_tiles = [&](int k, int rows) {
    const HOpt &o = hb->h_opts[k];
    for (int64_t i0 = 0; i0 < o.nS; i0 += rows) vtl.push_back(Tile{k, (int32_t)i0});
  };
  if (!hb->var_split) {
    for (int k : hb->order) add_tiles(k, hb->var_rows);
    hb->vgroups.push_back({hb->var_tpl, 0, 0, (int)vtl.size()});
  } else {
    for (int t = 1; t <= 64; t *= 2) {
      const int first = (int)vtl.size();
      for (int k : hb->order)
        if (var_tpl_for(hb->h_opts[k].nv) == t) add_tiles(k, 256 / t);
      if ((int)vtl.size() > first) hb->vgroups.push_back({t, 0, first, (int)vtl.size() - first});
    }
  }
  FDADI_REQUIRE((int64_t)vtl.size() <= hb->cap_vtiles, FDADI_ERR_STATE,
                "variance tile list exceeds its capacity");
  FDADI_TRY_HIP(hipMemcpy(hb->d_vtiles, vtl.data(), sizeof(Tile) * vtl.size(),
                          hipMemcpyHostToDevice));
  hb->nvtiles = (int)vtl.size();
  return FDADI_OK;
}

template <int MODE, int T, int NL, int ML>
int launch_spot_t(const fdadi_hb *hb, const fdadi_hb::SweepGroup &g, const double *U,
                  const double *Y, double *out, hipStream_t s) {
  constexpr int TPL = T / NL;
  // chunk carries of the scans, the next stage's explicit term (MAXL per
  // thread); wide tiles add their table rows (MAXL rows of 12 fields per chunk)
  const size_t ex = MODE == SM_IMPL ? 0 : (size_t)ML * T;
  const size_t tab = NL == 4 ? 0 : (size_t)TPL * ML * kSpFields;
  const size_t carry = NL == 4 ? T / 4 : 3 * (size_t)NL * (TPL + 1);
  const size_t lds = sizeof(double) * (carry + ex + tab);
  FDADI_RET(allow_lds((const void *)spot_sweep_kernel<MODE, T, NL, ML>, lds));
  // wide tiles: as many work-groups as run at once (two of 256 threads or one
  // of 512 per CU, as the LDS allows: one of 88 KB on 8 columns of 16 rows,
  // where the second half of 512 began after the first half's whole share,
  // 1,024 uneven grids in 553 us a stage, 525 now), each taking tile after tile
  const int slots = NL == 4 ? g.ntiles : 256 * std::min<int>(512 / T, kCuLds / lds);
  hipLaunchKernelGGL((spot_sweep_kernel<MODE, T, NL, ML>), dim3(std::min(g.ntiles, slots)),
                     dim3(T), lds, s, ctx_of(hb), hb->d_stiles + g.first, g.ntiles, U, Y, out);
  FDADI_CHECK_LAUNCH();
  return FDADI_OK;
}

template <int MODE, int NL>
int launch_spot_wide(const fdadi_hb *hb, const fdadi_hb::SweepGroup &g, const double *U,
                     const double *Y, double *out, hipStream_t s) {
  const bool long_rows = g.maxl == 2 * kMAXLs;
  if constexpr (NL == 16) {
    if (g.maxl == kMAXLs3) {
      if (g.threads == 256) return launch_spot_t<MODE, 256, NL, kMAXLs3>(hb, g, U, Y, out, s);
      if (g.threads == 512) return launch_spot_t<MODE, 512, NL, kMAXLs3>(hb, g, U, Y, out, s);
    }
  }
  if constexpr (NL != 32) {  // 32-column tiles: 512 threads (16 lanes per line)
    switch (g.threads * 2 + (long_rows ? 1 : 0)) {
      case 512: return launch_spot_t<MODE, 256, NL, kMAXLs>(hb, g, U, Y, out, s);
      case 513: return launch_spot_t<MODE, 256, NL, 2 * kMAXLs>(hb, g, U, Y, out, s);
    }
  }
  switch (g.threads * 2 + (long_rows ? 1 : 0)) {
    case 1024: return launch_spot_t<MODE, 512, NL, kMAXLs>(hb, g, U, Y, out, s);
    case 1025: return launch_spot_t<MODE, 512, NL, 2 * kMAXLs>(hb, g, U, Y, out, s);
  }
  set_error("spot sweep: unsupported shape for 8-, 16- or 32-column tiles");
  return FDADI_ERR_UNSUPPORTED;
}

template <int MODE>
int launch_spot_group(const fdadi_hb *hb, const fdadi_hb::SweepGroup &g, const double *U,
                      const double *Y, double *out, hipStream_t s) {
  if (hb->spot_nl == 32) return launch_spot_wide<MODE, 32>(hb, g, U, Y, out, s);
  if (hb->spot_nl == 16) return launch_spot_wide<MODE, 16>(hb, g, U, Y, out, s);
  if (hb->spot_nl == 8) return launch_spot_wide<MODE, 8>(hb, g, U, Y, out, s);
  if (g.maxl == 2 * kMAXLs) {
    switch (g.threads) {
      case 256: return launch_spot_t<MODE, 256, 4, 2 * kMAXLs>(hb, g, U, Y, out, s);
      case 512: return launch_spot_t<MODE, 512, 4, 2 * kMAXLs>(hb, g, U, Y, out, s);
    }
    set_error("spot sweep: unsupported thread count for 16 rows per thread");
    return FDADI_ERR_UNSUPPORTED;
  }
  switch (g.threads) {
    case 64: return launch_spot_t<MODE, 64, 4, kMAXLs>(hb, g, U, Y, out, s);
    case 128: return launch_spot_t<MODE, 128, 4, kMAXLs>(hb, g, U, Y, out, s);
    case 256: return launch_spot_t<MODE, 256, 4, kMAXLs>(hb, g, U, Y, out, s);
    case 512: return launch_spot_t<MODE, 512, 4, kMAXLs>(hb, g, U, Y, out, s);
  }
  set_error("spot sweep: unsupported thread count");
  return FDADI_ERR_UNSUPPORTED;
}

// One spot-sweep stage: a launch per group.
template <int MODE>
int launch_spot(const fdadi_hb *hb, const double *U, const double *Y, double *out,
                hipStream_t s) {
  for (const fdadi_hb::SweepGroup &g : hb->sgroups)
    FDADI_RET(launch_spot_group<MODE>(hb, g, U, Y, out, s));
  return FDADI_OK;
}

template <int MODE, int TPL>
int launch_var_t(const fdadi_hb *hb, const fdadi_hb::SweepGroup &g, const double *W, double *out,
                 hipStream_t s) {
  // LDS: three tables and 256/TPL lines of TPL chunks (pitch kMAXL + 1) + 1.
  const size_t lds = sizeof(double) * (3 + 256 / TPL) * (TPL * (kMAXL + 1) + 1);
  FDADI_RET(allow_lds((const void *)var_sweep_kernel<MODE, TPL, kMAXL>, lds));
  hipLaunchKernelGGL((var_sweep_kernel<MODE, TPL, kMAXL>), dim3(g.ntiles), dim3(256), lds, s,
                     ctx_of(hb), hb->d_vtiles + g.first, W, out);
  FDADI_CHECK_LAUNCH();
  return FDADI_OK;
}

// One variance-sweep stage: a launch per group.
template <int MODE>
int launch_var(const fdadi_hb *hb, const double *W, double *out, hipStream_t s) {
  for (const fdadi_hb::SweepGroup &g : hb->vgroups) {
    int st = FDADI_ERR_UNSUPPORTED;
    switch (g.threads) {
      case 1: st = launch_var_t<MODE, 1>(hb, g, W, out, s); break;
      case 2: st = launch_var_t<MODE, 2>(hb, g, W, out, s); break;
      case 4: st = launch_var_t<MODE, 4>(hb, g, W, out, s); break;
      case 8: st = launch_var_t<MODE, 8>(hb, g, W, out, s); break;
      case 16: st = launch_var_t<MODE, 16>(hb, g, W, out, s); break;
      case 32: st = launch_var_t<MODE, 32>(hb, g, W, out, s); break;
      case 64: st = launch_var_t<MODE, 64>(hb, g, W, out, s); break;
      default: set_error("variance sweep: unsupported lanes per line");
    }
    FDADI_RET(st);
  }
  return FDADI_OK;
}

// Optional per-stage event pairs (fdadi_hb_step_timed); null = untimed.
struct StageEvents {
  hipEvent_t *ev;  // 2 per stage, in launch order
  int next;
};

int mark(StageEvents *t, hipStream_t s) {
  if (!t) return FDADI_OK;
  FDADI_TRY_HIP(hipEventRecord(t->ev[t->next++], s));
  return FDADI_OK;
}

#define STAGE(call)                 \
  do {                              \
    FDADI_RET(mark(tm, s));         \
    FDADI_RET(call);                \
    FDADI_RET(mark(tm, s));         \
  } while (0)

// One time step of the configured scheme (stage list of the module comment).
int step_once(fdadi_hb *hb, hipStream_t s, StageEvents *tm = nullptr) {
  double *U = hb->d_state, *W = hb->d_w1, *Y2 = hb->d_y2;
  switch (hb->scheme) {
    case FDADI_SCHEME_DOUGLAS:
      STAGE((launch_spot<SM_FIRST>(hb, U, nullptr, W, s)));
      STAGE((launch_var<VM_PLAIN>(hb, W, U, s)));
      return FDADI_OK;
    case FDADI_SCHEME_IMPLICIT:
      STAGE((launch_var<VM_IMPL>(hb, U, W, s)));
      STAGE((launch_spot<SM_IMPL>(hb, W, nullptr, U, s)));
      return FDADI_OK;
    case FDADI_SCHEME_HV:
      STAGE((launch_spot<SM_FIRST>(hb, U, nullptr, W, s)));
      STAGE((launch_var<VM_PLAIN>(hb, W, Y2, s)));
      STAGE((launch_spot<SM_HV>(hb, U, Y2, W, s)));
      STAGE((launch_var<VM_PLAIN>(hb, W, U, s)));
      return FDADI_OK;
    case FDADI_SCHEME_CS:
      STAGE((launch_spot<SM_FIRST>(hb, U, nullptr, W, s)));
      STAGE((launch_var<VM_PLAIN>(hb, W, Y2, s)));
      STAGE((launch_spot<SM_CS>(hb, U, Y2, W, s)));
      STAGE((launch_var<VM_PLAIN>(hb, W, U, s)));
      return FDADI_OK;
    case FDADI_SCHEME_MCS:
      STAGE((launch_spot<SM_FIRST>(hb, U, nullptr, W, s)));
      STAGE((launch_var<VM_PLAIN>(hb, W, Y2, s)));
      STAGE((launch_spot<SM_MCS>(hb, U, Y2, W, s)));
      STAGE((launch_var<VM_PLAIN>(hb, W, U, s)));
      return FDADI_OK;
  }
  set_error("fdadi_hb_step: engine not configured (call fdadi_hb_configure)");
  return FDADI_ERR_STATE;
}

// Spot and variance tables from the meshes and parameters on the device.
int build_tables(fdadi_hb *hb, hipStream_t s) {
  hipLaunchKernelGGL(spot_tables_kernel, dim3(grid_for(hb->sp_n, 256)), dim3(256), 0, s,
                     hb->d_opts, hb->nopt, hb->d_sp_row, hb->d_spots, hb->d_sp, hb->sp_n,
                     hb->d_spr);
  FDADI_CHECK_LAUNCH();
  hipLaunchKernelGGL(var_tables_kernel, dim3(grid_for(hb->vt_n, 256)), dim3(256), 0, s,
                     hb->d_opts, hb->d_vt_row, hb->d_vars, hb->d_vt, hb->vt_n);
  FDADI_CHECK_LAUNCH();
  return FDADI_OK;
}

// Step sizes of the configured scheme and the time-invariant factorisations
// of I - tdt A0 and I - tdt A1, on the device.  theta and the dt multiplier
// come from the device scalars d_theta / d_scale when given (nothing is read
// back to the host and nothing synchronises), else from hb->theta /
// hb->dt_scale (synchronises).
int refactor(fdadi_hb *hb, hipStream_t s, const double *d_theta = nullptr,
             const double *d_scale = nullptr, bool capturing = false) {
  const bool dev = d_theta || d_scale;
  // the device copy of the options is current after fdadi_hb_update_dev (and
  // is made current before a capture, which records kernels only)
  if (!hb->opts_on_device && !capturing)
    FDADI_TRY_HIP(hipMemcpyAsync(hb->d_opts, hb->h_opts.data(), sizeof(HOpt) * hb->nopt,
                                 hipMemcpyHostToDevice, s));
  const bool reuse = d_theta == hb->d_slots;  // refactorisation with the kept pair
  hipLaunchKernelGGL(step_scalars_kernel, dim3(grid_for(hb->nopt, 64)), dim3(64), 0, s,
                     hb->d_opts, hb->nopt, hb->d_base_dt, d_theta, d_scale, hb->theta,
                     hb->dt_scale, (int)(hb->scheme == FDADI_SCHEME_IMPLICIT),
                     reuse ? nullptr : hb->d_slots);
  FDADI_CHECK_LAUNCH();
  hipLaunchKernelGGL(factor_kernel, dim3(hb->nopt + hb->nftiles), dim3(64), 0, s, ctx_of(hb),
                     hb->d_opts, hb->nopt, hb->d_vars, hb->d_vt, hb->d_ftiles, hb->d_rd0);
  FDADI_CHECK_LAUNCH();
  if (!dev && !capturing) FDADI_TRY_HIP(hipStreamSynchronize(s));
  return FDADI_OK;
}

void drop_graph(fdadi_hb *hb) {
  if (hb->gexec) {
    (void)hipGraphExecDestroy(hb->gexec);
    hb->gexec = nullptr;
  }
  if (hb->graph) {
    (void)hipGraphDestroy(hb->graph);
    hb->graph = nullptr;
  }
}

void free_hb(fdadi_hb *hb) {
  if (!hb) return;
  if (hb->gexec) (void)hipGraphExecDestroy(hb->gexec);
  if (hb->graph) (void)hipGraphDestroy(hb->graph);
  for (hipEvent_t e : hb->events) (void)hipEventDestroy(e);
  (void)fdadi_arena_destroy(hb->arena);
  delete hb;
}

}  // namespace
}  // namespace fdadi

extern "C" {

int fdadi_hb_create(int32_t nopt, const fdadi_heston_option *opts, const double *spots,
                    const double *vars, void *stream, fdadi_hb **out) {
  FDADI_REQUIRE(out && opts && spots && vars && nopt > 0, FDADI_ERR_ARG,
                "fdadi_hb_create: bad arguments");
  hipStream_t s = as_stream(stream);
  fdadi_hb *hb = new fdadi_hb();
  hb->nopt = nopt;
  hb->h_opts.resize(nopt);
  hb->base_dt.resize(nopt);
  int64_t so = 0, vo = 0, off = 0;
  std::vector<int64_t> sp_row, vt_row;
  for (int k = 0; k < nopt; ++k) {
    const fdadi_heston_option &q = opts[k];
    if (q.nS < 4 || q.nv < 4) {
      free_hb(hb);
      set_error("fdadi_hb_create: option " + std::to_string(k) +
                ": grid needs at least 4 points per axis");
      return FDADI_ERR_ARG;
    }
    if (q.nS > 2048 || q.nv > 1024) {
      free_hb(hb);
      set_error("fdadi_hb_create: option " + std::to_string(k) +
                ": the fused engine supports nS <= 2048 and nv <= 1024");
      return FDADI_ERR_UNSUPPORTED;
    }
    HOpt &o = hb->h_opts[k];
    o = HOpt{};
    o.nS = q.nS;
    o.nv = q.nv;
    o.off = off;
    o.so = so;
    o.vo = vo;
    o.r = q.r;
    o.kappa = q.kappa;
    o.theta = q.theta;
    o.sigma = q.sigma;
    o.rho = q.rho;
    o.dt = q.dt;
    o.barrier = q.barrier ? 1 : 0;
    hb->base_dt[k] = q.dt;
    for (int64_t i = 0; i < q.nS; ++i) sp_row.push_back(k);
    for (int64_t j = 0; j < q.nv; ++j) vt_row.push_back(k);
    so += q.nS;
    vo += q.nv;
    off += q.nS * q.nv;
    hb->nSmax = std::max<int64_t>(hb->nSmax, q.nS);
    hb->nvmax = std::max<int64_t>(hb->nvmax, q.nv);
  }
  hb->sp_n = so;
  hb->vt_n = vo;
  hb->total = off;
  // Tiles, largest options first (the dispatcher then balances the tail).
  std::vector<int> order(nopt);
  std::iota(order.begin(), order.end(), 0);
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
    return hb->h_opts[a].nS * hb->h_opts[a].nv > hb->h_opts[b].nS * hb->h_opts[b].nv;
  });
  std::vector<Tile> ft;
  for (int k : order) {
    const HOpt &o = hb->h_opts[k];
    for (int64_t j0 = 0; j0 < o.nv; j0 += 64) ft.push_back(Tile{k, (int32_t)j0});
  }
  hb->nftiles = (int)ft.size();
  spot_shape(hb->nSmax, 0, 4, &hb->spot_threads, &hb->spot_maxl);
  hb->order = order;
  hb->var_tpl = var_tpl_for(hb->nvmax);
  hb->var_rows = 256 / hb->var_tpl;
  // Every device buffer of the engine is carved from one arena (one
  // hipMalloc); the tile lists get the capacity of their largest launch
  // shape (4-column spot tiles, variance tiles of 4 rows) so that changing
  // shapes later allocates nothing.
  for (int k = 0; k < nopt; ++k) {
    hb->cap_stiles += (hb->h_opts[k].nv + 3) / 4;
    hb->cap_vtiles += (hb->h_opts[k].nS + 3) / 4;
  }
  struct Part {
    void **p;
    int64_t bytes;
  };
  const Part parts[] = {
      {(void **)&hb->d_opts, (int64_t)sizeof(HOpt) * nopt},
      {(void **)&hb->d_spots, 8 * so},
      {(void **)&hb->d_vars, 8 * vo},
      {(void **)&hb->d_sp, 8 * SP_NF * so},
      {(void **)&hb->d_vt, 8 * VT_NF * vo},
      {(void **)&hb->d_spr, 8 * 16 * so},
      {(void **)&hb->d_state, 8 * off},
      {(void **)&hb->d_w1, 8 * off},
      {(void **)&hb->d_y2, 8 * off},
      {(void **)&hb->d_rd0, 8 * off},
      {(void **)&hb->d_sp_row, 8 * so},
      {(void **)&hb->d_vt_row, 8 * vo},
      {(void **)&hb->d_stiles, (int64_t)sizeof(Tile) * hb->cap_stiles},
      {(void **)&hb->d_vtiles, (int64_t)sizeof(Tile) * hb->cap_vtiles},
      {(void **)&hb->d_ftiles, (int64_t)sizeof(Tile) * (int64_t)ft.size()},
      {(void **)&hb->d_base_dt, 8 * (int64_t)nopt},
      {(void **)&hb->d_slots, 16},
  };
  int64_t total_bytes = 0;
  for (const Part &q : parts) total_bytes += (q.bytes + 255) / 256 * 256;
  if (fdadi_arena_create(total_bytes, &hb->arena) != FDADI_OK) {
    const std::string msg = fdadi_last_error();
    free_hb(hb);
    set_error("fdadi_hb_create: " + msg);
    return FDADI_ERR_HIP;
  }
  for (const Part &q : parts) {
    double *d = nullptr;
    (void)fdadi_arena_alloc(hb->arena, (q.bytes + 7) / 8, &d);  // fits by construction
    *q.p = d;
  }
  hipError_t e = hipSuccess;
  auto up = [&](void *dst, const void *src, size_t bytes) {
    if (e == hipSuccess && bytes) e = hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice);
  };
  up(hb->d_opts, hb->h_opts.data(), sizeof(HOpt) * nopt);
  up(hb->d_spots, spots, sizeof(double) * so);
  up(hb->d_vars, vars, sizeof(double) * vo);
  up(hb->d_sp_row, sp_row.data(), sizeof(int64_t) * so);
  up(hb->d_vt_row, vt_row.data(), sizeof(int64_t) * vo);
  up(hb->d_ftiles, ft.data(), sizeof(Tile) * ft.size());
  up(hb->d_base_dt, hb->base_dt.data(), sizeof(double) * nopt);
  if (e == hipSuccess && build_spot_tiles(hb) != FDADI_OK) e = hipErrorUnknown;
  if (e == hipSuccess && build_var_tiles(hb) != FDADI_OK) e = hipErrorUnknown;
  if (e == hipSuccess && build_tables(hb, s) != FDADI_OK) e = hipErrorUnknown;
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) {
    free_hb(hb);
    set_error(std::string("fdadi_hb_create: ") + hipGetErrorString(e));
    return FDADI_ERR_HIP;
  }
  *out = hb;
  return FDADI_OK;
}

int fdadi_hb_destroy(fdadi_hb *hb) {
  free_hb(hb);
  return FDADI_OK;
}

int fdadi_hb_configure(fdadi_hb *hb, int scheme, double theta, double dt_scale, void *stream) {
  FDADI_REQUIRE(hb, FDADI_ERR_ARG, "fdadi_hb_configure: null engine");
  FDADI_REQUIRE(scheme >= FDADI_SCHEME_IMPLICIT && scheme <= FDADI_SCHEME_HV, FDADI_ERR_ARG,
                "fdadi_hb_configure: unknown scheme");
  FDADI_REQUIRE(dt_scale > 0, FDADI_ERR_ARG, "fdadi_hb_configure: dt_scale must be positive");
  hipStream_t s = as_stream(stream);
  // A captured graph stays valid while the scheme (the kernel sequence) is
  // unchanged: theta and dt live in device memory and are re-read each step.
  const bool keep_graph = scheme == hb->scheme;
  hb->scheme = scheme;
  hb->theta = theta;
  hb->dt_scale = dt_scale;
  hb->dev_scalars = false;
  FDADI_RET(refactor(hb, s));
  if (!keep_graph) {
    if (hb->gexec) {
      (void)hipGraphExecDestroy(hb->gexec);
      hb->gexec = nullptr;
    }
    if (hb->graph) {
      (void)hipGraphDestroy(hb->graph);
      hb->graph = nullptr;
    }
  }
  return FDADI_OK;
}

int fdadi_hb_configure_dev(fdadi_hb *hb, int scheme, const double *d_theta,
                           const double *d_dt_scale, void *stream) {
  FDADI_REQUIRE(hb && d_theta && d_dt_scale, FDADI_ERR_ARG,
                "fdadi_hb_configure_dev: bad arguments");
  FDADI_REQUIRE(scheme >= FDADI_SCHEME_IMPLICIT && scheme <= FDADI_SCHEME_HV, FDADI_ERR_ARG,
                "fdadi_hb_configure_dev: unknown scheme");
  const bool keep_graph = scheme == hb->scheme;
  hb->scheme = scheme;
  hb->dev_scalars = true;
  FDADI_RET(refactor(hb, as_stream(stream), d_theta, d_dt_scale));
  if (!keep_graph) {
    if (hb->gexec) {
      (void)hipGraphExecDestroy(hb->gexec);
      hb->gexec = nullptr;
    }
    if (hb->graph) {
      (void)hipGraphDestroy(hb->graph);
      hb->graph = nullptr;
    }
  }
  return FDADI_OK;
}

int fdadi_hb_update(fdadi_hb *hb, int32_t nopt, const fdadi_heston_option *opts,
                    const double *spots, const double *vars, void *stream) {
  FDADI_REQUIRE(hb && opts && spots && vars, FDADI_ERR_ARG, "fdadi_hb_update: bad arguments");
  FDADI_REQUIRE(nopt == hb->nopt, FDADI_ERR_ARG,
                "fdadi_hb_update: option count differs from the engine's");
  for (int k = 0; k < nopt; ++k)
    FDADI_REQUIRE(opts[k].nS == hb->h_opts[k].nS && opts[k].nv == hb->h_opts[k].nv,
                  FDADI_ERR_ARG,
                  "fdadi_hb_update: option " + std::to_string(k) + ": grid shape differs");
  hipStream_t s = as_stream(stream);
  for (int k = 0; k < nopt; ++k) {
    HOpt &o = hb->h_opts[k];
    const fdadi_heston_option &q = opts[k];
    o.r = q.r;
    o.kappa = q.kappa;
    o.theta = q.theta;
    o.sigma = q.sigma;
    o.rho = q.rho;
    o.dt = q.dt;
    o.barrier = q.barrier ? 1 : 0;
    hb->base_dt[k] = q.dt;
  }
  // The host arrays may be pageable: synchronous copies, after the stream's
  // earlier work (which may still read the tables) has finished.
  FDADI_TRY_HIP(hipStreamSynchronize(s));
  hb->opts_on_device = false;
  FDADI_TRY_HIP(hipMemcpy(hb->d_opts, hb->h_opts.data(), sizeof(HOpt) * nopt,
                          hipMemcpyHostToDevice));
  FDADI_TRY_HIP(hipMemcpy(hb->d_spots, spots, sizeof(double) * hb->sp_n, hipMemcpyHostToDevice));
  FDADI_TRY_HIP(hipMemcpy(hb->d_vars, vars, sizeof(double) * hb->vt_n, hipMemcpyHostToDevice));
  FDADI_TRY_HIP(hipMemcpy(hb->d_base_dt, hb->base_dt.data(), sizeof(double) * nopt,
                          hipMemcpyHostToDevice));
  FDADI_RET(build_tables(hb, s));
  if (hb->scheme >= 0) {
    if (hb->dev_scalars)
      FDADI_RET(refactor(hb, s, hb->d_slots, hb->d_slots + 1));
    else
      FDADI_RET(refactor(hb, s));
  }
  FDADI_TRY_HIP(hipStreamSynchronize(s));
  return FDADI_OK;
}

int fdadi_hb_update_dev(fdadi_hb *hb, const double *d_params, const double *d_spots,
                        const double *d_vars, void *stream) {
  FDADI_REQUIRE(hb && d_params, FDADI_ERR_ARG, "fdadi_hb_update_dev: bad arguments");
  hipStream_t s = as_stream(stream);
  hipLaunchKernelGGL(set_params_kernel, dim3(grid_for(hb->nopt, 64)), dim3(64), 0, s,
                     hb->d_opts, hb->nopt, d_params, hb->d_base_dt);
  FDADI_CHECK_LAUNCH();
  if (d_spots)
    FDADI_TRY_HIP(hipMemcpyAsync(hb->d_spots, d_spots, sizeof(double) * hb->sp_n,
                                 hipMemcpyDeviceToDevice, s));
  if (d_vars)
    FDADI_TRY_HIP(hipMemcpyAsync(hb->d_vars, d_vars, sizeof(double) * hb->vt_n,
                                 hipMemcpyDeviceToDevice, s));
  hb->opts_on_device = true;
  FDADI_RET(build_tables(hb, s));
  // theta and the dt multiplier of the configured scheme stay in d_slots
  if (hb->scheme >= 0) FDADI_RET(refactor(hb, s, hb->d_slots, hb->d_slots + 1));
  return FDADI_OK;
}

int fdadi_hb_call_payoff(fdadi_hb *hb, const double *d_strikes, void *stream) {
  FDADI_REQUIRE(hb && d_strikes, FDADI_ERR_ARG, "fdadi_hb_call_payoff: bad arguments");
  hipLaunchKernelGGL(call_payoff_kernel, dim3(hb->sp_n), dim3(128), 0, as_stream(stream),
                     hb->d_opts, hb->d_sp_row, hb->d_spots, hb->sp_n, d_strikes, hb->d_state);
  FDADI_CHECK_LAUNCH();
  return FDADI_OK;
}

int fdadi_hb_read_bicubic(const fdadi_hb *hb, const double *d_S0, const double *d_v0,
                          double *d_out, void *stream) {
  FDADI_REQUIRE(hb && d_S0 && d_v0 && d_out, FDADI_ERR_ARG,
                "fdadi_hb_read_bicubic: bad arguments");
  hipLaunchKernelGGL(read_bicubic_kernel, dim3(grid_for(hb->nopt, 64)), dim3(64), 0,
                     as_stream(stream), hb->d_opts, hb->nopt, hb->d_spots, hb->d_vars, hb->d_state,
                     d_S0, d_v0, d_out);
  FDADI_CHECK_LAUNCH();
  return FDADI_OK;
}

int fdadi_hb_state(fdadi_hb *hb, double **d_state, int64_t *total) {
  FDADI_REQUIRE(hb, FDADI_ERR_ARG, "fdadi_hb_state: null engine");
  if (d_state) *d_state = hb->d_state;
  if (total) *total = hb->total;
  return FDADI_OK;
}

int fdadi_hb_offsets(const fdadi_hb *hb, int64_t *offsets) {
  FDADI_REQUIRE(hb && offsets, FDADI_ERR_ARG, "fdadi_hb_offsets: bad arguments");
  for (int k = 0; k < hb->nopt; ++k) offsets[k] = hb->h_opts[k].off;
  return FDADI_OK;
}

int fdadi_hb_step(fdadi_hb *hb, int32_t nsteps, void *stream) {
  FDADI_REQUIRE(hb, FDADI_ERR_ARG, "fdadi_hb_step: null engine");
  FDADI_REQUIRE(nsteps >= 0, FDADI_ERR_ARG, "fdadi_hb_step: negative step count");
  hipStream_t s = as_stream(stream);
  for (int32_t n = 0; n < nsteps; ++n) FDADI_RET(step_once(hb, s));
  return FDADI_OK;
}

int fdadi_hb_step_timed(fdadi_hb *hb, int32_t nsteps, void *stream, double *stage_ms,
                        int32_t max_stages, int32_t *nstages) {
  FDADI_REQUIRE(hb && stage_ms && nstages && nsteps > 0, FDADI_ERR_ARG,
                "fdadi_hb_step_timed: bad arguments");
  // ADI stages per step (a stage is one launch per group of its sweep)
  FDADI_REQUIRE(hb->scheme >= 0, FDADI_ERR_STATE, "fdadi_hb_step_timed: engine not configured");
  const int per =
      hb->scheme == FDADI_SCHEME_DOUGLAS || hb->scheme == FDADI_SCHEME_IMPLICIT ? 2 : 4;
  FDADI_REQUIRE(per <= max_stages, FDADI_ERR_ARG, "fdadi_hb_step_timed: stage_ms too short");
  hipStream_t s = as_stream(stream);
  const size_t need = (size_t)2 * per * nsteps;
  while (hb->events.size() < need) {
    hipEvent_t e;
    FDADI_TRY_HIP(hipEventCreate(&e));
    hb->events.push_back(e);
  }
  StageEvents tm{hb->events.data(), 0};
  for (int32_t n = 0; n < nsteps; ++n) FDADI_RET(step_once(hb, s, &tm));
  FDADI_TRY_HIP(hipStreamSynchronize(s));
  for (int k = 0; k < per; ++k) stage_ms[k] = 0.0;
  for (int32_t n = 0; n < nsteps; ++n)
    for (int k = 0; k < per; ++k) {
      float ms = 0.f;
      const size_t b = (size_t)2 * (n * per + k);
      FDADI_TRY_HIP(hipEventElapsedTime(&ms, hb->events[b], hb->events[b + 1]));
      stage_ms[k] += ms;
    }
  *nstages = per;
  return FDADI_OK;
}

int fdadi_hb_capture(fdadi_hb *hb, int32_t nsteps, void *stream) {
  FDADI_REQUIRE(hb, FDADI_ERR_ARG, "fdadi_hb_capture: null engine");
  FDADI_REQUIRE(nsteps > 0, FDADI_ERR_ARG, "fdadi_hb_capture: step count must be positive");
  FDADI_REQUIRE(hb->scheme >= 0, FDADI_ERR_STATE, "fdadi_hb_capture: engine not configured");
  FDADI_REQUIRE(stream, FDADI_ERR_ARG, "fdadi_hb_capture: needs a created stream");
  hipStream_t s = as_stream(stream);
  if (hb->gexec) {
    (void)hipGraphExecDestroy(hb->gexec);
    hb->gexec = nullptr;
  }
  if (hb->graph) {
    (void)hipGraphDestroy(hb->graph);
    hb->graph = nullptr;
  }
  FDADI_TRY_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
  int st = FDADI_OK;
  for (int32_t n = 0; n < nsteps && st == FDADI_OK; ++n) st = step_once(hb, s);
  hipGraph_t g = nullptr;
  hipError_t e = hipStreamEndCapture(s, &g);
  if (st != FDADI_OK) {
    if (g) (void)hipGraphDestroy(g);
    return st;
  }
  if (e != hipSuccess) {
    set_error(std::string("fdadi_hb_capture: ") + hipGetErrorString(e));
    return FDADI_ERR_HIP;
  }
  hb->graph = g;
  FDADI_TRY_HIP(hipGraphInstantiate(&hb->gexec, g, nullptr, nullptr, 0));
  return FDADI_OK;
}

int fdadi_hb_capture_solve(fdadi_hb *hb, int scheme, double theta, int32_t smoothing,
                           int32_t nsteps, void *stream) {
  FDADI_REQUIRE(hb, FDADI_ERR_ARG, "fdadi_hb_capture_solve: null engine");
  FDADI_REQUIRE(scheme >= FDADI_SCHEME_IMPLICIT && scheme <= FDADI_SCHEME_HV, FDADI_ERR_ARG,
                "fdadi_hb_capture_solve: unknown scheme");
  FDADI_REQUIRE(smoothing >= 0 && nsteps > 0, FDADI_ERR_ARG,
                "fdadi_hb_capture_solve: smoothing >= 0 and a positive step count");
  FDADI_REQUIRE(stream, FDADI_ERR_ARG, "fdadi_hb_capture_solve: needs a created stream");
  hipStream_t s = as_stream(stream);
  drop_graph(hb);
  // the device copy of the options made current here: the capture records
  // kernels only (no host copy, no synchronisation)
  if (!hb->opts_on_device) {
    FDADI_TRY_HIP(hipMemcpyAsync(hb->d_opts, hb->h_opts.data(), sizeof(HOpt) * hb->nopt,
                                 hipMemcpyHostToDevice, s));
    FDADI_TRY_HIP(hipStreamSynchronize(s));
    hb->opts_on_device = true;
  }
  const int prev_scheme = hb->scheme;
  const double prev_theta = hb->theta, prev_scale = hb->dt_scale;
  const bool prev_dev = hb->dev_scalars;
  hb->dev_scalars = false;
  FDADI_TRY_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
  int st = FDADI_OK;
  if (smoothing > 0) {
    // 2 * smoothing implicit steps of half the step
    hb->scheme = FDADI_SCHEME_IMPLICIT;
    hb->theta = 1.0;
    hb->dt_scale = 0.5;
    st = refactor(hb, s, nullptr, nullptr, true);
    for (int32_t n = 0; n < 2 * smoothing && st == FDADI_OK; ++n) st = step_once(hb, s);
  }
  if (st == FDADI_OK) {
    hb->scheme = scheme;
    hb->theta = theta;
    hb->dt_scale = 1.0;
    st = refactor(hb, s, nullptr, nullptr, true);
  }
  for (int32_t n = 0; n < nsteps && st == FDADI_OK; ++n) st = step_once(hb, s);
  hipGraph_t g = nullptr;
  hipError_t e = hipStreamEndCapture(s, &g);
  if (st != FDADI_OK || e != hipSuccess) {
    // nothing ran: the engine keeps its previous configuration
    if (g) (void)hipGraphDestroy(g);
    hb->scheme = prev_scheme;
    hb->theta = prev_theta;
    hb->dt_scale = prev_scale;
    hb->dev_scalars = prev_dev;
    if (st != FDADI_OK) return st;
    set_error(std::string("fdadi_hb_capture_solve: ") + hipGetErrorString(e));
    return FDADI_ERR_HIP;
  }
  hb->graph = g;
  FDADI_TRY_HIP(hipGraphInstantiate(&hb->gexec, g, nullptr, nullptr, 0));
  // the capture recorded the refactorisations without running them: run the
  // last one now, so that eager steps after this call see `scheme` as well
  return refactor(hb, s);
}

int fdadi_hb_replay(fdadi_hb *hb, void *stream) {
  FDADI_REQUIRE(hb && hb->gexec, FDADI_ERR_STATE, "fdadi_hb_replay: no captured graph");
  FDADI_TRY_HIP(hipGraphLaunch(hb->gexec, as_stream(stream)));
  return FDADI_OK;
}

int fdadi_hb_set_shape(fdadi_hb *hb, int kind, int threads, int lines) {
  FDADI_REQUIRE(hb && (kind == 0 || kind == 1), FDADI_ERR_ARG, "fdadi_hb_set_shape: bad kind");
  FDADI_REQUIRE(kind == 0 || lines == 0, FDADI_ERR_UNSUPPORTED,
                "fdadi_hb_set_shape: variance tiles follow from the lanes per line (pass 0)");
  if (kind == 0) {
    FDADI_REQUIRE(threads == -1 || threads == 0 || threads == 64 || threads == 128 ||
                      threads == 256 || threads == 512,
                  FDADI_ERR_ARG,
                  "fdadi_hb_set_shape: threads must be a power of two in [64, 512], 0 or -1");
    const int nl = lines == 0 ? 4 : lines;
    if (nl == 32) {
      // the last column must fall on a tile's last lane (see from_prev2_col)
      for (const HOpt &o : hb->h_opts)
        FDADI_REQUIRE(o.nv >= 32, FDADI_ERR_ARG,
                      "fdadi_hb_set_shape: 32-column spot tiles need at least 32 variance nodes");
    }
    if (threads == -1) {
      int t = 0, ml = 0;
      FDADI_RET(spot_shape(1, 0, nl, &t, &ml));  // validates nl
      const auto c = spot_candidates(nl);
      for (const HOpt &o : hb->h_opts)
        FDADI_REQUIRE(spot_group_of(c, nl, o.nS) >= 0, FDADI_ERR_ARG,
                      "fdadi_hb_set_shape: no spot shape covers a line of " +
                          std::to_string(o.nS) + " nodes");
      hb->spot_split = true;
    } else {
      int t = 0, ml = 0;
      FDADI_RET(spot_shape(hb->nSmax, threads, nl, &t, &ml));
      hb->spot_split = false;
      hb->spot_threads = t;
      hb->spot_maxl = ml;
    }
    hb->spot_nl = nl;
    FDADI_RET(build_spot_tiles(hb));
  } else {
    // kind 1: `threads` = lanes per variance line (power of two <= 64), or
    // -1: per option, the fewest lanes that cover its line
    if (threads == -1) {
      hb->var_split = true;
    } else {
      const int t = threads == 0 ? var_tpl_for(hb->nvmax) : threads;
      FDADI_REQUIRE(t >= 1 && t <= 64 && (t & (t - 1)) == 0, FDADI_ERR_ARG,
                    "fdadi_hb_set_shape: lanes per variance line must be a power of two <= 64");
      FDADI_REQUIRE((int64_t)t * kMAXL >= hb->nvmax, FDADI_ERR_ARG,
                    "fdadi_hb_set_shape: too few lanes for the longest variance line");
      hb->var_split = false;
      hb->var_tpl = t;
      hb->var_rows = 256 / t;
    }
    FDADI_RET(build_var_tiles(hb));
  }
  if (hb->gexec) {
    (void)hipGraphExecDestroy(hb->gexec);
    hb->gexec = nullptr;
  }
  if (hb->graph) {
    (void)hipGraphDestroy(hb->graph);
    hb->graph = nullptr;
  }
  return FDADI_OK;
}

int fdadi_hb_get_shape(const fdadi_hb *hb, int kind, int *threads, int *lines) {
  FDADI_REQUIRE(hb && (kind == 0 || kind == 1), FDADI_ERR_ARG, "fdadi_hb_get_shape: bad kind");
  if (threads)
    *threads = kind == 0 ? (hb->spot_split ? -1 : hb->spot_threads)
                         : (hb->var_split ? -1 : hb->var_tpl);
  if (lines) *lines = kind == 0 ? hb->spot_nl : (hb->var_split ? 0 : hb->var_rows);
  return FDADI_OK;
}

int fdadi_hb_launches_per_step(const fdadi_hb *hb, int *n) {
  FDADI_REQUIRE(hb && n, FDADI_ERR_ARG, "fdadi_hb_launches_per_step: bad arguments");
  // one launch per group of each sweep stage
  const int pair = (int)(hb->sgroups.size() + hb->vgroups.size());
  switch (hb->scheme) {
    case FDADI_SCHEME_DOUGLAS:
    case FDADI_SCHEME_IMPLICIT: *n = pair; break;
    default: *n = 2 * pair; break;
  }
  return FDADI_OK;
}

}  // extern "C"
