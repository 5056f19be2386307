// Fused batched 0D steady-state Newton solver, FP64, one 64-lane wavefront per instance.
//
// Reference: bte_0d3v_batched.steady_state_solve / get_rhs_and_jacobian
// (BESolver/python/bte_0d3v_batched.py:602-821, 882-979).  The reference forms the
// dense Jacobian J = Q^T L Q - mu I in the (n-1)-dim basis Q of u-perp and inverts it.
// Here the same Newton step is obtained from the bordered system in the original
// B-spline basis (L = M^-1 K):
//      (K - mu M) y = c M uhat + d M x,   uhat^T y = uhat^T x,   d = w.y - mu
// (d = 0 reproduces the reference's Jacobian, which omits the derivative of the
// growth term; d free gives the exact Jacobian).  The step is computed in residual form
// (a third right-hand side carries the compensated residual), see k_newton0d.  K - mu M is sparse: a narrow
// band (|offset| <= bw) plus the inelastic gain band.  Ordering the radial index
// from high to low energy puts the gain band strictly below the diagonal, so LU
// without pivoting keeps U inside the narrow band and the fill stays in L, which is
// never stored: the forward substitution runs during the factorisation.
//
// Data layout (all vectors in the permuted order i' = (np_r-1-p)*ns + l):
//   * shared per grid: operator values in row profile storage (columns
//     first_col[i]..min(i+bw, n-1)), nop arrays: C_0..C_{S-1}, C_Tg, A_E, M
//   * per instance: K profile (sum of the scaled operators, built for the whole
//     batch by k_prepare0d), U rows (WP doubles each).
// Slot mapping: slot s is row s % 16 of tile s / 16 (factor_tiles).  A host schedule
// assigns rows to slots so that no two rows share a slot whose columns are read at the
// same time.
//
// This header holds the device code and the launch templates; it is included by the
// translation units that instantiate them per window width (bz_solver0d_w<W>.hip) and by
// bz_solver0d.hip (C entry points, set-up and QoI kernels).  Everything but the argument
// structures and the per-window dispatch functions is TU-local (anonymous namespace).
#pragma once
#include <algorithm>
#include <type_traits>
#include "bz_common.h"
#include "../../include/bz.h"

namespace bz0d {

struct GridDev {
  int n, ns, npr, bw, S, nop, P, nslots, max_row;
  const int* first_col;     // [n]
  const int* prof_off;      // [n+1]
  const double* opprof;     // [nop][P]
  const int* slot_first;    // [nslots]
  const int* sched_next;    // [n]
  const double* muhat;      // [n]  M uhat
  const double* uhat;       // [n]
  const double* u;          // [n]
  const double* wsp;        // [nop-1][n]  W_m = Op_m^T M^-1 u (zero rows: not in the growth term)
  const double* mchol;      // [n][4]  banded Cholesky of M (permuted), L[i, i-d*ns]
  const int* chunk_levels;  // [ceil(n/W)] register levels alive in each W-step chunk
  const unsigned* ent_rc;   // [P] (row << 16) | column of every profile entry
  int keep_mass;            // the staged mass factor has LDS of its own (set by the launch)
};

struct BatchDev {
  int B;
  const double* n0;         // [B]
  const double* Tg;         // [B]
  const double* E;          // [B]
  const double* ns_by_n0;   // [S][B]
  double* x;                // (n, B) original order, in/out
  double* kprof;            // [B][P] scratch
  double* urows;            // [B][n][WP] scratch
  double* vec;              // [B][4][n] scratch (row 0: growth vector of the instance)
  int* iters;               // [B]
  int* status;              // [B]  0 converged, 1 max_iter, 2 line search failed
  double* res_abs;          // [B]
  double* res0;             // [B]
  double atol, rtol, alpha_min, alpha_rho, ls_c;
  int max_iter, mode;       // mode 0: reference Jacobian (d = 0), 1: exact Jacobian
  double tg_scale;          // coefficient of C_Tg is n0 * Tg * tg_scale
  const double* tol_abs;    // [B] per-instance absolute tolerance, or null: atol + rtol * r0
  double* lprof;            // [B][P] stored L factor (transient step), or null
};

struct EEDev {
  const double* ccA;    // [npr][7][7][ns][ns][ns]
  const double* ccB;
  const double* h;      // (B, n) original order
  const double* g;
  const double* negam;  // [B]
  const double* h_lo;   // (B, n) or null
  const double* g_lo;
};

// Per-window dispatch (one translation unit per window width W, the instantiated tile counts
// of that window): steady Newton (ee: NULL or the frozen e-e potentials), transient step,
// e-e factorisation and preconditioner application.  Each returns BZ_EINVAL when g.nslots
// needs more tiles than the largest instance has.
#define BZ0D_DECLARE_WINDOW(W)                                                                         \
  int steady_w##W(const GridDev& g, const BatchDev& b, hipStream_t s, const EEDev* ee);               \
  int transient_w##W(const GridDev& g, const BatchDev& b, double cdt, const double* ustart, double* avg, \
                     hipStream_t s);                                                                   \
  int ee_factor_w##W(const GridDev& g, const BatchDev& b, const int* active, double* lprof, double* z1, \
                     double* s1, hipStream_t s);                                                       \
  int ee_apply_w##W(const GridDev& g, const BatchDev& b, const int* active, const double* lprof,       \
                    const double* z1, const double* s1, const double* v, double* out, double* outT,    \
                    hipStream_t s);
BZ0D_DECLARE_WINDOW(8)
BZ0D_DECLARE_WINDOW(11)
BZ0D_DECLARE_WINDOW(12)
BZ0D_DECLARE_WINDOW(17)
BZ0D_DECLARE_WINDOW(20)
#undef BZ0D_DECLARE_WINDOW

}  // namespace bz0d

namespace {

using namespace bz;
using namespace bz0d;

constexpr int kMaxOps = 16;
// rows of the per-instance work array b.vec (each n doubles): 0 growth vector w, 1 x, 2 M x,
// 3 third right-hand side, 4..10 the unshifted values of K on the band of M (row i, offset d: entry
// 7 i + d of the seven rows in k_newton0d, entry i of row 4 + d in k_newton0d_lane), 11 the Newton
// step
constexpr int kVecRows = 12;
// exact-Newton line search: residual evaluations per step, and the step length below which an
// accepted step counts as a stall
constexpr int kMaxTrials = 8;
constexpr double kStallAlpha = 1e-2;



__device__ __forceinline__ int orig_index(int i, int ns, int npr) {
  const int q = i / ns, l = i - q * ns;
  return (npr - 1 - q) * ns + l;
}

__device__ __forceinline__ double fast_rcp(double a) {
  double r = __builtin_amdgcn_rcp(a);
  r = fma(r, fma(-a, r, 1.0), r);
  r = fma(r, fma(-a, r, 1.0), r);
  return r;
}

// Compensated (s, e) += the pair of another lane.
template <int CTRL>
__device__ __forceinline__ void dd_reduce(double& s, double& e) {
#pragma clang fp contract(off)
  const double s2 = dpp_move<CTRL>(s), e2 = dpp_move<CTRL>(e);
  const double t = s + s2, z = t - s;
  const double er = (s - (t - z)) + (s2 - z);
  s = t;
  e = e + e2 + er;
}

// Pointers into LDS, marked as such: a function the compiler keeps out of line would
// otherwise access LDS with generic (flat) instructions, which also wait on global loads.
typedef __attribute__((address_space(3))) double lds_double;
typedef __attribute__((address_space(3))) int lds_int;
typedef __attribute__((address_space(1))) double glb_double;

__device__ __forceinline__ double dot(const double* __restrict__ a, const double* __restrict__ b, int n, int lane) {
  double s = 0.0;
  for (int i = lane; i < n; i += 64) s = fma(a[i], b[i], s);
  return wave_sum(s);
}

// y = M x from the M profile (M is l-block diagonal, radial 7-band: columns i + d*ns, |d| <= 3).
__device__ void mass_matvec(int n, int ns, const double* __restrict__ mprof, const int2* __restrict__ rt,
                            const double* __restrict__ x, double* __restrict__ y, int lane) {
  for (int i = lane; i < n; i += 64) {
    const int base = rt[i].y;
    double s = 0.0;
#pragma unroll
    for (int d = -3; d <= 3; ++d) {
      const int c = i + d * ns;
      if (c >= 0 && c < n) s = fma(mprof[base + c], x[c], s);
    }
    y[i] = s;
  }
}

// ---------------------------------------------------------------- matrix-core profile LU
//
// The elimination runs in blocks of four pivots on the FP64 matrix cores.  Alive rows sit in
// slots, 16 to a tile; a tile holds, per lane 16 q + row (q = 0..3), column 4 h + q of its row
// for the column groups h = g (the panel) and g + 1 .. g + NG (what the upper bandwidth of four
// pivots reaches), one register each, and the three right-hand sides (q = which one).  That is
// the operand layout of v_mfma_f64_4x4x4f64 (A: lane i + 4 b + 16 k, B: lane j + 4 b + 16 k,
// D: lane j + 4 b + 16 i, b the block) and of v_mfma_f64_16x16x4f64 (A: lane i + 16 k, B: lane
// j + 16 k, accumulator element m of lane l: D[4 m + l / 16][l % 16]), so a panel register is
// an operand as it stands and nothing is transposed between steps:
//   multipliers  L^T = U11^-T panel^T         one 4x4x4 per tile
//   update       window^T -= U12^T L^T        one 16x16x4 per tile (ring and right-hand sides)
// The pivot rows of a block are published through LDS (they may sit in any slot); every lane
// factorises the 4 x 4 pivot block in registers and eliminates the column of U it supplies.
// Bound: the chain publish -> 4 x 4 LU (four reciprocals) -> two matrix instructions per block
// with one wavefront per SIMD, issue slots with two.  One row per lane and one pivot per step on
// the vector pipe took about 200 instructions per pivot for 28 multiply-adds; here it is about
// 75.
typedef double v4d __attribute__((ext_vector_type(4)));
typedef unsigned int v2u __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) v4d lds_v4d;

__device__ __forceinline__ double mfma4(double a, double b, double c) {
  return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ v4d mfma16(double a, double b, v4d c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Column groups of four right of a pivot block that its U rows reach (bw <= W - 1).
template <int W>
constexpr int trail_groups() { return (W + 2) / 4; }

// Rows of one instance's profile (or of its U rows) read through a buffer descriptor: an offset
// past the end reads as zero, which is how columns outside a row's profile are masked.
struct ProfileBuf {
  __amdgpu_buffer_rsrc_t r;
};
constexpr int kOutside = 0x40000000;       // beyond every profile (n < 32768, P * 8 < 2^30 checked on the host)

__device__ __forceinline__ ProfileBuf profile_buf(const double* p, int count) {
  return {__builtin_amdgcn_make_buffer_rsrc((void*)p, 0, count * 8, 0x00020000)};
}
__device__ __forceinline__ double buf_load(const ProfileBuf& b, int byte) {
  const v2u v = __builtin_amdgcn_raw_buffer_load_b64(b.r, byte, 0, 0);
  return __hiloint2double((int)v.y, (int)v.x);
}

// A store past the end is dropped.
__device__ __forceinline__ void buf_store(const ProfileBuf& b, int byte, double v) {
  v2u w;
  w.x = (unsigned)__double2loint(v);
  w.y = (unsigned)__double2hiint(v);
  __builtin_amdgcn_raw_buffer_store_b64(w, b.r, byte, 0, 0);
}

// The lane index hidden from the optimiser: what a phase derives from it is formed where the
// phase starts and not kept in registers (spilled, in the end) through all other phases.
__device__ __forceinline__ int fresh_lane(int lane) {
  asm volatile("" : "+v"(lane));
  return lane;
}

// The value taken out of its register at this point of the program, so that a load may refill the
// register (else the compiler may take it later, load into another one and copy at the loop edge,
// waiting for every load there).
__device__ __forceinline__ double moved(double v) {
  asm volatile("" : "+v"(v));
  return v;
}

__device__ __forceinline__ bool wave_any(bool p) { return __builtin_amdgcn_ballot_w64(p) != 0; }

__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Entries lane, lane + 64, ... of a global vector of n, eight loads in flight: f(i, value), i < n.
template <class F>
__device__ __forceinline__ void for_entries(const ProfileBuf& a, int n, int lane, F f) {
  for (int i0 = lane; i0 - lane < n; i0 += 512) {
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = buf_load(a, 8 * (i0 + 64 * u));
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (i0 + 64 * u < n) f(i0 + 64 * u, v[u]);
  }
}

// Dot product with a vector in LDS in compensated arithmetic (per-lane TwoProduct/TwoSum
// accumulation, then a compensated butterfly across the wavefront): about as accurate as a sum in
// twice FP64.
__device__ double dot_dd(const double* __restrict__ a, const double* __restrict__ b, int n, int lane) {
  double s = 0.0, c = 0.0;
  for_entries(profile_buf(a, n), n, lane, [&](int i, double v) { two_sum_acc(v, b[i], s, c); });
#pragma unroll
  for (int off = 32; off >= 16; off >>= 1) {
#pragma clang fp contract(off)
    const double s2 = __shfl_xor(s, off, 64), c2 = __shfl_xor(c, off, 64);
    const double t = s + s2, z = t - s;
    const double e = (s - (t - z)) + (s2 - z);
    s = t;
    c = c + c2 + e;
  }
  dd_reduce<kDppRor8>(s, c);
  dd_reduce<kDppRor4>(s, c);
  dd_reduce<kDppXor2>(s, c);
  dd_reduce<kDppXor1>(s, c);
  return s + c;
}

// Row sums of the instance profile, sum_c k[row][c] x[c], eight lanes to a row and eight rows at
// a time (64-byte segments of a row per load; rows taken harmonic by harmonic, so the eight rows
// of a pass have about the same length).  A step is 32 columns of the eight rows; the entries of
// the next two steps are in flight while one is summed (a step waited on memory for several
// times what its sums take).  DD: -k x in compensated arithmetic (s, e), else the plain sum in
// s.  fin(row, s, e) runs on one lane per row.
template <bool DD, class Fin>
__device__ __forceinline__ void row_sums(int n, int ns, int npr, int bw, int P, const int2* __restrict__ rt,
                                         const double* __restrict__ kp, const double* __restrict__ x_, int lane,
                                         Fin fin) {
  lane = fresh_lane(lane);
  const ProfileBuf kb = profile_buf(kp, P);
  const lds_double* x = (const lds_double*)x_;
  const int sub = lane & 7;
  int p = lane >> 3, l = 0, row = 0, c = 0, lc = -1, off = 0;      // the row whose entries are fetched next
  struct Step {
    double k[4];
    int c, row;
    bool last;
  };
  auto set_row = [&]() {
    while (p >= npr && l < ns) {
      p -= npr;
      ++l;
    }
    const bool ok = l < ns;
    row = ok ? p * ns + l : -1;
    const int2 v = rt[ok ? row : 0];
    lc = ok ? min(row + bw, n - 1) : -1;
    c = (v.x & 0xffff) + sub;
    off = 8 * v.y;
  };
  auto fetch = [&](Step& s) {
    s.c = c;
    s.row = row;
#pragma unroll
    for (int u = 0; u < 4; ++u) s.k[u] = buf_load(kb, c + 8 * u <= lc ? off + 8 * (c + 8 * u) : kOutside);
    s.last = !__any(c + 32 <= lc);
    if (s.last) {
      p += 8;
      set_row();
    } else {
      c += 32;
    }
  };
  double s = 0.0, e = 0.0;
  auto sum = [&](const Step& b) {
    double xv[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) xv[u] = x[min(b.c + 8 * u, n - 1)];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if constexpr (DD) two_sum_acc(-b.k[u], xv[u], s, e);
      else s = fma(b.k[u], xv[u], s);
    }
    if (b.last) {
      if constexpr (DD) {
        dd_reduce<kDppXor1>(s, e);
        dd_reduce<kDppXor2>(s, e);
        dd_reduce<kDppHalfMirror>(s, e);
      } else {
        s += dpp_move<kDppXor1>(s);
        s += dpp_move<kDppXor2>(s);
        s += dpp_move<kDppHalfMirror>(s);
      }
      if (b.row >= 0 && sub == 0) fin(b.row, s, e);
      s = 0.0;
      e = 0.0;
    }
  };
  Step b0, b1, b2;
  set_row();
  fetch(b0);
  fetch(b1);
  do {
    fetch(b2);
    sum(b0);
    fetch(b0);
    sum(b1);
    fetch(b1);
    sum(b2);
  } while (__any(b0.row >= 0));
}

// Row table, one int2 per row i: x = first profile column of i (low 16 bits) | (next row
// in i's slot << 16, -1 for none), y = profile offset of i minus that column (entries of
// the row are kprof[y + c]).
__device__ __forceinline__ void fill_rowtab(const GridDev& g, int2* __restrict__ rt, int lane) {
  for (int i = lane; i < g.n; i += 64) {
    const int fc = g.first_col[i];
    int2 v;
    v.x = (int)((unsigned)(fc & 0xffff) | ((unsigned)g.sched_next[i] << 16));
    v.y = g.prof_off[i] - fc;
    rt[i] = v;
  }
}

// The row whose columns a slot is reading.  Row i reads the groups first_col >> 2 .. (i >> 2) +
// NG; the schedule gives its successor no column before group (i >> 2) + NG + 1.  LEFT: only the
// columns left of the row's pivot block (the stored L factor).  The table entry of the row after
// it, and the entry value y of the row itself, are read from LDS when the row is taken up and
// used only later, so no step waits for them.
template <int NG, bool LEFT>
struct SlotRow {
  int row, ent, off8, end8;            // kNone without a row; ent: first column, next row << 16
  int tx, ty;                          // table entry of the next row
  double y;
  static constexpr int kNone = 0x7ffffff0;
  __device__ __forceinline__ int fc() const { return row != kNone ? ent & 0xffff : kNone; }
  __device__ __forceinline__ void take(const lds_int* rt, const lds_double* yl, int r, int n, int bw) {
    const bool ok = r >= 0;
    row = ok ? r : kNone;
    ent = ok ? tx : -65536;
    off8 = ty * 8;
    end8 = ok ? off8 + 8 * (LEFT ? r & ~3 : min(r + bw, n - 1) + 1) : (int)0x80000000;
    y = yl[max(r, 0)];
    tx = rt[2 * max(ent >> 16, 0)];
    ty = rt[2 * max(ent >> 16, 0) + 1];
  }
  __device__ __forceinline__ void init(const lds_int* rt, const lds_double* yl, int r, int n, int bw) {
    tx = rt[2 * max(r, 0)];
    ty = rt[2 * max(r, 0) + 1];
    take(rt, yl, r, n, bw);
  }
  __device__ __forceinline__ void advance(const lds_int* rt, const lds_double* yl, int h, int n, int bw) {
    const bool past = row < 4 * (h - NG);
    if (wave_any(past))
      if (past) take(rt, yl, ent >> 16, n, bw);
  }
  // Byte offset of the row's entry in column c8 / 8, past the end of the profile outside the row.
  // Without LEFT, columns left of the row's first read other rows' entries: their group is masked
  // when it becomes the panel.
  __device__ __forceinline__ int at(int c8) const {
    const int o = off8 + c8;
    return o < end8 && (!LEFT || c8 >= 8 * (ent & 0xffff)) ? o : kOutside;
  }
};

// 4 x 4 LU without pivoting of the pivot block a[k][c], and what the block step needs of it.
struct PivotBlock {
  double l10, l20, l21, l30, l31, l32;      // unit lower factor
  double u01, u02, u03, u12, u13, u23;      // strict upper factor
  double r0, r1, r2, r3;                    // reciprocals of the diagonal
  __device__ __forceinline__ void factor(v4d c0, v4d c1, v4d c2, v4d c3) {   // columns
    r0 = fast_rcp(c0[0]);
    l10 = c0[1] * r0; l20 = c0[2] * r0; l30 = c0[3] * r0;
    u01 = c1[0]; u02 = c2[0]; u03 = c3[0];
    const double a11 = fma(-l10, u01, c1[1]);
    r1 = fast_rcp(a11);
    u12 = fma(-l10, u02, c2[1]);
    u13 = fma(-l10, u03, c3[1]);
    l21 = fma(-l20, u01, c1[2]) * r1;
    l31 = fma(-l30, u01, c1[3]) * r1;
    const double a22 = fma(-l21, u12, fma(-l20, u02, c2[2]));
    r2 = fast_rcp(a22);
    u23 = fma(-l21, u13, fma(-l20, u03, c3[2]));
    l32 = fma(-l31, u12, fma(-l30, u02, c2[3])) * r2;
    r3 = fast_rcp(fma(-l32, u23, fma(-l31, u13, fma(-l30, u03, c3[3]))));
  }
};

// L^-1 of a block column v (four pivot rows): the substitution of the elimination itself
__device__ __forceinline__ v4d lower_apply(double l10, double l20, double l21, double l30, double l31, double l32,
                                           v4d v) {
  v4d u;
  u[0] = v[0];
  u[1] = fma(-l10, u[0], v[1]);
  u[2] = fma(-l21, u[1], fma(-l20, u[0], v[2]));
  u[3] = fma(-l32, u[2], fma(-l31, u[1], fma(-l30, u[0], v[3])));
  return u;
}

__device__ __forceinline__ double pick4(v4d v, int k) {
  const double a = (k & 1) ? v[1] : v[0], b = (k & 1) ? v[3] : v[2];
  return (k & 2) ? b : a;
}

// Factorise A = K - mu M (the instance profile already holds it; permuted order, no pivoting)
// and forward-eliminate NRHS (1 to 3) right-hand sides whose entry values are read from Y1, Y2,
// Y3 when a row enters its slot (never after its own pivot step); Y*[j] receive the eliminated
// values.  U goes to urows, row j at urows[j * WP]: offset d >= 1 holds -U[j][j + d] for columns
// right of the pivot block, and the block's own part holds U11^-1 (upper triangular, at the same
// offsets as U11).  SL: the multipliers of L at the profile positions of lout.
// s_piv: 16 (NG + 2) doubles of LDS, 32-byte aligned.
template <int W, int T, bool SL, int NRHS>
__device__ __forceinline__ void factor_tiles(const GridDev& g, const double* __restrict__ kprof, const int2* __restrict__ rt_,
                             double* __restrict__ y1_, double* __restrict__ y2_, double* __restrict__ y3_,
                             double* __restrict__ piv_, double* __restrict__ urows, int lane,
                             double* __restrict__ lout_ = nullptr) {
  lane = fresh_lane(lane);
  constexpr int NG = trail_groups<W>(), WP = (W + 1) & ~1, NX = NG > 4 ? NG - 4 : 0;
  constexpr bool Y16 = NG <= 3;                      // the right-hand sides ride in the 16x16x4 tile
  constexpr int YR = Y16 ? NG : 0;                   // as its element YR
  // With five groups the compiler, where it keeps part of a tile in accumulation registers, pairs the
  // publishing stores with wrong offsets (8, 6 and 4 doubles for 64, 48 and 32 in the assembly of
  // W = 20 with five tiles and more: an offset in units of eight divided by eight once more).
  // Volatile stores are not paired.
  using PubPtr = std::conditional_t<(NX > 0), volatile lds_double*, lds_double*>;
  const int n = g.n, bw = g.bw;
  const int q = lane >> 4, a16 = lane & 15, i4 = lane & 3;
  const ProfileBuf kb = profile_buf(kprof, g.P), ub = profile_buf(urows, n * WP);
  glb_double* lout = (glb_double*)lout_;
  const lds_int* rt = (const lds_int*)rt_;
  lds_double* piv = (lds_double*)piv_;
  lds_double* yq = (lds_double*)(q == 0 ? y1_ : (q == 1 || NRHS < 3) ? y2_ : y3_);        // entry values of this lane
  const int qq = a16 & 3, m = a16 >> 2;
  lds_double* yw = (lds_double*)(qq == 0 ? y1_ : (qq == 1 || NRHS < 3) ? y2_ : y3_);      // where eliminated ones go
  const bool ywl = Y16 ? (m == NG && qq < NRHS) : (a16 < NRHS);
  // where this lane's entry of U12 (per position u of the block in the ring) and of U11^-1 goes
  // inside the four U rows of a block
  int uo[NG], ux[NX ? NX * NG : 1];
#pragma unroll
  for (int u = 0; u < NG; ++u) {
    const int o = 4 * (m > u ? m - u : m - u + NG) + qq - q;
    uo[u] = (m < NG && o <= bw) ? (q * WP + o) * 8 : kOutside;
#pragma unroll
    for (int x = 0; x < NX; ++x) {
      const int ox = 4 * (4 + x > u ? 4 + x - u : 4 + x - u + NG) + i4 - q;
      ux[u * NX + x] = (a16 < 4 && ox <= bw) ? (q * WP + ox) * 8 : kOutside;
    }
  }
  const int ui_o = (a16 < 4 && i4 >= q) ? (q * WP + i4 - q) * 8 : kOutside;

  // Per tile: P the panel, R4 ring registers 0..3 (and the right-hand sides), RX ring register 4
  // and Y when they do not fit the 16x16x4 tile, F the groups read ahead.
  SlotRow<NG, false> st[T];
  int crow[T], cfc[T];                               // row being eliminated in the slot, its first column
  int coff[SL ? T : 1];                              // and profile offset (SL)
  double P[T], F[T][NG], RX[NX ? T : 1], Y[Y16 ? 1 : T];
  v4d R4[T];
#pragma unroll
  for (int t = 0; t < T; ++t) {
    const int slot = 16 * t + a16;
    const int row = slot < g.nslots ? g.slot_first[slot] : -1;
    st[t].init(rt, yq, row, n, bw);
    crow[t] = st[t].row;
    cfc[t] = st[t].fc();
    if constexpr (SL) coff[t] = st[t].off8 >> 3;
    const double y0 = (q < NRHS && row >= 0) ? st[t].y : 0.0;
    P[t] = q >= cfc[t] ? buf_load(kb, st[t].at(8 * q)) : 0.0;
    R4[t] = v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 1; s <= NG; ++s) {
      const double v = buf_load(kb, st[t].at(8 * (4 * s + q)));
      if (s % NG < 4) R4[t][s % NG < 4 ? s % NG : 0] = v;
      else RX[NX ? t : 0] = v;
    }
    if constexpr (Y16) R4[t][YR] = y0;
    else Y[t] = y0;
#pragma unroll
    for (int s = 0; s < NG; ++s) {
      st[t].advance(rt, yq, NG + 1 + s, n, bw);
      F[t][s] = buf_load(kb, st[t].at(8 * (4 * (NG + 1 + s) + q)));
    }
  }
  // Wait for the loads so far here, once: with them in flight at the loop entry, in another order
  // than on its edge, the compiler's wait analysis would put full waits into every round.
  // (s_waitcnt fields: vmcnt 0, expcnt 7, lgkmcnt 15.)
  __builtin_amdgcn_s_waitcnt(0x0F70);
  // Whole rounds of NG blocks (the ring positions are constants); a block past the last row
  // factorises the identity on empty tiles and its stores fall past the end.  An exit inside a
  // round would put register copies, and so a wait for every load ahead, on the loop edge.
  const int nb = (n + 3) >> 2;
  for (int g0 = 0; g0 < nb; g0 += NG) {
#pragma unroll
    for (int u = 0; u < NG; ++u) {
      const int gb = g0 + u;
      // --- publish the pivot rows: column col, row k of the block at piv[4 col + k]; the columns
      // are the panel, the ring groups in order and the right-hand sides.  Rows past n - 1 are
      // rows of the identity.
      if (4 * gb + 4 > n) {
        for (int e = lane; e < 16 * (NG + 2); e += 64)
          if (4 * gb + (e & 3) >= n) piv[e] = (e >> 2) == (e & 3) ? 1.0 : 0.0;
      }
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const int rel = crow[t] - 4 * gb;
        const bool mine = (unsigned)rel < 4u;
        if (wave_any(mine)) {
          if (mine) {
            PubPtr pk = (PubPtr)(piv + 4 * q + rel);
            pk[0] = P[t];
#pragma unroll
            for (int r = 0; r < NG; ++r) pk[16 * (r > u ? r - u : r - u + NG)] = r < 4 ? R4[t][r < 4 ? r : 0] : RX[NX ? t : 0];
            pk[16 * (NG + 1)] = Y16 ? R4[t][YR] : Y[Y16 ? 0 : t];
          }
          // The slot's next row, already the one being read: no column of it has arrived yet;
          // what the ring still holds is the old row's and is masked as it becomes the panel.
          const double y0 = (q < NRHS && st[t].row != SlotRow<NG, false>::kNone) ? st[t].y : 0.0;
          P[t] = mine ? 0.0 : P[t];
          if constexpr (Y16) R4[t][YR] = mine ? y0 : R4[t][YR];
          else Y[t] = mine ? y0 : Y[t];
          crow[t] = mine ? st[t].row : crow[t];
          cfc[t] = mine ? st[t].fc() : cfc[t];
          if constexpr (SL) coff[t] = mine ? st[t].off8 >> 3 : coff[t];
        }
      }
      // --- where the next group of every slot is read from
      int nx_o[T];
#pragma unroll
      for (int t = 0; t < T; ++t) {
        st[t].advance(rt, yq, gb + 2 * NG + 1, n, bw);
        nx_o[t] = st[t].at(8 * (4 * (gb + 2 * NG + 1) + q));
      }
      wave_lds_fence();
      const lds_v4d* pc = (const lds_v4d*)piv;
      // the column of U this lane supplies: ring register m (or the right-hand sides)
      const v4d vc = pc[4 * (m < NG ? (m > u ? m - u : m - u + NG) : NG + 1) + qq];
      v4d vx[NX + 1];
#pragma unroll
      for (int x = 0; x < NX; ++x) vx[x] = pc[4 * (4 + x > u ? 4 + x - u : 4 + x - u + NG) + i4];
      if constexpr (!Y16) vx[NX] = pc[4 * (NG + 1) + i4];
      PivotBlock pb;
      pb.factor(pc[0], pc[1], pc[2], pc[3]);
      // column i4 of U11^-1; this lane's entry is row q of it
      v4d xi;
      xi[3] = i4 == 3 ? pb.r3 : 0.0;
      xi[2] = fma(-pb.u23, xi[3], i4 == 2 ? 1.0 : 0.0) * pb.r2;
      xi[1] = fma(-pb.u12, xi[2], fma(-pb.u13, xi[3], i4 == 1 ? 1.0 : 0.0)) * pb.r1;
      xi[0] = fma(-pb.u01, xi[1], fma(-pb.u02, xi[2], fma(-pb.u03, xi[3], i4 == 0 ? 1.0 : 0.0))) * pb.r0;
      const double ui = pick4(xi, q);
      const double nu = -pick4(lower_apply(pb.l10, pb.l20, pb.l21, pb.l30, pb.l31, pb.l32, vc), q);
      double nx[NX + 1];
#pragma unroll
      for (int x = 0; x < NX + (Y16 ? 0 : 1); ++x)
        nx[x] = -pick4(lower_apply(pb.l10, pb.l20, pb.l21, pb.l30, pb.l31, pb.l32, vx[x]), q);
      // --- multipliers of every tile, then the updates (independent products back to back)
      double l[T];
#pragma unroll
      for (int t = 0; t < T; ++t) l[t] = mfma4(ui, P[t], 0.0);
#pragma unroll
      for (int t = 0; t < T; ++t) {
        R4[t] = mfma16(nu, l[t], R4[t]);
        if constexpr (NX > 0) RX[t] = mfma4(nx[0], l[t], RX[t]);
        if constexpr (!Y16) Y[t] = mfma4(nx[NX], l[t], Y[t]);
      }
      // --- U rows, U11^-1, eliminated right-hand sides
      buf_store(ub, uo[u] + gb * (4 * WP * 8), nu);
      buf_store(ub, ui_o + gb * (4 * WP * 8), ui);
#pragma unroll
      for (int x = 0; x < NX; ++x) buf_store(ub, ux[u * NX + x] + gb * (4 * WP * 8), nx[x]);
      const int j = 4 * gb + q;
      if (ywl && j < n) yw[j] = Y16 ? -nu : -nx[NX];
      if constexpr (SL) {
#pragma unroll
        for (int t = 0; t < T; ++t)
          if (4 * gb + q >= cfc[t]) lout[coff[t] + 4 * gb + q] = l[t];
        // the strict lower part of the pivot block's own factor
        if (a16 < q && j < n) {
          const int c = 4 * gb + a16;
          if (c >= (rt[2 * j] & 0xffff)) {
            const double lv = q == 1 ? pb.l10 : q == 2 ? (a16 == 0 ? pb.l20 : pb.l21)
                                                       : (a16 == 0 ? pb.l30 : a16 == 1 ? pb.l31 : pb.l32);
            lout[rt[2 * j + 1] + c] = lv;
          }
        }
      }
      // --- the next panel, the group read NG blocks ago into the ring, and the next read
      constexpr int RN = NG;
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const int r = (u + 1) % RN;
        const bool in = 4 * gb + 4 + q >= cfc[t];
        if (r < 4) {
          P[t] = in ? R4[t][r < 4 ? r : 0] : 0.0;
          R4[t][r < 4 ? r : 0] = moved(F[t][u]);
        } else {
          P[t] = in ? RX[NX ? t : 0] : 0.0;
          RX[NX ? t : 0] = moved(F[t][u]);
        }
        F[t][u] = buf_load(kb, nx_o[t]);
      }
    }
  }
}

// Forward solve L y = b with the unit lower factor stored by factor_tiles<SL = true>, one
// right-hand side in Y (entry values in, eliminated values out; in place).  The same slots and
// blocks with the stored multipliers streamed as panels: per tile and block one load and one
// 4x4x4 product.  The order of the operations on a row is the factorisation's.
template <int W, int T>
__device__ __forceinline__ void forward_tiles(const GridDev& g, const double* __restrict__ lprof, const int2* __restrict__ rt_,
                              double* __restrict__ y_, double* __restrict__ piv_, int lane) {
  lane = fresh_lane(lane);
  constexpr int NG = trail_groups<W>(), PF = NG + 2;        // at its pivot step a slot already reads its next row
  const int n = g.n, bw = g.bw;
  const int q = lane >> 4, a16 = lane & 15;
  const ProfileBuf lb = profile_buf(lprof, g.P);
  const lds_int* rt = (const lds_int*)rt_;
  lds_double* yl = (lds_double*)y_;
  lds_double* piv = (lds_double*)piv_;
  SlotRow<NG, true> st[T];
  int crow[T];
  double Y[T], F[T][PF], D[PF];
  // entry (q, a16) of the block's own unit lower factor, a16 < q
  auto diag = [&](int gb) -> double {
    const int j = 4 * gb + q, c = 4 * gb + a16;
    const int jr = min(j, n - 1);
    const bool ok = a16 < q && j < n && c >= (rt[2 * jr] & 0xffff);
    return buf_load(lb, ok ? 8 * (rt[2 * jr + 1] + c) : kOutside);
  };
#pragma unroll
  for (int t = 0; t < T; ++t) {
    const int slot = 16 * t + a16;
    const int row = slot < g.nslots ? g.slot_first[slot] : -1;
    st[t].init(rt, yl, row, n, bw);
    crow[t] = st[t].row;
    Y[t] = row >= 0 ? st[t].y : 0.0;
  }
#pragma unroll
  for (int s = 0; s < PF; ++s) {
#pragma unroll
    for (int t = 0; t < T; ++t) {
      st[t].advance(rt, yl, s, n, bw);
      F[t][s] = buf_load(lb, st[t].at(8 * (4 * s + q)));
    }
    D[s] = diag(s);
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);                 // as in factor_tiles
  const int nb = (n + 3) >> 2;
  for (int g0 = 0; g0 < nb; g0 += PF) {
#pragma unroll
    for (int u = 0; u < PF; ++u) {
      const int gb = g0 + u;
      if (lane < 4 && 4 * gb + lane >= n) piv[lane] = 0.0;
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const int rel = crow[t] - 4 * gb;
        const bool mine = (unsigned)rel < 4u;
        if (wave_any(mine)) {
          if (mine && q == 0) piv[rel] = Y[t];
          Y[t] = mine ? (st[t].row != SlotRow<NG, true>::kNone ? st[t].y : 0.0) : Y[t];
          crow[t] = mine ? st[t].row : crow[t];
        }
      }
      int nx_o[T];
#pragma unroll
      for (int t = 0; t < T; ++t) {
        st[t].advance(rt, yl, gb + PF, n, bw);
        nx_o[t] = st[t].at(8 * (4 * (gb + PF) + q));
      }
      wave_lds_fence();
      const v4d v = *(const lds_v4d*)piv;
      auto rl = [&](int k, int c) -> double {
        const int l = 16 * k + c;
        return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(D[u]), l),
                                __builtin_amdgcn_readlane(__double2loint(D[u]), l));
      };
      const v4d y = lower_apply(rl(1, 0), rl(2, 0), rl(2, 1), rl(3, 0), rl(3, 1), rl(3, 2), v);
      const double yk = pick4(y, q);
      if (a16 == 0 && 4 * gb + q < n) yl[4 * gb + q] = yk;
#pragma unroll
      for (int t = 0; t < T; ++t) {
        Y[t] = mfma4(-yk, F[t][u], Y[t]);
        F[t][u] = buf_load(lb, nx_o[t]);
      }
      D[u] = diag(gb + PF);
    }
  }
}

// Back substitution U z = y for the NRHS right-hand sides held in Y1/Y2(/Y3) (in place), blocks
// of four rows: z_g = U11^-1 (y_g - sum_s U_(g,g+s) z_(g+s)), every product one 4x4x4 whose
// result is the next one's operand as it stands; only two of them wait on the block before.
template <int W, int NRHS>
__device__ __forceinline__ void back_tiles(const GridDev& g, const double* __restrict__ urows, double* __restrict__ Y1,
                           double* __restrict__ Y2, double* __restrict__ Y3, int lane) {
  lane = fresh_lane(lane);
  constexpr int NG = trail_groups<W>(), WP = (W + 1) & ~1, PD = NG <= 3 ? 2 * NG : NG;
  const int n = g.n, bw = g.bw;
  const int q = lane >> 4, j4 = lane & 3, b4 = (lane >> 2) & 3;
  const ProfileBuf ub = profile_buf(urows, n * WP);
  lds_double* yj = (lds_double*)(j4 == 0 || NRHS < 2 ? Y1 : (j4 == 1 || NRHS < 3) ? Y2 : Y3);
  const bool live = j4 < NRHS;
  // operand A[i][k]: lane i + 4 b + 16 k; byte offsets inside a block's four rows
  int uo[NG + 1];
  uo[0] = q >= j4 ? (j4 * WP + q - j4) * 8 : kOutside;
#pragma unroll
  for (int s = 1; s <= NG; ++s) uo[s] = 4 * s + q - j4 <= bw ? (j4 * WP + 4 * s + q - j4) * 8 : kOutside;
  const int nb = (n + 3) >> 2;
  const int nu = (nb + PD - 1) / PD * PD;             // blocks past the last read as zero rows
  double A[PD][NG + 1], Z[NG];
#pragma unroll
  for (int s = 0; s < NG; ++s) Z[s] = 0.0;
  // in the order of the loop, so that the compiler's wait analysis sees one order
#pragma unroll
  for (int u = PD - 1; u >= 0; --u) {
#pragma unroll
    for (int s = NG; s >= 0; --s) A[u][s] = buf_load(ub, uo[s] + (nu - PD + u) * (4 * WP * 8));
    __builtin_amdgcn_sched_barrier(0);
  }
  // Rows past the last have zero rows of U, U11^-1 among them, so any finite value does there.
  auto rhs = [&](int gb) -> double { return yj[min(max(4 * gb + q, 0), n - 1)]; };
  double yn = rhs(nu - 1), yn2 = rhs(nu - 2);
  for (int g0 = nu - PD; g0 >= 0; g0 -= PD) {
#pragma unroll
    for (int u = PD - 1; u >= 0; --u) {
      const int gb = g0 + u;
      double acc = yn;
      yn = yn2;
      yn2 = rhs(gb - 2);
#pragma unroll
      for (int s = NG; s >= 1; --s) acc = mfma4(A[u][s], Z[(u + s) % NG], acc);
      const double z = mfma4(A[u][0], acc, 0.0);
      Z[u % NG] = z;
      if (b4 == 0 && live && 4 * gb + q < n) yj[4 * gb + q] = z;
      // rows of block gb - PD; a negative block is past the end as an unsigned offset
#pragma unroll
      for (int s = NG; s >= 0; --s) A[u][s] = buf_load(ub, uo[s] + (gb - PD) * (4 * WP * 8));
    }
  }
}

// The radial mass Cholesky factor staged for mass_solve, rows of four: lc[4 q + d] for d <= q % 4
// is entry (q, q - d) of the inverse of the 4 x 4 diagonal block that row q lies in, for d > q % 4
// the factor's own entry L[q, q - d] (zero before the first column); rows past the last are zero.
// One lane per block, 16 doubles a block.
__device__ void stage_mass(const GridDev& g, double* __restrict__ lc, int lane) {
  lane = fresh_lane(lane);
  const int nb = (g.npr + 3) >> 2;
  for (int b = lane; b < nb; b += 64) {
    double L[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int q = 4 * b + i;
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const double v = g.mchol[(size_t)(min(q, g.npr - 1) * g.ns) * 4 + d];
        L[i][d] = q >= g.npr ? (d == 0 ? 1.0 : 0.0) : (q - d >= 0 ? v : 0.0);
      }
    }
    const double i0 = 1.0 / L[0][0], i1 = 1.0 / L[1][0], i2 = 1.0 / L[2][0], i3 = 1.0 / L[3][0];
    const double x10 = -(L[1][1] * i0) * i1;
    const double x21 = -(L[2][1] * i1) * i2;
    const double x20 = -fma(L[2][2], i0, L[2][1] * x10) * i2;
    const double x32 = -(L[3][1] * i2) * i3;
    const double x31 = -fma(L[3][2], i1, L[3][1] * x21) * i3;
    const double x30 = -fma(L[3][3], i0, fma(L[3][2], x10, L[3][1] * x20)) * i3;
    const double o[4][4] = {{i0, L[0][1], L[0][2], L[0][3]},
                            {i1, x10, L[1][2], L[1][3]},
                            {i2, x21, x20, L[2][3]},
                            {i3, x32, x31, x30}};
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int d = 0; d < 4; ++d) lc[16 * b + 4 * i + d] = 4 * b + i < g.npr ? o[i][d] : 0.0;
  }
}

// In-place solve M z = b in the permuted order: every l-block (stride ns) is the reversed radial
// mass block with half bandwidth 3, lc from stage_mass.  Blocks of four rows as 4x4x4 matrix
// products, the harmonics in the columns (ns <= 16): y_g = D_g (b_g - S_g y_(g-1)), then
// z_g = D_g^T (y_g - S_(g+1)^T z_(g+1)); the result of a product is the next one's operand as it
// stands, so a block waits on two products (about 260 dependent steps of four multiply-adds and
// their LDS reads before).
__device__ void mass_solve(int ns, int npr, const double* __restrict__ lc_, double* __restrict__ b_, int lane) {
  lane = fresh_lane(lane);
  const lds_double* lc = (const lds_double*)lc_;
  lds_double* b = (lds_double*)b_;
  constexpr int CH = 8;                               // blocks whose operands are read together
  const int i = lane & 3, k = lane >> 4, col = lane & 15;
  const int nb = (npr + 3) >> 2;
  // Operands A[i][k]: -S_g at (row i, offset 4 + i - k) where i < k, D_g at (i, i - k) where
  // i >= k, and the transposes; rows past the last are zero, the first block's S is zero.
  const int oS = 4 * i + ((4 + i - k) & 3), oD = 4 * i + ((i - k) & 3);
  const int oSt = 4 * k + ((4 + k - i) & 3), oDt = 4 * k + ((k - i) & 3);
  const double mS = i < k ? -1.0 : 0.0, mD = i >= k ? 1.0 : 0.0;
  const double mSt = k < i ? -1.0 : 0.0, mDt = k >= i ? 1.0 : 0.0;
  const int cc = min(col, ns - 1);
  auto at = [&](int g) -> int { return max(0, min(4 * g + k, npr - 1)) * ns + cc; };
  auto put = [&](int g, double v) {
    if (g >= 0 && 4 * g + k < npr && col < ns) b[(4 * g + k) * ns + col] = v;
  };
  double y = 0.0;
  for (int g0 = 0; g0 < nb; g0 += CH) {
    double S[CH], D[CH], v[CH];
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int g = min(g0 + u, nb - 1);
      S[u] = lc[16 * g + oS];
      D[u] = lc[16 * g + oD];
      v[u] = b[at(g)];
    }
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      y = mfma4(D[u] * mD, mfma4(S[u] * mS, y, v[u]), 0.0);
      if (g0 + u < nb) put(g0 + u, y);
    }
  }
  double z = 0.0;
  for (int g0 = nb - 1; g0 >= 0; g0 -= CH) {
    double S[CH], D[CH], v[CH];
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int g = max(g0 - u, 0);
      S[u] = lc[16 * min(g + 1, nb - 1) + oSt];       // the last block multiplies z = 0
      D[u] = lc[16 * g + oDt];
      v[u] = b[at(g)];
    }
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      z = mfma4(D[u] * mDt, mfma4(S[u] * mSt, z, v[u]), 0.0);
      put(g0 - u, z);
    }
  }
}

constexpr int kPrepIG = 4;         // instances per thread of k_prepare0d

// Per-instance K profile (sum of the scaled operators) and growth vector, all instances at once.
__global__ __launch_bounds__(256) void k_prepare0d(GridDev g, BatchDev b) {
  // One thread per entry (the profile, then the growth vector), kPrepIG instances at a time, so that
  // an operator entry is read once for them and the instances' coefficients are scalars.  What
  // bounds it: the bytes of the profiles written, next to about nine FP64 instructions per operator
  // and entry.  A flat loop over all entries with a 64-bit division each took 448 us for 4096
  // instances of n = 387 (598 MB), this 314.
  const int nk = g.nop - 1, S = g.S;
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e >= g.P + g.n) return;
  const bool prof = e < g.P;
  const int i = prof ? e : e - g.P;
  const double* op = (prof ? g.opprof : g.wsp) + i;
  const size_t step = prof ? g.P : g.n;
  for (int i0 = blockIdx.y * kPrepIG; i0 < b.B; i0 += gridDim.y * kPrepIG) {
    // compensated: on the band of M the elastic and gas-temperature terms cancel at low
    // energy, and a plain sum would round K there at the scale of the terms
    double v[kPrepIG], c[kPrepIG];
#pragma unroll
    for (int u = 0; u < kPrepIG; ++u) v[u] = c[u] = 0.0;
    for (int m = 0; m < nk; ++m) {
      const double o = op[m * step];
#pragma unroll
      for (int u = 0; u < kPrepIG; ++u) {
        const int inst = min(i0 + u, b.B - 1);
        const double n0 = b.n0[inst];
        double cm;
        if (m < S) cm = n0 * b.ns_by_n0[(size_t)m * b.B + inst];
        else if (m == S) cm = n0 * b.Tg[inst] * b.tg_scale;
        else cm = b.E[inst];
        two_sum_acc(cm, o, v[u], c[u]);
      }
    }
#pragma unroll
    for (int u = 0; u < kPrepIG; ++u)
      if (i0 + u < b.B) {
        const size_t inst = i0 + u;
        double* out = prof ? b.kprof + inst * g.P : b.vec + inst * kVecRows * g.n;
        out[i] = v[u] + c[u];
      }
  }
}

// LDS: the published pivot block PIV first (32-byte aligned), four n-vectors R0..R3, the staged
// mass factor LC (mass_len doubles), then the row table (int2 per row).  Where LC would cost a
// wavefront per CU or pass 64 KB it shares R1..R2 (with a pad after R2) and is staged again for
// every residual.
__host__ __device__ __forceinline__ int mass_len(int npr) { return 16 * ((npr + 3) / 4); }
__host__ __device__ __forceinline__ int zpad(int n, int npr) {
  return mass_len(npr) > 2 * n ? mass_len(npr) - 2 * n : 0;
}

template <int W>
__host__ __device__ constexpr int piv_len() { return 16 * (trail_groups<W>() + 2); }

// Waves per SIMD the register state of T tiles leaves room for (a tile holds 2 NG + 2 doubles and
// its read position per lane); one wave may also use the accumulation registers.
template <int W, int T>
constexpr int tile_waves() { return T * (trail_groups<W>() + 2) <= 30 ? 2 : 1; }

// `vecs` n-vectors beside R1 and R2; sets g.keep_mass
template <int W>
size_t newton_lds_bytes(GridDev& g, int vecs) {
  const size_t rest = (size_t)((vecs + 2) * g.n + piv_len<W>()) * sizeof(double) + (size_t)g.n * sizeof(int2);
  const size_t keep = rest + (size_t)mass_len(g.npr) * sizeof(double), share = rest + (size_t)zpad(g.n, g.npr) * sizeof(double);
  constexpr size_t cu = 160 * 1024;
  g.keep_mass = keep <= 64 * 1024 && (cu / keep >= 8 || cu / keep == cu / share);
  return g.keep_mass ? keep : share;
}

// Profiles and U rows are read through 32-bit byte offsets below kOutside.
inline bool fits_offsets(const GridDev& g) { return g.P > 0 && g.P < kOutside / 8 && g.n < 32768; }

// |(I - uhat uhat^T) v|, v in LDS (two passes: explicit projection, no |v|^2 - (u.v)^2
// cancellation).
__device__ double proj_norm(const double* v, const ProfileBuf& uh, int n, int lane) {
  double su = 0.0;
  for_entries(uh, n, lane, [&](int i, double u) { su = fma(u, v[i], su); });
  su = wave_sum(su);
  double s2 = 0.0;
  for_entries(uh, n, lane, [&](int i, double u) {
    const double rp = v[i] - su * u;
    s2 = fma(rp, rp, s2);
  });
  return sqrt(wave_sum(s2));
}

// Fused Newton loop of one instance (one 64-lane wavefront), residual form.
//
// F(x) = M^-1 K x - mu(x) x, mu(x) = w.x, is the reference's residual before the projection
// P = I - uhat uhat^T (bte_0d3v_batched.py:779-783); with K' = K - mu M, F = M^-1 K' x.  The
// exact Newton step p with uhat.p = 0 satisfies K' p = c M uhat + d M x - K' x, d = w.p
// (the reference's Jacobian, mode 0, takes d = 0).
//  * Residual evaluation at a point x (row_pass): x is put on u.x = 1, mu = w.x (compensated
//    dot); one pass over the rows (eight lanes to a row) sets the band of M in the profile to
//    K' = K - mu M from the unshifted values of K (saved at the first pass; the difference is
//    formed exactly and rounded once) and forms, in compensated arithmetic (TwoProduct by fma,
//    TwoSum), the right-hand side y3 = c' M uhat - K' x for the coefficient c' of the step
//    that led to x; T = M^-1 y3, and P F = -P T.  Near convergence y3 -> 0 and is computed to
//    about twice FP64 precision, so the fixed point follows the residual rather than the
//    roundoff of the factorisation.
//  * Step: K' is factorised with the three right-hand sides M uhat, M x, y3:
//    z1 = K'^-1 M uhat, z2 = K'^-1 M x, delta = K'^-1 y3 = c' z1 - x, and
//    p = delta + a z1 + d z2 with (a, d) from uhat.p = 0 and w.p = d (mode 0: d = 0),
//    c = c' + a.  Near convergence K' is nearly singular with x close to its null vector:
//    z1 ~ x / c and z2 are large.  c' tracks c, so delta stays of the size of x; the M x
//    coefficient is not carried over (d -> 0 at the solution), so no large multiple of z2
//    enters delta only to cancel against d z2.
//  * Armijo backtracking (bte_0d3v_batched.py:936-952) on the true residual |P F(x + al p)|,
//    evaluated by the same row pass; the accepted trial's evaluation is the next iteration's.
//    (With z1 and z2 nearly parallel the 2x2 system cancels: a, d are then accurate only in
//    combination, and a residual predicted from them is not; the true residual is.)
// Global scratch rows of the instance (b.vec, kVecRows x n): 0 growth vector w, 1 x (the
// base point of the line search), 2 M x, 3 y3, 4..10 unshifted K on the band of M, 11 p.
template <int W, int T>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(tile_waves<W, T>()))) void k_newton0d(GridDev g, BatchDev b) {
  extern __shared__ __align__(32) double lds[];
  const int n = g.n, lane = threadIdx.x, inst = blockIdx.x;
  constexpr int WP = (W + 1) & ~1;
  double* PIV = lds;                                       // published pivot block
  double* R0 = PIV + piv_len<W>();                         // x; y3 -> delta -> p during a step
  double* R1 = R0 + n;                                     // M uhat -> z1
  double* R2 = R1 + n;                                     // M x -> z2
  double* LC = g.keep_mass ? R2 + n : R1;                  // staged mass factor (R1..R2 free in a residual)
  double* R3 = R2 + n + (g.keep_mass ? mass_len(g.npr) : zpad(n, g.npr));   // y3 -> T = M^-1 y3
  int2* SC = reinterpret_cast<int2*>(R3 + n);

  double* kprof = b.kprof + (size_t)inst * g.P;           // K, then K - mu M on the band of M
  const double* __restrict__ mprof = g.opprof + (size_t)(g.nop - 1) * g.P;
  const double* __restrict__ UH = g.uhat;
  double* WV = b.vec + (size_t)inst * kVecRows * n;
  double* XG = WV + n;
  double* MXG = XG + n;
  double* Y3G = MXG + n;
  double* KB0 = Y3G + n;                                   // [n][7] unshifted K on the band of M
  double* PG = KB0 + 7 * n;                                // the step p
  double* urows = b.urows + (size_t)inst * n * WP;

  // ---------------- row table into LDS, initial iterate (original (n,B) layout -> permuted)
  fill_rowtab(g, SC, lane);
  if (g.keep_mass) stage_mass(g, LC, lane);
  for (int i = lane; i < n; i += 64) R0[i] = b.x[(size_t)orig_index(i, g.ns, g.npr) * b.B + inst];
  const ProfileBuf mb = profile_buf(mprof, g.P), kpb = profile_buf(kprof, g.P), kbb = profile_buf(KB0, 7 * n),
                   muhb = profile_buf(g.muhat, n), uhb = profile_buf(UH, n), wvb = profile_buf(WV, n);
  __syncthreads();

  // residual at the point in R0 for the coefficient cq: x normalised in place, K' in the
  // profile, y3 in R3 and Y3G, M x in MXG, T = M^-1 y3 in R3; returns |P F(x)| = |P T|
  bool first = true;
  auto evaluate = [&](double cq) -> double {
    const double ux = dot_dd(g.u, R0, n, lane);
    for (int i = lane; i < n; i += 64) R0[i] = R0[i] / ux;
    __syncthreads();
    const double mu = dot_dd(WV, R0, n, lane);
    // the band of M, lane d of eight on offset d - 3 of a row, eight rows to a pass and the loads
    // of NB passes in flight
    constexpr int NB = 10;
    for (int i0 = lane >> 3; i0 - (lane >> 3) < n; i0 += 8 * NB) {
      const int d = lane & 7;
      double mv[NB], kv[NB];
      int eo[NB];
#pragma unroll
      for (int u = 0; u < NB; ++u) {
        const int i = i0 + 8 * u, c = i + (d - 3) * g.ns;
        const bool ok = i < n && d < 7 && c >= 0 && c < n;
        eo[u] = ok ? 8 * (SC[min(i, n - 1)].y + c) : kOutside;
        mv[u] = buf_load(mb, eo[u]);
        kv[u] = first ? buf_load(kpb, eo[u]) : buf_load(kbb, ok ? 8 * (7 * i + d) : kOutside);
      }
#pragma unroll
      for (int u = 0; u < NB; ++u) {
#pragma clang fp contract(off)
        const int i = i0 + 8 * u, c = i + (d - 3) * g.ns;
        const double xc = R0[max(0, min(c, n - 1))];         // weight zero outside the row
        if (first) buf_store(kbb, eo[u] != kOutside ? 8 * (7 * i + d) : kOutside, kv[u]);
        const double pm = mu * mv[u];
        const double pe = fma(mu, mv[u], -pm);
        const double hi = kv[u] - pm;                        // TwoSum(kv, -pm)
        const double z = hi - kv[u];
        const double lo = ((kv[u] - (hi - z)) + (-pm - z)) - pe;
        const double kr = hi + lo;                           // K' rounded once
        buf_store(kpb, eo[u], kr);
        double mx = mv[u] * xc, corr = (lo - (kr - hi)) * xc;  // K' - kr, to the residual
        mx += dpp_move<kDppXor1>(mx);
        corr += dpp_move<kDppXor1>(corr);
        mx += dpp_move<kDppXor2>(mx);
        corr += dpp_move<kDppXor2>(corr);
        mx += dpp_move<kDppHalfMirror>(mx);
        corr += dpp_move<kDppHalfMirror>(corr);
        if (d == 0 && i < n) {
          R2[i] = corr;
          MXG[i] = mx;
        }
      }
    }
    first = false;
    __syncthreads();                                       // K' of every row before any row is summed
    row_sums<true>(n, g.ns, g.npr, g.bw, g.P, SC, kprof, R0, lane, [&](int i, double s, double e) {
      R3[i] = s;
      R1[i] = e;
    });
    __syncthreads();
    for_entries(muhb, n, lane, [&](int i, double mh) {
      double s = R3[i], e = R1[i] - R2[i];
      two_sum_acc(cq, mh, s, e);
      const double y3 = s + e;
      R3[i] = y3;
      Y3G[i] = y3;
    });
    __syncthreads();
    if (!g.keep_mass) stage_mass(g, LC, lane);
    __syncthreads();
    mass_solve(g.ns, g.npr, LC, R3, lane);
    __syncthreads();
    return proj_norm(R3, uhb, n, lane);
  };

  double cp = 0.0;
  int stalls = 0;
  double rt = evaluate(0.0);
  const double r0 = rt;
  const double tol = b.tol_abs ? b.tol_abs[inst] : b.atol + b.rtol * r0;
  double rprev = rt;
  int it = 0, status = 1;

  for (;;) {
    // stopping test on the true residual of x.  Mode 0 follows the reference loop
    // (bte_0d3v_batched.py:926-957): its test uses |F| of the previous iterate, refreshed
    // after the step every 10th iteration.
    const double tval = (b.mode != 0 || it == 0 || ((it - 1) % 10) == 0) ? rt : rprev;
    rprev = rt;
    if (!(tval > tol)) { status = 0; break; }
    if (it >= b.max_iter) { status = 1; break; }
    // ---- right-hand sides and factorisation of K'
    for_entries(profile_buf(Y3G, n), n, lane, [&](int i, double v) {
      XG[i] = R0[i];
      R0[i] = v;
    });
    for_entries(muhb, n, lane, [&](int i, double v) { R1[i] = v; });
    for_entries(profile_buf(MXG, n), n, lane, [&](int i, double v) { R2[i] = v; });
    __syncthreads();
    factor_tiles<W, T, false, 3>(g, kprof, SC, R1, R2, R0, PIV, urows, lane);
    __syncthreads();
    back_tiles<W, 3>(g, urows, R1, R2, R0, lane);
    __syncthreads();
    // ---- step p = delta + a z1 + b z2
    double s11 = 0.0, s12 = 0.0, s13 = 0.0, wz1 = 0.0, wz2 = 0.0, wz3 = 0.0;
    for_entries(uhb, n, lane, [&](int i, double v) {
      s11 = fma(v, R1[i], s11);
      s12 = fma(v, R2[i], s12);
      s13 = fma(v, R0[i], s13);
    });
    for_entries(wvb, n, lane, [&](int i, double v) {
      wz1 = fma(v, R1[i], wz1);
      wz2 = fma(v, R2[i], wz2);
      wz3 = fma(v, R0[i], wz3);
    });
    s11 = wave_sum(s11); s12 = wave_sum(s12); s13 = wave_sum(s13);
    wz1 = wave_sum(wz1); wz2 = wave_sum(wz2); wz3 = wave_sum(wz3);
    double a, bb;
    if (b.mode == 0) {
      a = -s13 / s11;
      bb = 0.0;
    } else {
      const double s22 = wz2 - 1.0;
      const double e2 = -wz3;
      const double det = s11 * s22 - s12 * wz1;
      a = (-s13 * s22 - s12 * e2) / det;
      bb = (s11 * e2 + wz1 * s13) / det;
    }
    const double c_new = cp + a;
    for (int i = lane; i < n; i += 64) PG[i] = fma(a, R1[i], fma(bb, R2[i], R0[i]));
    __syncthreads();
    // ---- line search on the true residual at x + al p
    const double rbase = rt;
    const double ae2 = rt * rt;
    double alpha = 1.0;
    bool diverged = false;
    int trials = 0;
    for (;;) {
      for (int i = lane; i < n; i += 64) R0[i] = fma(alpha, PG[i], XG[i]);
      __syncthreads();
      const double rnew = evaluate(c_new);
      ++trials;
      if (!(0.5 * rnew * rnew > 0.5 * ae2 - b.ls_c * alpha * ae2)) {
        rt = rnew;
        break;
      }
      // exact Newton: at most kMaxTrials evaluations per step (a step that needs more does
      // not lead to a root; see the stall rule below)
      if (b.mode != 0 && trials >= kMaxTrials) { diverged = true; break; }
      if (b.mode == 0) {
        alpha *= b.alpha_rho;                                // the reference's backtracking
      } else {
        // exact Newton direction: slope of 0.5 |P F|^2 at 0 is -|P F|^2; the minimiser of the
        // quadratic through f(0), f'(0), f(alpha), kept within [alpha / 10, alpha_rho alpha]
        const double f0 = 0.5 * ae2, g0 = -ae2, f1 = 0.5 * rnew * rnew;
        const double den = 2.0 * (f1 - f0 - g0 * alpha);
        double aq = (den > 0.0) ? -g0 * alpha * alpha / den : b.alpha_rho * alpha;
        aq = fmin(fmax(aq, 0.1 * alpha), b.alpha_rho * alpha);
        alpha = (aq == aq) ? aq : b.alpha_rho * alpha;      // NaN guard
      }
      if (alpha < b.alpha_min) { diverged = true; break; }
    }
    if (diverged) {
      // back to x: its profile, y3 and M x are re-formed if the caller continues
      for (int i = lane; i < n; i += 64) R0[i] = XG[i];
      __syncthreads();
      status = 2;
      break;
    }
    cp = c_new;
    ++it;
    // exact Newton: two steps in a row accepted only at alpha < kStallAlpha, or reducing |r|
    // by less than 10 %, make a stalled iteration (measured on the 4096-instance batch: no
    // instance that converges backtracks below alpha = 0.3; the instances without a root of
    // the batched residual stall at |r| / |r0| ~ 1e-3 with such steps)
    if (b.mode != 0) {
      stalls = (alpha < kStallAlpha || rt > 0.9 * rbase) ? stalls + 1 : 0;
      if (stalls >= 2) { status = 2; break; }
    }
  }

  // ---------------- write back (original order)
  for (int i = lane; i < n; i += 64) b.x[(size_t)orig_index(i, g.ns, g.npr) * b.B + inst] = R0[i];
  if (lane == 0) {
    b.iters[inst] = it;
    b.status[inst] = status;
    b.res_abs[inst] = rt;
    b.res0[inst] = r0;
  }
}

// K profile += ne gamma_a [cc_a(., h) + cc_b(., g)]: the e-e operator of every instance at
// its current potentials, entry (row (p,q), column (k,l)) = sum_{r,s} cc[(p,q),(k,l),(r,s)] h[(r,s)]
// (the M-space form of cc = M^-1 (cc_a hl_op + cc_b gl_op), bte_0d3v_batched.py:462-468).
__global__ void k_ee_profile_add(GridDev g, BatchDev b, EEDev e) {
  const long total = (long)b.B * g.P;
  const int ns = g.ns, n = g.n, npr = g.npr;
  const int nc = ns * ns * ns;
  for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += (long)gridDim.x * blockDim.x) {
    const int inst = (int)(idx / g.P);
    const int ent = (int)(idx - (long)inst * g.P);
    const unsigned rc = g.ent_rc[ent];
    const int oi = orig_index((int)(rc >> 16), ns, npr), oj = orig_index((int)(rc & 0xffffu), ns, npr);
    const int p = oi / ns, q = oi - p * ns, k = oj / ns, l = oj - k * ns;
    const int dk = k - p;
    if (dk < -3 || dk > 3) continue;
    const double* hv = e.h + (size_t)inst * n;
    const double* gv = e.g + (size_t)inst * n;
    const double* hl = e.h_lo ? e.h_lo + (size_t)inst * n : nullptr;
    const double* gl = e.g_lo ? e.g_lo + (size_t)inst * n : nullptr;
    // Compensated sum: near v_max the products cancel to ~1e-6 of their size, so a plain
    // FP64 sum carries order-dependent errors that bias the e-e fixed point.
    double s = 0.0, c = 0.0;
    for (int dr = -3; dr <= 3; ++dr) {
      const int r = p + dr;
      if (r < 0 || r >= npr) continue;
      const size_t base = (((size_t)p * 7 + (dk + 3)) * 7 + (dr + 3)) * nc + (size_t)(q * ns + l) * ns;
      for (int ss = 0; ss < ns; ++ss) {
        two_sum_acc(e.ccA[base + ss], hv[r * ns + ss], s, c);
        two_sum_acc(e.ccB[base + ss], gv[r * ns + ss], s, c);
        if (hl) c = fma(e.ccA[base + ss], hl[r * ns + ss], fma(e.ccB[base + ss], gl[r * ns + ss], c));
      }
    }
    b.kprof[idx] = fma(e.negam[inst], s + c, b.kprof[idx]);
  }
}

inline int launch_prepare(const GridDev& g, const BatchDev& b, hipStream_t stream, const EEDev* ee = nullptr) {
  const dim3 grid((g.P + g.n + 255) / 256, std::min((b.B + kPrepIG - 1) / kPrepIG, 65535));
  hipLaunchKernelGGL(k_prepare0d, grid, dim3(256), 0, stream, g, b);
  BZ_LAUNCH_CHECK();
  if (ee) {
    const int blocks = (int)std::min<long>(((long)b.B * g.P + 255) / 256, 8192);
    hipLaunchKernelGGL(k_ee_profile_add, dim3(blocks), dim3(256), 0, stream, g, b, *ee);
    BZ_LAUNCH_CHECK();
  }
  return BZ_OK;
}

template <int W, int T>
int launch_newton(GridDev g, const BatchDev& b, hipStream_t stream, const EEDev* ee = nullptr) {
  const size_t lds = newton_lds_bytes<W>(g, 2);
  if (lds > 64 * 1024 || !fits_offsets(g)) return BZ_EINVAL;
  const int rc = launch_prepare(g, b, stream, ee);
  if (rc != BZ_OK) return rc;
  hipLaunchKernelGGL((k_newton0d<W, T>), dim3(b.B), dim3(64), lds, stream, g, b);
  BZ_LAUNCH_CHECK();
  return BZ_OK;
}

// One backward-Euler step of every instance (bte_0d3v_batched.solve "transient" and
// newton_solver_batched, bte_0d3v_batched.py:59-126, 1068-1139):
//   G(x) = (x - u) - c P (M^-1 K x - mu(x) x),  P = I - uhat uhat^T,  c = dt tau,
// with x - u kept orthogonal to uhat.  The reference's Newton iteration freezes the
// Jacobian I - c Q^T (M^-1 K - mu(u) I) Q at the start of the step and takes full steps.
// In the original basis that step is
//   (K - mu' M) z_G = M G,  (K - mu' M) z_u = M uhat,  mu' = mu(u) + 1/c,
//   x <- x + (z_G - gamma z_u) / c,  gamma = uhat.z_G / uhat.z_u,
// so every iteration factorises the same matrix K - mu' M with the two right-hand
// sides, and the iterates are the reference's.  The iteration count and the stopping
// test follow the reference loop (the convergence test of an iterate is made before
// its update, and the update is still applied), per instance.
template <int W, int T>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(tile_waves<W, T>()))) void k_transient0d(GridDev g, BatchDev b,
                                                                                           double cdt,
                                                                                           const double* ustart,
                                                                                           double* avg) {
  extern __shared__ __align__(32) double lds[];
  const int n = g.n, lane = threadIdx.x, inst = blockIdx.x;
  constexpr int WP = (W + 1) & ~1;
  double* PIV = lds;
  double* X = PIV + piv_len<W>();
  double* Z1 = X + n;
  double* Z2 = Z1 + n;
  double* LC = g.keep_mass ? Z2 + n : Z1;
  double* AV = Z2 + n + (g.keep_mass ? mass_len(g.npr) : zpad(n, g.npr));
  double* U0 = AV + n;
  int2* SC = reinterpret_cast<int2*>(U0 + n);

  double* kprof = b.kprof + (size_t)inst * g.P;
  const double* __restrict__ mprof = g.opprof + (size_t)(g.nop - 1) * g.P;
  const double* __restrict__ UH = g.uhat;
  const double* __restrict__ WV = b.vec + (size_t)inst * kVecRows * n;
  double* urows = b.urows + (size_t)inst * n * WP;

  fill_rowtab(g, SC, lane);
  if (g.keep_mass) stage_mass(g, LC, lane);
  for (int i = lane; i < n; i += 64) {
    const size_t o = (size_t)orig_index(i, g.ns, g.npr) * b.B + inst;
    X[i] = b.x[o];                              // initial iterate
    U0[i] = ustart ? ustart[o] : b.x[o];        // state at the start of the step
  }
  __syncthreads();

  const ProfileBuf uhb = profile_buf(UH, n), wvb = profile_buf(WV, n);
  // frozen shift: the profile holds K; make it K - mu' M, mu' from the start state
  const double mu0 = dot(WV, U0, n, lane);
  const double mup = mu0 + 1.0 / cdt;
  for (int k = lane; k < 7 * n; k += 64) {
    const int i = k / 7, dd = k - 7 * (k / 7) - 3;
    const int c = i + dd * g.ns;
    if (c >= 0 && c < n) {
      const int e = SC[i].y + c;
      kprof[e] = fma(-mup, mprof[e], kprof[e]);
    }
  }
  __syncthreads();

  // G(X) into AV; returns |G|
  auto residual = [&]() -> double {
    if (!g.keep_mass) stage_mass(g, LC, lane);
    row_sums<false>(n, g.ns, g.npr, g.bw, g.P, SC, kprof, X, lane, [&](int i, double s, double) { AV[i] = s; });
    __syncthreads();
    mass_solve(g.ns, g.npr, LC, AV, lane);
    __syncthreads();
    double mu = 0.0;
    for_entries(wvb, n, lane, [&](int i, double v) { mu = fma(v, X[i], mu); });
    mu = wave_sum(mu);
    double su = 0.0;
    for_entries(uhb, n, lane, [&](int i, double uh) {
      const double a = fma(mup, X[i], AV[i]) - mu * X[i];      // M^-1 K x - mu x
      AV[i] = a;
      su = fma(uh, a, su);
    });
    su = wave_sum(su);
    double s2 = 0.0;
    for_entries(uhb, n, lane, [&](int i, double uh) {
      const double gi = (X[i] - U0[i]) - cdt * (AV[i] - su * uh);
      AV[i] = gi;
      s2 = fma(gi, gi, s2);
    });
    __syncthreads();
    return sqrt(wave_sum(s2));
  };

  // With b.lprof the frozen matrix is factorised once (its multipliers stored in the
  // instance's profile positions of lprof, z_u = (K - mu' M)^-1 M uhat kept in vec row 1);
  // later iterations forward-solve with the stored L and back-substitute one right-hand side.
  double* lp = b.lprof ? b.lprof + (size_t)inst * g.P : nullptr;
  double* ZU = b.vec + (size_t)inst * kVecRows * n + n;
  double su = 1.0;
  const double r0 = residual();
  double rr = r0;
  bool conv = (r0 < b.atol);
  int it = 0;
  while (!conv && it < b.max_iter) {
    if (it > 0) rr = residual();
    conv = (rr / r0 < b.rtol) || (rr < b.atol);
    mass_matvec(n, g.ns, mprof, SC, AV, Z2, lane);
    if (it == 0 || lp == nullptr) {
      for (int i = lane; i < n; i += 64) Z1[i] = g.muhat[i];
      __syncthreads();
      if (lp) factor_tiles<W, T, true, 2>(g, kprof, SC, Z1, Z2, nullptr, PIV, urows, lane, lp);
      else factor_tiles<W, T, false, 2>(g, kprof, SC, Z1, Z2, nullptr, PIV, urows, lane);
      __syncthreads();
      back_tiles<W, 2>(g, urows, Z1, Z2, nullptr, lane);
      __syncthreads();
      su = dot(UH, Z1, n, lane);
      if (lp)
        for (int i = lane; i < n; i += 64) ZU[i] = Z1[i];
    } else {
      __syncthreads();
      forward_tiles<W, T>(g, lp, SC, Z2, PIV, lane);
      __syncthreads();
      back_tiles<W, 1>(g, urows, Z2, nullptr, nullptr, lane);
      for_entries(profile_buf(ZU, n), n, lane, [&](int i, double v) { Z1[i] = v; });
      __syncthreads();
    }
    double gam = 0.0;
    for_entries(uhb, n, lane, [&](int i, double uh) { gam = fma(uh, Z2[i], gam); });
    gam = wave_sum(gam) / su;
    const double ic = 1.0 / cdt;
    for (int i = lane; i < n; i += 64) X[i] = fma(ic, Z2[i] - gam * Z1[i], X[i]);
    __syncthreads();
    ++it;
  }

  for (int i = lane; i < n; i += 64) {
    const size_t o = (size_t)orig_index(i, g.ns, g.npr) * b.B + inst;
    b.x[o] = X[i];
    if (avg) avg[o] += U0[i] + X[i];
  }
  if (lane == 0) {
    b.iters[inst] = it;
    b.status[inst] = conv ? 0 : 1;
    b.res_abs[inst] = rr;
    b.res0[inst] = r0;
  }
}

template <int W, int T>
int launch_transient(GridDev g, const BatchDev& b, double cdt, const double* ustart, double* avg,
                     hipStream_t stream) {
  const size_t lds = newton_lds_bytes<W>(g, 3);
  if (lds > 64 * 1024 || !fits_offsets(g)) return BZ_EINVAL;
  const int rc = launch_prepare(g, b, stream);
  if (rc != BZ_OK) return rc;
  hipLaunchKernelGGL((k_transient0d<W, T>), dim3(b.B), dim3(64), lds, stream, g, b, cdt, ustart, avg);
  BZ_LAUNCH_CHECK();
  return BZ_OK;
}

}  // namespace

// Runs `launch<W, T>` with the smallest instantiated tile count T that holds g.nslots slots.
#define BZ0D_FOR_TILES(W_, launch, g, ...)                      \
  const int tiles = ((g).nslots + 15) / 16;                     \
  if (tiles <= 3) return launch<W_, 3>(g, __VA_ARGS__);         \
  if (tiles <= 5) return launch<W_, 5>(g, __VA_ARGS__);         \
  if (tiles <= 8) return launch<W_, 8>(g, __VA_ARGS__);         \
  if (tiles <= 12) return launch<W_, 12>(g, __VA_ARGS__);       \
  if (W_ >= 17 && tiles <= 16) return launch<W_, (W_ >= 17 ? 16 : 12)>(g, __VA_ARGS__); \
  return BZ_EINVAL;
