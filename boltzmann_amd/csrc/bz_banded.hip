// Batched triangular sweeps and products of the 1D3V solver (gfx950, FP64).
//
// Every kernel here works on many independent short recurrences (one per
// system: an x-line, a radial line or an angular line of the 1D3V state).  The
// systems are stored row by row, (bsz, N) with N contiguous, which the reference
// walks with one thread per system and stride-N loads.  Here one wavefront takes
// 64 systems and works through chunks of CH positions: coalesced loads (consecutive
// lanes read consecutive columns of one system) into registers, from there to LDS,
// and every lane sweeps its own system from LDS, keeping the last ND-1 solution
// values in registers; the loads of the next chunk are in flight meanwhile.  Tiles
// are stored in the order of the sweep, so lanes of either direction run the same code.
// Products (no recurrence) use one thread per output element.
#include <algorithm>

#include "bz_common.h"

namespace {

constexpr int TS = 64;   // systems per workgroup (one wavefront)

enum Kind { K_BIDIAG = 0, K_BANDED = 1, K_ADV_VR = 2, K_ADV_VT = 3, K_ADV_X = 4, K_XSTEP = 5 };

struct SweepArgs {
  // per-system coefficients (K_BIDIAG: diag, subdiag; K_BANDED: diags)
  const double* diag;
  const double* sdiag;
  const double* diags;
  // shared advection operators (K_ADV_*) and the per-system advection speed inputs
  const double* DL;
  const double* DR;
  const double* p0;      // vr: Ex   vt: Ex   x: vr
  const double* p1;      // vr: cos  vt: vr   x: cos
  double dt;
  const double* b;
  double* out;
  int bsz, N, lower;
  int Nr, Nvt, Nx;
  const int* lower_of;   // K_XSTEP: direction of system s is lower_of[s % Nvt]
};

// advection speed and direction of system s (rawkernel.py:183-192, 249-254, 316-322)
template <int KIND>
__device__ __forceinline__ void adv_speed(const SweepArgs& a, int s, double& av, bool& fwd) {
  if (KIND == K_ADV_VR) {
    const int ix = s / a.Nvt, ivt = s % a.Nvt;
    av = -a.p0[ix] * a.p1[ivt];
    fwd = av >= 0;
  } else if (KIND == K_ADV_VT) {
    const int ix = s / a.Nr, ivr = s % a.Nr;
    av = a.p0[ix] / a.p1[ivr];
    fwd = -av >= 0;
  } else {
    const int ivr = s / a.Nvt, ivt = s % a.Nvt;
    av = a.p0[ivr] * a.p1[ivt];
    fwd = av >= 0;
  }
}

constexpr int kOutside = 0x40000000;               // past the end of every output buffer
typedef unsigned v2u __attribute__((ext_vector_type(2)));

__device__ __forceinline__ void out_store(const __amdgpu_buffer_rsrc_t& b, int byte, double v) {
  v2u w;
  w.x = (unsigned)__double2loint(v);
  w.y = (unsigned)__double2hiint(v);
  __builtin_amdgcn_raw_buffer_store_b64(w, b, byte, 0, 0);
}

// The order of LDS operations within the one wavefront of a workgroup.
__device__ __forceinline__ void tile_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One wavefront per 64 systems.  What bounds it: with thousands of systems (banded, bidiagonal)
// the bytes of the coefficients, with few long ones (the radial advection lines) the instructions
// of N dependent positions.  So the next chunk's loads (CH * (NC + 1) per lane, 20 to 40 KB a
// wavefront) are issued before the sweep of the present one, the sweep is straight-line code
// over the CH positions (tiles in sweep order; positions past the end repeat the last one and are
// not stored, couplings to rows before the first are staged as zero), and the advection tables
// are staged through LDS with the chunk, with the reciprocal of the denominator off the chain and
// the quotient corrected by its remainder: 100 us against 99 without the correction, whose error
// against twice FP64 was 6 % above that of a division in the angular lines (9.5e-17 and 8.9e-17
// in the 2-norm; 8.9e-17 with it).  The general solves keep the division and its order.  Measured against staging, sweeping and
// storing in turn: 16 x 100 radial lines of 671 points, x and angular lines of the same state,
// 650 -> 100 us together; 20000 systems of 259, four diagonals, two solves, a product and a
// bidiagonal solve 909 -> 281 us.
template <int KIND, int ND, bool LONG>
__global__ __launch_bounds__(TS) void k_sweep(SweepArgs a) {
  constexpr bool BIDIAG = (KIND == K_BIDIAG || KIND == K_XSTEP);
  constexpr bool ADV = !BIDIAG && KIND != K_BANDED;
  constexpr int NC = (KIND == K_BANDED) ? ND : (BIDIAG ? 2 : 0);   // staged coefficient tiles
  constexpr int CH = NC > 5 ? 8 : 16;
  constexpr int ST = CH + 1;                                       // LDS row stride (doubles)
  constexpr int RP = TS / CH;                                      // systems per load instruction
  constexpr int NTD = ADV ? 2 * CH * ND : 1;                       // advection coefficients of a chunk
  constexpr int TL = (NTD + TS - 1) / TS;
  __shared__ double tb[TS * ST];
  __shared__ double tc[(NC > 0 ? NC : 1) * TS * ST];
  __shared__ double td[NTD];

  const int lane = threadIdx.x;
  const int sys0 = blockIdx.x * TS;
  const int s = sys0 + lane;
  const bool active = s < a.bsz;
  const int N = a.N;
  const int lr = lane / CH, lo = lane % CH;       // system and position of a lane's loads

  double av = 0.0;
  bool fwd = ADV ? true : (a.lower != 0);
  if (ADV && active) adv_speed<KIND>(a, s, av, fwd);
  if (KIND == K_XSTEP && active) fwd = a.lower_of[s % a.Nvt] != 0;
  const unsigned long long dirs = __ballot(fwd);  // direction of every system of the wavefront
  const double t = av * a.dt;

  double B[CH], C[NC > 0 ? NC : 1][CH], D[TL];
  auto fetch = [&](int k) {
    const int p = min(k * CH + lo, N - 1);
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int r = u * RP + lr;
      const bool f = (KIND == K_BANDED || KIND == K_BIDIAG) ? fwd : ((dirs >> r) & 1) != 0;
      const int c = f ? p : N - 1 - p;
      const size_t sr = min(sys0 + r, a.bsz - 1);
      B[u] = a.b[sr * N + c];
      if constexpr (KIND == K_BANDED) {
#pragma unroll
        for (int d = 0; d < ND; ++d) C[d][u] = a.diags[(sr * ND + d) * N + c];
      } else if constexpr (BIDIAG) {
        C[0][u] = a.diag[sr * N + c];
        // coupling of row c to its upwind neighbour: subdiag[c-1] (lower) or subdiag[c] (upper)
        const int sc = f ? c - 1 : c;
        C[1][u] = N > 1 ? a.sdiag[sr * (N - 1) + max(0, min(sc, N - 2))] : 0.0;
      }
    }
    if constexpr (ADV) {
      // coefficient d of position q: D[d][c -+ d], both directions
#pragma unroll
      for (int i = 0; i < TL; ++i) {
        const int e = min(lane + TS * i, NTD - 1);
        const int f = e / (CH * ND), q = (e / ND) % CH, d = e % ND;
        const int pp = min(k * CH + q, N - 1);
        const int j = max(0, min(f ? pp - d : N - 1 - pp + d, N - 1));
        D[i] = (f ? a.DL : a.DR)[(size_t)d * N + j];
        if (pp < d) D[i] = 0.0;
      }
    }
  };

  double y[ND > 1 ? ND - 1 : 1];
#pragma unroll
  for (int d = 0; d < (ND > 1 ? ND - 1 : 1); ++d) y[d] = 0.0;

  // Results past the end of a line or of the batch fall outside the buffer and are dropped: with a
  // branch for each store the compiler could not count the stores in flight and waited for all of
  // them before the next chunk.  (LONG: lines whose 64 rows pass the buffer's 2^30 bytes.)
  const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc(
      a.out + (size_t)sys0 * N, 0, LONG ? 0 : min(TS, a.bsz - sys0) * N * 8, 0x00020000);

  const int nchunk = (N + CH - 1) / CH;
  fetch(0);
  // the first loads complete here, so that the waits inside the loop count only its own
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(0x0F70);
  for (int k = 0; k < nchunk; ++k) {
    const int p = k * CH + lo;
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int at = (u * RP + lr) * ST + lo;
      // the x-step zeroes the inflow value of every system before its sweep
      tb[at] = (KIND == K_XSTEP && p == 0) ? 0.0 : B[u];
#pragma unroll
      for (int d = 0; d < NC; ++d) tc[d * TS * ST + at] = p >= d ? C[d][u] : 0.0;
    }
    if constexpr (ADV) {
#pragma unroll
      for (int i = 0; i < TL; ++i)
        if (lane + TS * i < NTD) td[lane + TS * i] = D[i];
    }
    tile_fence();
    fetch(k + 1);                       // past the last chunk: the last position again, not used
    const double* mt = td + (fwd ? CH * ND : 0);
    // The right-hand sides all at once (results go into the same tile) and, for the advection
    // lines, the coefficients off the recurrence.
    double rhs[CH], den[ADV ? CH : 1], rden[ADV ? CH : 1];
#pragma unroll
    for (int q = 0; q < CH; ++q) rhs[q] = tb[lane * ST + q];
    if constexpr (ADV) {
#pragma unroll
      for (int q = 0; q < CH; ++q) {
        den[q] = fma(t, mt[q * ND], 1.0);
        rden[q] = 1.0 / den[q];
      }
    }
#pragma unroll
    for (int q = 0; q < CH; ++q) {
      const double bi = rhs[q];
      double val;
      if constexpr (BIDIAG) {
        const double sv = tc[(TS + lane) * ST + q] * y[0];
        val = (bi - sv) / tc[lane * ST + q];
      } else if constexpr (KIND == K_BANDED) {
        double sv = 0.0;
#pragma unroll
        for (int d = 1; d < ND; ++d) sv += tc[(d * TS + lane) * ST + q] * y[d - 1];
        val = (bi - sv) / tc[lane * ST + q];
      } else {
        double sv = 0.0;
#pragma unroll
        for (int d = ND - 1; d >= 1; --d) sv = fma(mt[q * ND + d], y[d - 1], sv);
        // num / den, rounded once: a product with the rounded reciprocal and one correction by its
        // remainder (Markstein).  Infinities, overflow and a zero denominator leave no remainder
        // to correct by and are the product's.
        const double num = fma(-t, sv, bi);
        const double q0 = num * rden[q];
        const double q1 = fma(fma(-den[q], q0, num), rden[q], q0);
        val = q1 == q1 ? q1 : q0;
      }
#pragma unroll
      for (int d = (ND > 1 ? ND - 2 : 0); d >= 1; --d) y[d] = y[d - 1];
      y[0] = val;
      tb[lane * ST + q] = val;
    }
    tile_fence();
    double v[CH];
#pragma unroll
    for (int u = 0; u < CH; ++u) v[u] = tb[(u * RP + lr) * ST + lo];
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int r = u * RP + lr;
      const bool f = (KIND == K_BANDED || KIND == K_BIDIAG) ? fwd : ((dirs >> r) & 1) != 0;
      const int c = f ? p : N - 1 - p;
      if constexpr (!LONG) {
        out_store(out, p < N ? 8 * (r * N + c) : kOutside, v[u]);
      } else if (p < N && sys0 + r < a.bsz) {
        a.out[(size_t)(sys0 + r) * N + c] = v[u];
      }
    }
    tile_fence();
  }
}

// The x-step's bidiagonal upwind solves as a parallel scan: one wavefront per system.  Along
// the sweep the solution obeys o_p = a_p o_(p-1) + b_p (a_p = -s_p / d_p, b_p = rhs_p / d_p,
// a_0 = 0 and rhs_0 = 0: the inflow value is zeroed), a composition of affine maps.  Each
// lane composes the maps of PER consecutive positions, the 64 lane maps are combined by a
// shuffle scan (6 steps), and each lane then re-runs its positions from the value entering
// its segment.  Every map has |a_p| < 1 (upwind, diagonally dominant), so the re-association
// changes the result only at rounding level.  The sequential sweep needed N dependent steps
// per system on 64 systems per wavefront; this takes N / 64 per system.
template <int PER>
__global__ __launch_bounds__(64) void k_xstep_scan(const double* __restrict__ diag, const double* __restrict__ sdiag,
                                                   const int* __restrict__ lower_of, const double* __restrict__ rhs,
                                                   double* __restrict__ out, int bsz, int Nvt, int N) {
  const int s = blockIdx.x;
  const int lane = threadIdx.x;
  if (s >= bsz) return;
  const bool fwd = lower_of[s % Nvt] != 0;
  const size_t row = (size_t)s * N;
  const size_t srow = (size_t)s * (N - 1);
  double al[PER], be[PER];
  double A = 1.0, B = 0.0;
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int p = lane * PER + q;                 // position along the sweep
    double a = 1.0, b = 0.0;                      // identity beyond the end
    if (p < N) {
      const int c = fwd ? p : N - 1 - p;          // matrix row
      const double inv = 1.0 / diag[row + c];
      const int sc = fwd ? c - 1 : c;             // coupling to the upwind neighbour
      const double sv = (p >= 1) ? sdiag[srow + sc] : 0.0;
      const double r = (p >= 1) ? rhs[row + c] : 0.0;
      a = -sv * inv;
      b = r * inv;
    }
    al[q] = a;
    be[q] = b;
    B = fma(a, B, b);
    A = a * A;
  }
  // inclusive scan of the lane maps: (A, B) <- (A, B) o (A_prev, B_prev)
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const double Ap = __shfl_up(A, off, 64);
    const double Bp = __shfl_up(B, off, 64);
    if (lane >= off) {
      B = fma(A, Bp, B);
      A = A * Ap;
    }
  }
  // value entering this lane's segment: the end of the previous lane's (position 0 has a = 0)
  double o = __shfl_up(B, 1, 64);
  if (lane == 0) o = 0.0;
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int p = lane * PER + q;
    o = fma(al[q], o, be[q]);
    if (p < N) out[row + (fwd ? p : N - 1 - p)] = o;
  }
}

template <int KIND, int ND>
void launch_one(const SweepArgs& a, hipStream_t st) {
  const dim3 grid((a.bsz + TS - 1) / TS), block(TS);
  if (a.N < (1 << 20)) hipLaunchKernelGGL((k_sweep<KIND, ND, false>), grid, block, 0, st, a);
  else hipLaunchKernelGGL((k_sweep<KIND, ND, true>), grid, block, 0, st, a);
}

template <int KIND>
int launch_sweep(const SweepArgs& a, int nd, hipStream_t st) {
  switch (nd) {
    case 1: launch_one<KIND, 1>(a, st); break;
    case 2: launch_one<KIND, 2>(a, st); break;
    case 3: launch_one<KIND, 3>(a, st); break;
    case 4: launch_one<KIND, 4>(a, st); break;
    case 5: launch_one<KIND, 5>(a, st); break;
    case 6: launch_one<KIND, 6>(a, st); break;
    case 7: launch_one<KIND, 7>(a, st); break;
    case 8: launch_one<KIND, 8>(a, st); break;
    default: return BZ_EINVAL;
  }
  BZ_LAUNCH_CHECK();
  return BZ_OK;
}

template <int KIND>
int launch_bidiag(const SweepArgs& a, hipStream_t st) {
  launch_one<KIND, 2>(a, st);
  BZ_LAUNCH_CHECK();
  return BZ_OK;
}

// out[s, i] = sum_{d=0}^{ND-1} diags[s, d, i] * b[s, i -/+ d]  (rawkernel.py:111-166)
__global__ void k_banded_mv(const double* __restrict__ diags, const double* __restrict__ b, double* __restrict__ out,
                            int bsz, int nd, int N, int lower) {
  const size_t total = (size_t)bsz * N;
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (size_t)gridDim.x * blockDim.x) {
    const int s = (int)(e / N), i = (int)(e % N);
    const double* dg = diags + (size_t)s * nd * N;
    const double* bs = b + (size_t)s * N;
    double acc = 0.0;
    for (int d = 0; d < nd; ++d) {
      const int j = lower ? i - d : i + d;
      if (j < 0 || j >= N) break;
      acc += dg[(size_t)d * N + i] * bs[j];
    }
    out[e] = acc;
  }
}

// x = U^-1 b, U block upper triangular with unit diagonal blocks, BSR (indptr, indices,
// data[nnzb][bsz][bsz]); b and x column-major (n, nrhs).  One workgroup takes R right-hand
// sides (bsz*R threads); thread (r, q) owns row r of every block row of rhs q.
__global__ void k_bsr_upper_unit(const double* __restrict__ data, const int* __restrict__ indptr,
                                 const int* __restrict__ indices, int nbr, int nrhs, int bsz, int R,
                                 const double* __restrict__ b, double* __restrict__ x) {
  extern __shared__ double xs[];            // [R][bsz]
  const int r = threadIdx.x % bsz, q = threadIdx.x / bsz;
  const int rhs = blockIdx.x * R + q;
  const bool act = (q < R) && (rhs < nrhs);
  const size_t n = (size_t)nbr * bsz;
  for (int i = nbr - 1; i >= 0; --i) {
    double bi = act ? b[(size_t)rhs * n + (size_t)i * bsz + r] : 0.0;
    const int a0 = indptr[i], a1 = indptr[i + 1];
    for (int idx = a0; idx < a1; ++idx) {
      const int j = indices[idx];
      if (j <= i || j >= nbr) continue;      // diagonal (unit) and lower blocks are not used
      if (act) xs[q * bsz + r] = x[(size_t)rhs * n + (size_t)j * bsz + r];
      __syncthreads();
      if (act) {
        const double* A = data + (size_t)idx * bsz * bsz + (size_t)r * bsz;
        double sacc = 0.0;
        for (int c = 0; c < bsz; ++c) sacc += A[c] * xs[q * bsz + c];
        bi -= sacc;
      }
      __syncthreads();
    }
    if (act) x[(size_t)rhs * n + (size_t)i * bsz + r] = bi;
    __syncthreads();
  }
}

// out[r, l, x] = sum_i P[l, i] in[r, i, x]: P (m, k) applied to every (k, nx) slab of
// in (nr, k, nx); consecutive threads take consecutive x.
__global__ void k_slab_left_mult(const double* __restrict__ P, int m, int k, const double* __restrict__ in, int nr,
                                 int nx, double* __restrict__ out) {
  const size_t total = (size_t)nr * m * nx;
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (size_t)gridDim.x * blockDim.x) {
    const int x = (int)(e % nx);
    const size_t rl = e / nx;
    const int l = (int)(rl % m), r = (int)(rl / m);
    const double* src = in + (size_t)r * k * nx + x;
    const double* pl = P + (size_t)l * k;
    double acc = 0.0;
    for (int i = 0; i < k; ++i) acc += pl[i] * src[(size_t)i * nx];
    out[e] = acc;
  }
}

}  // namespace

extern "C" {

int bz_slab_left_mult(const double* P, int m, int k, const double* in, int nr, int nx, double* out,
                      hipStream_t stream) {
  if (m < 1 || k < 1 || nr < 0 || nx < 0 || !P || !in || !out) return BZ_EINVAL;
  const size_t total = (size_t)nr * m * nx;
  if (total == 0) return BZ_OK;
  const int blocks = (int)std::min<size_t>((total + 255) / 256, 16384);
  hipLaunchKernelGGL(k_slab_left_mult, dim3(blocks), dim3(256), 0, stream, P, m, k, in, nr, nx, out);
  BZ_LAUNCH_CHECK();
  return BZ_OK;
}

int bz_bidiag_solve_batched(const double* diag, const double* subdiag, const double* b, double* out, int bsz, int N,
                            int lower, hipStream_t stream) {
  if (bsz < 0 || N < 1 || !diag || !b || !out || (N > 1 && !subdiag)) return BZ_EINVAL;
  if (bsz == 0) return BZ_OK;
  SweepArgs a{};
  a.diag = diag; a.sdiag = subdiag; a.b = b; a.out = out; a.bsz = bsz; a.N = N; a.lower = lower;
  return launch_bidiag<K_BIDIAG>(a, stream);
}

int bz_xstep_bidiag_solve(const double* diag, const double* subdiag, const int* lower_of, const double* b,
                          double* out, int Nr, int Nvt, int Nx, hipStream_t stream) {
  if (Nr < 1 || Nvt < 1 || Nx < 2 || !diag || !subdiag || !lower_of || !b || !out) return BZ_EINVAL;
  SweepArgs a{};
  a.diag = diag; a.sdiag = subdiag; a.lower_of = lower_of; a.b = b; a.out = out;
  a.bsz = Nr * Nvt; a.N = Nx; a.Nr = Nr; a.Nvt = Nvt; a.Nx = Nx;
  const int bsz = Nr * Nvt;
  const int per = (Nx + 63) / 64;
  if (per > 16) return launch_bidiag<K_XSTEP>(a, stream);       // long lines: the chunked sweep
  const dim3 grid(bsz), block(64);
  if (per <= 2) hipLaunchKernelGGL((k_xstep_scan<2>), grid, block, 0, stream, diag, subdiag, lower_of, b, out, bsz, Nvt, Nx);
  else if (per <= 4) hipLaunchKernelGGL((k_xstep_scan<4>), grid, block, 0, stream, diag, subdiag, lower_of, b, out, bsz, Nvt, Nx);
  else if (per <= 8) hipLaunchKernelGGL((k_xstep_scan<8>), grid, block, 0, stream, diag, subdiag, lower_of, b, out, bsz, Nvt, Nx);
  else hipLaunchKernelGGL((k_xstep_scan<16>), grid, block, 0, stream, diag, subdiag, lower_of, b, out, bsz, Nvt, Nx);
  BZ_LAUNCH_CHECK();
  return BZ_OK;
}

int bz_banded_tri_solve_batched(const double* diags, const double* b, double* out, int bsz, int ndiags, int N,
                                int lower, hipStream_t stream) {
  if (bsz < 0 || N < 1 || ndiags < 1 || ndiags > 8 || !diags || !b || !out) return BZ_EINVAL;
  if (bsz == 0) return BZ_OK;
  SweepArgs a{};
  a.diags = diags; a.b = b; a.out = out; a.bsz = bsz; a.N = N; a.lower = lower;
  return launch_sweep<K_BANDED>(a, ndiags, stream);
}

int bz_banded_tri_mv_batched(const double* diags, const double* b, double* out, int bsz, int ndiags, int N, int lower,
                             hipStream_t stream) {
  if (bsz < 0 || N < 1 || ndiags < 1 || !diags || !b || !out) return BZ_EINVAL;
  const size_t total = (size_t)bsz * N;
  if (total == 0) return BZ_OK;
  const int blocks = (int)std::min<size_t>((total + 255) / 256, 16384);
  hipLaunchKernelGGL(k_banded_mv, dim3(blocks), dim3(256), 0, stream, diags, b, out, bsz, ndiags, N, lower);
  BZ_LAUNCH_CHECK();
  return BZ_OK;
}

static int adv_common(int kind, const double* DL, const double* DR, const double* p0, const double* p1, double dt,
                      const double* b, double* out, int ndiags, int Nr, int Nvt, int Nx, hipStream_t stream) {
  if (Nr < 1 || Nvt < 1 || Nx < 1 || ndiags < 1 || ndiags > 8 || !DL || !DR || !p0 || !p1 || !b || !out)
    return BZ_EINVAL;
  SweepArgs a{};
  a.DL = DL; a.DR = DR; a.p0 = p0; a.p1 = p1; a.dt = dt; a.b = b; a.out = out;
  a.Nr = Nr; a.Nvt = Nvt; a.Nx = Nx;
  if (kind == K_ADV_VR) { a.bsz = Nx * Nvt; a.N = Nr; return launch_sweep<K_ADV_VR>(a, ndiags, stream); }
  if (kind == K_ADV_VT) { a.bsz = Nx * Nr; a.N = Nvt; return launch_sweep<K_ADV_VT>(a, ndiags, stream); }
  a.bsz = Nr * Nvt; a.N = Nx;
  return launch_sweep<K_ADV_X>(a, ndiags, stream);
}

int bz_adv_vr_be(const double* D_LtoR, const double* D_RtoL, const double* Ex, const double* cos_vt, double dt,
                 const double* b, double* out, int ndiags, int Nr, int Nvt, int Nx, hipStream_t stream) {
  return adv_common(K_ADV_VR, D_LtoR, D_RtoL, Ex, cos_vt, dt, b, out, ndiags, Nr, Nvt, Nx, stream);
}

int bz_adv_vt_be(const double* D_LtoR, const double* D_RtoL, const double* Ex, const double* vr, double dt,
                 const double* b, double* out, int ndiags, int Nr, int Nvt, int Nx, hipStream_t stream) {
  return adv_common(K_ADV_VT, D_LtoR, D_RtoL, Ex, vr, dt, b, out, ndiags, Nr, Nvt, Nx, stream);
}

int bz_adv_x_be(const double* D_LtoR, const double* D_RtoL, const double* vr, const double* cos_vt, double dt,
                const double* b, double* out, int ndiags, int Nr, int Nvt, int Nx, hipStream_t stream) {
  return adv_common(K_ADV_X, D_LtoR, D_RtoL, vr, cos_vt, dt, b, out, ndiags, Nr, Nvt, Nx, stream);
}

int bz_bsr_upper_unit_solve(const double* data, const int* indptr, const int* indices, int nbr, int nrhs, int bsz,
                            const double* b, double* out, hipStream_t stream) {
  if (nbr < 1 || nrhs < 0 || bsz < 1 || bsz > 256 || !data || !indptr || !indices || !b || !out) return BZ_EINVAL;
  if (nrhs == 0) return BZ_OK;
  const int R = std::max(1, 256 / bsz);
  const int grid = (nrhs + R - 1) / R;
  hipLaunchKernelGGL(k_bsr_upper_unit, dim3(grid), dim3(bsz * R), (size_t)R * bsz * sizeof(double), stream, data,
                     indptr, indices, nbr, nrhs, bsz, R, b, out);
  BZ_LAUNCH_CHECK();
  return BZ_OK;
}

}  // extern "C"
