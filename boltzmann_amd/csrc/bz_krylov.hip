// Building blocks of restarted GMRES on the device (gfx950, FP64).
//
// The Krylov basis is stored row by row, V[j*ldv + e] (one contiguous vector per row),
// so every operation below streams whole vectors with consecutive threads on
// consecutive elements.  Reductions are two-pass and deterministic: each workgroup
// writes the partial sum of its chunk, and one wavefront per output adds the partials
// in a fixed order.  Orthogonalisation is classical Gram-Schmidt applied twice (two
// block dot products and two block updates per Arnoldi step, independent of the step
// count), which has the stability of modified Gram-Schmidt in FP64.
#include <algorithm>

#include "bz_common.h"

namespace {

constexpr int NT = 256;

// partial[j * nblk + blockIdx.x] = sum over this block's chunk of V[j][e] * u[e]; grid (nblk, nv)
__global__ __launch_bounds__(NT) void k_multi_dot_partial(const double* __restrict__ V, long ldv,
                                                          const double* __restrict__ u, long n, long chunk,
                                                          double* __restrict__ partial) {
  __shared__ double red[NT / 64];
  const int j = blockIdx.y;
  const long a = (long)blockIdx.x * chunk, b = std::min(n, a + chunk);
  const double* v = V + (long)j * ldv;
  double acc = 0.0;
  for (long e = a + threadIdx.x; e < b; e += NT) acc = fma(v[e], u[e], acc);
  acc = bz::wave_sum(acc);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0;
    for (int w = 0; w < NT / 64; ++w) s += red[w];
    partial[(long)j * gridDim.x + blockIdx.x] = s;
  }
}

// out[j * ostride] = (accumulate ? out : 0) + s_j with s_j = sum_b partial[j * nblk + b] (or its
// square root); out2[j] = s_j as well when out2 is given
__global__ void k_reduce_partials(const double* __restrict__ partial, int nblk, int nv, double* out, int ostride,
                                  int accumulate, int take_sqrt, double* out2) {
  const int j = blockIdx.x;
  if (j >= nv) return;
  double acc = 0.0;
  for (int b = threadIdx.x; b < nblk; b += 64) acc += partial[(long)j * nblk + b];
  acc = bz::wave_sum(acc);
  if (threadIdx.x == 0) {
    const double v = take_sqrt ? sqrt(acc) : acc;
    if (out2) out2[j] = v;
    out[(long)j * ostride] = accumulate ? out[(long)j * ostride] + v : v;
  }
}

// dst[e] = src[e] + sign * sum_j coef[j * cstride] * V[j][e]
__global__ void k_vt_axpy(const double* __restrict__ V, long ldv, int nv, const double* __restrict__ coef, int cstride,
                          double sign, const double* src, double* dst, long n) {
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x) {
    double s = 0.0;
    for (int j = 0; j < nv; ++j) s = fma(coef[(long)j * cstride], V[(long)j * ldv + e], s);
    dst[e] = src[e] + sign * s;
  }
}

// y = x / s[0]; nothing is written when s[0] == 0 (Arnoldi breakdown)
__global__ void k_scale_inv(const double* __restrict__ x, const double* __restrict__ s, double* y, long n) {
  const double d = s[0];
  if (d == 0.0) return;
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x) y[e] = x[e] / d;
}

// min_y |H y - beta e_0| for the (m+1) x m upper Hessenberg H (row stride ldh), by Givens
// rotations on a copy; one thread (m is the restart length, at most a few dozen).
__global__ void k_hess_lstsq(const double* __restrict__ H, int ldh, int m, const double* __restrict__ beta,
                             double* __restrict__ R, double* __restrict__ y) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  // R: (m+1) x m work copy, g: right-hand side stored in y[m+1 ...]
  double* g = y + m;
  for (int r = 0; r <= m; ++r)
    for (int c = 0; c < m; ++c) R[r * m + c] = H[(long)r * ldh + c];
  for (int r = 0; r <= m; ++r) g[r] = 0.0;
  g[0] = beta[0];
  for (int c = 0; c < m; ++c) {
    const double a = R[c * m + c], b = R[(c + 1) * m + c];
    const double rr = hypot(a, b);
    const double cs = (rr == 0.0) ? 1.0 : a / rr, sn = (rr == 0.0) ? 0.0 : b / rr;
    for (int k = c; k < m; ++k) {
      const double t1 = R[c * m + k], t2 = R[(c + 1) * m + k];
      R[c * m + k] = cs * t1 + sn * t2;
      R[(c + 1) * m + k] = -sn * t1 + cs * t2;
    }
    const double g1 = g[c], g2 = g[c + 1];
    g[c] = cs * g1 + sn * g2;
    g[c + 1] = -sn * g1 + cs * g2;
  }
  for (int c = m - 1; c >= 0; --c) {
    double s = g[c];
    for (int k = c + 1; k < m; ++k) s -= R[c * m + k] * y[k];
    y[c] = (R[c * m + c] != 0.0) ? s / R[c * m + c] : 0.0;
  }
}

// ---------------------------------------------------------------- one Arnoldi step in three launches
// The vector part of a step (classical Gram-Schmidt, the norm, the scaling, the rotation of the new
// column) as k_orth_dots, k_orth_update and k_orth_finish.  The reductions end in the kernel that
// needs them: every workgroup adds the few hundred partial sums of the kernel before it, in one
// order, so no launch and no gap is spent on a reduction, the rotation runs in the first workgroup
// while the others scale, and |w|^2 is accumulated where w is written.  What bounds it: the rows of
// V in the dots and the update (8 n bytes each), launch latency for small n.  Measured as whole
// implicit steps against separate dot, reduce, update, dot, reduce, scale and rotation launches,
// steps past convergence done in full: n = 1.07e6 4427 -> 3718 us, n = 21000 1064 -> 758 us.  A set
// stop flag turns every launch into a no-op.
constexpr int OT = 512;        // threads
constexpr int OJ = 4;          // basis vectors per workgroup in the dots
constexpr int OH = 256;        // basis vectors whose coefficients are held at a time in the update

__device__ __forceinline__ double block_sum(double v, double* red) {   // OT threads, all get the sum
  v = bz::wave_sum(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
#pragma unroll
  for (int w = 0; w < OT / 64; ++w) s += red[w];
  return s;
}

// partial[j * gridDim.x + blockIdx.x] = sum over this block's chunk of V[j][e] u[e],
// j = OJ blockIdx.y ...
__global__ __launch_bounds__(OT) void k_orth_dots(const double* __restrict__ V, long ldv, int nv,
                                                  const double* __restrict__ u, long n, long chunk,
                                                  double* __restrict__ partial, const int* __restrict__ done) {
  if (*done) return;
  __shared__ double red[OT / 64][OJ];
  const int j0 = blockIdx.y * OJ;
  const long a = (long)blockIdx.x * chunk, b = std::min(n, a + chunk);
  const double* v[OJ];
#pragma unroll
  for (int j = 0; j < OJ; ++j) v[j] = V + (long)std::min(j0 + j, nv - 1) * ldv;
  double acc[OJ] = {0.0, 0.0, 0.0, 0.0};
  long e = a + threadIdx.x;
  for (; e + OT < b; e += 2 * OT) {
    const double u0 = u[e], u1 = u[e + OT];
    double v0[OJ], v1[OJ];
#pragma unroll
    for (int j = 0; j < OJ; ++j) {
      v0[j] = v[j][e];
      v1[j] = v[j][e + OT];
    }
#pragma unroll
    for (int j = 0; j < OJ; ++j) acc[j] = fma(v1[j], u1, fma(v0[j], u0, acc[j]));
  }
  if (e < b) {
    const double u0 = u[e];
#pragma unroll
    for (int j = 0; j < OJ; ++j) acc[j] = fma(v[j][e], u0, acc[j]);
  }
#pragma unroll
  for (int j = 0; j < OJ; ++j) {
    const double w = bz::wave_sum(acc[j]);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][j] = w;
  }
  __syncthreads();
  if (threadIdx.x < OJ && j0 + (int)threadIdx.x < nv) {
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < OT / 64; ++w) t += red[w][threadIdx.x];
    partial[(long)(j0 + threadIdx.x) * gridDim.x + blockIdx.x] = t;
  }
}

// h_j = sum of the nblk partials of vector j (to column H[., col], added to it when accumulate);
// w -= sum_j h_j V_j; with norm_partial also the block's part of |w|^2
__global__ __launch_bounds__(OT) void k_orth_update(const double* __restrict__ V, long ldv, int nv,
                                                    const double* __restrict__ partial, int nblk,
                                                    double* __restrict__ w, long n, long chunk,
                                                    double* __restrict__ H, int ldh, int col, int accumulate,
                                                    double* __restrict__ norm_partial, const int* __restrict__ done) {
  if (*done) return;
  __shared__ double h[OH], red[OT / 64];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const long a = (long)blockIdx.x * chunk, b = std::min(n, a + chunk);
  double sq = 0.0;
  for (int j0 = 0; j0 < nv; j0 += OH) {
    const int nj = std::min(OH, nv - j0);
    for (int j = wave; j < nj; j += OT / 64) {
      double t = 0.0;
      for (int k = lane; k < nblk; k += 64) t += partial[(long)(j0 + j) * nblk + k];
      t = bz::wave_sum(t);
      if (lane == 0) {
        h[j] = t;
        if (blockIdx.x == 0) {
          double* hp = H + (long)(j0 + j) * ldh + col;
          *hp = accumulate ? *hp + t : t;
        }
      }
    }
    __syncthreads();
    const bool last = j0 + OH >= nv;
    const double* Vj = V + (long)j0 * ldv;
    for (long e0 = a + threadIdx.x; e0 < b; e0 += 2 * OT) {
      const long e1 = e0 + OT < b ? e0 + OT : e0;
      double s0 = 0.0, s1 = 0.0;
      int j = 0;
      for (; j + 4 <= nj; j += 4) {
        double v0[4], v1[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          v0[i] = Vj[(long)(j + i) * ldv + e0];
          v1[i] = Vj[(long)(j + i) * ldv + e1];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          s0 = fma(h[j + i], v0[i], s0);
          s1 = fma(h[j + i], v1[i], s1);
        }
      }
      for (; j < nj; ++j) {
        s0 = fma(h[j], Vj[(long)j * ldv + e0], s0);
        s1 = fma(h[j], Vj[(long)j * ldv + e1], s1);
      }
      const double w0 = w[e0] - s0, w1 = w[e1] - s1;
      w[e0] = w0;
      if (e1 != e0) w[e1] = w1;
      if (last) sq = fma(w0, w0, e1 != e0 ? fma(w1, w1, sq) : sq);
    }
    __syncthreads();
  }
  if (norm_partial) {
    const double t = block_sum(sq, red);
    if (threadIdx.x == 0) norm_partial[blockIdx.x] = t;
  }
}

// The new column h[0..i] of the triangular factor (h[r] at h[r * hs]) under the rotations before
// it, its own rotation, the rotated right-hand side and the stop test; hn = H[i+1][i].
__device__ void rotate_column(double* h, long hs, const double* cs, const double* sn, int i, double hn, double* cs_out,
                              double* sn_out, double* g, double tol, int* done, int* kdone) {
  double a = h[0];
  for (int k = 0; k < i; ++k) {
    const double b = h[(k + 1) * hs], c = cs[k], s = sn[k];
    h[k * hs] = c * a + s * b;
    a = -s * a + c * b;
  }
  const double r = hypot(a, hn);
  const double c = (r > 0.0) ? a / r : 1.0, s = (r > 0.0) ? hn / r : 0.0;
  *cs_out = c;
  *sn_out = s;
  h[i * hs] = r;
  const double gi = g[i], gn = -s * gi;
  g[i] = c * gi;
  g[i + 1] = gn;
  if (fabs(gn) <= tol || hn == 0.0) {
    *kdone = i + 1;
    __hip_atomic_store(done, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// hn = |w| from the partial sums, V_(i+1) = w / hn (not written when hn = 0); the first workgroup
// rotates column i of H and may set the stop flag while others of this launch have not read it yet.
// So one thread reads it for its workgroup (all of whose wavefronts then agree on the barriers and
// on hn), and a workgroup that finds it set skips its part of V_(i+1) as a whole: no later step and
// no solution reads that row.
__global__ __launch_bounds__(OT) void k_orth_finish(const double* __restrict__ norm_partial, int nblk,
                                                    const double* __restrict__ w, double* __restrict__ Vn, long n,
                                                    double* __restrict__ H, int ldh, int i, double* __restrict__ cs,
                                                    double* __restrict__ sn, double* __restrict__ g,
                                                    const double* __restrict__ tol, int* done, int* kdone) {
  constexpr int CL = 512;                            // columns up to this length are rotated in LDS
  __shared__ double red[OT / 64], hc[CL], sc[CL], ss[CL];
  __shared__ int stop;
  double t = 0.0;
  for (int k = threadIdx.x; k < nblk; k += OT) t += norm_partial[k];
  if (threadIdx.x == 0) stop = __hip_atomic_load(done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  if (stop) return;
  const double hn = sqrt(block_sum(t, red));
  if (hn != 0.0)
    for (long e = (long)blockIdx.x * OT + threadIdx.x; e < n; e += (long)gridDim.x * OT) Vn[e] = w[e] / hn;
  if (blockIdx.x != 0) return;
  if (i < CL) {
    if ((int)threadIdx.x <= i) {
      hc[threadIdx.x] = H[(long)threadIdx.x * ldh + i];
      sc[threadIdx.x] = cs[threadIdx.x];
      ss[threadIdx.x] = sn[threadIdx.x];
    }
    __syncthreads();
    if (threadIdx.x == 0) rotate_column(hc, 1, sc, ss, i, hn, cs + i, sn + i, g, tol[0], done, kdone);
    __syncthreads();
    if ((int)threadIdx.x <= i) H[(long)threadIdx.x * ldh + i] = hc[threadIdx.x];
  } else if (threadIdx.x == 0) {
    rotate_column(H + i, ldh, cs, sn, i, hn, cs + i, sn + i, g, tol[0], done, kdone);
  }
  if (threadIdx.x == 0) H[(long)(i + 1) * ldh + i] = 0.0;
}

// r = b - ax (ax NULL: r = b) and the block's part of |r|^2
__global__ __launch_bounds__(OT) void k_gmres_residual(const double* __restrict__ b, const double* ax, double* r, long n,
                                                       long chunk, double* __restrict__ partial) {
  __shared__ double red[OT / 64];
  const long a = (long)blockIdx.x * chunk, z = std::min(n, a + chunk);
  double sq = 0.0;
  for (long e = a + threadIdx.x; e < z; e += OT) {
    const double v = ax ? b[e] - ax[e] : b[e];
    if (r) r[e] = v;
    sq = fma(v, v, sq);
  }
  const double t = block_sum(sq, red);
  if (threadIdx.x == 0) partial[blockIdx.x] = t;
}

// stat: |r|, |b|, tol = max(atol, rtol |b|), steps of the cycle.  of: 0 the residual's norm (and
// the step count), 1 the right-hand side's (and the tolerance), 2 both at once (r = b).
__global__ __launch_bounds__(OT) void k_gmres_stat(const double* __restrict__ partial, int nblk, int of, double atol,
                                                   double rtol, const int* __restrict__ kdone, double* stat) {
  __shared__ double red[OT / 64];
  double t = 0.0;
  for (int k = threadIdx.x; k < nblk; k += OT) t += partial[k];
  const double v = sqrt(block_sum(t, red));
  if (threadIdx.x == 0) {
    if (of != 1) {
      stat[0] = v;
      stat[3] = (double)*kdone;
    }
    if (of != 0) {
      stat[1] = v;
      stat[2] = fmax(atol, rtol * v);
    }
  }
}

// Start of a cycle from r, |r| in stat[0]: V_0 = r / |r|, g = (|r|, 0, ...), the flags
__global__ __launch_bounds__(OT) void k_gmres_begin(const double* __restrict__ r, const double* __restrict__ stat,
                                                    double* __restrict__ V0, long n, int m, double* __restrict__ g,
                                                    double* __restrict__ tol, int* done, int* kdone) {
  const double beta = stat[0];
  if (beta != 0.0)
    for (long e = (long)blockIdx.x * OT + threadIdx.x; e < n; e += (long)gridDim.x * OT) V0[e] = r[e] / beta;
  if (blockIdx.x != 0) return;
  for (int k = threadIdx.x; k <= m; k += OT) g[k] = k == 0 ? beta : 0.0;
  if (threadIdx.x == 0) {
    tol[0] = stat[2];
    *done = beta < stat[2] ? 1 : 0;
    *kdone = beta < stat[2] ? 0 : m;
  }
}

// x += V y, R y = g over the k = *kdone steps of the cycle.  Every workgroup solves for y itself,
// column by column (64 rows at a time in flight), from an LDS copy of R up to order 64.
__global__ __launch_bounds__(OT) void k_gmres_solution(const double* __restrict__ V, long ldv,
                                                       const double* __restrict__ H, int ldh,
                                                       const double* __restrict__ g, const int* __restrict__ kdone,
                                                       double* __restrict__ x, long n, int kmax) {
  extern __shared__ double y[];                      // m, then R up to order 64
  double* R = y + kmax;
  const int k = *kdone;
  const bool lds = kmax <= 64;
  for (int j = threadIdx.x; j < k; j += OT) y[j] = g[j];
  if (lds)
    for (int e = threadIdx.x; e < k * k; e += OT) R[e] = H[(long)(e / k) * ldh + e % k];
  __syncthreads();
  for (int r = k - 1; r >= 0; --r) {
    const double yr = y[r] / (lds ? R[r * k + r] : H[(long)r * ldh + r]);
    __syncthreads();
    for (int j = threadIdx.x; j <= r; j += OT)
      y[j] = j == r ? yr : y[j] - (lds ? R[j * k + r] : H[(long)j * ldh + r]) * yr;
    __syncthreads();
  }
  for (long e = (long)blockIdx.x * OT + threadIdx.x; e < n; e += (long)gridDim.x * OT) {
    double s = 0.0;
#pragma unroll 4
    for (int j = 0; j < k; ++j) s = fma(y[j], V[(long)j * ldv + e], s);
    x[e] += s;
  }
}

// x += V y over the first *kdone rows: rows past the last step may hold anything
__global__ __launch_bounds__(OT) void k_gmres_add(const double* __restrict__ V, long ldv, const double* __restrict__ y,
                                                  const int* __restrict__ kdone, double* __restrict__ x, long n) {
  const int k = *kdone;
  for (long e = (long)blockIdx.x * OT + threadIdx.x; e < n; e += (long)gridDim.x * OT) {
    double s = 0.0;
#pragma unroll 4
    for (int j = 0; j < k; ++j) s = fma(y[j], V[(long)j * ldv + e], s);
    x[e] += s;
  }
}

int orth_blocks(long n, long per) { return (int)std::max<long>(1, std::min<long>(256, (n + per - 1) / per)); }

int grid_for(long n) { return (int)std::min<long>((n + NT - 1) / NT, 8192); }

// bin[x] = argmin_i |E[x] - Ev[i]| (first minimum), the preconditioner membership of
// glow1d_boltzmann.vspace_pc_setup
__global__ void k_nearest_bin(const double* __restrict__ E, int nx, const double* __restrict__ Ev, int nb,
                              int* __restrict__ bin) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= nx) return;
  const double e = E[x];
  int best = 0;
  double bd = fabs(e - Ev[0]);
  for (int i = 1; i < nb; ++i) {
    const double d = fabs(e - Ev[i]);
    if (d < bd) { bd = d; best = i; }
  }
  bin[x] = best;
}

// y[i, x] = sum_k P[bin[x]][i, k] u[k, x]; u, y (dof, nx) with x fastest.  Consecutive
// threads take consecutive x; neighbouring points share a bin, so the rows of P they
// read are the same cache lines.
__global__ void k_binned_block_apply(const double* __restrict__ P, int dof, const int* __restrict__ bin,
                                     const double* __restrict__ u, int nx, double* __restrict__ y) {
  const long total = (long)dof * nx;
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (long)gridDim.x * blockDim.x) {
    const int x = (int)(e % nx), i = (int)(e / nx);
    const double* row = P + ((long)bin[x] * dof + i) * dof;
    double s = 0.0;
    for (int k = 0; k < dof; ++k) s = fma(row[k], u[(long)k * nx + x], s);
    y[e] = s;
  }
}

// y = x - c (Kx + E[col] Ax) for (dof, nx) arrays: the backward-Euler v-space operator
// I - dt tau (n0 np0 (C + Tg C_T) + E A) applied from the two operator products
__global__ void k_vstep_combine(const double* __restrict__ x, const double* __restrict__ Kx,
                                const double* __restrict__ Ax, const double* __restrict__ E, double c, int nx,
                                long total, double* __restrict__ y) {
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (long)gridDim.x * blockDim.x)
    y[e] = x[e] - c * (Kx[e] + E[e % nx] * Ax[e]);
}

// ---------------------------------------------------------------- batched GMRES (many small systems)
// B independent systems of size n, one wavefront each.  Basis V[(j * B + b) * n + e],
// j = 0..m; the Hessenberg columns are reduced by Givens rotations as they arrive, so
// R[b][col * m + row] holds the triangular factor, g[b][0..m] the rotated right-hand
// side and |g[b][k]| the residual norm after k steps.

__device__ __forceinline__ double wdot(const double* __restrict__ a, const double* __restrict__ b, int n) {
  double s = 0.0;
  for (int e = threadIdx.x; e < n; e += 64) s = fma(a[e], b[e], s);
  return bz::wave_sum(s);
}

// Arnoldi step i of every active system: orthogonalise w[b] (the operator applied to
// the preconditioned V_i) against V_0..V_i (classical Gram-Schmidt, twice), append
// V_{i+1}, rotate the new column, update the residual estimate; a system whose residual
// reaches target[b] (or whose basis breaks down) becomes inactive with kdim = i + 1.
__global__ __launch_bounds__(64) void k_arnoldi_batched(int n, int B, int m, int i, double* __restrict__ V,
                                                        const double* __restrict__ w, double* __restrict__ R,
                                                        double* __restrict__ cs, double* __restrict__ sn,
                                                        double* __restrict__ g, const double* __restrict__ target,
                                                        int* __restrict__ active, int* __restrict__ kdim,
                                                        double* __restrict__ resid) {
  extern __shared__ double lds[];
  const int inst = blockIdx.x, lane = threadIdx.x;
  if (!active[inst]) return;
  double* W = lds;
  double* HC = W + n;          // [m + 2] Hessenberg column
  double* T = HC + m + 2;      // [m + 1] projections of one pass
  for (int e = lane; e < n; e += 64) W[e] = w[(size_t)inst * n + e];
  for (int j = lane; j <= i + 1; j += 64) HC[j] = 0.0;
  __syncthreads();
  for (int rep = 0; rep < 2; ++rep) {
    // four dot products side by side (each in the order of wdot): their loads and their sums
    // across the wavefront overlap
    for (int j0 = 0; j0 <= i; j0 += 4) {
      double s[4] = {0.0, 0.0, 0.0, 0.0};
      for (int e = lane; e < n; e += 64) {
        double vj[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) vj[u] = V[((size_t)min(j0 + u, i) * B + inst) * n + e];
#pragma unroll
        for (int u = 0; u < 4; ++u) s[u] = fma(vj[u], W[e], s[u]);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) s[u] = bz::wave_sum(s[u]);
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (lane == 0 && j0 + u <= i) { T[j0 + u] = s[u]; HC[j0 + u] += s[u]; }
    }
    __syncthreads();
    for (int e = lane; e < n; e += 64) {
      double s = W[e];
      int j = 0;
      for (; j + 4 <= i + 1; j += 4) {
        double vj[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) vj[u] = V[((size_t)(j + u) * B + inst) * n + e];
#pragma unroll
        for (int u = 0; u < 4; ++u) s = fma(-T[j + u], vj[u], s);
      }
      for (; j <= i; ++j) s = fma(-T[j], V[((size_t)j * B + inst) * n + e], s);
      W[e] = s;
    }
    __syncthreads();
  }
  const double hn = sqrt(wdot(W, W, n));
  const double inv = hn > 0.0 ? 1.0 / hn : 0.0;
  double* Vn = V + ((size_t)(i + 1) * B + inst) * n;
  for (int e = lane; e < n; e += 64) Vn[e] = W[e] * inv;
  if (lane == 0) {
    HC[i + 1] = hn;
    double* csb = cs + (size_t)inst * m;
    double* snb = sn + (size_t)inst * m;
    double* gb = g + (size_t)inst * (m + 1);
    for (int j = 0; j < i; ++j) {
      const double a = HC[j], b2 = HC[j + 1];
      HC[j] = fma(csb[j], a, snb[j] * b2);
      HC[j + 1] = fma(-snb[j], a, csb[j] * b2);
    }
    const double a = HC[i], b2 = HC[i + 1];
    const double r = hypot(a, b2);
    const double c = r > 0.0 ? a / r : 1.0, s = r > 0.0 ? b2 / r : 0.0;
    csb[i] = c;
    snb[i] = s;
    HC[i] = r;
    const double gi = gb[i];
    gb[i] = c * gi;
    gb[i + 1] = -s * gi;
    double* Rb = R + (size_t)inst * m * m + (size_t)i * m;
    for (int j = 0; j <= i; ++j) Rb[j] = HC[j];
    const double res = fabs(gb[i + 1]);
    resid[inst] = res;
    kdim[inst] = i + 1;
    if (res <= target[inst] || !(hn > 0.0) || i + 1 >= m) active[inst] = 0;
  }
}

// out[b] = sum_j y_j V_j[b] with R y = g (the first kdim[b] steps); zero when kdim[b] = 0
__global__ __launch_bounds__(64) void k_gmres_combine_batched(int n, int B, int m, const double* __restrict__ V,
                                                              const double* __restrict__ R,
                                                              const double* __restrict__ g,
                                                              const int* __restrict__ kdim, double* __restrict__ out) {
  __shared__ double Y[64];
  const int inst = blockIdx.x, lane = threadIdx.x;
  const int k = kdim[inst];
  if (lane == 0) {
    const double* Rb = R + (size_t)inst * m * m;
    const double* gb = g + (size_t)inst * (m + 1);
    for (int r = k - 1; r >= 0; --r) {
      double s = gb[r];
      for (int c = r + 1; c < k; ++c) s = fma(-Rb[(size_t)c * m + r], Y[c], s);
      Y[r] = Rb[(size_t)r * m + r] != 0.0 ? s / Rb[(size_t)r * m + r] : 0.0;
    }
  }
  __syncthreads();
  for (int e = lane; e < n; e += 64) {
    double s = 0.0;
    for (int j = 0; j < k; ++j) s = fma(Y[j], V[((size_t)j * B + inst) * n + e], s);
    out[(size_t)inst * n + e] = s;
  }
}

}  // namespace

extern "C" {

int bz_multi_dot(const double* V, long ldv, int nv, const double* u, long n, double* partial, int nblk, double* out,
                 int ostride, int accumulate, int take_sqrt, double* out2, hipStream_t stream) {
  if (nv < 1 || n < 1 || nblk < 1 || ldv < n || !V || !u || !partial || !out || ostride < 1) return BZ_EINVAL;
  const long chunk = (n + nblk - 1) / nblk;
  hipLaunchKernelGGL(k_multi_dot_partial, dim3(nblk, nv), dim3(NT), 0, stream, V, ldv, u, n, chunk, partial);
  BZ_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_reduce_partials, dim3(nv), dim3(64), 0, stream, partial, nblk, nv, out, ostride, accumulate,
                     take_sqrt, out2);
  BZ_LAUNCH_CHECK();
  return BZ_OK;
}

int bz_vt_axpy(const double* V, long ldv, int nv, const double* coef, int cstride, double sign, const double* src,
               double* dst, long n, hipStream_t stream) {
  if (nv < 0 || n < 1 || ldv < n || !V || !coef || !src || !dst || cstride < 1) return BZ_EINVAL;
  hipLaunchKernelGGL(k_vt_axpy, dim3(grid_for(n)), dim3(NT), 0, stream, V, ldv, nv, coef, cstride, sign, src, dst, n);
  BZ_LAUNCH_CHECK();
  return BZ_OK;
}

int bz_scale_inv(const double* x, const double* s, double* y, long n, hipStream_t stream) {
  if (n < 1 || !x || !s || !y) return BZ_EINVAL;
  hipLaunchKernelGGL(k_scale_inv, dim3(grid_for(n)), dim3(NT), 0, stream, x, s, y, n);
  BZ_LAUNCH_CHECK();
  return BZ_OK;
}

// partial: (m + 1) * 256 doubles.  The last 256 hold |w|^2.
int bz_gmres_orthogonalise(double* V, long ldv, int m, int i, double* w, long n, int passes, double* partial, double* H,
                           int ldh, double* cs, double* sn, double* g, const double* tol, int* done, int* kdone,
                           hipStream_t stream) {
  if (n < 1 || ldv < n || m < 1 || i < 0 || i >= m || passes < 1 || ldh <= i || !V || !w || !partial || !H || !cs ||
      !sn || !g || !tol || !done || !kdone)
    return BZ_EINVAL;
  if ((i + OJ) / OJ > 65535) return BZ_EINVAL;
  const int nblk = orth_blocks(n, 2 * OT);
  const long chunk = (n + nblk - 1) / nblk;
  double* np = partial + (long)m * 256;
  for (int p = 0; p < passes; ++p) {
    hipLaunchKernelGGL(k_orth_dots, dim3(nblk, (i + OJ) / OJ), dim3(OT), 0, stream, V, ldv, i + 1, w, n, chunk, partial,
                       done);
    BZ_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_orth_update, dim3(nblk), dim3(OT), 0, stream, V, ldv, i + 1, partial, nblk, w, n, chunk, H, ldh,
                       i, p > 0 ? 1 : 0, p + 1 == passes ? np : nullptr, done);
    BZ_LAUNCH_CHECK();
  }
  hipLaunchKernelGGL(k_orth_finish, dim3(orth_blocks(n, OT) * 2), dim3(OT), 0, stream, np, nblk, w,
                     V + (long)(i + 1) * ldv, n, H, ldh, i, cs, sn, g, tol, done, kdone);
  BZ_LAUNCH_CHECK();
  return BZ_OK;
}

int bz_gmres_norm(const double* b, const double* ax, double* r, long n, double* partial, int of, double atol, double rtol,
                  const int* kdone, double* stat, hipStream_t stream) {
  if (n < 1 || !b || !partial || !kdone || !stat || of < 0 || of > 2) return BZ_EINVAL;
  const int nblk = orth_blocks(n, 2 * OT);
  hipLaunchKernelGGL(k_gmres_residual, dim3(nblk), dim3(OT), 0, stream, b, ax, r, n, (n + nblk - 1) / nblk, partial);
  BZ_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_gmres_stat, dim3(1), dim3(OT), 0, stream, partial, nblk, of, atol, rtol, kdone, stat);
  BZ_LAUNCH_CHECK();
  return BZ_OK;
}

int bz_gmres_begin(const double* r, const double* stat, double* V0, long n, int m, double* g, double* tol, int* done,
                   int* kdone, hipStream_t stream) {
  if (n < 1 || m < 1 || !r || !stat || !V0 || !g || !tol || !done || !kdone) return BZ_EINVAL;
  hipLaunchKernelGGL(k_gmres_begin, dim3(orth_blocks(n, OT) * 2), dim3(OT), 0, stream, r, stat, V0, n, m, g, tol, done,
                     kdone);
  BZ_LAUNCH_CHECK();
  return BZ_OK;
}

int bz_gmres_solution(const double* V, long ldv, int m, const double* H, int ldh, const double* g, const int* kdone,
                      double* x, long n, hipStream_t stream) {
  if (n < 1 || ldv < n || m < 1 || m > 8000 || ldh < m || !V || !H || !g || !kdone || !x) return BZ_EINVAL;
  hipLaunchKernelGGL(k_gmres_solution, dim3(orth_blocks(n, OT) * 2), dim3(OT),
                     (size_t)(m <= 64 ? m + m * m : m) * sizeof(double), stream, V, ldv, H, ldh, g, kdone, x, n, m);
  BZ_LAUNCH_CHECK();
  return BZ_OK;
}

int bz_gmres_add(const double* V, long ldv, const double* y, const int* kdone, double* x, long n, hipStream_t stream) {
  if (n < 1 || ldv < n || !V || !y || !kdone || !x) return BZ_EINVAL;
  hipLaunchKernelGGL(k_gmres_add, dim3(orth_blocks(n, OT) * 2), dim3(OT), 0, stream, V, ldv, y, kdone, x, n);
  BZ_LAUNCH_CHECK();
  return BZ_OK;
}

int bz_nearest_bin(const double* E, int nx, const double* Ev, int nb, int* bin, hipStream_t stream) {
  if (nx < 0 || nb < 1 || !E || !Ev || !bin) return BZ_EINVAL;
  if (nx == 0) return BZ_OK;
  hipLaunchKernelGGL(k_nearest_bin, dim3((nx + 255) / 256), dim3(256), 0, stream, E, nx, Ev, nb, bin);
  BZ_LAUNCH_CHECK();
  return BZ_OK;
}

int bz_binned_block_apply(const double* P, int dof, const int* bin, const double* u, int nx, double* y,
                          hipStream_t stream) {
  if (dof < 1 || nx < 1 || !P || !bin || !u || !y) return BZ_EINVAL;
  hipLaunchKernelGGL(k_binned_block_apply, dim3(grid_for((long)dof * nx)), dim3(NT), 0, stream, P, dof, bin, u, nx, y);
  BZ_LAUNCH_CHECK();
  return BZ_OK;
}

int bz_vstep_combine(const double* x, const double* Kx, const double* Ax, const double* E, double c, int dof, int nx,
                     double* y, hipStream_t stream) {
  if (dof < 1 || nx < 1 || !x || !Kx || !Ax || !E || !y) return BZ_EINVAL;
  const long total = (long)dof * nx;
  hipLaunchKernelGGL(k_vstep_combine, dim3(grid_for(total)), dim3(NT), 0, stream, x, Kx, Ax, E, c, nx, total, y);
  BZ_LAUNCH_CHECK();
  return BZ_OK;
}

int bz_hess_lstsq(const double* H, int ldh, int m, const double* beta, double* work, double* y, hipStream_t stream) {
  if (m < 1 || ldh < m || !H || !beta || !work || !y) return BZ_EINVAL;
  hipLaunchKernelGGL(k_hess_lstsq, dim3(1), dim3(64), 0, stream, H, ldh, m, beta, work, y);
  BZ_LAUNCH_CHECK();
  return BZ_OK;
}

int bz_arnoldi_batched(int n, int B, int m, int i, double* V, const double* w, double* R, double* cs, double* sn,
                       double* g, const double* target, int* active, int* kdim, double* resid, hipStream_t stream) {
  if (n < 1 || B < 1 || m < 1 || m > 64 || i < 0 || i >= m || !V || !w || !R || !cs || !sn || !g || !target ||
      !active || !kdim || !resid)
    return BZ_EINVAL;
  const size_t lds = (size_t)(n + 2 * m + 3) * sizeof(double);
  if (lds > 64 * 1024) return BZ_EINVAL;
  hipLaunchKernelGGL(k_arnoldi_batched, dim3(B), dim3(64), lds, stream, n, B, m, i, V, w, R, cs, sn, g, target, active,
                     kdim, resid);
  BZ_LAUNCH_CHECK();
  return BZ_OK;
}

int bz_gmres_combine_batched(int n, int B, int m, const double* V, const double* R, const double* g, const int* kdim,
                             double* out, hipStream_t stream) {
  if (n < 1 || B < 1 || m < 1 || m > 64 || !V || !R || !g || !kdim || !out) return BZ_EINVAL;
  hipLaunchKernelGGL(k_gmres_combine_batched, dim3(B), dim3(64), 0, stream, n, B, m, V, R, g, kdim, out);
  BZ_LAUNCH_CHECK();
  return BZ_OK;
}

}  // extern "C"
