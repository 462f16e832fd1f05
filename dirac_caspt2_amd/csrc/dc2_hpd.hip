// Resolvents of the A and C subspaces without an eigendecomposition of B~.
//
// solve_A/C_subspace.F90:197-257 diagonalise B~ = W w W^H and sum |W^H y_k|^2 / (alpha_k + w)
// over the perturbers k.  Both sums follow from u_k = (B~ + alpha_k)^-1 y_k alone:
//   e2 = -sum_k Re(y_k^H u_k),  sumc2 = sum_k |u_k|^2,
// and A and C have few perturbers (inactive or secondary spinors), so the systems are solved
// by conjugate gradients with the diagonal preconditioner Re B~_ii + alpha_k, every perturber
// with its own shift and step lengths and all of them sharing one product B~ P per iteration.
#include "dc2_kernels.hpp"

namespace dc2 {

namespace {

constexpr int CG_T = 256, CG_EMAX = 8;   // threads per column, rows per thread at most
constexpr int64_t CG_NMAX = (int64_t)CG_T * CG_EMAX;
constexpr double CG_TOL2 = 1e-28;        // squared relative residual at which a column is done
constexpr int CG_CHUNK = 8, CG_ITMAX = 240;   // iterations between two looks at the states, at most

enum { CG_ACTIVE = 0, CG_DONE = 1, CG_BAD = 2 };

// sums over the workgroup of two doubles, the same in every thread (fixed order)
__device__ inline void cg_sum2(double& a, double& b, double* red) {
  a = wave_add(a);
  b = wave_add(b);
  __syncthreads();   // red may still be read from the sum before
  if ((threadIdx.x & 63) == 0) {
    red[2 * (threadIdx.x >> 6)] = a;
    red[2 * (threadIdx.x >> 6) + 1] = b;
  }
  __syncthreads();
  a = red[0] + red[2] + red[4] + red[6];
  b = red[1] + red[3] + red[5] + red[7];
}

// x = 0, r = y, z = r / d, p = z; rho = r^H z, stop = CG_TOL2 |y|^2
__global__ __launch_bounds__(CG_T) void k_cg_init(int n, const cplx* __restrict__ Bt, const double* __restrict__ alpha,
                                                  const cplx* __restrict__ Y, cplx* __restrict__ X,
                                                  cplx* __restrict__ R, cplx* __restrict__ P,
                                                  double* __restrict__ rho, double* __restrict__ stop,
                                                  int* __restrict__ state) {
  __shared__ double red[8];
  const int k = blockIdx.x;
  const int64_t o = (int64_t)n * k;
  const double al = alpha[k];
  double yy = 0.0, rz = 0.0, low = 1.0;
  for (int i = threadIdx.x; i < n; i += CG_T) {
    const cplx y = Y[o + i];
    const double d = Bt[i + (int64_t)n * i].x + al;
    const cplx z = cscale(y, 1.0 / d);
    X[o + i] = mk(0.0, 0.0);
    R[o + i] = y;
    P[o + i] = z;
    yy += cabs2(y);
    rz += y.x * z.x + y.y * z.y;
    if (!(d > 0.0)) low = 0.0;
  }
  double bad = 1.0 - low;
  cg_sum2(yy, rz, red);
  double dummy = 0.0;
  cg_sum2(bad, dummy, red);
  if (threadIdx.x == 0) {
    rho[k] = rz;
    stop[k] = CG_TOL2 * yy;
    state[k] = bad > 0.0 || !(yy < 1e300) ? CG_BAD : (yy == 0.0 ? CG_DONE : CG_ACTIVE);
  }
}

// One iteration of every active column with Q = B~ P formed before: a workgroup per column
// keeps the column's x, r, p and q in registers between its two reductions, so that an
// iteration is one product and this one launch (16 n bytes read and written per vector).
template <int E>
__global__ __launch_bounds__(CG_T) void k_cg_step(int n, const cplx* __restrict__ Bt, const double* __restrict__ alpha,
                                                  const cplx* __restrict__ Q, cplx* __restrict__ X,
                                                  cplx* __restrict__ R, cplx* __restrict__ P,
                                                  double* __restrict__ rho, const double* __restrict__ stop,
                                                  int* __restrict__ state) {
  __shared__ double red[8];
  const int k = blockIdx.x;
  if (state[k] != CG_ACTIVE) return;   // uniform
  const int64_t o = (int64_t)n * k;
  const double al = alpha[k], rz = rho[k];
  cplx p[E], q[E], x[E], r[E];
  double d[E];
  double pq = 0.0, zero = 0.0;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int i = threadIdx.x + CG_T * e;
    p[e] = q[e] = x[e] = r[e] = mk(0.0, 0.0);
    d[e] = 1.0;
    if (i < n) {
      p[e] = P[o + i];
      q[e] = Q[o + i];
      x[e] = X[o + i];
      r[e] = R[o + i];
      d[e] = Bt[i + (int64_t)n * i].x + al;
    }
  }
#pragma unroll
  for (int e = 0; e < E; ++e) {
    q[e] = mk(fma(al, p[e].x, q[e].x), fma(al, p[e].y, q[e].y));
    pq += p[e].x * q[e].x + p[e].y * q[e].y;
  }
  cg_sum2(pq, zero, red);
  const double a = rz / pq;
  double rzn = 0.0, rr = 0.0;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    x[e] = mk(fma(a, p[e].x, x[e].x), fma(a, p[e].y, x[e].y));
    r[e] = mk(fma(-a, q[e].x, r[e].x), fma(-a, q[e].y, r[e].y));
    const double s = cabs2(r[e]);
    rr += s;
    rzn += s / d[e];
  }
  cg_sum2(rzn, rr, red);
  const double b = rzn / rz;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int i = threadIdx.x + CG_T * e;
    if (i < n) {
      const double id = 1.0 / d[e];
      X[o + i] = x[e];
      R[o + i] = r[e];
      P[o + i] = mk(fma(b, p[e].x, r[e].x * id), fma(b, p[e].y, r[e].y * id));
    }
  }
  if (threadIdx.x == 0) {
    rho[k] = rzn;
    if (!(pq > 0.0) || !(rr < 1e300)) state[k] = CG_BAD;   // not positive definite (or not finite)
    else if (rr <= stop[k]) state[k] = CG_DONE;
  }
}

// out: {one past the last active column, columns that failed}
__global__ __launch_bounds__(CG_T) void k_cg_poll(int npert, const int* __restrict__ state, int* __restrict__ out) {
  __shared__ int last, bad;
  if (threadIdx.x == 0) last = bad = 0;
  __syncthreads();
  for (int k = threadIdx.x; k < npert; k += CG_T) {
    if (state[k] == CG_ACTIVE) atomicMax(&last, k + 1);
    if (state[k] == CG_BAD) atomicAdd(&bad, 1);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    out[0] = last;
    out[1] = bad;
  }
}

// with Q = B~ X: the residual |y - (B~ + alpha) x|^2 against |y|^2 (a column outside the bound
// is marked as failed) and the column's -Re(y^H x) and |x|^2
__global__ __launch_bounds__(CG_T) void k_cg_energy(int n, const double* __restrict__ alpha,
                                                    const cplx* __restrict__ Y, const cplx* __restrict__ X,
                                                    const cplx* __restrict__ Q, double bound2,
                                                    double* __restrict__ partial, int* __restrict__ state) {
  __shared__ double red[8];
  const int k = blockIdx.x;
  const int64_t o = (int64_t)n * k;
  const double al = alpha[k];
  double e = 0.0, s = 0.0, rr = 0.0, yy = 0.0;
  for (int i = threadIdx.x; i < n; i += CG_T) {
    const cplx x = X[o + i], y = Y[o + i], q = Q[o + i];
    const double rx = y.x - q.x - al * x.x, ry = y.y - q.y - al * x.y;
    e -= y.x * x.x + y.y * x.y;
    s += cabs2(x);
    rr += rx * rx + ry * ry;
    yy += cabs2(y);
  }
  cg_sum2(e, s, red);
  cg_sum2(rr, yy, red);
  if (threadIdx.x == 0) {
    partial[2 * k] = e;
    partial[2 * k + 1] = s;
    if (!(rr <= bound2 * yy)) state[k] = CG_BAD;
  }
}

template <int E>
void step(hipStream_t s, int n, int nact, const cplx* Bt, const double* alpha, const cplx* Q, cplx* X, cplx* R, cplx* P,
          double* rho, const double* stop, int* state) {
  hipLaunchKernelGGL((k_cg_step<E>), dim3(nact), dim3(CG_T), 0, s, n, Bt, alpha, Q, X, R, P, rho, stop, state);
}

}  // namespace

int64_t cg_max_n() { return CG_NMAX; }
int64_t cg_work_bytes(int64_t n, int64_t npert) { return npert * (4 * n * 16 + 2 * 8 + 4) + 256 + 64; }

bool cg_resolvent(hipStream_t s, int64_t n, int64_t npert, const cplx* Bt, const cplx* Y, const double* alpha,
                  void* work, int* host2, double* partial, double* out2, int* iterations) {
  DC2_CHECK(n >= 1 && n <= CG_NMAX && npert >= 1 && npert < (1ll << 24), 1, "cg_resolvent: size out of range");
  cplx* X = reinterpret_cast<cplx*>(work);
  cplx* R = X + n * npert;
  cplx* P = R + n * npert;
  cplx* Q = P + n * npert;
  double* rho = reinterpret_cast<double*>(Q + n * npert);
  double* stop = rho + npert;
  int* out = reinterpret_cast<int*>(stop + npert);   // {last, bad}
  int* state = out + 16;
  const cplx one = mk(1.0, 0.0), zero = mk(0.0, 0.0);
  const int ni = (int)n, E = (int)((n + CG_T - 1) / CG_T);
  hipLaunchKernelGGL(k_cg_init, dim3((unsigned)npert), dim3(CG_T), 0, s, ni, Bt, alpha, Y, X, R, P, rho, stop, state);
  DC2_HIP(hipGetLastError());
  auto poll = [&]() {
    hipLaunchKernelGGL(k_cg_poll, dim3(1), dim3(CG_T), 0, s, (int)npert, state, out);
    DC2_HIP(hipMemcpyAsync(host2, out, 2 * sizeof(int), hipMemcpyDeviceToHost, s));
    DC2_HIP(hipStreamSynchronize(s));
    return host2[1] == 0;
  };
  int nact = (int)npert, it = 0;
  while (nact > 0) {
    // the shifts grow along the perturbers (their orbital energies are ascending), so the
    // columns converge from the last one on and the products shrink at every poll
    for (int c = 0; c < CG_CHUNK; ++c, ++it) {
      zgemm(s, 'N', 'N', n, nact, n, one, Bt, n, 0, P, n, 0, zero, Q, n, 0, 1);
      // rows per thread: the smallest instance that holds n, so that a column stays in registers
      // with few rows past n (280 columns of 1274 rows: 9.9 us with five, 10.3 with eight)
      if (E <= 1) step<1>(s, ni, nact, Bt, alpha, Q, X, R, P, rho, stop, state);
      else if (E <= 2) step<2>(s, ni, nact, Bt, alpha, Q, X, R, P, rho, stop, state);
      else if (E <= 4) step<4>(s, ni, nact, Bt, alpha, Q, X, R, P, rho, stop, state);
      else if (E <= 5) step<5>(s, ni, nact, Bt, alpha, Q, X, R, P, rho, stop, state);
      else step<8>(s, ni, nact, Bt, alpha, Q, X, R, P, rho, stop, state);
      DC2_HIP(hipGetLastError());
    }
    if (!poll()) return false;
    nact = host2[0];
    if (nact > 0 && it >= CG_ITMAX) return false;
  }
  if (iterations) *iterations = std::max(it, 1);
  // a column whose true residual has drifted from the recursive one is refused; over 8 to 16
  // active spinors and strong and weak correlation it stays below 1.6e-14, and on matrices with
  // conditions up to 6e4 the sums were exact to rounding or nearer to exact ones than an
  // eigendecomposition's (by up to 270 times)
  zgemm(s, 'N', 'N', n, npert, n, one, Bt, n, 0, X, n, 0, zero, Q, n, 0, 1);
  hipLaunchKernelGGL(k_cg_energy, dim3((unsigned)npert), dim3(CG_T), 0, s, ni, alpha, Y, X, Q, 1e-24, partial, state);
  sum_partials(s, npert, partial, out2);
  return poll();
}

// ------------------------------------------------------------------ Cholesky whitening
//
// When no eigenvalue of a metric S lies below the linear-dependency threshold, every
// orthonormalisation of its space gives the same resolvents, and S = U^H U with L^-1 = U^-H
// replaces the eigendecomposition: B~ = L^-1 B L^-H, y = L^-1 V.  That no eigenvalue is below
// the threshold is decided by a second factorisation, of S - sigma I, whose pivots are all
// positive exactly when every eigenvalue of S is above sigma (to rounding, as for an
// eigensolver).  Both are factorised side by side as a batch of two: the panels are a chain of
// dependent steps, each too small to fill the device.
//
// Per step of NB = 64 rows: k_chol_step, in which every workgroup eliminates the diagonal
// block redundantly (64 steps with one workgroup barrier each, the block in registers) and
// then multiplies its 64 columns of the block row by the block's inverse factor on the matrix
// cores, and one trailing update of the upper tiles (zherk_trailing).  L^-1 from the inverse
// diagonal blocks by merging neighbours, [[X, 0], [-Z U12^H X, Z]], doubling the block size.
//
// Bound by the chain of the 20 steps at n = 1274 (42 us for the last to 81 us for the first: the
// elimination 34, with the block row's product 48, the update 10 to 30), against 13.4 ms for the
// tridiagonalisation and 9 ms for the divide and conquer, back-transformation and scaled products
// it replaces; the two factorisations, L^-1 and B~ take 3.3 ms beside the other lanes.  324 spinors, FP64: 49.7 -> 39.9 ms per energy, split 37.7.

namespace {

constexpr int CH_NB = LOW_P, CH_LS = CH_NB + 1;   // 64: the Gram matrix of low_iterate is one block

struct Shifts {
  double v[3];
};

// W[b] (np x np), b < nmat: S - shift_b I in the leading n x n corner, the unit matrix below it
__global__ __launch_bounds__(256) void k_chol_pack(int n, int np, const cplx* __restrict__ S, int64_t lds, int nmat,
                                                   Shifts shift, cplx* __restrict__ W) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= (int64_t)np * np) return;
  const int i = (int)(t % np), j = (int)(t / np);
  const bool in = i < n && j < n;
  const cplx v = in ? S[i + lds * j] : mk(i == j ? 1.0 : 0.0, 0.0);
  for (int b = 0; b < nmat; ++b)
    W[(int64_t)np * np * b + t] = mk(in && i == j ? v.x - shift.v[b] : v.x, v.y);
}

// Step kb: block row kb of U = L^H from W, and (workgroup 0 of matrices 0 and 2) the inverse of
// its diagonal block into Li[0] and Li[1].  flag[b] is set when a pivot of matrix b is not positive.
__global__ __launch_bounds__(256) void k_chol_step(int np, int kb, const cplx* __restrict__ W, cplx* __restrict__ U,
                                                   cplx* __restrict__ Li, int* __restrict__ flag) {
  __shared__ cplx rowb[2][CH_NB], colb[2][CH_NB];
  __shared__ double Ar[CH_NB][CH_LS], Ai[CH_NB][CH_LS], Br[CH_NB][CH_LS], Bi[CH_NB][CH_LS];
  typedef double d4 __attribute__((ext_vector_type(4)));
  const int64_t nn = (int64_t)np * np;
  const int b = blockIdx.y, tid = threadIdx.x;
  W += nn * b;
  U += nn * b;
  const int k0 = kb * CH_NB, n0 = k0 + CH_NB * (int)blockIdx.x;
  // this workgroup's columns of the block row, in flight during the elimination
  if (blockIdx.x > 0) {
    for (int e = tid; e < CH_NB * CH_NB; e += 256) {
      const int kk = e % CH_NB, nn_ = e / CH_NB;
      const cplx v = W[(k0 + kk) + (int64_t)np * (n0 + nn_)];
      Br[kk][nn_] = v.x;
      Bi[kk][nn_] = v.y;
    }
  }
  // thread (r, c) owns rows r + 16 x and columns c + 16 y; the lower triangle from the upper one
  const int r = tid & 15, c = tid >> 4;
  cplx a[4][4];
#pragma unroll
  for (int x = 0; x < 4; ++x)
#pragma unroll
    for (int y = 0; y < 4; ++y) {
      const int i = r + 16 * x, j = c + 16 * y;
      const cplx v = W[(k0 + (i < j ? i : j)) + (int64_t)np * (k0 + (i < j ? j : i))];
      a[x][y] = i < j ? v : (i == j ? mk(v.x, 0.0) : cconj(v));
    }
  if (r == 0)
#pragma unroll
    for (int y = 0; y < 4; ++y) rowb[0][c + 16 * y] = a[0][y];
  if (c == 0)
#pragma unroll
    for (int x = 0; x < 4; ++x) colb[0][r + 16 * x] = a[x][0];
  __syncthreads();
  bool ok = true;
  // elimination of column j from the rows below it, the multipliers taking its place: the strict
  // lower triangle becomes the inverse of the unit factor, the diagonal keeps the pivots
#pragma unroll
  for (int xj = 0; xj < 4; ++xj) {
    for (int jr = 0; jr < 16; ++jr) {
      const int j = 16 * xj + jr, par = j & 1;
      double piv = rowb[par][j].x;
      if (!(piv > 0.0)) {
        ok = false;
        piv = 1.0;
      }
      const double ip = 1.0 / piv;
      cplx rw[4];
#pragma unroll
      for (int y = 0; y < 4; ++y) rw[y] = rowb[par][c + 16 * y];
      // column j itself lies in the registers y = xj of the threads c = jr: a_ij is dropped and
      // -m takes its place (0 - m 1)
      const bool own = c == jr;
      if (own) rw[xj] = mk(1.0, 0.0);
#pragma unroll
      for (int x = xj; x < 4; ++x) {   // rows below 16 xj are done
        const int i = r + 16 * x;
        if (i > j) {
          const cplx m = cscale(colb[par][i], ip);
          if (own) a[x][xj] = mk(0.0, 0.0);
#pragma unroll
          for (int y = 0; y < 4; ++y) {
            a[x][y].x = fma(-m.x, rw[y].x, fma(m.y, rw[y].y, a[x][y].x));
            a[x][y].y = fma(-m.x, rw[y].y, fma(-m.y, rw[y].x, a[x][y].y));
          }
        }
      }
      // publish row and column j + 1 (static register indices: the next block of 16 at jr = 15)
      const int q = (j + 1) & 15;
      if (jr < 15) {
        if (r == q)
#pragma unroll
          for (int y = 0; y < 4; ++y) rowb[par ^ 1][c + 16 * y] = a[xj][y];
        if (c == q)
#pragma unroll
          for (int x = 0; x < 4; ++x) colb[par ^ 1][r + 16 * x] = a[x][xj];
      } else if (xj < 3) {
        if (r == 0)
#pragma unroll
          for (int y = 0; y < 4; ++y) rowb[par ^ 1][c + 16 * y] = a[xj < 3 ? xj + 1 : 3][y];
        if (c == 0)
#pragma unroll
          for (int x = 0; x < 4; ++x) colb[par ^ 1][r + 16 * x] = a[x][xj < 3 ? xj + 1 : 3];
      }
      __syncthreads();
    }
  }
  if (!ok && tid == 0 && blockIdx.x == 0) flag[b] = 1;
  // row i of the inverse factor: the unit inverse's row over the square root of its pivot
#pragma unroll
  for (int x = 0; x < 4; ++x)
#pragma unroll
    for (int y = 0; y < 4; ++y)
      if (r + 16 * x == c + 16 * y) colb[0][r + 16 * x] = a[x][y];
  __syncthreads();
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    const int i = r + 16 * x;
    const double pv = colb[0][i].x;
    const double s = 1.0 / sqrt(pv > 0.0 ? pv : 1.0);
#pragma unroll
    for (int y = 0; y < 4; ++y) {
      const int j = c + 16 * y;
      const cplx v = i > j ? cscale(a[x][y], s) : mk(i == j ? s : 0.0, 0.0);
      Ar[j][i] = v.x;   // [k][m]
      Ai[j][i] = v.y;
      if (blockIdx.x == 0 && b != 1) Li[nn * (b >> 1) + (k0 + i) + (int64_t)np * (k0 + j)] = v;
    }
  }
  __syncthreads();
  if (blockIdx.x == 0) return;
  // U[k0 + m, n0 + n] = sum_k Linv[m][k] W[k0 + k, n0 + n]
  const int lane = tid & 63, wave = tid >> 6;
  const int wm = (wave & 1) * 32, wn = (wave >> 1) * 32;
  d4 accr[2][2], acci[2][2];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y) {
      accr[x][y] = d4{0.0, 0.0, 0.0, 0.0};
      acci[x][y] = d4{0.0, 0.0, 0.0, 0.0};
    }
  for (int kk = 0; kk < CH_NB; kk += 4) {
    const int kl = kk + (lane >> 4);
    double ar[2], ai[2], br[2], bi[2];
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      ar[x] = Ar[kl][wm + 16 * x + (lane & 15)];
      ai[x] = Ai[kl][wm + 16 * x + (lane & 15)];
      br[x] = Br[kl][wn + 16 * x + (lane & 15)];
      bi[x] = Bi[kl][wn + 16 * x + (lane & 15)];
    }
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < 2; ++y) {
        accr[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar[x], br[y], accr[x][y], 0, 0, 0);
        accr[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(-ai[x], bi[y], accr[x][y], 0, 0, 0);
        acci[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar[x], bi[y], acci[x][y], 0, 0, 0);
        acci[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai[x], br[y], acci[x][y], 0, 0, 0);
      }
  }
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row = wm + 16 * x + (lane >> 4) + 4 * q, col = wn + 16 * y + (lane & 15);
        U[(k0 + row) + (int64_t)np * (n0 + col)] = mk(accr[x][y][q], acci[x][y][q]);
      }
}

// Lanczos on S^-1 = L^-H L^-1: w = S^-1 v_j is given; alpha_j, the next vector and beta_j.
// One workgroup; n <= 1024 * LZ_E.
constexpr int LZ_T = 1024, LZ_E = 2, LZ_STEPS = 256;
__global__ __launch_bounds__(LZ_T) void k_lanczos(int n, int j, const cplx* __restrict__ w, cplx* __restrict__ v,
                                                  cplx* __restrict__ vold, double* __restrict__ ab) {
  __shared__ double red[16];
  auto sum = [&](double x) {
    x = wave_add(x);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
    __syncthreads();
    double t = 0.0;
    for (int q = 0; q < 16; ++q) t += red[q];
    return t;
  };
  cplx wv[LZ_E], vv[LZ_E];
  const double bo = j > 0 ? ab[2 * (j - 1) + 1] : 0.0;
  double a = 0.0;
#pragma unroll
  for (int e = 0; e < LZ_E; ++e) {
    const int i = threadIdx.x + LZ_T * e;
    wv[e] = vv[e] = mk(0.0, 0.0);
    if (i < n) {
      vv[e] = v[i];
      wv[e] = w[i];
      if (j > 0) {
        const cplx o = vold[i];
        wv[e] = mk(wv[e].x - bo * o.x, wv[e].y - bo * o.y);
      }
    }
    a += vv[e].x * wv[e].x + vv[e].y * wv[e].y;
  }
  a = sum(a);
  double b2 = 0.0;
#pragma unroll
  for (int e = 0; e < LZ_E; ++e) {
    wv[e] = mk(wv[e].x - a * vv[e].x, wv[e].y - a * vv[e].y);
    b2 += cabs2(wv[e]);
  }
  const double b = sqrt(sum(b2)), ib = b > 0.0 ? 1.0 / b : 0.0;
#pragma unroll
  for (int e = 0; e < LZ_E; ++e) {
    const int i = threadIdx.x + LZ_T * e;
    if (i < n) {
      vold[i] = vv[e];
      v[i] = cscale(wv[e], ib);
    }
  }
  if (threadIdx.x == 0) {
    ab[2 * j] = a;
    ab[2 * j + 1] = b;
  }
}

// Steps j0 .. j1-1 of the same iteration in one workgroup for n <= LZS_N: L^-1 stays in this
// compute unit's reach (L2), a step is two triangular matrix-vector products and two sums.
// Thread (row r, part q) of LZS_P = 1024 / LZS_N sums the columns k = q mod LZS_P of row r for
// L^-1 v; a wave per column sums over rows for L^-H t.  5 us a step at n = 196 against 25 for
// four launches.
constexpr int LZS_N = 256, LZS_P = 1024 / LZS_N;
__global__ __launch_bounds__(1024) void k_lanczos_small(int n, int np, int j0, int j1, const cplx* __restrict__ Li,
                                                        cplx* __restrict__ vg, cplx* __restrict__ voldg,
                                                        double* __restrict__ ab) {
  __shared__ cplx v[LZS_N], vold[LZS_N], t[LZS_N], w[LZS_N], part[LZS_P][LZS_N];
  __shared__ double red[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  auto sum = [&](double x) {
    x = wave_add(x);
    __syncthreads();
    if (lane == 0) red[wave] = x;
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < 16; ++q) s += red[q];
    return s;
  };
  // all LZS_N entries: the rounds of eight below multiply the ones past n by zeros of L^-1, which
  // what an earlier workgroup left in LDS (a NaN) would survive
  if (tid < LZS_N) {
    v[tid] = tid < n ? vg[tid] : mk(0.0, 0.0);
    vold[tid] = tid < n && j0 > 0 ? voldg[tid] : mk(0.0, 0.0);
  }
  double bo = j0 > 0 ? ab[2 * (j0 - 1) + 1] : 0.0;
  __syncthreads();
  for (int j = j0; j < j1; ++j) {
    const int r = tid % LZS_N, q = tid / LZS_N;
    cplx acc = mk(0.0, 0.0);
    if (r < n) {
      // eight loads in flight (past the diagonal L^-1 holds zeros; np >= n columns)
      for (int k0 = q; k0 <= r; k0 += 8 * LZS_P) {
        cplx l[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int k = k0 + u * LZS_P;
          l[u] = k <= r ? Li[r + (int64_t)np * k] : mk(0.0, 0.0);
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) cfma(acc, l[u], v[min(k0 + u * LZS_P, LZS_N - 1)]);
      }
    }
    part[q][r] = acc;
    __syncthreads();
    if (tid < n) {
      cplx s = part[0][tid];
#pragma unroll
      for (int u = 1; u < LZS_P; ++u) s = cadd(s, part[u][tid]);
      t[tid] = s;
    }
    __syncthreads();
    for (int k0 = wave; k0 < n; k0 += 64) {   // w_k = sum_{i >= k} conj(Li_ik) t_i, four columns at a time
      cplx a[4];
#pragma unroll
      for (int h = 0; h < 4; ++h) a[h] = mk(0.0, 0.0);
#pragma unroll
      for (int u = 0; u < LZS_N / 64; ++u) {
        const int i = lane + 64 * u;
        if (64 * u >= n) break;   // uniform
        cplx l[4];
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          const int k = k0 + 16 * h;
          l[h] = (k < n && i >= k && i < n) ? Li[i + (int64_t)np * k] : mk(0.0, 0.0);
        }
        const cplx ti = i < n ? t[i] : mk(0.0, 0.0);
#pragma unroll
        for (int h = 0; h < 4; ++h) cfma(a[h], cconj(l[h]), ti);
      }
#pragma unroll
      for (int h = 0; h < 4; ++h) a[h] = wave_add(a[h]);
      if (lane == 0)
#pragma unroll
        for (int h = 0; h < 4; ++h)
          if (k0 + 16 * h < n) w[k0 + 16 * h] = a[h];
    }
    __syncthreads();
    cplx x = mk(0.0, 0.0), y = mk(0.0, 0.0);
    if (tid < n) {
      x = v[tid];
      y = mk(w[tid].x - bo * vold[tid].x, w[tid].y - bo * vold[tid].y);
    }
    const double a = sum(x.x * y.x + x.y * y.y);
    y = mk(y.x - a * x.x, y.y - a * x.y);
    const double b = sqrt(sum(cabs2(y))), ib = b > 0.0 ? 1.0 / b : 0.0;
    if (tid < n) {
      vold[tid] = x;
      v[tid] = cscale(y, ib);
    }
    if (tid == 0) {
      ab[2 * j] = a;
      ab[2 * j + 1] = b;
    }
    bo = b;
    __syncthreads();
  }
  if (tid < n) {
    vg[tid] = v[tid];
    voldg[tid] = vold[tid];
  }
}

// a start vector with a part along every direction: unit-modulus entries of an integer hash (the
// first steps of splitmix64's finaliser)
__global__ void k_lanczos_start(int n, cplx* __restrict__ v) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  uint64_t z = 0x9E3779B97F4A7C15ull * (uint64_t)(i + 1);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z ^= z >> 27;
  double sn, cs;
  sincospi(2.0 * (double)(z >> 11) * 0x1.0p-53, &sn, &cs);
  const double s = 1.0 / sqrt((double)n);
  v[i] = mk(cs * s, sn * s);
}

}  // namespace

int64_t chol_np(int64_t n) { return (n + CH_NB - 1) / CH_NB * CH_NB; }
int64_t chol_work_elems(int64_t n, int nmat) { return 2 * nmat * chol_np(n) * chol_np(n); }

void chol_factor(hipStream_t s, int64_t n, const cplx* S, int64_t lds, int nmat, const double* shifts, cplx* work,
                 cplx* Li, int* flags) {
  const int64_t np = chol_np(n), nn = np * np;
  DC2_CHECK(n >= 1 && n <= 4096 && nmat >= 1 && nmat <= 3, 1, "chol_factor: n must be in 1..4096");
  const int nb = (int)(np / CH_NB);
  cplx* W = work;
  cplx* U = W + nmat * nn;
  Shifts sh{{0.0, 0.0, 0.0}};
  for (int b = 0; b < nmat; ++b) sh.v[b] = shifts[b];
  DC2_HIP(hipMemsetAsync(flags, 0, 3 * sizeof(int), s));
  hipLaunchKernelGGL(k_chol_pack, dim3(cdiv(nn, 256)), dim3(256), 0, s, (int)n, (int)np, S, lds, nmat, sh, W);
  fill_zero(s, Li, nmat == 3 ? 2 * nn : nn);
  for (int kb = 0; kb < nb; ++kb) {
    hipLaunchKernelGGL(k_chol_step, dim3(nb - kb, nmat), dim3(256), 0, s, (int)np, kb, W, U, Li, flags);
    const int64_t k0 = (int64_t)kb * CH_NB, k1 = k0 + CH_NB;
    zherk_trailing(s, np - k1, CH_NB, U + k0 + np * k1, np, nn, W + k1 + np * k1, np, nn, nmat);
  }
  DC2_HIP(hipGetLastError());
}

void chol_invert(hipStream_t s, int64_t n, cplx* work, int nmat, int b, cplx* Li) {
  const int64_t np = chol_np(n), nn = np * np;
  const int nb = (int)(np / CH_NB);
  cplx* W = work;
  const cplx* U = work + nmat * nn + nn * b;
  const cplx one = mk(1.0, 0.0), mone = mk(-1.0, 0.0), zero = mk(0.0, 0.0);
  // merges of neighbouring blocks (sizes in units of CH_NB): blocks of c, the last one shorter;
  // T (in W, which the factorisation no longer needs) holds Z U12^H
  for (int64_t c = 1; c < nb; c *= 2) {
    const int64_t pairs = nb / (2 * c), step = 2 * c * CH_NB, h = c * CH_NB;
    if (pairs > 0) {
      zgemm(s, 'N', 'C', h, h, h, one, Li + h + np * h, np, step * (np + 1), U + np * h, np, step * (np + 1), zero, W, h,
            h * h, pairs);
      zgemm(s, 'N', 'N', h, h, h, mone, W, h, h * h, Li, np, step * (np + 1), zero, Li + h, np, step * (np + 1), pairs);
    }
    const int64_t rest = nb - 2 * c * pairs;   // a full block and a shorter one remain
    if (rest > c) {
      const int64_t o = pairs * step, t = (rest - c) * CH_NB;
      zgemm(s, 'N', 'C', t, h, t, one, Li + (o + h) * (np + 1), np, 0, U + o + np * (o + h), np, 0, zero, W, t, 0, 1);
      zgemm(s, 'N', 'N', t, h, h, mone, W, t, 0, Li + o * (np + 1), np, 0, zero, Li + (o + h) + np * o, np, 0, 1);
    }
  }
}

void chol_inverse(hipStream_t s, int64_t n, const cplx* S, int64_t lds, double sigma, cplx* work, cplx* Li, int* flags) {
  const double shifts[2] = {0.0, sigma};
  chol_factor(s, n, S, lds, 2, shifts, work, Li, flags);
  chol_invert(s, n, work, 2, 0, Li);
}

// ------------------------------------------------------------------ the lowest eigenvectors
//
// Subspace iteration with (G + delta)^-1 = L^-H L^-1 on LOW_P columns: two products with the
// explicit inverse factor and an orthonormalisation by the Cholesky factor of the columns'
// 64 x 64 Gram matrix per step.

namespace {

// start columns: unit-modulus entries of an integer hash (splitmix64's finaliser)
__global__ void k_low_start(int64_t count, int n, cplx* __restrict__ x) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= count) return;
  uint64_t z = 0x9E3779B97F4A7C15ull * (uint64_t)(i + 1);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z ^= z >> 31;
  double sn, cs;
  sincospi(2.0 * (double)(z >> 11) * 0x1.0p-53, &sn, &cs);
  const double s = 1.0 / sqrt((double)n);
  x[i] = mk(cs * s, sn * s);
}

}  // namespace

int64_t low_work_elems(int64_t n) { return 2 * n * LOW_P + 2 * 3 * LOW_P * LOW_P + 64; }

// X <- X L^-H with X^H X = L L^H, passes times: once keeps the iterated columns apart, the last
// step takes three, to orthonormality at rounding (one pass leaves eps times the condition of the
// columns' Gram matrix, which is far from 1)
static void low_orth(hipStream_t s, int64_t n, cplx* X, cplx* Y, cplx* small, int* flags, int passes) {
  const cplx one = mk(1.0, 0.0), zero = mk(0.0, 0.0);
  const int64_t p = LOW_P, pp = p * p;
  cplx *Gm = small, *U = small + pp, *Li = small + 2 * pp;
  for (int q = 0; q < passes; ++q) {
    zgemm(s, 'C', 'N', p, p, n, one, X, n, 0, X, n, 0, zero, Gm, p, 0, 1);
    hipLaunchKernelGGL(k_chol_step, dim3(1, 1), dim3(256), 0, s, (int)p, 0, Gm, U, Li, flags);
    zgemm(s, 'N', 'C', n, p, p, one, X, n, 0, Li, p, 0, zero, Y, n, 0, 1);
    DC2_HIP(hipMemcpyAsync(X, Y, n * p * sizeof(cplx), hipMemcpyDeviceToDevice, s));
  }
}

void low_start(hipStream_t s, int64_t n, cplx* X) {
  hipLaunchKernelGGL(k_low_start, dim3(cdiv(n * LOW_P, 256)), dim3(256), 0, s, n * LOW_P, (int)n, X);
  DC2_HIP(hipGetLastError());
}

void low_iterate(hipStream_t s, int64_t n, const cplx* G, const cplx* Li, int steps, cplx* X, cplx* work, cplx* H,
                 int* flags) {
  const int64_t np = chol_np(n), p = LOW_P;
  const cplx one = mk(1.0, 0.0), zero = mk(0.0, 0.0);
  cplx *Y = work, *Z = Y + n * p, *small = Z + n * p;
  DC2_HIP(hipMemsetAsync(flags, 0, 3 * sizeof(int), s));
  for (int t = 0; t < steps; ++t) {
    zgemm(s, 'N', 'N', n, p, n, one, Li, np, 0, X, n, 0, zero, Y, n, 0, 1);
    zgemm(s, 'C', 'N', n, p, n, one, Li, np, 0, Y, n, 0, zero, X, n, 0, 1);
    low_orth(s, n, X, Y, small, flags, t + 1 < steps ? 1 : 3);
  }
  zgemm(s, 'N', 'N', n, p, n, one, G, n, 0, X, n, 0, zero, Y, n, 0, 1);
  zgemm(s, 'C', 'N', p, p, n, one, X, n, 0, Y, n, 0, zero, H, p, 0, 1);
  DC2_HIP(hipGetLastError());
}

bool chol_lambda_min(hipStream_t s, int64_t n, const cplx* Li, cplx* work, double* host, double& lambda) {
  const int64_t np = chol_np(n);
  DC2_CHECK(n >= 1 && n <= (int64_t)LZ_T * LZ_E, 1, "chol_lambda_min: n must be in 1..2048");
  cplx *v = work, *vold = v + n, *t = vold + n, *w = t + n;
  double* ab = reinterpret_cast<double*>(w + n);
  const cplx one = mk(1.0, 0.0), zero = mk(0.0, 0.0);
  hipLaunchKernelGGL(k_lanczos_start, dim3(cdiv(n, 256)), dim3(256), 0, s, (int)n, v);
  const int steps = (int)std::min<int64_t>(n, LZ_STEPS);
  for (int j = 0, seen = 0; j < steps;) {
    const int stop = std::min(steps, j + (j == 0 ? 24 : 16));
    if (n <= LZS_N) {
      hipLaunchKernelGGL(k_lanczos_small, dim3(1), dim3(1024), 0, s, (int)n, (int)np, j, stop, Li, v, vold, ab);
      j = stop;
    }
    for (; j < stop; ++j) {
      zgemm(s, 'N', 'N', n, 1, n, one, Li, np, 0, v, n, 0, zero, t, n, 0, 1);
      zgemm(s, 'C', 'N', n, 1, n, one, Li, np, 0, t, n, 0, zero, w, n, 0, 1);
      hipLaunchKernelGGL(k_lanczos, dim3(1), dim3(LZ_T), 0, s, (int)n, j, w, v, vold, ab);
    }
    DC2_HIP(hipGetLastError());
    DC2_HIP(hipMemcpyAsync(host + 2 * seen, ab + 2 * seen, 2 * (j - seen) * sizeof(double), hipMemcpyDeviceToHost, s));
    DC2_HIP(hipStreamSynchronize(s));
    seen = j;
    // the largest eigenvalue theta of the tridiagonal by bisection on its Sturm count, and the
    // last component of its eigenvector by the three-term recurrence from the end
    double hi = 0.0;
    for (int i = 0; i < j; ++i)
      hi = std::max(hi, host[2 * i] + (i ? host[2 * i - 1] : 0.0) + (i + 1 < j ? host[2 * i + 1] : 0.0));
    if (!(hi > 0.0 && hi < 1e300)) return false;
    double lo = 0.0;
    for (int k = 0; k < 200 && hi - lo > 4e-16 * hi; ++k) {
      const double mid = 0.5 * (lo + hi);
      bool above = false;   // some eigenvalue > mid: a positive pivot of T - mid
      double d = 1.0;
      for (int i = 0; i < j && !above; ++i) {
        const double b = i ? host[2 * i - 1] : 0.0;
        d = host[2 * i] - mid - (i ? b * b / d : 0.0);
        above = d >= 0.0;
      }
      (above ? lo : hi) = mid;
    }
    const double theta = hi;
    double sq = 1.0, x = 1.0, xn = 0.0;   // x_{j-1} = 1, going down
    for (int i = j - 1; i > 0; --i) {
      const double b = host[2 * i - 1];
      if (!(b > 0.0)) break;   // an invariant subspace: the rest does not couple
      const double xp = ((theta - host[2 * i]) * x - (i + 1 < j ? host[2 * i + 1] : 0.0) * xn) / b;
      xn = x;
      x = xp;
      sq += x * x;
      if (sq > 1e280) break;
    }
    // residual of the Ritz pair against theta; the eigenvalue's error is its square over the gap
    if (host[2 * j - 1] <= 1e-7 * theta * std::sqrt(sq)) {
      lambda = 1.0 / theta;
      return true;
    }
  }
  return false;
}

}  // namespace dc2
