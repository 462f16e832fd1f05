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
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    a += __shfl_xor(a, o, 64);
    b += __shfl_xor(b, o, 64);
  }
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
  zgemm(s, 'N', 'N', n, npert, n, one, Bt, n, 0, X, n, 0, zero, Q, n, 0, 1);
  hipLaunchKernelGGL(k_cg_energy, dim3((unsigned)npert), dim3(CG_T), 0, s, ni, alpha, Y, X, Q, 1e-24, partial, state);
  sum_partials(s, npert, partial, out2);
  return poll();
}

}  // namespace dc2
