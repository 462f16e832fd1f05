// Complex FP64 GEMM on CDNA4 matrix cores (v_mfma_f64_16x16x4f64).
//
// One workgroup = 4 wave64s along m, each with 16 rows and up to 64 columns of complex C in
// 16x16 MFMA tiles; a complex multiply-add is four real MFMAs.  Operands go through
// double-buffered LDS as complex numbers.
//
// Used for: the four one-index integral transforms (module_intra.F90), the
// RDM contractions (density_matrix.F90), the V contractions and the
// (U L^-1/2)^H B (U L^-1/2) products of every solve_X_subspace.  Single products
// whose output has too few 64x64 tiles (the block Davidson of the CI matrix) go to
// plain FP64 kernels instead: one wave per output row over a long K, one thread per
// output over a short K, one thread per row for at most 8 columns over a long K.
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdlib>
#include <map>
#include <mutex>
#include <tuple>

#include "dc2_common.hpp"

namespace dc2 {

typedef double d4 __attribute__((ext_vector_type(4)));

namespace {
constexpr int64_t kLd32 = 1ll << 22;   // below it the byte offsets within a tile fit 32 bits (63 ld 16 < 2^32)
constexpr int BM = 64, BK = 16;   // rows of an output tile; granule of the split-K chunks

// tri: zeros the operands are known to have, which end a tile's K loop early: TRI_A op(A) lower
// triangular (k <= m), TRI_B op(B) upper triangular (k <= n)
enum { TRI_NONE = 0, TRI_A = 1, TRI_B = 2 };
// k_zgemm: one workgroup = 4 waves along m, each with FN fragments of 16 x 16 (a tile of 64 x
// 16 FN), K in tiles of KB through double-buffered LDS, one workgroup barrier per K tile.
//
// What bounds it: the FP64 matrix units, and every vector instruction beside them (at 0.9
// others per product the units were busy 84% of the time, at 0.24-0.49 94-96%).  So the loop
// over full K tiles has no branch and no edge test: it runs in rounds of two tiles (constant
// LDS offsets), offsets are formed once, rows and columns past the edges are read from the
// last valid one (their outputs are never stored), and the partial K tile at the end has its
// own code, zeroed in both operands and multiplied up to its last group of four.  A column
// tile at the edge multiplies only the fragments that hold columns (zg_loop exists for every
// count).  The next tile's loads are issued before the current one is multiplied, and stored to
// the other buffer after it.  __launch_bounds__(256, 2): with the whole register file to itself
// the compiler kept the accumulators in AGPRs and moved all of them to VGPRs and back per tile.
//
// Measured against the kernel it replaces (64 x 64 tiles, single-buffered planes): 252000 x 280
// x 280 'T','N' 3170 -> 2250 us (70 TF/s), 41984 x 164 x 164 238 -> 153, 2352000 x 30 x 30
// 870 -> 523, 322752 x 14 x 14 72 -> 26 (5.6 TB/s), 1274^3 'C','N' 410 -> 300, 2048^3 1190 -> 970.
template <char OPA, char OPB, int FN, int KB>
struct ZgTile {
  static constexpr int TM = BM, TN = 16 * FN;
  static constexpr bool AK = OPA != 'N', BKc = OPB == 'N' || OPB == 'R';   // contiguous along k
  static constexpr int NA = TM * KB / 256, NB = (TN * KB + 255) / 256;
  // rows of LDS padded by one element: 2.8 conflict cycles per LDS instruction, against 17 with
  // none, 5 with two and 10 with four (counters, 'T','N')
  static constexpr int LA = TM + 1, LB = TN + 1;
};

// the part of the kernel that depends on the number F of fragments with valid columns
template <char OPA, char OPB, int FN, int KB, int F, class OFF>
__device__ __forceinline__ void zg_loop(const cplx* __restrict__ At, const cplx* __restrict__ Bt, int64_t lda, int64_t ldb,
                                        int mrem, int nrem, int ktot, cplx* __restrict__ As, cplx* __restrict__ Bs,
                                        d4 (&accr)[FN], d4 (&acci)[FN]) {
  using T = ZgTile<OPA, OPB, FN, KB>;
  constexpr int TM = T::TM, TN = T::TN, NA = T::NA, NB = T::NB, LA = T::LA, LB = T::LB;
  constexpr bool AK = T::AK, BKc = T::BKc;
  const int tid = threadIdx.x, lane = tid & 63, wm = (tid >> 6) * 16;
  const int64_t stepA = AK ? KB : lda * KB, stepB = BKc ? KB : ldb * KB;
  cplx ra[NA], rb[NB];
  OFF oa[NA], ob[NB];   // byte offsets within a tile
#pragma unroll
  for (int r = 0; r < NA; ++r) {
    const int e = tid + 256 * r, mm = AK ? e / KB : e % TM, kk = AK ? e % KB : e / TM;
    const int m = mm < mrem ? mm : mrem - 1;
    oa[r] = (OFF)(16 * (AK ? lda * m + kk : m + lda * kk));
  }
#pragma unroll
  for (int r = 0; r < NB; ++r) {
    const int e = tid + 256 * r, nn = BKc ? e / KB : e % TN, kk = (BKc ? e % KB : e / TN) % KB;
    const int n = nn < nrem ? nn : nrem - 1;
    ob[r] = (OFF)(16 * (BKc ? ldb * n + kk : n + ldb * kk));
  }
  auto at = [](const cplx* p, OFF o) {
    return *reinterpret_cast<const cplx*>(reinterpret_cast<const char*>(p) + o);
  };
  auto gload = [&]() {
#pragma unroll
    for (int r = 0; r < NA; ++r) ra[r] = at(At, oa[r]);
#pragma unroll
    for (int r = 0; r < NB; ++r) rb[r] = at(Bt, ob[r]);
  };
  // the last, partial tile: read up to its last k, zero past it
  auto gload_part = [&](int krem) {
#pragma unroll
    for (int r = 0; r < NA; ++r) {
      const int e = tid + 256 * r, kk = AK ? e % KB : e / TM;
      ra[r] = at(At, kk < krem ? oa[r] : oa[r] - (OFF)(16 * (AK ? 1 : lda) * (kk - krem + 1)));
      if (kk >= krem) ra[r] = mk(0.0, 0.0);
    }
#pragma unroll
    for (int r = 0; r < NB; ++r) {
      const int e = tid + 256 * r, kk = (BKc ? e % KB : e / TN) % KB;
      rb[r] = at(Bt, kk < krem ? ob[r] : ob[r] - (OFF)(16 * (BKc ? 1 : ldb) * (kk - krem + 1)));
      if (kk >= krem) rb[r] = mk(0.0, 0.0);
    }
  };
  // LDS positions of this thread's elements and fragments in buffer 0 (bytes; the other buffer
  // is AB / BB further on)
  constexpr int AB = KB * LA, BB = KB * LB;
  auto sstore = [&](int buf) {
    cplx* as = As + buf * AB;
    cplx* bs = Bs + buf * BB;
#pragma unroll
    for (int r = 0; r < NA; ++r) {
      const int e = tid + 256 * r, mm = AK ? e / KB : e % TM, kk = AK ? e % KB : e / TM;
      as[kk * LA + mm] = OPA == 'C' ? cconj(ra[r]) : ra[r];
    }
#pragma unroll
    for (int r = 0; r < NB; ++r) {
      const int e = tid + 256 * r, nn = BKc ? e / KB : e % TN, kk = BKc ? e % KB : e / TN;
      if (TN * KB % 256 == 0 || e < TN * KB) bs[kk * LB + nn] = (OPB == 'R' || OPB == 'C') ? cconj(rb[r]) : rb[r];
    }
  };
  const cplx* as0 = As + (lane >> 4) * LA + wm + (lane & 15);
  const cplx* bs0 = Bs + (lane >> 4) * LB + (lane & 15);
  auto mul4 = [&](int buf, int kk) {   // four k of the tile in buffer buf
    cplx b[F];
    const cplx a = as0[buf * AB + kk * LA];
#pragma unroll
    for (int j = 0; j < F; ++j) b[j] = bs0[buf * BB + kk * LB + 16 * j];
    // the transposed fragment (rows n), so that a lane's column index runs along m: the stores
    // of C write 16 consecutive elements; dependent products are 2 F apart
#pragma unroll
    for (int j = 0; j < F; ++j) {
      accr[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(b[j].x, a.x, accr[j], 0, 0, 0);
      acci[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(b[j].y, a.x, acci[j], 0, 0, 0);
    }
    const double na = -a.y;
#pragma unroll
    for (int j = 0; j < F; ++j) {
      accr[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(b[j].y, na, accr[j], 0, 0, 0);
      acci[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(b[j].x, a.y, acci[j], 0, 0, 0);
    }
  };
  auto mul = [&](int buf) {
#pragma unroll
    for (int kk = 0; kk < KB; kk += 4) mul4(buf, kk);
  };
  const int nfull = ktot / KB, rem = ktot - nfull * KB;
  if (nfull > 0) {
    gload();
    sstore(0);
    __syncthreads();
    // two tiles per round, so that the buffer is a constant and the loop has no branches
    int t = 1;
    for (; t + 1 < nfull; t += 2) {
      At += stepA;
      Bt += stepB;
      gload();
      mul(0);
      sstore(1);
      __syncthreads();
      At += stepA;
      Bt += stepB;
      gload();
      mul(1);
      sstore(0);
      __syncthreads();
    }
    const bool odd = t < nfull;
    if (odd) {
      At += stepA;
      Bt += stepB;
      gload();
      mul(0);
      sstore(1);
      __syncthreads();
    }
    // the last full tile, in buffer odd
    if (rem > 0) {
      At += stepA;
      Bt += stepB;
      gload_part(rem);
    }
    mul(odd);
    if (rem > 0) {
      sstore(!odd);
      __syncthreads();
      for (int kk = 0; kk < rem; kk += 4) mul4(!odd, kk);
    }
  } else if (rem > 0) {
    gload_part(rem);
    sstore(0);
    __syncthreads();
    for (int kk = 0; kk < rem; kk += 4) mul4(0, kk);
  }
}

// blockIdx.z = batch index * sk + K-split index; split kz covers K in [kz*kchunk, (kz+1)*kchunk)
// and writes its partial product to C + kz * sC (the split-K workspace) when sk > 1.  UPPER:
// only the tiles that reach the upper triangle (a Hermitian product; the others leave at
// once).  OFF: offsets within a tile, 32 bits where the leading dimensions allow it.
template <char OPA, char OPB, int FN, int KB, bool UPPER = false, class OFF = uint32_t>
__global__ __launch_bounds__(256, 2) void k_zgemm(int64_t M, int64_t N, int64_t Kfull, cplx alpha,
                                                  const cplx* __restrict__ A, int64_t lda, int64_t sA,
                                                  const cplx* __restrict__ B, int64_t ldb, int64_t sB,
                                                  cplx beta, cplx* __restrict__ C, int64_t ldc, int64_t sC, int sk,
                                                  int64_t kchunk, int tri) {
  using T = ZgTile<OPA, OPB, FN, KB>;
  constexpr int TM = T::TM, TN = T::TN;
  int64_t mt, nt;
  xcd_tile(gridDim.x, gridDim.y, blockIdx.x, blockIdx.y, mt, nt);
  // An XCD gets consecutive row blocks, whose work grows or shrinks along a triangle: the first
  // with the last, the second with the last but one ... evens it out (upper tiles of m = 1274, k
  // = 3432: 479 us, 686 with the rows in order)
  if (UPPER || tri != TRI_NONE) mt = (mt & 1) ? gridDim.x - 1 - mt / 2 : mt / 2;
  if (UPPER && mt * TM > nt * TN + TN - 1) return;   // uniform
  __shared__ cplx As[2 * KB * T::LA], Bs[2 * KB * T::LB];
  const int64_t bz = blockIdx.z / sk, kz = blockIdx.z % sk;
  C += (sk > 1 ? bz * sk + kz : bz) * sC;
  const int64_t kbeg = kz * kchunk;
  int64_t kend = (kbeg + kchunk < Kfull) ? kbeg + kchunk : Kfull;
  if (tri == TRI_A && kend > (mt + 1) * TM) kend = (mt + 1) * TM;
  if (tri == TRI_B && kend > (nt + 1) * TN) kend = (nt + 1) * TN;
  const int64_t m0 = mt * TM, n0 = nt * TN;
  const int mrem = (int)(M - m0 < TM ? M - m0 : TM), nrem = (int)(N - n0 < TN ? N - n0 : TN);
  const cplx* At = A + bz * sA + (T::AK ? lda * m0 + kbeg : m0 + lda * kbeg);
  const cplx* Bt = B + bz * sB + (T::BKc ? ldb * n0 + kbeg : n0 + ldb * kbeg);
  d4 accr[FN], acci[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    accr[j] = d4{0.0, 0.0, 0.0, 0.0};
    acci[j] = d4{0.0, 0.0, 0.0, 0.0};
  }
  const int f = (nrem + 15) / 16, ktot = (int)(kend - kbeg);   // uniform
  if (f == FN) zg_loop<OPA, OPB, FN, KB, FN, OFF>(At, Bt, lda, ldb, mrem, nrem, ktot, As, Bs, accr, acci);
  else if (FN > 1 && f == 1) zg_loop<OPA, OPB, FN, KB, 1, OFF>(At, Bt, lda, ldb, mrem, nrem, ktot, As, Bs, accr, acci);
  else if (FN > 2 && f == 2)
    zg_loop<OPA, OPB, FN, KB, (FN > 2 ? 2 : 1), OFF>(At, Bt, lda, ldb, mrem, nrem, ktot, As, Bs, accr, acci);
  else if (FN > 3 && f == 3)
    zg_loop<OPA, OPB, FN, KB, (FN > 3 ? 3 : 1), OFF>(At, Bt, lda, ldb, mrem, nrem, ktot, As, Bs, accr, acci);
  // D[row][col] of a 16x16 MFMA tile sits in element (row / 4) of lane col + 16 * (row % 4)
  // (measured on gfx950 with a one-hot probe of the builtin); rows are n here
  const int lane = threadIdx.x & 63, wm = (threadIdx.x >> 6) * 16;
  const bool beta_zero = (beta.x == 0.0 && beta.y == 0.0);
  const int64_t row = m0 + wm + (lane & 15);
#pragma unroll
  for (int j = 0; j < FN; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t col = n0 + 16 * j + (lane >> 4) + 4 * r;
      if (row < M && col < N) {
        const cplx acc = mk(accr[j][r], acci[j][r]);
        cplx out = cmul(alpha, acc);
        if (!beta_zero) cfma(out, beta, C[row + ldc * col]);
        C[row + ldc * col] = out;
      }
    }
}

// ---- shapes with too few output tiles for the MFMA kernel (the block Davidson of the CI
// matrix: Rayleigh-matrix columns, Gram-Schmidt coefficients, subspace updates, H x)

__device__ inline cplx out_value(cplx acc, cplx alpha, cplx beta, const cplx* c) {
  cplx out = cmul(alpha, acc);
  if (beta.x != 0.0 || beta.y != 0.0) cfma(out, beta, *c);
  return out;
}

// op(A) = A^H or A^T, op(B) = B or conj(B) with a small output (M x N): both operands are read
// along K, contiguous.  One wave per row m and up to 4 columns; the lanes stride over K and
// their partial sums meet in a fixed butterfly, so the result does not depend on timing.
constexpr int DOT_NB = 4, DOT_U = 4;
template <char OPA, char OPB>
__global__ __launch_bounds__(256) void k_zgemm_dot(int64_t M, int64_t N, int64_t K, cplx alpha,
                                                   const cplx* __restrict__ A, int64_t lda,
                                                   const cplx* __restrict__ B, int64_t ldb, cplx beta,
                                                   cplx* __restrict__ C, int64_t ldc) {
  const int lane = threadIdx.x & 63;
  const int64_t w = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);   // wave-uniform
  const int64_t nb = (N + DOT_NB - 1) / DOT_NB;
  if (w >= M * nb) return;
  const int64_t m = w % M, n0 = (w / M) * DOT_NB;
  const int nn = (int)(N - n0 < DOT_NB ? N - n0 : DOT_NB);
  cplx acc[DOT_NB];
#pragma unroll
  for (int j = 0; j < DOT_NB; ++j) acc[j] = mk(0.0, 0.0);
  const cplx* a = A + lda * m;
  const cplx* b = B + ldb * n0;
  // DOT_U strides of K per round: all their loads are issued before the first multiply
  for (int64_t k0 = lane; k0 < K; k0 += 64 * DOT_U) {
    cplx x[DOT_U], y[DOT_U][DOT_NB];
#pragma unroll
    for (int u = 0; u < DOT_U; ++u) {
      const int64_t k = k0 + 64 * u;
      x[u] = k < K ? a[k] : mk(0.0, 0.0);
#pragma unroll
      for (int j = 0; j < DOT_NB; ++j) y[u][j] = (k < K && j < nn) ? b[k + ldb * j] : mk(0.0, 0.0);
    }
#pragma unroll
    for (int u = 0; u < DOT_U; ++u) {
      if (k0 + 64 * u >= K) break;
      const cplx xv = OPA == 'C' ? cconj(x[u]) : x[u];
#pragma unroll
      for (int j = 0; j < DOT_NB; ++j)
        if (j < nn) cfma(acc[j], xv, OPB == 'R' ? cconj(y[u][j]) : y[u][j]);
    }
  }
#pragma unroll
  for (int j = 0; j < DOT_NB; ++j) {
    double re = acc[j].x, im = acc[j].y;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      re += __shfl_xor(re, off);
      im += __shfl_xor(im, off);
    }
    acc[j] = mk(re, im);
  }
  if (lane < nn) {
    cplx s = acc[0];
#pragma unroll
    for (int j = 1; j < DOT_NB; ++j)
      if (lane == j) s = acc[j];
    cplx* c = C + m + ldc * (n0 + lane);
    *c = out_value(s, alpha, beta, c);
  }
}

// The same products with very few outputs (the block Davidson's Rayleigh columns and
// Gram-Schmidt coefficients: at most a few hundred rows over K = ndet): one workgroup per row m
// and up to 4 columns, its 256 threads striding over K; the partial sums meet in a butterfly
// per wave and then in wave order through LDS, so the result does not depend on timing.
template <char OPA, char OPB>
__global__ __launch_bounds__(256) void k_zgemm_dotwg(int64_t M, int64_t N, int64_t K, cplx alpha,
                                                     const cplx* __restrict__ A, int64_t lda,
                                                     const cplx* __restrict__ B, int64_t ldb, cplx beta,
                                                     cplx* __restrict__ C, int64_t ldc) {
  __shared__ cplx part[4][DOT_NB];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t w = blockIdx.x;
  const int64_t m = w % M, n0 = (w / M) * DOT_NB;
  const int nn = (int)(N - n0 < DOT_NB ? N - n0 : DOT_NB);
  cplx acc[DOT_NB];
#pragma unroll
  for (int j = 0; j < DOT_NB; ++j) acc[j] = mk(0.0, 0.0);
  const cplx* a = A + lda * m;
  const cplx* b = B + ldb * n0;
  for (int64_t k0 = tid; k0 < K; k0 += 256 * DOT_U) {
    cplx x[DOT_U], y[DOT_U][DOT_NB];
#pragma unroll
    for (int u = 0; u < DOT_U; ++u) {
      const int64_t k = k0 + 256 * u;
      x[u] = k < K ? a[k] : mk(0.0, 0.0);
#pragma unroll
      for (int j = 0; j < DOT_NB; ++j) y[u][j] = (k < K && j < nn) ? b[k + ldb * j] : mk(0.0, 0.0);
    }
#pragma unroll
    for (int u = 0; u < DOT_U; ++u) {
      if (k0 + 256 * u >= K) break;
      const cplx xv = OPA == 'C' ? cconj(x[u]) : x[u];
#pragma unroll
      for (int j = 0; j < DOT_NB; ++j)
        if (j < nn) cfma(acc[j], xv, OPB == 'R' ? cconj(y[u][j]) : y[u][j]);
    }
  }
#pragma unroll
  for (int j = 0; j < DOT_NB; ++j) {
    double re = acc[j].x, im = acc[j].y;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      re += __shfl_xor(re, off);
      im += __shfl_xor(im, off);
    }
    if (lane == 0) part[wave][j] = mk(re, im);
  }
  __syncthreads();
  if (tid < nn) {
    cplx s = part[0][tid];
#pragma unroll
    for (int q = 1; q < 4; ++q) s = cadd(s, part[q][tid]);
    cplx* c = C + m + ldc * (n0 + tid);
    *c = out_value(s, alpha, beta, c);
  }
}

// op(A) = A, op(B) = B or conj(B) with a short K: one thread per output element
template <char OPB>
__global__ __launch_bounds__(256) void k_zgemm_smallk(int64_t M, int64_t N, int64_t K, cplx alpha,
                                                      const cplx* __restrict__ A, int64_t lda,
                                                      const cplx* __restrict__ B, int64_t ldb, cplx beta,
                                                      cplx* __restrict__ C, int64_t ldc) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= M * N) return;
  const int64_t m = i % M, n = i / M;
  cplx acc = mk(0.0, 0.0);
  for (int64_t k = 0; k < K; ++k) {
    cplx y = B[k + ldb * n];
    if (OPB == 'R') y = cconj(y);
    cfma(acc, A[m + lda * k], y);
  }
  cplx* c = C + m + ldc * n;
  *c = out_value(acc, alpha, beta, c);
}

// op(A) = A, op(B) = B or conj(B) with at most TS_NMAX columns and a long K: thread = row m,
// all columns; blockIdx.y = K-split index, partial products to W[kz][n][m] (summed by
// k_splitk_reduce in a fixed order)
constexpr int TS_NMAX = 8, TS_U = 8, TS_KMAX = 64;
template <char OPB>
__global__ __launch_bounds__(256) void k_zgemm_tall(int64_t M, int64_t N, int64_t K, const cplx* __restrict__ A,
                                                    int64_t lda, const cplx* __restrict__ B, int64_t ldb,
                                                    cplx* __restrict__ W, int64_t kchunk) {
  __shared__ cplx Bs[TS_KMAX][TS_NMAX];   // this split's rows of op(B), read as broadcasts
  const int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t kz = blockIdx.y, k0 = kz * kchunk;
  const int kc = (int)((k0 + kchunk < K ? k0 + kchunk : K) - k0);   // <= TS_KMAX (host-checked)
  for (int e = threadIdx.x; e < kc * N; e += blockDim.x) {
    const int kk = e % kc, j = e / kc;
    const cplx y = B[k0 + kk + ldb * j];
    Bs[kk][j] = OPB == 'R' ? cconj(y) : y;
  }
  __syncthreads();
  if (m >= M) return;
  cplx acc[TS_NMAX];
#pragma unroll
  for (int j = 0; j < TS_NMAX; ++j) acc[j] = mk(0.0, 0.0);
  const cplx* a = A + m + lda * k0;
  // TS_U rows of K per round: their loads of A are issued before the first multiply
  for (int kb = 0; kb < kc; kb += TS_U) {
    cplx x[TS_U];
#pragma unroll
    for (int u = 0; u < TS_U; ++u) x[u] = kb + u < kc ? a[lda * (kb + u)] : mk(0.0, 0.0);
#pragma unroll
    for (int u = 0; u < TS_U; ++u) {
      if (kb + u >= kc) break;
#pragma unroll
      for (int j = 0; j < TS_NMAX; ++j)
        if (j < N) cfma(acc[j], x[u], Bs[kb + u][j]);
    }
  }
  cplx* w = W + M * N * kz + m;
#pragma unroll
  for (int j = 0; j < TS_NMAX; ++j)   // static indices: acc stays in registers
    if (j < N) w[M * j] = acc[j];
}

// the strict lower triangle as the conjugate of the upper one, the diagonal real
__global__ void k_lower_from_upper(int64_t m, cplx* __restrict__ C, int64_t ldc) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= m * m) return;
  const int64_t i = t % m, j = t / m;
  if (i > j) C[i + ldc * j] = cconj(C[j + ldc * i]);
  else if (i == j) C[i + ldc * j].y = 0.0;
}

// C = sum_kz W[kz] on and above the diagonal (the split-K partials of a Hermitian product,
// summed in a fixed order), the strict lower triangle as the conjugate of the upper one
__global__ void k_herk_reduce(int64_t m, int sk, const cplx* __restrict__ W, cplx* __restrict__ C, int64_t ldc) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= m * m) return;
  const int64_t i = t % m, j = t / m;
  if (i > j) return;
  cplx acc = mk(0.0, 0.0);
  int z = 0;
  for (; z + 4 <= sk; z += 4) {
    cplx v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = W[t + m * m * (z + u)];
#pragma unroll
    for (int u = 0; u < 4; ++u) acc = cadd(acc, v[u]);
  }
  for (; z < sk; ++z) acc = cadd(acc, W[t + m * m * z]);
  C[i + ldc * j] = acc;
  if (i < j) C[j + ldc * i] = cconj(acc);
}

// C = alpha * sum_kz W[kz] + beta * C (the split-K partial products, fixed summation order);
// blockIdx.y: the product of a batch (partials W + (bz sk + kz) M N, output C + bz sC)
__global__ void k_splitk_reduce(int64_t M, int64_t N, int sk, const cplx* __restrict__ W, cplx alpha, cplx beta,
                                cplx* __restrict__ C, int64_t ldc, int64_t sC) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= M * N) return;
  W += (int64_t)blockIdx.y * sk * M * N;
  C += (int64_t)blockIdx.y * sC;
  const int64_t m = i % M, n = i / M;
  cplx acc = mk(0.0, 0.0);
  int z = 0;
  for (; z + 8 <= sk; z += 8) {   // eight loads in flight, summed in order
    cplx v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = W[i + M * N * (z + u)];
#pragma unroll
    for (int u = 0; u < 8; ++u) acc = cadd(acc, v[u]);
  }
  for (; z < sk; ++z) acc = cadd(acc, W[i + M * N * z]);
  cplx out = cmul(alpha, acc);
  if (beta.x != 0.0 || beta.y != 0.0) cfma(out, beta, C[m + ldc * n]);
  C[m + ldc * n] = out;
}

// grow-only split-K workspaces, one per stream (kernels on one stream run in order).  The
// owner of a stream releases its workspace before destroying the stream; the map itself is
// never destroyed, so no device memory is freed by static destructors at process exit,
// when the HIP runtime may already be gone.
std::mutex g_ws_mu;
std::map<hipStream_t, DevBuf<cplx>>* g_ws = new std::map<hipStream_t, DevBuf<cplx>>;
cplx* splitk_workspace(hipStream_t s, size_t n) {
  std::lock_guard<std::mutex> lk(g_ws_mu);
  DevBuf<cplx>& b = (*g_ws)[s];
  b.ensure(n);
  return b.get();
}

GemmStats* g_stats = nullptr;
// The variants of k_zgemm: 1 FN 4, KB 8; 2 FN 2, KB 16; 3 FN 1, KB 16; 4 FN 1, KB 8
struct Variant {
  int fn, kb;
};
constexpr Variant kVariants[5] = {{0, 0}, {4, 8}, {2, 16}, {1, 16}, {1, 8}};

// The variant of a product by its sizes.  FN 4 keeps the matrix units busiest (A is read once
// per 64 columns) and needs at most 64 columns or more than four tiles per compute unit to do so;
// short of that the narrower tiles spread the product over more workgroups (1274 x 280 x 1274:
// 76 us with FN 1, 114 with FN 4; 2048^3: 968 with FN 2, 1010 with FN 4).  At most 32 columns
// take the tile they fill, and K <= 8 the shorter K tile (600000 x 8 x 8: 24 us against 33).
int pick_variant(int64_t M, int64_t N, int64_t K, int64_t batch) {
  const int64_t mt = cdiv(M, BM) * batch;
  if (N <= 16) return K <= 8 ? 4 : 3;
  if (N <= 32) return mt >= 256 ? 2 : 3;
  if (N <= 64 ? mt >= 256 : mt * cdiv(N, 64) > 1024) return 1;
  return mt * cdiv(N, 32) > 1024 ? 2 : 3;
}

// DC2_GEMM_VARIANT: 1..4 that variant for every product, 0 no kernels for skinny shapes
int g_variant = [] {
  const char* v = std::getenv("DC2_GEMM_VARIANT");
  return v ? std::atoi(v) : -1;
}();
std::mutex g_stats_mu;
thread_local int g_tag = 0;
thread_local bool g_no_ws = false;

// tuned choices by exact shape (heap, never destroyed; looked up only when not empty)
struct TuneKey {
  char oa, ob;
  int64_t M, N, K, batch;
  bool operator<(const TuneKey& o) const {
    return std::tie(oa, ob, M, N, K, batch) < std::tie(o.oa, o.ob, o.M, o.N, o.K, o.batch);
  }
};
struct TuneChoice {
  int variant, split;
};
std::mutex g_tune_mu;
std::map<TuneKey, TuneChoice>* g_tune = new std::map<TuneKey, TuneChoice>;
std::atomic<bool> g_tune_any{false};

bool tuned_choice(char oa, char ob, int64_t M, int64_t N, int64_t K, int64_t batch, TuneChoice& c) {
  if (!g_tune_any.load(std::memory_order_relaxed)) return false;
  std::lock_guard<std::mutex> lk(g_tune_mu);
  auto it = g_tune->find(TuneKey{oa, ob, M, N, K, batch});
  if (it == g_tune->end()) return false;
  c = it->second;
  return true;
}

// Kernels for the shapes the 64x64 MFMA tiles serve badly (single products only): small
// outputs with A read along K (k_zgemm_dot), a short K (k_zgemm_smallk), at most 8 columns
// and a long K (k_zgemm_tall).  Returns false when the MFMA kernel is the one to use.
template <char OPA, char OPB>
bool launch_skinny(hipStream_t s, int64_t M, int64_t N, int64_t K, cplx alpha, const cplx* A, int64_t lda,
                   const cplx* B, int64_t ldb, cplx beta, cplx* C, int64_t ldc) {
  constexpr bool b_along_k = OPB == 'N' || OPB == 'R';
  if constexpr ((OPA == 'C' || OPA == 'T') && b_along_k) {
    // a few outputs, or a matrix-vector product over a long K (one wave per output row
    // reads its column of A once; on 64 x 64 MFMA tiles N = 1 would use 1/64 of each tile)
    if (M * N > 2048 && !(N <= DOT_NB && K >= 256)) return false;
    const int64_t waves = M * ((N + DOT_NB - 1) / DOT_NB);
    if (waves < 512 && K >= 1024) {   // too few rows to keep the device busy: a workgroup per row
      hipLaunchKernelGGL((k_zgemm_dotwg<OPA, OPB>), dim3((unsigned)waves), dim3(256), 0, s, M, N, K, alpha, A,
                         lda, B, ldb, beta, C, ldc);
      return true;
    }
    hipLaunchKernelGGL((k_zgemm_dot<OPA, OPB>), dim3((unsigned)cdiv(waves, 4)), dim3(256), 0, s, M, N, K, alpha, A,
                       lda, B, ldb, beta, C, ldc);
    return true;
  } else if constexpr (OPA == 'N' && b_along_k) {
    if (K <= 64 && M * N <= 65536) {
      hipLaunchKernelGGL((k_zgemm_smallk<OPB>), dim3((unsigned)cdiv(M * N, 256)), dim3(256), 0, s, M, N, K, alpha, A,
                         lda, B, ldb, beta, C, ldc);
      return true;
    }
    if (N > TS_NMAX || K <= 64 || M > 65536 || g_no_ws) return false;
    const int64_t rb = cdiv(M, 256);
    const int64_t want = std::max<int64_t>(cdiv(K, TS_KMAX), std::min<int64_t>({cdiv(256, rb), 32, cdiv(K, 16)}));
    const int64_t kchunk = cdiv(K, want), sk = cdiv(K, kchunk);
    if (kchunk > TS_KMAX || sk >= 65536) return false;
    cplx* W = splitk_workspace(s, (size_t)sk * M * N);
    hipLaunchKernelGGL((k_zgemm_tall<OPB>), dim3((unsigned)rb, (unsigned)sk), dim3(256), 0, s, M, N, K, A, lda, B,
                       ldb, W, kchunk);
    hipLaunchKernelGGL(k_splitk_reduce, dim3(cdiv(M * N, 256)), dim3(256), 0, s, M, N, (int)sk, W, alpha, beta, C,
                       ldc, (int64_t)0);
    return true;
  }
  return false;
}

// force_variant > 0: that MFMA variant and split-K factor force_split (the tuner's trials; no
// skinny kernels, no table lookup)
template <char OPA, char OPB>
void launch(hipStream_t s, int64_t M, int64_t N, int64_t K, cplx alpha, const cplx* A, int64_t lda, int64_t sA,
            const cplx* B, int64_t ldb, int64_t sB, cplx beta, cplx* C, int64_t ldc, int64_t sC, int64_t batch,
            int force_variant = 0, int force_split = 1) {
  GemmRecord r{};
  const bool acct = g_stats && g_stats->on;
  if (acct) {
    DC2_HIP(hipEventCreate(&r.a));
    DC2_HIP(hipEventCreate(&r.b));
    DC2_HIP(hipEventRecord(r.a, s));
  }
  auto record = [&](bool mfma) {
    if (!acct) return;
    r.mfma = mfma;
    DC2_HIP(hipEventRecord(r.b, s));
    r.flops = 8.0 * (double)M * (double)N * (double)K * (double)batch;
    r.tag = g_tag;
    r.opA = OPA;
    r.opB = OPB;
    r.M = M;
    r.N = N;
    r.K = K;
    r.batch = batch;
    std::lock_guard<std::mutex> lk(g_stats_mu);
    g_stats->rec.push_back(r);
  };
  if (force_variant == 0 && batch == 1 && g_variant != 0 &&
      launch_skinny<OPA, OPB>(s, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc)) {
    DC2_HIP(hipGetLastError());
    record(false);
    return;
  }
  int variant = g_variant >= 1 && g_variant <= 4 ? g_variant : pick_variant(M, N, K, batch);
  TuneChoice tc{0, 0};
  int want_split = 0;   // 0: the rule below
  if (force_variant > 0) {
    variant = force_variant;
    want_split = force_split;
  } else if (g_variant != 0 && tuned_choice(OPA, OPB, M, N, K, batch, tc)) {
    variant = tc.variant;
    want_split = tc.split;
  }
  if (cdiv(N, 16 * kVariants[variant].fn) >= 65536) variant = 1;   // the grid's second dimension
  // split K over workgroups when the output has few tiles and K is long (1274 x 280 x 1274: 360
  // tiles, 92 us unsplit, 76 in three)
  const int64_t tn = 16 * kVariants[variant].fn;
  const int64_t tiles = (int64_t)cdiv(M, BM) * cdiv(N, tn) * batch;
  int sk = 1;
  int64_t kchunk = K;
  if (want_split == 0 && tiles < 512 && K >= 256) {
    want_split = (int)std::min<int64_t>(K / 128, (1024 + tiles - 1) / tiles);
    want_split = std::max(2, std::min(want_split, 64));
  }
  if (want_split > 1) {
    kchunk = ((K + want_split - 1) / want_split + BK - 1) / BK * BK;
    sk = (int)((K + kchunk - 1) / kchunk);
  }
  if (batch * sk >= 65536 || g_no_ws) {   // one grid dimension holds batch x split
    sk = 1;
    kchunk = K;
  }
  cplx* Cw = C;
  int64_t ldw = ldc, sw = sC;
  cplx a1 = alpha, b1 = beta;
  if (sk > 1) {
    Cw = splitk_workspace(s, (size_t)sk * M * N * batch);
    ldw = M;
    sw = M * N;
    a1 = mk(1.0, 0.0);
    b1 = mk(0.0, 0.0);
  }
  DC2_CHECK(cdiv(N, tn) < 65536, 1, "zgemm: matrix too large for the grid");
  const dim3 grid(cdiv(M, BM), cdiv(N, tn), (unsigned)(batch * sk));
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, M, N, K, a1, A, lda, sA, B, ldb, sB, b1, Cw, ldw, sw, sk, kchunk,
                       (int)TRI_NONE);
  };
  if (lda < kLd32 && ldb < kLd32) {
    switch (variant) {
      case 1: go(k_zgemm<OPA, OPB, 4, 8>); break;
      case 2: go(k_zgemm<OPA, OPB, 2, 16>); break;
      case 3: go(k_zgemm<OPA, OPB, 1, 16>); break;
      default: go(k_zgemm<OPA, OPB, 1, 8>); break;
    }
  } else {
    switch (variant) {
      case 1: go(k_zgemm<OPA, OPB, 4, 8, false, uint64_t>); break;
      case 2: go(k_zgemm<OPA, OPB, 2, 16, false, uint64_t>); break;
      case 3: go(k_zgemm<OPA, OPB, 1, 16, false, uint64_t>); break;
      default: go(k_zgemm<OPA, OPB, 1, 8, false, uint64_t>); break;
    }
  }
  if (sk > 1)
    hipLaunchKernelGGL(k_splitk_reduce, dim3(cdiv(M * N, 256), (unsigned)batch), dim3(256), 0, s, M, N, sk, Cw, alpha,
                       beta, C, ldc, sC);
  DC2_HIP(hipGetLastError());
  record(true);
}

template <char OPA>
void dispatchB(char opB, hipStream_t s, int64_t M, int64_t N, int64_t K, cplx alpha, const cplx* A, int64_t lda,
               int64_t sA, const cplx* B, int64_t ldb, int64_t sB, cplx beta, cplx* C, int64_t ldc, int64_t sC,
               int64_t batch, int fv = 0, int fs = 1) {
  switch (opB) {
    case 'N': launch<OPA, 'N'>(s, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, batch, fv, fs); break;
    case 'R': launch<OPA, 'R'>(s, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, batch, fv, fs); break;
    case 'T': launch<OPA, 'T'>(s, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, batch, fv, fs); break;
    case 'C': launch<OPA, 'C'>(s, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, batch, fv, fs); break;
    default: throw Error(1, "zgemm: bad opB");
  }
}

void dispatch(hipStream_t s, char opA, char opB, int64_t M, int64_t N, int64_t K, cplx alpha, const cplx* A,
              int64_t lda, int64_t sA, const cplx* B, int64_t ldb, int64_t sB, cplx beta, cplx* C, int64_t ldc,
              int64_t sC, int64_t batch, int fv = 0, int fs = 1) {
  switch (opA) {
    case 'N': dispatchB<'N'>(opB, s, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, batch, fv, fs); break;
    case 'T': dispatchB<'T'>(opB, s, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, batch, fv, fs); break;
    case 'C': dispatchB<'C'>(opB, s, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, batch, fv, fs); break;
    default: throw Error(1, "zgemm: bad opA");
  }
}
}  // namespace

void set_gemm_stats(GemmStats* st) {
  std::lock_guard<std::mutex> lk(g_stats_mu);
  g_stats = st;
}
void set_gemm_tag(int tag) { g_tag = tag; }
void set_gemm_no_workspace(bool on) { g_no_ws = on; }

void release_stream_workspace(hipStream_t s) {
  std::lock_guard<std::mutex> lk(g_ws_mu);
  g_ws->erase(s);
}

void zgemm(hipStream_t s, char opA, char opB, int64_t M, int64_t N, int64_t K, cplx alpha, const cplx* A,
           int64_t lda, int64_t sA, const cplx* B, int64_t ldb, int64_t sB, cplx beta, cplx* C, int64_t ldc,
           int64_t sC, int64_t batch) {
  if (M <= 0 || N <= 0 || batch <= 0) return;
  DC2_CHECK(batch < 65536, 1, "zgemm: batch too large for one grid dimension");
  DC2_CHECK(cdiv(M, BM) < (1u << 31) && cdiv(N, 64) < 65536, 1, "zgemm: matrix too large for the grid");
  dispatch(s, opA, opB, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, batch);
}

// C (m x m, ldc) = A A^H for A (m x k, lda): the tiles on and above the diagonal on the MFMA
// kernel, then the lower triangle as the conjugate of the upper one.  Few tiles over a long
// k (the determinant-space Gram matrices: 350 upper tiles of 64 x 16 over k = 1728) are split
// over k towards 2048 workgroups, at most 12 chunks of at least 128, summed in a fixed order by
// k_herk_reduce (m = 792, k = 1728: 140 us unsplit, 103 / 115 / 102 / 103 / 100 / 108 us in 2 / 3
// / 4 / 6 / 8 / 12 chunks; m = 210, k = 1000: 51, 29 / 22 / 18 / 20 / 16 / 19).  split: 0 this
// rule, >= 1 that many k chunks (1: unsplit).
void zherk_upper(hipStream_t s, int64_t m, int64_t k, const cplx* A, int64_t lda, cplx* C, int64_t ldc, int split) {
  zgemm_herm(s, m, k, A, lda, A, lda, C, ldc, split);
}

// C (m x m, ldc) = A B^H for A, B (m x k) whose product is Hermitian (B = D A with D real
// diagonal over k, or B = A): the same upper-tile product and mirror as zherk_upper
void zgemm_herm(hipStream_t s, int64_t m, int64_t k, const cplx* A, int64_t lda, const cplx* B, int64_t ldb, cplx* C,
                int64_t ldc, int split) {
  if (m <= 0) return;
  DC2_CHECK(cdiv(m, BM) < 65536, 1, "zgemm_herm: matrix too large for the grid");
  DC2_CHECK(split >= 0 && split <= 64, 1, "zgemm_herm: split 0..64");
  const cplx one = mk(1.0, 0.0), zero = mk(0.0, 0.0);
  // tiles of 64 x 16: finer along the diagonal and enough workgroups without splitting k far
  const int64_t T = cdiv(m, BM), Tn = cdiv(m, 16), tiles = T * (Tn + 4) / 2;
  DC2_CHECK(Tn < 65536, 1, "zgemm_herm: matrix too large for the grid");
  int64_t want = split;
  if (want == 0 && tiles < 1024 && k >= 256) want = std::min<int64_t>(std::min<int64_t>(k / 128, cdiv(2048, tiles)), 12);
  int64_t kchunk = k;
  int sk = 1;
  if (want > 1 && k > 0) {
    kchunk = (cdiv(k, want) + BK - 1) / BK * BK;
    sk = (int)cdiv(k, kchunk);
  }
  cplx* W = sk > 1 ? splitk_workspace(s, (size_t)sk * m * m) : C;
  const dim3 grid(T, Tn, (unsigned)sk);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, m, m, k, one, A, lda, (int64_t)0, B, ldb, (int64_t)0, zero, W,
                       sk > 1 ? m : ldc, m * m, sk, kchunk, (int)TRI_NONE);
  };
  if (lda < kLd32 && ldb < kLd32) go(k_zgemm<'N', 'C', 1, 16, true>);
  else go(k_zgemm<'N', 'C', 1, 16, true, uint64_t>);
  if (sk > 1) hipLaunchKernelGGL(k_herk_reduce, dim3(cdiv(m * m, 256)), dim3(256), 0, s, m, sk, W, C, ldc);
  else hipLaunchKernelGGL(k_lower_from_upper, dim3(cdiv(m * m, 256)), dim3(256), 0, s, m, C, ldc);
  DC2_HIP(hipGetLastError());
}

// C <- C - A^H A on and above the diagonal (m x m, A k x m with k short), batched by strides:
// the trailing update of a Cholesky factorisation
void zherk_trailing(hipStream_t s, int64_t m, int64_t k, const cplx* A, int64_t lda, int64_t sA, cplx* C, int64_t ldc,
                    int64_t sC, int64_t batch) {
  if (m <= 0) return;
  const int64_t T = cdiv(m, BM), Tn = cdiv(m, 32);
  DC2_CHECK(Tn < 65536 && batch < 65536 && lda < kLd32, 1, "zherk_trailing: matrix too large");
  dim3 grid(T, Tn, (unsigned)batch);
  hipLaunchKernelGGL((k_zgemm<'C', 'N', 2, 16, true>), grid, dim3(256), 0, s, m, m, k, mk(-1.0, 0.0), A, lda, sA, A,
                     lda, sA, mk(1.0, 0.0), C, ldc, sC, 1, k, (int)TRI_NONE);
  DC2_HIP(hipGetLastError());
}

// C = L B L^H (n x n, Hermitian B, L lower triangular with zeros above the diagonal): T = L B,
// then the upper tiles of T L^H and their mirror; the K loops end at the triangle's edge, so
// the two products take 1/2 and 1/3 of the full ones
void zgemm_congruence(hipStream_t s, int64_t n, const cplx* L, int64_t ldl, const cplx* B, int64_t ldb, cplx* T,
                      cplx* C, int64_t ldc) {
  if (n <= 0) return;
  const int64_t t = cdiv(n, BM), tn = cdiv(n, 16);
  DC2_CHECK(tn < 65536 && ldl < kLd32 && ldb < kLd32, 1, "zgemm_congruence: matrix too large");
  const cplx one = mk(1.0, 0.0), zero = mk(0.0, 0.0);
  dim3 grid(t, tn, 1);
  hipLaunchKernelGGL((k_zgemm<'N', 'N', 1, 16>), grid, dim3(256), 0, s, n, n, n, one, L, ldl, (int64_t)0, B, ldb,
                     (int64_t)0, zero, T, n, (int64_t)0, 1, n, (int)TRI_A);
  hipLaunchKernelGGL((k_zgemm<'N', 'C', 1, 16, true>), grid, dim3(256), 0, s, n, n, n, one, T, n, (int64_t)0, L, ldl,
                     (int64_t)0, zero, C, ldc, (int64_t)0, 1, n, (int)TRI_B);
  hipLaunchKernelGGL(k_lower_from_upper, dim3(cdiv(n * n, 256)), dim3(256), 0, s, n, C, ldc);
  DC2_HIP(hipGetLastError());
}

void gemm_set_choice(char opA, char opB, int64_t M, int64_t N, int64_t K, int64_t batch, int variant, int split) {
  DC2_CHECK(variant >= 1 && variant <= 4 && split >= 1 && split <= 64, 1, "gemm choice: variant 1..4, split 1..64");
  std::lock_guard<std::mutex> lk(g_tune_mu);
  (*g_tune)[TuneKey{opA, opB, M, N, K, batch}] = TuneChoice{variant, split};
  g_tune_any.store(true);
}

void gemm_clear_choices() {
  std::lock_guard<std::mutex> lk(g_tune_mu);
  g_tune->clear();
  g_tune_any.store(false);
}

int64_t gemm_choice_count() {
  std::lock_guard<std::mutex> lk(g_tune_mu);
  return (int64_t)g_tune->size();
}

namespace {
// p[i] = seeded values in (-0.5, 0.5) + i (-0.5, 0.5) from a 64-bit integer hash of (seed, i)
// (splitmix64's finaliser), a grid-stride loop
__global__ __launch_bounds__(256) void k_fill_hash(cplx* __restrict__ p, int64_t n, uint64_t seed) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    uint64_t z = seed + 0x9E3779B97F4A7C15ull * (uint64_t)(i + 1);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    const double re = (double)(z >> 40) * (1.0 / 16777216.0) - 0.5;
    const double im = (double)((z >> 16) & 0xFFFFFF) * (1.0 / 16777216.0) - 0.5;
    p[i] = mk(re, im);
  }
}

void fill_hash(hipStream_t s, cplx* p, int64_t n, uint64_t seed) {
  if (n <= 0) return;
  const int64_t blocks = std::min<int64_t>(cdiv(n, 256), 65535);
  hipLaunchKernelGGL(k_fill_hash, dim3((unsigned)blocks), dim3(256), 0, s, p, n, seed);
  DC2_HIP(hipGetLastError());
}
}  // namespace

void gemm_tune(hipStream_t s, char opA, char opB, int64_t M, int64_t N, int64_t K, int64_t batch, int reps,
               double* out) {
  DC2_CHECK(M > 0 && N > 0 && K > 0 && batch > 0 && batch < 65536 && reps >= 1, 1, "gemm_tune: invalid shape");
  DC2_CHECK(std::string("NTC").find(opA) != std::string::npos && std::string("NRTC").find(opB) != std::string::npos, 1,
            "gemm_tune: bad op");
  // scratch operands with seeded nonzero values (an all-zero product draws less power than
  // the real one, so its clocks and timings could differ)
  const int64_t lda = opA == 'N' ? M : K, ldb = (opB == 'N' || opB == 'R') ? K : N;
  const int64_t sA = M * K, sB = K * N, sC = M * N;
  DevBuf<cplx> A((size_t)(sA * batch)), B((size_t)(sB * batch)), C((size_t)(sC * batch));
  fill_hash(s, A.get(), sA * batch, 0x5eed0001ull);
  fill_hash(s, B.get(), sB * batch, 0x5eed0002ull);
  DC2_HIP(hipMemsetAsync(C.get(), 0, sC * batch * sizeof(cplx), s));
  hipEvent_t e0, e1;
  DC2_HIP(hipEventCreate(&e0));
  DC2_HIP(hipEventCreate(&e1));
  const cplx one = mk(1.0, 0.0), zero = mk(0.0, 0.0);
  auto time = [&](int fv, int fs) {   // fv = 0: the built-in choice (the table is bypassed below)
    dispatch(s, opA, opB, M, N, K, one, A.get(), lda, sA, B.get(), ldb, sB, zero, C.get(), M, sC, batch, fv, fs);
    DC2_HIP(hipEventRecord(e0, s));
    for (int r = 0; r < reps; ++r)
      dispatch(s, opA, opB, M, N, K, one, A.get(), lda, sA, B.get(), ldb, sB, zero, C.get(), M, sC, batch, fv, fs);
    DC2_HIP(hipEventRecord(e1, s));
    DC2_HIP(hipEventSynchronize(e1));
    float ms = 0.0f;
    DC2_HIP(hipEventElapsedTime(&ms, e0, e1));
    return 1e-3 * ms / reps;
  };
  // the built-in choice: variant g_variant and the split-K rule, without a table entry
  bool had = false;
  TuneChoice prev{0, 0};
  {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    auto it = g_tune->find(TuneKey{opA, opB, M, N, K, batch});
    if (it != g_tune->end()) { had = true; prev = it->second; g_tune->erase(it); }
    g_tune_any.store(!g_tune->empty());
  }
  const double t_builtin = time(0, 1);
  if (had) gemm_set_choice(opA, opB, M, N, K, batch, prev.variant, prev.split);
  double best = INFINITY;
  int bv = 1, bs = 1;
  for (int v = 1; v <= 4; ++v) {
    const int64_t tiles = (int64_t)cdiv(M, BM) * cdiv(N, 16 * kVariants[v].fn) * batch;
    if (cdiv(N, 16 * kVariants[v].fn) >= 65536) continue;
    for (int sp : {1, 2, 4, 8, 16, 32}) {
      if (sp > 1 && (K < 2 * BK * sp || tiles * sp > 4096 || batch * sp >= 65536)) continue;
      const double t = time(v, sp);
      if (t < best) { best = t; bv = v; bs = sp; }
    }
  }
  DC2_HIP(hipEventDestroy(e0));
  DC2_HIP(hipEventDestroy(e1));
  DC2_HIP(hipStreamSynchronize(s));   // the scratch operands are freed next
  if (best < t_builtin) {
    gemm_set_choice(opA, opB, M, N, K, batch, bv, bs);
  } else {   // the built-in choice stays (it may split K by a factor outside the candidates)
    std::lock_guard<std::mutex> lk(g_tune_mu);
    g_tune->erase(TuneKey{opA, opB, M, N, K, batch});
    g_tune_any.store(!g_tune->empty());
    bv = bs = 0;
    best = t_builtin;
  }
  out[0] = bv;
  out[1] = bs;
  out[2] = best;
  out[3] = t_builtin;
}

}  // namespace dc2
