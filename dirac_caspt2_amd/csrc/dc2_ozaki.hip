// Split-precision complex GEMM (Ozaki scheme) on CDNA4 INT8 matrix cores.
//
// C = A * B (complex FP64, alpha = 1, beta = 0) for the integral-transform passes,
// A[m][k] = in[k + lda*m] ('T') and B[k][j] = U[k + ldb*j] or its conjugate ('N'/'R').
//
// Every row m of A (and column j of B) is scaled by a power of two 2^-e so that its
// largest real or imaginary part lies in [1/2, 1), then cut into S signed 7-bit digits:
//   a = sum_{p<S} d_p 2^{-7(p+1)} + r 2^{-7S},  d_p in [-127, 127],  |r| < 1,
// each extraction exact in FP64.  A complex product is two real GEMMs over K' = 2K:
//   Re C = [Ar | Ai] [Br ; -Bi],   Im C = [Ar | Ai] [Bi ; Br]
// (conjugated B flips the sign of Bi; digit negation is exact), real and imaginary digits of one
// k side by side.  The digit products
// of level L = p + q < S are accumulated exactly in INT32 with
// v_mfma_i32_16x16x64_i8 (|sum| <= S * K' * 127^2 < 2^31 for K' <= 8192) and
// recombined in FP64 as sum_L 2^{-7(L+2)} acc_L, smallest level first, times
// 2^{e_m + f_j}.  Dropped levels (L >= S) and the residuals bound the error by
// about (S + 1) 2^{-7S} K' max|row of A| max|column of B|.
//
// The slices are stored in the matrix unit's operand order: 1 KB for 16 rows, 64 of K' and one
// digit p, lane l's 16 bytes (row l & 15, K' 16 (l >> 4) ...) at 16 l, the S digits of one (rows,
// K' chunk) one after another (the k of a chunk in the order that k_oz_split loads well, the same
// for A and B: the sums are exact in any order).  A fragment is then one contiguous load straight into LDS, and one
// conflict-free read from there.
#include "dc2_kernels.hpp"

namespace dc2 {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int OZ_FRAG = 1024;   // bytes of a fragment: 16 rows x 64 of K' (32 complex k)
constexpr int OZ_BN = 32;

// exponent e with max(|re|, |im|) * 2^-e in [1/2, 1) (0 for a zero vector)
__device__ inline int scale_exponent(double amax) {
  if (!(amax > 0.0)) return 0;
  return ilogb(amax) + 1;
}

// the S base-128 digits of |x| 2^-e (most significant first, bits 7 (S - 1 - p)); x |x| < 2^e
template <int S>
__device__ inline uint64_t digits_of(double x, int e) {
  const double v = ldexp(fabs(x), 7 * S - e);   // exact: below 2^56, cut to an integer here
  if (7 * S <= 31) return (uint32_t)v;
  const double hi = trunc(v * 0x1p-32);
  return ((uint64_t)(uint32_t)hi << 32) | (uint32_t)fma(hi, -0x1p32, v);
}

// Workgroup = 16 rows of A, or 16 columns of B for its Re or its Im part (blocks after A's:
// Re, Im in turn); a wave takes every fourth K' chunk of 32 complex k, lane (row, g) the k = 4 u
// + g of it: 64 contiguous bytes per row in, 16 bytes per digit out, the wave's stores 1 KB in a
// row (8 consecutive k a lane, 16 bytes per line and load: 0.21 ms).  NH > 0: the row's elements
// stay in registers between the pass for the largest one and the digits (NH chunks a wave, K <=
// 128 NH), so that A is read once.  Bound by its traffic: 394 MB in, 305 MB out for 88199 x 279
// and 6 digits in 0.136 ms, 5.1 TB/s; 0.18 ms with a wave per row and byte stores.
template <int S, int NH>
__global__ __launch_bounds__(256) void k_oz_split(int64_t M, int64_t N, int64_t K, int64_t nkc, int64_t rbA,
                                                  const cplx* __restrict__ A, int64_t lda,
                                                  const cplx* __restrict__ B, int64_t ldb, int conj,
                                                  int8_t* __restrict__ A8, int8_t* __restrict__ B8,
                                                  int* __restrict__ expo) {
  __shared__ double mx[4][16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
  const bool isA = blockIdx.x < rbA;
  const int64_t c = blockIdx.x - rbA, rb = isA ? blockIdx.x : c >> 1;
  const int ri = isA ? 0 : (int)(c & 1);   // 1: the Im part, digits (conj Im B, Re B)
  const int64_t row = 16 * rb + r;
  const bool valid = row < (isA ? M : N);
  const cplx* x = isA ? A + lda * row : B + ldb * row;
  auto load = [&](int64_t kc, cplx* z) {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int64_t k = 32 * kc + 4 * u + g;
      z[u] = valid && k < K ? x[k] : mk(0.0, 0.0);
    }
  };
  constexpr int H = NH > 0 ? NH : 1;
  cplx z[H][8];
  double amax = 0.0;
  if (NH > 0) {
#pragma unroll
    for (int h = 0; h < H; ++h) load(wave + 4 * h, z[h]);
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
      for (int u = 0; u < 8; ++u) amax = fmax(amax, fmax(fabs(z[h][u].x), fabs(z[h][u].y)));
  } else {
    for (int64_t kc = wave; kc < nkc; kc += 4) {
      load(kc, z[0]);
#pragma unroll
      for (int u = 0; u < 8; ++u) amax = fmax(amax, fmax(fabs(z[0][u].x), fabs(z[0][u].y)));
    }
  }
  amax = fmax(amax, __shfl_xor(amax, 16, 64));
  amax = fmax(amax, __shfl_xor(amax, 32, 64));
  if (lane < 16) mx[wave][lane] = amax;
  __syncthreads();
  amax = fmax(fmax(mx[0][r], mx[1][r]), fmax(mx[2][r], mx[3][r]));
  const int e = scale_exponent(amax);
  if (threadIdx.x < 16 && valid && ri == 0) expo[(isA ? 0 : M) + row] = e;
  // A: (re, im); B's Re part: (Re B, -conj Im B), its Im part: (conj Im B, Re B)
  const bool neg_im = isA ? false : (ri == 0) == (conj > 0);
  int8_t* out = isA ? A8 + rb * nkc * S * OZ_FRAG : B8 + (rb * nkc * 2 + ri) * S * OZ_FRAG;
  const int64_t step = (isA ? 1 : 2) * S * OZ_FRAG;
  auto put = [&](int64_t kc, const cplx* z) {
    v4i o[S];
#pragma unroll
    for (int p = 0; p < S; ++p) o[p] = v4i{0, 0, 0, 0};
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const uint64_t dr = digits_of<S>(z[u].x, e), di = digits_of<S>(z[u].y, e);
      const int sr = z[u].x < 0.0 ? -1 : 0, si = (z[u].y < 0.0) != neg_im ? -1 : 0;
#pragma unroll
      for (int p = 0; p < S; ++p) {
        const int a = (((int)(dr >> (7 * (S - 1 - p))) & 127) ^ sr) - sr;
        const int b = (((int)(di >> (7 * (S - 1 - p))) & 127) ^ si) - si;
        const int lo = ri ? b : a, hi = ri ? a : b;
        o[p][u >> 1] |= ((lo & 255) | (hi & 255) << 8) << (16 * (u & 1));
      }
    }
#pragma unroll
    for (int p = 0; p < S; ++p) *reinterpret_cast<v4i*>(out + kc * step + p * OZ_FRAG + 16 * lane) = o[p];
  };
  if (NH > 0) {
#pragma unroll
    for (int h = 0; h < H; ++h)
      if (wave + 4 * h < nkc) put(wave + 4 * h, z[h]);
  } else {
    for (int64_t kc = wave; kc < nkc; kc += 4) {
      load(kc, z[0]);
      put(kc, z[0]);
    }
  }
}

typedef __attribute__((address_space(1))) void gvoid;
typedef __attribute__((address_space(3))) void lvoid;

// C[m + ldc*j] = sum_L 2^{-7(L+2)} (acc_L) * 2^{ea[m] + eb[j]} for the re and im GEMMs.
// Workgroup: WM x 2 waves, tile 32 WM x 32; wave (wm, wn) owns rows 32 wm .. and columns 16 wn
// .. (two 16x16 tiles along m, S levels of each, Re and Im: 16 S accumulators).  The next K'
// chunk's fragments go to the other half of LDS (72 KB a half at S = 6, WM = 4) while this
// one's 2 S (S + 1) MFMAs per wave run; WM = 2 where two halves of WM = 4 exceed 160 KB.
// Bound by LDS and the matrix units together: a chunk's 264 KB through LDS are 2100 cycles, its
// MFMAs 2700 (88199 x 279 x 279, S = 6: 0.50 ms, 2.4e15 operations/s; 0.91 ms with the fragments
// loaded from L2 into registers).  Measured and not better: four tiles along m a wave and one
// wave per SIMD (0.64 ms), one LDS half and three 64 x 32 workgroups a compute unit (0.56),
// workgroups that stay for several tiles (0.53).
template <int S, int WM>
__global__ __launch_bounds__(128 * WM) void k_oz_gemm(int64_t M, int64_t N, int64_t nkc, int64_t rbA, int64_t rbB,
                                                      const int8_t* __restrict__ A8, const int8_t* __restrict__ B8,
                                                      const int* __restrict__ expo, cplx* __restrict__ C,
                                                      int64_t ldc) {
  constexpr int NA = 2 * WM * S, NB = 4 * S, NF = NA + NB, NW = 2 * WM;
  __shared__ __align__(16) int8_t sh[2][NF * OZ_FRAG];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave % WM, wn = wave / WM;
  int64_t mt, nt;
  xcd_tile(gridDim.x, gridDim.y, blockIdx.x, blockIdx.y, mt, nt);
  // this wave's fragments of a chunk; blocks past the last are copies of it, whose results are
  // not stored
  constexpr int NU = (NF + NW - 1) / NW;
  const int8_t* src[NU];
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    const int f = wave + NW * u;
    if (f < NA) {
      const int64_t rb = 2 * WM * mt + f / S;
      src[u] = A8 + ((rb < rbA ? rb : rbA - 1) * nkc * S + f % S) * OZ_FRAG;
    } else {
      const int64_t cb = 2 * nt + (f - NA) / (2 * S);
      src[u] = B8 + ((cb < rbB ? cb : rbB - 1) * nkc * (2 * S) + (f - NA) % (2 * S)) * OZ_FRAG;
    }
  }
  auto stage = [&](int buf) {
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int f = wave + NW * u;
      if (NF % NW != 0 && f >= NF) break;
      __builtin_amdgcn_global_load_lds((gvoid*)(src[u] + 16 * lane), (lvoid*)&sh[buf][f * OZ_FRAG], 16, 0, 0);
      src[u] += (f < NA ? S : 2 * S) * OZ_FRAG;
    }
  };
  v4i accr[S][2], acci[S][2];
#pragma unroll
  for (int L = 0; L < S; ++L)
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      accr[L][t] = v4i{0, 0, 0, 0};
      acci[L][t] = v4i{0, 0, 0, 0};
    }
  stage(0);
  __builtin_amdgcn_s_waitcnt(0);   // the loads into LDS of this wave; the barrier for the others'
  __syncthreads();
  for (int64_t kc = 0; kc < nkc; ++kc) {
    const int buf = (int)(kc & 1);
    if (kc + 1 < nkc) stage(buf ^ 1);
    const int8_t* pa = &sh[buf][2 * wm * S * OZ_FRAG + 16 * lane];
    const int8_t* pb = &sh[buf][(NA + 2 * wn * S) * OZ_FRAG + 16 * lane];
    v4i a[S][2];
#pragma unroll
    for (int p = 0; p < S; ++p)
#pragma unroll
      for (int t = 0; t < 2; ++t) a[p][t] = *reinterpret_cast<const v4i*>(pa + (t * S + p) * OZ_FRAG);
#pragma unroll
    for (int q = 0; q < S; ++q) {
      const v4i br = *reinterpret_cast<const v4i*>(pb + q * OZ_FRAG);
      const v4i bi = *reinterpret_cast<const v4i*>(pb + (S + q) * OZ_FRAG);
#pragma unroll
      for (int p = 0; p < S - q; ++p)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          accr[p + q][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(br, a[p][t], accr[p + q][t], 0, 0, 0);
          acci[p + q][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(bi, a[p][t], acci[p + q][t], 0, 0, 0);
        }
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
  }
  // D[i][j] of a 16x16 tile: lane j + 16*(i/4), element i%4 (measured on gfx950); B's columns
  // are the rows i here, so that a store takes 16 consecutive m of four columns
  const int r16 = lane & 15, g = lane >> 4;
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int64_t m = 32 * (WM * mt + wm) + 16 * t + r16;
    if (m >= M) continue;
    const int em = expo[m];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t j = OZ_BN * nt + 16 * wn + 4 * g + r;
      if (j >= N) continue;
      double re = (double)accr[S - 1][t][r], im = (double)acci[S - 1][t][r];
#pragma unroll
      for (int L = S - 2; L >= 0; --L) {
        re = fma(re, 0x1p-7, (double)accr[L][t][r]);
        im = fma(im, 0x1p-7, (double)acci[L][t][r]);
      }
      const int sc = em + expo[M + j] - 14;
      C[m + ldc * j] = mk(ldexp(re, sc), ldexp(im, sc));
    }
  }
}

template <int S>
void oz_launch(hipStream_t s, char opB, int64_t M, int64_t N, int64_t K, const cplx* A, int64_t lda, const cplx* B,
               int64_t ldb, cplx* C, int64_t ldc, int8_t* work, int* expo) {
  constexpr int WM = S <= 6 ? 4 : 2;
  const int64_t nkc = (K + 31) / 32, rbA = (M + 15) / 16, rbB = (N + 15) / 16;
  int8_t* A8 = work;
  int8_t* B8 = A8 + S * rbA * nkc * OZ_FRAG;
  const int conj = opB == 'R' ? -1 : 1;
  // up to K = 384 a row's elements are held (96 registers a thread): 279 and 280, the sizes of
  // the largest transforms, take 3 chunks a wave
  auto split = nkc <= 4 ? k_oz_split<S, 1> : nkc <= 12 ? k_oz_split<S, 3> : k_oz_split<S, 0>;
  hipLaunchKernelGGL(split, dim3((unsigned)(rbA + 2 * rbB)), dim3(256), 0, s, M, N, K, nkc, rbA, A, lda, B, ldb, conj,
                     A8, B8, expo);
  hipLaunchKernelGGL((k_oz_gemm<S, WM>), dim3(cdiv(M, 32 * WM), cdiv(N, OZ_BN)), dim3(128 * WM), 0, s, M, N, nkc, rbA,
                     rbB, A8, B8, expo, C, ldc);
  DC2_HIP(hipGetLastError());
}

}  // namespace

int64_t zgemm_ozaki_work_bytes(int slices, int64_t M, int64_t N, int64_t K) {
  return (int64_t)slices * ((M + 15) / 16 + 2 * ((N + 15) / 16)) * ((K + 31) / 32) * OZ_FRAG;
}

void zgemm_ozaki(hipStream_t s, int slices, char opB, int64_t M, int64_t N, int64_t K, const cplx* A, int64_t lda,
                 const cplx* B, int64_t ldb, cplx* C, int64_t ldc, int8_t* work, int* expo) {
  if (M <= 0 || N <= 0) return;
  DC2_CHECK(K >= 1 && K <= 4096, 1, "zgemm_ozaki: K must be in 1..4096");
  DC2_CHECK(opB == 'N' || opB == 'R', 1, "zgemm_ozaki: opB must be N or R");
  DC2_CHECK(M < (1ll << 33) && cdiv(N, OZ_BN) < 65536, 1,
            "zgemm_ozaki: matrix too large for the grid");
  switch (slices) {
    case 3: oz_launch<3>(s, opB, M, N, K, A, lda, B, ldb, C, ldc, work, expo); break;
    case 4: oz_launch<4>(s, opB, M, N, K, A, lda, B, ldb, C, ldc, work, expo); break;
    case 5: oz_launch<5>(s, opB, M, N, K, A, lda, B, ldb, C, ldc, work, expo); break;
    case 6: oz_launch<6>(s, opB, M, N, K, A, lda, B, ldb, C, ldc, work, expo); break;
    case 7: oz_launch<7>(s, opB, M, N, K, A, lda, B, ldb, C, ldc, work, expo); break;
    case 8: oz_launch<8>(s, opB, M, N, K, A, lda, B, ldb, C, ldc, work, expo); break;
    default: throw Error(1, "zgemm_ozaki: slices must be in 3..8");
  }
}

}  // namespace dc2
