// FP64 dense linear algebra for B formation on the device: an MFMA GEMM, a
// blocked Cholesky factorisation of the Coulomb metric and the forward
// substitution B = L^-1 (P|mn).
//
// These replace NOPT's metric route, S05_calc + dsyevd (src/matr.cpp:205-250,
// 372-401) and the per-build V^-1/2 products (src/RI.cpp:128-138, 152-156):
// the metric is factored once per geometry and folded into B.
#include "linalg.hpp"

namespace nopt {
namespace {

struct GemmArgs {
  const double *A, *B;
  double* C;
  long lda, ldb, ldc;
  int M, N, K;
  double alpha, beta;
  bool lower;
  int mt, nt;
};

// C = alpha A op(B) + beta C in 64 x 64 tiles: four waves of
// 32 x 32, slabs of 16 terms through double-buffered LDS (the slab requested a
// slab earlier is stored and the next one requested before the products, one
// barrier per slab; four blocks per CU). op(B) = B (rows k, TB false) or the
// transpose of B (rows n, TB true). Loads are single values, sixteen lanes or
// more per line, so any leading dimension will do. LDS rows of 18 (k fastest)
// and 80 doubles (n fastest) keep the operand reads on distinct banks.
// lower: only tiles that hold elements on or below the diagonal are formed.
// The tiles of one XCD are consecutive blocks of supertiles of 8 tile columns,
// column fastest, so that the blocks in flight on an XCD share their operands
// in its L2.
template <bool TB>
__global__ __launch_bounds__(256, 4) void k_gemm_f64(GemmArgs p) {
  __shared__ __attribute__((aligned(16))) double As[2][64][18];
  __shared__ __attribute__((aligned(16))) double Bs[2][TB ? 64 * 18 : 16 * 80];
  const int t = threadIdx.x, lane = t & 63, lr = lane & 15, g = lane >> 4, w = t >> 6;
  const int wr = 32 * (w >> 1), wc = 32 * (w & 1);
  const int total = p.mt * p.nt, per_xcd = total / 8, xcd = blockIdx.x % 8;
  const int idx = xcd * per_xcd + min(xcd, total % 8) + blockIdx.x / 8;
  const int sc = idx / (8 * p.mt), wid = min(8, p.nt - 8 * sc), in = idx - 8 * sc * p.mt;
  const int m0 = in / wid * 64, n0 = (8 * sc + in % wid) * 64;
  if (p.lower && n0 > m0 + 63) return;
  // loader: A value (row t / 16 + 16 u, term t % 16); B the same with TB, else (term t / 64 + 4 u, column t % 64)
  const int ar = t >> 4, ak = t & 15, bk = t >> 6, bn = t & 63;
  const double *pa[4], *pb[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    pa[u] = p.A + (long)min(m0 + ar + 16 * u, p.M - 1) * p.lda;
    pb[u] = TB ? p.B + (long)min(n0 + ar + 16 * u, p.N - 1) * p.ldb : p.B + min(n0 + bn, p.N - 1);
  }
  double xa[4], xb[4];
  auto gload = [&](int k) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int ka = k + ak, kb = TB ? ka : k + bk + 4 * u;
      const double va = pa[u][min(ka, p.K - 1)];
      const double vb = TB ? pb[u][min(kb, p.K - 1)] : pb[u][(long)min(kb, p.K - 1) * p.ldb];
      xa[u] = ka < p.K ? va : 0.0;
      xb[u] = kb < p.K ? vb : 0.0;
    }
  };
  auto lstore = [&](int buf) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      As[buf][ar + 16 * u][ak] = xa[u];
      Bs[buf][TB ? (ar + 16 * u) * 18 + ak : (bk + 4 * u) * 80 + bn] = xb[u];
    }
  };
  d4_t acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = d4_t{0, 0, 0, 0};
  gload(0);
  lstore(0);
  gload(16);
  __syncthreads();
  int cur = 0;
  for (int k = 0; k < p.K; k += 16, cur ^= 1) {
    lstore(cur ^ 1);
    gload(k + 32);
    double a[4][2], b[4][2];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        a[ks][i] = As[cur][wr + i * 16 + lr][4 * ks + g];
        b[ks][i] = Bs[cur][TB ? (wc + i * 16 + lr) * 18 + 4 * ks + g : (4 * ks + g) * 80 + wc + i * 16 + lr];
      }
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = mfma_f64(a[ks][i], b[ks][j], acc[i][j]);
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = m0 + wr + i * 16 + acc_row<double>(lane, v), col = n0 + wc + j * 16 + lr;
        if (row < p.M && col < p.N) {
          double r = p.alpha * acc[i][j][v];
          double* c = p.C + (long)row * p.ldc + col;
          if (p.beta != 0.0) r += p.beta * *c;
          *c = r;
        }
      }
}

hipError_t launch_gemm(bool transB, int M, int N, int K, double alpha, const double* A, long lda, const double* B,
                       long ldb, double beta, double* C, long ldc, bool lower, hipStream_t s) {
  if (M <= 0 || N <= 0) return hipSuccess;
  if (K <= 0) return hipErrorInvalidValue;
  const GemmArgs p{A, B, C, lda, ldb, ldc, M, N, K, alpha, beta, lower, (M + 63) / 64, (N + 63) / 64};
  if ((long)p.mt * p.nt > 0x7fffffffL) return hipErrorInvalidValue;
  if (transB)
    k_gemm_f64<true><<<(unsigned)(p.mt * p.nt), 256, 0, s>>>(p);
  else
    k_gemm_f64<false><<<(unsigned)(p.mt * p.nt), 256, 0, s>>>(p);
  return hipGetLastError();
}

// ---------------------------------------------------------------- Cholesky
constexpr int NB = 64;

// Factors the kb x kb diagonal block at (k0, k0) of A in place (lower, its
// strict upper part zeroed) and writes the inverse of the factor, 64 x 64 with
// the rows and columns beyond kb those of a unit matrix, to Xd. One block of
// four waves; the 64 x 64 block lives in LDS as 4 x 4 blocks of 16 (rows and
// columns beyond kb those of a unit matrix). A
// panel of 16 columns is factored by one wave with a row per lane and the
// columns in registers (pivot and row values by lane reads), the blocks right
// of it are updated on the matrix cores. The inverse starts from those of the
// diagonal 16 x 16 blocks (a column per lane, a wave per block) and adds the
// subdiagonals one after the other, X_ij = -X_ii sum_l L_il X_lj, the sum going
// back into the matrix unit from its accumulators.
// A non-positive pivot sets *info = k0 + j + 1 (first one wins) and is replaced
// by 1 so that the kernels stay finite.
// The chain of 64 dependent columns bounds it: 26 us (148 us with a thread per
// element and three barriers per column).
__global__ __launch_bounds__(256) void k_potrf_inv(double* A, double* Xd, long lda, int k0, int kb, int* info) {
  __shared__ double L[NB][NB + 1], V[NB][NB + 1];
  const int t = threadIdx.x, lane = t & 63, lr = lane & 15, g = lane >> 4, w = t >> 6;
  for (int e = t; e < NB * NB; e += 256) {
    const int i = e / NB, j = e % NB;
    L[i][j] = i < kb && j <= i ? A[(long)(k0 + i) * lda + k0 + j] : i == j ? 1.0 : 0.0;
    V[i][j] = 0.0;
  }
  __syncthreads();
  for (int p = 0; p < 4; ++p) {
    if (w == 0) {
      double a[16];
#pragma unroll
      for (int c = 0; c < 16; ++c) a[c] = L[lane][16 * p + c];
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        double d = lane_read(a[j], 16 * p + j);
        if (!(d > 0.0)) {
          if (lane == 0) atomicCAS(info, 0, k0 + 16 * p + j + 1);
          d = 1.0;
        }
        const double s = sqrt(d);
        a[j] = lane == 16 * p + j ? s : a[j] / s;
#pragma unroll
        for (int c = j + 1; c < 16; ++c) a[c] -= a[j] * lane_read(a[j], 16 * p + c);
      }
#pragma unroll
      for (int c = 0; c < 16; ++c)
        if (lane >= 16 * p + c) L[lane][16 * p + c] = a[c];
    }
    __syncthreads();
    // blocks (ti, tj), p < tj <= ti < 4: one to three waves' worth each
    int b = 0;
    for (int ti = p + 1; ti < 4; ++ti)
      for (int tj = p + 1; tj <= ti; ++tj, ++b) {
        if (b % 4 != w) continue;
        d4_t c;
#pragma unroll
        for (int v = 0; v < 4; ++v) c[v] = L[16 * ti + g + 4 * v][16 * tj + lr];
#pragma unroll
        for (int s = 0; s < 4; ++s)
          c = mfma_f64(-L[16 * ti + lr][16 * p + 4 * s + g], L[16 * tj + lr][16 * p + 4 * s + g], c);
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (16 * ti + g + 4 * v >= 16 * tj + lr) L[16 * ti + g + 4 * v][16 * tj + lr] = c[v];
      }
    __syncthreads();
  }
  // inverses of the diagonal blocks: wave w, block w, column lr (lanes 0..15)
  if (lane < 16) {
    double x[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      double v = r == lr ? 1.0 : 0.0;
#pragma unroll
      for (int l = 0; l < 16; ++l)
        if (l < r) v -= L[16 * w + r][16 * w + l] * x[l];
      x[r] = v / L[16 * w + r][16 * w + r];
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) V[16 * w + r][16 * w + lr] = x[r];
  }
  __syncthreads();
  for (int d = 1; d < 4; ++d) {
    if (w < 4 - d) {
      const int i = w + d, j = w;
      d4_t c = d4_t{0, 0, 0, 0}, x = d4_t{0, 0, 0, 0};
      for (int l = j; l < i; ++l)
#pragma unroll
        for (int s = 0; s < 4; ++s)
          c = mfma_f64(L[16 * i + lr][16 * l + 4 * s + g], V[16 * l + 4 * s + g][16 * j + lr], c);
#pragma unroll
      for (int s = 0; s < 4; ++s) x = mfma_f64(-V[16 * i + lr][16 * i + 4 * s + g], c[s], x);
#pragma unroll
      for (int v = 0; v < 4; ++v) V[16 * i + g + 4 * v][16 * j + lr] = x[v];
    }
    __syncthreads();
  }
  for (int e = t; e < NB * NB; e += 256) {
    const int i = e / NB, j = e % NB;
    if (i < kb && j < kb) A[(long)(k0 + i) * lda + k0 + j] = j <= i ? L[i][j] : 0.0;
    Xd[e] = V[i][j];
  }
}

// ------------------------------------------------- triangular block solves
// T (64 x 128, row stride kTS in LDS, also in the accumulators t of the eight
// waves of 32 x 32) <- L_kk^-1 T for the kb x kb diagonal block Lkk (row stride
// ld) with the inverse Xkk of k_potrf_inv: x = X T, then one step of
// refinement, x += X (T - L x), which brings the residual of the product with
// the inverse down to that of a substitution (without it the fitted B of small
// alkanes and water clusters had a ten times larger error). Rows of T beyond
// kb are zero and stay so. The result is in x; T is overwritten.
constexpr int kTS = 144;
__device__ __forceinline__ void block_solve(double (*T)[kTS], const d4_t (&t)[2][2], d4_t (&x)[2][2],
                                            const double* __restrict__ Lkk, long ld,
                                            const double* __restrict__ Xkk, int kb, int wr, int wc, int lr, int g) {
  // c += sign * M[rows of the wave][:] T over the terms below the wave's last row
  auto mul = [&](const double* M, long ldm, bool inv, double sign, d4_t (&c)[2][2]) {
    for (int k = 0; k < wr + 32; k += 16) {
      double a[4][2], b[4][2];
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int row = wr + i * 16 + lr, col = k + 4 * ks + g;
          const double v = inv ? M[row * ldm + col] : M[(long)min(row, kb - 1) * ldm + min(col, kb - 1)];
          a[ks][i] = sign * (inv || (row < kb && col < kb) ? v : 0.0);
          b[ks][i] = T[col][wc + i * 16 + lr];
        }
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) c[i][j] = mfma_f64(a[ks][i], b[ks][j], c[i][j]);
    }
  };
  auto put = [&](const d4_t (&c)[2][2]) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) T[wr + i * 16 + g + 4 * v][wc + j * 16 + lr] = c[i][j][v];
    __syncthreads();
  };
  d4_t r[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      x[i][j] = d4_t{0, 0, 0, 0};
      r[i][j] = t[i][j];
    }
  mul(Xkk, NB, true, 1.0, x);
  put(x);
  mul(Lkk, ld, false, -1.0, r);
  put(r);
  mul(Xkk, NB, true, 1.0, x);
}

// Rows i >= k0 + kb of the panel at column k0: P L_kk^T = A, P overwrites A.
// 128 rows per block, as the columns of T = A^T.
__global__ __launch_bounds__(512) void k_panel(double* A, long lda, int n, int k0, int kb,
                                               const double* __restrict__ Xd) {
  __shared__ double T[NB][kTS];
  const int t = threadIdx.x, lane = t & 63, lr = lane & 15, g = lane >> 4, w = t >> 6;
  const int wr = 32 * (w >> 2), wc = 32 * (w & 3);
  const int r0 = k0 + kb + blockIdx.x * 128;
  for (int e = t; e < 128 * NB; e += 512) {
    const int row = e / NB, k = e % NB;
    T[k][row] = r0 + row < n && k < kb ? A[(long)(r0 + row) * lda + k0 + k] : 0.0;
  }
  __syncthreads();
  d4_t tt[2][2], x[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) tt[i][j][v] = T[wr + i * 16 + g + 4 * v][wc + j * 16 + lr];
  block_solve(T, tt, x, A + (long)k0 * (lda + 1), lda, Xd, kb, wr, wc, lr, g);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) T[wr + i * 16 + g + 4 * v][wc + j * 16 + lr] = x[i][j][v];
  __syncthreads();
  for (int e = t; e < 128 * NB; e += 512) {
    const int row = e / NB, k = e % NB;
    if (r0 + row < n && k < kb) A[(long)(r0 + row) * lda + k0 + k] = T[k][row];
  }
}

// B (n x ncol, ldb) <- L^-1 B for the rows r0 .. r1, 128 columns per block from
// the first to the last row block without leaving the kernel: for each block of 64 rows the products
// of L with the rows solved so far (slabs of 16 terms of both through
// double-buffered LDS, as in k_gemm_f64; the solved rows come back from the
// block's own stores), then the diagonal block. Eight waves of 32 x 32.
// The flops n^2 ncol bound it, and for few columns the chain of row blocks (a
// block's next row block needs its last): 2.7 ms for 1206 x 31375 (246 blocks),
// 26 ms for 2366 x 120295, 26 TFLOP/s; a launch per row block, each with a pass
// over all rows below, took 6.4 and 58 ms.
__global__ __launch_bounds__(512, 4) void k_trsm_f64(const double* __restrict__ L, long ldl, int n,
                                                     const double* __restrict__ Xd, double* B, long ldb,
                                                     long ncol, int r0, int r1) {
  __shared__ __attribute__((aligned(16))) double sm[NB * kTS];
  double(*As)[64][18] = reinterpret_cast<double(*)[64][18]>(sm);                   // [2]
  double(*Bs)[16][kTS] = reinterpret_cast<double(*)[16][kTS]>(sm + 2 * 64 * 18);   // [2]
  double(*T)[kTS] = reinterpret_cast<double(*)[kTS]>(sm);
  static_assert(2 * 64 * 18 + 2 * 16 * kTS <= NB * kTS, "slabs inside T");
  const int t = threadIdx.x, lane = t & 63, lr = lane & 15, g = lane >> 4, w = t >> 6;
  const int wr = 32 * (w >> 2), wc = 32 * (w & 3);
  const long c0 = (long)blockIdx.x * 128;
  // loader: L value (row t / 16 + 32 u, term t % 16), B value (term t / 128 + 4 u, column t % 128)
  const int ar = t >> 4, ak = t & 15, bk = t >> 7, bn = t & 127;
  const double* pb = B + min(c0 + bn, ncol - 1);
  for (int k0 = r0; k0 < r1; k0 += NB) {
    const int kb = min(NB, n - k0);
    d4_t acc[2][2], tt[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = d4_t{0, 0, 0, 0};
    if (k0 > 0) {
      const double* pa[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) pa[u] = L + (long)min(k0 + ar + 32 * u, n - 1) * ldl;
      double xa[2], xb[4];
      auto gload = [&](int k) {  // (the slab after the last: that one again, unused)
        const int kk = min(k, k0 - 16);
#pragma unroll
        for (int u = 0; u < 2; ++u) xa[u] = pa[u][kk + ak];
#pragma unroll
        for (int u = 0; u < 4; ++u) xb[u] = pb[(long)(kk + bk + 4 * u) * ldb];
      };
      auto lstore = [&](int buf) {
#pragma unroll
        for (int u = 0; u < 2; ++u) As[buf][ar + 32 * u][ak] = xa[u];
#pragma unroll
        for (int u = 0; u < 4; ++u) Bs[buf][bk + 4 * u][bn] = xb[u];
      };
      gload(0);
      lstore(0);
      gload(16);
      __syncthreads();
      int cur = 0;
      for (int k = 0; k < k0; k += 16, cur ^= 1) {
        lstore(cur ^ 1);
        gload(k + 32);
        double a[4][2], b[4][2];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            a[ks][i] = As[cur][wr + i * 16 + lr][4 * ks + g];
            b[ks][i] = Bs[cur][4 * ks + g][wc + i * 16 + lr];
          }
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] = mfma_f64(a[ks][i], b[ks][j], acc[i][j]);
        __syncthreads();
      }
    }
    // T = B_k - sum (rows beyond n: zero)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = wr + i * 16 + g + 4 * v;
          const long col = min(c0 + wc + j * 16 + lr, ncol - 1);
          tt[i][j][v] = row < kb ? B[(long)(k0 + row) * ldb + col] - acc[i][j][v] : 0.0;
          T[row][wc + j * 16 + lr] = tt[i][j][v];
        }
    __syncthreads();
    d4_t x[2][2];
    block_solve(T, tt, x, L + (long)k0 * (ldl + 1), ldl, Xd + (long)(k0 / NB) * NB * NB, kb, wr, wc, lr, g);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = wr + i * 16 + g + 4 * v;
          const long col = c0 + wc + j * 16 + lr;
          if (row < kb && col < ncol) B[(long)(k0 + row) * ldb + col] = x[i][j][v];
        }
    __threadfence();  // the rows are read back by other waves of the block
    __syncthreads();
  }
}

__global__ void k_zero_upper(double* A, long lda, int n) {
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (long)n * n) return;
  const long i = e / n, j = e % n;
  if (j > i) A[i * lda + j] = 0.0;
}

__global__ void k_set_int(int* p, int v) { *p = v; }

}  // namespace

hipError_t gemm_f64(bool transB, int M, int N, int K, double alpha, const double* A, long lda,
                    const double* B, long ldb, double beta, double* C, long ldc,
                    hipStream_t s) {
  return launch_gemm(transB, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, false, s);
}

long chol_inverse_count(int n) { return (long)(n + NB - 1) / NB * NB * NB; }

hipError_t cholesky_f64(double* A, long lda, int n, double* Xd, int* d_info, hipStream_t s) {
  k_set_int<<<1, 1, 0, s>>>(d_info, 0);
  for (int k0 = 0; k0 < n; k0 += NB) {
    const int kb = n - k0 < NB ? n - k0 : NB, rest = n - k0 - kb;
    double* X = Xd + (long)(k0 / NB) * NB * NB;
    k_potrf_inv<<<1, 256, 0, s>>>(A, X, lda, k0, kb, d_info);
    if (rest <= 0) break;
    k_panel<<<(unsigned)((rest + 127) / 128), 512, 0, s>>>(A, lda, n, k0, kb, X);
    const double* P = A + (long)(k0 + kb) * lda + k0;
    const hipError_t e = launch_gemm(true, rest, rest, kb, -1.0, P, lda, P, lda, 1.0, A + (long)(k0 + kb) * (lda + 1),
                                     lda, true, s);
    if (e != hipSuccess) return e;
  }
  k_zero_upper<<<(int)(((long)n * n + 255) / 256), 256, 0, s>>>(A, lda, n);
  return hipGetLastError();
}

hipError_t trsm_lower_f64(const double* L, long ldl, int n, const double* Xd, double* B, long ldb, long ncol, int r0,
                          int r1, hipStream_t s) {
  if (ncol <= 0 || r0 >= r1) return hipSuccess;
  if (ncol > 128L * 0x7fffffff || r0 < 0 || r0 % NB || r1 > n || (r1 < n && r1 % NB)) return hipErrorInvalidValue;
  k_trsm_f64<<<(unsigned)((ncol + 127) / 128), 512, 0, s>>>(L, ldl, n, Xd, B, ldb, ncol, r0, r1);
  return hipGetLastError();
}

}  // namespace nopt
