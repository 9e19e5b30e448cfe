// FP64 contractions of the build on the 16x16x4 FP64 matrix cores. One such
// product occupies its SIMD for 64 cycles (78.6 TFLOP/s over 1024 SIMDs at
// 2.4 GHz; back to back from registers 67-68 TFLOP/s are reached, a barrier
// every sixteen products costs a tenth of that), and FP64 vector instructions
// share that unit. What keeps a kernel from the rate is work on padding, waits
// at barriers, and the address unit, which looks up every 128-byte line that a
// load instruction touches.
#include "fp64.hpp"

namespace nopt {
namespace {

// ------------------------------------------------------------ half-transform
// X[r][c] = sum_n B[r][n] C[c][n] over the rows r = Q*nbf + m of all functions,
// taken as pair rows (row m of the functions 2p and 2p + 1) in one range p*nbf + m
// without padding of the rows of a pair, and with ND > 0 the partial sums of
// gamma_d[Q] = sum_mn B[Q][m][n] D_d[m][n].
//
// A block takes 64 pair rows and 16 NT columns, a wave 16 pair rows of them. Only
// C passes through LDS (all four waves read it; slabs of 16, double buffered,
// one barrier per slab of 16 NT products per wave); a wave's rows of B go
// straight from global memory to its registers, a row's 16 values of a slab in
// two loads back to back, so that the second finds its line in the L1, and are
// requested again for the next slab as soon as their products are issued. Row m
// of D serves both functions of the pair: with rows of one function, as many
// loads and registers went to D as to B. The order of the terms is free: in a step of
// eight, lane l holds the terms 2 (l / 16) and 2 (l / 16) + 1 of row l % 16 of
// either operand, the first for one product, the second for the next.
//
// At C20H42 (490 functions, 2366 auxiliary functions, 81 orbitals, one
// density) 1.75 ms, 53 TFLOP/s of useful products (62 as issued: 96 columns),
// against 2.85 ms with B and C staged through LDS by loads of 64-byte lane
// stride in 128-row tiles per function; 1.69 ms without the density. With up to
// four column tiles it runs at the rate of B's reads, and the pairs tell: the
// gradient at 298 functions and 49 orbitals 640 -> 593 us, two densities of 192
// functions 274 -> 264, the host call at 250 functions and 41 orbitals 474 -> 456.
// Four waves per SIMD where 128 registers (nearly) hold the kernel, up to three
// column tiles and one density: that call 455 -> 440 us with four against three.
// Extra columns by vector instructions and wave tiles of 16, 48 or 64 rows were slower.
//
// The column groups of a row tile are consecutive blocks of one XCD, so that
// the second finds B in its L2. gpart[d*gstride + 2*(tile + p) + i] is the part
// of gamma_d[2p + i] in row tile `tile` (consecutive (tile, pair)s that share
// rows have consecutive sums tile + p).
constexpr int kHalfRows = kHalfF64Rows;  // pair rows
template <int NT, int ND, int OCC>
__global__ __launch_bounds__(256, OCC) void k_half_f64(const double* __restrict__ B, long ld, int naux, int nbf,
                                                       const double* __restrict__ Cp, const double* __restrict__ Dp,
                                                       long dstride, double* __restrict__ X, int ldx,
                                                       double* __restrict__ gpart, long gstride, int ntile,
                                                       int groups) {
  constexpr int MI = 2, NC = 16 * NT, CPT = (NC * 8 + 255) / 256;
  __shared__ __attribute__((aligned(16))) double sm[2][NC][18];
  const int t = threadIdx.x, lane = t & 63, lr = lane & 15, g = lane >> 4, w = t >> 6;
  const int local = blockIdx.x / 8, cg = local % groups, tile = (local / groups) * 8 + (int)(blockIdx.x % 8);
  if (tile >= ntile) return;
  const long rb = (long)tile * kHalfRows, prows = (long)((naux + 1) / 2) * nbf;  // pair rows: the block's first, all
  const long p0 = rb / nbf;
  const int m0 = (int)(rb % nbf);
  // row of function i of the pair of pair row rb + x, counted from (2 p0, m0);
  // of an odd last function's missing partner that function's (not written)
  auto row_of = [&](int x, int i) {
    const int p = (m0 + x) / nbf, m = (m0 + x) % nbf;
    return (2 * p + (2 * (p0 + p) + i < naux ? i : 0)) * nbf + m - m0;
  };
  const char* Bb = reinterpret_cast<const char*>(B + (2 * p0 * nbf + m0) * ld);
  const char* Db = reinterpret_cast<const char*>(Dp);
  const char* Cb = reinterpret_cast<const char*>(Cp);
  // byte offsets of the lane's rows (beyond the last pair row: that one again, not written)
  const int xr = (int)min((long)(w * 16 + lr), prows - 1 - rb);
  unsigned ao[MI];
#pragma unroll
  for (int i = 0; i < MI; ++i) ao[i] = 8u * ((unsigned)row_of(xr, i) * (unsigned)ld + 2u * g);
  const unsigned dof = 8u * ((unsigned)((m0 + xr) % nbf) * (unsigned)ld + 2u * g);
  // C loader: 16-byte chunk e % 8 of column e / 8 (a column beyond ldx repeats the last one, not written)
  unsigned co[CPT];
#pragma unroll
  for (int u = 0; u < CPT; ++u) {
    const int e = min(t + 256 * u, NC * 8 - 1);
    co[u] = 8u * (unsigned)(min(cg * NC + (e >> 3), ldx - 1) * (int)ld + 2 * (e & 7));
  }
  d2_t a[MI][2], d[ND ? ND : 1][2], cr[CPT];
  auto aload = [&](int i, long k) {
#pragma unroll
    for (int h = 0; h < 2; ++h) a[i][h] = *reinterpret_cast<const d2_t*>(Bb + 8 * k + ao[i] + 64 * h);
    if (i == MI - 1) {  // both rows' terms with the old ones are done
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int q = 0; q < ND; ++q)
          d[q][h] = *reinterpret_cast<const d2_t*>(Db + 8 * (q * dstride + k) + dof + 64 * h);
    }
  };
  auto cload = [&](long k) {
#pragma unroll
    for (int u = 0; u < CPT; ++u) cr[u] = *reinterpret_cast<const d2_t*>(Cb + 8 * k + co[u]);
  };
  auto cstore = [&](int buf) {
#pragma unroll
    for (int u = 0; u < CPT; ++u) {
      const int e = t + 256 * u;
      if ((u + 1) * 256 <= NC * 8 || e < NC * 8) *reinterpret_cast<d2_t*>(&sm[buf][e >> 3][2 * (e & 7)]) = cr[u];
    }
  };
  d4_t acc[MI][NT];
  double rd[MI][ND ? ND : 1];
#pragma unroll
  for (int i = 0; i < MI; ++i) {
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = d4_t{0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < ND; ++q) rd[i][q] = 0.0;
  }
#pragma unroll
  for (int i = 0; i < MI; ++i) aload(i, 0);
  cload(0);
  cstore(0);
  __syncthreads();
  int cur = 0;
  for (int k0 = 0; k0 < nbf; k0 += 16, cur ^= 1) {
    const int kn = k0 + 16 < nbf ? k0 + 16 : k0;  // the last slab again, unused, after the last
    cload(kn);
#pragma unroll
    for (int i = 0; i < MI; ++i) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        d2_t cc[NT];
#pragma unroll
        for (int j = 0; j < NT; ++j) cc[j] = *reinterpret_cast<const d2_t*>(&sm[cur][j * 16 + lr][8 * h + 2 * g]);
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
          for (int j = 0; j < NT; ++j) acc[i][j] = mfma_f64(a[i][h][e], cc[j][e], acc[i][j]);
#pragma unroll
        for (int q = 0; q < ND; ++q)
          rd[i][q] = fma(a[i][h][1], d[q][h][1], fma(a[i][h][0], d[q][h][0], rd[i][q]));
      }
      aload(i, kn);
      // keeps the operand reads of the next rows, and their registers, behind these products
      __builtin_amdgcn_sched_barrier(0);
    }
    cstore(cur ^ 1);
    __syncthreads();
  }
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int x = w * 16 + acc_row<double>(lane, v);
    if (rb + x >= prows) continue;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      if (i && 2 * (p0 + (m0 + x) / nbf) + i >= naux) continue;
      double* xo = X + (2 * p0 * nbf + m0 + row_of(x, i)) * ldx + cg * NC;
#pragma unroll
      for (int j = 0; j < NT; ++j)
        if (cg * NC + j * 16 + lr < ldx) xo[j * 16 + lr] = acc[i][j][v];
    }
  }
  if constexpr (ND > 0) {
    if (cg != 0) return;
    double(*red)[MI][kHalfRows] = reinterpret_cast<double(*)[MI][kHalfRows]>(&sm[0][0][0]);
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int q = 0; q < ND; ++q) {
        double x = rd[i][q];
        x += __shfl_xor(x, 16, 64);
        x += __shfl_xor(x, 32, 64);
        if (g == 0) red[q][i][w * 16 + lr] = x;
      }
    __syncthreads();
    // a wave per pair of functions: its rows inside the tile, one per lane
    static_assert(kHalfRows == 64, "a lane per pair row");
    const int xe = (int)min((long)kHalfRows, prows - rb), np = (m0 + xe - 1) / nbf;  // the tile's rows, its last pair
    for (int p = w; p <= np; p += 4) {
      const bool in = lane < xe && (m0 + lane) / nbf == p;
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int q = 0; q < ND; ++q) {
          const double x = warp_sum(in ? red[q][i][lane] : 0.0);
          if (lane == 0) gpart[q * gstride + 2 * (tile + p0 + p) + i] = x;
        }
    }
  }
}

// ---------------------------------------------------------------- Coulomb
// Jpart[d][s][m][n] = sum_{Q in split s} gamma[d][Q] B[Q][m][n] over the lower
// triangle, for ND densities at once (B is read once). A block owns the row
// pair (p, nbf-1-p): nbf+1 elements, read as aligned pairs of columns (a
// row's last pair may include its first upper element, which lies inside the
// row because ld > nbf and is not written). The Q loop is unrolled so that UNR
// loads per thread are in flight. gamma[d*gstride + Q], or with grows > 0 its
// partials as the FP64 half-transform leaves them (launch_half_f64).
template <int ND>
__device__ __forceinline__ void k_jpart_body(int p, int s, double* gs /* ND x the longest split */,
                                             const double* __restrict__ B, long ld, int nbf, int naux,
                                             const double* __restrict__ gamma, long gstride, int grows, int ns,
                                             double* __restrict__ Jpart, long jstride) {
  constexpr int UNR = ND == 1 ? 8 : 4;
  const int q0 = (int)((long)naux * s / ns), q1 = (int)((long)naux * (s + 1) / ns);
  const int len = q1 - q0;
  for (int q = q0 + threadIdx.x; q < q1; q += blockDim.x)
#pragma unroll
    for (int d = 0; d < ND; ++d) {
        const double* gd = gamma + d * gstride + q;  // (2 (q / 2) + q % 2)
      double v = 0.0;
      if (grows > 0) {  // partials of the FP64 half-transform: one per tile of grows pair rows that holds rows of q
        const long r = (long)(q / 2) * nbf;
        const int t1 = (int)((r + nbf - 1) / grows);
#pragma unroll 4
        for (int tl = (int)(r / grows); tl <= t1; ++tl) v += gd[2 * tl];
      } else {
        v = gd[0];
      }
      gs[d * len + q - q0] = v;
    }
  __syncthreads();
  auto g = [&](int d, int i) { return gs[d * len + i]; };
  const int m1 = p, m2 = nbf - 1 - p;
  const int s1 = (m1 + 2) / 2, s2 = (m2 != m1) ? (m2 + 2) / 2 : 0;
  const long qstride = (long)nbf * ld;
  for (int slot = threadIdx.x; slot < s1 + s2; slot += blockDim.x) {
    const int row = slot < s1 ? m1 : m2;
    const int col = 2 * (slot < s1 ? slot : slot - s1);
    const double* bp = B + (long)q0 * qstride + (long)row * ld + col;
    double a0[ND], a1[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) a0[d] = a1[d] = 0.0;
    int q = q0;
    for (; q + UNR <= q1; q += UNR) {
      double2 v[UNR];
#pragma unroll
      for (int u = 0; u < UNR; ++u) v[u] = *reinterpret_cast<const double2*>(bp + (long)u * qstride);
#pragma unroll
      for (int u = 0; u < UNR; ++u)
#pragma unroll
        for (int d = 0; d < ND; ++d) {
          a0[d] += g(d, q - q0 + u) * v[u].x;
          a1[d] += g(d, q - q0 + u) * v[u].y;
        }
      bp += (long)UNR * qstride;
    }
    for (; q < q1; ++q) {
      const double2 v = *reinterpret_cast<const double2*>(bp);
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        a0[d] += g(d, q - q0) * v.x;
        a1[d] += g(d, q - q0) * v.y;
      }
      bp += qstride;
    }
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      double* Js = Jpart + d * jstride + (long)s * nbf * nbf;
      Js[(long)row * nbf + col] = a0[d];
      if (col + 1 <= row) Js[(long)row * nbf + col + 1] = a1[d];
    }
  }
}
template <int ND>
__global__ __launch_bounds__(256) void k_jpart(JF64 a) {
  extern __shared__ double gs[];
  k_jpart_body<ND>(blockIdx.x, blockIdx.y, gs, a.B, a.ld, a.nbf, a.naux, a.gamma, a.gstride, a.grows, a.nsplit,
                   a.Jpart, a.jstride);
}

// ------------------------------------------------------------------ exchange
// Tiles of 64 x 64 with four waves of 32 x 32, four blocks per CU. The
// contraction runs over (Q, orbital) as one index, kpad orbitals per function
// without padding between functions, in slabs of 16 through double-buffered
// LDS: the slab requested a slab earlier is stored and the one after it
// requested before the products, one barrier per slab. Rows of 18 doubles keep
// the operand reads (lane l: row l % 16, term l / 16) on distinct banks. A wave
// whose quadrant holds no output (above the diagonal, beyond nbf) only loads;
// which wave takes which quadrant turns with the split, so that the idle ones
// do not all fall on the same SIMD. Rows beyond nbf read row nbf - 1 (their
// products are not read). Blocks are numbered so that each XCD owns a
// contiguous range of the (split, tile) pairs, tile fastest: the tiles of a
// split read the same rows of X from that XCD's L2.
//
// At C20H42 (490 functions, 2366 auxiliary functions, 96 padded orbitals)
// 1.13-1.20 ms alone against 1.45 ms with 128 x 128 tiles, whole diagonal
// tiles and 16-byte loads at a lane stride of 64 bytes; with the J pass beside
// it both are held up by what they read from memory (X about four times over:
// the tiles of a split drift apart by more than L2 holds). A wave that keeps a
// 64 x 64 tile in registers and reads its operands straight from global memory,
// without LDS or barriers, takes 0.94 instead of 0.98 ms alone at 84 orbitals,
// but 1.5 instead of 1.3 ms beside the J pass. Four blocks per CU: with two,
// or a barrier every 8 or 32 orbitals, it is 5-15 % slower.
__device__ __forceinline__ void k_syrk_f64_body(const double* __restrict__ X, long ldx, int nbf, int naux, int kpad,
                                                int ntiles, int nsplit, double* __restrict__ Kpart) {
  constexpr int T = kSyrkF64Tile;
  __shared__ __attribute__((aligned(16))) double sm[2][2][T][18];
  const int t = threadIdx.x, lane = t & 63, lr = lane & 15, g = lane >> 4;
  const int total = ntiles * nsplit, per_xcd = total / 8, xcd = blockIdx.x % 8;
  const int gidx = xcd * per_xcd + min(xcd, total % 8) + blockIdx.x / 8;
  const int tile = gidx % ntiles, sp = gidx / ntiles;
  int bi, bj;
  tri_tile(tile, bi, bj);
  const int q0 = (int)((long)naux * sp / nsplit), q1 = (int)((long)naux * (sp + 1) / nsplit), nq = q1 - q0;
  const int wq = ((t >> 6) + sp) & 3, wr = 32 * (wq >> 1), wc = 32 * (wq & 1);
  const bool live = __builtin_amdgcn_readfirstlane(bi * T + wr < nbf && bj * T + wc <= bi * T + wr);
  // loader: 16-byte chunk t % 8 of the rows t / 8 and t / 8 + 32 of both
  // operands; the chunk's orbitals ki, ki + 1 of the split's function kq
  const int lrow = t >> 3, lch = t & 7;
  const long qstride = (long)nbf * ldx;
  const double* src[4];
#pragma unroll
  for (int u = 0; u < 4; ++u)
    src[u] = X + q0 * qstride + (long)min((u < 2 ? bi : bj) * T + lrow + 32 * (u & 1), nbf - 1) * ldx;
  const int dq = 16 / kpad, di = 16 % kpad;
  int kq = 2 * lch / kpad, ki = 2 * lch % kpad;
  d2_t x[4];
  auto gload = [&]() {
    // beyond the split's last function: the first one, counted zero
    const bool ok = kq < nq;
    const long o = ok ? kq * qstride + ki : 0L;
#pragma unroll
    for (int u = 0; u < 4; ++u) x[u] = *reinterpret_cast<const d2_t*>(src[u] + o);
    if (!ok) {
#pragma unroll
      for (int u = 0; u < 4; ++u) x[u] = d2_t{0.0, 0.0};
    }
    ki += di;
    kq += dq;
    if (ki >= kpad) {
      ki -= kpad;
      ++kq;
    }
  };
  auto lstore = [&](int buf) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
      *reinterpret_cast<d2_t*>(&sm[buf][u >> 1][lrow + 32 * (u & 1)][2 * lch]) = x[u];
  };
  d4_t acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = d4_t{0, 0, 0, 0};
  const int nsl = (int)(((long)nq * kpad + 15) / 16);
  gload();
  lstore(0);
  gload();
  __syncthreads();
  for (int sl = 0; sl < nsl; ++sl) {
    const int cur = sl & 1;
    lstore(cur ^ 1);
    gload();
    if (live) {
      double a[4][2], b[4][2];
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          a[ks][i] = sm[cur][0][wr + i * 16 + lr][4 * ks + g];
          b[ks][i] = sm[cur][1][wc + i * 16 + lr][4 * ks + g];
        }
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) acc[i][j] = mfma_f64(a[ks][i], b[ks][j], acc[i][j]);
    }
    __syncthreads();
  }
  if (!live) return;
  double* Kt = Kpart + ((long)sp * ntiles + tile) * T * T;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        Kt[(wr + i * 16 + acc_row<double>(lane, v)) * T + wc + j * 16 + lr] = acc[i][j][v];
}
__global__ __launch_bounds__(256, 4) void k_syrk_f64(const double* __restrict__ X, long ldx, int nbf, int naux,
                                                     int kpad, int ntiles, int nsplit,
                                                     double* __restrict__ Kpart) {
  k_syrk_f64_body(X, ldx, nbf, naux, kpad, ntiles, nsplit, Kpart);
}
// The exchange, and behind its blocks the J pass in the same launch: the two do
// not depend on each other, one is bound by the matrix unit and the other by
// memory, and a launch of its own costs a small build more than its J pass
// takes (one water molecule 27.1 -> 23.2 us).
template <int ND>
__global__ __launch_bounds__(256, 4) void k_syrk_j_f64(const double* __restrict__ X, long ldx, int nbf, int naux,
                                                       int kpad, int ntiles, int nsplit, double* __restrict__ Kpart,
                                                       JF64 a) {
  __shared__ double gs[kRideGamma];
  const int b = (int)blockIdx.x - ntiles * nsplit, np = (a.nbf + 1) / 2;
  if (b < 0)
    k_syrk_f64_body(X, ldx, nbf, naux, kpad, ntiles, nsplit, Kpart);
  else
    k_jpart_body<ND>(b % np, b / np, gs, a.B, a.ld, a.nbf, a.naux, a.gamma, a.gstride, a.grows, a.nsplit, a.Jpart,
                     a.jstride);
}

// ---------------------------------------------------- active-space integrals
// R_Q[a2][a1] = sum_mn C2[a2][n] B_Q[m][n] C1[a1][m] for one Q per block (Cp:
// the rows of C2, then those of C1, ldc values each, zero from nbf on).
//
// Bound by the read of B, of which only the lower triangle W (diagonal halved)
// is read: R = C2 W^T C1^T + C2 W C1^T. A wave takes strips of 16 rows in
// zigzag order (their lengths grow with the row), forms U = W [C2; C1]^T of the
// strip on the matrix cores, and adds both products with the strip's columns of
// C1 and C2: U leaves the accumulators in the layout of either operand (lane
// l, item v: row l / 16 + 4 v, column l % 16), so it goes back into the matrix
// unit as it is. The waves' sums are added in their order. R is written in
// groups of 32 functions, [Q / 32][a2*na + a1][Q % 32] (zero for Q >= naux), the
// form in which the exchange kernel contracts it over Q.
// For 240 functions, 1160 auxiliary functions and 10 active orbitals 106 us
// (958 us with one row at a time per wave on the vector unit, lane sums after
// every row), and 5 us for the contraction over Q (290 us in one thread per
// element).
template <int NT>
__global__ __launch_bounds__(256, NT == 1 ? 4 : 2) void k_active_half(const double* __restrict__ B, long ld, int nbf,
                                                                      int naux, const double* __restrict__ Cp,
                                                                      int ldc, int na, double* __restrict__ R) {
  __shared__ double part[4][NT * NT * 256];
  const int Q = blockIdx.x, t = threadIdx.x, lane = t & 63, lr = lane & 15, g = lane >> 4, w = t >> 6;
  double* Rq = R + (long)(Q / kActiveGroup) * na * na * kActiveGroup + Q % kActiveGroup;
  if (Q >= naux) {
    for (int e = t; e < na * na; e += 256) Rq[(long)e * kActiveGroup] = 0.0;
    return;
  }
  const double* Bq = B + (long)Q * nbf * ld + 2 * g;
  // rows of C2 (tiles 0 .. NT-1) and C1 (NT .. 2 NT-1); rows beyond na repeat the last one (not written)
  const double* cp[2 * NT];
#pragma unroll
  for (int j = 0; j < 2 * NT; ++j)
    cp[j] = Cp + (long)((j < NT ? 0 : na) + min((j % NT) * 16 + lr, na - 1)) * ldc;
  d4_t r[NT][NT];  // [a2 tile][a1 tile]
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) r[i][j] = d4_t{0, 0, 0, 0};
  const int ns = (nbf + 15) / 16;
  for (int rnd = 0; 4 * rnd < ns; ++rnd) {
    const int st = 4 * rnd + ((rnd & 1) ? 3 - w : w), m0 = 16 * st;
    if (st >= ns) continue;
    const double* br = Bq + (long)min(m0 + lr, nbf - 1) * ld;
    d4_t u[2 * NT];
#pragma unroll
    for (int j = 0; j < 2 * NT; ++j) u[j] = d4_t{0, 0, 0, 0};
    d2_t b[2], bn[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) b[h] = *reinterpret_cast<const d2_t*>(br + 8 * h);
    for (int n0 = 0; n0 <= m0; n0 += 16) {
      d2_t c[2 * NT][2];
#pragma unroll
      for (int j = 0; j < 2 * NT; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h) c[j][h] = *reinterpret_cast<const d2_t*>(cp[j] + n0 + 8 * h + 2 * g);
      const int nn = n0 < m0 ? n0 + 16 : n0;
#pragma unroll
      for (int h = 0; h < 2; ++h) bn[h] = *reinterpret_cast<const d2_t*>(br + nn + 8 * h);
      if (n0 == m0) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const int n = 8 * h + 2 * g + e;
            b[h][e] = n < lr ? b[h][e] : n == lr ? 0.5 * b[h][e] : 0.0;
          }
      }
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
          for (int j = 0; j < 2 * NT; ++j) u[j] = mfma_f64(b[h][e], c[j][h][e], u[j]);
#pragma unroll
      for (int h = 0; h < 2; ++h) b[h] = bn[h];
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      double cm[2 * NT];
#pragma unroll
      for (int j = 0; j < 2 * NT; ++j) cm[j] = cp[j][m0 + 4 * v + g];
#pragma unroll
      for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          r[i][j] = mfma_f64(u[i][v], cm[NT + j], r[i][j]);
          r[i][j] = mfma_f64(cm[i], u[NT + j][v], r[i][j]);
        }
    }
  }
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        part[w][(i * 16 + acc_row<double>(lane, v)) * (16 * NT) + j * 16 + lr] = r[i][j][v];
  __syncthreads();
  for (int e = t; e < na * na; e += 256) {
    const int i = (e / na) * (16 * NT) + e % na;
    Rq[(long)e * kActiveGroup] = ((part[0][i] + part[1][i]) + part[2][i]) + part[3][i];
  }
}

}  // namespace

int half_f64_nt(long ncol, int* groups) {
  const int t = (int)std::max(1L, (ncol + 15) / 16);
  *groups = (t + 7) / 8;
  return (t + *groups - 1) / *groups;
}

hipError_t launch_half_f64(int nt, int groups, int nd, hipStream_t s, const double* B, long ld, int naux, int nbf,
                           const double* Cp, const double* Dp, long dstride, double* X, long ldx, double* gpart) {
  const int ntile = half_f64_tiles(naux, nbf);
  if (nd < 0 || nd > kHalfF64Dens || groups < 1 || 16L * nt * groups < ldx || 16L * nt * (groups - 1) >= ldx ||
      ldx % 2 || ld % 16 || ld < nbf || (nd && (!Dp || !gpart)) || ld * std::max(ldx, 2L * kHalfF64Rows) > 1L << 28 ||
      ld * (nbf + kHalfF64Rows) >= 1L << 28)
    return hipErrorInvalidValue;
  const unsigned grid = (unsigned)((ntile + 7) / 8 * 8 * groups);
#define NOPT_HALF_F64(NT_, ND_)                                                                                  \
  if (nt == NT_ && nd == ND_)                                                                                    \
    k_half_f64<NT_, ND_, (NT_ <= 3 && ND_ < 2 ? 4 : NT_ <= 4 ? 3 : 2)><<<grid, 256, 0, s>>>(B, ld, naux, nbf, Cp, Dp, dstride, X, (int)ldx, \
                                                                 gpart, half_f64_gstride(naux, nbf), ntile, groups);
#define NOPT_HALF_F64_ND(NT_) NOPT_HALF_F64(NT_, 0) NOPT_HALF_F64(NT_, 1) NOPT_HALF_F64(NT_, 2)
  NOPT_HALF_F64_ND(1)
  NOPT_HALF_F64_ND(2)
  NOPT_HALF_F64_ND(3)
  NOPT_HALF_F64_ND(4)
  NOPT_HALF_F64_ND(5)
  NOPT_HALF_F64_ND(6)
  NOPT_HALF_F64_ND(7)
  NOPT_HALF_F64_ND(8)
#undef NOPT_HALF_F64_ND
#undef NOPT_HALF_F64
  return nt < 1 || nt > 8 ? hipErrorInvalidValue : hipGetLastError();
}

hipError_t launch_active_half(hipStream_t s, const double* B, long ld, int nbf, int naux, const double* Cp, int ldc,
                              int na, double* R) {
  if (na < 1 || na > 32 || ldc < (nbf + 15) / 16 * 16 || ldc % 2 || ld < (nbf + 15) / 16 * 16)
    return hipErrorInvalidValue;
  const unsigned grid = (unsigned)((naux + kActiveGroup - 1) / kActiveGroup * kActiveGroup);
  if (na <= 16)
    k_active_half<1><<<grid, 256, 0, s>>>(B, ld, nbf, naux, Cp, ldc, na, R);
  else
    k_active_half<2><<<grid, 256, 0, s>>>(B, ld, nbf, naux, Cp, ldc, na, R);
  return hipGetLastError();
}

int syrk_f64_splits(int nsplit, int naux, int kpad) {
  return (int)std::max(1L, std::min((long)nsplit, (long)naux * kpad / 32));
}

hipError_t launch_jpart_f64(const JF64& a, int nd, hipStream_t s) {
  const dim3 grid((a.nbf + 1) / 2, a.nsplit);
  const size_t lds = sizeof(double) * nd * ((a.naux + a.nsplit - 1) / a.nsplit);
  switch (nd) {
    case 1: k_jpart<1><<<grid, 256, lds, s>>>(a); break;
    case 2: k_jpart<2><<<grid, 256, lds, s>>>(a); break;
    case 3: k_jpart<3><<<grid, 256, lds, s>>>(a); break;
    case 4: k_jpart<4><<<grid, 256, lds, s>>>(a); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

bool jpart_rides_f64(int nd, int naux, int nsplit) {
  return nd >= 1 && nd <= 2 && (long)nd * ((naux + nsplit - 1) / nsplit) <= kRideGamma;
}

hipError_t launch_syrk_f64(int ntiles, int nsplit, hipStream_t s, const double* X, long ldx, int nbf, int naux,
                           int kpad, double* Kpart, const JF64* j, int nd) {
  const int kt = (nbf + kSyrkF64Tile - 1) / kSyrkF64Tile;
  if (nsplit < 1 || nsplit > naux || ntiles != kt * (kt + 1) / 2 || kpad < 4 || kpad % 4 || kpad > ldx || ldx % 2 || (reinterpret_cast<uintptr_t>(X) & 15))
    return hipErrorInvalidValue;
  if (j && !jpart_rides_f64(nd, j->naux, j->nsplit)) return hipErrorInvalidValue;
  const unsigned nx = (unsigned)(ntiles * nsplit), njb = j ? (unsigned)((j->nbf + 1) / 2 * j->nsplit) : 0u;
  if (!j)
    k_syrk_f64<<<nx, 256, 0, s>>>(X, ldx, nbf, naux, kpad, ntiles, nsplit, Kpart);
  else if (nd == 1)
    k_syrk_j_f64<1><<<nx + njb, 256, 0, s>>>(X, ldx, nbf, naux, kpad, ntiles, nsplit, Kpart, *j);
  else
    k_syrk_j_f64<2><<<nx + njb, 256, 0, s>>>(X, ldx, nbf, naux, kpad, ntiles, nsplit, Kpart, *j);
  return hipGetLastError();
}

}  // namespace nopt
