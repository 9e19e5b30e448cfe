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
__global__ __launch_bounds__(256, 4) void k_syrk_f64(const double* __restrict__ X, long ldx, int nbf, int naux,
                                                     int kpad, int ntiles, int nsplit,
                                                     double* __restrict__ Kpart) {
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

}  // namespace

int syrk_f64_splits(int nsplit, int naux, int kpad) {
  return (int)std::max(1L, std::min((long)nsplit, (long)naux * kpad / 32));
}

hipError_t launch_syrk_f64(int ntiles, int nsplit, hipStream_t s, const double* X, long ldx, int nbf, int naux,
                           int kpad, double* Kpart) {
  const int kt = (nbf + kSyrkF64Tile - 1) / kSyrkF64Tile;
  if (nsplit < 1 || nsplit > naux || ntiles != kt * (kt + 1) / 2 || kpad < 4 || kpad % 4 || kpad > ldx || ldx % 2 || (reinterpret_cast<uintptr_t>(X) & 15))
    return hipErrorInvalidValue;
  k_syrk_f64<<<(unsigned)(ntiles * nsplit), 256, 0, s>>>(X, ldx, nbf, naux, kpad, ntiles, nsplit, Kpart);
  return hipGetLastError();
}

}  // namespace nopt
