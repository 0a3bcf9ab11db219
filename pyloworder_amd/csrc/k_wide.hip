// FP64 MFMA Grams of wide problems (256 < real columns <= 2048): the tall-skinny SVD
// of n columns beyond what one register-resident Gram holds.  Columns are cut into
// stripes of W = 128.
//
//   k_wgram_f64 : one (row chunk, stripe pair I <= J) per workgroup:
//                 G[I, J] = Yc_I^T Yc_J over the chunk's rows, 32-row tiles of
//                 both stripes in LDS (two buffers, the next tile in registers), 64
//                 16x16 output blocks (8 per wave; the 36 upper ones when I == J).
//                 The chunk's partial Gram lands in its NBp x NBp slab at (I W, J W);
//                 only blocks with I <= J are written, the reductions read the upper
//                 triangle only.  The FP64 matrix rate bounds it.  Loading each tile
//                 between two barriers took 11.9 ms for 1M x 512 float32, this 5.2
//                 (float64 9.3 -> 5.9).
//   k_wxgram_f64: the cross product of two operands the same way, unbuffered.
// Yc is the row-centred input (center 1: minus the row mean; 2: also divided
// by the row variance; the FP64 statistics come from a prior pass), so the
// centring costs nothing extra.  Element types: TS the real storage type
// (complex data is read as its interleaved real view).
#include "common.hpp"
#include "f64_common.hpp"
#include "kernels.hpp"

namespace {

constexpr int WS = 128;       // stripe width
constexpr int WTR = 32;       // rows per tile
constexpr int WNT = 512;      // threads per workgroup (8 waves)

template <class TS, bool VAR>
__global__ __launch_bounds__(WNT) void k_wgram_f64(const TS* __restrict__ X, int64_t ldx, int64_t m, int n, int center,
                                                   const double* __restrict__ mean, const double* __restrict__ var,
                                                   int kstr, int64_t tpc, double* __restrict__ part, int NBp) {
  constexpr int LD = 2 * WS + 2;
  __shared__ double S[2][WTR * LD];
  // pair p -> (I, J), I <= J, row-major over the upper triangle of kstr stripes
  int p = blockIdx.y, I = 0;
  while (p >= kstr - I) { p -= kstr - I; I++; }
  const int J = I + p;
  const bool diag = I == J;
  const int w = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)), l = threadIdx.x & 63, kr = l >> 4, cc = l & 15;
  // the wave's blocks: row w of the 8 x 8, or 4 or 5 consecutive ones of the 36 upper
  int bi = w, bj = 0, cnt = 8;
  if (diag) {
    int b = 36 * w / 8;
    cnt = 36 * (w + 1) / 8 - b;
    bi = 0;
    while (b >= 8 - bi) b -= 8 - bi++;
    bj = bi + b;
  }
  const int right = diag ? 0 : WS;  // columns of the right operand in the tile
  d4 acc[8];
#pragma unroll
  for (int s = 0; s < 8; s++) acc[s] = d4{0, 0, 0, 0};
  const int64_t ntiles = ceil_div(m, WTR);
  const int64_t t0 = int64_t(blockIdx.x) * tpc;
  const int64_t t1 = t0 + tpc < ntiles ? t0 + tpc : ntiles;
  RowStage<TS, WTR, WS, VAR> sa, sb;
  auto fetch = [&](int64_t t) {
    const int64_t row0 = (t < t1 ? t : t1 - 1) * WTR;
    sa.fetch(X, ldx, m, n, row0, I * WS, center, mean, var);
    if (!diag) sb.fetch(X, ldx, m, n, row0, J * WS, center, mean, var);
  };
  auto put = [&](int64_t t) {
    double* d = S[(t - t0) & 1];
    sa.template put<LD>(d, 0, m, n, t * WTR, I * WS, center, false, nullptr, nullptr);
    if (!diag) sb.template put<LD>(d, WS, m, n, t * WTR, J * WS, center, false, nullptr, nullptr);
  };
  fetch(t0);
  put(t0);
  fetch(t0 + 1);
  lds_barrier();
  for (int64_t t = t0; t < t1; t++) {
    const double* base = S[(t - t0) & 1] + kr * LD + cc;
    double a[WTR / 4];
    int x = bi, y = bj, cur = -1;
#pragma unroll
    for (int s = 0; s < 8; s++) {
      if (s < cnt) {
        if (x != cur) {
#pragma unroll
          for (int kk = 0; kk < WTR / 4; kk++) a[kk] = base[4 * kk * LD + 16 * x];
          cur = x;
        }
        double b[WTR / 4];
#pragma unroll
        for (int kk = 0; kk < WTR / 4; kk++) b[kk] = base[4 * kk * LD + right + 16 * y];
#pragma unroll
        for (int kk = 0; kk < WTR / 4; kk++) acc[s] = mfma64(a[kk], b[kk], acc[s]);
        if (++y == 8) y = diag ? ++x : 0;
      }
    }
    if (t + 1 < t1) {
      put(t + 1);
      fetch(t + 2);
    }
    lds_barrier();
  }
  double* P = part + int64_t(blockIdx.x) * NBp * NBp;
#pragma unroll
  for (int s = 0; s < 8; s++) {
    if (s < cnt) {
#pragma unroll
      for (int r = 0; r < 4; r++)
        P[int64_t(I * WS + bi * 16 + 4 * r + kr) * NBp + J * WS + bj * 16 + cc] = acc[s][r];
      if (++bj == 8) bj = diag ? ++bi : 0;
    }
  }
}

// P[chunk] (PBp x QBp) += A^T B over the chunk's rows, A m x p, B m x q: one
// (row chunk, stripe I of A, stripe J of B) per workgroup
template <class TA, class TB>
__global__ __launch_bounds__(WNT) void k_wxgram_f64(const TA* __restrict__ A, int64_t lda, int p,
                                                    const TB* __restrict__ B, int64_t ldb, int q, int64_t m, int kq,
                                                    int64_t tpc, double* __restrict__ part, int PBp, int QBp) {
  __shared__ double S[WTR][2 * WS + 2];
  const int I = blockIdx.y / kq, J = blockIdx.y % kq;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, kr = l >> 4, cc = l & 15;
  d4 acc[8];
#pragma unroll
  for (int s = 0; s < 8; s++) acc[s] = d4{0, 0, 0, 0};
  const int64_t ntiles = ceil_div(m, WTR);
  const int64_t t0 = int64_t(blockIdx.x) * tpc;
  const int64_t t1 = t0 + tpc < ntiles ? t0 + tpc : ntiles;
  for (int64_t t = t0; t < t1; t++) {
    __syncthreads();
    for (int idx = threadIdx.x; idx < WTR * 2 * WS; idx += WNT) {
      const int r = idx / (2 * WS), c = idx % (2 * WS);
      const int64_t row = t * WTR + r;
      double v = 0.0;
      if (c < WS) {
        const int col = I * WS + c;
        if (row < m && col < p) v = double(A[row * lda + col]);
      } else {
        const int col = J * WS + (c - WS);
        if (row < m && col < q) v = double(B[row * ldb + col]);
      }
      S[r][c] = v;
    }
    __syncthreads();
#pragma unroll 2
    for (int kk = 0; kk < WTR / 4; kk++) {
      const double* srow = S[kk * 4 + kr];
#pragma unroll
      for (int s = 0; s < 8; s++) {
        const int b = w * 8 + s, bi = b >> 3, bj = b & 7;
        acc[s] = mfma64(srow[bi * 16 + cc], srow[WS + bj * 16 + cc], acc[s]);
      }
    }
  }
  double* P = part + int64_t(blockIdx.x) * PBp * QBp;
#pragma unroll
  for (int s = 0; s < 8; s++) {
    const int b = w * 8 + s, bi = b >> 3, bj = b & 7;
#pragma unroll
    for (int r = 0; r < 4; r++)
      P[int64_t(I * WS + bi * 16 + 4 * r + kr) * QBp + J * WS + bj * 16 + cc] = acc[s][r];
  }
}

}  // namespace

int wide_stripe() { return WS; }
int wide_tile_rows() { return WTR; }

int launch_wgram_f64(hipStream_t st, pc_dtype dt, const void* X, int64_t ldx, int64_t m, int n, int center,
                     const double* mean, const double* var, int chunks, int64_t tpc, double* part, int NBp) {
  const int kstr = int(ceil_div(n, WS));
  if (kstr * WS > NBp) return -1;
  const dim3 g(unsigned(chunks), unsigned(kstr * (kstr + 1) / 2));
  auto go = [&](auto x, auto vc) {
    typedef typename std::remove_const<typename std::remove_pointer<decltype(x)>::type>::type TS;
    constexpr bool VAR = decltype(vc)::value;
    hipLaunchKernelGGL((k_wgram_f64<TS, VAR>), g, dim3(WNT), 0, st, x, ldx, m, n, center, mean, var, kstr, tpc, part,
                       NBp);
  };
  auto typed = [&](auto x) {
    if (center == 2) go(x, std::true_type{});
    else go(x, std::false_type{});
  };
  if (dt == PC_F64) typed((const double*)X);
  else if (dt == PC_F32) typed((const float*)X);
  else
    return -1;
  return 0;
}

// partial slabs (chunks x PBp x QBp) of A^T B, A m x p and B m x q of one real
// storage type; PBp, QBp multiples of the stripe width
int launch_wxgram_f64(hipStream_t st, pc_dtype dt, const void* A, int64_t lda, int p, const void* B, int64_t ldb,
                      int q, int64_t m, int chunks, int64_t tpc, double* part, int PBp, int QBp) {
  const int kp = int(ceil_div(p, WS)), kq = int(ceil_div(q, WS));
  if (kp * WS > PBp || kq * WS > QBp || int64_t(kp) * kq > 65535) return -1;
  const dim3 g(unsigned(chunks), unsigned(kp * kq));
  if (dt == PC_F64)
    hipLaunchKernelGGL((k_wxgram_f64<double, double>), g, dim3(WNT), 0, st, (const double*)A, lda, p,
                       (const double*)B, ldb, q, m, kq, tpc, part, PBp, QBp);
  else if (dt == PC_F32)
    hipLaunchKernelGGL((k_wxgram_f64<float, float>), g, dim3(WNT), 0, st, (const float*)A, lda, p, (const float*)B,
                       ldb, q, m, kq, tpc, part, PBp, QBp);
  else
    return -1;
  return 0;
}
