// FP64 dense kernels for real n x n matrices (the small dense stage of the POD
// core), n <= 512: shifted Cholesky, pivoted Cholesky, the triangular inverse and
// Householder QR with explicit Q.  The factorisations are blocked, the Cholesky ones
// on one workgroup: matrices live in global memory (L2-resident at these sizes),
// panels in LDS or registers, and the updates run on v_mfma_f64_16x16x4f64.
//
// f64 MFMA 16x16x4 lane layout (wave64): lane l holds A[l % 16][l / 16] and
// B[l / 16][l % 16]; accumulator register r holds D[4 r + l / 16][l % 16].
// Included by solve.hip after k_small.hip (uses NT, block_max, mfma64s, d4s).

namespace dense {

constexpr int PW = 32;           // panel width
constexpr int DMAX = 512;        // widest matrix

// DPP move of a double (both 32-bit halves), lanes that the row mask leaves
// out return `old`
template <int CTRL, int ROWS>
PC_DEV double dpp_f64(double x, double old) {
  const long long xi = __builtin_bit_cast(long long, x), oi = __builtin_bit_cast(long long, old);
  const int lo = __builtin_amdgcn_update_dpp(int(oi), int(xi), CTRL, ROWS, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(int(oi >> 32), int(xi >> 32), CTRL, ROWS, 0xF, false);
  return __builtin_bit_cast(double, (long long)(unsigned)lo | ((long long)hi << 32));
}
PC_DEV double readlane63_f64(double x) {
  const long long xi = __builtin_bit_cast(long long, x);
  const int lo = __builtin_amdgcn_readlane(int(xi), 63), hi = __builtin_amdgcn_readlane(int(xi >> 32), 63);
  return __builtin_bit_cast(double, (long long)(unsigned)lo | ((long long)hi << 32));
}
// Sum over the 64 lanes of a wave, returned to every lane: within each row
// of 16 lanes two quad permutations and two rotations (by 4, by 8) leave the
// row's sum in all its lanes; row 0 is added into row 1 and row 2 into row 3
// (row_bcast:15), then row 1 into rows 2 and 3 (row_bcast:31), so lane 63
// holds every lane once.  Call with the whole wave active.
PC_DEV double wave_sum_dpp(double v) {
  v += dpp_f64<0xB1, 0xF>(v, 0.0);   // quad_perm [1,0,3,2]
  v += dpp_f64<0x4E, 0xF>(v, 0.0);   // quad_perm [2,3,0,1]
  v += dpp_f64<0x124, 0xF>(v, 0.0);  // row_ror:4
  v += dpp_f64<0x128, 0xF>(v, 0.0);  // row_ror:8
  v += dpp_f64<0x142, 0xA>(v, 0.0);  // row_bcast:15 into rows 1, 3
  v += dpp_f64<0x143, 0xC>(v, 0.0);  // row_bcast:31 into rows 2, 3
  return readlane63_f64(v);
}
// Maximum over the 64 lanes, returned to every lane
PC_DEV int wave_max_dpp_i32(int v) {
  v = max(v, __builtin_amdgcn_update_dpp(v, v, 0xB1, 0xF, 0xF, false));
  v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x4E, 0xF, 0xF, false));
  v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x124, 0xF, 0xF, false));
  v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x128, 0xF, 0xF, false));
  v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x142, 0xA, 0xF, false));
  v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x143, 0xC, 0xF, false));
  return __builtin_amdgcn_readlane(v, 63);
}
// x of lane i (wave-uniform), to every lane
PC_DEV double lane_read_f64(double x, int i) {
  const long long b = __builtin_bit_cast(long long, x);
  const int lo = __builtin_amdgcn_readlane(int(b), i), hi = __builtin_amdgcn_readlane(int(b >> 32), i);
  return __builtin_bit_cast(double, (long long)(unsigned)lo | ((long long)hi << 32));
}
// 1 / sqrt(d), d > 0: the hardware's estimate (2^-24) and two Newton steps
PC_DEV double rsqrt_f64(double d) {
  double y = __builtin_amdgcn_rsq(d);
#pragma unroll
  for (int k = 0; k < 2; k++) y = fma(0.5 * y, fma(-d * y, y, 1.0), y);
  return y;
}
// r = sqrt(d) from y = 1 / sqrt(d), and x / r = q + (x - q r) y, q = x y: each result
// corrected by its residual, as a square root and a division would round it
PC_DEV double sqrt_from(double d, double y) {
  const double r = d * y;
  return fma(0.5 * y, fma(-r, r, d), r);
}
PC_DEV double div_by(double x, double r, double y) {
  const double q = x * y;
  return fma(fma(-q, r, x), y, q);
}
// LDS and memory accesses of one wave in program order across its lanes
PC_DEV void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// f(I), f(I + 1), ... f(N - 1), the number a constant
template <int I, int N, class F>
PC_DEV void static_for(F f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<I + 1, N>(f);
  }
}
// The upper tiles of any grid, numbered from its last one: tile k is e / 256 rows and
// e % 256 columns before the last, e = tab[k]
constexpr int kMaxTiles = (DMAX / 16) * (DMAX / 16 + 1) / 2;
PC_DEV void tile_table(unsigned short* tab, int nt, int tid, int nth) {
  for (int e = tid; e < nt * nt; e += nth) {
    const int b = e / nt, a = e % nt;
    if (a <= b) tab[b * (b + 1) / 2 + a] = (unsigned short)(256 * b + a);
  }
}
// f(I, J, acc) over a wave's upper tiles of an nt x nt grid, acc loaded by g(I, J, acc),
// BATCH tiles at a time: their loads are waited for once, before the first of the
// batch's stores (the counter of outstanding accesses covers both, so a wait between
// them would be one for the stores).  g and f keep clear of branches for the same
// reason, and because a branch costs as much as a tile's product.
template <int NW, int BATCH, class L, class F>
PC_DEV void fold_tiles(int w, int nt, const unsigned short* tab, L g, F f) {
  const int count = nt * (nt + 1) / 2;
  for (int t = w; t < count; t += NW * BATCH) {
    int I[BATCH], J[BATCH];
    d4s acc[BATCH];
#pragma unroll
    for (int d = 0; d < BATCH; d++) {
      const int e = __builtin_amdgcn_readfirstlane(tab[min(t + d * NW, count - 1)]);
      I[d] = nt - 1 - (e >> 8);
      J[d] = nt - 1 - (e & 255);
    }
#pragma unroll
    for (int d = 0; d < BATCH; d++) g(I[d], J[d], acc[d]);
#pragma unroll
    for (int d = 0; d < BATCH; d++) asm volatile("" : "+v"(acc[d][0]), "+v"(acc[d][1]), "+v"(acc[d][2]), "+v"(acc[d][3]));
#pragma unroll
    for (int d = 0; d < BATCH; d++)
      if (t + d * NW < count) f(I[d], J[d], acc[d]);
  }
}

}  // namespace dense

// ---------------------------------------------------------------------------
// Shifted Cholesky, real (n <= DMAX): R upper with R^T R = G + tau I, tau =
// shift_rel * max G_ii.  Right-looking with 16-wide panels; a pivot below tau/2
// (rounding made G indefinite at that scale) restarts with tau *= 8.
// status[0] = 1 on a non-finite Gram or when 20 restarts did not suffice.
//
// What bounds it is the chain of pivots, so wave 0 alone factors each 16 x 16
// diagonal block, lane c holding column c in registers: a pivot and its row reach
// the other lanes by lane reads, no barrier and no LDS in the chain (four waves a
// SIMD sharing it, each step behind three barriers: 460 us at n = 256, now 165).  The
// panel's rows are one forward substitution per thread in registers, the trailing
// update MFMA tiles loaded four at a time.  CN: columns P has room for.
// ---------------------------------------------------------------------------
constexpr int kCholThreads = 512;
constexpr int CW = 16;  // panel width: at 32 the factorisation of a block is 60 KB of unrolled code, fetched anew for each
template <int CN>
__global__ __launch_bounds__(kCholThreads) void k_chol_fast(const double* G, int ldg, int n, double shift_rel,
                                                            double* R, int ldr, int* status) {
  using namespace dense;
  constexpr int NW = kCholThreads / 64, LD = CN + 1, DLD = CW + 2;
  static_assert(CN - CW <= kCholThreads, "one thread per panel column");
  __shared__ double P[CW * LD];
  __shared__ __attribute__((aligned(16))) double Dt[CW * DLD];  // column i of the factored block at Dt[i * DLD]
  __shared__ double Ds[CW * DLD];                               // the block to be factored
  __shared__ double ri_s[CW];
  __shared__ unsigned short tab[kMaxTiles];
  __shared__ double sh[32];
  __shared__ int restart;
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, lr = l & 15, lk = l >> 4;
  tile_table(tab, (n + 15) >> 4, tid, kCholThreads);
  double dmax = 0.0;
  for (int i = tid; i < n; i += kCholThreads) dmax = fmax(dmax, G[int64_t(i) * ldg + i]);
  dmax = block_max(dmax, sh);
  if (!isfinite(dmax)) {
    if (tid == 0) status[0] = 1;
    dmax = 1.0;
  }
  double tau = shift_rel * dmax;
  if (!(tau > 0.0)) tau = 1.0;
  for (int attempt = 0; attempt < 20; attempt++) {
    if (tid == 0) restart = 0;
    for (int e = tid; e < CW * CW; e += kCholThreads) {
      const int i = e >> 4, j = e & 15;
      Ds[i * DLD + j] = i < n && j < n ? G[int64_t(i) * ldg + j] + (i == j ? tau : 0.0) : 0.0;
    }
    __syncthreads();
    for (int k0 = 0; k0 < n; k0 += CW) {
      const int bs = min(CW, n - k0);
      // the first panel reads G, the later ones the trailing block left in R
      const double* A = k0 ? R : G;
      const int64_t lda = k0 ? ldr : ldg;
      const double add = k0 ? 0.0 : tau;  // the shift of the diagonal (the update adds it for the later panels)
      const int c1 = k0 + bs, nt = n - c1, ntl = (nt + 15) >> 4;
      // this thread's column of the panel, on its way while the block is factored
      double x[CW];
      const bool own = tid < 16 * ntl, in = tid < nt;
      if (own) {
        const double* src = A + int64_t(k0) * lda + (in ? c1 + tid : 0);
#pragma unroll
        for (int i = 0; i < CW; i++) x[i] = src[int64_t(i) * lda];  // nt > 0: bs = CW
      }
      if (w == 0) {
        const int c = l & 15;
        double a[CW], ri = 1.0;
#pragma unroll
        for (int i = 0; i < CW; i++) {
          const double v = Ds[i * DLD + c];
          a[i] = c < bs ? (i <= c ? v : 0.0) : (i == c ? 1.0 : 0.0);
        }
        bool bad = false, low = false;
#pragma unroll
        for (int j = 0; j < CW; j++) {
          double d = lane_read_f64(a[j], j);
          if (!isfinite(d)) {
            bad = bad || !low;  // what follows a failed pivot may well overflow
            d = tau;
          } else if (j < bs && d < 0.5 * tau) {
            low = true;
            d = tau;
          }
          const double y = rsqrt_f64(d);
          const double r = sqrt_from(d, y);
          a[j] = c == j ? r : div_by(a[j], r, y);
          if (c == j) ri = y;
#pragma unroll
          for (int i = j + 1; i < CW; i++) a[i] = fma(-lane_read_f64(a[j], i), a[j], a[i]);
        }
        if (l < CW) {
          ri_s[c] = ri;
#pragma unroll
          for (int i = 0; i < CW; i++) Dt[c * DLD + i] = i <= c ? a[i] : 0.0;
        }
        if (l == 0) {
          if (bad) status[0] = 1;
          if (low) restart = 1;
        }
      }
      __syncthreads();
      if (restart) break;
      for (int e = tid; e < CW * CW; e += kCholThreads) {
        const int i = e >> 4, j = e & 15;
        if (i < bs && j < bs) R[int64_t(k0 + i) * ldr + k0 + j] = Dt[j * DLD + i];
      }
      // panel: rows k0..k0+bs-1 of R right of the block, D^T X = A, a column per thread
      if (own) {
#pragma unroll
        for (int i = 0; i < CW; i++) {
          double s = in ? x[i] : 0.0;
#pragma unroll
          for (int t = 0; t < i; t++) s = fma(-Dt[i * DLD + t], x[t], s);
          x[i] = div_by(s, Dt[i * DLD + i], ri_s[i]);
          P[i * LD + tid] = x[i];
          if (in) R[int64_t(k0 + i) * ldr + c1 + tid] = x[i];
        }
      }
      __syncthreads();
      // trailing update (upper tiles): A[c1:, c1:] -= P^T P; the next panel's block also to LDS
      fold_tiles<NW, 4>(
          w, ntl, tab,
          [&](int I, int J, d4s& acc) {
            const double* src = A + int64_t(c1) * lda + c1 + min(16 * J + lr, nt - 1);
#pragma unroll
            for (int r = 0; r < 4; r++) acc[r] = src[min(16 * I + 4 * r + lk, nt - 1) * int(lda)];
          },
          [&](int I, int J, d4s acc) {
#pragma unroll
            for (int r = 0; r < 4; r++) acc[r] = -(I == J && 4 * r + lk == lr ? acc[r] + add : acc[r]);
#pragma unroll
            for (int k = 0; k < CW; k += 4)
              acc = mfma64s(P[(k + lk) * LD + 16 * I + lr], P[(k + lk) * LD + 16 * J + lr], acc);
            double* dst = R + (c1 + 16 * I + lk) * ldr + c1 + 16 * J + lr;
            if (J == 0) {
#pragma unroll
              for (int r = 0; r < 4; r++) Ds[(4 * r + lk) * DLD + lr] = -acc[r];
            } else if (16 * J + 16 <= nt) {  // I <= J: all rows too
#pragma unroll
              for (int r = 0; r < 4; r++) dst[4 * r * ldr] = -acc[r];
            } else {
#pragma unroll
              for (int r = 0; r < 4; r++)
                if (16 * I + 4 * r + lk < nt && 16 * J + lr < nt) dst[4 * r * ldr] = -acc[r];
            }
          });
      __syncthreads();
    }
    const int again = restart;
    __syncthreads();
    if (!again) {
      // strictly lower part
      for (int i = w; i < n; i += NW)
        for (int j = l; j < i; j += 64) R[int64_t(i) * ldr + j] = 0.0;
      return;
    }
    tau *= 8.0;
  }
  if (tid == 0) status[0] = 1;
}

// ---------------------------------------------------------------------------
// Pivoted Cholesky with rank detection, real (n <= 256 C): P^T G P = R^T R.  Row j
// of R picks the unpivoted column p with the largest Schur diagonal (ties to the
// lower index), R[j][q] = (A[p][q] - sum_{t in panel, t < j} R[t][p] R[t][q]) /
// sqrt(d_p); after 32 rows they are folded into A.  Stops when the largest
// remaining diagonal is <= tol * max(diag G) (rank); perm[rank..] lists the
// unpivoted columns in increasing order.
//
// The pivot steps form one chain: largest diagonal, its row of A from L2, new row,
// diagonals.  One wave per SIMD, thread t owning columns t + 256 c: with 16 waves
// the chain's scalar work was issued four times per SIMD (2.0 us a step), with one
// wave its LDS traffic and selections came one after the other (1.7 us).  The panel's
// products run while A's row comes.  One
// barrier per step, over which the waves exchange their largest diagonals.
// The fold runs on MFMA and writes the Schur complement of the remaining columns
// only, compacted (in increasing order) into the other of two buffers: a third of
// the products that a fold of all columns does.  n = 256: 568 -> 270 us (1,800
// cycles a step, a fifth of the time in the folds).
//
// A, B: n x n workspaces.  R leaves with its columns in G's order (R[t][q], only
// the columns unpivoted before row t's panel written); k_pchol_cols permutes them.
// ---------------------------------------------------------------------------
constexpr int kPcholThreads = 256;
template <int C>
__global__ __launch_bounds__(kPcholThreads) void k_pchol_fast(const double* G, int ldg, int n, double tol, double* A,
                                                              double* B, double* R, int ldr, int* perm, int* rank_out,
                                                              int* status) {
  using namespace dense;
  constexpr int NTH = kPcholThreads, NW = NTH / 64, N = NTH * C, LD = PW + 2;
  __shared__ __attribute__((aligned(16))) double P[N * LD];  // entry t of column q at P[q * LD + t]
  __shared__ double dgs[N];          // diagonals, compacted
  __shared__ short id[N], al[N];     // column of a position; its position before the fold
  __shared__ short prm[N];           // the pivots
  __shared__ double cand_v[2][NW];   // the waves' largest diagonals and their positions
  __shared__ int cand_p[2][NW];
  __shared__ int kept[NW * C];
  __shared__ unsigned short tab[kMaxTiles];
  __shared__ double sh[32];
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, lr = l & 15, lk = l >> 4;
  tile_table(tab, (n + 15) >> 4, tid, NTH);
  double dmax = 0.0;
  for (int q = tid; q < n; q += NTH) {
    const double d = G[int64_t(q) * ldg + q];
    dmax = fmax(dmax, d);
    dgs[q] = d;
    id[q] = short(q);
  }
  for (int e = tid; e < N * LD; e += NTH) P[e] = 0.0;
  dmax = block_max(dmax, sh);
  if (!(dmax > 0.0) || !isfinite(dmax)) {
    for (int q = tid; q < n; q += NTH) perm[q] = q;
    if (tid == 0) {
      rank_out[0] = 0;
      if (!isfinite(dmax)) atomicOr(status, 16);
    }
    return;
  }
  const double thr = tol * dmax;
  const double* S = G;  // Schur complement of the na remaining columns
  int64_t lds = ldg;
  int na = n, rank = n;
  for (int k0 = 0; k0 < n; k0 += PW) {
    const int bs = min(PW, n - k0);
    // dq: the Schur diagonal, -2 once pivoted, -1 if NaN (never a pivot), -3 beyond na
    double dq[C];
#pragma unroll
    for (int c = 0; c < C; c++) {
      const int q = tid + NTH * c;
      const double d = q < na ? dgs[q] : -3.0;
      dq[c] = d == d ? d : -1.0;
#pragma unroll
      for (int t = 0; t < PW; t++) P[q * LD + t] = 0.0;
    }
    // The wave's largest diagonal (lowest position of several) into slot sl, by the high
    // words, which order non-negative doubles and put the negative marks last; the
    // low words only if several lanes share the highest.
    auto offer = [&](int sl) {
      double v = dq[0];
      int q = tid;
#pragma unroll
      for (int c = 1; c < C; c++)
        if (dq[c] > v) {
          v = dq[c];
          q = tid + NTH * c;
        }
      const int hi = __double2hiint(v), lo = __double2loint(v);
      const int hm = wave_max_dpp_i32(hi);
      uint64_t at = __ballot(hi == hm);
      if (at & (at - 1)) {
        const int lm = wave_max_dpp_i32(hi == hm ? int(unsigned(lo) >> 1) : 0);  // 31 bits: signed order
        const bool top = hi == hm && int(unsigned(lo) >> 1) == lm;
        at = __ballot(top && (lo & 1));
        if (!at) at = __ballot(top);
        if (C > 1 && (at & (at - 1))) {  // equal: the lowest position, not the lowest lane
          int best = 1 << 30;
          for (uint64_t m = at; m; m &= m - 1) best = min(best, __builtin_amdgcn_readlane(q, __builtin_ctzll(m)));
          at = __ballot(q == best && ((at >> l) & 1));
        }
      }
      if (l == __builtin_ctzll(at)) {
        cand_v[sl][w] = v;
        cand_p[sl][w] = q;
      }
    };
    offer(0);
    __syncthreads();
    int jj = 0;
    for (; jj < bs; jj++) {
      const int sl = jj & 1;
      double bk[NW];
      int pk[NW];
#pragma unroll
      for (int k = 0; k < NW; k++) {
        bk[k] = cand_v[sl][k];
        pk[k] = cand_p[sl][k];
      }
      double b = bk[0];
      int p = pk[0];
#pragma unroll
      for (int k = 1; k < NW; k++) {
        const bool up = bk[k] > b || (C > 1 && bk[k] == b && pk[k] < p);
        b = up ? bk[k] : b;
        p = up ? pk[k] : p;
      }
      p = __builtin_amdgcn_readfirstlane(p);
      if (__ballot(b > thr) == 0) break;
      double x[C], s[C][4];
#pragma unroll
      for (int c = 0; c < C; c++) {
        const int q = tid + NTH * c;
        x[c] = S[int64_t(p) * lds + (q < na ? q : 0)];
        s[c][0] = s[c][1] = s[c][2] = s[c][3] = 0.0;
      }
      const double y = rsqrt_f64(b), r = sqrt_from(b, y);
      // The products of column p's panel entries (the same address in every lane) and this
      // thread's (zero from entry jj on) run while A's row comes.  jd hides jj, or the
      // compiler makes a loop of its own for each group of entries (32 KB of code).
      int jd = jj;
      asm volatile("" : "+s"(jd));
#pragma unroll
      for (int t0 = 0; t0 < PW; t0 += 8)
        if (t0 < jd) {
          double pp[8], pr[C][8];
#pragma unroll
          for (int t = 0; t < 8; t++) {
            pp[t] = P[p * LD + t0 + t];
#pragma unroll
            for (int c = 0; c < C; c++) pr[c][t] = P[(tid + NTH * c) * LD + t0 + t];
          }
#pragma unroll
          for (int t = 0; t < 8; t++)
#pragma unroll
            for (int c = 0; c < C; c++) s[c][t & 3] = fma(pp[t], pr[c][t], s[c][t & 3]);
        }
      if (tid == 0) prm[k0 + jj] = short(p);  // as positions until the panel's end
#pragma unroll
      for (int c = 0; c < C; c++) {
        const int q = tid + NTH * c;
        double v = div_by(x[c] - ((s[c][0] + s[c][1]) + (s[c][2] + s[c][3])), r, y);
        double d = fmax(fma(-v, v, dq[c]), 0.0);
        asm volatile("" : "+v"(v), "+v"(d));  // selections, no branches around them
        v = q == p ? r : dq[c] <= -2.0 ? 0.0 : v;
        dq[c] = q == p ? -2.0 : dq[c] >= 0.0 ? d : dq[c];
        P[q * LD + jj] = v;
      }
      offer(sl ^ 1);
      __syncthreads();
    }
    // the remaining columns, in order, move up
    int mine[C];
#pragma unroll
    for (int c = 0; c < C; c++) {
      const uint64_t m = __ballot(dq[c] > -2.0);
      mine[c] = __builtin_popcountll(m & ((uint64_t(1) << l) - 1));
      if (l == 0) kept[c * NW + w] = __builtin_popcountll(m);
    }
    __syncthreads();
    int nr = 0;
#pragma unroll
    for (int k = 0; k < NW * C; k++) {
#pragma unroll
      for (int c = 0; c < C; c++)
        if (k < c * NW + w) mine[c] += kept[k];
      nr += kept[k];
    }
#pragma unroll
    for (int c = 0; c < C; c++)
      if (dq[c] > -2.0) {
        al[mine[c]] = short(tid + NTH * c);
        dgs[mine[c]] = dq[c];
      }
    if (tid < jj) prm[k0 + tid] = id[prm[k0 + tid]];
#pragma unroll
    for (int c = 0; c < C; c++) {
      const int q = tid + NTH * c;
      if (q < na) {
        double* o = R + int64_t(k0) * ldr + id[q];
        for (int t = 0; t < jj; t++) o[int64_t(t) * ldr] = P[q * LD + t];
      }
    }
    __syncthreads();
    short nid[C];  // columns of this thread's positions after the fold
#pragma unroll
    for (int c = 0; c < C; c++) nid[c] = tid + NTH * c < nr ? id[al[tid + NTH * c]] : short(0);
    if (jj < bs || k0 + bs >= n) {
      rank = k0 + jj;
#pragma unroll
      for (int c = 0; c < C; c++)
        if (tid + NTH * c < nr) prm[rank + tid + NTH * c] = nid[c];
      break;
    }
    // fold the panel into the remaining columns (upper tiles, mirrored)
    double* D = S == A ? B : A;
    fold_tiles<NW, 6>(
        w, (nr + 15) >> 4, tab,
        [&](int I, int J, d4s& acc) {
          const double* src = S + al[min(16 * J + lr, nr - 1)];
#pragma unroll
          for (int r = 0; r < 4; r++) acc[r] = src[al[min(16 * I + 4 * r + lk, nr - 1)] * int(lds)];
        },
        [&](int I, int J, d4s acc) {
          acc = -acc;
          const int pi = al[min(16 * I + lr, nr - 1)] * LD + lk, pj = al[min(16 * J + lr, nr - 1)] * LD + lk;
#pragma unroll
          for (int k = 0; k < PW; k += 4) acc = mfma64s(P[pi + k], P[pj + k], acc);
          const int row = 16 * I + lk, col = 16 * J + lr;
          double *d0 = D + row * n + col, *d1 = D + col * n + row;
          if (16 * J + 16 <= nr) {  // I <= J: all rows too; a diagonal tile is its own mirror
#pragma unroll
            for (int r = 0; r < 4; r++) {
              d0[4 * r * n] = -acc[r];
              d1[4 * r] = -acc[r];
            }
          } else {
#pragma unroll
            for (int r = 0; r < 4; r++)
              if (row + 4 * r < nr && col < nr) {
                d0[4 * r * n] = -acc[r];
                d1[4 * r] = -acc[r];
              }
          }
        });
    __syncthreads();
#pragma unroll
    for (int c = 0; c < C; c++)
      if (tid + NTH * c < nr) id[tid + NTH * c] = nid[c];
    S = D;
    lds = n;
    na = nr;
    __syncthreads();
  }
  __syncthreads();
  for (int q = tid; q < n; q += NTH) perm[q] = prm[q];
  if (tid == 0) rank_out[0] = rank;
}

// R[t][c] <- R[t][perm[c]] (c >= t, t < rank), 0 elsewhere; one wave per row
template <int C>
__global__ __launch_bounds__(256) void k_pchol_cols(double* R, int ldr, int n, const int* perm, const int* rank) {
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6), l = threadIdx.x & 63;
  if (t >= n) return;
  double* r = R + int64_t(t) * ldr;
  const bool in = t < rank[0];
  double v[C];
#pragma unroll
  for (int c = 0; c < C; c++) {
    const int q = l + 64 * c, p = q < n ? perm[q] : 0;
    const double x = r[p >= 0 && p < n ? p : 0];
    v[c] = in && q >= t ? x : 0.0;
  }
  // a lane's stores come after every lane's loads
#pragma unroll
  for (int c = 0; c < C; c++) asm volatile("" : "+v"(v[c]));
  dense::wave_fence();
#pragma unroll
  for (int c = 0; c < C; c++)
    if (l + 64 * c < n) r[l + 64 * c] = v[c];
}

// ---------------------------------------------------------------------------
// Householder QR of a real n x n matrix (n <= 64 RW), A = Q R, Q explicit.
// LAPACK conventions (beta = -sign(alpha) ||x||, tau = (beta - alpha) / beta).
// Panels of 32 columns are factored on one workgroup (k_hqr_panel: the column loop,
// V^T V, T of the compact WY form); the block reflector I - V T V^T updates the
// trailing columns after each panel, and Q, accumulated backwards, one workgroup per
// 32-column strip (k_hqr_strip).  work: n*n (the factored matrix) + n (tau) +
// 32*32*ceil(n/32) (T).
//
// The column loop is a chain (norm, reflector, its products with the other columns),
// so the panel lives in the registers of one wave per SIMD, wave w holding columns
// w + 4 k, lane l rows l + 64 q: only the reflector goes through LDS, one barrier per
// column, and a wave reduces its columns' dot products together.  n = 256: a panel 69
// -> 29 us (on 16 waves, each forming the reflector and summing its columns' products
// one after the other), a strip 9 to 25 -> 10 us.
// ---------------------------------------------------------------------------
// d[v] summed over the 64 lanes, in the lanes l with l % 4 = v % 4 of set[v / 4]
template <int CNT>
PC_DEV void wave_sums(const double (&d)[CNT], double (&set)[(CNT + 3) / 4]) {
  using namespace dense;
  const bool b0 = threadIdx.x & 1, b1 = threadIdx.x & 2;
  constexpr int HALF = (CNT + 1) / 2;
  double h[HALF];
#pragma unroll
  for (int k = 0; k < HALF; k++) {
    const double x = d[2 * k], y = 2 * k + 1 < CNT ? d[2 * k + 1] : d[2 * k];
    h[k] = (b0 ? y : x) + dpp_f64<0xB1, 0xF>(b0 ? x : y, 0.0);  // lane l ^ 1
  }
#pragma unroll
  for (int k = 0; k < (CNT + 3) / 4; k++) {
    const double x = h[2 * k], y = 2 * k + 1 < HALF ? h[2 * k + 1] : h[2 * k];
    double v = (b1 ? y : x) + dpp_f64<0x4E, 0xF>(b1 ? x : y, 0.0);  // lane l ^ 2
    v += dpp_f64<0x124, 0xF>(v, 0.0);                               // row_ror:4
    v += dpp_f64<0x128, 0xF>(v, 0.0);                               // row_ror:8
    // rows 0 and 1, 2 and 3, then the halves: the swaps leave both terms in every lane
    auto both = [](double u, auto swap) {
      const long long bits = __builtin_bit_cast(long long, u);
      const auto lo = swap(unsigned(bits)), hi = swap(unsigned(bits >> 32));
      return __builtin_bit_cast(double, (long long)lo[0] | ((long long)hi[0] << 32)) +
             __builtin_bit_cast(double, (long long)lo[1] | ((long long)hi[1] << 32));
    };
    v = both(v, [](unsigned x) { return __builtin_amdgcn_permlane16_swap(x, x, false, false); });
    v = both(v, [](unsigned x) { return __builtin_amdgcn_permlane32_swap(x, x, false, false); });
    set[k] = v;
  }
}

constexpr int kHqrThreads = 256;
template <int RW>
__global__ __launch_bounds__(kHqrThreads) void k_hqr_panel(const double* __restrict__ A, int lda, int n, int pp,
                                                           double* __restrict__ work) {
  using namespace dense;
  constexpr int NW = kHqrThreads / 64, K = PW / NW, LD = 64 * RW + 1;
  __shared__ double Pn[PW * LD];  // panel columns (column c at Pn[c * LD], rows relative to the panel start)
  __shared__ double Xs[PW * (PW + 1)];  // V^T V
  __shared__ double Ts[PW * (PW + 1)];
  __shared__ double vb[2][64 * RW], tau_s[PW];
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, lr = l & 15, lk = l >> 4;
  double* Wm = work;
  double* tau = work + int64_t(n) * n;
  double* Tg = tau + n;
  const int c0 = pp * PW, bs = min(PW, n - c0), mr = n - c0;
  {
    const double* src = pp ? Wm + int64_t(c0) * n + c0 : A;  // the first panel comes from A
    const int lds = pp ? n : lda, c = tid & 31, i0 = tid >> 5;
    constexpr int PER = 64 * RW / (kHqrThreads / 32);
    double v[PER];
#pragma unroll
    for (int u = 0; u < PER; u++) v[u] = src[min(i0 + 8 * u, mr - 1) * lds + min(c, bs - 1)];
#pragma unroll
    for (int u = 0; u < PER; u++) Pn[c * LD + i0 + 8 * u] = c < bs && i0 + 8 * u < mr ? v[u] : 0.0;
  }
  if (tid < PW) tau_s[tid] = 0.0;
  __syncthreads();
  double a[K][RW];  // column w + NW k, row l + 64 q
#pragma unroll
  for (int k = 0; k < K; k++)
#pragma unroll
    for (int q = 0; q < RW; q++) a[k][q] = Pn[(w + NW * k) * LD + l + 64 * q];
  static_for<0, K>([&](auto kc) {
    constexpr int k = decltype(kc)::value;
#pragma unroll 1
    for (int o = 0; o < NW; o++) {
      const int j = NW * k + o;
      if (j >= bs) break;
      double* v_s = vb[o & 1];
      if (w == o) {
        // rows above j are R's; s: the squares below
        double s = l > j ? a[k][0] * a[k][0] : 0.0;
#pragma unroll
        for (int q = 1; q < RW; q++) s = fma(a[k][q], a[k][q], s);
        s = wave_sum_dpp(s);
        const double al = lane_read_f64(a[k][0], j);
        double tj = 0.0, sc = 0.0, beta = al;
        if (s != 0.0) {
          const double anorm = sqrt(al * al + s);
          beta = al >= 0 ? -anorm : anorm;
          tj = (beta - al) / beta;
          sc = 1.0 / (al - beta);
        }
#pragma unroll
        for (int q = 0; q < RW; q++) {
          const bool below = q > 0 || l > j;
          const double v = a[k][q] * sc;
          a[k][q] = below ? v : l == j ? beta : a[k][q];
          v_s[l + 64 * q] = below ? v : l == j ? 1.0 : 0.0;
        }
        if (l == 0) tau_s[j] = tj;
      }
      __syncthreads();
      double v[RW], d[K - k], set[(K - k + 3) / 4];
#pragma unroll
      for (int q = 0; q < RW; q++) v[q] = v_s[l + 64 * q];
      const double tj = tau_s[j];
#pragma unroll
      for (int x = k; x < K; x++) {
        d[x - k] = v[0] * a[x][0];
#pragma unroll
        for (int q = 1; q < RW; q++) d[x - k] = fma(v[q], a[x][q], d[x - k]);
      }
      wave_sums<K - k>(d, set);
#pragma unroll
      for (int x = k; x < K; x++) {
        double f = tj * lane_read_f64(set[(x - k) / 4], (x - k) % 4);
        if (x == k && w <= o) f = 0.0;  // columns up to j are done
#pragma unroll
        for (int q = 0; q < RW; q++) a[x][q] = fma(-v[q], f, a[x][q]);
      }
    }
  });
#pragma unroll
  for (int k = 0; k < K; k++)
#pragma unroll
    for (int q = 0; q < RW; q++) Pn[(w + NW * k) * LD + l + 64 * q] = a[k][q];
  __syncthreads();
  // V: unit diagonal, zero above
  auto vget = [&](int i, int c) -> double {
    const double v = Pn[c * LD + i];
    return i < c ? 0.0 : (i == c ? 1.0 : v);
  };
  // V^T V into Xs: four 16 x 16 tiles, one wave each, two accumulators over alternating
  // k-steps (rows beyond mr are zero, and so are columns beyond bs below the diagonal)
  {
    const int I = w >> 1, J = w & 1, ca = 16 * I + lr, cb = 16 * J + lr;
    d4s a0 = {0.0, 0.0, 0.0, 0.0}, a1 = {0.0, 0.0, 0.0, 0.0};
    const int kend = min(64 * RW, (mr + 7) & ~7);
#pragma unroll 4
    for (int k0 = 0; k0 < kend; k0 += 8) {
      a0 = mfma64s(vget(k0 + lk, ca), vget(k0 + lk, cb), a0);
      a1 = mfma64s(vget(k0 + 4 + lk, ca), vget(k0 + 4 + lk, cb), a1);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) Xs[(16 * I + 4 * r + lk) * (PW + 1) + cb] = a0[r] + a1[r];
  }
  __syncthreads();
  // T of the compact WY form.  T^-1 = diag(1 / tau) + strictly upper
  // (V^T V) (Puglisi 1992), so in 16 x 16 blocks T11 and T22 come from back
  // substitution, one lane per column in registers: T_jj = tau_j,
  // T_ij = -tau_i sum_{k = i+1..j} (V^T V)_ik T_kj; multiplying by tau_i
  // (not dividing by 1 / tau_i) keeps a trivial reflector (tau_i = 0) exact,
  // its row and column of T zero.  Then T12 = -T11 (V^T V)_12 T22 on MFMA.
  // The other waves store the panel meanwhile.
  if (w == 0) {
    {
      // lane jl of half-wave `base / 16` owns column jl of block (base, base)
      const int base = 16 * ((l >> 4) & 1), jl = l & 15;
      double tc[16];
#pragma unroll
      for (int i = 15; i >= 0; i--) {
        double acc = 0.0;
#pragma unroll
        for (int k = i + 1; k < 16; k++) acc += Xs[(base + i) * (PW + 1) + base + k] * tc[k];
        const double ti = tau_s[base + i];
        tc[i] = i == jl ? ti : (i < jl ? -ti * acc : 0.0);
      }
      if (l < 32) {
#pragma unroll
        for (int i = 0; i < 16; i++) Ts[(base + i) * (PW + 1) + base + jl] = tc[i];
      }
      if (l < 16)
        for (int i = 0; i < 16; i++) Ts[(16 + i) * (PW + 1) + jl] = 0.0;
    }
    wave_fence();
    // W = (V^T V)_12 T22 into the lower-left block of Xs (not read again)
    d4s acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k0 = 0; k0 < 16; k0 += 4)
      acc = mfma64s(Xs[lr * (PW + 1) + 16 + k0 + lk], Ts[(16 + k0 + lk) * (PW + 1) + 16 + lr], acc);
#pragma unroll
    for (int r = 0; r < 4; r++) Xs[(16 + 4 * r + lk) * (PW + 1) + lr] = acc[r];
    wave_fence();
    acc = d4s{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k0 = 0; k0 < 16; k0 += 4)
      acc = mfma64s(Ts[lr * (PW + 1) + k0 + lk], Xs[(16 + k0 + lk) * (PW + 1) + lr], acc);
#pragma unroll
    for (int r = 0; r < 4; r++) Ts[(4 * r + lk) * (PW + 1) + 16 + lr] = -acc[r];
    wave_fence();
    for (int e = l; e < PW * PW; e += 64) Tg[int64_t(pp) * PW * PW + e] = Ts[(e >> 5) * (PW + 1) + (e & 31)];
    if (l < bs) tau[c0 + l] = tau_s[l];
  } else {
    const int c = tid & 31;
    if (c < bs)
      for (int i = (tid - 64) >> 5; i < mr; i += 6) Wm[int64_t(c0 + i) * n + c0 + c] = Pn[c * LD + i];
  }
}

// One workgroup per 32-column strip: qmode 0 updates the trailing columns of Wm after
// panel pp (those of the first panel come from A), qmode 1 applies panel pp's block
// reflector to Q.  A wave holds the strip's rows 16 (w + 4 u) .. + 15 in registers in the
// products' accumulator layout, which is the right operand's of X = V^T B: entry r of
// tile u is row 4 r + lk of the tile, the four rows of one k-step.  X is the sum of the
// waves' parts, Y = T^T X or T X, and the same registers are the accumulators of
// B - V Y, so B is read and written once and never staged.
template <int RW>
__global__ __launch_bounds__(kHqrThreads) void k_hqr_strip(const double* A, int lda, int n, int pp, int qmode,
                                                           double* work, double* Q, int ldq) {
  using namespace dense;
  constexpr int NW = kHqrThreads / 64, LD = 64 * RW + 1, XLD = PW + 1;
  __shared__ double Pn[PW * LD];
  __shared__ double Xs[NW - 1][PW * XLD];
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, lr = l & 15, lk = l >> 4;
  double* Wm = work;
  const double* T = work + int64_t(n) * n + n + int64_t(pp) * PW * PW;
  const int c0 = pp * PW, bs = min(PW, n - c0), mr = n - c0;
  const int cst = qmode ? c0 : c0 + bs;  // first column of the updated block
  const int ncols = n - cst, s0 = 32 * blockIdx.x;
  if (s0 >= ncols) return;
  double* B = qmode ? Q + int64_t(c0) * ldq + cst : Wm + int64_t(c0) * n + cst;
  const int ldb = qmode ? ldq : n;
  const double* Bin = !qmode && pp == 0 ? A + cst : B;
  const int ldi = !qmode && pp == 0 ? lda : ldb;
  // V below the diagonal (its diagonal is 1), the strip and this wave's tile of T: every
  // load goes out before the first is waited for
  const int ti = w >> 1, tj = w & 1;  // this wave's tile of Y
  d4s b[RW][2];
  double tv[PW / 4];
  {
    const int c = tid & 31, i0 = tid >> 5;
    constexpr int PER = 64 * RW / (kHqrThreads / 32);
    double v[PER];
#pragma unroll
    for (int u = 0; u < PER; u++) v[u] = Wm[(c0 + min(i0 + 8 * u, mr - 1)) * n + c0 + min(c, bs - 1)];
#pragma unroll
    for (int u = 0; u < RW; u++)
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int r = 0; r < 4; r++)
          b[u][h][r] = Bin[min(16 * (w + NW * u) + 4 * r + lk, mr - 1) * ldi + min(s0 + 16 * h + lr, ncols - 1)];
#pragma unroll
    for (int k = 0; k < PW / 4; k++) {
      const int i = 16 * ti + lr, x = 4 * k + lk;
      tv[k] = qmode ? T[i * PW + x] : T[x * PW + i];
    }
#pragma unroll
    for (int u = 0; u < PER; u++) {
      const int i = i0 + 8 * u;
      Pn[c * LD + i] = i < mr && c < bs && i >= c ? (i == c ? 1.0 : v[u]) : 0.0;
    }
#pragma unroll
    for (int u = 0; u < RW; u++)
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int r = 0; r < 4; r++)
          if (16 * (w + NW * u) + 4 * r + lk >= mr) b[u][h][r] = 0.0;
  }
  __syncthreads();
  d4s x[2][2] = {};
#pragma unroll
  for (int u = 0; u < RW; u++)
    if (16 * (w + NW * u) < mr) {
#pragma unroll
      for (int r = 0; r < 4; r++)
#pragma unroll
        for (int I = 0; I < 2; I++) {
          const double v = Pn[(16 * I + lr) * LD + 16 * (w + NW * u) + 4 * r + lk];
#pragma unroll
          for (int h = 0; h < 2; h++) x[I][h] = mfma64s(v, b[u][h][r], x[I][h]);
        }
    }
  if (w > 0) {
#pragma unroll
    for (int I = 0; I < 2; I++)
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int r = 0; r < 4; r++) Xs[w - 1][(16 * I + 4 * r + lk) * XLD + 16 * h + lr] = x[I][h][r];
  }
  __syncthreads();
  if (w == 0) {
#pragma unroll
    for (int I = 0; I < 2; I++)
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int e = (16 * I + 4 * r + lk) * XLD + 16 * h + lr;
          Xs[0][e] = (x[I][h][r] + Xs[0][e]) + (Xs[1][e] + Xs[2][e]);
        }
  }
  __syncthreads();
  {
    d4s y = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < PW / 4; k++) y = mfma64s(tv[k], Xs[0][(4 * k + lk) * XLD + 16 * tj + lr], y);
#pragma unroll
    for (int r = 0; r < 4; r++) Xs[1][(16 * ti + 4 * r + lk) * XLD + 16 * tj + lr] = -y[r];
  }
  __syncthreads();
  double yv[PW / 4][2];
#pragma unroll
  for (int k = 0; k < PW / 4; k++)
#pragma unroll
    for (int h = 0; h < 2; h++) yv[k][h] = Xs[1][(4 * k + lk) * XLD + 16 * h + lr];
#pragma unroll
  for (int u = 0; u < RW; u++) {
    const int i0 = 16 * (w + NW * u);
    if (i0 < mr) {
#pragma unroll
      for (int k = 0; k < PW / 4; k++) {
        const double v = Pn[(4 * k + lk) * LD + i0 + lr];
#pragma unroll
        for (int h = 0; h < 2; h++) b[u][h] = mfma64s(v, yv[k][h], b[u][h]);
      }
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int r = 0; r < 4; r++)
          if (i0 + 4 * r + lk < mr && s0 + 16 * h + lr < ncols)
            B[int64_t(i0 + 4 * r + lk) * ldb + s0 + 16 * h + lr] = b[u][h][r];
    }
  }
}

// R (upper part of the factored matrix) and Q = I before the backward accumulation
__global__ __launch_bounds__(256) void k_hqr_rq(int n, const double* __restrict__ work, double* __restrict__ R,
                                                int ldr, double* __restrict__ Q, int ldq) {
  const int64_t idx = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (idx >= int64_t(n) * n) return;
  const int i = int(idx / n), j = int(idx % n);
  R[int64_t(i) * ldr + j] = i <= j ? work[idx] : 0.0;
  Q[int64_t(i) * ldq + j] = i == j ? 1.0 : 0.0;
}

// W = R^-1 for an upper triangular R (n <= 64 C, row-major, zeros below), one
// wavefront per column j of W: the back substitution R w = e_j runs from i = j down
// to 0 with the right-hand side r in registers (lane l owns rows l + 64 q):
//   w_i = r_i / R_ii,   r_k -= R_ki w_i  (k < i).
// The columns of R a stretch of ST steps needs are staged in LDS, rows padded to an
// odd number of doubles so that the lanes of a wave read one column without bank
// conflicts.  A workgroup's four waves solve four neighbouring columns on the same
// stretches, so the staging, which took 85 % of the time of a lone wave, has four
// times the loads in flight and is done once for the four (n = 256: 97 -> 27 us).
// The chain of a step is two lane reads and four FMAs (125 cycles): the row block
// that holds r_i is known when the code is compiled and rows at or below i, which
// nothing reads again, are updated with the others, so no selection or mask is in it.
// rank: R's rows from rank[0] on are zero and count as the identity's.
template <int C>
__global__ __launch_bounds__(256) void k_trinv_cols(const double* __restrict__ R, int ldr, int n,
                                                    const int* __restrict__ rank, double* __restrict__ W, int ldw) {
  constexpr int ST = C <= 4 ? 64 : 32, LD = ST + 1, PER = 64 / ST;
  __shared__ double Rs[64 * C * LD];
  const int jw = n - 1 - 4 * int(blockIdx.x);  // the workgroup's last column; the longest go first
  const int j = jw - int(threadIdx.x >> 6), l = threadIdx.x & 63;
  const int rk0 = rank ? rank[0] : n;
  double r[C], w[C];
#pragma unroll
  for (int q = 0; q < C; q++) {
    r[q] = (l + 64 * q == j) ? 1.0 : 0.0;
    w[q] = 0.0;
  }
#pragma unroll
  for (int g = C - 1; g >= 0; g--)  // rows 64 g .. 64 g + 63
#pragma unroll
    for (int h = PER - 1; h >= 0; h--) {
      const int c0 = 64 * g + ST * h;
      if (c0 > jw) continue;
      // eight steps at a time up to the workgroup's last column: below row j (i > j) the
      // right-hand side is zero and the diagonal counts as 1, so those steps do nothing
      const int cl = j - c0 < ST - 1 ? j - c0 : ST - 1;
      __syncthreads();  // the previous stretch has been read
      {
        constexpr int ROWS = 256 / ST;  // rows a pass of the workgroup loads
        const int lc = threadIdx.x % ST, r0 = threadIdx.x / ST;
        const bool ok = c0 + lc < n;
        const double* src = R + (ok ? c0 + lc : 0);
        double v[64 * C / ROWS];
#pragma unroll
        for (int u = 0; u < 64 * (g + 1) / ROWS; u++) {
          const int k = r0 + ROWS * u;
          v[u] = src[k < n ? int64_t(k) * ldr : 0];
        }
#pragma unroll
        for (int u = 0; u < 64 * (g + 1) / ROWS; u++) {
          const int k = r0 + ROWS * u;
          Rs[k * LD + lc] = ok && k < n ? v[u] : 0.0;
        }
      }
      __syncthreads();
      // The stretch's diagonal and its reciprocals, one division per lane in
      // parallel.  A step's quotient is then q0 = r y refined by one residual
      // step, q0 + (r - d q0) y (the last step of Newton-Markstein division),
      // so the division leaves the step's dependency chain.
      const int ld = l % ST;
      const double dgl = ld <= cl && c0 + ld < rk0 ? Rs[(c0 + ld) * LD + ld] : 1.0;
      const double dl = 1.0 / dgl;
      for (int t8 = min(jw - c0, ST - 1) & ~7; t8 >= 0; t8 -= 8) {
#pragma unroll
        for (int t = t8 + 7; t >= t8; --t) {
          double rk[C];
#pragma unroll
          for (int q = 0; q <= g; q++) rk[q] = Rs[(l + 64 * q) * LD + t];
          const int tl = ST * h + t;  // the lane of row c0 + t
          const double rt = dense::lane_read_f64(r[g], tl), d = dense::lane_read_f64(dgl, t),
                       y = dense::lane_read_f64(dl, t);
          const double q0 = rt * y;
          const double wi = fma(fma(-d, q0, rt), y, q0);
          w[g] = l == tl ? wi : w[g];
#pragma unroll
          for (int q = 0; q <= g; q++) r[q] = fma(-rk[q], wi, r[q]);
        }
      }
    }
  if (j < 0) return;
#pragma unroll
  for (int q = 0; q < C; q++) {
    const int k = l + 64 * q;
    if (k < n) W[int64_t(k) * ldw + j] = k <= j ? w[q] : 0.0;
  }
}
