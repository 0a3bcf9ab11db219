// FP64 MFMA streaming kernels for narrow operands (at most 64 real columns, or a
// product whose W fits one CU's LDS): every wave works on its own rows, straight
// from global memory to MFMA fragments, with no barrier in the row loop.
//
// What bounds these sizes is HBM (30 columns: 4 flop / B in P1, the FP64 matrix
// rate needs 15), so the point is bytes in flight.  Staging 32-row tiles in LDS
// with two barriers per tile left one 4 KB tile per workgroup in flight; here each
// of the 8 waves of a workgroup holds its current rows and loads the next ones.
//
// v_mfma_f64_16x16x4f64 (wave64, lane l, i = l % 16, g = l / 16):
//   A (16x4): A[i][g]    B (4x16): B[g][i]    D (16x16), reg r: D[4 r + g][i]
// Two facts make LDS unnecessary:
//   - in a Gram both operands of rows k..k+3 are the same fragment Y[k + g][16 J + i];
//   - the D registers of Z = Y W are themselves such fragments of Z (register r is
//     rows 4 r .. 4 r + 3), so P2's Gram takes them as they are.
// Measured (MI355X) against LDS-staged 32-row tiles: 129 x 200,000 x 30 float32
// (SPOD) P1 1.54 -> 0.91 ms, P2 2.78 -> 1.65 ms, U = Y W 2.47 -> 1.39 ms (4.4 TB/s, a copy
// reaches 4.7); 1M x 64 float64 P1 195 -> 144 us, P2 423 -> 228 us, product 282 -> 194 us;
// 8M x 64 by 64 x 256 float32 (reconstruct) 7.19 -> 4.61 ms (57 TFLOP/s); A^T B of
// 700,001 x 64 and x 48 float32 189 -> 109 us.
//
// Loads are V elements per lane (V = 1, 2, 4 by alignment).  In the Grams the V
// elements go to V column blocks (block c V + e holds the physical columns
// 16 V c + V i + e), undone when the slab is written; in the products they go to V
// k-steps (a sum over k may take its terms in any order) and W is laid out in LDS
// to match.
#include "common.hpp"
#include "f64_common.hpp"
#include "kernels.hpp"
#include <algorithm>

namespace {

constexpr int DNT = 512;        // 8 waves
constexpr int DNW = DNT / 64;
// A row chunk of a Gram over more than 32 columns is a workgroup's of 8 waves, 16 rows
// each per turn, which sum their parts through LDS; up to 32 columns one of 4 waves', or
// a wave's of its own, whose slab is written from registers (chunk_waves).
// So a workgroup has 256 threads up to 32 columns (129 x 200,000 x 30 float32 P1 0.96 ->
// 0.91 ms), but 512 in a P2 of one wave a chunk, where the waves share one copy of W (1.80
// -> 1.65 ms).
constexpr int gram_threads(int NB, int WPC, bool P2) { return NB <= 32 && !(P2 && WPC == 1) ? 256 : DNT; }
// Waves of a chunk over at most 32 columns.  Real ones: 4, since with one a lone problem
// leaves the chip half idle or more (4M x 8 float32 SVD 587 us, with 4 waves 402; P2 of
// 5000 x 32 23 and 12 us).  Complex ones, the blocks of a spectral POD, many in a launch:
// one, its rows summed in ascending order, which fixes the phase that a noise mode's
// vector has (64 of 130,000 x 15 in one launch 2.49 ms, with 4 waves a chunk 2.63).
inline int chunk_waves(bool cplx) { return cplx ? 1 : 4; }

template <class TS, int V>
PC_DEV void load_vec(const TS* p, TS* o) {
  if constexpr (V == 1) {
    o[0] = p[0];
  } else {
    typedef TS vt __attribute__((ext_vector_type(V)));
    const vt q = *reinterpret_cast<const vt*>(p);
#pragma unroll
    for (int e = 0; e < V; e++) o[e] = q[e];
  }
}
template <class TO, int V>
PC_DEV void store_vec(TO* p, const TO* o) {
  if constexpr (V == 1) {
    p[0] = o[0];
  } else {
    typedef TO vt __attribute__((ext_vector_type(V)));
    vt q;
#pragma unroll
    for (int e = 0; e < V; e++) q[e] = o[e];
    *reinterpret_cast<vt*>(p) = q;
  }
}

// Sum the NBLK accumulators of NW waves in wave order through red (NW KB; NW / 4 blocks
// at a time) and hand every entry (block, i, j, value) to `put`.
template <int NBLK, int NW, class Put>
PC_DEV void sum_waves(const d4* acc, double* red, Put put) {
  constexpr int BP = NW / 4;  // blocks whose entries the threads of NW waves are
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
#pragma unroll
  for (int b0 = 0; b0 < NBLK; b0 += BP) {
    __syncthreads();
#pragma unroll
    for (int u = 0; u < BP; u++)
      if (b0 + u < NBLK)
#pragma unroll
        for (int r = 0; r < 4; r++) red[(w * BP + u) * 256 + r * 64 + l] = acc[b0 + u][r];
    __syncthreads();
    const int u = threadIdx.x >> 8, e = threadIdx.x & 255;
    if (b0 + u < NBLK) {
      double s = 0.0;
#pragma unroll
      for (int q = 0; q < NW; q++) s += red[(q * BP + u) * 256 + e];
      put(b0 + u, 4 * (e >> 6) + ((e >> 4) & 3), e & 15, s);
    }
  }
}
constexpr int red_size(int NW) { return NW * (NW / 4) * 256; }  // doubles

// Upper blocks (I, J) of a chunk's Gram to `put`: from registers, or summed over its waves
template <int nb, int WPC, class Put>
PC_DEV void store_gram(const d4* acc, double* red, Put put) {
  constexpr int NBLK = nb * (nb + 1) / 2;
  if constexpr (WPC == 1) {
    const int l = threadIdx.x & 63;
    int b = 0;
#pragma unroll
    for (int I = 0; I < nb; I++)
#pragma unroll
      for (int J = I; J < nb; J++, b++)
#pragma unroll
        for (int r = 0; r < 4; r++) put(I, J, 4 * r + (l >> 4), l & 15, acc[b][r]);
  } else {
    sum_waves<NBLK, WPC>(acc, red, [&](int blk, int pi, int pj, double s) {
      int I = 0, o = 0;
      while (o + nb - I <= blk) o += nb - I++;
      put(I, I + blk - o, pi, pj, s);
    });
  }
}

// fragments of 4 RS rows (RS k-steps) of a row-major operand: v[r][c V + e] is row
// base + 4 r + g, column 16 V c + V i + e.  Rows beyond the range repeat its last
// row, columns beyond n column 0: masked by the caller.
template <class TS, int NBF, int V, int RS>
PC_DEV void load_rows(const TS* __restrict__ X, int64_t ldx, int n, int64_t base, int64_t row1, TS (*v)[NBF]) {
  const int l = threadIdx.x & 63, i = l & 15, g = l >> 4;
#pragma unroll
  for (int r = 0; r < RS; r++) {
    const int64_t row = base + 4 * r + g;
    const TS* xr = X + (row < row1 ? row : row1 - 1) * ldx;
#pragma unroll
    for (int c = 0; c < NBF / V; c++) {
      const int col = 16 * V * c + V * i;
      load_vec<TS, V>(xr + (col < n ? col : 0), &v[r][c * V]);
    }
  }
}

// P1: partial Gram of the (centred) rows of a chunk
template <class TS, int NB, int V, int WPC>
__global__ __launch_bounds__(gram_threads(NB, WPC, false)) void k_dgram_f64(const TS* __restrict__ X, int64_t ldx, int64_t m, int n, int center,
                                                   double* mean_out, double* var_out, int chunks, int64_t rpc,
                                                   double* __restrict__ part, int64_t zx, int64_t zb) {
  X = zoff(X, zx);
  mean_out = zoff(mean_out, zb);
  var_out = zoff(var_out, zb);
  part = zoff(part, zb);
  constexpr int nb = NB / 16, NBLK = nb * (nb + 1) / 2;
  __shared__ double red[WPC > 1 ? red_size(WPC) : 1];
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, i = l & 15, g = l >> 4;
  const int64_t chunk = int64_t(blockIdx.x) * (gram_threads(NB, WPC, false) / 64 / WPC) + w / WPC;
  if (WPC == 1 && chunk >= chunks) return;
  const int64_t row0 = chunk * rpc;
  const int64_t row1 = row0 + rpc < m ? row0 + rpc : m;
  bool cv[nb];
#pragma unroll
  for (int b = 0; b < nb; b++) cv[b] = 16 * V * (b / V) + V * i + b % V < n;
  const double nd = n, inv_n = 1.0 / nd;
  d4 acc[NBLK];
#pragma unroll
  for (int b = 0; b < NBLK; b++) acc[b] = d4{0, 0, 0, 0};
  TS cur[4][nb], nxt[4][nb];
  int64_t t = row0 + 16 * (w % WPC);
  if (t < row1) load_rows<TS, nb, V, 4>(X, ldx, n, t, row1, cur);
  for (; t < row1; t += 16 * WPC) {
    if (t + 16 * WPC < row1) load_rows<TS, nb, V, 4>(X, ldx, n, t + 16 * WPC, row1, nxt);
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int64_t row = t + 4 * r + g;
      const bool rv = row < row1;
      double f[nb];
#pragma unroll
      for (int b = 0; b < nb; b++) f[b] = rv && cv[b] ? double(cur[r][b]) : 0.0;
      if (center) {
        double s = 0.0;
#pragma unroll
        for (int b = 0; b < nb; b++) s += f[b];
        const double mu = div_n(row16_sum(s), nd, inv_n);
#pragma unroll
        for (int b = 0; b < nb; b++) f[b] = rv && cv[b] ? f[b] - mu : 0.0;
        if (center == 2) {
          double s2 = 0.0;
#pragma unroll
          for (int b = 0; b < nb; b++) s2 += f[b] * f[b];
          const double var = div_n(row16_sum(s2), nd, inv_n);
          divide_rows<nb>(f, var);
#pragma unroll
          for (int b = 0; b < nb; b++) f[b] = rv && cv[b] ? f[b] : 0.0;
          if (rv && i == 0) var_out[row] = var;
        }
        if (rv && i == 0) mean_out[row] = mu;
      }
      int b = 0;
#pragma unroll
      for (int I = 0; I < nb; I++)
#pragma unroll
        for (int J = I; J < nb; J++, b++) acc[b] = mfma64(f[I], f[J], acc[b]);
    }
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
      for (int b = 0; b < nb; b++) cur[r][b] = nxt[r][b];
  }
  double* P = part + chunk * NB * NB;
  auto put = [&](int I, int J, int pi, int pj, double s) {
    const int pr = 16 * V * (I / V) + V * pi + I % V, pc = 16 * V * (J / V) + V * pj + J % V;
    if (I == J && pr > pc) return;
    P[int64_t(pr < pc ? pr : pc) * NB + (pr < pc ? pc : pr)] = s;
  };
  store_gram<nb, WPC>(acc, red, put);
}

// A fragments of 16 rows for the products: a[c V + e] is row base + i, column
// 4 V c + V g + e (k-step c V + e)
template <class TS, int KS, int V>
PC_DEV void load_afrag(const TS* __restrict__ X, int64_t ldx, int n, int64_t row, int64_t row1, TS* a) {
  const int g = (threadIdx.x & 63) >> 4;
  const TS* xr = X + (row < row1 ? row : row1 - 1) * ldx;
#pragma unroll
  for (int c = 0; c < KS / V; c++) {
    const int col = 4 * V * c + V * g;
    if (4 * V * c < n) load_vec<TS, V>(xr + (col < n ? col : 0), a + c * V);  // uniform: whole k-steps beyond n stay out
  }
}
// their values: centred, zero beyond the rows and columns
template <class TS, int KS, int V>
PC_DEV void afrag_values(const TS* x, double* a, int n, bool rv, int center, double mu, double var) {
  const int g = (threadIdx.x & 63) >> 4;
#pragma unroll
  for (int st = 0; st < KS; st++) a[st] = center ? double(x[st]) - mu : double(x[st]);
  if (center == 2) divide_rows<KS>(a, var);
#pragma unroll
  for (int st = 0; st < KS; st++) a[st] = rv && 4 * V * (st / V) + V * g + st % V < n ? a[st] : 0.0;
}
// W (ld ldw) into LDS in B-fragment order: Wl[(st nbl + J) 64 + l] is row
// 4 V (st / V) + V g + st % V, column col0 + colmap(J, i); zero beyond n rows / ldw columns
template <int NTHR, int KS, int NBL, int V, class Map>
PC_DEV void stage_w(const double* __restrict__ W, int n, int ldw, int col0, double* Wl, Map colmap) {
  constexpr int ALL = KS * NBL * 64, U = ALL / NTHR < 16 ? (ALL + NTHR - 1) / NTHR : 16;
  for (int i0 = threadIdx.x; i0 < ALL; i0 += U * NTHR) {
    double v[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int idx = i0 + u * NTHR, lane = idx & 63, sj = idx >> 6, st = sj / NBL, J = sj - st * NBL;
      const int k = 4 * V * (st / V) + V * (lane >> 4) + st % V, col = col0 + colmap(J, lane & 15);
      const bool in = idx < ALL && k < n && col < ldw;
      v[u] = W[in ? int64_t(k) * ldw + col : 0];
      v[u] = in ? v[u] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < U; u++)
      if (ALL % (U * NTHR) == 0 || i0 + u * NTHR < ALL) Wl[i0 + u * NTHR] = v[u];
  }
}

// P2: Z = Yc W in registers, then its Gram.  W is upper triangular: column block J
// takes the k-steps below 16 (J + 1) only (the rest are exact zeros).
template <class TS, int NB, int V, int WPC>
__global__ __launch_bounds__(gram_threads(NB, WPC, true)) void k_dzgram_f64(const TS* __restrict__ X, int64_t ldx, int64_t m, int n, int center,
                                                    const double* mean_in, const double* var_in,
                                                    const double* __restrict__ W, int chunks, int64_t rpc,
                                                    double* __restrict__ part, int64_t zx, int64_t zb) {
  X = zoff(X, zx);
  mean_in = zoff(mean_in, zb);
  var_in = zoff(var_in, zb);
  W = zoff(W, zb);
  part = zoff(part, zb);
  constexpr int nb = NB / 16, NBLK = nb * (nb + 1) / 2, KS = NB / 4;
  constexpr int WL = KS * nb * 64, RL = WPC > 1 ? red_size(WPC) : 1;
  __shared__ double sm[WL > RL ? WL : RL];  // W fragments, then the waves' partial Grams
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, i = l & 15;
  stage_w<gram_threads(NB, WPC, true), KS, nb, V>(W, n, NB, 0, sm, [](int J, int j) { return 16 * J + j; });
  const int64_t chunk = int64_t(blockIdx.x) * (gram_threads(NB, WPC, true) / 64 / WPC) + w / WPC;
  const int64_t row0 = chunk * rpc;
  const int64_t row1 = WPC == 1 && chunk >= chunks ? row0 : row0 + rpc < m ? row0 + rpc : m;
  d4 acc[NBLK];
#pragma unroll
  for (int b = 0; b < NBLK; b++) acc[b] = d4{0, 0, 0, 0};
  TS cur[KS] = {}, nxt[KS] = {};
  double mu = 0.0, var = 1.0, mu_n = 0.0, var_n = 1.0;
  auto load = [&](int64_t t, TS* a, double& mu_, double& var_) {
    const int64_t row = t + i, rc = row < row1 ? row : row1 - 1;
    load_afrag<TS, KS, V>(X, ldx, n, row, row1, a);
    if (center) mu_ = mean_in[rc];
    if (center == 2) var_ = var_in[rc];
  };
  int64_t t = row0 + 16 * (w % WPC);
  if (t < row1) load(t, cur, mu, var);
  __syncthreads();
  for (; t < row1; t += 16 * WPC) {
    if (t + 16 * WPC < row1) load(t + 16 * WPC, nxt, mu_n, var_n);
    const bool rv = t + i < row1;
    asm volatile("" ::: "memory");  // keep W's fragments in LDS: hoisted into registers they spill
    d4 z[nb];
#pragma unroll
    for (int J = 0; J < nb; J++) z[J] = d4{0, 0, 0, 0};
    double a[KS];
    afrag_values<TS, KS, V>(cur, a, n, rv, center, mu, var);
#pragma unroll
    for (int st = 0; st < KS; st++) {
#pragma unroll
      for (int J = 0; J < nb; J++)
        if (4 * V * (st / V) < 16 * (J + 1)) z[J] = mfma64(a[st], sm[(st * nb + J) * 64 + l], z[J]);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
      int b = 0;
#pragma unroll
      for (int I = 0; I < nb; I++)
#pragma unroll
        for (int J = I; J < nb; J++, b++) acc[b] = mfma64(z[I][r], z[J][r], acc[b]);
    }
#pragma unroll
    for (int st = 0; st < KS; st++) cur[st] = nxt[st];
    mu = mu_n;
    var = var_n;
  }
  if (WPC == 1 && chunk >= chunks) return;
  double* P = part + chunk * NB * NB;
  store_gram<nb, WPC>(acc, sm, [&](int I, int J, int pi, int pj, double s) {
    if (I == J && pi > pj) return;
    P[int64_t(16 * I + pi) * NB + 16 * J + pj] = s;
  });
}

// C = Yc W, W (KB x ldw, at most 128 KB of it per column slice) resident in LDS.
// A wave takes R 16-row blocks per turn, every k in registers, and writes CV
// consecutive columns per lane.  blockIdx.y: column slice of NCB.
template <class TS, class TO, int KB, int NCB, int V, int CV>
__global__ __launch_bounds__(DNT) void k_dgemm_f64(const TS* __restrict__ X, int64_t ldx, int64_t m, int n, int center,
                                                   const double* mean_in, const double* var_in,
                                                   const double* __restrict__ W, int ldw, int nc,
                                                   TO* __restrict__ C, int64_t ldc, int64_t zx, int64_t zb,
                                                   int64_t zc) {
  X = zoff(X, zx);
  mean_in = zoff(mean_in, zb);
  var_in = zoff(var_in, zb);
  W = zoff(W, zb);
  C = zoff(C, zc);
  constexpr int KS = KB / 4, nbl = NCB / 16, R = KB > 64 ? 1 : 2;
  __shared__ double Wl[KS * nbl * 64];
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, i = l & 15, g = l >> 4;
  const int col0 = blockIdx.y * NCB;
  const int64_t step = int64_t(gridDim.x) * DNW * 16 * R;
  TS cur[R][KS] = {}, nxt[R][KS] = {};
  double mu[R] = {}, var[R], mu_n[R] = {}, var_n[R];
#pragma unroll
  for (int q = 0; q < R; q++) var[q] = var_n[q] = 1.0;
  auto load = [&](int64_t t, int n_, TS (*a)[KS], double* mu_, double* var_) {
#pragma unroll
    for (int q = 0; q < R; q++) {
      const int64_t row = t + 16 * q + i, rc = row < m ? row : m - 1;
      load_afrag<TS, KS, V>(X, ldx, n_, row, m, a[q]);
      if (center) mu_[q] = mean_in[rc];
      if (center == 2) var_[q] = var_in[rc];
    }
  };
  int64_t t = (int64_t(blockIdx.x) * DNW + w) * 16 * R;
  if (t < m) load(t, n, cur, mu, var);
  stage_w<DNT, KS, nbl, V>(W, n, ldw, col0, Wl, [](int J, int j) { return 16 * CV * (J / CV) + CV * j + J % CV; });
  __syncthreads();
  for (; t < m; t += step) {
    // n anew each turn: the columns' clamps and masks, kept over the loop, spilled registers
    int nn = n;
    asm volatile("" : "+s"(nn));
    if (t + step < m) load(t + step, nn, nxt, mu_n, var_n);
    double a[R][KS];
#pragma unroll
    for (int q = 0; q < R; q++)
      afrag_values<TS, KS, V>(cur[q], a[q], nn, t + 16 * q + i < m, center, mu[q], var[q]);
#pragma unroll 1
    for (int q0 = 0; q0 < nbl / CV; q0++) {
      if (col0 + 16 * CV * q0 >= nc) break;
      d4 z[R][CV];
#pragma unroll
      for (int q = 0; q < R; q++)
#pragma unroll
        for (int u = 0; u < CV; u++) z[q][u] = d4{0, 0, 0, 0};
      // X k-steps at a time, beyond 32 inputs their fragments read while the X before are
      // multiplied.  A branch round each step left every product waiting for its read:
      // 500,000 x 128 by 128 x 128 float64 391 -> 315 us.  Up to 16, where a step is a quarter
      // of the products and more, the steps beyond n stay out one load's width at a time
      // (250,000 x 3 by 3 x 64 float32 21 us in fours, 16 so)
      constexpr int AHEAD = KB > 32 ? 1 : 0, XM = CV == 4 ? 2 : 4, X = KB > 16 || V > XM ? XM : V;
      const double* wq = Wl + q0 * CV * 64 + l;
      double b[1 + AHEAD][X][CV];
      auto read = [&](int c) {
#pragma unroll
        for (int x = 0; x < X; x++)
#pragma unroll
          for (int u = 0; u < CV; u++) b[c & AHEAD][x][u] = wq[((X * c + x) * nbl + u) * 64];
      };
      if (AHEAD) read(0);
#pragma unroll
      for (int c = 0; c < KS / X; c++)
        if (4 * V * (X * c / V) < n) {
          if (!AHEAD || c + 1 < KS / X) read(c + AHEAD);
#pragma unroll
          for (int x = 0; x < X; x++)
#pragma unroll
            for (int u = 0; u < CV; u++)
#pragma unroll
              for (int q = 0; q < R; q++) z[q][u] = mfma64(a[q][X * c + x], b[c & AHEAD][x][u], z[q][u]);
        }
      const int col = col0 + 16 * CV * q0 + CV * i;
#pragma unroll
      for (int q = 0; q < R; q++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int64_t row = t + 16 * q + 4 * r + g;
          TO o[CV];
#pragma unroll
          for (int u = 0; u < CV; u++) o[u] = TO(z[q][u][r]);
          if (row < m && col < nc) store_vec<TO, CV>(C + row * ldc + col, o);
        }
    }
#pragma unroll
    for (int q = 0; q < R; q++) {
#pragma unroll
      for (int st = 0; st < KS; st++) cur[q][st] = nxt[q][st];
      mu[q] = mu_n[q];
      var[q] = var_n[q];
    }
  }
}

// cross product of a chunk's rows: A^T B, both at most 64 columns
template <class TS, int PB, int QB, int V>
__global__ __launch_bounds__(DNT) void k_dxgram_f64(const TS* __restrict__ A, int64_t lda, int p,
                                                    const TS* __restrict__ B, int64_t ldb, int q, int64_t m,
                                                    int64_t rpc, double* __restrict__ part) {
  constexpr int pb = PB / 16, qb = QB / 16, NBLK = pb * qb;
  // k-steps per turn: current and next rows beside the accumulators in 256 registers
  constexpr int RS = (pb + qb) * int(sizeof(TS)) * 2 + NBLK * 8 > 200 ? 2 : 4;
  constexpr int unit = DNW * 4 * RS;
  __shared__ double red[red_size(DNW)];
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, i = l & 15, g = l >> 4;
  const int64_t row0 = int64_t(blockIdx.x) * rpc;
  const int64_t row1 = row0 + rpc < m ? row0 + rpc : m;
  bool ca[pb], cb[qb];
#pragma unroll
  for (int b = 0; b < pb; b++) ca[b] = 16 * V * (b / V) + V * i + b % V < p;
#pragma unroll
  for (int b = 0; b < qb; b++) cb[b] = 16 * V * (b / V) + V * i + b % V < q;
  d4 acc[NBLK];
#pragma unroll
  for (int b = 0; b < NBLK; b++) acc[b] = d4{0, 0, 0, 0};
  TS xa[RS][pb], xb[RS][qb], na[RS][pb], nq[RS][qb];
  int64_t t = row0 + 4 * RS * w;
  if (t < row1) {
    load_rows<TS, pb, V, RS>(A, lda, p, t, row1, xa);
    load_rows<TS, qb, V, RS>(B, ldb, q, t, row1, xb);
  }
  for (; t < row1; t += unit) {
    if (t + unit < row1) {
      load_rows<TS, pb, V, RS>(A, lda, p, t + unit, row1, na);
      load_rows<TS, qb, V, RS>(B, ldb, q, t + unit, row1, nq);
    }
#pragma unroll
    for (int r = 0; r < RS; r++) {
      const bool rv = t + 4 * r + g < row1;
      double fa[pb], fb[qb];
#pragma unroll
      for (int b = 0; b < pb; b++) fa[b] = rv && ca[b] ? double(xa[r][b]) : 0.0;
#pragma unroll
      for (int b = 0; b < qb; b++) fb[b] = rv && cb[b] ? double(xb[r][b]) : 0.0;
#pragma unroll
      for (int I = 0; I < pb; I++)
#pragma unroll
        for (int J = 0; J < qb; J++) acc[I * qb + J] = mfma64(fa[I], fb[J], acc[I * qb + J]);
    }
#pragma unroll
    for (int r = 0; r < RS; r++) {
#pragma unroll
      for (int b = 0; b < pb; b++) xa[r][b] = na[r][b];
#pragma unroll
      for (int b = 0; b < qb; b++) xb[r][b] = nq[r][b];
    }
  }
  double* P = part + int64_t(blockIdx.x) * PB * QB;
  sum_waves<NBLK, DNW>(acc, red, [&](int blk, int pi, int pj, double s) {
    const int I = blk / qb, J = blk - I * qb;
    P[int64_t(16 * V * (I / V) + V * pi + I % V) * QB + 16 * V * (J / V) + V * pj + J % V] = s;
  });
}

template <int N> using Int = std::integral_constant<int, N>;

template <class F>
int with_nb(int n, F&& f) {
  if (n <= 16) return f(Int<16>{});
  if (n <= 32) return f(Int<32>{});
  if (n <= 48) return f(Int<48>{});
  if (n <= 64) return f(Int<64>{});
  return -1;
}

// widest vector (4, 2, 1 elements, at most 16 bytes) that n columns, the leading
// dimension and the base address allow; max: the caller's limit
template <class TS>
int vec_width(const void* p, int64_t ld, int64_t n, int64_t zstride, int max) {
  for (int v = int(16 / sizeof(TS)); v > 1; v /= 2)
    if (v <= max && n % v == 0 && ld % v == 0 && reinterpret_cast<uintptr_t>(p) % (v * sizeof(TS)) == 0 &&
        zstride % int64_t(v * sizeof(TS)) == 0)
      return v;
  return 1;
}
template <class TS, class F>
int with_vec(int v, F&& f) {
  if constexpr (sizeof(TS) == 4)
    if (v >= 4) return f(Int<4>{});
  if (v >= 2) return f(Int<2>{});
  return f(Int<1>{});
}

// K class, and row turns of the direct product over n inputs
int gemm_k(int n) { return n <= 16 ? 16 : n <= 32 ? 32 : n <= 64 ? 64 : 128; }
int64_t gemm_turns(int64_t m, int n) { return ceil_div(m, DNW * (n > 64 ? 16 : 32)); }
// Workgroups per slice of s columns, one per CU: all slices side by side, or one after the
// other where that is less work for the CU with the most of it (a last slice of few
// columns leaves its workgroups idle beside the others).
int64_t gemm_workgroups(int64_t turns, int nc, int s) {
  const int64_t shared = std::max<int64_t>(1, 256 / ceil_div(nc, s));
  return ceil_div(turns, 256) * nc < ceil_div(turns, shared) * s ? 256 : shared;
}
// Columns of W that a workgroup keeps in LDS: a power of two, at most 128 KB of it.  X is
// read once per slice, and a slice writes only a part of each row, so a tall product takes
// the widest (1.5M x 5 by 5 x 41 float64 in halves 285 us, whole 152); one of few rows (nz
// problems together) takes the narrowest of which every CU holds a workgroup at once
// (1024 x 128 by 128 x 256 float64: 16 workgroups of 128 columns 44 us, 256 of 16 columns
// 20, where the call's launch is what is left; 5000 rows: 36 us with 128, 23 with 64, 30
// with 32, which take two rounds).
int gemm_slice(int64_t m, int n, int nc, int nz) {
  const int64_t turns = gemm_turns(m, n) * nz;
  int most = n > 64 ? 128 : 256;
  while (most > 16 && most / 2 >= nc) most /= 2;
  auto slices = [&](int s) { return ceil_div(nc, s); };
  if (turns * slices(most) > 256) {
    if (n <= 32) return most;
    // several turns each, beyond 32 inputs, where the matrix units bound them: half as
    // many columns where that shortens the longest workgroup's work by a fifth and X, read
    // once per slice, stays in the caches
    auto work = [&](int s) { return ceil_div(turns, gemm_workgroups(turns, nc, s)) * s; };
    const int half = most / 2;
    return half >= 16 && 5 * work(half) <= 4 * work(most) && slices(half) * m * n * 8 <= (int64_t(128) << 20) ? half : most;
  }
  while (most > 16 && turns * slices(most / 2) <= 256) most /= 2;
  return most;
}

template <class TS>
int dgram_t(hipStream_t st, const TS* X, int64_t ldx, int64_t m, int n, int center, const double* mean_in,
            const double* var_in, double* mean_out, double* var_out, const double* W, int chunks, int64_t tpc,
            double* part, const PassBatch& bz) {
  const int wpc = n > 32 ? DNW : chunk_waves(bz.cplx);
  const int64_t rpc = tpc * 32 * (wpc == 1 ? 1 : 4);
  return with_nb(n, [&](auto nbc) {
    constexpr int NB = decltype(nbc)::value;
    // the Gram's V column blocks have to exist: 48 columns are three blocks; up to 32
    // columns Z's k-steps stay in ascending order
    const int vmax = W ? (NB <= 32 ? 1 : 4) : NB == 64 ? 4 : NB == 32 ? 2 : 1;
    return with_vec<TS>(vec_width<TS>(X, ldx, n, bz.zx, vmax), [&](auto vc) {
      constexpr int V = decltype(vc)::value;
      auto go = [&](auto wc) {
        constexpr int WPC = decltype(wc)::value, N1 = gram_threads(NB, WPC, false), N2 = gram_threads(NB, WPC, true);
        const dim3 g(unsigned(ceil_div(chunks, (W ? N2 : N1) / 64 / WPC)), 1, unsigned(bz.nz));
        if (W) {
          if constexpr (NB > 32 || V == 1)
            hipLaunchKernelGGL((k_dzgram_f64<TS, NB, V, WPC>), g, dim3(N2), 0, st, X, ldx, m, n, center, mean_in,
                               var_in, W, chunks, rpc, part, bz.zx, bz.zb);
        } else {
          if constexpr ((NB / 16) % V == 0)
            hipLaunchKernelGGL((k_dgram_f64<TS, NB, V, WPC>), g, dim3(N1), 0, st, X, ldx, m, n, center, mean_out,
                               var_out, chunks, rpc, part, bz.zx, bz.zb);
        }
      };
      if constexpr (NB > 32) go(Int<DNW>{});
      else if (wpc == 1) go(Int<1>{});
      else go(Int<4>{});
      return 0;
    });
  });
}

// Unused LDS that keeps a direct product of up to 32 inputs alone on its CU: where C is
// beyond the 256 MB cache and its rows, of more than a line, begin inside lines, a line that
// two rows share is written to HBM twice unless the waves in flight are few (1.5M x 8 by
// 8 x 41 float64 203 us with two workgroups a CU, 145 with one; by 8 x 60 268 and 228;
// 700,000 x 8 by 8 x 41, C of 230 MB, 76 and 76).  Shorter rows, and rows of whole lines,
// take the waves (4M x 8 by 8 x 20 float32 with one 1.3 times as long).
inline size_t alone_lds(int kb, size_t wl, int64_t rows, int nc, int64_t ldc, size_t size) {
  const int64_t pitch = ldc * int64_t(size);
  const bool split = kb <= 32 && pitch > 128 && pitch % 128 != 0 && rows * nc * int64_t(size) > (int64_t(256) << 20);
  return split && wl < 84 * 1024 ? 84 * 1024 - wl : 0;
}
template <class TS, class TO>
int dgemm_t(hipStream_t st, const TS* X, int64_t ldx, int64_t m, int n, int center, const double* mean_in,
            const double* var_in, const double* W, int ldw, int nc, int chunks, TO* C, int64_t ldc,
            const PassBatch& bz) {
  const int vx = vec_width<TS>(X, ldx, n, bz.zx, 4), vc = vec_width<TO>(C, ldc, nc, bz.zc, 4);
  auto go = [&](auto kc, auto ncc) {
    constexpr int KB = decltype(kc)::value, NCB = decltype(ncc)::value;
    return with_vec<TS>(vx, [&](auto v_) {
      return with_vec<TO>(NCB / 16 < vc ? NCB / 16 : vc, [&](auto c_) {
        constexpr int V = decltype(v_)::value, CV = decltype(c_)::value;
        const size_t pad = alone_lds(KB, size_t(KB) * NCB * sizeof(double), m * bz.nz, nc, ldc, sizeof(TO));
        if constexpr ((NCB / 16) % CV == 0)
          hipLaunchKernelGGL((k_dgemm_f64<TS, TO, KB, NCB, V, CV>),
                             dim3(unsigned(chunks), unsigned(ceil_div(nc, NCB)), unsigned(bz.nz)), dim3(DNT), pad, st, X,
                             ldx, m, n, center, mean_in, var_in, W, ldw, nc, C, ldc, bz.zx, bz.zb, bz.zc);
        return 0;
      });
    });
  };
  auto cols = [&](auto kc) {
    constexpr int KB = decltype(kc)::value;
    const int slice = gemm_slice(m, n, nc, bz.nz);
    if (slice == 16) return go(kc, Int<16>{});
    if (slice == 32) return go(kc, Int<32>{});
    if (slice == 64) return go(kc, Int<64>{});
    if (slice == 128) return go(kc, Int<128>{});
    if constexpr (KB <= 64) return go(kc, Int<256>{});
    return -1;
  };
  if (n <= 16) return cols(Int<16>{});
  if (n <= 32) return cols(Int<32>{});
  if (n <= 64) return cols(Int<64>{});
  if (n <= 128) return cols(Int<128>{});
  return -1;
}

template <class TS>
int dxgram_t(hipStream_t st, const TS* A, int64_t lda, int p, const TS* B, int64_t ldb, int q, int64_t m, int chunks,
             int64_t tpc, double* part) {
  return with_nb(p, [&](auto pc_) {
    return with_nb(q, [&](auto qc_) {
      constexpr int PB = decltype(pc_)::value, QB = decltype(qc_)::value;
      constexpr int VM = PB == 64 && QB == 64 ? 4 : PB % 32 == 0 && QB % 32 == 0 ? 2 : 1;
      const int va = vec_width<TS>(A, lda, p, 0, VM), vb = vec_width<TS>(B, ldb, q, 0, VM);
      return with_vec<TS>(va < vb ? va : vb, [&](auto vc) {
        constexpr int V = decltype(vc)::value;
        if constexpr (V <= VM)
          hipLaunchKernelGGL((k_dxgram_f64<TS, PB, QB, V>), dim3(unsigned(chunks)), dim3(DNT), 0, st, A, lda, p, B,
                             ldb, q, m, tpc * 128, part);
        return 0;
      });
    });
  });
}

}  // namespace

// Row chunks of the direct Grams (at least one: of no rows it writes zeros), from m and the
// columns alone; *tpc: turns of 128 rows, or of 32 where a chunk is one wave's.  At most
// 1024 up to 32 columns and 512 (two workgroups per CU) beyond, where a slab is 32 KB to
// write and sum.  Few rows: as few turns as that gives (P2 of 5000 x 64 with two turns a
// chunk 17 us, with one 11), for complex columns at least 128 and 256 rows a chunk.
int d64_gram_chunks(int64_t m, int n, bool cplx, int64_t* tpc) {
  int64_t tiles, per;
  if (n <= 32 && chunk_waves(cplx) == 1) {
    tiles = ceil_div(m, 32);
    per = ceil_div(tiles, stream_chunks(m, 32));
  } else {
    tiles = ceil_div(m, 128);
    per = std::max<int64_t>(cplx ? 2 : 1, ceil_div(tiles, n <= 32 ? 1024 : 512));
  }
  *tpc = per;
  return tiles < 1 ? 1 : int(ceil_div(tiles, per));
}
// Workgroups of the direct product per column slice, no more than there are turns of work.
// One per CU in all beyond 32 inputs, whose rows fill its registers: with more, waiting
// for a CU, each took one or two turns with nothing loaded ahead and staged W for them
// (250,000 x 64 by 64 x 64 float64: 977 workgroups 76 us, 256 workgroups 60).  Up to 32
// inputs HBM bounds the pass, and as many as W's LDS allows keep more bytes in flight
// (4M x 8 by 8 x 8: 137 us with one per CU, 107 with four), beyond 16 while each has four
// turns (250,000 x 30 by 30 x 30: 33 us with one turn each, 27 with four).
int d64_gemm_chunks(int64_t m, int n, int nc) {
  const int64_t turns = gemm_turns(m, n);
  const int slice = gemm_slice(m, n, nc, 1);
  int64_t want = gemm_workgroups(turns, nc, slice);
  if (n <= 32) {
    const int64_t lds = int64_t(gemm_k(n)) * 8 * slice, fit = lds > 40 * 1024 ? 2 : 4;
    const int64_t all = n <= 16 ? 256 * fit : std::min(256 * fit, std::max<int64_t>(256, ceil_div(turns, 4)));
    want = std::max<int64_t>(1, all / ceil_div(nc, slice));
  }
  return turns < 1 ? 1 : int(std::min(turns, want));
}

// row chunks of the direct cross products, turns of 128 rows
int d64_xgram_chunks(int64_t m, int64_t* tpc) { return d64_gram_chunks(m, kDirectGram, false, tpc); }

int launch_d64_gram(hipStream_t st, pc_dtype dt, const void* X, int64_t ldx, int64_t m, int n, int center,
                    const double* mean_in, const double* var_in, double* mean_out, double* var_out, const double* W,
                    int chunks, int64_t tpc, double* part, const PassBatch& bz) {
  if (dt == PC_F64)
    return dgram_t<double>(st, (const double*)X, ldx, m, n, center, mean_in, var_in, mean_out, var_out, W, chunks, tpc,
                           part, bz);
  return dgram_t<float>(st, (const float*)X, ldx, m, n, center, mean_in, var_in, mean_out, var_out, W, chunks, tpc,
                        part, bz);
}
int launch_d64_gemm(hipStream_t st, pc_dtype dt, const void* X, int64_t ldx, int64_t m, int n, int center,
                    const double* mean_in, const double* var_in, const double* W, int ldw, int nc, int chunks, void* C,
                    int64_t ldc, const PassBatch& bz) {
  if (dt == PC_F64)
    return dgemm_t<double, double>(st, (const double*)X, ldx, m, n, center, mean_in, var_in, W, ldw, nc, chunks,
                                   (double*)C, ldc, bz);
  return dgemm_t<float, float>(st, (const float*)X, ldx, m, n, center, mean_in, var_in, W, ldw, nc, chunks, (float*)C,
                               ldc, bz);
}
int launch_d64_xgram(hipStream_t st, pc_dtype dt, const void* A, int64_t lda, int p, const void* B, int64_t ldb, int q,
                     int64_t m, int chunks, int64_t tpc, double* part) {
  if (dt == PC_F64)
    return dxgram_t<double>(st, (const double*)A, lda, p, (const double*)B, ldb, q, m, chunks, tpc, part);
  return dxgram_t<float>(st, (const float*)A, lda, p, (const float*)B, ldb, q, m, chunks, tpc, part);
}
