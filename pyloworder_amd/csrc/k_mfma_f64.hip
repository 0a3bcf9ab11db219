// FP64 MFMA streaming kernels (v_mfma_f64_16x16x4f64) for operands wider than
// k_direct_f64.hip takes: Grams of 65 to 256 columns, products over more than 128
// inputs (any number of them).
//
// A pass over the tall matrix A (m x n, row-major) is split over workgroups: the Grams
// into `chunks` contiguous row ranges, 8 waves each (one partial NB x NB slab per
// chunk, summed in a fixed order afterwards, so results never depend on scheduling),
// the product into 32-row tiles dealt in turn.
//   gram  : the upper 16x16 blocks of Y^T Y in registers,
//   zgram : Z = Y W (W n x n upper triangular, FP64, from L2) into LDS, then Z^T Z,
//   gemm  : C = Y W (W K x nc from L2),
//   xgram : A^T B for two tall operands (projection, sketches).
//
// The FP64 matrix rate bounds all of them (256 columns: 32 flop / B in a Gram, the
// rate needs 15), so what matters is that no SIMD waits: rows arrive in registers
// while the previous tile is multiplied (RowStage), barriers leave global loads in
// flight, W of the next 16 k-steps is loaded before the products of the current ones,
// and NB comes in steps of 32 columns, not in powers of two.
// Measured (MI355X; a large library product reaches 72.6 TFLOP/s): 8M x 256 float64
// P1 11.3 -> 10.4 ms, P2 23.4 -> 23.0 (its 256-column form has 160 bytes a lane in
// scratch), U = Y W 20.8 -> 20.2 (52 TFLOP/s).  Counters: the matrix units are busy in 62
// to 70 % of the cycles, which run at 2.1 to 2.4 GHz;
// 400,003 x 151 float32 (160 columns instead of 256) P1 0.77 -> 0.26, P2 1.53 -> 0.53,
// U 1.07 -> 0.55 ms; 1M x 512 float32 Z 13.8 -> 6.6 (its zero blocks skipped), U 13.9 ->
// 9.9 ms.
#include "common.hpp"
#include "f64_common.hpp"
#include "kernels.hpp"

namespace {

constexpr int TR = 32;       // rows per tile
constexpr int NTH = 512;     // threads per workgroup
// rows from which a product takes 64-row tiles: eight of them for each CU
constexpr int64_t kTallProduct = 1 << 17;
constexpr int NWV = NTH / 64;
constexpr int PADD = 2;      // LDS row padding (doubles): rows 4 banks apart

// Accumulate the Gram of the tile S (TR rows of LD doubles) into the wave's slots: its
// upper blocks are SL consecutive ones of the row-major triangle from (I, J) on, so
// the left operand is read once per run of equal I.  A slot's 8 k-steps are read
// before its products; the SIMD's other wave multiplies meanwhile.
template <int LD, int SL>
PC_DEV void gram_tile(const double* S, int I, int J, int nslot, int nb, d4* acc) {
  const int l = threadIdx.x & 63, kr = l >> 4, cc = l & 15;
  const double* base = S + kr * LD + cc;
  double a[TR / 4];
  int cur = -1;
#pragma unroll
  for (int s = 0; s < SL; s++) {
    if (s < nslot) {
      if (I != cur) {
#pragma unroll
        for (int kk = 0; kk < TR / 4; kk++) a[kk] = base[4 * kk * LD + 16 * I];
        cur = I;
      }
      double b[TR / 4];
#pragma unroll
      for (int kk = 0; kk < TR / 4; kk++) b[kk] = base[4 * kk * LD + 16 * J];
#pragma unroll
      for (int kk = 0; kk < TR / 4; kk++) acc[s] = mfma64(a[kk], b[kk], acc[s]);
      if (++J == nb) J = ++I;
    }
  }
}
// first slot (I, J) of the wave and its count, the NBLK upper blocks dealt evenly
template <int NB>
PC_DEV void wave_blocks(int& I, int& J, int& cnt) {
  constexpr int nb = NB / 16, NBLK = nb * (nb + 1) / 2;
  const int w = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  int b = NBLK * w / NWV;
  cnt = NBLK * (w + 1) / NWV - b;
  I = 0;
  while (b >= nb - I) b -= nb - I++;
  J = I + b;
}
template <int NB, int SL>
PC_DEV void store_blocks(const d4* acc, int I, int J, int cnt, double* P) {
  const int l = threadIdx.x & 63, kr = l >> 4, cc = l & 15;
#pragma unroll
  for (int s = 0; s < SL; s++) {
    if (s < cnt) {
#pragma unroll
      for (int r = 0; r < 4; r++) P[int64_t(I * 16 + 4 * r + kr) * NB + J * 16 + cc] = acc[s][r];
      if (++J == NB / 16) J = ++I;
    }
  }
}
constexpr int gram_slots(int NB) { return ((NB / 16) * (NB / 16 + 1) / 2 + NWV - 1) / NWV; }

// P1: two LDS tiles, one barrier per tile
template <class TS, int NB, bool VAR>
__global__ __launch_bounds__(NTH) void k_gram_f64(const TS* __restrict__ X, int64_t ldx, int64_t m, int n, int center,
                                                  double* mean_out, double* var_out, int64_t tiles_per_chunk,
                                                  double* __restrict__ part, int64_t zx, int64_t zb) {
  X = zoff(X, zx);
  mean_out = zoff(mean_out, zb);
  var_out = zoff(var_out, zb);
  part = zoff(part, zb);
  constexpr int SL = gram_slots(NB), LD = NB + PADD;
  __shared__ double S[2][TR * LD];
  int I, J, cnt;
  wave_blocks<NB>(I, J, cnt);
  d4 acc[SL];
#pragma unroll
  for (int s = 0; s < SL; s++) acc[s] = d4{0, 0, 0, 0};
  const int64_t ntiles = ceil_div(m, TR);
  const int64_t t0 = int64_t(blockIdx.x) * tiles_per_chunk;
  const int64_t t1 = t0 + tiles_per_chunk < ntiles ? t0 + tiles_per_chunk : ntiles;
  RowStage<TS, TR, NB, VAR> st;
  auto fetch = [&](int64_t t) {
    st.fetch(X, ldx, m, n, (t < t1 ? t : t1 - 1) * TR, 0, 0, nullptr, nullptr);
  };
  auto put = [&](int64_t t) {
    st.template put<LD>(S[(t - t0) & 1], 0, m, n, t * TR, 0, center, true, mean_out, var_out);
  };
  fetch(t0);
  put(t0);
  fetch(t0 + 1);
  lds_barrier();
  for (int64_t t = t0; t < t1; t++) {
    gram_tile<LD, SL>(S[(t - t0) & 1], I, J, cnt, NB / 16, acc);
    if (t + 1 < t1) {
      put(t + 1);
      fetch(t + 2);
    }
    lds_barrier();
  }
  store_blocks<NB, SL>(acc, I, J, cnt, part + int64_t(blockIdx.x) * NB * NB);
}

// Column blocks of Z for a wave, at most two (a < b, -1: none), each with both 16-row
// blocks.  Block J takes J + 1 of W's 16-row blocks (W is upper triangular), so the
// blocks are dealt to the four SIMDs largest first and back and forth; waves 2 k and
// 2 k + 1 share a SIMD, the first takes its 1st and 4th block, the other the 2nd and 3rd.
template <int NB>
PC_DEV void wave_zblocks(int& a, int& b) {
  constexpr int nb = NB / 16;
  const int w = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)), k = w >> 1;
  auto nth = [&](int q) {  // q-th block of SIMD k
    const int J = nb - 1 - (4 * q + ((q & 1) ? 3 - k : k));
    return J >= 0 ? J : -1;
  };
  b = nth(w & 1 ? 1 : 0);
  a = nth(w & 1 ? 2 : 3);
}

// P2: Z = Yc W into LDS, then its Gram
template <class TS, int NB, bool VAR>
__global__ __launch_bounds__(NTH) void k_zgram_f64(const TS* __restrict__ X, int64_t ldx, int64_t m, int n, int center,
                                                   const double* mean_in, const double* var_in,
                                                   const double* __restrict__ W, int64_t tiles_per_chunk,
                                                   double* __restrict__ part, int64_t zx, int64_t zb) {
  X = zoff(X, zx);
  mean_in = zoff(mean_in, zb);
  var_in = zoff(var_in, zb);
  W = zoff(W, zb);
  part = zoff(part, zb);
  constexpr int SL = gram_slots(NB), LD = NB + PADD;
  __shared__ double S[TR * LD], Zs[TR * LD];
  const int l = threadIdx.x & 63, kr = l >> 4, cc = l & 15;
  int I, J, cnt, Ja, Jb;
  wave_blocks<NB>(I, J, cnt);
  wave_zblocks<NB>(Ja, Jb);
  d4 acc[SL];
#pragma unroll
  for (int s = 0; s < SL; s++) acc[s] = d4{0, 0, 0, 0};
  const int64_t ntiles = ceil_div(m, TR);
  const int64_t t0 = int64_t(blockIdx.x) * tiles_per_chunk;
  const int64_t t1 = t0 + tiles_per_chunk < ntiles ? t0 + tiles_per_chunk : ntiles;
  RowStage<TS, TR, NB, VAR> st;
  auto fetch = [&](int64_t t) {
    st.fetch(X, ldx, m, n, (t < t1 ? t : t1 - 1) * TR, 0, center, mean_in, var_in);
  };
  auto put = [&](int64_t t) { st.template put<LD>(S, 0, m, n, t * TR, 0, center, false, nullptr, nullptr); };
  const double* wl = W + int64_t(kr) * NB + cc;
  // W rows 16 kb .. of column block Jc (A- and B-operand steps 4 kk)
  auto load_w = [&](int kb, int Jc, double* b) {
#pragma unroll
    for (int kk = 0; kk < 4; kk++) b[kk] = wl[int64_t(16 * kb + 4 * kk) * NB + 16 * Jc];
  };
  const int steps = (Jb + 1) + (Ja + 1);  // of 16 k: block Jb's, then block Ja's
  auto load_step = [&](int s, double* b) {
    s = s < steps ? s : steps - 1;
    load_w(s <= Jb ? s : s - Jb - 1, s <= Jb ? Jb : Ja, b);
  };
  fetch(t0);
  put(t0);
  fetch(t0 + 1);
  lds_barrier();
  for (int64_t t = t0; t < t1; t++) {
    d4 z[2][2];
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int R = 0; R < 2; R++) z[u][R] = d4{0, 0, 0, 0};
    if (steps > 0) {
      // W is loaded two steps ahead (the loads are unconditional, so that their number
      // is known and the products wait for their own only)
      double w0[4], w1[4];
      load_step(0, w0);
      load_step(1, w1);
      auto step = [&](int s, int kb, d4* zz) {
        double w2[4];
        load_step(s + 2, w2);
        const double* sr = S + cc * LD + 16 * kb + kr;
        double x[2][4];
#pragma unroll
        for (int R = 0; R < 2; R++)
#pragma unroll
          for (int kk = 0; kk < 4; kk++) x[R][kk] = sr[16 * R * LD + 4 * kk];
#pragma unroll
        for (int kk = 0; kk < 4; kk++)
#pragma unroll
          for (int R = 0; R < 2; R++) zz[R] = mfma64(x[R][kk], w0[kk], zz[R]);
#pragma unroll
        for (int kk = 0; kk < 4; kk++) {
          w0[kk] = w1[kk];
          w1[kk] = w2[kk];
        }
      };
#pragma unroll 1
      for (int kb = 0; kb <= Jb; kb++) step(kb, kb, z[1]);
#pragma unroll 1
      for (int kb = 0; kb <= Ja; kb++) step(Jb + 1 + kb, kb, z[0]);
    }
    lds_barrier();  // the tile is multiplied, and the Gram of the one before read
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const int Jc = u ? Jb : Ja;
      if (Jc >= 0) {
#pragma unroll
        for (int R = 0; R < 2; R++)
#pragma unroll
          for (int r = 0; r < 4; r++) Zs[(16 * R + 4 * r + kr) * LD + 16 * Jc + cc] = z[u][R][r];
      }
    }
    if (t + 1 < t1) {
      put(t + 1);
      fetch(t + 2);
    }
    lds_barrier();
    gram_tile<LD, SL>(Zs, I, J, cnt, NB / 16, acc);
  }
  store_blocks<NB, SL>(acc, I, J, cnt, part + int64_t(blockIdx.x) * NB * NB);
}

// Product C[m x nc] = Yc W, W (K rows up to a multiple of 16, zero beyond K; ld ldw).
// 16 NR-row tiles, the K columns in chunks of KC; blockIdx.y: slice of 256 columns.  A
// wave's loads and stores complete in order, so W of the next rows waits behind the
// next tile's rows and the last one's stores, and only other waves fill that time.
// Wave w forms the NR 16-row blocks of the column blocks w + NW i of the slice, so each
// element of W it loads from the L2 feeds NR products.  NR = 4 on eight waves, one
// workgroup per CU, for tall inputs: half the traffic of W and half as many of those
// waits per row (8M x 256 float64 62.1 -> 61.3 ms, 1M x 512 38.4 -> 37.2 ms for the
// whole solves); NR = 2 on four waves, two workgroups per CU, where 64-row tiles would be
// too few or the columns leave half of the waves idle.
// upper: W is upper triangular with 16 x 16 blocks (block (kb, J) is zero for kb > J).
template <class TS, class TO, int KC, bool VAR, int NR, int NW>
__global__ __launch_bounds__(64 * NW) void k_gemm_f64(const TS* __restrict__ X, int64_t ldx, int64_t m, int K, int center,
                                                  const double* mean_in, const double* var_in,
                                                  const double* __restrict__ W, int64_t ldw, int nc, int upper,
                                                  TO* __restrict__ C, int64_t ldc, int64_t zx, int64_t zb,
                                                  int64_t zc) {
  X = zoff(X, zx);
  mean_in = zoff(mean_in, zb);
  var_in = zoff(var_in, zb);
  W = zoff(W, zb);
  C = zoff(C, zc);
  constexpr int LD = KC + PADD, TRG = 16 * NR, NI = 16 / NW, SH = NW == 8 ? 3 : 2;
  __shared__ double S[TRG * LD];
  const int w = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)), l = threadIdx.x & 63, kr = l >> 4, cc = l & 15;
  const int Jg = 16 * blockIdx.y + w;
  const int nkb = (K + 15) / 16, nch = (K + KC - 1) / KC;
  int nJ = 0;  // this wave's column blocks inside nc
#pragma unroll
  for (int i = 0; i < NI; i++) nJ += 16 * (Jg + NW * i) < nc;
  const int64_t ntl = ceil_div(m, TRG);
  RowStage<TS, TRG, KC, VAR, 64 * NW> st;
  d4 acc[NR][NI];
#pragma unroll
  for (int R = 0; R < NR; R++)
#pragma unroll
    for (int i = 0; i < NI; i++) acc[R][i] = d4{0, 0, 0, 0};
  int64_t t = blockIdx.x;
  int ch = 0;
  if (t < ntl) st.fetch(X, ldx, m, K, t * TRG, 0, center, mean_in, var_in);
  while (t < ntl) {
    st.template put<LD>(S, 0, m, K, t * TRG, ch * KC, center, false, nullptr, nullptr);
    const bool last = ch + 1 == nch;
    const int64_t tn = last ? t + gridDim.x : t;
    const int chn = last ? 0 : ch + 1;
    const int kb0 = ch * (KC / 16), kb1 = nkb - kb0 < KC / 16 ? nkb - kb0 : KC / 16;
    const double* wl = W + int64_t(16 * kb0 + kr) * ldw + 16 * Jg + cc;
    // a block of W's rows takes part in column block Jg + NW i from lo(kb) on
    auto lo = [&](int kb) {
      if (!upper) return 0;
      const int d = kb0 + kb - Jg;
      return d <= 0 ? 0 : (d + NW - 1) >> SH;
    };
    // Unconditional (column blocks beyond the wave's last repeat it): were the loads
    // behind branches, their number would be unknown and the products of the current
    // rows would wait for the next ones'.
    auto load_w = [&](int kb, double (*b)[4]) {
#pragma unroll
      for (int i = 0; i < NI; i++)
#pragma unroll
        for (int kk = 0; kk < 4; kk++)
          b[i][kk] = wl[int64_t(16 * kb + 4 * kk) * ldw + 16 * NW * (i < nJ ? i : nJ - 1)];
    };
    double wc[NI][4], wn[NI][4];
    if (nJ > 0) load_w(0, wc);
    st.fetch(X, ldx, m, K, (tn < ntl ? tn : t) * TRG, chn * KC, center, mean_in, var_in);
    lds_barrier();
#pragma unroll 1
    for (int kb = 0; nJ > 0 && kb < kb1; kb++) {
      const int from = lo(kb);
      if (from >= nJ) break;  // every later block is zero too
      load_w(kb + 1 < kb1 ? kb + 1 : kb, wn);
      const double* sr = S + cc * LD + 16 * kb + kr;
      double x[NR][4];
#pragma unroll
      for (int R = 0; R < NR; R++)
#pragma unroll
        for (int kk = 0; kk < 4; kk++) x[R][kk] = sr[16 * R * LD + 4 * kk];
#pragma unroll
      for (int i = 0; i < NI; i++)
        if (i < nJ && i >= from) {
#pragma unroll
          for (int kk = 0; kk < 4; kk++)
#pragma unroll
            for (int R = 0; R < NR; R++) acc[R][i] = mfma64(x[R][kk], wc[i][kk], acc[R][i]);
        }
#pragma unroll
      for (int i = 0; i < NI; i++)
#pragma unroll
        for (int kk = 0; kk < 4; kk++) wc[i][kk] = wn[i][kk];
    }
    if (last) {
      TO* ct = C + (t * TRG + kr) * ldc + 16 * Jg + cc;
      const bool whole = (t + 1) * TRG <= m && 16 * (Jg + NW * (nJ - 1) + 1) <= nc;  // no edge in the wave's blocks
#pragma unroll
      for (int i = 0; i < NI; i++) {
        const int col = 16 * (Jg + NW * i) + cc;
#pragma unroll
        for (int R = 0; R < NR; R++) {
          if (i < nJ && whole) {
#pragma unroll
            for (int r = 0; r < 4; r++) ct[(16 * R + 4 * r) * ldc + 16 * NW * i] = TO(acc[R][i][r]);
          } else if (i < nJ) {
#pragma unroll
            for (int r = 0; r < 4; r++)
              if (t * TRG + 16 * R + 4 * r + kr < m && col < nc) ct[(16 * R + 4 * r) * ldc + 16 * NW * i] = TO(acc[R][i][r]);
          }
          acc[R][i] = d4{0, 0, 0, 0};
        }
      }
    }
    t = tn;
    ch = chn;
    lds_barrier();
  }
}

// ---------------------------------------------------------------------------
// cross Gram: P[chunk] += A^T B, A m x p (p <= PB), B m x q (q <= QB)
// ---------------------------------------------------------------------------
template <class TA, class TB, int PB, int QB>
__global__ __launch_bounds__(NTH) void k_xgram_f64(const TA* __restrict__ A, int64_t lda, int p,
                                                   const TB* __restrict__ B, int64_t ldb, int q, int64_t m,
                                                   int64_t tiles_per_chunk, double* __restrict__ part) {
  constexpr int pb = PB / 16, qb = QB / 16;
  constexpr int NBLK = pb * qb;
  constexpr int SL = (NBLK + 7) / 8;
  __shared__ double SA[TR][PB + PADD];
  __shared__ double SB[TR][QB + PADD];
  int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  int kr = l >> 4, cc = l & 15;
  d4 acc[SL];
#pragma unroll
  for (int s = 0; s < SL; s++) acc[s] = d4{0, 0, 0, 0};
  int64_t ntiles = ceil_div(m, TR);
  int64_t t0 = int64_t(blockIdx.x) * tiles_per_chunk;
  int64_t t1 = t0 + tiles_per_chunk < ntiles ? t0 + tiles_per_chunk : ntiles;
  for (int64_t t = t0; t < t1; t++) {
    __syncthreads();
    for (int idx = threadIdx.x; idx < TR * PB; idx += NTH) {
      int r = idx / PB, c = idx % PB;
      int64_t row = t * TR + r;
      SA[r][c] = (row < m && c < p) ? double(A[row * lda + c]) : 0.0;
    }
    for (int idx = threadIdx.x; idx < TR * QB; idx += NTH) {
      int r = idx / QB, c = idx % QB;
      int64_t row = t * TR + r;
      SB[r][c] = (row < m && c < q) ? double(B[row * ldb + c]) : 0.0;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < TR / 4; kk++) {
#pragma unroll
      for (int s = 0; s < SL; s++) {
        int b = w + 8 * s;
        if (b < NBLK) {
          int I = b / qb, J = b % qb;
          acc[s] = mfma64(SA[kk * 4 + kr][I * 16 + cc], SB[kk * 4 + kr][J * 16 + cc], acc[s]);
        }
      }
    }
  }
  double* P = part + int64_t(blockIdx.x) * PB * QB;
#pragma unroll
  for (int s = 0; s < SL; s++) {
    int b = w + 8 * s;
    if (b < NBLK) {
      int I = b / qb, J = b % qb;
#pragma unroll
      for (int r = 0; r < 4; r++) P[int64_t(I * 16 + 4 * r + kr) * QB + J * 16 + cc] = acc[s][r];
    }
  }
}

template <class F>
int dispatch_nb(int n, F&& f) {
  if (n <= 96) return f(std::integral_constant<int, 96>{});
  if (n <= 128) return f(std::integral_constant<int, 128>{});
  if (n <= 160) return f(std::integral_constant<int, 160>{});
  if (n <= 192) return f(std::integral_constant<int, 192>{});
  if (n <= 224) return f(std::integral_constant<int, 224>{});
  if (n <= 256) return f(std::integral_constant<int, 256>{});
  return -1;
}
// rows divided by their variance (center 2) take kernels of their own: the divisions
// cost the others registers that a 256-column Gram does not have
template <class F>
void with_var(int center, F&& f) {
  if (center == 2) f(std::true_type{});
  else f(std::false_type{});
}
// operand widths of the cross products
template <class F>
int dispatch_xnb(int n, F&& f) {
  if (n <= 16) return f(std::integral_constant<int, 16>{});
  if (n <= 32) return f(std::integral_constant<int, 32>{});
  if (n <= 48) return f(std::integral_constant<int, 48>{});
  if (n <= 64) return f(std::integral_constant<int, 64>{});
  if (n <= 128) return f(std::integral_constant<int, 128>{});
  if (n <= 256) return f(std::integral_constant<int, 256>{});
  return -1;
}

}  // namespace

int f64_nb(int n) { return n <= 64 ? int(round_up(n < 1 ? 1 : n, 16)) : n <= 256 ? int(round_up(n, 32)) : -1; }
int f64_xnb(int n) { return n <= 64 ? f64_nb(n) : n <= 128 ? 128 : n <= 256 ? 256 : -1; }
// Row chunks of the Gram passes over n columns (k_direct_f64.hip up to 64): at most
// 512, two per CU in turn, so that half the slabs of 1024 are written and summed
int f64_gram_chunks(int64_t m, int n, bool cplx, int64_t* tpc) {
  if (n <= kDirectGram) return d64_gram_chunks(m, n, cplx, tpc);
  const int64_t tiles = ceil_div(m, TR);
  int64_t per = ceil_div(tiles, 512);
  if (per < 4) per = 4;
  *tpc = per;
  return tiles < 1 ? 1 : int(ceil_div(tiles, per));
}
// cross products take the direct kernel when both operands are narrow
int f64_xgram_chunks(int64_t m, int p, int q, int64_t* tpc) {
  if (p <= kDirectGram && q <= kDirectGram) return d64_xgram_chunks(m, tpc);
  const int c = stream_chunks(m, TR);
  *tpc = ceil_div(ceil_div(m, TR), c);
  return c;
}
// rows of one turn of a product pass over n inputs, and its workgroups: at most 512 of the
// tiled kernel's (two per CU at a time, or one after the other with 64-row tiles)
static bool gemm_tall(int64_t m, int nc) { return nc > 128 && m >= kTallProduct; }
int f64_gemm_rows(int64_t m, int n, int nc) {
  return n > kDirectProduct ? (gemm_tall(m, nc) ? 2 * TR : TR) : n > 64 ? 128 : 256;
}
int f64_gemm_chunks(int64_t m, int n, int nc) {
  if (n <= kDirectProduct) return d64_gemm_chunks(m, n, nc);
  const int64_t tiles = ceil_div(m, f64_gemm_rows(m, n, nc));
  return tiles < 1 ? 1 : int(tiles < 512 ? tiles : 512);
}

// P1 / P2 launchers -----------------------------------------------------------
template <class TS>
static int launch_gram_t(hipStream_t st, const TS* X, int64_t ldx, int64_t m, int n, int center,
                         const double* mean_in, const double* var_in, double* mean_out, double* var_out,
                         const double* W, int chunks, int64_t tpc, double* part, const PassBatch& bz) {
  return dispatch_nb(n, [&](auto nbc) {
    constexpr int NB = decltype(nbc)::value;
    const dim3 g(unsigned(chunks), 1, unsigned(bz.nz));
    with_var(center, [&](auto vc) {
      constexpr bool VAR = decltype(vc)::value;
      if (W)
        hipLaunchKernelGGL((k_zgram_f64<TS, NB, VAR>), g, dim3(NTH), 0, st, X, ldx, m, n, center, mean_in, var_in, W,
                           tpc, part, bz.zx, bz.zb);
      else
        hipLaunchKernelGGL((k_gram_f64<TS, NB, VAR>), g, dim3(NTH), 0, st, X, ldx, m, n, center, mean_out, var_out,
                           tpc, part, bz.zx, bz.zb);
    });
    return 0;
  });
}

int launch_gram_f64(hipStream_t st, pc_dtype dt, const void* X, int64_t ldx, int64_t m, int n, int center,
                    const double* mean_in, const double* var_in, double* mean_out, double* var_out, const double* W,
                    int chunks, int64_t tpc, double* part, const PassBatch& bz) {
  if (n <= kDirectGram)
    return launch_d64_gram(st, dt, X, ldx, m, n, center, mean_in, var_in, mean_out, var_out, W, chunks, tpc, part, bz);
  if (dt == PC_F64)
    return launch_gram_t<double>(st, (const double*)X, ldx, m, n, center, mean_in, var_in, mean_out, var_out, W,
                                 chunks, tpc, part, bz);
  return launch_gram_t<float>(st, (const float*)X, ldx, m, n, center, mean_in, var_in, mean_out, var_out, W, chunks,
                              tpc, part, bz);
}

template <class TS, class TO>
static int launch_gemm_t(hipStream_t st, const TS* X, int64_t ldx, int64_t m, int n, int center,
                         const double* mean_in, const double* var_in, const double* W, int64_t ldw, int nc, int chunks,
                         int upper, TO* C, int64_t ldc, const PassBatch& bz) {
  return dispatch_nb(n < 160 ? 160 : n > 256 ? 256 : n, [&](auto kc) {
    constexpr int KC = decltype(kc)::value;
    if constexpr (KC > kDirectProduct) {
      with_var(center, [&](auto vc) {
        constexpr bool VAR = decltype(vc)::value;
        const dim3 g(unsigned(chunks), unsigned(ceil_div(nc, 256)), unsigned(bz.nz));
        if (gemm_tall(m, nc))
          hipLaunchKernelGGL((k_gemm_f64<TS, TO, KC, VAR, 4, 8>), g, dim3(512), 0, st, X, ldx, m, n, center, mean_in,
                             var_in, W, ldw, nc, upper, C, ldc, bz.zx, bz.zb, bz.zc);
        else
          hipLaunchKernelGGL((k_gemm_f64<TS, TO, KC, VAR, 2, 4>), g, dim3(256), 0, st, X, ldx, m, n, center, mean_in,
                             var_in, W, ldw, nc, upper, C, ldc, bz.zx, bz.zb, bz.zc);
      });
      return 0;
    }
    return -1;
  });
}

int launch_gemm_f64(hipStream_t st, pc_dtype dt, const void* X, int64_t ldx, int64_t m, int n, int center,
                    const double* mean_in, const double* var_in, const double* W, int64_t ldw, int nc, int chunks,
                    void* C, int64_t ldc, const PassBatch& bz, bool out_f64, bool upper) {
  if (n <= kDirectProduct && !out_f64)
    return launch_d64_gemm(st, dt, X, ldx, m, n, center, mean_in, var_in, W, int(ldw), nc, chunks, C, ldc, bz);
  if (dt == PC_F64)
    return launch_gemm_t<double, double>(st, (const double*)X, ldx, m, n, center, mean_in, var_in, W, ldw, nc, chunks,
                                         upper ? 1 : 0, (double*)C, ldc, bz);
  if (out_f64)
    return launch_gemm_t<float, double>(st, (const float*)X, ldx, m, n, center, mean_in, var_in, W, ldw, nc, chunks,
                                        upper ? 1 : 0, (double*)C, ldc, bz);
  return launch_gemm_t<float, float>(st, (const float*)X, ldx, m, n, center, mean_in, var_in, W, ldw, nc, chunks,
                                     upper ? 1 : 0, (float*)C, ldc, bz);
}

template <class T>
static int launch_xgram_t(hipStream_t st, const T* A, int64_t lda, int p, const T* B, int64_t ldb, int q, int64_t m,
                          int chunks, int64_t tpc, double* part) {
  int pb = f64_xnb(p), qb = f64_xnb(q);
  if (pb < 0 || qb < 0) return -1;
  if (int64_t(pb) * qb > 128 * 256) return -1;  // register budget: at most 128 blocks
  return dispatch_xnb(pb, [&](auto pc_) {
    constexpr int PB = decltype(pc_)::value;
    return dispatch_xnb(qb, [&](auto qc_) {
      constexpr int QB = decltype(qc_)::value;
      if constexpr (PB * QB <= 128 * 256 && (PB > kDirectGram || QB > kDirectGram)) {
        hipLaunchKernelGGL((k_xgram_f64<T, T, PB, QB>), dim3(chunks), dim3(NTH), 0, st, A, lda, p, B, ldb, q, m, tpc,
                           part);
        return 0;
      } else {
        return -1;
      }
    });
  });
}

int launch_xgram_f64(hipStream_t st, pc_dtype dt, const void* A, int64_t lda, int p, const void* B, int64_t ldb, int q,
                     int64_t m, int chunks, int64_t tpc, double* part) {
  if (p <= kDirectGram && q <= kDirectGram)
    return launch_d64_xgram(st, dt, A, lda, p, B, ldb, q, m, chunks, tpc, part);
  if (dt == PC_F64)
    return launch_xgram_t<double>(st, (const double*)A, lda, p, (const double*)B, ldb, q, m, chunks, tpc, part);
  return launch_xgram_t<float>(st, (const float*)A, lda, p, (const float*)B, ldb, q, m, chunks, tpc, part);
}
