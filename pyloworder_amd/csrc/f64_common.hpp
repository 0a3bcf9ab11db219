// Device helpers shared by the FP64 MFMA streaming kernels.
//
// v_mfma_f64_16x16x4f64 (wave64, lane l, i = l % 16, g = l / 16):
//   A (16x4): A[i][g]    B (4x16): B[g][i]    D (16x16), reg r: D[4 r + g][i]
#pragma once
#include "common.hpp"

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

PC_DEV d4 mfma64(double a, double b, d4 c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }

// Workgroup barrier for LDS traffic only: __syncthreads() would also wait for the
// outstanding global loads of the next tile.
PC_DEV void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <int CTRL>
PC_DEV double dpp_move(double x) {
  const long long b = __builtin_bit_cast(long long, x);
  const int lo = __builtin_amdgcn_update_dpp(0, int(b), CTRL, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_update_dpp(0, int(b >> 32), CTRL, 0xF, 0xF, true);
  return __builtin_bit_cast(double, (long long)(unsigned)lo | ((long long)hi << 32));
}
// sum over the 16 lanes of a DPP row, in every lane
PC_DEV double row16_sum(double v) {
  v += dpp_move<0xB1>(v);   // quad_perm [1,0,3,2]
  v += dpp_move<0x4E>(v);   // quad_perm [2,3,0,1]
  v += dpp_move<0x141>(v);  // row_half_mirror
  v += dpp_move<0x140>(v);  // row_mirror
  return v;
}
// s / n with iv = 1 / n: the quotient and one residual step
PC_DEV double div_n(double s, double n, double iv) {
  const double q = s * iv;
  return fma(fma(-n, q, s), iv, q);
}

// x /= var.  Called under a uniform branch and opaque to the optimiser, which would
// otherwise run the divisions (17 FP64 instructions an element) for every centring
// and select their result.
template <int N>
PC_DEV void divide_rows(double* x, double var) {
  asm volatile("" : "+v"(var));
#pragma unroll
  for (int q = 0; q < N; q++) x[q] /= var;
}

// Rows of a row-major operand on their way to LDS: NTHR threads hold ROWS x COLS
// elements, thread (lane32, r0) = (tid % 32, tid / 32) rows r0 + RG p and columns
// lane32 + 32 q, so a load instruction reads 32 consecutive elements of two rows.
// fetch() only issues loads (clamped, so nothing branches); put() centres (VAR: and
// divides by the row variance), masks and stores them as FP64.
template <class TS, int ROWS, int COLS, bool VAR, int NTHR = 512>
struct RowStage {
  static constexpr int RG = NTHR / 32, P = ROWS / RG, Q = COLS / 32;
  TS v[P][Q];
  double mu[P], var[VAR ? P : 1];

  // rows row0 .., columns col0 .. of X (m x n); the statistics of the rows when given
  PC_DEV void fetch(const TS* __restrict__ X, int64_t ldx, int64_t m, int n, int64_t row0, int col0, int center,
                    const double* mean, const double* vars) {
    const int lane = threadIdx.x & 31, r0 = threadIdx.x >> 5;
#pragma unroll
    for (int p = 0; p < P; p++) {
      const int64_t row = row0 + r0 + RG * p, rc = row < m ? row : m - 1;
#pragma unroll
      for (int q = 0; q < Q; q++) {
        const int c = col0 + lane + 32 * q;
        v[p][q] = X[rc * ldx + (c < n ? c : 0)];
      }
      if (center && mean) mu[p] = mean[rc];
      if constexpr (VAR)
        if (vars) var[p] = vars[rc];
    }
  }
  // S[row][s0 + column], LD doubles per row.  stats: the row mean (and variance) come
  // from the staged columns themselves (all n of them) and are stored when asked for
  template <int LD>
  PC_DEV void put(double* S, int s0, int64_t m, int n, int64_t row0, int col0, int center, bool stats,
                  double* mean_out, double* var_out) {
    const int lane = threadIdx.x & 31, r0 = threadIdx.x >> 5;
    const double nd = n, inv_n = 1.0 / nd;
#pragma unroll
    for (int p = 0; p < P; p++) {
      const int64_t row = row0 + r0 + RG * p;
      const bool rv = row < m;
      double x[Q];
#pragma unroll
      for (int q = 0; q < Q; q++) x[q] = rv && col0 + lane + 32 * q < n ? double(v[p][q]) : 0.0;
      if (center) {
        double mu_ = mu[p];
        [[maybe_unused]] double var_ = VAR ? var[p] : 1.0;
        if (stats) {
          double s = 0.0;
#pragma unroll
          for (int q = 0; q < Q; q++) s += x[q];
          s = row16_sum(s);
          mu_ = div_n(s + __shfl_xor(s, 16), nd, inv_n);
          if constexpr (VAR) {
            double s2 = 0.0;
#pragma unroll
            for (int q = 0; q < Q; q++) {
              const double d = col0 + lane + 32 * q < n ? x[q] - mu_ : 0.0;
              s2 += d * d;
            }
            s2 = row16_sum(s2);
            var_ = div_n(s2 + __shfl_xor(s2, 16), nd, inv_n);
            if (rv && lane == 0 && var_out) var_out[row] = var_;
          }
          if (rv && lane == 0 && mean_out) mean_out[row] = mu_;
        }
#pragma unroll
        for (int q = 0; q < Q; q++) x[q] = rv && col0 + lane + 32 * q < n ? x[q] - mu_ : 0.0;
        if constexpr (VAR) {
          divide_rows<Q>(x, var_);
#pragma unroll
          for (int q = 0; q < Q; q++) x[q] = rv && col0 + lane + 32 * q < n ? x[q] : 0.0;  // 0 / 0 beyond the edges
        }
      }
#pragma unroll
      for (int q = 0; q < Q; q++) S[(r0 + RG * p) * LD + s0 + lane + 32 * q] = x[q];
    }
  }
};

}  // namespace
