// Real one-sided block Jacobi driven by the columns' Gram matrix (included by
// solve.hip after k_small.hip).  H (n x n, column-major) is rotated from the right
// until its columns are orthogonal, J collects the rotations.
//
// The columns form nb2 blocks of GB = 16.  A sweep is
//   k_bjac_gram : G = H^T H from the current columns, and the one-sided test
//                 |G_uv| <= tol sqrt(G_uu G_vv) on every pair.  A sweep whose test
//                 finds nothing ends the iteration.
//   k_bjac_pair : nb2 - 1 round-robin steps, one launch each.  A step pairs the
//                 blocks; each pair's rotation Q (32 x 32 orthogonal) comes from one
//                 cyclic sweep of two-sided rotations on its 32 x 32 block of G, and
//                 G <- Q^T G Q, H <- H Q, J <- J Q follow in the same launch.
// G is only kept between two tests of a sweep; convergence is always decided on a
// Gram computed afresh from the columns.
//
// Latency is the cost (one step's rounds depend on each other), so a step is one
// launch: workgroup (p, q) forms the rotations of pairs p and q itself, side by side
// on two halves of 256 threads, while its part of G, H and J is already on its way
// from memory, and applies them to G[pair p, pair q] and to 32 rows of H and J.
// That costs nb2 / 2 times the rotations on otherwise idle CUs.  It replaced two
// launches per step (rotations on one workgroup per pair from a Gram computed there,
// then the products): 22.3 -> 10.7 us per step at n = 200 under the profiler (of it
// 6.4 us are the 16 rounds, 0.4 us each: LDS exchange 155 cycles, angle 150, shuffle
// 58), 20.2 us for the first step of a sweep; the iteration of 20,000 x 200 took 2.9
// ms and takes 1.5.  n <= 32 is one launch (six launches of the pair kernel before:
// 196 -> 64 us at n = 8).
// Above kJacFused columns the rotations are formed once per pair in a launch of
// their own: (n / 32)^2 workgroups repeating them no longer run beside each other.

constexpr int GB = 16;
constexpr int GC = 2 * GB;
constexpr int GLD = GC + 1;
constexpr int kJacFused = 512;
// dstate: [0] negligible squared norm and [1] power-of-two scale of G (its trace about
// 2^96: products of its entries neither overflow nor underflow, and those above the
// negligible norm are within float's range), from kBjacQOff
// the nb2 / 2 pair rotations of the unfused steps
constexpr int kBjacQOff = 4;
inline int64_t bjac_dstate_len(int n) {
  int64_t nb2 = (int64_t(n) + GB - 1) / GB;
  nb2 += nb2 & 1;
  if (nb2 < 16) nb2 = 16;
  return kBjacQOff + (nb2 / 2) * GC * GC + nb2 / 2;
}

// lane i of a 16-lane row reads lane (i + 1) % 16
PC_DEV double row16_next(double x) {
  const long long b = __builtin_bit_cast(long long, x);
  const int lo = __builtin_amdgcn_update_dpp(0, int(b), 0x12F, 0xF, 0xF, true);  // row_ror:15
  const int hi = __builtin_amdgcn_update_dpp(0, int(b >> 32), 0x12F, 0xF, 0xF, true);
  return __builtin_bit_cast(double, (long long)(unsigned)lo | ((long long)hi << 32));
}

// Rotation zeroing the off-diagonal c of [[a, c], [c, b]]: u' = cs u - sn v,
// v' = sn u + cs v, tan(2 theta) = 2 c / (b - a), |theta| <= pi / 4; the identity when
// c passes the orthogonality test or a column is negligible.  The angle only steers
// convergence, so it comes from float estimates (half-angle formulas, relative error
// about 1e-6); what has to hold to rounding is cs^2 + sn^2 = 1, and the FP64 step
// (cs, sn) (1 + e / 2 + 3 e^2 / 8), e = 1 - cs^2 - sn^2, does that to e^3.  The test is
// FP64.  (256 -> 150 cycles of a round's chain against FP64 estimates with Newton
// steps.)  Against the angle in FP64 by square root and division, over 128 matrices each of
// 16 to 100 columns and condition 1e10, 1e12 and 1e14: the same singular values to three
// digits of their error, V orthogonal to 2e-15 to 4e-15 (2e-15 to 1e-14 with the other).
// G's scale keeps d, c of any active pair far inside float's range.
PC_DEV bool jac_active(double a, double b, double c, double negl, double tol2) {
  return a > negl && b > negl && c * c > tol2 * a * b;
}
PC_DEV void jac_angle(double a, double b, double c, double negl, double tol2, double& cs, double& sn) {
  const float d = float(b - a), e = float(c + c);
  const float rm = __builtin_amdgcn_rcpf(fmaxf(fabsf(d), fabsf(e)));
  const float dn = fabsf(d) * rm, em = e * rm, en = d < 0.0f ? -em : em;
  const float y = __builtin_amdgcn_rsqf(fmaf(dn, dn, en * en));  // 1 / hypot
  const float w = fmaf(0.5f * dn, y, 0.5f);                      // cos^2(theta)
  const float r = __builtin_amdgcn_rsqf(w);
  const double c0 = double(w * r), s0 = double(0.5f * en * y * r);
  double f = fma(-c0, c0, 1.0);
  f = fma(-s0, s0, f);
  f = f * fma(f, 0.375, 0.5);
  const bool act = jac_active(a, b, c, negl, tol2);
  cs = act ? fma(c0, f, c0) : 1.0;
  sn = act ? fma(s0, f, s0) : 0.0;
}

// LDS of one pair's rounds
template <bool FULL>
struct JacPair {
  double A[GB], B[GB];            // the diagonal
  double X[2][2][GB * (GB + 1)];  // G_vu and G_vv, which move between threads
  double G[2][FULL ? GC * GLD : 1], Q[2][FULL ? GC * GLD : 1];
};

// One cyclic sweep of two-sided rotations on a pair's 32 x 32 block of G by 256
// threads (t); every thread of the workgroup calls it (barriers inside).  Thread
// (bp, bq) = (t / 16, t % 16) comes with g = G at rows {u_bp, v_bp}, columns {u_bq,
// v_bq}, u_k = k, v_k = 16 + k, and leaves with q = the rotation's rows 2 bp, 2 bp + 1
// at columns u_bq, v_bq.  FULL: also the pairs inside the two blocks (15 rounds of
// both side by side, through LDS) before the 16 rounds of pairs across them, in which
// round s pairs u_k with v_{k+s}: u's data stay with their thread, v's move on by one
// pair per round, along bq by DPP, along bp through LDS.  One barrier per round.
// players < 16 (even): no column beyond the first `players` exists, so players - 1
// rounds meet every pair.
template <bool FULL>
PC_DEV void jac_rounds(JacPair<FULL>& S, int t, double negl, double tol2, const double (&g)[4], double (&q)[4],
                       int players = GB, bool cross = true) {
  const int bp = t >> 4, bq = t & 15;
  double guu = g[0], guv = g[1], gvu = g[2], gvv = g[3];
  q[0] = 2 * bp == bq ? 1.0 : 0.0;
  q[1] = 2 * bp == bq + GB ? 1.0 : 0.0;
  q[2] = 2 * bp + 1 == bq ? 1.0 : 0.0;
  q[3] = 2 * bp + 1 == bq + GB ? 1.0 : 0.0;
  if constexpr (FULL) {
    S.G[0][bp * GLD + bq] = guu;
    S.G[0][bp * GLD + GB + bq] = guv;
    S.G[0][(GB + bp) * GLD + bq] = gvu;
    S.G[0][(GB + bp) * GLD + GB + bq] = gvv;
    S.Q[0][2 * bp * GLD + bq] = q[0];
    S.Q[0][2 * bp * GLD + GB + bq] = q[1];
    S.Q[0][(2 * bp + 1) * GLD + bq] = q[2];
    S.Q[0][(2 * bp + 1) * GLD + GB + bq] = q[3];
    // Positions, not columns: the players of each block's circle schedule sit at
    // positions 0..players - 1, pair k of block k / 8 at positions k & 7 and players - 1 -
    // (k & 7), and every result is stored where its player sits in the next round (slot
    // k moves to k - 1, slot 1 to the last, slot 0 stays), so a thread's addresses never
    // change.  After players - 1 rounds everybody is back.  The (empty) positions
    // beyond pair up among themselves and stay.
    auto first = [&](int k) { return 2 * k < players ? k : 2 * k; };
    auto second = [&](int k) { return 2 * k < players ? players - 1 - k : 2 * k + 1; };
    auto next = [&](int k) { return k == 0 || k >= players ? k : k == 1 ? players - 1 : k - 1; };
    const int ob = 2 * (bp & 8), oq = 2 * (bq & 8);
    const int up = ob + first(bp & 7), vp = ob + second(bp & 7), uq = oq + first(bq & 7), vq = oq + second(bq & 7);
    const int upn = ob + next(up - ob), vpn = ob + next(vp - ob);
    const int uqn = oq + next(uq - oq), vqn = oq + next(vq - oq);
    __syncthreads();
#pragma unroll 2
    for (int s = 0; s < players - 1; s++) {
      const double *G0 = S.G[s & 1], *Q0 = S.Q[s & 1];
      double *G1 = S.G[~s & 1], *Q1 = S.Q[~s & 1];
      double cq, sq;
      jac_angle(G0[uq * GLD + uq], G0[vq * GLD + vq], G0[uq * GLD + vq], negl, tol2, cq, sq);
      const double cp = __shfl(cq, bp), sp = __shfl(sq, bp);
      const double a = G0[up * GLD + uq], b = G0[up * GLD + vq], c = G0[vp * GLD + uq], d = G0[vp * GLD + vq];
      const double xa = cq * a - sq * b, xb = sq * a + cq * b, xc = cq * c - sq * d, xd = sq * c + cq * d;
      G1[upn * GLD + uqn] = cp * xa - sp * xc;
      G1[upn * GLD + vqn] = cp * xb - sp * xd;
      G1[vpn * GLD + uqn] = sp * xa + cp * xc;
      G1[vpn * GLD + vqn] = sp * xb + cp * xd;
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int row = (2 * bp + h) * GLD;
        const double x = Q0[row + uq], y = Q0[row + vq];
        Q1[row + uqn] = cq * x - sq * y;
        Q1[row + vqn] = sq * x + cq * y;
      }
      __syncthreads();
    }
    constexpr int last = (GB - 1) & 1;
    guu = S.G[last][bp * GLD + bq];
    guv = S.G[last][bp * GLD + GB + bq];
    gvu = S.G[last][(GB + bp) * GLD + bq];
    gvv = S.G[last][(GB + bp) * GLD + GB + bq];
    q[0] = S.Q[last][2 * bp * GLD + bq];
    q[1] = S.Q[last][2 * bp * GLD + GB + bq];
    q[2] = S.Q[last][(2 * bp + 1) * GLD + bq];
    q[3] = S.Q[last][(2 * bp + 1) * GLD + GB + bq];
  }
  if (!cross) return;
  // Round s's rotation k needs G_uu, G_vv, G_uv of pair k: the last two are the
  // diagonals of what moved in the round before (G_uv as its mirror G_vu), the first
  // every thread carries along for its own k = bq.
  if (bp == bq) {
    S.A[bp] = guu;
    S.X[0][0][bp * (GB + 1) + bq] = gvu;
    S.X[0][1][bp * (GB + 1) + bq] = gvv;
  }
  __syncthreads();
  double a = S.A[bq];
  const int mine = bp * (GB + 1) + bq, diag = bq * (GB + 2);
  const int pm = (bp + GB - 1) & 15, qm = (bq + GB - 1) & 15;
  const int to0 = pm * (GB + 1) + bq, to1 = pm * (GB + 1) + qm;
#pragma unroll 2
  for (int s = 0; s < GB; s++) {
    const int cur = s & 1, nxt = cur ^ 1;
    const double c = S.X[cur][0][diag], b = S.X[cur][1][diag];
    if (s > 0) {
      gvu = S.X[cur][0][mine];
      gvv = S.X[cur][1][mine];
    }
    double cq, sq;
    jac_angle(a, b, c, negl, tol2, cq, sq);
    const double cp = __shfl(cq, bp), sp = __shfl(sq, bp);
    const double xa = cq * guu - sq * guv, xb = sq * guu + cq * guv;
    const double xc = cq * gvu - sq * gvv, xd = sq * gvu + cq * gvv;
    S.X[nxt][0][to0] = sp * xa + cp * xc;
    S.X[nxt][1][to1] = sp * xb + cp * xd;
    guu = cp * xa - sp * xc;
    guv = row16_next(cp * xb - sp * xd);
    a = cq * (cq * a - sq * c) - sq * (cq * c - sq * b);
    const double q0 = cq * q[0] - sq * q[1], q1 = sq * q[0] + cq * q[1];
    const double q2 = cq * q[2] - sq * q[3], q3 = sq * q[2] + cq * q[3];
    q[0] = q0;
    q[1] = row16_next(q1);
    q[2] = q2;
    q[3] = row16_next(q3);
    __syncthreads();
  }
}

// G (n x n, row-major, both triangles) = scale H^T H, one 16 x 16 tile I <= J per
// workgroup, the rows split over its 4 waves; state[1 + sweep] is set when some pair
// of columns fails the orthogonality test.
__global__ __launch_bounds__(256) void k_bjac_gram(const double* __restrict__ H, int ldh, int n, int nt,
                                                   double* __restrict__ G, int sweep, int* state,
                                                   const double* dstate, double tol2) {
  __shared__ double red[4][256], nrm[2][4][16];
  if (state[0]) return;
  int I = 0, J = int(blockIdx.x);
  while (J >= nt - I) J -= nt - I++;
  J += I;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, i = l & 15, g = l >> 4;
  const int ca = 16 * I + i, cb = 16 * J + i;
  const double* ha = H + int64_t(ca < n ? ca : 0) * ldh;
  const double* hb = H + int64_t(cb < n ? cb : 0) * ldh;
  d4s acc = {0.0, 0.0, 0.0, 0.0};
  double sa = 0.0, sb = 0.0;
  for (int k0 = 32 * w; k0 < n; k0 += 128) {
    double a[8], b[8];
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const int k = k0 + 4 * u + g;
      a[u] = k < n && ca < n ? ha[k] : 0.0;
      b[u] = k < n && cb < n ? hb[k] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < 8; u++) {
      acc = mfma64s(a[u], b[u], acc);
      sa = fma(a[u], a[u], sa);
      sb = fma(b[u], b[u], sb);
    }
  }
#pragma unroll
  for (int o = 16; o < 64; o <<= 1) {
    sa += __shfl_xor(sa, o);
    sb += __shfl_xor(sb, o);
  }
#pragma unroll
  for (int r = 0; r < 4; r++) red[w][r * 64 + l] = acc[r];
  if (g == 0) {
    nrm[0][w][i] = sa;
    nrm[1][w][i] = sb;
  }
  __syncthreads();
  const int e = threadIdx.x, ri = 4 * (e >> 6) + ((e >> 4) & 3), rj = e & 15;  // D layout of register e / 64
  const double sc = dstate[1], negl = dstate[0];
  const double c = sc * ((red[0][e] + red[1][e]) + (red[2][e] + red[3][e]));
  const double a = sc * ((nrm[0][0][ri] + nrm[0][1][ri]) + (nrm[0][2][ri] + nrm[0][3][ri]));
  const double b = sc * ((nrm[1][0][rj] + nrm[1][1][rj]) + (nrm[1][2][rj] + nrm[1][3][rj]));
  const int row = 16 * I + ri, col = 16 * J + rj;
  if (row <= col && col < n) {
    G[int64_t(row) * n + col] = c;
    G[int64_t(col) * n + row] = c;
    if (row < col && jac_active(a, b, c, negl, tol2)) state[1 + sweep] = 1;  // any thread's 1 is the same 1
  }
}

// MODE 0: rotations and products; 1: rotations of pairs 2 b, 2 b + 1 only, into Qg;
// 2: products only, from Qg.
// FULL: the first step of a sweep.
template <int MODE, bool FULL>
__global__ __launch_bounds__(512) void k_bjac_pair(double* __restrict__ H, int ldh, int n, double* __restrict__ J,
                                                   int ldj, const double* __restrict__ Gin, double* __restrict__ Gout,
                                                   int nb2, int step, int sweep, int* state,
                                                   const double* __restrict__ dstate, double* __restrict__ Qg,
                                                   double tol2) {
  __shared__ JacPair<FULL> S[2];
  __shared__ double Qs[2][GC * GLD];
  __shared__ int need[2];
  const int done = state[0], rotate = state[1 + sweep];
  const int np = nb2 / 2;
  const int p = MODE == 1 ? 2 * blockIdx.x : blockIdx.x % np, q = MODE == 1 ? p + 1 : blockIdx.x / np;
  const int h = threadIdx.x >> 8, t = threadIdx.x & 255;
  // column blocks of pairs p and q; every index below is one of these plus an offset,
  // and out-of-range elements are read at column 0 and masked (no branches, so the
  // loads go out together)
  const int bp0 = GB * rr_player(p, step, nb2), bp1 = GB * rr_player(nb2 - 1 - p, step, nb2);
  const int bq0 = GB * rr_player(q < np ? q : p, step, nb2), bq1 = GB * rr_player(nb2 - 1 - (q < np ? q : p), step, nb2);
  auto at = [&](const double* M, int ld, int row, int col) {
    const bool in = row < n && col < n;
    const double v = M[in ? int64_t(row) * ld + col : 0];
    return in ? v : 0.0;
  };
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, i = l & 15, g = l >> 4;
  // this thread's part of its pair's G
  double gg[4] = {0.0, 0.0, 0.0, 0.0};
  if (MODE != 2) {
    const int bp = t >> 4, bq = t & 15, b0 = h ? bq0 : bp0, b1 = h ? bq1 : bp1;
    gg[0] = at(Gin, n, b0 + bp, b0 + bq);
    gg[1] = at(Gin, n, b0 + bp, b1 + bq);
    gg[2] = at(Gin, n, b1 + bp, b0 + bq);
    gg[3] = at(Gin, n, b1 + bp, b1 + bq);
#pragma unroll
    for (int k = 0; k < 4; k++) asm volatile("" : "+v"(gg[k]));  // read with the flags, not after them
  }
  if (done) return;
  if (!rotate) {  // the sweep's test found every pair orthogonal
    if (step == 0 && blockIdx.x == 0 && threadIdx.x == 0) state[0] = 1;
    return;
  }
  // operands of the products, in flight during the rounds.  Waves 0-3: G[pair p, pair
  // q] (p <= q), both 16-row halves; waves 4-7: rows 32 q .. of H and J, pair p
  const bool gpart = w < 4;
  double fa[GC / 4], fb[GC / 4];
  const int hr = 32 * q + 16 * ((w >> 1) & 1) + i;
  if (MODE != 1) {
    if (gpart) {
#pragma unroll
      for (int kk = 0; kk < GC / 4; kk++) {  // G is symmetric: read along its rows
        const int ck = (kk < 4 ? bq0 : bq1) + 4 * (kk & 3) + g;
        fa[kk] = at(Gin, n, ck, bp0 + i);
        fb[kk] = at(Gin, n, ck, bp1 + i);
      }
    } else {
#pragma unroll
      for (int kk = 0; kk < GC / 4; kk++) {
        const int ck = (kk < 4 ? bp0 : bp1) + 4 * (kk & 3) + g;
        fa[kk] = at(H, ldh, ck, hr);
        fb[kk] = at(J, ldj, ck, hr);
      }
    }
  }
  const double negl = dstate[0];
  if (threadIdx.x < 2) need[threadIdx.x] = 0;
  if constexpr (MODE != 2) {
    const int bp = t >> 4, bq = t & 15;
    if (bp == bq) {
      S[h].A[bp] = gg[0];
      S[h].B[bp] = gg[3];
    }
    __syncthreads();
    // The first step of a sweep rotates every pair of its 32 columns, later steps the
    // 256 pairs across the blocks: each pair of columns once per sweep
    bool any = jac_active(S[h].A[bp], S[h].B[bq], gg[1], negl, tol2);
    if (FULL && bp < bq)
      any = any || jac_active(S[h].A[bp], S[h].A[bq], gg[0], negl, tol2) ||
            jac_active(S[h].B[bp], S[h].B[bq], gg[3], negl, tol2);
    if (any) need[h] = 1;
    __syncthreads();
    double qq[4];
    if (need[0] | need[1]) {
      jac_rounds<FULL>(S[h], t, negl, tol2, gg, qq);
    } else {
      qq[0] = 2 * bp == bq ? 1.0 : 0.0;
      qq[1] = 2 * bp == bq + GB ? 1.0 : 0.0;
      qq[2] = 2 * bp + 1 == bq ? 1.0 : 0.0;
      qq[3] = 2 * bp + 1 == bq + GB ? 1.0 : 0.0;
    }
    if constexpr (MODE == 1) {
      const int mine = h ? q : p;
      if (mine < np) {
        double* o = Qg + int64_t(mine) * GC * GC + 2 * bp * GC;
        o[bq] = qq[0];
        o[GB + bq] = qq[1];
        o[GC + bq] = qq[2];
        o[GC + GB + bq] = qq[3];
      }
      return;
    }
    double* o = Qs[h] + 2 * bp * GLD;
    o[bq] = qq[0];
    o[GB + bq] = qq[1];
    o[GLD + bq] = qq[2];
    o[GLD + GB + bq] = qq[3];
  } else {
    const double* src = Qg + int64_t(h ? q : p) * GC * GC;
    for (int e = t; e < GC * GC; e += 256) Qs[h][(e >> 5) * GLD + (e & 31)] = src[e];
  }
  __syncthreads();
  if (gpart) {
    if (p > q) return;
    // tile (ti, tj) of Qp^T (G Qq); the accumulators of G Qq are operand fragments
    const int ti = w >> 1, tj = w & 1;
    d4s x0 = {0.0, 0.0, 0.0, 0.0}, x1 = x0, o = x0;
#pragma unroll
    for (int kk = 0; kk < GC / 4; kk++) {
      const double b = Qs[1][(4 * kk + g) * GLD + 16 * tj + i];
      x0 = mfma64s(fa[kk], b, x0);
      x1 = mfma64s(fb[kk], b, x1);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) o = mfma64s(Qs[0][(4 * r + g) * GLD + 16 * ti + i], x0[r], o);
#pragma unroll
    for (int r = 0; r < 4; r++) o = mfma64s(Qs[0][(16 + 4 * r + g) * GLD + 16 * ti + i], x1[r], o);
    const int cc = (tj ? bq1 : bq0) + i;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int lr = 16 * ti + 4 * r + g, rr = (ti ? bp1 : bp0) + 4 * r + g;
      if (rr < n && cc < n && (p < q || lr <= 16 * tj + i)) {  // one value for both triangles
        Gout[int64_t(rr) * n + cc] = o[r];
        Gout[int64_t(cc) * n + rr] = o[r];
      }
    }
  } else {
    // (H Q)^T = Q^T H^T: lanes run along the rows of a column
    const int cB = w & 1;
    d4s oh = {0.0, 0.0, 0.0, 0.0}, oj = oh;
#pragma unroll
    for (int kk = 0; kk < GC / 4; kk++) {
      const double a = Qs[0][(4 * kk + g) * GLD + 16 * cB + i];
      oh = mfma64s(a, fa[kk], oh);
      oj = mfma64s(a, fb[kk], oj);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int cc = (cB ? bp1 : bp0) + 4 * r + g;
      if (cc < n && hr < n) {
        H[int64_t(cc) * ldh + hr] = oh[r];
        J[int64_t(cc) * ldj + hr] = oj[r];
      }
    }
  }
}

// n <= 32: every column in one pair, iterated to convergence on one workgroup.  A sweep
// is n - 1 rounds (n even) up to 16 columns, 31 beyond: n = 8 76 -> 31 us.
__global__ __launch_bounds__(256) void k_bjac_one(double* __restrict__ H, int ldh, int n, double* __restrict__ J,
                                                  int ldj, int* state, const double* dstate, double tol2,
                                                  int max_sweeps) {
  __shared__ JacPair<true> S;
  __shared__ double M[2][GC * GLD], Qs[GC * GLD];  // H and J, column c at c * GLD
  const int t = threadIdx.x, w = t >> 6, l = t & 63, i = l & 15, g = l >> 4, bp = t >> 4, bq = t & 15;
  for (int e = t; e < GC * GC; e += 256) {
    const int c = e >> 5, r = e & 31;
    M[0][c * GLD + r] = c < n && r < n ? H[int64_t(c) * ldh + r] : 0.0;
    M[1][c * GLD + r] = c == r ? 1.0 : 0.0;
  }
  const double negl = dstate[0], sc = dstate[1];
  const int I = w >> 1, Jt = w & 1;  // this wave's tile
  bool done = false;
  for (int it = 0; it < max_sweeps; it++) {
    __syncthreads();
    d4s a4 = {0.0, 0.0, 0.0, 0.0};
    // tile (1, 0) as the mirror of (0, 1): G stays symmetric
    const int ta = I <= Jt ? I : Jt, tb = I <= Jt ? Jt : I;
#pragma unroll
    for (int kk = 0; kk < GC / 4; kk++)
      a4 = mfma64s(M[0][(16 * ta + i) * GLD + 4 * kk + g], M[0][(16 * tb + i) * GLD + 4 * kk + g], a4);
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int x = 16 * ta + 4 * r + g, y = 16 * tb + i;
      if (I <= Jt) S.G[0][x * GLD + y] = sc * a4[r];
      else S.G[0][y * GLD + x] = sc * a4[r];
    }
    __syncthreads();
    bool any = false;
    for (int e = t; e < GC * GC; e += 256) {
      const int u = e >> 5, v = e & 31;
      if (u < v)
        any = any || jac_active(S.G[0][u * GLD + u], S.G[0][v * GLD + v], S.G[0][u * GLD + v], negl, tol2);
    }
    double gg[4] = {S.G[0][bp * GLD + bq], S.G[0][bp * GLD + GB + bq], S.G[0][(GB + bp) * GLD + bq],
                    S.G[0][(GB + bp) * GLD + GB + bq]};
    if (!__syncthreads_or(any)) {
      done = true;
      break;
    }
    double qq[4];
    jac_rounds<true>(S, t, negl, tol2, gg, qq, n <= GB ? (n < 2 ? 2 : (n + 1) & ~1) : GB, n > GB);
    double* o = Qs + 2 * bp * GLD;
    o[bq] = qq[0];
    o[GB + bq] = qq[1];
    o[GLD + bq] = qq[2];
    o[GLD + GB + bq] = qq[3];
    __syncthreads();
    // M <- M Q, tile (rows 16 Jt, columns 16 I) of each, transposed as above
    d4s om[2];
#pragma unroll
    for (int k = 0; k < 2; k++) {
      om[k] = d4s{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int kk = 0; kk < GC / 4; kk++)
        om[k] = mfma64s(Qs[(4 * kk + g) * GLD + 16 * I + i], M[k][(4 * kk + g) * GLD + 16 * Jt + i], om[k]);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 2; k++)
#pragma unroll
      for (int r = 0; r < 4; r++) M[k][(16 * I + 4 * r + g) * GLD + 16 * Jt + i] = om[k][r];
  }
  __syncthreads();
  for (int e = t; e < n * n; e += 256) {
    const int c = e / n, r = e - c * n;
    H[int64_t(c) * ldh + r] = M[0][c * GLD + r];
    J[int64_t(c) * ldj + r] = M[1][c * GLD + r];
  }
  if (t == 0 && done) state[0] = 1;
}
