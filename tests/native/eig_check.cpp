// Residuals of eig.hpp's eigenpairs on the host (one lane), for random and special matrices:
// |A v - lambda v| within 64 n eps |A| for unit v, the trace kept, conjugate pairs together.
#include <complex>
#include <cstdio>
#include <random>
#include <vector>

#include "eig.hpp"

typedef std::complex<double> cd;

static bool check(const std::vector<double>& A, int n, const char* what) {
  std::vector<double> H(A), Z(n * n), E(n * n), wr(n), wi(n), ort(n), V(2 * n * (n + 3));
  const eig::Serial one;
  const int ld = n + 3;
  if (eig::real_eig(one, H.data(), Z.data(), E.data(), wr.data(), wi.data(), ort.data(), n) != 0) {
    std::printf("%s n = %d: no convergence\n", what, n);
    return false;
  }
  eig::normalise(one, Z.data(), wi.data(), n, V.data(), ld);
  double norm = 0, tr = 0, sum = 0;
  for (int i = 0; i < n; i++) {
    tr += A[i * n + i];
    sum += wr[i];
    for (int j = 0; j < n; j++) norm += A[i * n + j] * A[i * n + j];
  }
  norm = std::sqrt(norm);
  const double tol = 64 * n * 2.220446049250313e-16 * norm;
  if (std::fabs(tr - sum) > tol) return std::printf("%s n = %d: trace %g, sum %g\n", what, n, tr, sum), false;
  for (int j = 0; j < n; j++) {
    if (wi[j] > 0 && !(j + 1 < n && wr[j + 1] == wr[j] && wi[j + 1] == -wi[j]))
      return std::printf("%s n = %d: %d has no conjugate beside it\n", what, n, j), false;
    double r2 = 0, v2 = 0;
    for (int i = 0; i < n; i++) {
      auto v = [&](int k) { return cd(V[2 * (k * ld + j)], V[2 * (k * ld + j) + 1]); };
      cd s = 0;
      for (int k = 0; k < n; k++) s += A[i * n + k] * v(k);
      r2 += std::norm(s - cd(wr[j], wi[j]) * v(i));
      v2 += std::norm(v(i));
    }
    if (!(std::sqrt(r2) <= tol) || !(std::fabs(v2 - 1) <= 1e-12))
      return std::printf("%s n = %d: pair %d residual %g (%g), |v|^2 %g\n", what, n, j, std::sqrt(r2), tol, v2), false;
  }
  return true;
}

int main() {
  std::mt19937_64 g(5);
  std::normal_distribution<double> N;
  bool ok = true;
  for (int n = 1; n <= 40; n++) {
    std::vector<double> A(n * n), T(n * n), S(n * n), C(n * n), B(n * n);
    for (int i = 0; i < n; i++)
      for (int j = 0; j < n; j++) {
        A[i * n + j] = N(g);
        T[i * n + j] = j > i ? N(g) : j == i ? i + 1.0 : 0.0;
        S[i * n + j] = i <= j ? N(g) : S[j * n + i];
        C[i * n + j] = i == (j + 1) % n ? 1.0 : 0.0;
        B[i * n + j] = N(g) * std::pow(10.0, 0.2 * (i % 5));
      }
    ok = check(A, n, "random") && check(T, n, "triangular") && check(S, n, "symmetric") && check(C, n, "cyclic") &&
         check(B, n, "graded") && ok;
  }
  std::puts(ok ? "eig check passed" : "eig check failed");
  return ok ? 0 : 1;
}
