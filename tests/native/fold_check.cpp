// Test helper: the folded screen of the stencil-lattice search
// (pyhea_amd/csrc/hea_screen.h: refresh_fold, fold_bound, screen_fold, the
// templates the kernel instantiates) against the oracle's sequential updates
// (oracle/hcs_oracle.cpp), and the stencil detection (hea_stencil.h).
//
//   fold_check <problem.bin> <lattices> <drift> <seed> <beta_scale>
//   fold_check --detect <problem.bin>      prints "<shell set> <edge>"
//   fold_check --steps <trials> <seed>     safe_step_within on random sequences
//
// For every unlike-species pair of random drifted lattices:
// |err(P) - err(G) - X(P)| <= 2 beta (times <beta_scale>), with beta from the
// tables' own bounds, and again after <= 8 further swaps with beta taken before
// them (fold_bound_ahead).  Prints "ok <pairs> <max ratio>" or the first
// failure, exit 1.  The problem file is
// screen_check.cpp's.
#include <stdio.h>
#include <stdlib.h>

#include <algorithm>
#include <random>
#include <string>
#include <vector>

#include "hcs_oracle.cpp"
#include "hea_screen.h"
#include "hea_stencil.h"

namespace {

constexpr int KM = 8;
struct D2 {
  double x, y;
};
struct Args {
  int N, K, S;
  int Z[HEA_MAX_S];
  double delta[HEA_MAX_S], weight[HEA_MAX_S];
};
// the templates write through const tables (pointers in the kernels)
struct TabView {
  double *E0, *R, *B;
  const double *tgt, *C, *conc;
  D2* UV;
  int idx(int s, int i, int j) const { return (s * KM + i) * KM + j; }
  int uvx(int s, int i, int j) const { return (s * KM + i) * (KM + 1) + j; }
};

bool read_all(FILE* f, void* p, size_t n) { return fread(p, 1, n, f) == n; }

}  // namespace

// Sequences of +-delta with partial sums within n steps of g end at
// fma(net, r, g) whenever safe_step_within returns r != 0: random entries and
// entries n + 3 to n + 40 steps from a binade edge, where the bound decides.
int steps_mode(long trials, uint64_t seed) {
  std::mt19937_64 rng(seed);
  std::uniform_real_distribution<double> U(0.0, 1.0);
  long fast = 0, cases = 0;
  for (long t = 0; t < trials; ++t) {
    const int n = 1 + (int)(rng() % 30), sites = 100 + (int)(rng() % 500000);
    const double delta = 1.0 / (24.0 * sites);
    const double edge = ldexp(1.0, -1 - (int)(rng() % 6));
    const double g = (t & 1) ? edge * (1.0 + U(rng))
                             : edge + ((rng() & 1) ? 1.0 : -1.0) * delta * (n + 40.0 * U(rng));
    if (!(g > delta)) continue;
    ++cases;
    const double r = safe_step_within(g, delta, n);
    if (r == 0.0) continue;
    for (int q = 0; q < 4; ++q) {
      double v = g;
      int net = 0;
      for (int i = 0; i < 4 * n; ++i) {
        int st = (q == 0) ? -1 : (q == 1) ? 1 : ((rng() & 1) ? 1 : -1);
        if (net + st > n || net + st < -n) st = -st;
        v = st > 0 ? v + delta : v - delta;
        net += st;
        ++fast;
        if (__builtin_bit_cast(uint64_t, v) !=
            __builtin_bit_cast(uint64_t, fma((double)net, r, g))) {
          printf("step: g %.17g delta %.17g n %d net %d\n", g, delta, n, net);
          return 1;
        }
      }
    }
  }
  printf("ok %ld %ld\n", cases, fast);
  return 0;
}

int main(int argc, char** argv) {
  if (argc == 4 && std::string(argv[1]) == "--steps")
    return steps_mode(atol(argv[2]), strtoull(argv[3], nullptr, 10));
  const bool detect = argc == 3 && std::string(argv[1]) == "--detect";
  if (!detect && argc != 6) return 2;
  FILE* f = fopen(argv[detect ? 2 : 1], "rb");
  if (!f) return 2;
  int32_t hdr[6];
  if (!read_all(f, hdr, sizeof hdr)) return 2;
  const int N = hdr[0], K = hdr[1], S = hdr[2];
  const int32_t Z[3] = {hdr[3], hdr[4], hdr[5]};
  int sumZ = 0;
  for (int s = 0; s < S; ++s) sumZ += Z[s];
  std::vector<int32_t> nbr((size_t)N * sumZ), counts(K);
  std::vector<double> weight(S), target((size_t)S * K * K);
  if (!read_all(f, nbr.data(), 4 * nbr.size()) || !read_all(f, counts.data(), 4 * K) ||
      !read_all(f, weight.data(), 8 * S) || !read_all(f, target.data(), 8 * target.size()))
    return 2;
  fclose(f);
  if (detect) {
    int edge = 0;
    const int lt = hea_stencil_detect(nbr.data(), N, S, Z, &edge);
    printf("%d %d\n", lt, edge);
    return 0;
  }
  const int n_lat = atoi(argv[2]), n_drift = atoi(argv[3]);
  std::mt19937_64 rng(strtoull(argv[4], nullptr, 10));
  const double beta_scale = atof(argv[5]);
  const Problem P = make_problem(N, K, S, Z, nbr.data(), counts.data(), weight.data(),
                                 target.data());
  Args A{};
  A.N = N;
  A.K = K;
  A.S = S;
  for (int s = 0; s < S; ++s) {
    A.Z[s] = Z[s];
    A.delta[s] = 1.0 / (double)(Z[s] * N);
    A.weight[s] = weight[s];
  }
  const int TAB = HEA_MAX_S * KM * KM;
  std::vector<double> E0(TAB), R(TAB), B(TAB), tgt(TAB), C(TAB), conc(KM);
  std::vector<D2> UV(HEA_MAX_S * KM * (KM + 1), D2{0.0, 0.0});
  const TabView T{E0.data(), R.data(), B.data(), tgt.data(), C.data(), conc.data(), UV.data()};
  for (int a = 0; a < K; ++a) conc[a] = (double)counts[a] / (double)N;
  for (int s = 0; s < S; ++s)
    for (int i = 0; i < K; ++i)
      for (int j = 0; j < K; ++j) {
        const double c = -A.delta[s] / (conc[i] * conc[j]);
        tgt[T.idx(s, i, j)] = target[(size_t)s * K * K + i * K + j];
        C[T.idx(s, i, j)] = c;
        UV[T.uvx(s, i, j)].y = 2.0 * weight[s] * c * c;
      }
  using PK = Pack<KM>;
  long long pairs = 0;
  double max_ratio = 0.0;
  std::vector<uint8_t> lat(N), lat2(N);
  for (int li = 0; li < n_lat; ++li) {
    int k = 0;
    for (int a = 0; a < K; ++a)
      for (int c = 0; c < counts[a]; ++c) lat[k++] = (uint8_t)a;
    std::shuffle(lat.begin(), lat.end(), rng);
    Gamma g;
    recount_gamma(P, lat.data(), g);
    for (int d = 0; d < n_drift; ++d) {
      int i = (int)(rng() % N), j = (int)(rng() % N);
      while (lat[i] == lat[j]) j = (int)(rng() % N);
      incremental(P, lat.data(), g, i, j);
    }
    double beta = 0.0;
    for (int s = 0; s < S; ++s) {
      double most = 0.0;
      for (int i = 0; i < K; ++i)
        for (int j = i; j < K; ++j) {
          refresh_fold(A, T, s, i, j, g.at(i, j, s));
          most = std::max(most, B[T.idx(s, i, j)]);
        }
      beta += most;
    }
    beta *= 2.0 * 1.01 * beta_scale;
    // the window of a round of up to 8 further swaps, then such swaps
    for (int round = 0; round < 2; ++round) {
    if (round == 1) {
      beta = 0.0;
      for (int s = 0; s < S; ++s) {
        double most = 0.0;
        for (int i = 0; i < K; ++i)
          for (int j = i; j < K; ++j)
            most = std::max(most, fold_bound_ahead(A, T, s, i, j, g.at(i, j, s), 8));
        beta += most;
      }
      beta *= 2.0 * 1.01 * beta_scale;
      for (int d = 0; d < 8; ++d) {
        int i = (int)(rng() % N), j = (int)(rng() % N);
        while (lat[i] == lat[j]) j = (int)(rng() % N);
        incremental(P, lat.data(), g, i, j);
      }
      for (int s = 0; s < S; ++s)
        for (int i = 0; i < K; ++i)
          for (int j = i; j < K; ++j) refresh_fold(A, T, s, i, j, g.at(i, j, s));
    }
    const double errG = error_of_gamma(P, g);
    for (int a1 = 0; a1 < N; ++a1)
      for (int a2 = 0; a2 < N; ++a2) {
        const int a = lat[a1], b = lat[a2];
        if (a == b) continue;
        ++pairs;
        PK::T MA[HEA_MAX_S] = {}, MB[HEA_MAX_S] = {};
        int c12[HEA_MAX_S] = {};
        for (int s = 0; s < S; ++s)
          for (int q = 0; q < Z[s]; ++q) {
            const int n1 = P.nb(a1, s, q);
            MA[s] += PK::one(lat[n1]);
            MB[s] += PK::one(lat[P.nb(a2, s, q)]);
            c12[s] += n1 == a2;
          }
        const double X = screen_fold<KM>(T, S, a, b, MA, MB, c12);
        Gamma g2 = g;
        lat2 = lat;
        incremental(P, lat2.data(), g2, a1, a2);
        const double dev = fabs(error_of_gamma(P, g2) - errG - X);
        max_ratio = std::max(max_ratio, dev / (2.0 * beta));
        if (!(dev <= 2.0 * beta)) {
          printf("bound: lattice %d pair (%d,%d): %.6g > 2 beta = %.6g\n", li, a1, a2, dev,
                 2.0 * beta);
          return 1;
        }
      }
    }
  }
  printf("ok %lld %.6g\n", pairs, max_ratio);
  return 0;
}
