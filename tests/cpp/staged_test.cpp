// CPU test of the staged J/K digestion (chronusq_public_amd/csrc/
// digest_staged.hpp) for waves whose quartets belong to two molecules of
// different sizes: every plane of a molecule ends at a page that may not be
// touched, so a read through the other molecule's planes ends the program.
// Prints one line per case and exits non-zero on a wrong sum.
#include <sys/mman.h>
#include <unistd.h>

#include <cstdio>
#include <cstring>
#include <random>

#include "digest_staged.hpp"

using namespace cqx;

namespace {

// n doubles that end at an inaccessible page
double *guarded(size_t n) {
  const size_t page = (size_t)sysconf(_SC_PAGESIZE), len = (n * sizeof(double) + page - 1) / page * page;
  char *p = static_cast<char *>(mmap(nullptr, len + page, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0));
  if (p == MAP_FAILED || mprotect(p + len, page, PROT_NONE)) std::exit(2);
  return reinterpret_cast<double *>(p + len) - n;
}

using K = Cls<2, 1, 2, 1>;
constexpr int kQuartets = 4, kXCap = 512;

// one tile: quartet q of molecule mols[q]; counts[k] planes of each kind
int run_case(const char *name, const int (&nbc)[2], const int (&mols)[kQuartets], const int (&counts)[4], int nq) {
  std::printf("%s ", name);
  std::fflush(stdout);
  std::mt19937_64 rng(7);
  std::normal_distribution<double> normal;
  PlaneSet ps{};
  MolPlanes mp[2] = {};
  int slot = 0;
  for (int k = 0; k < 4; ++k) {
    ps.kstart[k] = slot;
    ps.kcount[k] = counts[k];
    ps.kps[k] = 1;
    while (ps.kps[k] < counts[k]) ps.kps[k] *= 2;
    for (int p = 0; p < counts[k]; ++p, ++slot) {
      ps.mats |= (unsigned long long)(slot & 7) << (4 * slot);
      if (k == kKHer && (p & 1)) ps.negs |= 1u << slot;  // the imaginary part of a conjugated density
    }
  }
  std::vector<std::vector<double>> ref[2];
  for (int m = 0; m < 2; ++m) {
    mp[m].nbc = nbc[m];
    ref[m].resize(4);
    for (int k = 0; k < 4; ++k) {
      if (!counts[k]) continue;
      const size_t n = (size_t)nbc[m] * nbc[m] * ps.kps[k];
      double *x = guarded(n), *a = guarded(n);
      for (size_t e = 0; e < n; ++e) x[e] = normal(rng);
      std::memset(a, 0, n * sizeof(double));
      mp[m].kx[k] = x;
      mp[m].ka[k] = a;
      ref[m][k].assign(n, 0.0);
    }
  }
  ps.n = slot;
  ps.nmol = 2;
  ps.mols = mp;
  std::vector<double> I((size_t)kQuartets * K::NC), X(kXCap);
  for (double &v : I) v = normal(rng);
  int bf[kQuartets][4];
  unsigned mask[kQuartets];
  for (int q = 0; q < kQuartets; ++q) {
    // the second half at the very end of its molecule's functions
    for (int r = 0; r < 4; ++r) {
      const int last = nbc[mols[q]] - K::n(r);
      bf[q][r] = q >= nq / 2 ? last : (int)(rng() % (unsigned)(last + 1));
    }
    mask[q] = q == 0 ? 0xFFu : 0xFEu;  // contraction 0 screened out of the others
  }
  host_wave::run(64, [&](int lane) { digest_staged<K, kXCap>(I.data(), bf, mask, mols, nq, ps, X.data(), lane); });
  // the same updates term by term
  const int st[4] = {K::NCB * K::NCC * K::NCD, K::NCC * K::NCD, K::NCD, 1};
  for (int q = 0; q < nq; ++q)
    for (int k = 0; k < 4; ++k)
      for (int p = 0; p < counts[k]; ++p) {
        const int s = ps.kstart[k] + p, S = ps.kps[k], N = nbc[mols[q]];
        if (!((mask[q] >> ((ps.mats >> (4 * s)) & 15)) & 1u)) continue;
        const double coef = (k == kJHer ? 1.0 : 0.5) * (k == kKHer && ((ps.negs >> s) & 1u) ? -1.0 : 1.0);
        for (int t = 0; t < kDigestTerms.n[k]; ++t) {
          const signed char *role = kDigestTerms.t[k][t];
          int e[4];
          for (e[0] = 0; e[0] < K::NCA; ++e[0])
            for (e[1] = 0; e[1] < K::NCB; ++e[1])
              for (e[2] = 0; e[2] < K::NCC; ++e[2])
                for (e[3] = 0; e[3] < K::NCD; ++e[3]) {
                  const double v = I[(size_t)q * K::NC + e[0] * st[0] + e[1] * st[1] + e[2] * st[2] + e[3]];
                  auto at = [&](int r, int c) {
                    return ((size_t)(bf[q][r] + e[r]) + (size_t)(bf[q][c] + e[c]) * N) * S + p;
                  };
                  ref[mols[q]][k][at(role[0], role[1])] += coef * v * mp[mols[q]].kx[k][at(role[2], role[3])];
                }
        }
      }
  // Hermitian kinds may store the transposed element: compare A + A^H
  double worst = 0.0;
  for (int m = 0; m < 2; ++m)
    for (int k = 0; k < 4; ++k)
      for (int p = 0; p < counts[k]; ++p)
        for (int i = 0; i < nbc[m]; ++i)
          for (int j = 0; j < nbc[m]; ++j) {
            const size_t ij = ((size_t)i + (size_t)j * nbc[m]) * ps.kps[k] + p;
            const size_t ji = ((size_t)j + (size_t)i * nbc[m]) * ps.kps[k] + p;
            const bool her = k == kJHer || k == kKHer;
            const double sg = !her ? 0.0 : (ps.negs >> (ps.kstart[k] + p)) & 1u ? -1.0 : 1.0;
            const double *a = mp[m].ka[k];
            worst = std::max(worst, std::fabs(a[ij] + sg * a[ji] - ref[m][k][ij] - sg * ref[m][k][ji]));
          }
  // sums of a few hundred products of order one in another order
  const bool ok = worst < 1e-11;
  std::printf("%s %.1e\n", ok ? "ok" : "FAIL", worst);
  return ok ? 0 : 1;
}

}  // namespace

int main() {
  int bad = 0;
  const int large_first[2] = {61, 25}, small_first[2] = {25, 61};
  const int both[kQuartets] = {0, 1, 0, 1}, swapped[kQuartets] = {1, 0, 1, 0}, one[kQuartets] = {1, 1, 1, 1};
  const int rhf[4] = {1, 1, 0, 0}, cplx[4] = {1, 2, 0, 0}, nonher[4] = {0, 0, 1, 1}, wide[4] = {1, 8, 0, 0};
  for (const auto &nbc : {large_first, small_first}) {
    const char *o = nbc[0] > nbc[1] ? "large molecule first:" : "small molecule first:";
    std::printf("%s\n", o);
    bad += run_case("real J/K, one molecule", {nbc[0], nbc[1]}, one, rhf, 2);
    bad += run_case("real J/K", {nbc[0], nbc[1]}, both, rhf, 2);
    bad += run_case("real J/K, swapped", {nbc[0], nbc[1]}, swapped, rhf, 2);
    bad += run_case("real J/K, four quartets", {nbc[0], nbc[1]}, both, rhf, 4);
    bad += run_case("complex K", {nbc[0], nbc[1]}, both, cplx, 2);
    bad += run_case("non-Hermitian", {nbc[0], nbc[1]}, both, nonher, 2);
    bad += run_case("more planes than are staged", {nbc[0], nbc[1]}, both, wide, 2);
  }
  return bad ? 1 : 0;
}
