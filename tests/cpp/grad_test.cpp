// CPU test of a templated gradient kernel (chronusq_public_amd/csrc/
// eri_grad_impl.hpp) on quartets none of whose primitive pairs are left: they
// add nothing, whatever the block's LDS holds from the quartet before.
#include <cstdio>
#include <random>

#include "eri_grad_impl.hpp"

using namespace cqx;

template <int LA, int LB, int LC, int LD>
int run_case(const char *name) {
  using W = GradWave<LA, LB, LC, LD>;
  std::mt19937_64 rng(3);
  std::uniform_real_distribution<double> u(0.1, 1.0);
  const int nbc = W::K::NCA + W::K::NCB + W::K::NCC + W::K::NCD;
  PairRec bra{}, ket[2] = {};
  bra.a = 0;
  bra.b = 1;
  bra.bfb = W::K::NCA;
  for (int k = 0; k < 2; ++k) {
    ket[k].a = 2;
    ket[k].b = 3;
    ket[k].bfa = W::K::NCA + W::K::NCB;
    ket[k].bfb = ket[k].bfa + W::K::NCC;
    ket[k].pp_off = 2;
    ket[k].npp = k == 0 ? 1 : 0;  // the second has lost its primitive pairs
  }
  bra.npp = 2;
  PrimPair prims[3];
  double alpha[3];
  for (int k = 0; k < 3; ++k) {
    prims[k].p = 1.0 + u(rng);
    prims[k].rp = 1.0 / prims[k].p;
    prims[k].K = u(rng);
    for (double &x : prims[k].P) x = u(rng);
    alpha[k] = 0.5 * prims[k].p;
  }
  std::vector<double> rys(rys_tab_off(10)), X((size_t)nbc * nbc), acc[2];
  for (double &v : rys) v = 0.01 * u(rng);
  for (double &v : X) v = u(rng);
  const int atom[4] = {0, 1, 2, 3};
  GradLaunch a{};
  a.bra = &bra;
  a.ket = ket;
  a.nbra = 1;
  a.nket = 2;
  a.prims = prims;
  a.prim_alpha = alpha;
  a.rys = rys.data();
  a.shell_atom = atom;
  a.X = X.data();
  a.nmat = 1;
  a.nbc = nbc;
  a.kmask = 1;
  for (int k = 0; k < 2; ++k) {
    acc[k].assign((size_t)12 * nbc * nbc, 0.0);
    a.acc = acc[k].data();
    a.nq = 1 + k;  // the first quartet alone, then both
    host_wave::run(W::NT, [&](int) { grad_wave_kernel<LA, LB, LC, LD>(a); });
  }
  double most = 0.0, worst = 0.0;
  for (size_t e = 0; e < acc[0].size(); ++e) {
    most = std::max(most, std::fabs(acc[0][e]));
    worst = std::max(worst, std::fabs(acc[1][e] - acc[0][e]));
  }
  const bool ok = most > 0.0 && worst == 0.0;
  std::printf("%s %s %.1e of %.1e\n", name, ok ? "ok" : "FAIL", worst, most);
  return ok ? 0 : 1;
}

int main() {
  return run_case<1, 1, 1, 1>("(pp|pp)") + run_case<2, 1, 2, 1>("(dp|dp)") + run_case<2, 2, 2, 1>("(dd|dp)");
}
