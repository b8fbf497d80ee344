// Pairs of cells that the source lists hold, counted on the host from the same
// tables, for the CPU test of the lists' bound.
#include <cmath>
#include <vector>

#include "../../adaptive-multiresolution-dg_amd/csrc/fiber.hpp"
#include "../../adaptive-multiresolution-dg_amd/csrc/setup.hpp"

using namespace adg;

// table 0 point values, 1 flux and penalty, 2 constant coefficients (both
// signs); family 0 Lagrange, 1 Hermite (m = 3).  out: pairs with a block that
// is not zero outside the relation of the sweep-by-sweep form; for every level,
// the most sources up to a target's own level (n + 1 counts), then all pairs.
extern "C" int list_pairs(int table, int family, int k, int m, int n, long* out) {
  const Basis1D alpt(BasisKind::Alpert, k, n);
  const Basis1D intp(family ? BasisKind::Hermite : BasisKind::Lagrange, family ? 3 : m, n);
  const int ns = 1 << n, k1 = k + 1, m1 = m + 1;
  std::vector<char> nz(static_cast<size_t>(ns) * ns, 0);  // [target][source]
  auto add = [&](const std::vector<double>& t, int pf1, int pt1) {
    for (int s = 0; s < ns * pf1; ++s)
      for (int c = 0; c < ns * pt1; ++c)
        if (t[static_cast<size_t>(s) * ns * pt1 + c] != 0.) nz[static_cast<size_t>(c / pt1) * ns + s / pf1] = 1;
  };
  if (table == 0) {
    add(family ? alpt_at_herm_points(alpt, intp) : alpt_at_lagr_points(alpt, intp), k1, m1);
  } else {
    const OperatorTables aa(alpt, alpt);
    if (table == 1) {
      const OperatorTables la(intp, alpt);
      std::vector<double> f(la.ulft_vjp.size());
      for (size_t i = 0; i < f.size(); ++i) f[i] = la.ulft_vjp[i] + la.urgt_vjp[i];
      add(f, m1, k1);
      add(aa.ujp_vjp, k1, k1);
    } else {
      add(linear_operator_table(aa, 0.7), k1, k1);
      add(linear_operator_table(aa, -1.3), k1, k1);
    }
  }
  for (int l = 0; l <= n + 2; ++l) out[l] = 0;
  for (int st = 0; st < ns; ++st) {
    std::vector<char> rel(ns, 0);
    for_each_related(st, n, table != 0, LU_FULL, [&](int s) { rel[s] = 1; });
    const int lt = slot_level(st);
    long up = 0;
    for (int s = 0; s < ns; ++s) {
      if (!nz[static_cast<size_t>(st) * ns + s]) continue;
      if (!rel[s]) {
        if (table == 0) continue;  // (those lists hold nested cells only)
        ++out[0];
      }
      if (slot_level(s) <= lt) ++up;
      ++out[n + 2];
    }
    if (up > out[1 + lt]) out[1 + lt] = up;
  }
  return ns;
}
