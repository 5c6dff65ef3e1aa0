// Test of the device factorisation's own checks (GPU, not part of the
// library): a Schur matrix factors, and the same matrix with one struct row
// missing where the scatter looks it up is refused, not factored without the
// entries of that row.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <stdexcept>
#include <string>

#include "devfactor.hpp"
#include "mesh.hpp"
#include "ops.hpp"

using namespace pecs;

int main() {
  Params prm;
  prm.k = 2;
  prm.dt = 5e-4;
  const SolarCellMesh m = make_solarcell_mesh(3, GeometrySpec{});
  const RefTables T(prm.k);
  const BlockSPD S = schur_matrix(m.semi, build_ldg_ops(m.semi, T, prm), 1.0);
  FrontPlan plan;
  const SupernodalFactor F = cholesky_symbolic({&S}, 4, plan);
  const PackedFactor P = pack_layout(F);
  double *fwd = nullptr, *bwd = nullptr;
  if (hipMalloc(&fwd, P.nvals * sizeof(double)) || hipMalloc(&bwd, P.nvals * sizeof(double))) return 3;
  void* handle = factor_handle_create();
  auto error = [&](const PackedFactor& Q) -> std::string {
    try {
      factor_on_device(plan, F, Q, fwd, bwd, nullptr, handle);
    } catch (const std::exception& e) {
      return e.what();
    }
    return "";
  };
  const std::string whole = error(P);
  // a coupling of the first node with a struct row: its row's number is taken
  // by the next one (rows stay ascending)
  PackedFactor Q = P;
  std::string damaged;
  for (size_t i = 0; i < plan.sb_src.size() && damaged.empty(); ++i)
    for (int e = 0; e < plan.sb_nx[i] * plan.sb_ny[i] && damaged.empty(); ++e) {
      const int p = F.perm[plan.sb_x[i] + e / plan.sb_ny[i]], q = F.perm[plan.sb_y[i] + e % plan.sb_ny[i]];
      const SNode& N = F.nodes[plan.node_of[p]];
      if (plan.sb_val[i][e] == 0.0 || q < p) continue;
      const int r = front_row(q, N.p0, N.ns, N.ms, &F.rows[N.rows_off]) - N.ns;
      if (r < 0 || r + 1 >= N.ms) continue;
      Q.rows[N.rows_off + r] = Q.rows[N.rows_off + r + 1];
      damaged = error(Q);
      if (damaged.empty()) damaged = "factored";
    }
  factor_handle_destroy(handle);
  (void)hipFree(fwd);
  (void)hipFree(bwd);
  std::printf("whole: %s\ndamaged: %s\n", whole.c_str(), damaged.c_str());
  const bool ok = whole.empty() && damaged.find("outside their fronts") != std::string::npos;
  std::printf("%s\n", ok ? "OK" : "FAIL");
  return ok ? 0 : 1;
}
