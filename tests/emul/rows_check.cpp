// The 2D x-passes over blocks of neighbouring rows in the host emulation, with
// AddressSanitizer: three and six fields in, rows of many members in one block, and
// a last block that is partly empty.  Members against the FP64 oracle, the
// perturbation against a single-member context's recorded replay.  Exit status 0 =
// all passed.  TEST INFRASTRUCTURE ONLY.
#include <math.h>
#include <stdio.h>
#include <string.h>
#include <vector>
#include "oracle.h"
#include "psg.h"
#include "psg_newton.h"

typedef std::vector<double> V;

static double rel(const V &a, const V &b) {
  double m = 0, n = 0;
  for (size_t i = 0; i < a.size(); i++) { m = fmax(m, fabs(a[i] - b[i])); n = fmax(n, fabs(b[i])); }
  return m / (n > 0 ? n : 1);
}

// two steps of dt 0.005: FP64 roundings, or two increments of dt times FP32 products
static int rows_case(int nx, int ny, int batch, int prec) {
  const int steps = 2;
  const double alpha = (double)ny / nx, dt = 0.005, T = steps * dt * (1 + 1e-9), tol = prec ? 1e-6 : 1e-12;
  psg_config c;
  memset(&c, 0, sizeof c);
  c.flavour = PSG_NS2D; c.precision = prec; c.batch = batch; c.nx = nx; c.ny = ny; c.nz = 1; c.alpha = alpha;
  c.v2 = 1 / 40.0; c.dt = dt; c.force = PSG_FORCE_KOLMO; c.kf = 4.0; c.ampfor = -2.0; c.sc = 1.0;
  or_grid g;
  or_grid2(&g, nx, ny, alpha);
  const size_t n = 2 * g.nkt;
  V z[3] = {V(n), V(n), V(n)}, d(n), z1(n), dz1(n), z2(n), dz2(n), got(n);
  for (int m = 0; m < 3; m++) or_ic_ns2d_cfg(&g, 31 + m, 1.0, (orc *)z[m].data());
  or_ic_ns2d_cfg(&g, 47, 1.0, (orc *)d.data());
  or2_ctx *o = or2_create(nx, ny, alpha, c.v2, T / steps, 4, -2.0);
  V want[3] = {z[0], z[1], z[2]};
  for (V &w : want) or2_run(o, (orc *)w.data(), steps);
  or2_destroy(o);
  psg_ctx *many = nullptr, *one = nullptr;
  psg_config c1 = c;
  c1.batch = 1;
  if (psg_create(&c, &many) || psg_create(&c1, &one)) { printf("FAIL create\n"); return 1; }
  double worst = 0, pert = 0;
  // the tangent's six fields, then the plain step's three
  for (int tangent = 1; tangent >= 0; tangent--) {
    for (int m = 0; m < batch; m++) psg_set_state(many, m, z[m % 3].data());
    int rc = tangent ? psg_tangent(many, z[0].data(), d.data(), T, dt, 0, z1.data(), dz1.data()) : psg_run(many, steps);
    if (rc) { printf("FAIL run %d\n", rc); return 1; }
    for (int m = 0; m < batch; m++) {
      psg_get_state(many, m, got.data());
      worst = fmax(worst, rel(got, want[m % 3]));
    }
  }
  if (psg_tangent_many(one, z[0].data(), 1, d.data(), T, dt, 0, 0, z2.data(), dz2.data())) { printf("FAIL replay\n"); return 1; }
  pert = fmax(rel(dz1, dz2), rel(z1, z2));
  psg_destroy(many);
  psg_destroy(one);
  const bool ok = worst <= tol && pert <= 2 * tol;
  printf("%s %dx%d x %d %s: states %.2e, perturbation %.2e\n", ok ? "PASS" : "FAIL", nx, ny, batch, prec ? "fp32" : "fp64",
         worst, pert);
  fflush(stdout);
  return !ok;
}

int main() {
  int bad = 0;
  bad += rows_case(16, 16, 129, PSG_FP64);
  bad += rows_case(16, 16, 129, PSG_FP32BULK);
  bad += rows_case(512, 16, 129, PSG_FP32BULK);
  printf("%d failed\n", bad);
  return bad != 0;
}
