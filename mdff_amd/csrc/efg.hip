// efg.hip -- electric field gradient at the ions (doefg) for gfx950.
//
// Reference: multipole_ES (src/ewald.f90:49-314) with do_efg, its parts
//   real space   multipole_ES_dir  src/ewald_dir.f90:543-546, 577-582
//   reciprocal   multipole_ES_rec  src/ewald_rec.f90:116-148 (S(k)),
//                                  :209-216 (k_a k_b A Re(S e^{-ik.r})), :302, :351
//   self         src/ewald.f90:214-216; total x coul_unit :231
// and its copy into efg_t (src/engforce_driver.f90:171).
//
// Every part runs in FP64 whatever the precision form.  The reciprocal part
// is the second moments Re(W e) n n that the force evaluation's gather forms
// for dipole forces: with doefg it forms them for charges too, and one kernel
// here turns them into Cartesian components, adds the other parts and scales
// by coul_unit into the reference layout efg(3,3,natm); the reciprocal part
// only on the upper triangle and the diagonal, as the reference fills it.
// (Its own sums over k and atoms with a cos/sin per term took 660 of the 930
// us of a 4,096-ion evaluation with 22,050 k vectors.)
#include "common.h"

namespace {

// efg(3,3,n) column-major per atom.  dir: 6 per atom or null (no doefg: the
// self term alone); rf: the second moments, scaled by 2 (half mesh) x 4 pi / V.
__global__ void __launch_bounds__(256) k_efg_combine(int n, const double* __restrict__ dir, RecFinal rf,
                                                     const double* __restrict__ q, double self2, double coul,
                                                     double* __restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  constexpr int up[6] = {0, 4, 8, 3, 6, 7};   // (1,1) (2,2) (3,3) (1,2) (1,3) (2,3)
  constexpr int lo[3] = {1, 2, 5};            // (2,1) (3,1) (3,2) of xy, xz, yz
  constexpr int ra[6] = {0, 1, 2, 0, 0, 1}, rb[6] = {0, 1, 2, 1, 2, 2};
  double* o = out + 9 * (size_t)i;
  double h[3][3] = {};
  if (dir) {
    double v[9], g[3];
    rec_final_moments(rf, i, v, g);
    const double m[3][3] = {{v[3], v[6], v[7]}, {v[6], v[4], v[8]}, {v[7], v[8], v[5]}};
    double t[3][3];                            // B M
    for (int a = 0; a < 3; ++a)
      for (int e = 0; e < 3; ++e) t[a][e] = rf.b[a] * m[0][e] + rf.b[3 + a] * m[1][e] + rf.b[6 + a] * m[2][e];
    const double sc = 2.0 * rf.fpi_V * (2.0 * MDFF_PI) * (2.0 * MDFF_PI);
    for (int a = 0; a < 3; ++a)
      for (int b = a; b < 3; ++b) h[a][b] = sc * (t[a][0] * rf.b[b] + t[a][1] * rf.b[3 + b] + t[a][2] * rf.b[6 + b]);
  }
  for (int v = 0; v < 6; ++v) {
    const double d = dir ? dir[6 * (size_t)i + v] : 0.0;
    const double self = v < 3 ? -self2 * q[i] : 0.0;
    o[up[v]] = (d + h[ra[v]][rb[v]] + self) * coul;
    if (v >= 3) o[lo[v - 3]] = d * coul;
  }
}

}  // namespace

int efg_alloc(mdff_ctx* c) {
  if (c->efg) return MDFF_OK;
  const int n = c->n;
  // every entry is written by each efg_eval (its only caller)
  HIP_TRY(c, hipMalloc((void**)&c->efg, sizeof(double) * 9 * (size_t)n));
  if (!c->d.doefg || !c->d.lcoulomb) return MDFF_OK;
  HIP_TRY(c, hipMalloc((void**)&c->efg_dir, sizeof(double) * 6 * (size_t)n));
  return MDFF_OK;
}

void efg_free(mdff_ctx* c) {
  for (double* p : {c->efg, c->efg_dir})
    if (p) (void)hipFree(p);
  c->efg = c->efg_dir = nullptr;
}

// efg_t of a Coulomb evaluation whose atoms, lists and dipoles (c->mu) are
// current: with doefg the three parts, otherwise the self term alone.
int efg_eval(mdff_ctx* c) {
  MDFF_TRY(efg_alloc(c));
  const int n = c->n;
  const double alpha2 = c->alpha * c->alpha;
  const double selfa = c->alpha / sqrt(MDFF_PI), selfa2 = 2.0 * selfa * alpha2 / 3.0;
  if (c->d.doefg) MDFF_TRY(realspace_efg(c, c->efg_dir));
  // c->rfin: the force evaluation's moments, described for its force kernel
  hipLaunchKernelGGL(k_efg_combine, dim3(div_up(n, 256)), dim3(256), 0, c->stream, n,
                     c->d.doefg ? c->efg_dir : nullptr, c->rfin, c->q, 2.0 * selfa2, c->d.coul_unit, c->efg);
  HIP_TRY(c, hipGetLastError());
  return MDFF_OK;
}
