/* The FP64 Riemann solvers of rmhd_device.hpp at n interfaces normal to x, on the host: the
 * sweeps' common path (lean) and the full solver. rc: 0, an error, or kHlldDefer = 100 where
 * the common path hands the interface to the full solver (its flux is then not final). */
#include "rmhd_device.hpp"

using namespace maragpu;

extern "C" {

void lean(int solver, long n, const double *pl, const double *pr, double gamma, double pfloor, double *f, int *rc,
          double *lam, int *steps)
{
  PhysParams pp = {};
  pp.gamma = gamma;
  pp.pfloor = pfloor;
  pp.g1 = gamma / (gamma - 1.0);
  pp.gamf = (gamma - 1.0) / gamma;
  pp.igamma = 1.0 / gamma;
#pragma omp parallel for
  for (long i = 0; i < n; ++i) {
    const double *l = pl + 8 * i, *r = pr + 8 * i;
    FluxCounters fc = {0, 0, 0, 0};
    auto store = [&](int q, double v) { f[8 * i + q] = v; };
    lam[i] = 0.0;
    rc[i] = solver == RIEMANN_HLLD ? riemann_hlld_lean(l, r, pp, lam[i], fc, store)
          : solver == RIEMANN_HLLC ? riemann_hllx_lean<RIEMANN_HLLC>(l, r, pp, lam[i], store)
                                   : riemann_hllx_lean<RIEMANN_HLL>(l, r, pp, lam[i], store);
    steps[i] = fc.newton_iters;
  }
}

void full(int solver, long n, const double *pl, const double *pr, double gamma, double pfloor, double *f, int *rc,
          double *lam, int *steps)
{
#pragma omp parallel for
  for (long i = 0; i < n; ++i) {
    const double *l = pl + 8 * i, *r = pr + 8 * i;
    FluxCounters fc = {0, 0, 0, 0};
    lam[i] = 0.0;
    rc[i] = solver == RIEMANN_HLLD ? riemann_hlld<double, 1>(l, r, f + 8 * i, gamma, pfloor, lam[i], fc)
          : solver == RIEMANN_HLLC ? riemann_hllc<double, 1>(l, r, f + 8 * i, gamma, lam[i])
                                   : riemann_hll<double, 1>(l, r, f + 8 * i, gamma, lam[i]);
    steps[i] = fc.newton_iters;
  }
}

/* the predictor's flux of a physical state (plm-muscl) and the reference's, from its conserved state */
void side_flux(long n, const double *p, double gamma, double *lean_f, double *full_f)
{
  for (long i = 0; i < n; ++i) {
    const double *P = p + 8 * i;
    side_flux_lean(P, gamma / (gamma - 1.0), lean_f + 8 * i);
    double U[8], a, b;
    prim_to_cons(P, U, gamma - 1.0);
    flux_and_eigenvalues<double, 1, false>(U, P, full_f + 8 * i, a, b, gamma);
  }
}

/* plm at the face ahead of n values (behind, centre, ahead), in general and as the sweeps that
 * hand on take it, in FP64 and FP32 */
void plm_ahead(long n, const double *v, double theta, double *d, double *d_hand_on, float *f, float *f_hand_on)
{
  for (long i = 0; i < n; ++i) {
    const double a = v[3 * i], b = v[3 * i + 1], c = v[3 * i + 2];
    d[i] = plm<double>(a, b, c, 1.0, theta);
    d_hand_on[i] = plm<double, true>(a, b, c, 1.0, theta);
    f[i] = plm<float>((float)a, (float)b, (float)c, 1.0f, (float)theta);
    f_hand_on[i] = plm<float, true>((float)a, (float)b, (float)c, 1.0f, (float)theta);
  }
}

/* the Jiang-Shu reconstructions of the lean sweeps from n values v[-2..3], and the general ones:
 * both states of the interface, and the finite-difference flux from both sides */
void weno5(long n, const double *v, double *lean_f, double *full_f)
{
  for (long i = 0; i < n; ++i) {
    const double *a = v + 6 * i;
    double *l = lean_f + 4 * i, *f = full_f + 4 * i;
    weno5_js_pair(a[0], a[1], a[2], a[3], a[4], a[5], l[0], l[1]);
    l[2] = weno5_js_fd(a[0], a[1], a[2], a[3], a[4]);
    l[3] = weno5_js_fd(a[5], a[4], a[3], a[2], a[1]);
    f[0] = weno5<double, true>(a[0], a[1], a[2], a[3], a[4], IS_JS96, 0.0);
    f[1] = weno5<double, false>(a[1], a[2], a[3], a[4], a[5], IS_JS96, 0.0);
    f[2] = weno5<double, true, true>(a[0], a[1], a[2], a[3], a[4], IS_JS96, 0.0);
    f[3] = weno5<double, false, true>(a[1], a[2], a[3], a[4], a[5], IS_JS96, 0.0);
  }
}

}
