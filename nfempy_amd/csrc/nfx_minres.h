// The scalar recurrence of preconditioned MINRES (Paige-Saunders, as in SciPy's minres), shared by the
// launch-per-step kernels (nfx_krylov.hip) and the kernels that keep a whole solve resident.
#pragma once

#include "nfx_common.h"

namespace nfx {

struct MinresState {
  double beta, oldb, alfa, beta1;
  double dbar, epsln, oldeps, phibar, cs, sn;
  double delta, denom, phi;
  double s, ratio;  // 1/beta and beta/oldb for the next A kernel
  double rnorm2;    // scratch for norms
  double bnorm2;
  int stop;
  int pad;
};

// Scalar step of iteration k: beta_k, and the Givens rotation of iteration k-1.
__device__ __forceinline__ void minres_scalars(const MinresState& in, MinresState& out,
                                               double beta, int first) {
  out = in;
  if (first) {
    out.beta1 = beta;
    out.beta = beta;
    out.oldb = 0;
    out.alfa = 0;
    out.dbar = 0;
    out.epsln = 0;
    out.oldeps = 0;
    out.phibar = beta;
    out.cs = -1;
    out.sn = 0;
    out.delta = 0;
    out.denom = 0;
    out.phi = 0;
    out.s = beta > 0 ? 1.0 / beta : 0.0;
    out.ratio = 0;
    out.stop = beta > 0 ? 0 : 1;
    return;
  }
  const double alfa = in.alfa;
  const double oldb = in.beta;
  const double oldeps = in.epsln;
  const double delta = in.cs * in.dbar + in.sn * alfa;
  const double gbar = in.sn * in.dbar - in.cs * alfa;
  const double epsln = in.sn * beta;
  const double dbar = -in.cs * beta;
  double gamma = hypot(gbar, beta);
  if (gamma < 1e-300) gamma = 1e-300;
  out.oldb = oldb;
  out.beta = beta;
  out.oldeps = oldeps;
  out.delta = delta;
  out.epsln = epsln;
  out.dbar = dbar;
  out.cs = gbar / gamma;
  out.sn = beta / gamma;
  out.phi = out.cs * in.phibar;
  out.phibar = out.sn * in.phibar;
  out.denom = 1.0 / gamma;
  out.s = beta > 0 ? 1.0 / beta : 0.0;
  out.ratio = oldb > 0 ? beta / oldb : 0.0;
  if (!(beta > 0)) out.stop = 1;
}

// The update of iteration k - 1 from the scalars that minres_scalars left for it, in FP32: w from z of that
// iteration and the two w before it, x += phi w.
struct MinresStep {
  float sprev, oldeps, delta, denom, phi;
  __device__ __forceinline__ explicit MinresStep(const MinresState& st)
      : sprev(st.oldb > 0 ? (float)(1.0 / st.oldb) : 0.f),
        oldeps((float)st.oldeps),
        delta((float)st.delta),
        denom((float)st.denom),
        phi((float)st.phi) {}
  __device__ __forceinline__ float w(float z, float wa, float wb) const {
    return (z * sprev - oldeps * wa - delta * wb) * denom;
  }
};

}  // namespace nfx
