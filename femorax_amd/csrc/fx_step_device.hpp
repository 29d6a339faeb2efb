// The CentralDifference update of one equation (explicit_analysis.cpp:87-117, 712-722), for the
// update kernel and for the lattice kernels that run it where an equation's force is complete.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace fx {

// Point loads the fused update looks up at every equation (more take the separate kernels).
constexpr int kStepLoads = 4;

struct CdStep {
  double c2, c3;
  const double* m;
  const double* am;    // lumped alphaM mass, or null
  const double* dash;  // dampers outside the elements, or null
  double* um;          // in: U(n-1); out: U(n+1)
  const int8_t* dir;   // the DOF direction of each equation
  int32_t gdir;        // the excitation's direction, or -1
  double ag;           // its acceleration at this step's load time
  double* v;           // the recorded velocity and acceleration (in: v of the step before), or null
  double* a;
  double dt;
  int32_t nload;       // point loads P(q): f(q) -= P
  int32_t load_eq[kStepLoads];
  double load[kStepLoads];
};

// The effective ground-motion load on equation q (ground_load, explicit_analysis.cpp:48-58):
// -m(q) a_g when q acts in the excitation's direction.
__device__ inline double ground_load(const int8_t* dir, int32_t gdir, double ag, int64_t q, double mq) {
  double r = 0.0;
  if (gdir >= 0 && dir[q] == gdir) r -= mq * ag;
  return r;
}

// U(n+1) at equation q from the elements' force fq (their damping and body forces in it), U(n) = uq
// and U(n-1) = umq: R = -f - M a_g + P, U = R / (c3 m + c2 c), the dampers' force at the garbage
// velocity -c2 U(n-1).
__device__ inline double cd_next(const CdStep& g, int64_t q, double fq, double uq, double umq) {
  const double mq = g.m[q];
  for (int j = 0; j < g.nload; ++j)
    if (q == g.load_eq[j]) fq -= g.load[j];
  double cq = 0.0;
  if (g.am) cq += g.am[q];
  if (g.dash) {
    const double dq = g.dash[q];
    fq += dq * (umq * -g.c2);
    cq += dq;
  }
  const double ag = uq * (-2.0 * g.c3) + umq * g.c3;
  const double R = -fq - mq * ag + ground_load(g.dir, g.gdir, g.ag, q, mq);
  const double A = mq * g.c3 + cq * g.c2;
  return R / A;
}

// The equation's step stored: U(n+1) over U(n-1), and the recorded rates where they are asked for
// (they feed no later displacement: the dampers act at the garbage velocity).
__device__ inline void cd_store(const CdStep& g, int64_t q, double fq, double uq, double umq) {
  const double U = cd_next(g, q, fq, uq, umq);
  g.um[q] = U;
  if (!g.v) return;
  double Udot = U * 3.0;
  Udot += uq * -4.0;
  Udot += umq;
  Udot *= g.c2;
  const double Udotdot = (Udot - g.v[q]) / g.dt;
  g.v[q] = Udot;
  g.a[q] = Udotdot;
}

}  // namespace fx
