// Internal force of elastic stdBrick batches and the explicit CentralDifference and
// ExplicitDifference loops.
//
// For ElasticIsotropic the element force is linear: f = K u + C v - F_body (std_brick.hpp:
// 493-543 with element_operator's Factors). stdBrick lattices of 4- and 8-deep tiles form it in one
// tile pass (launch_box_force); the others run the operator kernels (K u, and C v with the operator
// coefficients (0, 1, 0)) plus a combine kernel, with F_body a vector built once per batch. The
// CentralDifference step (explicit_analysis.cpp:87-117, 712-722) is one device-resident loop:
// per step the force at the garbage velocity v_e = -c2 u(n-1) (where the elements damp), the
// point loads, and one update per equation that forms R = -f - M a_g + P, solves the diagonal
// system (c3 M + c2 C) U = R and writes U and, where they are asked for, the recorded velocity
// and acceleration: inside the tile pass on a lattice (up to kStepLoads point loads, no nodal
// damping), else in kernels of their own. U goes into u(n-1)'s buffer and the two buffers swap
// roles, so the update writes 3 vectors, not 4. ExplicitDifference (explicit_analysis.cpp:60-85) runs its
// predictor, the force at the predicted velocity and one fused update (a = R / m, the recorded
// velocity). Both add the ground-motion load of a uniform excitation (:48-58).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "fx_internal.hpp"
#include "fx_kernels.hpp"
#include "fx_step_device.hpp"

namespace fx {

namespace {

constexpr int kThreads = 256;

inline unsigned blocks_for(int64_t n) { return static_cast<unsigned>((n + kThreads - 1) / kThreads); }

__global__ void scale_kernel(int32_t n, double s, const double* __restrict__ x, double* __restrict__ y) {
  const int32_t q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q < n) y[q] = x[q] * s;
}

// f = Ku (+ Cv) - F_body
__global__ void force_combine_kernel(int32_t n, const double* __restrict__ ku, const double* __restrict__ cv,
                                     const double* __restrict__ body, double* __restrict__ f) {
  const int32_t q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n) return;
  double v = ku[q];
  if (cv) v += cv[q];
  if (body) v -= body[q];
  f[q] = v;
}

struct PointLoads {
  int32_t n;
  int32_t eq[kMaxPointLoads];
  double val[kMaxPointLoads];
};

// f(q) -= P(q): the point loads join the residual R = -f + P
__global__ void point_load_kernel(PointLoads p, double* f) {
  if (threadIdx.x == 0 && blockIdx.x == 0)
    for (int j = 0; j < p.n; ++j) f[p.eq[j]] -= p.val[j];
}

struct CdArgs {
  int32_t n;
  double dt;
  const double* f;     // K u (+ loads folded in)
  const double* fd;    // C v_e of the elements, or null
  const double* body;  // F_body, or null
  const double* u;     // U(n)
  double* v;
  double* a;
  CdStep s;
};

__global__ __launch_bounds__(kThreads) void cd_update_kernel(CdArgs g) {
  const int32_t q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= g.n) return;
  double fq = g.f[q];
  if (g.fd) fq += g.fd[q];
  if (g.body) fq -= g.body[q];
  cd_store(g.s, q, fq, g.u[q], g.s.um[q]);
}

// ExplicitDifference newStep (ed_predict, explicit_analysis.cpp:60-68): vh += dt a; u += dt vh.
__global__ __launch_bounds__(kThreads) void ed_predict_kernel(int32_t n, double dt, double* __restrict__ u,
                                                              double* __restrict__ vh, const double* __restrict__ a) {
  const int32_t q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n) return;
  vh[q] += a[q] * dt;
  u[q] += vh[q] * dt;
}

// ExplicitDifference solve and update (ed_correct, :70-85): a(n+1) = R / m with R = -f + the
// ground load; the recorded velocity vh + (dt/8)(3 a(n+1) + a(n)). The force f carries the
// elements' damping at vh; dampers outside the elements add dash * vh to it (no tangent term:
// the scheme is explicit in the velocity).
__global__ __launch_bounds__(kThreads) void ed_correct_kernel(CdArgs g) {
  const int32_t q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= g.n) return;
  const double mq = g.s.m[q], vh = g.s.um[q];
  double fq = g.f[q];
  if (g.fd) fq += g.fd[q];
  if (g.body) fq -= g.body[q];
  if (g.s.dash) fq += g.s.dash[q] * vh;
  const double R = -fq + ground_load(g.s.dir, g.s.gdir, g.s.ag, q, mq);
  const double a_new = R / mq;
  const double t = 3.0 * a_new + g.a[q];
  g.v[q] = vh + t * (g.dt * 0.125);
  g.a[q] = a_new;
}

}  // namespace

bool elements_damp(const fx_batch* b) {
  for (const DevParam& p : b->host_params)
    if (p.alphaM != 0.0 || p.betaK != 0.0 || p.betaKinit != 0.0 || p.betaKcomm != 0.0) return true;
  return false;
}

int force64(fx_batch* b, const double* u, const double* v, double* f, double* scratch) {
  if (b->pimy) {  // the return map (and the damping force at v)
    if (int rc = pimy_force64(b, u, v, f, false)) return rc;
  } else if (box_forms_force(b)) {
    if (int rc = launch_box_force(b, u, v && elements_damp(b) ? v : nullptr, 1.0, f, 0, nullptr)) return rc;
  } else {
    const int32_t n = b->neq;
    if (int rc = elements_apply64(b, fx_coeffs{1.0, 0.0, 0.0, 0}, u, f)) return rc;
    const double* cv = nullptr;
    if (v && elements_damp(b)) {
      if (int rc = elements_apply64(b, fx_coeffs{0.0, 1.0, 0.0, 0}, v, scratch)) return rc;
      cv = scratch;
    }
    if (cv || b->body)
      hipLaunchKernelGGL(force_combine_kernel, dim3(blocks_for(n)), dim3(kThreads), 0, b->ctx->stream, n, f, cv,
                         b->body, f);
    FX_HIP(b->ctx, hipGetLastError());
  }
  // the nodal masses' Rayleigh damping force alphaM m v (internal_force.cpp:366-374)
  if (v && b->nodal_am) return nodal_damping_force64(b, v, f);
  return FX_OK;
}

int cd_run(fx_batch* b, const fx_cd_desc& d, double* u, double* um, double* v, double* a) {
  fx_ctx* ctx = b->ctx;
  const int32_t n = b->neq;
  if (n == 0 || d.nsteps <= 0) return FX_OK;
  double* W = b->work;
  const size_t N = static_cast<size_t>(n);
  // state in the solver numbering
  double *U = u, *Um = um, *V = v, *Acc = a, *dash = const_cast<double*>(d.dash);
  if (b->internal) {
    U = W;
    Um = W + N;
    V = W + 2 * N;
    Acc = W + 3 * N;
    if (d.dash) dash = W + 6 * N;
    if (int rc = to_internal_all(b, VectorPairs{{{u, U}, {um, Um}, {v, V}, {a, Acc}, {d.dash, d.dash ? dash : nullptr}}})) return rc;
  }
  double* f = W + 4 * N;
  double* ve = W + 5 * N;
  double* fd = b->internal ? W + 7 * N : W + 6 * N;
  // the elements' damping force at the garbage velocity: by the operator (C v_e) for elastic
  // batches, inside the return-map force for PIMY batches
  // (the nodal masses' alphaM term joins the operator's, or follows the return-map force)
  const bool pdamp = b->pimy && elements_damp(b);
  const bool edamp = elements_damp(b) || b->nodal_am, damp = !b->pimy && edamp;
  const bool ed = d.scheme == 1;  // ExplicitDifference: um holds the element velocity vh
  const double c2 = 0.5 / d.dt, c3 = 1.0 / (d.dt * d.dt);
  // the excitation, evaluated where the reference's stage loop evaluates its loads: at t(n) for
  // CentralDifference, at t(n+1) for ExplicitDifference (explicit_analysis.cpp:699-722)
  int32_t loc = d.ground_series && d.ground_series->loc ? *d.ground_series->loc : 0;
  double time = d.time;
  auto ground_at = [&](int32_t k, double t) {
    if (d.ground_dir < 0) return 0.0;
    if (d.ground_series) return series_value(*d.ground_series, d.ground_factor, t, loc);
    return d.ground_accel[k];
  };
  PointLoads pl{};
  pl.n = d.nload;
  for (int j = 0; j < d.nload; ++j) pl.eq[j] = b->internal ? b->internal_of[d.load_eq[j]] : d.load_eq[j];
  CdArgs g{};
  g.n = n;
  g.dt = d.dt;
  g.f = f;
  g.fd = damp ? fd : nullptr;
  g.body = b->pimy ? nullptr : b->body;  // the return-map force carries the body force
  g.s.c2 = c2;
  g.s.c3 = c3;
  g.s.dt = d.dt;
  g.s.m = b->lumped_m;
  g.s.am = b->lumped_am;
  g.s.dash = dash;
  g.s.dir = b->eq_dir_dev;
  g.s.gdir = d.ground_dir;
  // node recorders after every step (explicit_analysis.cpp:724-731): u and the recorded v, a
  const bool rec = recorder_active(d.recorder), rec_rates = recorder_reads_rates(d.recorder);
  const int32_t* rmap = nullptr;
  if (rec)
    if (int rc = batch_internal_map(b, &rmap)) return rc;
  if (ed) {
    double* VH = Um;
    for (int32_t k = 0; k < d.nsteps; ++k) {
      hipLaunchKernelGGL(ed_predict_kernel, dim3(blocks_for(n)), dim3(kThreads), 0, ctx->stream, n, d.dt, U, VH, Acc);
      time += d.dt;
      g.s.ag = ground_at(k, time);
      if (damp)
        if (int rc = operator_apply64(b, fx_coeffs{0.0, 1.0, 0.0, 0}, VH, fd)) return rc;
      if (b->pimy) {
        if (int rc = pimy_force64(b, U, pdamp ? VH : nullptr, f, false)) return rc;
        if (b->nodal_am)
          if (int rc = nodal_damping_force64(b, VH, f)) return rc;
      } else if (int rc = operator_apply64(b, fx_coeffs{1.0, 0.0, 0.0, 0}, U, f)) {
        return rc;
      }
      if (pl.n > 0) {
        for (int j = 0; j < pl.n; ++j) pl.val[j] = d.load_hist[static_cast<size_t>(k) * pl.n + j];
        hipLaunchKernelGGL(point_load_kernel, dim3(1), dim3(64), 0, ctx->stream, pl, f);
      }
      g.u = U;
      g.s.um = VH;
      g.v = V;
      g.a = Acc;
      hipLaunchKernelGGL(ed_correct_kernel, dim3(blocks_for(n)), dim3(kThreads), 0, ctx->stream, g);
      if (b->pimy) std::swap(b->state_c, b->state_t);  // commit_state
      if (rec)
        if (int rc = recorder_record(d.recorder, time, n, U, V, Acc, rmap)) return rc;
    }
  }
  // a lattice step in two launches, the update run where each equation's force is complete (with
  // dashpots 64 B of vectors per equation and step become 48)
  const bool fused = !ed && box_forms_force(b) && !b->nodal_am && pl.n <= kStepLoads;
  for (int32_t k = 0; !ed && k < d.nsteps; ++k) {
    g.s.ag = ground_at(k, time);
    time += d.dt;
    // the recorded v and a only where a record reads them (of this step, so of every step) and in
    // the last two steps: the last step's acceleration needs the velocity of the step before
    const bool rates = rec_rates || k >= d.nsteps - 2;
    g.s.um = Um;
    g.s.v = rates ? V : nullptr;
    g.s.a = rates ? Acc : nullptr;
    if (fused) {
      CdStep s = g.s;
      s.nload = pl.n;
      for (int j = 0; j < pl.n; ++j) {
        s.load_eq[j] = pl.eq[j];
        s.load[j] = d.load_hist[static_cast<size_t>(k) * pl.n + j];
      }
      if (int rc = launch_box_force(b, U, damp ? Um : nullptr, -c2, nullptr, 0, &s)) return rc;
      std::swap(U, Um);
      if (rec)
        if (int rc = recorder_record(d.recorder, time, n, U, V, Acc, rmap)) return rc;
      continue;
    }
    if (edamp)
      hipLaunchKernelGGL(scale_kernel, dim3(blocks_for(n)), dim3(kThreads), 0, ctx->stream, n, -c2, Um, ve);
    if (damp)
      if (int rc = operator_apply64(b, fx_coeffs{0.0, 1.0, 0.0, 0}, ve, fd)) return rc;
    if (b->pimy) {
      if (int rc = pimy_force64(b, U, pdamp ? ve : nullptr, f, false)) return rc;
      if (b->nodal_am)
        if (int rc = nodal_damping_force64(b, ve, f)) return rc;
    } else if (int rc = operator_apply64(b, fx_coeffs{1.0, 0.0, 0.0, 0}, U, f)) {
      return rc;
    }
    if (pl.n > 0) {
      for (int j = 0; j < pl.n; ++j) pl.val[j] = d.load_hist[static_cast<size_t>(k) * pl.n + j];
      hipLaunchKernelGGL(point_load_kernel, dim3(1), dim3(64), 0, ctx->stream, pl, f);
    }
    g.u = U;
    hipLaunchKernelGGL(cd_update_kernel, dim3(blocks_for(n)), dim3(kThreads), 0, ctx->stream, g);
    std::swap(U, Um);  // U(n+1) sits in the old U(n-1) buffer
    if (b->pimy) std::swap(b->state_c, b->state_t);  // commit_state: the trial history becomes committed
    if (rec)
      if (int rc = recorder_record(d.recorder, time, n, U, V, Acc, rmap)) return rc;
  }
  FX_HIP(ctx, hipGetLastError());
  // back to the caller's buffers: u = U(n+1), um = U(n)
  if (b->internal) {
    if (int rc = to_external_all(b, VectorPairs{{{U, u}, {Um, um}, {V, v}, {Acc, a}}})) return rc;
  } else if (!ed && U != u) {  // an odd number of steps: the roles are swapped
    if (int rc = copy64(ctx, n, U, ve)) return rc;
    if (int rc = copy64(ctx, n, Um, U)) return rc;
    if (int rc = copy64(ctx, n, ve, Um)) return rc;
  }
  if (d.ground_series && d.ground_series->loc) *d.ground_series->loc = loc;
  FX_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return FX_OK;
}

}  // namespace fx
