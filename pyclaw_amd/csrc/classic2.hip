// classic2.hip -- 2D classic Clawpack unsplit wave-propagation step for gfx950:
// one fused kernel per step (unsplit.hpp: x- and y-slices of classic/step2.f90
// with flux2.f90, limiter.f90, philim.f90, the ghost fill as an index map and
// the CFL max-reduction), plus the device-controlled variant, with a one-wavefront
// kernel after it that applies Solver.evolve_to_time's accept/reject and next dt.
//
// A fused kernel was measured against a two-launch form (an x-sweep into a work
// array, then a y-sweep): on 1024^2 Euler FP64 the fused kernel takes 162 us,
// the two launches 78 + 132 us, because the slices' FP64 instruction count is
// the bound and the split pays the halo recomputation and the work round trip
// twice.
#include "variant.hpp"  // first: selects the arithmetic variant
#include <stdlib.h>

#include <algorithm>
#include <cmath>

#include "launch.hpp"
#include "unsplit.hpp"

namespace claw {
namespace CLAW_VNS {

template <class RS, typename T, bool KAHAN, bool AUX = false, bool CAPA = false>
__global__ void __launch_bounds__(256)
    __attribute__((amdgpu_waves_per_eu(unsplit_waves<RS, T, AUX, CAPA>())))
    k_unsplit(const UnsplitArgs<T> a) {
  // one Courant-number atomic per workgroup: one per wavefront serialises
  // (same address) over the thousands of wavefronts of a large grid
  block_atomic_max(unsplit_block<RS, T, KAHAN, AUX, CAPA>(a, (int)xcd_block()), a.cfl_bits);
}

// Device-resident stepping: one launch = one attempted step of
// Solver.evolve_to_time.  The state ping-pongs between two buffers; `ctl->cur`
// names the current one.  The last workgroup to finish applies the CFL check,
// accepts or rejects the step and computes the next dt (k_step_ctl after it).
template <class RS, typename T, bool KAHAN>
__global__ void __launch_bounds__(256)
    __attribute__((amdgpu_waves_per_eu(unsplit_waves<RS, T>())))
    k_unsplit_ctl(UnsplitArgs<T> a, StepCtl* ctl, CtlBuffers bufs) {
  if (ctl->done) return;   // uniform across the grid
  const int cur = ctl->cur;
  const double dt = ctl->dt;
  a.qin = (const T*)bufs.q[cur];
  a.qout = (T*)bufs.q[1 - cur];
  a.comp_in = (const T*)bufs.comp[cur];
  a.comp_out = (T*)bufs.comp[1 - cur];
  a.dtdx = T(dt / bufs.dx);
  a.dtdy = T(dt / bufs.dy);
  a.cfl_bits = &ctl->cfl_bits;
  block_atomic_max(unsplit_block<RS, T, KAHAN>(a, (int)xcd_block()), a.cfl_bits);
}

// The step's control after it (step_ctl_apply).
__global__ void __launch_bounds__(64) k_step_ctl(StepCtl* ctl) {
  if (threadIdx.x == 0) step_ctl_apply(ctl);
}

}  // namespace CLAW_VNS
}  // namespace claw

// ---------------------------------------------------------------- launchers
namespace claw {
namespace CLAW_VNS {

namespace {
// Blocks per strip.  Four wavefronts of a block solve its rows and one more, each
// after a warm-up worth about a row; a launch of k rounds of resident blocks costs
// k times that, and the smallest such cost is taken.  Blocks of at most 128 rows:
// longer ones leave nothing to fill in behind the early wavefronts (4096^2 FP64
// acoustics, 64 / 128 / 186 / 256 rows: 402, 403, 411, 438 us).  At least 7, two
// solves a wavefront: a grid that fills less than one round takes it (256^2 FP64
// acoustics, 3 / 7 / 11 / 15 / 19 rows: 11.2, 10.7, 12.2, 14.4, 16.3 us).
// CLAWHIP_UNSPLIT_ROWS overrides the solves per wavefront (tuning sweeps).
template <class Kernel>
int choose_blocks(Kernel kernel, int nstrips, int my, int waves_hint) {
  if (const char* env = getenv("CLAWHIP_UNSPLIT_ROWS")) {
    int h = atoi(env);
    if (h >= 1 && h <= 4096) return (my + 4 * h - 2) / (4 * h - 1);
  }
  // beyond two wavefronts per SIMD the measured gain of a third is smaller than
  // the halo rows the shorter marches add, so count at most two, unless the
  // kernel is compiled for more (unsplit_waves)
  const long long resident =
      resident_waves((const void*)kernel, waves_hint > 2 ? waves_hint : 2) / 4;
  if (resident == 0) return (my + 63) / 64;
  const int most = (my + 6) / 7, least = (my + 127) / 128;
  const double all = (double)my * nstrips / (4.0 * resident);   // rows of a wavefront, one round
  int best = most;
  double best_cost = 1e300;
  for (long long k = 1; all + k < best_cost; k++) {
    const int n = (int)std::min((long long)most, k * resident / nstrips);
    if (n < least) continue;
    const double rounds = std::ceil((double)nstrips * n / resident);
    const double cost = rounds * (((double)my / n + 1) / 4 + 1);
    if (cost < best_cost) {
      best = n;
      best_cost = cost;
    }
    if (n == most) break;
  }
  return best;
}

template <class RS, typename T, bool KAHAN, bool AUX = false, bool CAPA = false>
int run_unsplit(const clawhip_rp& rp, const void* q_in, const Geom& gin, void* q_out,
                const Geom& gout, const void* comp_in, void* comp_out, const int* lo, const int* hi, const int* refl,
                int ng, const int* method, const int* mthlim, double dx, double dy, double dt,
                unsigned long long* cfl_bits, hipStream_t stream, const AuxIn* aux = nullptr) {
  UnsplitArgs<T> a;
  a.aux = nullptr;
  a.naux = 0;
  a.capa = -1;
  if constexpr (AUX) {
    a.aux = (const T*)aux->p;
    a.gaux = aux->g;
    const int never[3] = {-1, -1, -1};
    a.bcaux = to_bc(aux->lo, aux->hi, never, 2);
    a.naux = method[6];
    a.capa = method[5] - 1;
  }
  a.rp = to_params<T>(rp);
  a.gin = gin; a.gout = gout;
  a.bc = to_bc(lo, hi, refl, 2);
  a.ng = ng; a.order = method[1]; a.trans = method[2];
  for (int w = 0; w < kMaxWaves; w++) a.mthlim[w] = w < RS::mwaves ? mthlim[w] : 0;
  a.dtdx = T(dt / dx); a.dtdy = T(dt / dy);
  a.nstrips = (gout.mx + 59) / 60;
  a.nrb = choose_blocks(k_unsplit<RS, T, KAHAN, AUX, CAPA>, a.nstrips, gout.my,
                        unsplit_waves<RS, T, AUX, CAPA>());
  a.qin = (const T*)q_in; a.qout = (T*)q_out;
  a.comp_in = (const T*)comp_in; a.comp_out = (T*)comp_out;
  a.cfl_bits = cfl_bits;
  const unsigned blocks = (unsigned)((long long)a.nstrips * a.nrb);
  hipLaunchKernelGGL((k_unsplit<RS, T, KAHAN, AUX, CAPA>), dim3(blocks), dim3(256), 0, stream, a);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : (int)e;
}

template <class RS, typename T, bool KAHAN>
int run_unsplit_ctl(const clawhip_rp& rp, const Geom& g, const int* lo, const int* hi,
                    const int* refl, int ng, const int* method, const int* mthlim,
                    StepCtl* ctl, const CtlBuffers& bufs, int nsteps, hipStream_t stream) {
  UnsplitArgs<T> a;
  a.rp = to_params<T>(rp);
  a.gin = g; a.gout = g;
  a.bc = to_bc(lo, hi, refl, 2);
  a.ng = ng; a.order = method[1]; a.trans = method[2];
  for (int w = 0; w < kMaxWaves; w++) a.mthlim[w] = w < RS::mwaves ? mthlim[w] : 0;
  a.dtdx = T(0); a.dtdy = T(0);
  a.nstrips = (g.mx + 59) / 60;
  a.nrb = choose_blocks(k_unsplit_ctl<RS, T, KAHAN>, a.nstrips, g.my, unsplit_waves<RS, T>());
  a.qin = nullptr; a.qout = nullptr; a.comp_in = nullptr; a.comp_out = nullptr;
  a.cfl_bits = nullptr;
  const unsigned blocks = (unsigned)((long long)a.nstrips * a.nrb);
  for (int n = 0; n < nsteps; n++) {
    hipLaunchKernelGGL((k_unsplit_ctl<RS, T, KAHAN>), dim3(blocks), dim3(256), 0, stream, a,
                       ctl, bufs);
    hipLaunchKernelGGL(k_step_ctl, dim3(1), dim3(64), 0, stream, ctl);
  }
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : (int)e;
}

template <template <typename> class RSF>
int dispatch_unsplit_ctl(int dtype, const clawhip_rp& rp, const Geom& g, const int* lo,
                         const int* hi, const int* refl, int ng, const int* method,
                         const int* mthlim, StepCtl* ctl, const CtlBuffers& bufs, int nsteps,
                         hipStream_t stream) {
  if (dtype != CLAWHIP_F32K)
    return run_unsplit_ctl<RSF<double>, double, false>(rp, g, lo, hi, refl, ng, method, mthlim,
                                                       ctl, bufs, nsteps, stream);
#if CLAW_FAST
  return run_unsplit_ctl<RSF<float>, float, true>(rp, g, lo, hi, refl, ng, method, mthlim, ctl,
                                                  bufs, nsteps, stream);
#else
  // FP32 + Kahan is dispatched to the fast variant only
  return CLAWHIP_E_ARG;
#endif
}

template <template <typename> class RSF>
int dispatch_unsplit(int dtype, const clawhip_rp& rp, const void* q_in, const Geom& gin,
                     void* q_out, const Geom& gout, const void* comp_in, void* comp_out, const int* lo, const int* hi,
                     const int* refl, int ng, const int* method, const int* mthlim, double dx,
                     double dy, double dt, unsigned long long* cfl_bits, hipStream_t stream) {
  if (dtype != CLAWHIP_F32K)
    return run_unsplit<RSF<double>, double, false>(rp, q_in, gin, q_out, gout, comp_in, comp_out, lo, hi,
                                                   refl, ng, method, mthlim, dx, dy, dt,
                                                   cfl_bits, stream);
#if CLAW_FAST
  return run_unsplit<RSF<float>, float, true>(rp, q_in, gin, q_out, gout, comp_in, comp_out, lo, hi, refl,
                                              ng, method, mthlim, dx, dy, dt, cfl_bits, stream);
#else
  // FP32 + Kahan is dispatched to the fast variant only
  return CLAWHIP_E_ARG;
#endif
}
// Solvers with aux fields: the aux window, with or without a capacity field.
template <class RS>
int dispatch_unsplit_aux(int dtype, const clawhip_rp& rp, const void* q_in, const Geom& gin,
                         void* q_out, const Geom& gout, const void* comp_in, void* comp_out,
                         const int* lo, const int* hi, const int* refl, int ng,
                         const int* method, const int* mthlim, double dx, double dy, double dt,
                         unsigned long long* cfl_bits, hipStream_t stream, const AuxIn& aux) {
  (void)rp;
  const bool capa = method[5] > 0;
  if (dtype != CLAWHIP_F32K) {
    using R = typename RS::template with<double>;
    return capa ? run_unsplit<R, double, false, true, true>(rp, q_in, gin, q_out, gout, comp_in,
                                                            comp_out, lo, hi, refl, ng, method,
                                                            mthlim, dx, dy, dt, cfl_bits, stream,
                                                            &aux)
                : run_unsplit<R, double, false, true, false>(rp, q_in, gin, q_out, gout, comp_in,
                                                             comp_out, lo, hi, refl, ng, method,
                                                             mthlim, dx, dy, dt, cfl_bits, stream,
                                                             &aux);
  }
#if CLAW_FAST
  using R = typename RS::template with<float>;
  return capa ? run_unsplit<R, float, true, true, true>(rp, q_in, gin, q_out, gout, comp_in,
                                                        comp_out, lo, hi, refl, ng, method, mthlim,
                                                        dx, dy, dt, cfl_bits, stream, &aux)
              : run_unsplit<R, float, true, true, false>(rp, q_in, gin, q_out, gout, comp_in,
                                                         comp_out, lo, hi, refl, ng, method,
                                                         mthlim, dx, dy, dt, cfl_bits, stream,
                                                         &aux);
#else
  // FP32 + Kahan is dispatched to the fast variant only
  return CLAWHIP_E_ARG;
#endif
}

template <int ME>
struct VCAdvectionOf {
  template <typename T>
  using with = VCAdvection<T, ME>;
};
template <template <typename> class RSF>
struct SolverOf {
  template <typename T>
  using with = RSF<T>;
};
}  // namespace

int launch_unsplit(const clawhip_rp& rp, int dtype, const void* q_in, const Geom& gin,
                   void* q_out, const Geom& gout, const void* comp_in, void* comp_out, const int* lo, const int* hi,
                   const int* refl, int ng, const int* method, const int* mthlim, double dx,
                   double dy, double dt, unsigned long long* cfl_bits, hipStream_t stream,
                   const AuxIn& aux) {
  if (rp.kind == CLAWHIP_RP_VC_ADVECTION || rp.kind == CLAWHIP_RP_VC_ADVECTION_2D) {
    if (!aux.p) return CLAWHIP_E_ARG;
    const int me = rp.kind == CLAWHIP_RP_VC_ADVECTION_2D ? 1 : rp.meqn;
#define CLAWHIP_VCA(ME)                                                                         \
  return dispatch_unsplit_aux<VCAdvectionOf<ME>>(dtype, rp, q_in, gin, q_out, gout, comp_in,   \
                                                 comp_out, lo, hi, refl, ng, method, mthlim,   \
                                                 dx, dy, dt, cfl_bits, stream, aux)
    switch (me) {
      case 1: CLAWHIP_VCA(1);
      case 2: CLAWHIP_VCA(2);
      case 3: CLAWHIP_VCA(3);
      case 4: CLAWHIP_VCA(4);
    }
#undef CLAWHIP_VCA
    return CLAWHIP_E_ARG;
  }
  if (rp.kind == CLAWHIP_RP_VC_ACOUSTICS) {
    if (!aux.p) return CLAWHIP_E_ARG;
    return dispatch_unsplit_aux<SolverOf<VCAcoustics>>(dtype, rp, q_in, gin, q_out, gout, comp_in,
                                                      comp_out, lo, hi, refl, ng, method, mthlim,
                                                      dx, dy, dt, cfl_bits, stream, aux);
  }
  if (rp.kind == CLAWHIP_RP_SHALLOW_FWAVE) {
    if (!aux.p) return CLAWHIP_E_ARG;
    return dispatch_unsplit_aux<SolverOf<ShallowFwave>>(dtype, rp, q_in, gin, q_out, gout,
                                                       comp_in, comp_out, lo, hi, refl, ng,
                                                       method, mthlim, dx, dy, dt, cfl_bits,
                                                       stream, aux);
  }
  if (aux.p) return CLAWHIP_E_ARG;
  switch (rp.kind) {
    case CLAWHIP_RP_ACOUSTICS:
      if (stiff(rp))
        return dispatch_unsplit<StiffAcoustics>(dtype, rp, q_in, gin, q_out, gout, comp_in,
                                                comp_out, lo, hi, refl, ng, method, mthlim, dx,
                                                dy, dt, cfl_bits, stream);
      return dispatch_unsplit<Acoustics>(dtype, rp, q_in, gin, q_out, gout, comp_in, comp_out, lo, hi, refl,
                                         ng, method, mthlim, dx, dy, dt, cfl_bits, stream);
    case CLAWHIP_RP_EULER:
      return dispatch_unsplit<Euler>(dtype, rp, q_in, gin, q_out, gout, comp_in, comp_out, lo, hi, refl, ng,
                                     method, mthlim, dx, dy, dt, cfl_bits, stream);
    case CLAWHIP_RP_SHALLOW:
      return dispatch_unsplit<Shallow>(dtype, rp, q_in, gin, q_out, gout, comp_in, comp_out, lo, hi, refl,
                                       ng, method, mthlim, dx, dy, dt, cfl_bits, stream);
    case CLAWHIP_RP_ADVECTION:
      return dispatch_unsplit<Advection>(dtype, rp, q_in, gin, q_out, gout, comp_in, comp_out, lo, hi, refl,
                                         ng, method, mthlim, dx, dy, dt, cfl_bits, stream);
    case CLAWHIP_RP_SHALLOW_HLLE:
      return dispatch_unsplit<ShallowHLLE>(dtype, rp, q_in, gin, q_out, gout, comp_in, comp_out,
                                           lo, hi, refl, ng, method, mthlim, dx, dy, dt,
                                           cfl_bits, stream);
    case CLAWHIP_RP_EULER5:
      return dispatch_unsplit<Euler5>(dtype, rp, q_in, gin, q_out, gout, comp_in, comp_out, lo, hi,
                                      refl, ng, method, mthlim, dx, dy, dt, cfl_bits, stream);
  }
  return CLAWHIP_E_KIND;
}

int launch_unsplit_ctl(const clawhip_rp& rp, int dtype, const Geom& g, const int* lo,
                       const int* hi, const int* refl, int ng, const int* method,
                       const int* mthlim, StepCtl* ctl, const CtlBuffers& bufs, int nsteps,
                       hipStream_t stream) {
  switch (rp.kind) {
    case CLAWHIP_RP_ACOUSTICS:
      if (stiff(rp))
        return dispatch_unsplit_ctl<StiffAcoustics>(dtype, rp, g, lo, hi, refl, ng, method,
                                                    mthlim, ctl, bufs, nsteps, stream);
      return dispatch_unsplit_ctl<Acoustics>(dtype, rp, g, lo, hi, refl, ng, method, mthlim, ctl,
                                             bufs, nsteps, stream);
    case CLAWHIP_RP_EULER:
      return dispatch_unsplit_ctl<Euler>(dtype, rp, g, lo, hi, refl, ng, method, mthlim, ctl,
                                         bufs, nsteps, stream);
    case CLAWHIP_RP_SHALLOW:
      return dispatch_unsplit_ctl<Shallow>(dtype, rp, g, lo, hi, refl, ng, method, mthlim, ctl,
                                           bufs, nsteps, stream);
    case CLAWHIP_RP_ADVECTION:
      return dispatch_unsplit_ctl<Advection>(dtype, rp, g, lo, hi, refl, ng, method, mthlim, ctl,
                                             bufs, nsteps, stream);
    case CLAWHIP_RP_SHALLOW_HLLE:
      return dispatch_unsplit_ctl<ShallowHLLE>(dtype, rp, g, lo, hi, refl, ng, method, mthlim,
                                               ctl, bufs, nsteps, stream);
    case CLAWHIP_RP_EULER5:
      return dispatch_unsplit_ctl<Euler5>(dtype, rp, g, lo, hi, refl, ng, method, mthlim, ctl,
                                          bufs, nsteps, stream);
  }
  return CLAWHIP_E_KIND;
}

}  // namespace CLAW_VNS
}  // namespace claw
