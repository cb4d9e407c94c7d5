// unsplit3.hip -- the unsplit 3D classic step (classic/step3.f90 with
// flux3.f90's transverse and double-transverse terms), FP64.
//
// step3 adds to each cell, in a fixed order, the updates of the 27 slices
// around it: 9 x-slices (k outer, j inner), 9 y-slices (k outer, i inner), 9
// z-slices (j outer, i inner) (step3.f90:120-580).  Every slice reads the old
// state, so the slices are independent; the order only matters for the sums.
// Two kernels per direction:
//   k_flux3<DIR>: for every slice of that direction, the flux3 results of each
//     cell along it -- qadd, fadd at its left interface, and the transverse
//     modifications gadd(m, 1:2, -1:1) and hadd -- into a work array.  The
//     slices' cells with their ghosts (n + 4 each) are laid end to end and a
//     wavefront takes 64 consecutive ones and owns the middle 60, so a slice
//     of any length fills the lanes (one strip a slice left 47 % of them idle
//     at n = 64); neighbours' values by DPP lane shifts as in the split sweeps.
//   k_apply3<DIR>: adds a direction's 9 slices to each cell, in the reference's
//     order and parenthesisation (bitwise equal to the oracle, whose step3 equals
//     the reference's own Fortran on every qbc cell).  A pass per direction lets
//     the lanes run along the slices, as the work array is laid out: with lanes
//     along x throughout, the y- and z-slices' 270 of a cell's 405 loads per
//     field touched a cache line each: at 96x64x80 one such pass took 1.23 ms,
//     the three take 0.28, and the step 0.73 instead of 1.86 ms (k_flux3
//     0.60 -> 0.42).
// Work: 14 * meqn doubles per cell and direction; x, then y, then z use the same
// array, so that a direction's results are read while they are cached.  Bound:
// HBM, by the work array's write and its 27-fold gather; the path exists for
// parity with ClawSolver3D's unsplit default, the split step is the fast 3D path.
#include <algorithm>
#include <type_traits>

#include "launch.hpp"

namespace claw {

template <typename T>
struct Step3Args {
  RPParams<T> rp;
  Geom g;            // the state's geometry (compact, or with stored ghosts)
  BCSpec bc;
  int ng, order, m3, m4;
  int mthlim[kMaxWaves];
  T dtdx, dtdy, dtdz;
  const T* qin;
  T* qout;           // compact output (k_apply3)
  T* work;           // the direction's component-major slice results
  long long wstride; // elements per component
  const T* qsum;     // k_apply3: what the direction's slices are added to, and its
  Geom gsum;         //   geometry (the old state, then qout)
  unsigned long long* cfl_bits;
};

// Extents of direction DIR's slices: normal length n, first transverse
// (gadd's, the next axis in the cycle) a, second (hadd's) b.
template <int DIR>
__device__ __host__ __forceinline__ void dir_extents(const Geom& g, int& n, int& na, int& nb) {
  if (DIR == 1) { n = g.mx; na = g.my; nb = g.mz; }
  else if (DIR == 2) { n = g.my; na = g.mz; nb = g.mx; }
  else { n = g.mz; na = g.mx; nb = g.my; }
}

// Slices are numbered so that consecutive ones lie next to each other in x (in y
// for the x-slices): the strided q rows of neighbouring slices share lines.
template <int DIR>
__device__ __forceinline__ void slice_ab(long long sl, int na, int nb, int& sa, int& sb) {
  if (DIR == 2) { sb = (int)(sl % (nb + 2)); sa = (int)(sl / (nb + 2)); }
  else { sa = (int)(sl % (na + 2)); sb = (int)(sl / (na + 2)); }
}
template <int DIR>
__device__ __forceinline__ long long slice_no(int a, int b, int na, int nb) {
  return DIR == 2 ? (long long)a * (nb + 2) + b : (long long)b * (na + 2) + a;
}

// component slots: 0..ME-1 qadd, ME..2ME-1 fadd, then gadd / hadd as
// 2ME + m + ME * (side - 1 + 2 * (off + 1)), H after the 6 ME of G.
template <int ME>
struct W3 {
  static constexpr int QA = 0, FA = ME, G = 2 * ME, H = 8 * ME, N = 14 * ME;
  __device__ static constexpr int gh(int base, int m, int side, int off) {
    return base + m + ME * ((side - 1) + 2 * (off + 1));
  }
};

template <class RS, int DIR>
__global__ void __launch_bounds__(256) k_flux3(const Step3Args<double> a) {
  using T = double;
  constexpr int ME = RS::meqn, MW = RS::mwaves;
  using WL = W3<ME>;
  const int lane = threadIdx.x & 63;
  const long long wid = xcd_block() * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int n, na, nb;
  dir_extents<DIR>(a.g, n, na, nb);
  const long long slices = (long long)(na + 2) * (nb + 2), cells = slices * (n + 4);
  // wavefronts past the last cell skip the work but reach the workgroup's
  // Courant-number reduction (a barrier): one atomic per workgroup
  const bool live = wid * 60 < cells;   // uniform per wavefront
  double cfl_wave = 0.0;
  if (live) {
    // the lane's place in the row of slices: cell c = -1..n+2 of slice (sa, sb);
    // lanes outside the row take its first or last cell and own nothing
    const long long first = wid * 60 / (n + 4);
    const int at = (int)(wid * 60 - first * (n + 4)) + lane - 2;
    const int hop = at < 0 ? 0 : at / (n + 4);
    const bool inside = (at >= 0 || first > 0) && first + hop < slices;
    // at < 0: the last cells of the slice before
    const long long sl = !inside ? (at < 0 ? 0 : slices - 1) : at < 0 ? first - 1 : first + hop;
    const int c = (!inside ? (at < 0 ? 0 : n + 3) : at < 0 ? at + n + 4 : at - hop * (n + 4)) - 1;
    int sa, sb;   // 0..na+1, 0..nb+1
    slice_ab<DIR>(sl, na, nb, sa, sb);
    const T dtn = DIR == 1 ? a.dtdx : (DIR == 2 ? a.dtdy : a.dtdz);
    // flux3's dtdy / dtdz: the first / second transverse direction's dt/d
    const T dt1 = DIR == 1 ? a.dtdy : (DIR == 2 ? a.dtdz : a.dtdx);
    const T dt2 = DIR == 1 ? a.dtdz : (DIR == 2 ? a.dtdx : a.dtdy);
    int i, j, k;
    if (DIR == 1) { i = c; j = sa; k = sb; }
    else if (DIR == 2) { j = c; k = sa; i = sb; }
    else { k = c; i = sa; j = sb; }
    T Q[ME], QL[ME];
    load_cell3<ME>(a.qin, a.g, a.bc, a.ng, i, j, k, Q);
    from_left(Q, QL);
    Watch<RS, T> seen;
    seen.see(Q);
    auto slice = [&](auto kind) __attribute__((always_inline)) {
    constexpr bool WIDE = decltype(kind)::value;
    T W[MW][ME], s[MW], am[ME], ap[ME];
    typename RS::Roe roe;
    RS::template rpn<DIR, WIDE>(a.rp, QL, Q, W, s, am, ap, roe);
    // Courant number over interfaces 1..n+1 (flux3.f90:214-221)
    T smax = T(0);
    if (lane >= 1 && inside && c >= 1 && c <= n + 1) {
  #pragma unroll
      for (int w = 0; w < MW; w++) smax = cfl_term(smax, fabs(s[w]));
    }
    cfl_wave = (double)dtn * (double)smax;
    // qadd(c) = (0 - dtn apdq(c)) - dtn amdq(c+1)  (flux3.f90:205-208)
    T amn[ME], qadd[ME];
    from_right(am, amn);
  #pragma unroll
    for (int m = 0; m < ME; m++) qadd[m] = (T(0) - dtn * ap[m]) - dtn * amn[m];
    // second-order correction (flux3.f90:224-259); cqxx carries the 0.5
    T cq[ME];
  #pragma unroll
    for (int m = 0; m < ME; m++) cq[m] = T(0);
    if (a.order != 1) {
      T Wn[MW][ME];
  #pragma unroll
      for (int w = 0; w < MW; w++) from_right(W[w], Wn[w]);
      T dotr[MW], dotl[MW];
      wave_dots<ME, MW>(W, Wn, dotr);
      from_left(dotr, dotl);
      limit_waves<ME, MW>(W, s, dotl, dotr, a.mthlim);
      const T dtdxave = T(0.5) * (dtn + dtn);
  #pragma unroll
      for (int w = 0; w < MW; w++) {
  #pragma unroll
        for (int m = 0; m < ME; m++) {
          const T sa2 = fabs(s[w]);
          const T f = a.rp.fwave ? copysign(T(1), s[w]) : sa2;
          cq[m] = cq[m] + T(0.5) * f * (T(1) - sa2 * dtdxave) * W[w][m];
        }
      }
    }
    T fadd[ME];
  #pragma unroll
    for (int m = 0; m < ME; m++) fadd[m] = T(0) + cq[m];

    // stores of this lane's cell c (cells 1..n; fadd at interfaces 1..n+1)
    const bool own = lane >= 2 && lane < 62 && inside && c >= 1;
    const bool own_cell = own && c <= n;
    const long long st = a.wstride;
    T* wk = a.work + slice_no<DIR>(sa, sb, na, nb) * (n + 1) + (c - 1);
    if (own && c <= n + 1) {
  #pragma unroll
      for (int m = 0; m < ME; m++) wk[(WL::FA + m) * st] = fadd[m];
    }
    if (own_cell) {
  #pragma unroll
      for (int m = 0; m < ME; m++) wk[(WL::QA + m) * st] = qadd[m];
    }
    const int m3 = a.m3, m4 = a.m4;
    T bmam[ME], bpam[ME], bmap[ME], bpap[ME], cmam[ME], cpam[ME], cmap[ME], cpap[ME];
    T bmcq[ME], bpcq[ME], cmcq[ME], cpcq[ME];
  #pragma unroll
    for (int m = 0; m < ME; m++) {
      bmam[m] = bpam[m] = bmap[m] = bpap[m] = cmam[m] = cpam[m] = cmap[m] = cpap[m] = T(0);
      bmcq[m] = bpcq[m] = cmcq[m] = cpcq[m] = T(0);
    }
    if (m3 > 0) {
      RS::template rpt3<DIR, 2, WIDE>(roe, am, bmam, bpam);
      RS::template rpt3<DIR, 2, WIDE>(roe, ap, bmap, bpap);
      RS::template rpt3<DIR, 3, WIDE>(roe, am, cmam, cpam);
      RS::template rpt3<DIR, 3, WIDE>(roe, ap, cmap, cpap);
      if (m3 == 2) {
        RS::template rpt3<DIR, 2, WIDE>(roe, cq, bmcq, bpcq);
        RS::template rpt3<DIR, 3, WIDE>(roe, cq, cmcq, cpcq);
      }
    }
    // One family of transverse modifications (gadd: family 0, split direction
    // 2, double-transverse factor dt2; hadd: family 1, direction 3, factor dt1)
    // for cell c: interface c's own terms as a running sum in statement order,
    // then interface c+1's terms for its left cell, shifted from the right lane
    // (flux3.f90:374-456, 488-580).  x*: the 2D splits (bm/bp of am and ap for
    // gadd, cm/cp for hadd); y*: the correction's split in that direction;
    // z*: the other direction's splits, which the double-transverse solve
    // splits again.
    auto family = [&](auto fam, const T (&xmam)[ME], const T (&xpam)[ME], const T (&xmap)[ME],
                      const T (&xpap)[ME], const T (&ymcq)[ME], const T (&ypcq)[ME],
                      const T (&zmam)[ME], const T (&zpam)[ME], const T (&zmap)[ME],
                      const T (&zpap)[ME], const T (&zmcq)[ME], const T (&zpcq)[ME], T dtf) {
      constexpr int FAM = decltype(fam)::value;
      constexpr int ICO = FAM == 0 ? 2 : 3;
      const T sixth = T(1) / T(6);
      T cmcpap[ME], cpcpap[ME], cmcpam[ME], cpcpam[ME], cmcmap[ME], cpcmap[ME], cmcmam[ME],
          cpcmam[ME];
      if (m3 > 0 && m4 > 0) {
        T x2[ME];
  #pragma unroll
        for (int m = 0; m < ME; m++) x2[m] = m4 == 2 ? zpap[m] - T(3) * zpcq[m] : zpap[m];
        RS::template rpt3<DIR, ICO, WIDE>(roe, x2, cmcpap, cpcpap);
  #pragma unroll
        for (int m = 0; m < ME; m++) x2[m] = m4 == 2 ? zpam[m] + T(3) * zpcq[m] : zpam[m];
        RS::template rpt3<DIR, ICO, WIDE>(roe, x2, cmcpam, cpcpam);
  #pragma unroll
        for (int m = 0; m < ME; m++) x2[m] = m4 == 2 ? zmap[m] - T(3) * zmcq[m] : zmap[m];
        RS::template rpt3<DIR, ICO, WIDE>(roe, x2, cmcmap, cpcmap);
  #pragma unroll
        for (int m = 0; m < ME; m++) x2[m] = m4 == 2 ? zmam[m] + T(3) * zmcq[m] : zmam[m];
        RS::template rpt3<DIR, ICO, WIDE>(roe, x2, cmcmam, cpcmam);
      }
  #pragma unroll
      for (int m = 0; m < ME; m++) {
        // [side][off + 1]: the running sums of cell c
        T v[2][3];
        v[0][0] = v[0][1] = v[0][2] = v[1][0] = v[1][1] = v[1][2] = T(0);
        // interface c+1's terms for this cell, shifted from the right lane
        T l0[2], l4[2], l3[2], lp[2], lm[2];
        if (m3 > 0) {
          v[0][1] = v[0][1] - T(0.5) * dtn * xmap[m];
          v[1][1] = v[1][1] - T(0.5) * dtn * xpap[m];
          l0[0] = T(0.5) * dtn * xmam[m];
          l0[1] = T(0.5) * dtn * xpam[m];
          if (m4 > 0) {
            v[1][1] = v[1][1] + sixth * dtn * dtf * (cpcpap[m] - cpcmap[m]);
            v[0][1] = v[0][1] + sixth * dtn * dtf * (cmcpap[m] - cmcmap[m]);
            v[1][2] = v[1][2] - sixth * dtn * dtf * cpcpap[m];
            v[0][2] = v[0][2] - sixth * dtn * dtf * cmcpap[m];
            v[1][0] = v[1][0] + sixth * dtn * dtf * cpcmap[m];
            v[0][0] = v[0][0] + sixth * dtn * dtf * cmcmap[m];
            l4[1] = sixth * dtn * dtf * (cpcpam[m] - cpcmam[m]);
            l4[0] = sixth * dtn * dtf * (cmcpam[m] - cmcmam[m]);
            lp[1] = sixth * dtn * dtf * cpcpam[m];
            lp[0] = sixth * dtn * dtf * cmcpam[m];
            lm[1] = sixth * dtn * dtf * cpcmam[m];
            lm[0] = sixth * dtn * dtf * cmcmam[m];
          }
          if (m3 >= 2) {
            v[1][1] = v[1][1] + dtn * ypcq[m];
            v[0][1] = v[0][1] + dtn * ymcq[m];
            l3[1] = dtn * ypcq[m];
            l3[0] = dtn * ymcq[m];
          }
  #pragma unroll
          for (int sd = 0; sd < 2; sd++) {
            v[sd][1] = v[sd][1] - from_right(l0[sd]);
            if (m4 > 0) {
              v[sd][1] = v[sd][1] + from_right(l4[sd]);
              v[sd][2] = v[sd][2] - from_right(lp[sd]);
              v[sd][0] = v[sd][0] + from_right(lm[sd]);
            }
            if (m3 >= 2) v[sd][1] = v[sd][1] - from_right(l3[sd]);
          }
        }
        if (own_cell) {
          constexpr int base = FAM == 0 ? WL::G : WL::H;
  #pragma unroll
          for (int sd = 0; sd < 2; sd++)
  #pragma unroll
            for (int o = 0; o < 3; o++)
              wk[WL::gh(base, m, sd + 1, o - 1) * st] = v[sd][o];
        }
      }
    };
    family(std::integral_constant<int, 0>(), bmam, bpam, bmap, bpap, bmcq, bpcq, cmam, cpam,
           cmap, cpap, cmcq, cpcq, dt2);
    // hadd's double-transverse input: the y-like splits with the correction
    family(std::integral_constant<int, 1>(), cmam, cpam, cmap, cpap, cmcq, cpcq, bmam, bpam,
           bmap, bpap, bmcq, bpcq, dt1);
    };
    // uniform over the wavefront (see Divided, rpn_either)
    const int way = a.rp.wide ? kPlain : seen.way();
    if (__builtin_expect(way == kShared, 1) ||
        (way == kLooked && __ballot(RS::template shear_alone<DIR>(QL, Q)) == 0ull))
      slice(std::false_type());
    else slice(std::true_type());
  }
  block_atomic_max(cfl_wave, a.cfl_bits);
}

// One slice's update of a cell at transverse offsets (DA, DB) from the slice
// (step3.f90:189-225 and the y / z equivalents): v is the cell's running value,
// wk field m's qadd of the slice (uniform), at the cell's byte offset in it (32
// bits: launch_step3 refuses a component of 4 GB).
template <int ME, int DA, int DB>
__device__ __forceinline__ double term3(double v, const double* wk, long long st, unsigned at,
                                        double dtn, double dt1, double dt2) {
  using WL = W3<ME>;
  auto W = [&](long long comp) {
    return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(wk + comp * st) + at);
  };
  auto G = [&](int side, int off) { return W(WL::gh(WL::G, 0, side, off)); };
  auto H = [&](int side, int off) { return W(WL::gh(WL::H, 0, side, off)); };
  if constexpr (DA == 0 && DB == 0) {
    const double qa = W(WL::QA);
    const double f0 = W(WL::FA);
    const double f1 =
        *reinterpret_cast<const double*>(reinterpret_cast<const char*>(wk + WL::FA * st + 1) + at);
    return v + qa - dtn * (f1 - f0) - dt1 * (G(2, 0) - G(1, 0)) - dt2 * (H(2, 0) - H(1, 0));
  }
  if constexpr (DA == -1 && DB == 0) return v - dt1 * G(1, 0) - dt2 * (H(2, -1) - H(1, -1));
  if constexpr (DA == -1 && DB == -1) return v - dt1 * G(1, -1) - dt2 * H(1, -1);
  if constexpr (DA == 0 && DB == -1) return v - dt1 * (G(2, -1) - G(1, -1)) - dt2 * H(1, 0);
  if constexpr (DA == 1 && DB == -1) return v + dt1 * G(2, -1) - dt2 * H(1, 1);
  if constexpr (DA == 1 && DB == 0) return v + dt1 * G(2, 0) - dt2 * (H(2, 1) - H(1, 1));
  if constexpr (DA == 1 && DB == 1) return v + dt1 * G(2, 1) + dt2 * H(2, 1);
  if constexpr (DA == 0 && DB == 1) return v - dt1 * (G(2, 1) - G(1, 1)) + dt2 * H(2, 0);
  return v - dt1 * G(1, 1) + dt2 * H(2, -1);   // (-1, 1)
}

// A thread per cell, numbered along the slices (consecutive lanes: consecutive
// cells of a slice), then as the slices are.
template <class RS, int DIR>
__global__ void __launch_bounds__(256) k_apply3(const Step3Args<double> a) {
  constexpr int ME = RS::meqn;
  const Geom& g = a.g;
  int n, na, nb;
  dir_extents<DIR>(g, n, na, nb);
  const long long cell = xcd_block() * 256 + threadIdx.x;
  if (cell >= (long long)n * na * nb) return;
  const int p = 1 + (int)(cell % n);
  const long long rest = cell / n;
  const int sa = 1 + (int)(DIR == 2 ? rest / nb : rest % na);
  const int sb = 1 + (int)(DIR == 2 ? rest % nb : rest / na);
  int i, j, k;
  if (DIR == 1) { i = p; j = sa; k = sb; }
  else if (DIR == 2) { j = p; k = sa; i = sb; }
  else { k = p; i = sa; j = sb; }
  const double* pin = cell_ptr3(a.qsum, a.gsum, i, j, k);
  Geom go = g;
  go.g = 0; go.rs = g.mx; go.ss = (long long)g.mx * g.my; go.fs = go.ss * g.mz;
  double* pout = cell_ptr3(a.qout, go, i, j, k);
  const double dtn = DIR == 1 ? a.dtdx : (DIR == 2 ? a.dtdy : a.dtdz);
  const double dt1 = DIR == 1 ? a.dtdy : (DIR == 2 ? a.dtdz : a.dtdx);
  const double dt2 = DIR == 1 ? a.dtdz : (DIR == 2 ? a.dtdx : a.dtdy);
  // elements from a slice to the next in a and in b
  const long long ea = (DIR == 2 ? nb + 2 : 1) * (long long)(n + 1);
  const long long eb = (DIR == 2 ? 1 : na + 2) * (long long)(n + 1);
  // byte offset of (p, slice (sa-1, sb-1)), the first of the 9
  const unsigned at =
      (unsigned)((slice_no<DIR>(sa - 1, sb - 1, na, nb) * (n + 1) + (p - 1)) * (long long)sizeof(double));
  const long long st = a.wstride;
#pragma unroll 1
  for (int m = 0; m < ME; m++) {
    const double* w = a.work + m * st;
    double v = pin[(long long)m * a.gsum.fs];
#define TERM(AA, BB) \
  v = term3<ME, -(AA), -(BB)>(v, w + ((AA) + 1) * ea + ((BB) + 1) * eb, st, at, dtn, dt1, dt2)
    if constexpr (DIR == 2) {   // y-slices (a = k', b = i'): k' outer, i' inner
      TERM(-1, -1); TERM(-1, 0); TERM(-1, 1);
      TERM(0, -1); TERM(0, 0); TERM(0, 1);
      TERM(1, -1); TERM(1, 0); TERM(1, 1);
    } else {   // x-slices (a = j', b = k'): k' outer; z-slices (a = i', b = j'): j' outer
      TERM(-1, -1); TERM(0, -1); TERM(1, -1);
      TERM(-1, 0); TERM(0, 0); TERM(1, 0);
      TERM(-1, 1); TERM(0, 1); TERM(1, 1);
    }
#undef TERM
    pout[(long long)m * go.fs] = v;
  }
}

namespace {
template <class RS, int DIR>
void launch_flux3(const Step3Args<double>& a, hipStream_t stream) {
  int n, na, nb;
  dir_extents<DIR>(a.g, n, na, nb);
  const long long cells = (long long)(na + 2) * (nb + 2) * (n + 4);
  hipLaunchKernelGGL((k_flux3<RS, DIR>), dim3((unsigned)((cells + 239) / 240)), dim3(256), 0,
                     stream, a);
}

template <class RS, int DIR>
void launch_apply3(const Step3Args<double>& a, hipStream_t stream) {
  const long long ncell = (long long)a.g.mx * a.g.my * a.g.mz;
  hipLaunchKernelGGL((k_apply3<RS, DIR>), dim3((unsigned)((ncell + 255) / 256)), dim3(256), 0,
                     stream, a);
}
}  // namespace

namespace {
// Elements of a component of each direction's slice results.
void step3_strides(int mx, int my, int mz, long long (&s)[3]) {
  s[0] = (long long)(mx + 1) * (my + 2) * (mz + 2);
  s[1] = (long long)(my + 1) * (mz + 2) * (mx + 2);
  s[2] = (long long)(mz + 1) * (mx + 2) * (my + 2);
}
}  // namespace

// The directions take the work array in turn: the largest one's results.
long long step3_work_elems(int meqn, int mx, int my, int mz) {
  long long s[3];
  step3_strides(mx, my, mz, s);
  return 14LL * meqn * std::max({s[0], s[1], s[2]});
}

int launch_step3(const clawhip_rp& rp, const void* q_in, const Geom& gin, void* q_out,
                 void* work, const int* lo, const int* hi, const int* refl, int ng,
                 const int* method, const int* mthlim, double dx, double dy, double dz,
                 double dt, unsigned long long* cfl, hipStream_t stream) {
  if (rp.kind != CLAWHIP_RP_EULER3) return CLAWHIP_E_KIND;
  using RS = Euler3<double>;
  Step3Args<double> a;
  a.rp = to_params<double>(rp);
  a.g = gin;
  a.bc = to_bc(lo, hi, refl, 3);
  a.ng = ng;
  a.order = method[1];
  a.m3 = method[2] / 10;
  a.m4 = method[2] - 10 * a.m3;
  for (int w = 0; w < kMaxWaves; w++) a.mthlim[w] = w < RS::mwaves ? mthlim[w] : 0;
  a.dtdx = dt / dx; a.dtdy = dt / dy; a.dtdz = dt / dz;
  a.qin = (const double*)q_in;
  a.qout = (double*)q_out;
  a.cfl_bits = cfl;
  const int mx = gin.mx, my = gin.my, mz = gin.mz;
  long long stride[3];
  step3_strides(mx, my, mz, stride);
  // k_apply3 addresses a component with 32 bits (state and work array together are then
  // beyond any device's memory)
  if (std::max({stride[0], stride[1], stride[2]}) * (long long)sizeof(double) >= 1LL << 32)
    return CLAWHIP_E_ARG;
  // the directions share the work array (the entry point refuses q_out == q_in,
  // so all of them read the old state); each adds its slices to the sum so far
  Geom go = gin;
  go.g = 0; go.rs = mx; go.ss = (long long)mx * my; go.fs = go.ss * mz;
  Step3Args<double> d[3] = {a, a, a};
  for (int k = 0; k < 3; k++) {
    d[k].work = (double*)work;
    d[k].wstride = stride[k];
    d[k].qsum = k == 0 ? a.qin : a.qout;
    d[k].gsum = k == 0 ? gin : go;
  }
  launch_flux3<RS, 1>(d[0], stream);
  launch_apply3<RS, 1>(d[0], stream);
  launch_flux3<RS, 2>(d[1], stream);
  launch_apply3<RS, 2>(d[1], stream);
  launch_flux3<RS, 3>(d[2], stream);
  launch_apply3<RS, 3>(d[2], stream);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : (int)e;
}

}  // namespace claw
