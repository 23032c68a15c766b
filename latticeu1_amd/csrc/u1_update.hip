// u1_update.hip -- checkerboard Metropolis and overrelaxation phases, hot start.
//
// One launch per (pass, parity, mu) phase, as the reference (update.cu:177-190,
// 227-231, 301-316, 379-394), or one k_pair launch for the phases (parity, 0)
// and (parity, 1) of a single lattice (see k_pair).  Within a phase no link
// reads a link of the same phase: the staple of (x, mu) reads theta_nu
// (nu != mu) and theta_mu at the other parity (staple.h:85-92), so the launch
// is race free.
//
// Work decomposition (instruction-issue bound, so indexing is kept scalar):
// a workgroup covers a contiguous chunk of one (z, t) plane of the half
// lattice (P = Nx/2 * Ny even/odd sites per plane), so z, t, their boundary
// tests and the +-z, +-t neighbour offsets are uniform (SGPR) values; a thread
// derives only (x/2, y) from its index in the plane.  All angle loads use a
// uniform 64-bit plane base plus a 32-bit byte offset, which maps to
// global_load with an SGPR base.
//
// FP64 parity contract with the host oracle (oracle/u1_oracle.cpp): the
// staple, the Metropolis weight and the OR reflection below perform the same
// IEEE operations in the same order as the oracle, on the same Philox words,
// with the same u1_math.h functions.  The library is compiled with
// -ffp-contract=off so that no FMA is formed implicitly.
//
// FP32-bulk variant: angles, staples, proposals, the Metropolis weight and the
// OR angle in binary32 with the hardware transcendentals (v_sin_f32,
// v_cos_f32, v_exp_f32, v_rcp_f32) and explicit FMAs; the periodic wrap into
// [-pi, pi] in binary64 (wrap_near_d), rounded once to binary32.  It reads the
// same Philox words as the FP64 path.  Its parity bar is statistical.
#include "u1_chain.h"
#include "u1_kernels.h"
#include "u1_link.h"

namespace u1d {

namespace {

// SPT even/odd sites per thread: sites chunk*SPT*bdim + k*bdim + tid, k < SPT,
// of one (z, t) plane.  All angle loads of all SPT sites are issued before the
// transcendental work, so each wave keeps SPT x 19 loads in flight.  Threads
// past the end of a plane work on the plane's last site (in bounds) and do not
// store.
//
// MEAS (MU >= 1, parity 1 of the last pass of a sweep): the logical
// workgroup L also writes row L of a.meas with its sums over the plaquettes of
// the planes (nu, MU), nu < MU, after the update -- [sum (1 - cos P), sum
// -sin P] in the space-space (MU < 3) or space-time (MU = 3) slot.  The three
// phases (1, 1), (1, 2), (1, 3) come after every link of those planes has
// reached its final value, and together cover all six planes once.
//
// A thread's share of a phase is the sites tid0 + k blockDim.x (k < SPT) of
// chunk b in phase_site numbering (bdim sites per chunk), from phase_sites.
// phase_load issues all of their angle loads; phase_compute forms the staples, updates and
// stores the links, adds the plaquette sums of its valid sites to v (MEAS) and
// the accepted hits of its wavefront to acc_wave; the caller reduces both.
template <typename Real, int SPT>
struct PhaseIn {
  PhaseSite ps[SPT];
  uint32_t same[SPT];
  StapleIn<Real> in[SPT];
  Real th[SPT];
};

// The thread's sites; returns true if the workgroup's plane is frozen
// (multilevel.cu:41,141 -- spatial links on slices t % ml == 0 are frozen; t
// is uniform over the workgroup, so the whole workgroup skips the phase).
template <int MU, int SPT>
__device__ __forceinline__ bool phase_sites(const PhaseArgs& a, const RepDesc& r, uint32_t b, uint32_t tid0,
                                            uint32_t bdim, PhaseSite (&ps)[SPT]) {
#pragma unroll
  for (int k = 0; k < SPT; ++k) phase_site(r, b, tid0 + k * blockDim.x, bdim, a.parity, ps[k]);
  return MU != 3 && a.ml != 0 && (ps[0].t & (uint32_t)(a.ml - 1)) == 0;
}

// The angle loads of the sites in q.ps (but the c, d angles of DEFM).
template <typename Real, int MU, int SPT, int DEFM = 0>
__device__ __forceinline__ void phase_load(const Real* __restrict__ lat_base, const PhaseArgs& a, const RepDesc& r,
                                           PhaseIn<Real, SPT>& q) {
  const Real* lat = lat_base + r.lat_off;
#pragma unroll
  for (int k = 0; k < SPT; ++k) {
    q.same[k] = (uint32_t)(a.parity * r.HV) + q.ps[k].id;
    const uint32_t opp = (uint32_t)((1 - a.parity) * r.HV) + q.ps[k].id;
    staple_load<Real, MU, DEFM>(lat, r, q.same[k], opp, q.ps[k].fwd, q.ps[k].bwd, q.in[k]);
    q.th[k] = ld(lat + (size_t)MU * r.V, q.same[k]);
  }
}

// The c, d angles of the directions in DEFM that phase_load left out --
// theta_nu(x) and theta_nu(x + mu - nu) at the link's own parity, written
// earlier in the same launch by another workgroup -- as device-scope loads.
template <typename Real, int MU, int SPT, int DEFM>
__device__ __forceinline__ void phase_load_dep(const Real* __restrict__ lat_base, const RepDesc& r,
                                               PhaseIn<Real, SPT>& q) {
  const Real* lat = lat_base + r.lat_off;
#pragma unroll
  for (int k = 0; k < SPT; ++k)
#pragma unroll
    for (int nu = 0; nu < 4; ++nu) {
      if (nu == MU || !((DEFM >> nu) & 1)) continue;
      const int j = nu < MU ? nu : nu - 1;
      const Real* pn = lat + (size_t)nu * r.V;
      q.in[k].c[j] = ldc(pn, q.same[k]);
      q.in[k].d[j] = ldc(pn, q.same[k] + (uint32_t)(q.ps[k].fwd[MU] + q.ps[k].bwd[nu]));
    }
}

// The two angles phase_load<..., DEFM = 1> left out -- theta_0 at the
// link's own parity at x and x + e1 - e0, both in the site's (z, t) plane --
// from lds_th, where phase 0 of this workgroup left the plane's new theta_0
// by in-plane index (id - pbase).
template <typename Real, int SPT>
__device__ __forceinline__ void phase_load_nu0_lds(const Real* lds_th, uint32_t pbase, PhaseIn<Real, SPT>& q) {
#pragma unroll
  for (int k = 0; k < SPT; ++k) {
    const uint32_t i = q.ps[k].id - pbase;
    q.in[k].c[0] = lds_th[i];
    q.in[k].d[0] = lds_th[i + (uint32_t)(q.ps[k].fwd[1] + q.ps[k].bwd[0])];
  }
}

// Phase (parity, 1) of a fused pair reads seven angles that phase (parity, 0)
// of the same site has already loaded, at the same addresses, and that
// neither phase writes: the link's own theta_1(x) (c of nu = 1 in phase 0),
// a = theta_0(x + e1) and b = theta_1(x + e0) of nu = 0 (b and a of nu = 1 in
// phase 0), and c = theta_nu(x), f = theta_nu(x - e_nu) of nu = 2, 3 (the
// same slots j = 1, 2 in both phases).  pair_shared keeps them from phase 0's
// staple angles, pair_take hands them to phase 1.
template <typename Real>
struct PairShared {
  Real th, a0, b0, c2, f2, c3, f3;
};
template <typename Real>
__device__ __forceinline__ PairShared<Real> pair_shared(const StapleIn<Real>& in0) {
  return {in0.c[0], in0.b[0], in0.a[0], in0.c[1], in0.f[1], in0.c[2], in0.f[2]};
}
template <typename Real>
__device__ __forceinline__ void pair_take(const PairShared<Real>& s, StapleIn<Real>& in1, Real& th1) {
  th1 = s.th;
  in1.a[0] = s.a0;
  in1.b[0] = s.b0;
  in1.c[1] = s.c2;
  in1.f[1] = s.f2;
  in1.c[2] = s.c3;
  in1.f[2] = s.f3;
}

// The phase-(parity, 1) angles of the sites in q.ps that neither the LDS
// exchange (c, d of nu = 0) nor pair_take provides: e, f of nu = 0 and a, b,
// d, e of nu = 2, 3 -- ten loads instead of seventeen (the addresses of
// staple_load for MU = 1).
template <typename Real, int SPT>
__device__ __forceinline__ void pair1_load(const Real* __restrict__ lat_base, const PhaseArgs& a, const RepDesc& r,
                                           PhaseIn<Real, SPT>& q) {
  const Real* lat = lat_base + r.lat_off;
  const Real* p0 = lat;
  const Real* p1 = lat + (size_t)r.V;
#pragma unroll
  for (int k = 0; k < SPT; ++k) {
    const PhaseSite& s = q.ps[k];
    q.same[k] = (uint32_t)(a.parity * r.HV) + s.id;
    const uint32_t opp = (uint32_t)((1 - a.parity) * r.HV) + s.id;
    q.in[k].e[0] = ld(p1, opp + s.bwd[0]);
    q.in[k].f[0] = ld(p0, opp + s.bwd[0]);
#pragma unroll
    for (int nu = 2; nu < 4; ++nu) {
      const Real* pn = lat + (size_t)nu * r.V;
      q.in[k].a[nu - 1] = ld(pn, opp + s.fwd[1]);
      q.in[k].b[nu - 1] = ld(p1, opp + s.fwd[nu]);
      q.in[k].d[nu - 1] = ld(pn, q.same[k] + s.fwd[1] + s.bwd[nu]);
      q.in[k].e[nu - 1] = ld(p1, opp + s.bwd[nu]);
    }
  }
}

// lds_th (nullable): the new angles are also written to lds_th[id - pbase],
// the site's index within its (z, t) plane (fused pairs, phase 0).  COH: the
// new angles are stored at device scope (fused passes).
template <typename Real, int MU, int KIND, int SPT, bool MEAS, bool COH = false>
__device__ __forceinline__ void phase_compute(Real* __restrict__ lat_base, const PhaseArgs& a, const RepDesc& r,
                                              PhaseIn<Real, SPT>& q, double (&v)[2], uint32_t& acc_wave,
                                              Real* lds_th = nullptr, uint32_t pbase = 0) {
  Real* pmu = lat_base + r.lat_off + (size_t)MU * r.V;
  const bool aniso = r.aniso != 1.0;
  const Real xi = sizeof(Real) == sizeof(float) ? (Real)r.aniso_f : (Real)r.aniso;
  const PhaseSite(&ps)[SPT] = q.ps;
  const uint32_t(&same)[SPT] = q.same;
  Staple<Real> S[SPT];
  Real th[SPT];
  PlaqPieces<Real> pp[SPT];
  uint32_t l[SPT];
  uint64_t vmask[SPT];  // lanes with a valid site
#pragma unroll
  for (int k = 0; k < SPT; ++k) {
    pp[k] = {0, 0, 0, 0};
    S[k] = staple_sum<Real, MU, MEAS>(q.in[k], xi, (Real)r.inv_aniso_f, aniso, &pp[k]);
    th[k] = q.th[k];
    l[k] = same[k] + (uint32_t)MU * (uint32_t)r.V;
    vmask[k] = KIND == KIND_METROPOLIS ? wave_mask(ps[k].valid) : 0;
  }
  update_angles<Real, KIND, SPT>(a, r, S, th, l, vmask, acc_wave);
#pragma unroll
  for (int k = 0; k < SPT; ++k)
    if (ps[k].valid) {
      if (COH)
        stc(pmu, same[k], th[k]);
      else
        st(pmu, same[k], th[k]);
      if (lds_th) lds_th[ps[k].id - pbase] = th[k];
    }
  if (MEAS) {
#pragma unroll
    for (int k = 0; k < SPT; ++k) add_plaquettes<Real, MU>(pp[k], th[k], ps[k].valid, v[0], v[1]);
  }
}

// Workgroup epilogue: the plaquette row L of a measuring phase (block_sum:
// every thread of the workgroup takes part) and the wavefront's accepts.
template <int MU, int KIND, bool MEAS>
__device__ __forceinline__ void phase_finish(const PhaseArgs& a, uint32_t L, double (&v)[2], uint32_t acc_wave) {
  if (MEAS) {
    const double o = block_sum<2>(v);
    if (threadIdx.x < 2) {
      const uint32_t c = MU == 3 ? 2 : 0;
      double* row = a.meas + 4 * (size_t)L + threadIdx.x;
      row[c] = o;
      row[2 - c] = 0.0;
    }
  }
  if (KIND == KIND_METROPOLIS && a.accepts && (threadIdx.x & 63) == 0 && acc_wave)
    atomicAdd(a.accepts, (unsigned long long)acc_wave);
}

template <typename Real, int MU, int KIND, bool BATCHED, int SPT, bool MEAS = false>
__global__ __launch_bounds__(512) void k_phase(Real* __restrict__ lat_base, PhaseArgs a) {
  const uint32_t block = fetch_args<sizeof(Real*) + sizeof(PhaseArgs)>(blockIdx.x);
  const uint32_t L = a.xcd ? xcd_remap(block, gridDim.x) : block;
  const RepDesc& r = BATCHED ? a.reps[a.blockmap[L]] : a.single;
  const uint32_t b = L - (uint32_t)r.blk_begin;
  double v[2] = {0.0, 0.0};
  uint32_t acc_wave = 0;
  PhaseIn<Real, SPT> q;
  // (phase_sites and the early exit written out here: through the helper,
  // hipcc turns the site arithmetic into divergent branches)
#pragma unroll
  for (int k = 0; k < SPT; ++k) phase_site(r, b, threadIdx.x + k * blockDim.x, SPT * blockDim.x, a.parity, q.ps[k]);
  if (MU != 3 && a.ml != 0 && (q.ps[0].t & (uint32_t)(a.ml - 1)) == 0) return;
  phase_load<Real, MU, SPT>(lat_base, a, r, q);
  phase_compute<Real, MU, KIND, SPT, MEAS>(lat_base, a, r, q, v, acc_wave);
  phase_finish<MU, KIND, MEAS>(a, L, v, acc_wave);
}

// The phases (parity, 0) and (parity, 1) of one single lattice in one launch.
// Workgroup L owns the whole (z, t) plane L (set_phase_blocks(r, P): one chunk
// per plane) and runs phase (parity, 0) over it, SPT * blockDim.x sites per
// step, then phase (parity, 1), with a workgroup barrier in between.  This is
// race free and gives the results of the two separate launches bit for bit:
//  * the staple of (x, 1) reads the phase-0 links theta_0 at this parity only
//    at x and x + e1 - e0, both in the same (z, t) plane, so in this
//    workgroup: phase 0 also leaves them in LDS (P angles of the plane, by
//    in-plane index), and phase 1 reads those two from there after the
//    barrier instead of reloading them;
//  * phase (parity, 0) reads theta_1 at this parity only at x and x + e0 - e1,
//    also in the same plane, so before this workgroup's phase 1 rewrites them
//    (its loads have returned before the barrier);
//  * nothing else either phase reads is written by the launch.
// The pair reads the lattice once (4V angles) and writes V/2 + V/2: 5V angles
// against 9V for two launches.  MEAS applies to phase (parity, 1).  Dynamic
// LDS: P angles (pair_lds_bytes).  Of phase 1's nineteen angles two come
// from LDS; in the first two forms below, seven more come from phase 0's loads
// of the same site (pair_shared), phase 1 loads ten, and both load at the same
// time:
//  * PAIR_ONE_STEP: one step covers the plane (P <= SPT * blockDim.x, SPT <= 3):
//    every load of phase 1 is issued before phase 0 computes, so phase 1 waits
//    on the barrier and two LDS reads only;
//  * PAIR_SKEW (SPT = 1): phase 1 follows phase 0 one step behind, with a barrier
//    after each step of phase 0, its angles kept in registers meanwhile.  Sites
//    are in row order, and a step covers at least two rows (step >= Nx): then
//    phase 1 of step k reads the new theta_0 of steps k and k + 1 only (and of
//    row 0, of step 0), and phase 0 of step k + 1 reads the old theta_1 of steps
//    k and k + 1 only (step 0: also of the last row, rewritten last).  All
//    workgroups of an XCD go through their planes at about the same pace, so
//    what a plane shares with its neighbours is read while it is in the L2;
//  * PAIR_LOOP (steps of less than two rows, or more sites per thread): phase 1
//    loads its seventeen angles after phase 0 of the whole plane, when at large
//    planes the L2 no longer has them.
// Binary32 overrelaxation pair, PAIR_LOOP or two steps before, PAIR_SKEW now: 563 ->
// 466 us at 96^4 (1.70 GB compulsory), 82 -> 63 us at 64^4, 24.2 -> 23.0 us at
// 48^4; Metropolis 651 -> 582, 120 -> 105 and 43.4 -> 39.8 us.  256 threads were
// best (occupancy 7 at 65 to 71 registers; two sites per thread: 123 registers
// and 5 to 30 % more time).
// FORM picks the form at compile time for a single lattice, whose plane size
// the host knows: each kernel then holds the code of its own form only.
// PAIR_ANY (batched replicas with planes too large for k_pair_packed) decides
// per workgroup between the last two; its descriptor is copied into registers
// (see k_pair_packed).
// The arguments before a (single lattices) are what the first loads depend on, as
// many as the dispatcher writes into scalar registers by itself (fourteen, build
// flag amdgpu-kernarg-preload-count): the kernel's first 0.4 us were the wait for
// the cold argument lines.  packed: shifts of the four magic divisions by five
// bits, parity, xcd, tile, ml.  Overrelaxation pair 5.67 -> 5.27 us and Metropolis
// 8.54 -> 8.06 us at 24^3 x 48, 5.33 -> 4.94 and 7.54 -> 7.10 us at 28 x 20 x 36 x 22.
enum { PAIR_ONE_STEP = 0, PAIR_SKEW = 1, PAIR_LOOP = 2, PAIR_ANY = 3 };
template <typename Real, int KIND, int SPT, bool MEAS, bool BATCHED = false, int FORM = PAIR_ANY>
__global__ __launch_bounds__(pair_max_block(sizeof(Real), SPT)) void k_pair(Real* __restrict__ lat_base, uint32_t N1,
                                                                          uint32_t N2, uint32_t N3, uint32_t nxh,
                                                                          uint32_t div_nxh_m, uint32_t div_nz_m,
                                                                          uint32_t div_tile_m, uint32_t div_bz_m,
                                                                          uint32_t packed, PhaseArgs a) {
  const uint32_t block = BATCHED ? fetch_args<sizeof(Real*) + 32 + sizeof(PhaseArgs)>(blockIdx.x) : blockIdx.x;
  extern __shared__ __align__(8) unsigned char pair_lds[];
  Real* th0 = reinterpret_cast<Real*>(pair_lds);
  if constexpr (!BATCHED) {
    a.parity = (int32_t)(packed >> 20 & 1u);
    a.xcd = packed >> 21 & 1u;
    a.ml = (int32_t)(packed >> 23 & 7u);
  }
  const uint32_t L = a.xcd ? xcd_remap(block, BATCHED ? gridDim.x : N2 * N3) : block;
  RepDesc r;
  if constexpr (BATCHED) {
    r = a.reps[a.blockmap[L]];
  } else {
    r = a.single;
    r.N[1] = (int32_t)N1;
    r.N[2] = (int32_t)N2;
    r.N[3] = (int32_t)N3;
    r.nxh = r.sy = (int32_t)nxh;
    r.sz = (int32_t)(nxh * N1);
    r.st = (int32_t)(nxh * N1 * N2);
    r.HV = (int32_t)(nxh * N1 * N2 * N3);
    r.V = 2 * r.HV;
    r.div_nxh_m = div_nxh_m;
    r.div_nz_m = div_nz_m;
    r.div_tile_m = div_tile_m;
    r.div_bz_m = div_bz_m;
    r.div_nxh_s = packed & 31u;
    r.div_nz_s = packed >> 5 & 31u;
    r.div_tile_s = packed >> 10 & 31u;
    r.div_bz_s = packed >> 15 & 31u;
    r.tile = packed >> 22 & 1u;
    r.tile_bz = N2 >> 1;
    r.tile_bt = N3 >> 2;
    r.bpp = 1;
    r.div_bpp_m = 1;  // division by 1
    r.div_bpp_s = 0;
    r.blk_begin = 0;
    r.lat_off = 0;
  }
  const uint32_t b = L - (uint32_t)r.blk_begin;  // the replica's plane (one chunk per plane)
  const uint32_t P = (uint32_t)r.nxh * (uint32_t)r.N[1];
  const uint32_t step = SPT * blockDim.x;
  double v0[2] = {0.0, 0.0}, v[2] = {0.0, 0.0};
  uint32_t acc0 = 0, acc1 = 0;
  uint32_t pbase = 0;  // the plane's first id
  // both phases' loads and phase 0 of the step at `base`; false: a frozen plane
  // (multilevel mask, uniform over the workgroup), frozen for both phases: the
  // whole workgroup leaves before the first barrier
  auto phase0 = [&](uint32_t base, PhaseIn<Real, SPT>& q1) -> bool {
    PhaseIn<Real, SPT> q0;
#pragma unroll
    for (int k = 0; k < SPT; ++k)
      phase_site(r, b, base + threadIdx.x + k * blockDim.x, step, a.parity, q0.ps[k]);
    if (a.ml != 0 && (q0.ps[0].t & (uint32_t)(a.ml - 1)) == 0) return false;
    pbase = ((uint32_t)q0.ps[0].z + (uint32_t)r.N[2] * q0.ps[0].t) * P;
#pragma unroll
    for (int k = 0; k < SPT; ++k) q1.ps[k] = q0.ps[k];  // the same sites
    phase_load<Real, 0, SPT>(lat_base, a, r, q0);
    pair1_load<Real, SPT>(lat_base, a, r, q1);
    phase_compute<Real, 0, KIND, SPT, false>(lat_base, a, r, q0, v0, acc0, th0, pbase);
#pragma unroll
    for (int k = 0; k < SPT; ++k) pair_take(pair_shared(q0.in[k]), q1.in[k], q1.th[k]);
    return true;
  };
  auto phase1 = [&](PhaseIn<Real, SPT>& q1) {
    phase_load_nu0_lds<Real, SPT>(th0, pbase, q1);
    phase_compute<Real, 1, KIND, SPT, MEAS>(lat_base, a, r, q1, v, acc1);
  };
  if (FORM == PAIR_ONE_STEP) {
    PhaseIn<Real, SPT> q1;
    if (!phase0(0, q1)) return;
    __syncthreads();
    phase1(q1);
  } else if (FORM == PAIR_SKEW || (FORM == PAIR_ANY && SPT == 1 && step >= 2 * (uint32_t)r.nxh)) {
    PhaseIn<Real, SPT> qa, qb;  // phase 1 of alternate steps
    if (!phase0(0, qa)) return;
    for (uint32_t base = step;; base += 2 * step) {
      if (base < P) phase0(base, qb);
      __syncthreads();
      phase1(qa);
      if (base >= P) break;
      if (base + step < P) phase0(base + step, qa);
      __syncthreads();
      phase1(qb);
      if (base + step >= P) break;
    }
  } else {
    for (uint32_t base = 0; base < P; base += step) {
      PhaseIn<Real, SPT> q;
      if (phase_sites<0, SPT>(a, r, b, base + threadIdx.x, step, q.ps)) return;  // frozen plane
      pbase = ((uint32_t)q.ps[0].z + (uint32_t)r.N[2] * q.ps[0].t) * P;
      phase_load<Real, 0, SPT>(lat_base, a, r, q);
      phase_compute<Real, 0, KIND, SPT, false>(lat_base, a, r, q, v0, acc0, th0, pbase);
    }
    __syncthreads();
    for (uint32_t base = 0; base < P; base += step) {
      PhaseIn<Real, SPT> q;
      phase_sites<1, SPT>(a, r, b, base + threadIdx.x, step, q.ps);
      phase_load<Real, 1, SPT, 1>(lat_base, a, r, q);
      phase_load_nu0_lds<Real, SPT>(th0, pbase, q);
      phase_compute<Real, 1, KIND, SPT, MEAS>(lat_base, a, r, q, v, acc1);
    }
  }
  phase_finish<1, KIND, MEAS>(a, L, v, acc0 + acc1);
}

// The same two phases for batched replicas whose planes fit one workgroup: a
// workgroup takes as many planes of one replica as it has room for, whole
// wavefronts each (64 sites per wavefront, map: replica and first
// wavefront-chunk), so that replicas with small planes fill it as well as those
// with large ones.  A replica descriptor carries set_phase_blocks(r, 64); it is
// copied into registers, since after the first store its fields could only be
// reloaded through the vector memory path.  Each wavefront is k_pair's one-step
// form: all loads of both phases before phase 0 computes, two angles through
// LDS (the plane's own part of it).  Measured, 64 replicas of 8^4 to 24^3 x 32
// (11.7 M sites), binary32: overrelaxation 49 us, 71 us as two launches;
// Metropolis 91 us and 94 us.  MEAS: phase (parity, 1) measures, one row per
// workgroup.
template <typename Real, int KIND, bool MEAS>
__global__ __launch_bounds__(pair_max_block(sizeof(Real), 1)) void k_pair_packed(Real* __restrict__ lat_base, PhaseArgs a,
                                                                               const WalkBlock* __restrict__ map) {
  const uint32_t block = fetch_args<sizeof(Real*) + sizeof(PhaseArgs) + sizeof(WalkBlock*)>(blockIdx.x);
  extern __shared__ __align__(8) unsigned char pair_lds[];
  const uint32_t L = a.xcd ? xcd_remap(block, gridDim.x) : block;
  const WalkBlock e = map[L];
  const RepDesc r = a.reps[e.x];
  const uint32_t P = (uint32_t)r.sz;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t sub = mdiv(wave, r.div_bpp_m, r.div_bpp_s);  // plane of the workgroup
  const uint32_t room = mdiv(blockDim.x >> 6, r.div_bpp_m, r.div_bpp_s);
  const bool active = sub < room && e.y + wave < (uint32_t)r.nblk;
  Real* th0 = reinterpret_cast<Real*>(pair_lds) + sub * P;
  double v[2] = {0.0, 0.0};
  uint32_t acc = 0, pbase = 0;
  PhaseIn<Real, 1> q0, q1;
  if (active) {
    phase_site(r, e.y + wave, threadIdx.x & 63u, 64u, a.parity, q0.ps[0]);
    pbase = ((uint32_t)q0.ps[0].z + (uint32_t)r.N[2] * q0.ps[0].t) * P;
    q1.ps[0] = q0.ps[0];
    phase_load<Real, 0, 1>(lat_base, a, r, q0);
    pair1_load<Real, 1>(lat_base, a, r, q1);
    phase_compute<Real, 0, KIND, 1, false>(lat_base, a, r, q0, v, acc, th0, pbase);
    pair_take(pair_shared(q0.in[0]), q1.in[0], q1.th[0]);
  }
  __syncthreads();
  if (active) {
    phase_load_nu0_lds<Real, 1>(th0, pbase, q1);
    phase_compute<Real, 1, KIND, 1, MEAS>(lat_base, a, r, q1, v, acc);
  }
  phase_finish<1, KIND, MEAS>(a, L, v, acc);
}

// Reads a completion counter at device scope (sees other XCDs' increments);
// the value is wave-uniform.
__device__ __forceinline__ uint32_t chain_poll(const uint32_t* p) {
  return __builtin_amdgcn_readfirstlane(__hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

// Waits (one wavefront) until the completion counter *p reaches target, with
// a sleep between polls; after kChainSpin polls it records a timeout in *err
// and returns.
__device__ __forceinline__ void chain_wait(const uint32_t* p, uint32_t target, uint32_t* err) {
  for (uint32_t n = 0; chain_poll(p) < target; ++n) {
    if (n == kChainSpin) {
      if ((threadIdx.x & 63) == 0) __hip_atomic_store(err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      return;
    }
    __builtin_amdgcn_s_sleep(8);
  }
}

// One phase-MU workgroup of a fused pass (k_chain): chunk `chunk` of plane
// (z, t).  Each wavefront on its own:
//  1. (MU > 0) reads the counters of the phase-(MU - 1) planes of chain_deps
//     once, before its other loads, so that this read overlaps them;
//  2. issues the loads that no workgroup of this launch writes: the angles at
//     the other parity, the link's own angle, and theta_nu (nu > MU) at this
//     parity, which phase nu only overwrites after this wavefront is counted;
//  3. (MU > 0) waits until those counters are complete, if the first read did
//     not find them so;
//  4. loads theta_nu (nu < MU) at this parity at device scope;
//  5. updates its links and stores them at device scope (plus the
//     measurement row, the accept count);
//  6. waits for its stores to complete (s_waitcnt vmcnt(0)) and adds 1 to
//     the (MU, plane) counter at device scope.
// A (mu, plane) counter is complete when every wavefront of the plane's bpp
// workgroups has added to it (tgt: the launch's value, bpp * blockDim.x / 64
// above the previous launch's).  Device-scope stores and loads make the
// exchange coherent across the XCDs' L2 caches without the whole-cache
// write-back and invalidation of an agent-scope fence.
template <typename Real, int MU, int KIND, int SPT, bool MEAS>
__device__ __forceinline__ void chain_phase(Real* __restrict__ lat_base, const PhaseArgs& a, const ChainArgs& c,
                                            int32_t z, uint32_t t, uint32_t chunk) {
  const RepDesc& r = a.single;
  const uint32_t npl = (uint32_t)r.N[2] * (uint32_t)r.N[3];
  const uint32_t plane = (uint32_t)z + (uint32_t)r.N[2] * t;
  constexpr int DEFM = (1 << MU) - 1;
  PhaseIn<Real, SPT> q;
#pragma unroll
  for (int k = 0; k < SPT; ++k)
    phase_site_zt(r, z, t, chunk * (SPT * blockDim.x) + threadIdx.x + k * blockDim.x, a.parity, q.ps[k]);
  const uint32_t* dep[2] = {nullptr, nullptr};
  uint32_t seen[2] = {0, 0};
  int ndep = 0;
  if (MU > 0) {
    int dz[2], dt[2];
    ndep = chain_deps(MU, z, (int)t, r.N[2], r.N[3], dz, dt);
    for (int i = 0; i < ndep; ++i) {
      dep[i] = c.cnt + (size_t)(MU - 1) * npl + (uint32_t)dz[i] + (uint32_t)r.N[2] * (uint32_t)dt[i];
      seen[i] = chain_poll(dep[i]);
    }
  }
  phase_load<Real, MU, SPT, DEFM>(lat_base, a, r, q);
  if (MU > 0) {
    for (int i = 0; i < ndep; ++i)
      if (seen[i] < c.tgt[MU - 1]) chain_wait(dep[i], c.tgt[MU - 1], c.err);
    phase_load_dep<Real, MU, SPT, DEFM>(lat_base, r, q);
  }
  double v[2] = {0.0, 0.0};
  uint32_t acc = 0;
  phase_compute<Real, MU, KIND, SPT, MEAS, true>(lat_base, a, r, q, v, acc);
  phase_finish<MU, KIND, MEAS>(a, (uint32_t)((MU > 0 ? MU - 1 : 0) * npl + plane) * (uint32_t)r.bpp + chunk, v, acc);
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wavefront's stores have completed
  if ((threadIdx.x & 63) == 0)
    __hip_atomic_fetch_add(c.cnt + (size_t)MU * npl + plane, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The phases (parity, 0..3) of one pass of a single lattice in one launch:
// workgroup b runs entry b >> 3 of the schedule list (u1_chain.h) on the
// tile of XCD b & 7.  Results are those of four separate launches, bit for
// bit: each link update does the same arithmetic on the same angles.  MEAS
// makes phases 1-3 measuring.
template <typename Real, int KIND, int SPT, bool MEAS>
__global__ __launch_bounds__(512) void k_chain(Real* __restrict__ lat_base, PhaseArgs a, ChainArgs c) {
  const uint32_t block = fetch_args<sizeof(Real*) + sizeof(PhaseArgs) + sizeof(ChainArgs)>(blockIdx.x);
  const uint32_t x = block & 7u;
  const uint32_t e = c.sched[block >> 3];
  const uint32_t w = e >> 10, chunk = (e >> 2) & 0xFFu;
  const uint32_t wt = mdiv(w, c.bz_m, c.bz_s);
  const uint32_t t = (x >> c.tz_log2) * c.bt + wt;
  const int32_t z = (int32_t)((x & ((1u << c.tz_log2) - 1u)) * c.bz + (w - wt * c.bz));
  switch (e & 3u) {
    case 0: chain_phase<Real, 0, KIND, SPT, false>(lat_base, a, c, z, t, chunk); break;
    case 1: chain_phase<Real, 1, KIND, SPT, MEAS>(lat_base, a, c, z, t, chunk); break;
    case 2: chain_phase<Real, 2, KIND, SPT, MEAS>(lat_base, a, c, z, t, chunk); break;
    default: chain_phase<Real, 3, KIND, SPT, MEAS>(lat_base, a, c, z, t, chunk); break;
  }
}

template <typename Real>
__global__ __launch_bounds__(256) void k_hotstart(Real* __restrict__ lat, RepDesc r) {
  const int64_t l = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (l >= 4 * (int64_t)r.V) return;
  const u1r::U32x4 w = u1r::draw(r.seed, (uint32_t)l, 0u, u1r::ctr2(u1r::STREAM_HOTSTART, 0, 0), r.c3);
  lat[l] = (Real)(u1m::K_PI * (2.0 * u1r::u01_d(w.v[0]) - 1.0));
}

template <typename Real, int KIND, bool BATCHED, int SPT>
hipError_t launch_mu(int mu, Real* lat, const PhaseArgs& a, int nblocks, int block, hipStream_t s) {
  if (a.meas != nullptr) {
    // measuring phases: mu >= 1, no multilevel mask
    if (mu < 1 || a.ml != 0) return hipErrorInvalidValue;
    switch (mu) {
      case 1: k_phase<Real, 1, KIND, BATCHED, SPT, true><<<nblocks, block, 0, s>>>(lat, a); break;
      case 2: k_phase<Real, 2, KIND, BATCHED, SPT, true><<<nblocks, block, 0, s>>>(lat, a); break;
      default: k_phase<Real, 3, KIND, BATCHED, SPT, true><<<nblocks, block, 0, s>>>(lat, a); break;
    }
    return hipGetLastError();
  }
  switch (mu) {
    case 0: k_phase<Real, 0, KIND, BATCHED, SPT><<<nblocks, block, 0, s>>>(lat, a); break;
    case 1: k_phase<Real, 1, KIND, BATCHED, SPT><<<nblocks, block, 0, s>>>(lat, a); break;
    case 2: k_phase<Real, 2, KIND, BATCHED, SPT><<<nblocks, block, 0, s>>>(lat, a); break;
    default: k_phase<Real, 3, KIND, BATCHED, SPT><<<nblocks, block, 0, s>>>(lat, a); break;
  }
  return hipGetLastError();
}

template <typename Real, int KIND, bool BATCHED>
hipError_t launch_spt(int spt, int mu, Real* lat, const PhaseArgs& a, int nblocks, int block, hipStream_t s) {
  if (spt == 2) return launch_mu<Real, KIND, BATCHED, 2>(mu, lat, a, nblocks, block, s);
  if (spt == 4) {
    // four sites per thread only for binary32 (binary64 would exceed the register budget)
    if (sizeof(Real) != sizeof(float)) return hipErrorInvalidValue;
    return launch_mu<Real, KIND, BATCHED, (sizeof(Real) == sizeof(float) ? 4 : 1)>(mu, lat, a, nblocks, block, s);
  }
  return launch_mu<Real, KIND, BATCHED, 1>(mu, lat, a, nblocks, block, s);
}

template <typename Real>
hipError_t launch_prec(int kind, int mu, Real* lat, const PhaseArgs& a, int nblocks, int block, int spt,
                       hipStream_t s) {
  const bool batched = a.reps != nullptr;
  if (kind == KIND_METROPOLIS)
    return batched ? launch_spt<Real, KIND_METROPOLIS, true>(spt, mu, lat, a, nblocks, block, s)
                   : launch_spt<Real, KIND_METROPOLIS, false>(spt, mu, lat, a, nblocks, block, s);
  return batched ? launch_spt<Real, KIND_OVERRELAX, true>(spt, mu, lat, a, nblocks, block, s)
                 : launch_spt<Real, KIND_OVERRELAX, false>(spt, mu, lat, a, nblocks, block, s);
}

template <typename Real, int KIND, int SPT, bool MEAS>
void launch_pair_form(int form, Real* lat, const PhaseArgs& a, int nblocks, int block, size_t lds, hipStream_t s) {
  const RepDesc& r = a.single;
  const uint32_t packed = r.div_nxh_s | r.div_nz_s << 5 | r.div_tile_s << 10 | r.div_bz_s << 15 |
                          (uint32_t)a.parity << 20 | (a.xcd ? 1u : 0u) << 21 | (r.tile ? 1u : 0u) << 22 |
                          (uint32_t)a.ml << 23;
  if constexpr (SPT <= 3)
    if (form == PAIR_ONE_STEP) {
      k_pair<Real, KIND, SPT, MEAS, false, PAIR_ONE_STEP><<<nblocks, block, lds, s>>>(lat, (uint32_t)r.N[1], (uint32_t)r.N[2], (uint32_t)r.N[3],
                                                                      (uint32_t)r.nxh, r.div_nxh_m, r.div_nz_m, r.div_tile_m, r.div_bz_m, packed, a);
      return;
    }
  if constexpr (SPT == 1)
    if (form == PAIR_SKEW) {
      k_pair<Real, KIND, SPT, MEAS, false, PAIR_SKEW><<<nblocks, block, lds, s>>>(lat, (uint32_t)r.N[1], (uint32_t)r.N[2], (uint32_t)r.N[3],
                                                                      (uint32_t)r.nxh, r.div_nxh_m, r.div_nz_m, r.div_tile_m, r.div_bz_m, packed, a);
      return;
    }
  k_pair<Real, KIND, SPT, MEAS, false, PAIR_LOOP><<<nblocks, block, lds, s>>>(lat, (uint32_t)r.N[1], (uint32_t)r.N[2], (uint32_t)r.N[3],
                                                                      (uint32_t)r.nxh, r.div_nxh_m, r.div_nz_m, r.div_tile_m, r.div_bz_m, packed, a);
}

template <typename Real, int KIND, int SPT>
hipError_t launch_pair_meas(Real* lat, const PhaseArgs& a, int nblocks, int block, size_t lds, hipStream_t s) {
  if (a.reps != nullptr) {  // batched replicas: no measuring pairs; the form per workgroup
    if constexpr (SPT > 2) return hipErrorInvalidValue;  // no ensemble shape has them
    else k_pair<Real, KIND, SPT, false, true><<<nblocks, block, lds, s>>>(lat, 0, 0, 0, 0, 0, 0, 0, 0, 0, a);
    return hipGetLastError();
  }
  // a single lattice: its plane and row size fix the form
  const int64_t P = (int64_t)a.single.nxh * a.single.N[1], step = (int64_t)SPT * block;
  const bool meas = a.meas != nullptr;
  const int form = SPT <= 3 && P <= step                   ? PAIR_ONE_STEP
                   : SPT == 1 && step >= 2 * a.single.nxh ? PAIR_SKEW
                                                           : PAIR_LOOP;
  if (meas)
    launch_pair_form<Real, KIND, SPT, true>(form, lat, a, nblocks, block, lds, s);
  else
    launch_pair_form<Real, KIND, SPT, false>(form, lat, a, nblocks, block, lds, s);
  return hipGetLastError();
}

template <typename Real, int KIND>
hipError_t launch_pair_spt(int spt, Real* lat, const PhaseArgs& a, int nblocks, int block, size_t lds,
                           hipStream_t s) {
  constexpr bool F = sizeof(Real) == sizeof(float);
  if (spt == 2) return launch_pair_meas<Real, KIND, 2>(lat, a, nblocks, block, lds, s);
  if (spt == 3) return launch_pair_meas<Real, KIND, (F ? 3 : 1)>(lat, a, nblocks, block, lds, s);
  if (spt == 4) return launch_pair_meas<Real, KIND, (F ? 4 : 1)>(lat, a, nblocks, block, lds, s);
  return launch_pair_meas<Real, KIND, 1>(lat, a, nblocks, block, lds, s);
}

template <typename Real>
hipError_t launch_pair_prec(int kind, Real* lat, const PhaseArgs& a, int nblocks, int block, int spt, size_t lds,
                            hipStream_t s) {
  if (kind == KIND_METROPOLIS) return launch_pair_spt<Real, KIND_METROPOLIS>(spt, lat, a, nblocks, block, lds, s);
  return launch_pair_spt<Real, KIND_OVERRELAX>(spt, lat, a, nblocks, block, lds, s);
}

template <typename Real, int KIND>
hipError_t launch_packed_meas(Real* lat, const PhaseArgs& a, const WalkBlock* map, int nblocks, int block, size_t lds,
                              hipStream_t s) {
  if (a.meas != nullptr)
    k_pair_packed<Real, KIND, true><<<nblocks, block, lds, s>>>(lat, a, map);
  else
    k_pair_packed<Real, KIND, false><<<nblocks, block, lds, s>>>(lat, a, map);
  return hipGetLastError();
}
template <typename Real>
hipError_t launch_packed_prec(int kind, Real* lat, const PhaseArgs& a, const WalkBlock* map, int nblocks, int block,
                              size_t lds, hipStream_t s) {
  return kind == KIND_METROPOLIS ? launch_packed_meas<Real, KIND_METROPOLIS>(lat, a, map, nblocks, block, lds, s)
                                 : launch_packed_meas<Real, KIND_OVERRELAX>(lat, a, map, nblocks, block, lds, s);
}

template <typename Real, int KIND, int SPT>
hipError_t launch_chain_meas(Real* lat, const PhaseArgs& a, const ChainArgs& c, int nblocks, int block,
                             hipStream_t s) {
  if (a.meas != nullptr)
    k_chain<Real, KIND, SPT, true><<<nblocks, block, 0, s>>>(lat, a, c);
  else
    k_chain<Real, KIND, SPT, false><<<nblocks, block, 0, s>>>(lat, a, c);
  return hipGetLastError();
}

template <typename Real>
hipError_t launch_chain_prec(int kind, Real* lat, const PhaseArgs& a, const ChainArgs& c, int nblocks, int block,
                             int spt, hipStream_t s) {
  if (kind == KIND_METROPOLIS)
    return spt == 2 ? launch_chain_meas<Real, KIND_METROPOLIS, 2>(lat, a, c, nblocks, block, s)
                    : launch_chain_meas<Real, KIND_METROPOLIS, 1>(lat, a, c, nblocks, block, s);
  return spt == 2 ? launch_chain_meas<Real, KIND_OVERRELAX, 2>(lat, a, c, nblocks, block, s)
                  : launch_chain_meas<Real, KIND_OVERRELAX, 1>(lat, a, c, nblocks, block, s);
}

}  // namespace

PhaseArgs with_f32_constants(const PhaseArgs& a) {
  PhaseArgs b = a;
  const float amp = a.proposal == 0 ? u1m::KF_PI : (float)a.step;
  b.pscale_f = amp * 0x1p-31f;
  b.poff_f = amp;
  b.thm_f = a.proposal == 0 ? 0.0f : 1.0f;
  return b;
}

hipError_t launch_phase(int prec, int kind, int mu, void* lat_base, const PhaseArgs& a, int nblocks, int block,
                        int spt, hipStream_t s) {
  if (prec == PREC_F64) return launch_prec<double>(kind, mu, (double*)lat_base, a, nblocks, block, spt, s);
  return launch_prec<float>(kind, mu, (float*)lat_base, with_f32_constants(a), nblocks, block, spt, s);
}

hipError_t launch_pair(int prec, int kind, void* lat_base, const PhaseArgs& a, int nblocks, int block, int spt,
                       int plane_sites, hipStream_t s) {
  // whole wavefronts within the kernel's launch bound; the plane's angles in LDS
  if (!(spt == 1 || spt == 2 || ((spt == 3 || spt == 4) && prec != PREC_F64))) return hipErrorInvalidValue;
  const int elem = prec == PREC_F64 ? 8 : 4;
  const int maxb = pair_max_block(elem, spt);
  if (block < 64 || block > maxb || block % 64 != 0 || plane_sites < 1 || plane_sites > pair_max_plane(elem) ||
      (a.meas != nullptr && (a.ml != 0 || a.reps != nullptr)))
    return hipErrorInvalidValue;
  // single lattice: one chunk per plane, one workgroup per plane, plane_sites
  // its plane (batched: the replica table and block map carry the same layout
  // per replica, plane_sites the largest plane)
  if (a.reps == nullptr && (a.single.bpp != 1 || nblocks != a.single.N[2] * a.single.N[3] ||
                            plane_sites != a.single.nxh * a.single.N[1]))
    return hipErrorInvalidValue;
  const size_t lds = (size_t)plane_sites * (size_t)elem;
  if (prec == PREC_F64) return launch_pair_prec<double>(kind, (double*)lat_base, a, nblocks, block, spt, lds, s);
  return launch_pair_prec<float>(kind, (float*)lat_base, with_f32_constants(a), nblocks, block, spt, lds, s);
}

hipError_t launch_pair_packed(int prec, int kind, void* lat_base, const PhaseArgs& a, const WalkBlock* map, int nblocks,
                              int block, hipStream_t s) {
  const int elem = prec == PREC_F64 ? 8 : 4;
  if (block < 64 || block > pair_max_block(elem, 1) || block % 64 != 0 || a.reps == nullptr || a.ml != 0 ||
      a.accepts != nullptr || map == nullptr || nblocks < 1)
    return hipErrorInvalidValue;
  const size_t lds = (size_t)block * (size_t)elem;
  if (prec == PREC_F64) return launch_packed_prec<double>(kind, (double*)lat_base, a, map, nblocks, block, lds, s);
  return launch_packed_prec<float>(kind, (float*)lat_base, with_f32_constants(a), map, nblocks, block, lds, s);
}

hipError_t launch_chain(int prec, int kind, void* lat_base, const PhaseArgs& a, const ChainArgs& c, int nblocks,
                        int block, int spt, hipStream_t s) {
  const RepDesc& r = a.single;
  const int64_t P = (int64_t)r.nxh * r.N[1], chunk = (int64_t)block * spt;
  // a single unmasked lattice in a tz x (8 / tz) tiling, its planes cut into
  // bpp chunks of block * spt sites, whole wavefronts within the launch bound
  const int tz = c.tz_log2 <= 3 ? 1 << c.tz_log2 : 0;
  if (!(spt == 1 || spt == 2) || block < 64 || block > 512 || block % 64 != 0 || a.reps != nullptr || a.ml != 0 ||
      !chain_possible(r.N[2], r.N[3], r.bpp, tz) || c.bz * (uint32_t)tz != (uint32_t)r.N[2] ||
      c.bt * (uint32_t)(8 / tz) != (uint32_t)r.N[3] || (int64_t)r.bpp * chunk < P ||
      (int64_t)(r.bpp - 1) * chunk >= P || nblocks <= 0 || nblocks % 8 != 0 || c.sched == nullptr ||
      c.cnt == nullptr || c.err == nullptr)
    return hipErrorInvalidValue;
  if (prec == PREC_F64) return launch_chain_prec<double>(kind, (double*)lat_base, a, c, nblocks, block, spt, s);
  return launch_chain_prec<float>(kind, (float*)lat_base, with_f32_constants(a), c, nblocks, block, spt, s);
}

hipError_t launch_hotstart(int prec, void* lat, const RepDesc& r, int block, hipStream_t s) {
  const int64_t n = 4 * (int64_t)r.V;
  const int nb = (int)((n + block - 1) / block);
  if (prec == PREC_F64)
    k_hotstart<double><<<nb, block, 0, s>>>((double*)lat + r.lat_off, r);
  else
    k_hotstart<float><<<nb, block, 0, s>>>((float*)lat + r.lat_off, r);
  return hipGetLastError();
}

}  // namespace u1d
