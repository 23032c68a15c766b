// u1_die.hip -- a whole sweep of a small lattice in one launch, on one die.
//
// A sweep of a lattice of a few ten thousand sites is a chain of 8 phases per
// pass that are each over in a microsecond; a launch per one or two phases, or
// a fused parity pass with completion counters at device scope, costs two to
// three microseconds per phase whatever the phase does.  Here one workgroup per
// CU of one XCD runs all passes, with a barrier between phases whose counter
// and data live in that XCD's L2 (measured, barrier and exchange: 0.6 to 0.9 us
// with 8 to 32 workgroups; 2.6 to 6.2 us at device scope with 32 to 256).
//
// The dispatcher hands workgroup b to XCD (b + const) % 8, so the launch has
// eight times the workgroups that work and all but every eighth leave at once.
// Nothing depends on that: before the first store every workgroup reports its
// XCD, and unless all report the same one, stores and counters go to device
// scope.
//
// Barrier and order (control words: u1_die_sync.h).  A phase's workgroup first waits for its stores, then
// counts itself; the next phase's loads of angles that the phase before wrote
// come after the counter is complete.  All angle loads pass the L1 (device
// scope; on one XCD the L2 serves them).  Of its eighteen staple angles a phase
// (parity, mu) reads two that the phase before it wrote -- theta_{mu-1} at x and
// x + mu - (mu-1), or for mu = 0 theta_3 at x + e0 and x - e3 -- so the loads and
// four of the six staple terms of a thread's first site run while the barrier
// completes.  Write after read: a phase overwrites theta_mu(parity), which the
// phase before reads, and every workgroup has consumed its loads before it
// counts itself.
//
// Multilevel masks (a.ml): between two frozen slices t % ml == 0 the links of a
// slab -- spatial on its other slices, temporal on all -- depend on each other
// and on frozen links only.  Each slab is a sweep of its own, on the XCD of its
// number, and slabs on one XCD share its CUs.
//
// All workgroups of a barrier must be resident at once: an XCD is given at most
// 32, one per CU, and if other work keeps some of them out, one does the sweep
// alone (u1_die_sync.h).  The waits are bounded all the same, and a timeout is
// reported, not hung on.
//
// Bound by latency: 4^4 takes as long as 8^4.  One Metropolis and three
// overrelaxation passes, against the tuned launches: binary64 8^4 70 us against
// 79, 12^3 x 8 81 against 91; binary32 8^4 38 us against 52, 12^3 x 16 51
// against 62, 16^3 x 8 level at 50.  With more sites one XCD's arithmetic
// takes over (binary64 12^3 x 16: 112 us against 95; binary32 16^4: 84 against
// 56).  Masked sweeps at 24^4, every slab by itself: level 2 binary32 59 us against
// 74, binary64 131 against 157; level 4 71 against 81, 162 against 178.
#include "u1_kernels.h"
#include "u1_link.h"

namespace u1d {

namespace {

// The accesses of DieSync: thread 0's relaxed atomics in device memory.
struct DieMem {
  static constexpr uint32_t kSpin = 1u << 24;  // polls before a wait gives up: several seconds
  uint32_t* ctl;  // DIE_CTL words
  uint32_t* err;
  uint32_t polls;  // for the others to begin (DieArgs::patience)

  __device__ __forceinline__ bool leader() const { return threadIdx.x == 0; }
  __device__ __forceinline__ void barrier() const {
    __syncthreads();
    asm volatile("" ::: "memory");
  }
  __device__ __forceinline__ uint32_t patience() const { return polls; }
  __device__ __forceinline__ void drain() const { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
  __device__ __forceinline__ void pause() const { __builtin_amdgcn_s_sleep(1); }
  __device__ __forceinline__ uint32_t xcd() const { return __builtin_amdgcn_s_getreg(20 | (3 << 11)); }  // XCC_ID
  // thread 0's v; a barrier
  __device__ __forceinline__ uint32_t broadcast(uint32_t v) const {
    __shared__ uint32_t word;
    if (threadIdx.x == 0) word = v;
    barrier();
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)word);
  }
  __device__ __forceinline__ uint32_t load(int word) const {
    return __hip_atomic_load(ctl + word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __device__ __forceinline__ void store(int word, uint32_t v) const {
    __hip_atomic_store(ctl + word, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  // local: counted and read on one XCD only
  __device__ __forceinline__ void add(int word, uint32_t v, bool local) const {
    if (local)
      __hip_atomic_fetch_add(ctl + word, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    else
      __hip_atomic_fetch_add(ctl + word, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __device__ __forceinline__ uint32_t fetch_add(int word, uint32_t v) const {
    return __hip_atomic_fetch_add(ctl + word, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __device__ __forceinline__ uint32_t cas(int word, uint32_t want, uint32_t v) const {
    __hip_atomic_compare_exchange_strong(ctl + word, &want, v, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
    return want;  // what was there
  }
  __device__ __forceinline__ void timed_out() const {
    __hip_atomic_store(err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
};

// Angles of direction j (not MU) of the staple; the two of the direction that
// the phase before wrote only with DEP.
template <typename Real, int MU>
struct DieLoad {
  static constexpr int LATE = MU == 0 ? 2 : MU - 1;  // j of the direction with late angles
  const Real* lat;
  const RepDesc& r;
  uint32_t same, opp;
  const int32_t (&fwd)[4];
  const int32_t (&bwd)[4];
  template <bool EARLY, bool DEP>
  __device__ __forceinline__ void dir(StapleIn<Real>& in, int j) const {
    const int nu = j < MU ? j : j + 1;
    const Real* pm = lat + (size_t)MU * r.V;
    const Real* pn = lat + (size_t)nu * r.V;
    const bool late = j == LATE;
    if (EARLY) {
      in.b[j] = ldc(pm, opp + fwd[nu]);
      in.e[j] = ldc(pm, opp + bwd[nu]);
    }
    if (late && MU == 0 ? DEP : EARLY) {
      in.a[j] = ldc(pn, opp + fwd[MU]);
      in.f[j] = ldc(pn, opp + bwd[nu]);
    }
    if (late && MU != 0 ? DEP : EARLY) {
      in.c[j] = ldc(pn, same);
      in.d[j] = ldc(pn, same + (uint32_t)(fwd[MU] + bwd[nu]));
    }
  }
};

// What changes from phase to phase, apart from MU.
struct DieStep {
  int kind;
  bool meas;   // the last pass's parity 1
};

// The even/odd sites of a workgroup's slab, spatial and temporal phases: n of
// them from base on, this thread's first + k stride of those.  Wavefronts are
// dealt to the workgroups in turn, so that a phase with half the sites still
// uses every CU (binary32 level-2 sweep at 24^4: 70 -> 59 us, level 4 110 -> 77).
struct DieSites {
  uint32_t base, n, base3, n3, first, stride;
};

// One body per MU for all passes and sites: the kernel runs each of them a few
// times only, and its instructions are cold in every cache when it begins.
template <typename Real, int MU, bool MEAS>
__device__ __forceinline__ void die_phase(Real* __restrict__ lat, const PhaseArgs& a, const RepDesc& r, DieSync<DieMem>& sync,
                                          const DieSites& own, uint32_t& acc, double (&v)[4], const DieStep& step) {
  const uint32_t first = own.first, stride = own.stride;
  const uint32_t n = MU == 3 ? own.n3 : own.n, base = MU == 3 ? own.base3 : own.base;
  constexpr int LATE = DieLoad<Real, MU>::LATE;
  const bool aniso = r.aniso != 1.0;
  const Real xi = sizeof(Real) == sizeof(float) ? (Real)r.aniso_f : (Real)r.aniso;
#pragma nounroll
  for (uint32_t i = first; i == first || i - (threadIdx.x & 63u) < n; i += stride) {
    const bool valid = i < n;  // others: the last site, nothing stored
    const uint32_t id = base + (valid ? i : n - 1u);
    Site s;
    site_of(r, (int32_t)id, a.parity, s);
    const uint32_t same = (uint32_t)(a.parity * r.HV) + id, opp = (uint32_t)((1 - a.parity) * r.HV) + id;
    const DieLoad<Real, MU> load{lat, r, same, opp, s.fwd, s.bwd};
    StapleIn<Real> in;
    StapleTerm<Real> term[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) load.template dir<true, false>(in, j);
    Real th[1] = {ldc(lat + (size_t)MU * r.V, same)};
#pragma unroll
    for (int j = 0; j < 3; ++j)
      if (j != LATE) term[j] = staple_term(in, j);
    if (i == first) sync.wait();
    load.template dir<false, true>(in, LATE);
    term[LATE] = staple_term(in, LATE);
    PlaqPieces<Real> pp = {0, 0, 0, 0};
    const Staple<Real> S[1] = {staple_of<Real, MU, MEAS>(term, xi, (Real)r.inv_aniso_f, aniso, &pp)};
    const uint32_t l[1] = {same + (uint32_t)MU * (uint32_t)r.V};
    const uint64_t vm[1] = {wave_mask(valid)};
    if (step.kind == KIND_METROPOLIS)
      update_angles<Real, KIND_METROPOLIS, 1>(a, r, S, th, l, vm, acc);
    else
      update_angles<Real, KIND_OVERRELAX, 1>(a, r, S, th, l, vm, acc);
    if (valid) {
      if (sync.one)
        st(lat + (size_t)MU * r.V, same, th[0]);
      else
        stc(lat + (size_t)MU * r.V, same, th[0]);
    }
    if (MEAS && MU > 0)
      if (step.meas) add_plaquettes<Real, MU>(pp, th[0], valid, v[MU == 3 ? 2 : 0], v[MU == 3 ? 3 : 1]);
  }
  sync.arrive();
}

template <typename Real, bool MEAS>
__global__ __launch_bounds__(die_max_block(sizeof(Real))) void k_die(Real* __restrict__ lat_base, PhaseArgs a, DieArgs d) {
  const uint32_t block = fetch_args<sizeof(Real*) + sizeof(PhaseArgs) + sizeof(DieArgs)>(blockIdx.x);
  const RepDesc& r = a.single;
  // place in the slab: by the XCD that the dispatcher hands the workgroup to, or in order
  const uint32_t k = d.in_order ? block : block >> 3, row = k / d.groups, wg = k - row * d.groups;
  const uint32_t slab = d.in_order ? row : 8u * row + (block & 7u);
  if (slab >= d.slabs) return;
  Real* lat = lat_base + r.lat_off;
  DieSync<DieMem> sync{{d.ctl + slab * DIE_CTL, d.err, d.patience}, d.groups, wg, d.groups, 0, false, false};
  sync.start();
  const uint32_t half = (uint32_t)r.st;  // even/odd sites of a slice
  const uint32_t t0 = slab * (uint32_t)a.ml, nt = a.ml ? min((uint32_t)a.ml, (uint32_t)r.N[3] - t0) : (uint32_t)r.N[3];
  const uint32_t frozen = a.ml ? 1u : 0u;
  DieSites own = {(t0 + frozen) * half, (nt - frozen) * half, t0 * half, nt * half,
                  ((threadIdx.x >> 6) * d.groups + wg) * 64u + (threadIdx.x & 63u), d.groups * blockDim.x};
  // In front of the first phase and not, as the other waits, behind its loads: the
  // choice there cost every phase registers (8^4 with plaquette 102 us per call, 97
  // here).  One addition carries both count and XCDs, and thread 0 hands on what it
  // polled: with an addition each, and a load by all threads, a sweep took 2 us more
  // (binary64 8^4 75.7 -> 73.9, binary32 16^3 x 8 55.4 -> 53.4).
  sync.started();
  if (sync.n == 0) {
    sync.leave();
    return;
  }
  if (sync.n != sync.all) {  // alone: all sites
    own.first = threadIdx.x;
    own.stride = blockDim.x;
  }
  uint32_t acc = 0;
  double v[4] = {0.0, 0.0, 0.0, 0.0};
  // (pass, parity) by (pass, parity)
  const int halves = 2 * (d.metrop + d.ovrn);
#pragma nounroll
  for (int h = 0; h < halves; ++h) {
    const bool metro = h < 2 * d.metrop;
    a.pass = (uint32_t)((metro ? h : h - 2 * d.metrop) >> 1);
    a.parity = h & 1;
    const DieStep step = {metro ? KIND_METROPOLIS : KIND_OVERRELAX, h == halves - 1};
    die_phase<Real, 0, MEAS>(lat, a, r, sync, own, acc, v, step);
    die_phase<Real, 1, MEAS>(lat, a, r, sync, own, acc, v, step);
    die_phase<Real, 2, MEAS>(lat, a, r, sync, own, acc, v, step);
    die_phase<Real, 3, MEAS>(lat, a, r, sync, own, acc, v, step);
    // four phases at a time: of at most 2^16 sites and 8190 hits each, acc holds them,
    // but not those of many passes
    if (a.accepts && (threadIdx.x & 63) == 0 && acc) atomicAdd(a.accepts, (unsigned long long)acc);
    acc = 0;
  }
  if (MEAS) {
    // one row per workgroup, folded in their order by the first
    const double o = block_sum<4>(v);
    if (threadIdx.x < 4) stc(a.meas, 4 * sync.wg + threadIdx.x, o);
    sync.arrive();
    if (sync.wg == 0) {
      sync.wait();
      if (threadIdx.x < 4) {
        double s = 0.0;
        for (uint32_t g = 0; g < sync.n; ++g) s += ldc(a.meas, 4 * g + threadIdx.x);
        d.out[threadIdx.x] = s * d.scale;
      }
    }
  }
  sync.leave();
}

template <typename Real>
hipError_t launch_die_prec(Real* lat, const PhaseArgs& a, const DieArgs& d, int block, hipStream_t s) {
  const uint32_t grid = 8u * die_rows(d.slabs) * d.groups;
  if (a.meas)
    k_die<Real, true><<<grid, block, 0, s>>>(lat, a, d);
  else
    k_die<Real, false><<<grid, block, 0, s>>>(lat, a, d);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_die(int prec, void* lat, const PhaseArgs& a, const DieArgs& d, int block, hipStream_t s) {
  const uint32_t ml = (uint32_t)a.ml, nt = (uint32_t)a.single.N[3];
  if (block < 64 || block > die_max_block(prec == PREC_F64 ? 8 : 4) || block % 64 != 0 || !(ml == 0 || ml == 2 || ml == 4) || nt % 2 != 0 ||
      d.slabs != die_slabs(a.ml, a.single.N[3]) || d.groups < 1 || die_rows(d.slabs) * d.groups > kDieGroups || a.reps ||
      d.metrop < 0 || d.ovrn < 0 || d.metrop + d.ovrn == 0 || !d.ctl || !d.err || (a.meas && (!d.out || ml != 0)))
    return hipErrorInvalidValue;
  if (prec == PREC_F64) return launch_die_prec<double>((double*)lat, a, d, block, s);
  return launch_die_prec<float>((float*)lat, with_f32_constants(a), d, block, s);
}

}  // namespace u1d
