// u1_walk.hip -- kernels of the diagonal walks (u1_walk.h): two checkerboard
// phases of a pass in one launch.  Every update is the phases' own arithmetic
// on the same angles (u1_link.h), so the results are those of two launches bit
// for bit.
#include "u1_walk.h"

#include "u1_link.h"

namespace u1d {

namespace {

typedef __attribute__((ext_vector_type(2))) uint32_t U32x2;

// The four directions' angles as raw buffers: an access is a uniform byte
// offset (a scalar register) plus a lane byte offset, with no 64-bit vector
// address to form.  Each buffer spans one direction's V angles (< 4 GiB).
template <typename Real>
struct WalkMem {
  __amdgpu_buffer_rsrc_t dir[4];
  __device__ __forceinline__ WalkMem(Real* lat, const RepDesc& r) {
#pragma unroll
    for (int mu = 0; mu < 4; ++mu)
      dir[mu] = __builtin_amdgcn_make_buffer_rsrc(lat + (size_t)mu * r.V, 0, (int)((uint32_t)r.V * (uint32_t)sizeof(Real)),
                                                  0x00027000);
  }
  __device__ __forceinline__ Real operator()(int mu, uint32_t base, uint32_t off) const {
    if constexpr (sizeof(Real) == 4)
      return __builtin_bit_cast(Real, __builtin_amdgcn_raw_buffer_load_b32(dir[mu], (int)off, (int)base, 0));
    else
      return __builtin_bit_cast(Real, __builtin_amdgcn_raw_buffer_load_b64(dir[mu], (int)off, (int)base, 0));
  }
  __device__ __forceinline__ void store(int mu, const WalkPos& p, Real v) const {
    const int base = __builtin_amdgcn_readfirstlane((int)p.base);  // uniform, which the compiler does not always see
    if constexpr (sizeof(Real) == 4)
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), dir[mu], (int)p.off, base, 0);
    else
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U32x2, v), dir[mu], (int)p.off, base, 0);
  }
};

// The six angles of direction DIR in the staple of a MU link (StapleIn).
template <typename Real, int MU, int DIR>
__device__ __forceinline__ void staple_dir(StapleIn<Real>& in, Real a, Real b, Real c, Real d, Real e, Real f) {
  constexpr int j = DIR < MU ? DIR : DIR - 1;
  in.a[j] = a;
  in.b[j] = b;
  in.c[j] = c;
  in.d[j] = d;
  in.e[j] = e;
  in.f[j] = f;
}

// One link update of a walk; returns the new angle.
template <typename Real, int MU, int KIND, bool MEAS>
__device__ __forceinline__ Real walk_update(const WalkMem<Real>& mem, const PhaseArgs& a, const RepDesc& r,
                                            const StapleIn<Real>& in, Real th_old, const WalkPos& p, bool valid,
                                            uint64_t vmask, double& re_sum, double& im_sum, uint32_t& acc) {
  const Real xi = sizeof(Real) == sizeof(float) ? (Real)r.aniso_f : (Real)r.aniso;
  PlaqPieces<Real> pp = {0, 0, 0, 0};
  const Staple<Real> S[1] = {staple_sum<Real, MU, MEAS>(in, xi, (Real)r.inv_aniso_f, r.aniso != 1.0, &pp)};
  Real th[1] = {th_old};
  const uint32_t l[1] = {p.off / (uint32_t)sizeof(Real) + (p.base / (uint32_t)sizeof(Real) + MU * (uint32_t)r.V)};
  const uint64_t vm[1] = {vmask};
  update_angles<Real, KIND, 1>(a, r, S, th, l, vm, acc);
  if (valid) mem.store(MU, p, th[0]);
  if (MEAS) add_plaquettes<Real, MU>(pp, th[0], valid, re_sum, im_sum);
  return th[0];
}

// Measured, binary32 overrelaxation, per launch against the two phase launches
// it replaces: 23.5 us against 31.2 us at 48^4 (lattice in the MALL), 407 us
// against 630 us at 96^4 (from HBM: 1.70 GB compulsory, 4.2 TB/s), 6.7 us
// against 8.5 us at 24^3 x 48, 5.1 us against 7.4 us at 24^4.  78 vector
// instructions per link (uniform form) where a phase issues 108-120: offsets
// instead of per-load addresses.  At 48^4 the vector units are 70 % busy and
// 108 workgroups per XCD of 64 sites each leave 12 of its 32 CUs with a fourth
// workgroup; segments of 32 sites halve that unit, which is why narrow strips
// win there in spite of their extra instructions.  Metropolis is bound by its
// arithmetic: level with two launches in the caches, 548 us against 659 us at
// 96^4.  Binary64 is arithmetic-bound throughout and seldom gains.
enum { WALK_PLAIN = 0, WALK_MEAS = 1, WALK_MASK = 2 };

// The two phases (parity, 2) and (parity, 3) of one lattice (walk_args).  MODE
// WALK_MEAS: also the plaquette sums of both, one row of a.meas per strip and
// diagonal; WALK_MASK: with the multilevel mask a.ml (frozen slices keep
// theta_2).  Every wavefront leaves the first new theta_2 of its segments in
// LDS, meets the barrier, and takes the last one it needs from there.
// BATCHED: all replicas of an ensemble (WalkBatch), each with its own
// descriptor, copied into registers before the first store.  64 replicas of
// 8^4 to 24^3 x 32 (11.7 M sites), binary32: overrelaxation 44 us against
// 63 us for the two phase launches, Metropolis 82 us against 91 us.
// The arguments before a (single lattices) are the fourteen words that the
// dispatcher writes into scalar registers, as for k_pair: what a walk needs before
// its first load.  packed: shifts of the four magic divisions by five bits, parity,
// log2 of width and sg, plain order.  Binary32 at 24^3 x 48: overrelaxation 6.07 ->
// 5.84 us, Metropolis 9.35 -> 9.17; binary64 at 24^3 x 12: overrelaxation 6.3 -> 6.1.
template <typename Real, int KIND, int MODE, bool UNIFORM, bool BATCHED = false>
__global__ __launch_bounds__(64 * walk_max_waves(sizeof(Real))) void k_walk(
    Real* __restrict__ lat_base, uint32_t N1, uint32_t N2, uint32_t N3, uint32_t nxh, uint32_t div_nxh_m,
    uint32_t div_nz_m, uint32_t div_nt_m, uint32_t gs_m, uint32_t orbits, uint32_t len, uint32_t seg_len,
    uint32_t packed, PhaseArgs a, WalkBatch w) {
  // binary64 Metropolis is short of scalar registers and reads its other arguments
  // again and again: all lines at once (8.0 us at 24^3 x 12, 8.6 without)
  constexpr bool FETCH = BATCHED || (sizeof(Real) == 8 && KIND == KIND_METROPOLIS);
  const uint32_t block =
      FETCH ? fetch_args<sizeof(Real*) + 48 + sizeof(PhaseArgs) + sizeof(WalkBatch)>(blockIdx.x) : blockIdx.x;
  using Walk = WalkZT<sizeof(Real), UNIFORM>;
  constexpr int A = Walk::A, B = Walk::B, C = Walk::C, D = Walk::D;
  constexpr bool MEAS = MODE == WALK_MEAS;
  __shared__ Real first[64 * walk_max_waves(sizeof(Real))];
  uint32_t strip, orbit;
  RepDesc r;
  WalkArgs wa;
  if constexpr (BATCHED) {
    const WalkBlock e = w.map[block];
    if (e.x == kWalkNone) return;
    r = a.reps[e.x];
    wa = w.args[e.x];
    (void)walk_place(wa, e.y, &strip, &orbit);  // never empty in plain order
  } else {
    a.parity = (int32_t)(packed >> 20 & 1u);
    r = a.single;
    r.N[1] = (int32_t)N1;
    r.N[2] = (int32_t)N2;
    r.N[3] = (int32_t)N3;
    r.nxh = r.sy = (int32_t)nxh;
    r.sz = (int32_t)(nxh * N1);
    r.st = (int32_t)(nxh * N1 * N2);
    r.HV = (int32_t)(nxh * N1 * N2 * N3);
    r.V = 2 * r.HV;
    r.lat_off = 0;
    r.div_nxh_m = div_nxh_m;
    r.div_nxh_s = packed & 31u;
    r.div_nz_m = div_nz_m;
    r.div_nz_s = packed >> 5 & 31u;
    const uint32_t wlog = packed >> 21 & 7u, sglog = packed >> 24 & 3u;
    const bool plain = (packed >> 26 & 1u) != 0;
    wa.nt_m = div_nt_m;
    wa.nt_s = packed >> 10 & 31u;
    wa.gs_m = gs_m;
    wa.gs_s = packed >> 15 & 31u;
    wa.orbits = (int32_t)orbits;
    wa.len = (int32_t)len;
    wa.seg = (int32_t)seg_len;
    wa.width = 1 << wlog;
    wa.strips = (int32_t)(((uint32_t)r.sz + (uint32_t)wa.width - 1u) >> wlog);
    wa.sg = plain ? 0 : 1 << sglog;
    wa.gs = plain ? wa.strips : (int32_t)(((uint32_t)wa.strips + (uint32_t)wa.sg - 1u) >> sglog);
    wa.go = plain ? wa.orbits : (int32_t)((orbits + (8u >> sglog) - 1u) >> (3u - sglog));
    wa.row = 0;
    if (!walk_place(wa, block, &strip, &orbit)) return;
  }
  // segment of this lane, and its place in the strip
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t seg = UNIFORM ? wave : threadIdx.x >> __builtin_ctz((uint32_t)wa.width);
  const uint32_t lane = UNIFORM ? threadIdx.x & 63u : threadIdx.x & (uint32_t)(wa.width - 1);
  const int32_t j0 = (int32_t)seg * wa.seg, j1 = min(j0 + wa.seg, wa.len);
  const int32_t steps = UNIFORM ? j1 - j0 : wa.seg;  // uniform over the wavefront
  const uint32_t P = (uint32_t)r.sz, site = strip * (uint32_t)wa.width + lane;
  const bool valid = site < P;
  Walk wk;
  // lanes past the end of the plane walk its last site and store nothing
  // (by magic: the compiler's divisions ran one after the other before the first
  // load: a sweep of 16 launches took 118.9 us at 24^3 x 48, binary32, 117.3 now)
  const uint32_t jt = orbit + (uint32_t)j0;
  wk.init(r, a.parity, valid ? site : P - 1, (int32_t)orbit,
          j0 - r.N[2] * (int32_t)mdiv((uint32_t)j0, r.div_nz_m, r.div_nz_s),
          (int32_t)(jt - (uint32_t)r.N[3] * mdiv(jt, wa.nt_m, wa.nt_s)));
  const WalkMem<Real> mem(lat_base + r.lat_off, r);
  const uint32_t ml1 = (uint32_t)a.ml - 1u;
  const uint64_t vmask = KIND == KIND_METROPOLIS ? wave_mask(valid) : 0;
  double v[4] = {0.0, 0.0, 0.0, 0.0};
  uint32_t acc = 0;
  auto update_a = [&](const RungSite<Real>& q, const WalkPos& p, const Rung<Real>& r0, const Rung<Real>& r1,
                      Real before) -> Real {
    const bool moves = MODE != WALK_MASK || ((uint32_t)p.t & ml1) != 0;
    if (MODE == WALK_MASK && UNIFORM && !moves) return q.x[0];  // uniform
    StapleIn<Real> in;
    staple_dir<Real, A, B>(in, r0.u[1], r1.u[0], q.x[1], before, r0.va, r0.vb);
    staple_dir<Real, A, C>(in, r0.u[2], q.ap[0], q.x[2], r0.w[0], q.am[0], q.f[0]);
    staple_dir<Real, A, D>(in, r0.u[3], q.ap[1], q.x[3], r0.w[1], q.am[1], q.f[1]);
    const uint64_t vm = MODE == WALK_MASK && KIND == KIND_METROPOLIS ? wave_mask(valid && moves) : vmask;
    const Real n = walk_update<Real, A, KIND, MEAS>(mem, a, r, in, q.x[0], p, valid && moves, vm, v[0], v[1], acc);
    return moves ? n : q.x[0];
  };
  auto update_b = [&](const RungSite<Real>& q, const WalkPos& p, Real ub, const Rung<Real>& r1, Real n0, Real n1) {
    StapleIn<Real> in;
    staple_dir<Real, B, A>(in, r1.u[0], ub, n0, n1, r1.vb, r1.va);
    staple_dir<Real, B, C>(in, r1.u[2], q.bp[0], q.x[2], r1.w[0], q.bm[0], q.f[0]);
    staple_dir<Real, B, D>(in, r1.u[3], q.bp[1], q.x[3], r1.w[1], q.bm[1], q.f[1]);
    walk_update<Real, B, KIND, MEAS>(mem, a, r, in, q.x[1], p, valid, vmask, v[2], v[3], acc);
  };
  WalkSegment<Real, Walk, WalkMem<Real>, decltype(update_a), decltype(update_b)> sg{wk, mem, update_a, update_b};
  if (steps > 0) first[threadIdx.x] = sg.first();
  __syncthreads();
  if (steps > 0)
    sg.template rest<KIND == KIND_OVERRELAX>(
        steps, [&] { return first[j1 == wa.len ? lane : threadIdx.x + (uint32_t)wa.width]; });
  if (MEAS) {
    const double o = block_sum<4>(v);
    if (threadIdx.x < 4)
      a.meas[4 * ((size_t)(uint32_t)wa.row + (size_t)orbit * (uint32_t)wa.strips + strip) + threadIdx.x] = o;
  }
  if (KIND == KIND_METROPOLIS && a.accepts && (threadIdx.x & 63) == 0 && acc)
    atomicAdd(a.accepts, (unsigned long long)acc);
}

template <typename Real, int KIND, int MODE>
hipError_t launch_walk_batch_width(Real* lat, const PhaseArgs& a, const WalkBatch& w, int nblk, int block, int width,
                                   hipStream_t s) {
  if (width == 64)
    k_walk<Real, KIND, MODE, true, true><<<nblk, block, 0, s>>>(lat, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, a, w);
  else
    k_walk<Real, KIND, MODE, false, true><<<nblk, block, 0, s>>>(lat, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, a, w);
  return hipGetLastError();
}
template <typename Real, int KIND>
hipError_t launch_walk_batch(Real* lat, const PhaseArgs& a, const WalkBatch& w, int nblk, int block, int width,
                             hipStream_t s) {
  return a.meas != nullptr ? launch_walk_batch_width<Real, KIND, WALK_MEAS>(lat, a, w, nblk, block, width, s)
                           : launch_walk_batch_width<Real, KIND, WALK_PLAIN>(lat, a, w, nblk, block, width, s);
}
template <typename Real>
hipError_t launch_walk_batch_prec(int kind, Real* lat, const PhaseArgs& a, const WalkBatch& w, int nblk, int block,
                                  int width, hipStream_t s) {
  return kind == KIND_METROPOLIS ? launch_walk_batch<Real, KIND_METROPOLIS>(lat, a, w, nblk, block, width, s)
                                 : launch_walk_batch<Real, KIND_OVERRELAX>(lat, a, w, nblk, block, width, s);
}

template <typename Real, int KIND, int MODE>
hipError_t launch_walk_width(Real* lat, const PhaseArgs& a, const WalkArgs& w, int block, hipStream_t s) {
  const RepDesc& r = a.single;
  auto* k = w.width == 64 ? k_walk<Real, KIND, MODE, true, false> : k_walk<Real, KIND, MODE, false, false>;
  const uint32_t packed = r.div_nxh_s | r.div_nz_s << 5 | w.nt_s << 10 | w.gs_s << 15 | (uint32_t)a.parity << 20 |
                          (uint32_t)__builtin_ctz((uint32_t)w.width) << 21 |
                          (w.sg ? (uint32_t)__builtin_ctz((uint32_t)w.sg) << 24 : 1u << 26);
  k<<<walk_blocks(w), block, 0, s>>>(lat, (uint32_t)r.N[1], (uint32_t)r.N[2], (uint32_t)r.N[3], (uint32_t)r.nxh,
                                     r.div_nxh_m, r.div_nz_m, w.nt_m, w.gs_m, (uint32_t)w.orbits, (uint32_t)w.len,
                                     (uint32_t)w.seg, packed, a, WalkBatch{});
  return hipGetLastError();
}

template <typename Real, int KIND>
hipError_t launch_walk_mode(Real* lat, const PhaseArgs& a, const WalkArgs& w, int block, hipStream_t s) {
  if (a.meas != nullptr) return launch_walk_width<Real, KIND, WALK_MEAS>(lat, a, w, block, s);
  if (a.ml != 0) return launch_walk_width<Real, KIND, WALK_MASK>(lat, a, w, block, s);
  return launch_walk_width<Real, KIND, WALK_PLAIN>(lat, a, w, block, s);
}

template <typename Real>
hipError_t launch_walk_prec(int kind, Real* lat, const PhaseArgs& a, const WalkArgs& w, int block, hipStream_t s) {
  return kind == KIND_METROPOLIS ? launch_walk_mode<Real, KIND_METROPOLIS>(lat, a, w, block, s)
                                 : launch_walk_mode<Real, KIND_OVERRELAX>(lat, a, w, block, s);
}

}  // namespace

hipError_t launch_walk(int prec, int kind, void* lat_base, const PhaseArgs& a, int block, int width, int sg,
                       hipStream_t s) {
  if (!walk_shape_ok(a.single, prec == PREC_F64 ? 8 : 4, block, width, sg) || a.reps != nullptr ||
      (a.meas != nullptr && a.ml != 0))
    return hipErrorInvalidValue;
  const WalkArgs w = walk_args(a.single, block / 64, width, sg);
  if (prec == PREC_F64) return launch_walk_prec<double>(kind, (double*)lat_base, a, w, block, s);
  return launch_walk_prec<float>(kind, (float*)lat_base, with_f32_constants(a), w, block, s);
}

hipError_t launch_walk_batched(int prec, int kind, void* lat_base, const PhaseArgs& a, const WalkBatch& w, int nblk,
                               int block, int width, hipStream_t s) {
  if (a.reps == nullptr || a.ml != 0 || nblk < 1) return hipErrorInvalidValue;
  if (prec == PREC_F64) return launch_walk_batch_prec<double>(kind, (double*)lat_base, a, w, nblk, block, width, s);
  return launch_walk_batch_prec<float>(kind, (float*)lat_base, with_f32_constants(a), w, nblk, block, width, s);
}

}  // namespace u1d
