// u1_measure.hip -- plaquette, Polyakov loop, Polyakov-loop volume (plain,
// analytic and stochastic multihit), correlator PP, layout conversions and
// plaquette fields.
//
// Reductions are deterministic: every workgroup writes its partial sums (DPP
// row sums within each wave64, then waves in order through LDS) to a partials
// buffer, and k_fold_rows / k_finish fold the rows in order -- replacing the reference's
// shared-memory fold plus one FP64 atomicAdd per block (reduce_block_1d.h:41-64,
// cudaAtomic.h:147-177), whose summation order is nondeterministic.  All sums
// are FP64 for both lattice precisions.
#include <algorithm>
#include <type_traits>

#include "u1_kernels.h"

namespace u1d {

namespace {

struct C64 {
  double re, im;
};
typedef double F64x2 __attribute__((ext_vector_type(2), aligned(8)));  // one 16-byte store, 8-byte aligned
// complex.h:205-217 ordering
__device__ __forceinline__ C64 cmul(C64 a, C64 b) { return {a.re * b.re - a.im * b.im, a.im * b.re + a.re * b.im}; }

// sin and cos of the measurement kernels: Prec's values (UMath<double>: but for
// sin(-0), a zero of either sign here).
template <typename Real>
__device__ __forceinline__ void msincos(Real x, Real* s, Real* c) {
  if constexpr (sizeof(Real) == 8)
    UMath<double>::sincos(x, s, c);
  else
    Prec<Real>::sincos(x, s, c);
}
template <typename Real>
__device__ __forceinline__ C64 exp_i(Real a) {
  Real s, c;
  msincos<Real>(a, &s, &c);
  return {(double)c, (double)s};
}

// Temporal-link staple (staple.h:79-102 with mu = TDir): all six staples are
// space-time, weight xi.  Same operation order as the update kernels (their
// space-space term is 0 / xi = 0).
template <typename Real>
__device__ __forceinline__ void staple_t(const Real* __restrict__ lat, const RepDesc& r, const Site& s, int32_t id,
                                         int32_t parity, Real& Sre, Real& Sim) {
  const int32_t same = parity * r.HV + id;
  const int32_t opp = (1 - parity) * r.HV + id;
  const Real* pm = lat + 3 * (int64_t)r.V;
  Real str = 0, sti = 0;
#pragma unroll
  for (int nu = 0; nu < 3; ++nu) {
    const Real* pn = lat + (int64_t)nu * r.V;
    const Real a = ld(pn, opp + s.fwd[3]);
    const Real b = ld(pm, opp + s.fwd[nu]);
    const Real c = ld(pn, same);
    const Real d = ld(pn, same + s.fwd[3] + s.bwd[nu]);
    const Real e = ld(pm, opp + s.bwd[nu]);
    const Real f = ld(pn, opp + s.bwd[nu]);
    const Real up = (a - b) - c;
    const Real lo = ((-d) - e) + f;
    Real su, cu, sl, cl;
    msincos<Real>(up, &su, &cu);
    msincos<Real>(lo, &sl, &cl);
    str += cu + cl;
    sti += su + sl;
  }
  const Real xi = (Real)r.aniso;
  Sre = (Real)0 + str * xi;
  Sim = (Real)0 + sti * xi;
}

// nhit Metropolis hits of a temporal link with its staple fixed; returns the
// sums of cos and sin of the angle after each hit.  The proposals are those of
// the update kernels (one FMA for a (2u - 1): the same bits as the two-step
// form).  NEAR: every lane's angle starts in [-pi, pi], so theta + delta needs
// one wrap step each way (|delta| <= pi); otherwise wrap_d's four.  Bound by
// its vector instructions: a binary32 hit takes 62 of them (80 before the FMA
// proposal, the single wrap steps and the sign flips of u1m::sincos_f) and half
// a Philox draw.  The 100-hit correlator at 24^3 x 48 takes 136 us, 200 us
// before (about 30 us of that from the hits).
template <typename Real, bool NEAR>
__device__ __forceinline__ C64 multihit_sum(const RepDesc& r, Real th, Real Sre, Real Sim, uint32_t l, int proposal,
                                            int nhit, double step, uint32_t stream, uint32_t c1, uint32_t c3) {
  Real s0, c0;
  msincos<Real>(th, &s0, &c0);
  Real re_old = Sre * c0 - Sim * s0;
  const Real beta = (Real)r.beta;
  double ac = 0.0, as = 0.0;
  auto hit = [&](uint32_t wu, uint32_t wb) {
    double x;
    if (proposal == 0) {
      x = __builtin_fma((double)wu, u1m::K_PI * 0x1p-31, -u1m::K_PI);
    } else {
      x = (double)th + __builtin_fma((double)wu, step * 0x1p-31, -step);
      x = NEAR ? u1m::wrap_step_d(x) : u1m::wrap_d(x);
    }
    const Real tn = (Real)x;
    Real sn, cn;
    if constexpr (sizeof(Real) == 8) UMath<double>::sincos_in_loop(tn, &sn, &cn);
    else Prec<Real>::sincos(tn, &sn, &cn);
    const Real re_new = Sre * cn - Sim * sn;
    bool ok;
    if constexpr (sizeof(Real) == 8) ok = UMath<double>::accept(beta * (re_new - re_old), wb, r.exp_small != 0);
    else ok = Prec<Real>::exp(beta * (re_new - re_old)) > Prec<Real>::u01(wb);
    if (ok) {
      th = tn;
      re_old = re_new;
      s0 = sn;
      c0 = cn;
    }
    ac += (double)c0;
    as += (double)s0;
  };
  // hits 2j and 2j + 1 read words (0, 1) and (2, 3) of one Philox call
  for (int h = 0; h < nhit; h += 2) {
    const u1r::U32x4 w = u1r::draw(r.seed, l, c1, u1r::ctr2(stream, 0, (uint32_t)(h >> 1)), c3);
    hit(w.v[0], w.v[1]);
    if (h + 1 < nhit) hit(w.v[2], w.v[3]);
  }
  return {ac, as};
}

// Temporal link value at even/odd site (id, parity) = s: e^{i theta_t}, the
// analytic multihit mean (lattice_functions.h:92-105) or the stochastic nhit
// mean.  MODE 0, 1, 2.
template <typename Real, int MODE>
__device__ __forceinline__ C64 temporal_value(const Real* __restrict__ lat, const RepDesc& r, const Site& s, int32_t id,
                                              int32_t parity, int proposal, int nhit, double step, uint32_t stream,
                                              uint32_t c1, uint32_t c3) {
  const int32_t l = id + parity * r.HV + 3 * r.V;
  if (MODE == 0) return exp_i<Real>(lat[l]);
  Real Sre, Sim;
  staple_t<Real>(lat, r, s, id, parity, Sre, Sim);
  if (MODE == 1) {
    // (binary64 at 32^3 x 16: 22.6 us per field with two divisions per series
    // term, 13.4 us with the polynomials)
    // conj(S) I1(x) / (I0(x) |S|), x = beta |S|: (beta / 2) conj(S) times a
    // function of x^2, so that no square root and one division are left
    const double sr = (double)Sre, si = (double)Sim, a2 = sr * sr + si * si;
    if (a2 == 0.0) return {0.0, 0.0};
    const double temp = 0.5 * r.beta * u1m::bessel_ratio_d(0.25 * (r.beta * r.beta) * a2);
    return {temp * sr, -temp * si};
  }
  const Real th = lat[l];
  // (the negated test also sends NaN the general way)
  const bool near = __all(!((double)th > 3.1415927410125733 || (double)th < -3.1415927410125733) && th == th);
  const C64 sum = near ? multihit_sum<Real, true>(r, th, Sre, Sim, (uint32_t)l, proposal, nhit, step, stream, c1, c3)
                       : multihit_sum<Real, false>(r, th, Sre, Sim, (uint32_t)l, proposal, nhit, step, stream, c1, c3);
  return {sum.re / (double)nhit, sum.im / (double)nhit};
}

// plaquette.cu:93-118: per site, sum over mu < nu of 1 - e^{iP}, split into
// space-space and space-time; P = ((t_mu(x) + t_nu(x+mu)) - t_mu(x+nu)) - t_nu(x).
//
// Decomposition as the update phases (one chunk of one (z, t) plane per
// workgroup, uniform z/t, SGPR-based loads, XCD-aware order), over both
// parities: the first nblk/2 workgroups of a replica take the even sites, the
// rest the odd sites.  SPT sites per thread.  A site reads its four links and
// the twelve forward neighbours it needs (16 loads; every link is read by four
// sites, mostly from L2).  The three plaquettes of each class are added in
// Real, then once per site into the FP64 accumulators.
template <typename Real, bool BATCHED, int SPT>
__global__ __launch_bounds__(256) void k_plaquette(const Real* __restrict__ lat_base, RepDesc single,
                                                   const RepDesc* reps, const uint16_t* blockmap,
                                                   double* __restrict__ partials) {
  const uint32_t L = xcd_remap(blockIdx.x, gridDim.x);
  const RepDesc& r = BATCHED ? reps[blockmap[L]] : single;
  const Real* lat = lat_base + r.lat_off;
  uint32_t b = L - (uint32_t)r.blk_begin;
  const uint32_t half = (uint32_t)r.nblk >> 1;
  const int32_t parity = b >= half ? 1 : 0;
  if (parity) b -= half;
  PhaseSite ps[SPT];
#pragma unroll
  for (int k = 0; k < SPT; ++k) phase_site(r, b, threadIdx.x + k * blockDim.x, SPT * blockDim.x, parity, ps[k]);
  Real tm[SPT][4], tf[SPT][4][4];  // tf[k][nu][mu] = theta_nu(x + mu), mu < nu or mu > nu
#pragma unroll
  for (int k = 0; k < SPT; ++k) {
    const uint32_t same = (uint32_t)(parity * r.HV) + ps[k].id;
    const uint32_t opp = (uint32_t)((1 - parity) * r.HV) + ps[k].id;
#pragma unroll
    for (int mu = 0; mu < 4; ++mu) tm[k][mu] = ld(lat + (size_t)mu * r.V, same);
#pragma unroll
    for (int mu = 0; mu < 4; ++mu)
#pragma unroll
      for (int nu = 0; nu < 4; ++nu)
        if (nu != mu) tf[k][nu][mu] = ld(lat + (size_t)nu * r.V, opp + ps[k].fwd[mu]);
  }
  double v[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int k = 0; k < SPT; ++k) {
    Real re[2] = {0, 0}, im[2] = {0, 0};
#pragma unroll
    for (int mu = 0; mu < 3; ++mu)
#pragma unroll
      for (int nu = mu + 1; nu < 4; ++nu) {
        const Real p = ((tm[k][mu] + tf[k][nu][mu]) - tf[k][mu][nu]) - tm[k][nu];
        Real sp, cp;
        msincos<Real>(p, &sp, &cp);
        const int c = nu == 3 ? 1 : 0;
        re[c] += (Real)1 - cp;
        im[c] -= sp;
      }
    if (ps[k].valid) {
      v[0] += (double)re[0];
      v[1] += (double)im[0];
      v[2] += (double)re[1];
      v[3] += (double)im[1];
    }
  }
  const double out = block_sum<4>(v);
  // row L (the logical workgroup): a batched fold reads each replica's rows
  // [blk_begin, blk_begin + nblk)
  if (threadIdx.x < 4) partials[4 * (int64_t)L + threadIdx.x] = out;
}

// polyakov.cu:60-77: sum of the temporal angles along t (in FP64), then e^{i.}.
template <typename Real>
__global__ __launch_bounds__(256) void k_polyakov(const Real* __restrict__ lat, RepDesc r,
                                                  double* __restrict__ partials) {
  const int32_t idx = (int32_t)(blockIdx.x * blockDim.x + threadIdx.x);
  double v[2] = {0.0, 0.0};
  if (idx < r.SV) {
    const int32_t half = r.SV / 2;
    const int32_t parity = idx >= half ? 1 : 0;
    const int32_t id = idx - parity * half;  // eo-id of (x, t = 0)
    const Real* pt = lat + 3 * (int64_t)r.V;
    double tmp = 0.0;
    // (loads in groups of eight: one after the other they were the whole time)
    int t = 0;
    for (; t + 8 <= r.N[3]; t += 8) {
      Real q[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) q[k] = pt[((parity + t + k) & 1) * r.HV + id + (t + k) * half];
#pragma unroll
      for (int k = 0; k < 8; ++k) tmp += (double)q[k];
    }
    for (; t < r.N[3]; ++t) tmp += (double)pt[((parity + t) & 1) * r.HV + id + t * half];
    double s, c;
    u1m::sincos_d(tmp, &s, &c);
    v[0] = c;
    v[1] = s;
  }
  const double out = block_sum<2>(v);
  if (threadIdx.x < 2) partials[2 * (int64_t)blockIdx.x + threadIdx.x] = out;
}

// Fold nblk partial rows of nv values in workgroup order; one workgroup per value.
// Up to kFoldRows rows it takes 2.3 to 4.5 us, a second level as much again: 2880
// rows of 4 values 3.2 us here, 2.8 us + 2.8 us and a launch in two levels.
__global__ __launch_bounds__(1024) void k_finish(const double* __restrict__ partials, int nblk, int nv, double scale,
                                                double* __restrict__ out) {
  const int k = blockIdx.x;
  double v[1] = {0.0};
  for (int i = threadIdx.x; i < nblk; i += blockDim.x) v[0] += partials[(int64_t)i * nv + k];
  const double o = block_sum<1>(v);
  if (threadIdx.x == 0) out[k] = o * scale;
}

// First level of a long fold: workgroup (g, k) adds rows [g R, g R + R) of
// column k into row g of l1 (same row layout, nv values per row).
__global__ __launch_bounds__(256) void k_fold_rows(const double* __restrict__ partials, int nrows, int nv, int R,
                                                   double* __restrict__ l1) {
  const int g = blockIdx.x, k = blockIdx.y;
  const int r0 = g * R, r1 = min(nrows, r0 + R);
  double v[1] = {0.0};
  for (int i = r0 + (int)threadIdx.x; i < r1; i += blockDim.x) v[0] += partials[(int64_t)i * nv + k];
  const double o = block_sum<1>(v);
  if (threadIdx.x == 0) l1[(int64_t)g * nv + k] = o;
}

// polyakov.cu:415-440 without multihit: P(x) = prod_t e^{i theta_t(x, t)},
// stored at the lexicographic spatial index (indexIdS).  The angles are loaded
// in groups of eight; the product keeps its order.
template <typename Real>
__global__ __launch_bounds__(256) void k_poly_volume(const Real* __restrict__ lat, RepDesc r, double* __restrict__ P) {
  const int32_t idx = (int32_t)(blockIdx.x * blockDim.x + threadIdx.x);
  if (idx >= r.SV) return;
  const int32_t half = r.SV / 2;
  const int32_t parity = idx >= half ? 1 : 0;
  const int32_t id = idx - parity * half;
  const Real* pt = lat + 3 * (int64_t)r.V;
  C64 res = {1.0, 0.0};
  int t = 0;
  for (; t + 8 <= r.N[3]; t += 8) {
    Real q[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) q[k] = pt[((parity + t + k) & 1) * r.HV + id + (t + k) * half];
#pragma unroll
    for (int k = 0; k < 8; ++k) res = cmul(res, exp_i<Real>(q[k]));
  }
  for (; t < r.N[3]; ++t) res = cmul(res, exp_i<Real>(pt[((parity + t) & 1) * r.HV + id + t * half]));
  Site s;
  site_of(r, id, parity, s);
  const int32_t j = s.x[0] + r.N[0] * (s.x[1] + r.N[1] * s.x[2]);
  P[2 * (int64_t)j] = res.re;
  P[2 * (int64_t)j + 1] = res.im;
}

// multilevel.cu:239-258: per-site temporal link at the lexicographic 4D index.
template <typename Real, int MODE>
__global__ __launch_bounds__(256) void k_temporal_links(const Real* __restrict__ lat, RepDesc r, int proposal, int nhit,
                                                        double step, uint32_t stream, uint32_t c1, uint32_t c3,
                                                        double* __restrict__ out) {
  const int32_t idx = (int32_t)(blockIdx.x * blockDim.x + threadIdx.x);
  if (idx >= r.V) return;
  const int32_t parity = idx >= r.HV ? 1 : 0;
  const int32_t id = idx - parity * r.HV;
  Site s;
  site_of(r, id, parity, s);
  const C64 v = temporal_value<Real, MODE>(lat, r, s, id, parity, proposal, nhit, step, stream, c1, c3);
  // lex = 2*id + (x0 & 1); x0 parity = (y + z + t + parity) & 1
  const int64_t j = 2 * (int64_t)id + (s.x[0] & 1);
  out[2 * j] = v.re;
  out[2 * j + 1] = v.im;
}

// Multilevel, level-2 step c = *ctr: the products of the temporal links of two
// slices, p2[l SV + x] = T(x, 2l) T(x, 2l + 1) (from 1, in the order of
// multilevel.cu:342-347; the product of the conjugates is its conjugate), into
// slot (c % n2) % slots of p2.  Philox counter word c1 = c.  The workgroup that
// finishes last advances the step counter, which the sweeps of the next step
// read: ctr[1] counts workgroups that have used ctr[0], so no launch of its
// own is needed for it (3.9 us per step).
template <typename Real, int MODE>
__global__ __launch_bounds__(256) void k_temporal_pairs(const Real* __restrict__ lat, RepDesc r, int proposal, int nhit,
                                                        double step, uint32_t stream, uint32_t c3,
                                                        double* __restrict__ p2, uint32_t* ctr, uint32_t n2,
                                                        uint32_t slots) {
  const uint32_t idx = blockIdx.x * blockDim.x + threadIdx.x, half = (uint32_t)r.SV / 2u;
  const uint32_t n = (uint32_t)r.SV * (uint32_t)(r.N[3] / 2), c = *(const volatile uint32_t*)ctr;
  if (idx < n) {
    const uint32_t l = idx / (uint32_t)r.SV, q = idx - l * (uint32_t)r.SV;
    const int32_t parity = q >= half ? 1 : 0;
    const int32_t i = (int32_t)(q - (parity ? half : 0u));  // eo-id of (x, t = 0)
    C64 p = {1.0, 0.0};
    int32_t odd = 0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int32_t id = i + (int32_t)((2 * l + h) * half), par = parity ^ h;
      Site s;
      site_of(r, id, par, s);
      odd = s.x[0] & 1;
      p = cmul(p, temporal_value<Real, MODE>(lat, r, s, id, par, proposal, nhit, step, stream, c, c3));
    }
    double* out = p2 + 2 * ((size_t)(c % n2 % slots) * n + (size_t)l * (uint32_t)r.SV + 2u * (uint32_t)i + (uint32_t)odd);
    out[0] = p.re;
    out[1] = p.im;
  }
  __syncthreads();  // every thread of the workgroup has used c
  if (threadIdx.x == 0 && atomicAdd(ctr + 1, 1u) == gridDim.x - 1) {
    ctr[1] = 0;
    ctr[0] = c + 1;
  }
}

// Product over t of a per-site temporal-link field (lexicographic 4D index),
// in t order as polyakov.cu:430-437: P(x) = prod_t T(x, t).  Loads in groups of
// eight (one after the other, with a wavefront per CU, they were the whole
// time: 14 us at 24^3 x 48), one wavefront per workgroup to spread the few of
// them over the CUs.
__global__ __launch_bounds__(64) void k_tprod(const double* __restrict__ tl, RepDesc r, double* __restrict__ P) {
  const int32_t j = (int32_t)(blockIdx.x * blockDim.x + threadIdx.x);
  if (j >= r.SV) return;
  C64 res = {1.0, 0.0};
  int t = 0;
  for (; t + 8 <= r.N[3]; t += 8) {
    C64 q[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int64_t m = j + (int64_t)(t + k) * r.SV;
      q[k] = {tl[2 * m], tl[2 * m + 1]};
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) res = cmul(res, q[k]);
  }
  for (; t < r.N[3]; ++t) {
    const int64_t m = j + (int64_t)t * r.SV;
    res = cmul(res, C64{tl[2 * m], tl[2 * m + 1]});
  }
  P[2 * (int64_t)j] = res.re;
  P[2 * (int64_t)j + 1] = res.im;
}

// Polyakov loops of the analytic multihit links, without the field between:
// P(x) = prod_t T(x, t), a workgroup for kPolySites spatial sites with one thread
// per link; the first row multiplies what the rows left in LDS, in t order as
// k_tprod.  A loop over t, for more slices than a workgroup has rows, made the
// compiler keep the constants of the special functions in registers (158, or
// spills): 14 us and more.  Calls with the correlator, two kernels before: 35.3 ->
// 31.2 us at 32^3 x 16 and 42.4 -> 34.1 us at 32^3 x 24, binary64, 32.3 -> 27.8 us
// at 24^3 x 32 and 90.9 -> 68.6 us at 48^3 x 32, binary32.
constexpr int kPolySites = 32;
template <typename Real>
__global__ __launch_bounds__(kPolySites * kPolyRows) void k_poly_links(const Real* __restrict__ lat, RepDesc r,
                                                                       double* __restrict__ P) {
  __shared__ C64 link[kPolyRows][kPolySites];
  const int32_t lane = (int32_t)threadIdx.x % kPolySites, t = (int32_t)threadIdx.x / kPolySites, half = r.SV / 2;
  const int32_t i = (int32_t)blockIdx.x * kPolySites + lane, idx = min(i, r.SV - 1);
  const int32_t parity = idx >= half ? 1 : 0, id = idx - parity * half;  // at t = 0
  Site s;
  site_of(r, id + t * half, (parity + t) & 1, s);
  link[t][lane] = temporal_value<Real, 1>(lat, r, s, id + t * half, (parity + t) & 1, 0, 0, 0.0, 0, 0, 0);
  __syncthreads();
  if (t == 0 && i < r.SV) {
    C64 res = {1.0, 0.0};
#pragma unroll 2
    for (int32_t k = 0; k < r.N[3]; ++k) res = cmul(res, link[k][lane]);
    const int32_t j = s.x[0] + r.N[0] * (s.x[1] + r.N[1] * s.x[2]);
    P[2 * (int64_t)j] = res.re;
    P[2 * (int64_t)j + 1] = res.im;
  }
}

// polyakov.cu:514-535: sum over x and the three spatial axes of
// P(x) conj(P(x + R e_dir)), R = 1..rmax; one partial row of 2*rmax per 256
// sites.  One R per workgroup (blockIdx.y): 15.6 us at 24^3 when a workgroup
// took all R in turn, two barriers each.
__global__ __launch_bounds__(256) void k_pp(const double* __restrict__ P, RepDesc r, int rmax,
                                            double* __restrict__ partials) {
  const int32_t id = (int32_t)(blockIdx.x * blockDim.x + threadIdx.x);
  const int32_t R = (int32_t)blockIdx.y + 1;
  double v[2] = {0.0, 0.0};
  if (id < r.SV) {
    const int32_t row = (int32_t)((uint32_t)id / (uint32_t)r.N[0]), x2 = (int32_t)((uint32_t)row / (uint32_t)r.N[1]);
    const int32_t x[3] = {id - row * r.N[0], row - x2 * r.N[1], x2};
    const int32_t stride[3] = {1, r.N[0], r.N[0] * r.N[1]};
    const C64 p0 = {P[2 * (int64_t)id], P[2 * (int64_t)id + 1]};
#pragma unroll
    for (int dir = 0; dir < 3; ++dir) {
      const int32_t y = (int32_t)((uint32_t)(x[dir] + R) % (uint32_t)r.N[dir]);
      const int64_t j = id + (int64_t)(y - x[dir]) * stride[dir];
      const C64 q = {P[2 * j], -P[2 * j + 1]};
      const C64 t = cmul(p0, q);
      v[0] += t.re;
      v[1] += t.im;
    }
  }
  const double o = block_sum<2>(v);
  if (threadIdx.x < 2) partials[((int64_t)blockIdx.x * rmax + (R - 1)) * 2 + threadIdx.x] = o;
}

// convertOrder.cu:32-63: even/odd <-> lexicographic, all four planes.  A thread
// takes the two sites 2e, 2e + 1 of a row, element e of both parities' arrays: all
// accesses in full lines.  24^4, binary64 (21 MB): 6.3 us before, with a thread
// per element, every other one of a line, and divisions.
template <typename Real>
__global__ __launch_bounds__(256) void k_convert_layout(const Real* __restrict__ in, Real* __restrict__ out,
                                                        RepDesc r, int eo_to_no) {
  typedef Real Two __attribute__((ext_vector_type(2), aligned(sizeof(Real))));
  const uint32_t e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (uint32_t)r.HV) return;
  Site s;
  site_of(r, (int32_t)e, 0, s);
  // the parity of the site with even x
  const uint32_t even = (uint32_t)(((s.x[1] + s.x[2] + s.x[3]) & 1) * r.HV) + e, odd = (uint32_t)r.HV + 2 * e - even;
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const size_t o = (size_t)d * r.V;
    if (eo_to_no) {
      const Two v = {in[o + even], in[o + odd]};
      *reinterpret_cast<Two*>(out + o + 2 * (size_t)e) = v;
    } else {
      const Two v = *reinterpret_cast<const Two*>(in + o + 2 * (size_t)e);
      out[o + even] = v.x;
      out[o + odd] = v.y;
    }
  }
}

template <typename A, typename B>
__global__ __launch_bounds__(256) void k_convert_precision(const A* __restrict__ in, B* __restrict__ out, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = (B)in[i];
}

__global__ __launch_bounds__(256) void k_fill_zero(uint32_t* __restrict__ p, int64_t nwords) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nwords) p[i] = 0u;
}

__global__ void k_increment(uint32_t* c) {
  if (threadIdx.x == 0 && blockIdx.x == 0) c[0] = c[0] + 1u;
}

// Sum over a workgroup of NT threads of NV values each; thread k < NV returns the
// k-th.  Through LDS: NT / 16 threads' values added by a thread, then their 16 sums
// by another.  block_sum shuffles every value through the wavefront, 24
// instructions each (plaquette fields at 24^4, twelve values: 15.7 -> 13.8 us).
template <int NV, int NT>
__device__ __forceinline__ double block_sum_wide(const double (&v)[NV]) {
  static_assert(16 * NV <= NT && NT % 16 == 0, "a thread per value and sixteenth");
  __shared__ double red[NV][NT + 1], part[NV][16];
#pragma unroll
  for (int k = 0; k < NV; ++k) red[k][threadIdx.x] = v[k];
  __syncthreads();
  const int k = (int)threadIdx.x / 16, q = (int)threadIdx.x % 16;
  if (k < NV) {
    double s = 0.0;
#pragma unroll
    for (int j = 0; j < NT / 16; ++j) s += red[k][16 * j + q];
    part[k][q] = s;
  }
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x < NV)
#pragma unroll
    for (int j = 0; j < 16; ++j) s += part[threadIdx.x][j];
  return s;
}

// plaquette_comps.cu:34-107: six plaquette components per site (spacetime) or
// per spatial site averaged over t, in SixPlaquette order
// (lattice_functions.h:38-45): (0,3) (1,3) (2,3) (1,2) (2,0) (0,1); field written
// at the lexicographic index, component-major; partial sums of the six means per
// workgroup.  EO: even/odd input, else lexicographic.
//
// A thread takes lexicographic sites, so the field is stored in full lines, and
// an even/odd input is read as two contiguous half rows.  A site's sixteen links
// are loaded at once; only the loop over t keeps a second set of sums.  At most
// kFoldRows workgroups, one set of sums each, so that the sums take one fold.
// 24^4, binary64 (42 MB, 8 us at the copy rate): 13.8 us, 17.8 us with a shuffled
// block sum, 24.8 us with even/odd
// threads, loads site by site and divisions for the coordinates.  All its
// wavefronts are resident at once and load, compute (800 vector instructions,
// 7 us) and store in step.
template <typename Real, bool EO, bool SPACETIME>
__global__ __launch_bounds__(256) void k_plaquette_fields(const Real* __restrict__ lat, RepDesc r,
                                                         double* __restrict__ field,
                                                         double* __restrict__ partials) {
  const uint32_t size = (uint32_t)(SPACETIME ? r.V : r.SV);
  double v[12];
#pragma unroll
  for (int k = 0; k < 12; ++k) v[k] = 0.0;
  for (uint32_t idx = blockIdx.x * blockDim.x + threadIdx.x; idx < size; idx += gridDim.x * blockDim.x) {
    double w[12];
#pragma unroll
    for (int k = 0; k < 12; ++k) w[k] = 0.0;
    const int nt = SPACETIME ? 1 : r.N[3];
    for (int t = 0; t < nt; ++t) {
      const uint32_t n = idx + (uint32_t)(t * r.SV);  // lexicographic site
      Site s;  // its row (of parity 0)
      site_of(r, (int32_t)(n >> 1), 0, s);
      const int32_t odd = (int32_t)(n & 1u), parity = (s.x[1] + s.x[2] + s.x[3] + odd) & 1;
      const bool last = odd && (s.x[0] >> 1) == r.nxh - 1;
      uint32_t here = n, nb[4];
      if (EO) {
        here = (uint32_t)(parity * r.HV) + (n >> 1);
        const uint32_t opp = (uint32_t)((1 - parity) * r.HV) + (n >> 1);
        nb[0] = opp + (uint32_t)(last ? 1 - r.nxh : odd);
#pragma unroll
        for (int mu = 1; mu < 4; ++mu) nb[mu] = opp + (uint32_t)s.fwd[mu];
      } else {
        nb[0] = n + (uint32_t)(last ? 1 - r.N[0] : 1);
#pragma unroll
        for (int mu = 1; mu < 4; ++mu) nb[mu] = n + 2u * (uint32_t)s.fwd[mu];
      }
      Real own[4], tf[4][4];  // tf[nu][mu] = theta_nu(x + mu)
#pragma unroll
      for (int mu = 0; mu < 4; ++mu) {
        own[mu] = ld(lat + (size_t)mu * r.V, here);
#pragma unroll
        for (int nu = 0; nu < 4; ++nu)
          if (nu != mu) tf[nu][mu] = ld(lat + (size_t)nu * r.V, nb[mu]);
      }
      constexpr int m[6] = {0, 1, 2, 1, 2, 0}, q[6] = {3, 3, 3, 2, 0, 1};
#pragma unroll
      for (int d = 0; d < 6; ++d) {
        const Real p = ((own[m[d]] + tf[q[d]][m[d]]) - tf[m[d]][q[d]]) - own[q[d]];
        const C64 e = exp_i<Real>(p);
        w[2 * d] += 1.0 - e.re;
        w[2 * d + 1] += -e.im;
      }
    }
    if (!SPACETIME)
#pragma unroll
      for (int k = 0; k < 12; ++k) w[k] /= (double)r.N[3];
#pragma unroll
    for (int d = 0; d < 6; ++d) {
      *reinterpret_cast<F64x2*>(field + 2 * ((size_t)idx + (size_t)d * size)) = F64x2{w[2 * d], w[2 * d + 1]};
      v[2 * d] += w[2 * d];
      v[2 * d + 1] += w[2 * d + 1];
    }
  }
  const double o = block_sum_wide<12, 256>(v);
  if (threadIdx.x < 12) partials[12 * (size_t)blockIdx.x + threadIdx.x] = o;
}

// Per-replica fold of batched plaquette partials, in workgroup order.
__global__ __launch_bounds__(256) void k_batched_finish(const double* __restrict__ partials,
                                                        const RepDesc* __restrict__ reps, double* __restrict__ out) {
  const RepDesc& r = reps[blockIdx.x];
  double v[4] = {0.0, 0.0, 0.0, 0.0};
  for (int i = threadIdx.x; i < r.nblk; i += blockDim.x)
    for (int k = 0; k < 4; ++k) v[k] += partials[4 * (int64_t)(r.blk_begin + i) + k];
  const double o = block_sum<4>(v);
  if (threadIdx.x < 4) out[4 * blockIdx.x + threadIdx.x] = o * (1.0 / (3.0 * (double)r.V));
}

// Per-replica fold of the plaquette rows written by the measuring update
// launches of a batched sweep (spans[sgi * nrep + replica]: its rows of each
// launch, in launch order), stored at the series row of the current sweep.
__global__ __launch_bounds__(256) void k_ensemble_plaquette_fold(const double* __restrict__ rows, int nseg,
                                                                 const RowSpan* __restrict__ spans,
                                                                 const RepDesc* __restrict__ reps, int nrep,
                                                                 const uint32_t* sweep_dev, const uint32_t* base_dev,
                                                                 int cap, double* __restrict__ series) {
  const RepDesc& r = reps[blockIdx.x];
  double v[4] = {0.0, 0.0, 0.0, 0.0};
  for (int sgi = 0; sgi < nseg; ++sgi) {
    const RowSpan span = spans[sgi * nrep + (int)blockIdx.x];
    for (int i = threadIdx.x; i < span.count; i += blockDim.x) {
      const double* row = rows + 4 * ((int64_t)span.begin + i);
      for (int k = 0; k < 4; ++k) v[k] += row[k];
    }
  }
  const double o = block_sum<4>(v);
  if (threadIdx.x < 4) {
    const uint32_t idx = *sweep_dev - *base_dev;
    if (idx < (uint32_t)cap)
      series[4 * ((int64_t)idx * nrep + blockIdx.x) + threadIdx.x] = o * (1.0 / (3.0 * (double)r.V));
  }
}

inline int nblocks(int64_t n, int block) { return (int)((n + block - 1) / block); }

}  // namespace

namespace {
template <typename Real, bool BATCHED>
hipError_t plaquette_spt(int spt, const Real* lat, const RepDesc& r, const RepDesc* reps, const uint16_t* map,
                         double* partials, int nblk, int block, hipStream_t st) {
  if (spt == 4 && sizeof(Real) == sizeof(float))
    k_plaquette<Real, BATCHED, 4><<<nblk, block, 0, st>>>(lat, r, reps, map, partials);
  else if (spt == 2)
    k_plaquette<Real, BATCHED, 2><<<nblk, block, 0, st>>>(lat, r, reps, map, partials);
  else if (spt == 1)
    k_plaquette<Real, BATCHED, 1><<<nblk, block, 0, st>>>(lat, r, reps, map, partials);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}
}  // namespace

hipError_t launch_plaquette(int prec, const void* lat, const RepDesc& r, double* partials, int nblk, int block,
                            int spt, hipStream_t st) {
  if (prec == PREC_F64)
    return plaquette_spt<double, false>(spt, (const double*)lat, r, nullptr, nullptr, partials, nblk, block, st);
  return plaquette_spt<float, false>(spt, (const float*)lat, r, nullptr, nullptr, partials, nblk, block, st);
}

hipError_t launch_plaquette_batched(int prec, const void* lat_base, const RepDesc* reps, const uint16_t* blockmap,
                                    double* partials, int nblk, int block, int spt, hipStream_t st) {
  RepDesc dummy{};
  if (prec == PREC_F64)
    return plaquette_spt<double, true>(spt, (const double*)lat_base, dummy, reps, blockmap, partials, nblk, block,
                                       st);
  return plaquette_spt<float, true>(spt, (const float*)lat_base, dummy, reps, blockmap, partials, nblk, block, st);
}

hipError_t launch_ensemble_plaquette_fold(const double* rows, int nseg, const RowSpan* spans, const RepDesc* reps,
                                          int nrep, const uint32_t* sweep_dev, const uint32_t* base_dev, int cap,
                                          double* series, hipStream_t st) {
  k_ensemble_plaquette_fold<<<nrep, 256, 0, st>>>(rows, nseg, spans, reps, nrep, sweep_dev, base_dev, cap, series);
  return hipGetLastError();
}

hipError_t launch_batched_finish(const double* partials, const RepDesc* reps, int nrep, double* out, hipStream_t st) {
  k_batched_finish<<<nrep, 256, 0, st>>>(partials, reps, out);
  return hipGetLastError();
}

hipError_t launch_polyakov(int prec, const void* lat, const RepDesc& r, double* partials, int nblk, int block,
                           hipStream_t st) {
  if (prec == PREC_F64)
    k_polyakov<double><<<nblk, block, 0, st>>>((const double*)lat, r, partials);
  else
    k_polyakov<float><<<nblk, block, 0, st>>>((const float*)lat, r, partials);
  return hipGetLastError();
}

hipError_t launch_finish_sums(const double* partials, int nblk, int nv, double scale, double* out, double* scratch,
                              hipStream_t st) {
  if (nblk <= kFoldRows) {
    k_finish<<<nv, std::min(1024, (nblk + 63) / 64 * 64), 0, st>>>(partials, nblk, nv, scale, out);
    return hipGetLastError();
  }
  const int G = fold_groups(nblk);
  k_fold_rows<<<dim3(G, nv), 256, 0, st>>>(partials, nblk, nv, kFoldRows, scratch);
  k_finish<<<nv, 256, 0, st>>>(scratch, G, nv, scale, out);
  return hipGetLastError();
}

hipError_t launch_poly_volume(int prec, const void* lat, const RepDesc& r, double* P, hipStream_t st) {
  const int block = 64, nb = nblocks(r.SV, block);
  if (prec == PREC_F64)
    k_poly_volume<double><<<nb, block, 0, st>>>((const double*)lat, r, P);
  else
    k_poly_volume<float><<<nb, block, 0, st>>>((const float*)lat, r, P);
  return hipGetLastError();
}

hipError_t launch_tprod(const double* tl, const RepDesc& r, double* P, hipStream_t st) {
  k_tprod<<<nblocks(r.SV, 64), 64, 0, st>>>(tl, r, P);
  return hipGetLastError();
}

hipError_t launch_poly_links(int prec, const void* lat, const RepDesc& r, double* P, hipStream_t st) {
  const int nb = nblocks(r.SV, kPolySites), block = kPolySites * r.N[3];
  if (r.N[3] > kPolyRows) return hipErrorInvalidValue;
  if (prec == PREC_F64)
    k_poly_links<double><<<nb, block, 0, st>>>((const double*)lat, r, P);
  else
    k_poly_links<float><<<nb, block, 0, st>>>((const float*)lat, r, P);
  return hipGetLastError();
}

hipError_t launch_temporal_links(int prec, const void* lat, const RepDesc& r, int mode, int proposal, int nhit,
                                 double step, uint32_t stream, uint32_t c1, uint32_t c3, double* out, hipStream_t st) {
  const int block = 256, nb = nblocks(r.V, block);
  auto go = [&](auto* l) {
    typedef std::remove_cv_t<std::remove_pointer_t<decltype(l)>> Real;
    auto* k = mode == 0 ? k_temporal_links<Real, 0> : mode == 1 ? k_temporal_links<Real, 1> : k_temporal_links<Real, 2>;
    k<<<nb, block, 0, st>>>(l, r, proposal, nhit, step, stream, c1, c3, out);
  };
  if (prec == PREC_F64) go((const double*)lat);
  else go((const float*)lat);
  return hipGetLastError();
}

hipError_t launch_temporal_pairs(int prec, const void* lat, const RepDesc& r, int mode, int proposal, int nhit,
                                 double step, uint32_t stream, uint32_t c3, double* p2, uint32_t* ctr, uint32_t n2,
                                 uint32_t slots, hipStream_t st) {
  const int block = 256, nb = nblocks((int64_t)r.SV * (r.N[3] / 2), block);
  auto go = [&](auto* l) {
    typedef std::remove_cv_t<std::remove_pointer_t<decltype(l)>> Real;
    auto* k = mode == 0 ? k_temporal_pairs<Real, 0> : mode == 1 ? k_temporal_pairs<Real, 1> : k_temporal_pairs<Real, 2>;
    k<<<nb, block, 0, st>>>(l, r, proposal, nhit, step, stream, c3, p2, ctr, n2, slots);
  };
  if (prec == PREC_F64) go((const double*)lat);
  else go((const float*)lat);
  return hipGetLastError();
}

hipError_t launch_pp(const double* P, const RepDesc& r, int rmax, double* partials, int nblk, int block,
                     hipStream_t st) {
  k_pp<<<dim3(nblk, rmax), block, 0, st>>>(P, r, rmax, partials);
  return hipGetLastError();
}

hipError_t launch_convert_layout(int prec, const void* in, void* out, const RepDesc& r, int eo_to_no, int block,
                                 hipStream_t st) {
  const int nb = nblocks(r.HV, block);
  if (prec == PREC_F64)
    k_convert_layout<double><<<nb, block, 0, st>>>((const double*)in, (double*)out, r, eo_to_no);
  else
    k_convert_layout<float><<<nb, block, 0, st>>>((const float*)in, (float*)out, r, eo_to_no);
  return hipGetLastError();
}

hipError_t launch_convert_precision(const void* in, int in_prec, void* out, int out_prec, int64_t n, int block,
                                    hipStream_t st) {
  const int nb = nblocks(n, block);
  if (in_prec == PREC_F64 && out_prec == PREC_F32)
    k_convert_precision<double, float><<<nb, block, 0, st>>>((const double*)in, (float*)out, n);
  else if (in_prec == PREC_F32 && out_prec == PREC_F64)
    k_convert_precision<float, double><<<nb, block, 0, st>>>((const float*)in, (double*)out, n);
  else if (in_prec == PREC_F64)
    k_convert_precision<double, double><<<nb, block, 0, st>>>((const double*)in, (double*)out, n);
  else
    k_convert_precision<float, float><<<nb, block, 0, st>>>((const float*)in, (float*)out, n);
  return hipGetLastError();
}

hipError_t launch_plaquette_fields(int prec, const void* lat, const RepDesc& r, int spacetime, int eo_order,
                                   double* field, double* partials, int nblk, int block, hipStream_t st) {
  const auto run = [&](auto* l) {
    using Real = std::remove_const_t<std::remove_pointer_t<decltype(l)>>;
    if (eo_order && spacetime)
      k_plaquette_fields<Real, true, true><<<nblk, block, 0, st>>>(l, r, field, partials);
    else if (eo_order)
      k_plaquette_fields<Real, true, false><<<nblk, block, 0, st>>>(l, r, field, partials);
    else if (spacetime)
      k_plaquette_fields<Real, false, true><<<nblk, block, 0, st>>>(l, r, field, partials);
    else
      k_plaquette_fields<Real, false, false><<<nblk, block, 0, st>>>(l, r, field, partials);
  };
  if (prec == PREC_F64)
    run((const double*)lat);
  else
    run((const float*)lat);
  return hipGetLastError();
}

hipError_t launch_fill_zero(void* p, int64_t bytes, hipStream_t st) {
  const int64_t nw = bytes / 4;
  if (nw > 0) k_fill_zero<<<nblocks(nw, 256), 256, 0, st>>>((uint32_t*)p, nw);
  return hipGetLastError();
}

hipError_t launch_increment(uint32_t* counter, hipStream_t st) {
  k_increment<<<1, 64, 0, st>>>(counter);
  return hipGetLastError();
}

}  // namespace u1d
