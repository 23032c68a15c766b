// u1_link.h -- one link update of the update kernels: the staple from its
// angles, the Metropolis hits, the overrelaxation reflection, and the plaquette
// sums of a measuring update.  Shared by the phase, pair and pass kernels
// (u1_update.hip) and the diagonal walks (u1_walk.hip), so that every launch
// form does the same arithmetic on the same angles.
#pragma once
#include "u1_kernels.h"

namespace u1d {

namespace {

template <typename Real>
struct Staple {
  Real re, im;
};

// Plaquette pieces of a link (x, MU) for the directions nu < MU: the sums of
// e^{i up_nu} (u) and e^{i lo_nu} (l).  With the link's new angle theta,
// theta + up_nu = -P_{nu,MU}(x) and theta + lo_nu = P_{nu,MU}(x - nu), so
// every plaquette of the planes (nu, MU), nu < MU, is one piece of exactly one
// odd-site MU link.
template <typename Real>
struct PlaqPieces {
  Real ur, ui, lr, li;
};

// First direction nu != mu of the space-time (st) or space-space class.
__host__ __device__ constexpr int first_nu(int mu, bool st) {
  for (int nu = 0; nu < 4; ++nu)
    if (nu != mu && ((mu == 3 || nu == 3) == st)) return nu;
  return -1;
}

// The 18 angles of the staple of link (x, MU) (staple.h:85-92): for the j-th
// direction nu != MU (j = nu for nu < MU, else nu - 1),
//   a = theta_nu(x+mu), b = theta_mu(x+nu), c = theta_nu(x),
//   d = theta_nu(x+mu-nu), e = theta_mu(x-nu), f = theta_nu(x-nu).
// fwd/bwd[d] are the eo-id offsets to x +- e_d.
template <typename Real>
struct StapleIn {
  Real a[3], b[3], c[3], d[3], e[3], f[3];
};

// Loads the staple angles.  The c and d angles of the directions nu in the
// bit mask DEFM (theta_nu at the link's own parity) are left out: for a fused
// pair (DEFM = 1) to phase_load_nu0_lds, for a fused pass to phase_load_dep.
template <typename Real, int MU, int DEFM = 0>
__device__ __forceinline__ void staple_load(const Real* __restrict__ lat, const RepDesc& r, uint32_t same,
                                            uint32_t opp, const int32_t (&fwd)[4], const int32_t (&bwd)[4],
                                            StapleIn<Real>& in) {
  const Real* pm = lat + (size_t)MU * r.V;
#pragma unroll
  for (int nu = 0; nu < 4; ++nu) {
    if (nu == MU) continue;
    const int j = nu < MU ? nu : nu - 1;
    const Real* pn = lat + (size_t)nu * r.V;
    in.a[j] = ld(pn, opp + fwd[MU]);
    in.b[j] = ld(pm, opp + fwd[nu]);
    if (!((DEFM >> nu) & 1)) {
      in.c[j] = ld(pn, same);
      in.d[j] = ld(pn, same + fwd[MU] + bwd[nu]);
    }
    in.e[j] = ld(pm, opp + bwd[nu]);
    in.f[j] = ld(pn, opp + bwd[nu]);
  }
}
// e^{i up} and e^{i lo} of one direction: cosines and sines.
template <typename Real>
struct StapleTerm {
  Real cu, su, cl, sl;
};
template <typename Real>
__device__ __forceinline__ StapleTerm<Real> staple_term(const StapleIn<Real>& in, int j) {
  const Real up = (in.a[j] - in.b[j]) - in.c[j];
  const Real lo = ((-in.d[j]) - in.e[j]) + in.f[j];
  StapleTerm<Real> t;
  UMath<Real>::sincos(up, &t.su, &t.cu);
  UMath<Real>::sincos(lo, &t.sl, &t.cl);
  return t;
}

// Staple of link (x, MU) (staple.h:79-102) from its terms (the j-th direction
// nu != MU), with the operation order of the oracle.  With MEAS the plaquette
// pieces are collected on the side (the staple is unchanged).
template <typename Real, int MU, bool MEAS = false>
__device__ __forceinline__ Staple<Real> staple_of(const StapleTerm<Real> (&term)[3], Real xi, Real inv_xi, bool aniso,
                                                  PlaqPieces<Real>* pp = nullptr) {
  Real ssr = 0, ssi = 0, str = 0, sti = 0;
#pragma unroll
  for (int nu = 0; nu < 4; ++nu) {
    if (nu == MU) continue;
    const StapleTerm<Real>& t = term[nu < MU ? nu : nu - 1];
    const Real ar = t.cu + t.cl, ai = t.su + t.sl;
    if (MEAS && nu < MU) {
      pp->ur += t.cu;
      pp->ui += t.su;
      pp->lr += t.cl;
      pp->li += t.sl;
    }
    // binary32: the first term of each class initialises its sum (the oracle's
    // 0 + x is kept in binary64, where the kernels match it bit for bit)
    const bool st_class = MU == 3 || nu == 3;
    const bool first = sizeof(Real) == sizeof(float) && nu == first_nu(MU, st_class);
    if (st_class) {
      str = first ? ar : str + ar;
      sti = first ? ai : sti + ai;
    } else {
      ssr = first ? ar : ssr + ar;
      ssi = first ? ai : ssi + ai;
    }
  }
  if constexpr (sizeof(Real) == sizeof(float)) {
    // binary32: the weighted form with no test of xi; at xi == 1 both weights
    // are exactly 1 and the fused sum equals the plain sum ss + st
    if (MU == 3) return {str * xi, sti * xi};  // no space-space staples
    return {__builtin_fmaf(ssr, inv_xi, str * xi), __builtin_fmaf(ssi, inv_xi, sti * xi)};
  } else {
    if (!aniso) return {ssr + str, ssi + sti};  // xi == 1: identical to ss/1 + st*1
    return {ssr / xi + str * xi, ssi / xi + sti * xi};
  }
}
template <typename Real, int MU, bool MEAS = false>
__device__ __forceinline__ Staple<Real> staple_sum(const StapleIn<Real>& in, Real xi, Real inv_xi, bool aniso,
                                                   PlaqPieces<Real>* pp = nullptr) {
  const StapleTerm<Real> t[3] = {staple_term(in, 0), staple_term(in, 1), staple_term(in, 2)};
  return staple_of<Real, MU, MEAS>(t, xi, inv_xi, aniso, pp);
}

template <typename Real>
struct MetroState {
  Real th, re_old;
};

// One Metropolis hit with a fixed staple (lattice_functions.h:68-80 in the
// Re(S e^{i theta}) form), binary64: the oracle's operations in its order.
// wu: proposal word, wb: accept-test word.  For theta + delta one wrap step
// each way suffices because |delta| <= step <= pi.
__device__ __forceinline__ bool metro_hit_f64(MetroState<double>& m, Staple<double> S, double beta, bool exp_small,
                                              int proposal, double step, uint32_t wu, uint32_t wb) {
  // a * (2u - 1) with u = wu 2^-32 as one FMA: 2u - 1 is exact in binary64,
  // so fma(wu, a 2^-31, -a) is the same correctly rounded product as the
  // oracle's two-step form (a 2^-31 is exact).
  double tn;
  if (proposal == 0)
    tn = __builtin_fma((double)wu, u1m::K_PI * 0x1p-31, -u1m::K_PI);
  else
    tn = u1m::wrap_step_d(m.th + __builtin_fma((double)wu, step * 0x1p-31, -step));
  double sn, cn;
  UMath<double>::sincos_in_loop(tn, &sn, &cn);
  const double re_new = S.re * cn - S.im * sn;
  const bool ok = UMath<double>::accept(beta * (re_new - m.re_old), wb, exp_small);
  if (ok) {
    m.th = tn;
    m.re_old = re_new;
  }
  return ok;
}

// The same hit in binary32, from the same two words.  The proposal is
// a (2 wu 2^-32 - 1) as one FMA, with a = pi (independent: pscale = pi 2^-31,
// poff = pi) or a = step (theta + delta).  theta + delta is not wrapped here:
// the caller wraps theta (x - 2 pi rint(x / 2 pi), any range) after every
// second pair of hits and after the last (|theta| <= pi + 4 step <= 5 pi in
// between, well inside the hardware sin/cos range).  The accept test
// exp(beta dRe) > wb 2^-32 is evaluated as 2^(beta log2(e) dRe + 32) > wb
// (bl2e = beta log2(e)): one v_exp_f32 and the word converted without scaling.
// thm is 1 for theta + delta and 0 for the independent proposal, so both
// forms are one more FMA (theta * thm + offset, rounded once).
__device__ __forceinline__ bool metro_hit_f32(MetroState<float>& m, Staple<float> S, float bl2e, float thm,
                                              float pscale, float poff, uint32_t wu, uint32_t wb) {
  const float tn = __builtin_fmaf(m.th, thm, __builtin_fmaf((float)wu, pscale, -poff));
  float sn, cn;
  UMath<float>::sincos(tn, &sn, &cn);
  const float re_new = __builtin_fmaf(S.re, cn, -(S.im * sn));
  const float x = __builtin_fmaf(bl2e, re_new - m.re_old, 32.0f);
  const bool ok = __builtin_amdgcn_exp2f(x) > (float)wb;
  if (ok) {
    m.th = tn;
    m.re_old = re_new;
  }
  return ok;
}

// New angles of SPT links from their staples: nhit Metropolis hits each (l:
// Philox counter word 0, the link index; the accepted hits of the lanes in
// vmask are added to acc_wave, a wave-uniform count from the accept masks kept
// on the scalar unit), or the overrelaxation reflection.
template <typename Real, int KIND, int SPT>
__device__ __forceinline__ void update_angles(const PhaseArgs& a, const RepDesc& r, const Staple<Real> (&S)[SPT],
                                              Real (&th)[SPT], const uint32_t (&l)[SPT], const uint64_t (&vmask)[SPT],
                                              uint32_t& acc_wave) {
  if (KIND == KIND_METROPOLIS) {
    MetroState<Real> m[SPT];
#pragma unroll
    for (int k = 0; k < SPT; ++k) {
      m[k].th = th[k];
      Real s0, c0;
      UMath<Real>::sincos(th[k], &s0, &c0);
      if constexpr (sizeof(Real) == sizeof(float))
        m[k].re_old = __builtin_fmaf(S[k].re, c0, -(S[k].im * s0));
      else
        m[k].re_old = S[k].re * c0 - S[k].im * s0;
    }
    const uint32_t sweep = a.sweep_dev ? *a.sweep_dev * a.sweep_mul + a.sweep : a.sweep;
    const Real beta = (Real)r.beta;
    const bool exp_small = r.exp_small != 0;
    // binary32 hit constants (metro_hit_f32), rounded on the host
    const float bl2e = r.bl2e_f;
    const float pscale = a.pscale_f, thm = a.thm_f;
    // kept in a vector register: the proposal FMA reads pscale and poff, and
    // one scalar register only (else a vector move per hit)
    float poff = a.poff_f;
    if constexpr (sizeof(Real) == sizeof(float)) asm("" : "+v"(poff));
    // hits in blocks of up to four (two Philox draws of four words each)
    for (int h4 = 0; h4 < a.nhit; h4 += 4) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int h = h4 + 2 * j;
        if (h >= a.nhit) break;
        const uint32_t c2 = u1r::ctr2(a.stream, a.pass, (uint32_t)(h >> 1));
#pragma unroll
        for (int k = 0; k < SPT; ++k) {
          const u1r::U32x4 w = u1r::draw(r.seed, l[k], sweep, c2, r.c3);
          if constexpr (sizeof(Real) == sizeof(float)) {
            const bool ok0 = metro_hit_f32(m[k], S[k], bl2e, thm, pscale, poff, w.v[0], w.v[1]);
            acc_wave += count_wave(ok0, vmask[k]);
            if (h + 1 < a.nhit) {
              const bool ok1 = metro_hit_f32(m[k], S[k], bl2e, thm, pscale, poff, w.v[2], w.v[3]);
              acc_wave += count_wave(ok1, vmask[k]);
            }
          } else {
            const bool ok0 = metro_hit_f64(m[k], S[k], beta, exp_small, a.proposal, a.step, w.v[0], w.v[1]);
            acc_wave += count_wave(ok0, vmask[k]);
            if (h + 1 < a.nhit) {
              const bool ok1 = metro_hit_f64(m[k], S[k], beta, exp_small, a.proposal, a.step, w.v[2], w.v[3]);
              acc_wave += count_wave(ok1, vmask[k]);
            }
          }
        }
      }
      // binary32: back into [-pi, pi] after each block, i.e. after every
      // second pair of hits and after the last (|theta| <= pi + 4 step in
      // between)
      if constexpr (sizeof(Real) == sizeof(float)) {
#pragma unroll
        for (int k = 0; k < SPT; ++k) m[k].th = (float)u1m::wrap_near_d((double)m[k].th);
      }
    }
#pragma unroll
    for (int k = 0; k < SPT; ++k) th[k] = m[k].th;
  } else {
#pragma unroll
    for (int k = 0; k < SPT; ++k) {
      // lattice_functions.h:83-89: theta' = -theta - 2 arg(S), wrapped
      const Real t2 = UMath<Real>::atan2(S[k].im, S[k].re);
      if constexpr (sizeof(Real) == sizeof(float))  // -theta - 2 t2 and the wrap in binary64
        th[k] = (float)u1m::wrap_near_d(__builtin_fma(-2.0, (double)t2, -(double)th[k]));
      else
        th[k] = UMath<double>::wrap(-th[k] - 2.0 * t2);
    }
  }
}

// Plaquette sums of one updated link (x, MU) from its pieces and new angle:
// sum over nu < MU of (1 - cos P), and of -sin P, added to re and im.
template <typename Real, int MU>
__device__ __forceinline__ void add_plaquettes(const PlaqPieces<Real>& pp, Real th, bool valid, double& re_sum,
                                               double& im_sum) {
  Real sn, cn;
  UMath<Real>::sincos(th, &sn, &cn);
  // sum cos(theta + up) + cos(theta + lo); sum sin(theta + up) - sin(theta + lo)
  const Real re = cn * (pp.ur + pp.lr) - sn * (pp.ui + pp.li);
  const Real im = sn * (pp.ur - pp.lr) + cn * (pp.ui - pp.li);
  if (valid) {
    re_sum += (double)(2 * MU) - (double)re;
    im_sum += (double)im;
  }
}

}  // namespace

}  // namespace u1d
