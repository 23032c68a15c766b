// u1_multilevel.hip -- tensor accumulation of the two-level multilevel
// Polyakov-loop correlator (reference multilevel.cu:331-553).
//
// Layout of one T2 / T4 layer (multilevel.cu:350): element (x, R, dir) at
//     x + SV*(R-1) + SV*Rmax*dir,  layer stride sz = SV*Rmax*3,
// complex FP64, interleaved (re, im).  All accumulation is FP64.
// The masked sublattice updates reuse the update kernels (ml = 4 or 2); the
// two-slice products of the temporal links come from k_temporal_pairs
// (u1_measure.hip), one slot of SV*Nt/2 complex values per level-2 step.
#include "u1_kernels.h"

namespace u1d {

namespace {

struct C64 {
  double re, im;
};
__device__ __forceinline__ C64 cmul(C64 a, C64 b) { return {a.re * b.re - a.im * b.im, a.im * b.re + a.re * b.im}; }
__device__ __forceinline__ C64 ldc(const double* p, int64_t i) {
  const double2 v = *(const double2*)(p + 2 * i);
  return {v.x, v.y};
}
__device__ __forceinline__ void stc64(double* p, int64_t i, C64 v) { *(double2*)(p + 2 * i) = {v.re, v.im}; }

// Level 2 over nslots level-2 steps and level 4 (multilevel.cu:331-360,
// 439-456):
//   l2[x, R, dir, layer] = sum over steps of p(x, layer) conj p(x + R e_dir, layer),
//   l4[., j] += (l2[., 2j] l2norm) (l2[., 2j+1] l2norm),
// each sum in step order.  One thread per (x, dir, j) and kMlR values of R: the
// two layers of j and kMlR distances accumulate in registers over all the
// steps, so the T2 tensor, 3 Rmax Nt/2 complex values per site, is not stored
// at all -- read and written once per step it was 191 MB per step at 24^4, 39 us
// of every step, and another 25 us per level-4 step to clear it.  Now a step
// costs 16 SV Nt/2 bytes per (dir, R block) from L2.  More steps than slots:
// the sums pass from launch to launch through l2 (null otherwise; LOAD, STORE).
constexpr int kMlR = 4;
template <bool LOAD, bool STORE>
__global__ __launch_bounds__(256) void k_ml_accum(const double* __restrict__ p2, int nslots, double* __restrict__ l2,
                                                  double* __restrict__ l4, RepDesc r, int rmax, double l2norm,
                                                  int first) {
  const uint32_t SV = (uint32_t)r.SV, x = blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= SV) return;
  const uint32_t nrb = (uint32_t)(rmax + kMlR - 1) / kMlR;
  const uint32_t dir = blockIdx.y / nrb, R0 = (blockIdx.y - dir * nrb) * kMlR + 1u, j = blockIdx.z;
  const uint32_t n0 = (uint32_t)r.N[0], n1 = (uint32_t)r.N[1], nd = (uint32_t)r.N[dir];
  const uint32_t x1x2 = x / n0, x0 = x - x1x2 * n0, x2 = x1x2 / n1, x1 = x1x2 - x2 * n1;
  const uint32_t xd = dir == 0 ? x0 : dir == 1 ? x1 : x2, stride = dir == 0 ? 1u : dir == 1 ? n0 : n0 * n1;
  const uint32_t step = SV * (uint32_t)(r.N[3] / 2);  // complex values per slot
  const int64_t sz = (int64_t)SV * rmax * 3, base = x + (int64_t)SV * (R0 - 1) + (int64_t)SV * rmax * dir;
  uint32_t y[kMlR];
  C64 s[kMlR][2];
#pragma unroll
  for (int k = 0; k < kMlR; ++k) {
    // R <= rmax = Nx/2, which may exceed the extent of another direction
    y[k] = x - xd * stride + (xd + R0 + k) % nd * stride;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      s[k][h] = {0.0, 0.0};
      if (LOAD && R0 + k <= (uint32_t)rmax) s[k][h] = ldc(l2, base + (int64_t)SV * k + sz * (2 * j + h));
    }
  }
  const double* p = p2 + 2 * (size_t)(2 * j) * SV;
  for (int n = 0; n < nslots; ++n, p += 2 * (size_t)step) {
    C64 a[2], b[kMlR][2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      a[h] = ldc(p, x + h * SV);
#pragma unroll
      for (int k = 0; k < kMlR; ++k) b[k][h] = ldc(p, y[k] + h * SV);
    }
#pragma unroll
    for (int k = 0; k < kMlR; ++k)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const C64 pl = cmul(a[h], C64{b[k][h].re, -b[k][h].im});
        s[k][h] = {pl.re + s[k][h].re, pl.im + s[k][h].im};
      }
  }
#pragma unroll
  for (int k = 0; k < kMlR; ++k) {
    if (R0 + k > (uint32_t)rmax) break;
    const int64_t at = base + (int64_t)SV * k;
    if (STORE) {
#pragma unroll
      for (int h = 0; h < 2; ++h) stc64(l2, at + sz * (2 * j + h), s[k][h]);
    } else {
      C64 pl = {1.0, 0.0};
#pragma unroll
      for (int h = 0; h < 2; ++h) pl = cmul(pl, C64{s[k][h].re * l2norm, s[k][h].im * l2norm});
      if (!first) {
        const C64 o = ldc(l4, at + sz * j);
        pl = {pl.re + o.re, pl.im + o.im};
      }
      stc64(l4, at + sz * j, pl);
    }
  }
}

// multilevel.cu:532-553: C(R) = sum_x sum_dir prod_j (l4[.,j] * l4norm);
// optional per-site field ppSpace; one partial row of 2*rmax per 256 sites, one
// R per workgroup (blockIdx.y).
__global__ __launch_bounds__(256) void k_ml_final(const double* __restrict__ l4, double* __restrict__ ppspace,
                                                  RepDesc r, int rmax, double l4norm,
                                                  double* __restrict__ partials) {
  const int32_t id = (int32_t)(blockIdx.x * blockDim.x + threadIdx.x), R = (int32_t)blockIdx.y;
  const int64_t sz = (int64_t)r.SV * rmax * 3;
  const int nl4 = r.N[3] / 4;
  double v[2] = {0.0, 0.0};
  if (id < r.SV) {
    C64 pl[3] = {{1.0, 0.0}, {1.0, 0.0}, {1.0, 0.0}};
    const int64_t base = id + (int64_t)r.SV * R;
    for (int j = 0; j < nl4; ++j)
#pragma unroll
      for (int dir = 0; dir < 3; ++dir) {
        const C64 q = ldc(l4, base + (int64_t)r.SV * rmax * dir + sz * j);
        pl[dir] = cmul(pl[dir], C64{q.re * l4norm, q.im * l4norm});
      }
#pragma unroll
    for (int dir = 0; dir < 3; ++dir) {
      v[0] += pl[dir].re;
      v[1] += pl[dir].im;
      if (ppspace) {  // the caller's memory: aligned for doubles only
        const int64_t at = base + (int64_t)r.SV * rmax * dir;
        ppspace[2 * at] = pl[dir].re;
        ppspace[2 * at + 1] = pl[dir].im;
      }
    }
  }
  const double o = block_sum<2>(v);
  if (threadIdx.x < 2) partials[((int64_t)blockIdx.x * rmax + R) * 2 + threadIdx.x] = o;
}

}  // namespace

hipError_t launch_ml_accum(const double* p2, int nslots, double* l2, bool load, bool store, double* l4,
                           const RepDesc& r, int rmax, double l2norm, bool first, hipStream_t st) {
  const int block = 256;
  const dim3 grid((unsigned)((r.SV + block - 1) / block), (unsigned)(3 * ((rmax + kMlR - 1) / kMlR)),
                  (unsigned)(r.N[3] / 4));
  auto* k = load ? (store ? k_ml_accum<true, true> : k_ml_accum<true, false>)
                 : (store ? k_ml_accum<false, true> : k_ml_accum<false, false>);
  k<<<grid, block, 0, st>>>(p2, nslots, l2, l4, r, rmax, l2norm, first ? 1 : 0);
  return hipGetLastError();
}

hipError_t launch_ml_final(const double* l4, double* ppspace, const RepDesc& r, int rmax, double l4norm,
                           double* partials, int nblk, int block, hipStream_t st) {
  k_ml_final<<<dim3(nblk, rmax), block, 0, st>>>(l4, ppspace, r, rmax, l4norm, partials);
  return hipGetLastError();
}

}  // namespace u1d
