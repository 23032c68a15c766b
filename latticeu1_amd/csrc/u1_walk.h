// u1_walk.h -- two checkerboard phases (parity, A) and (parity, B) in one
// launch, by wavefronts that walk along the diagonals e_B - e_A: the order of
// the updates and the addresses of the angles (k_walk in u1_walk.hip; emulated
// on the CPU against two sequential phases).
//
// Phase (parity, B) reads, of the links phase (parity, A) writes, only
// theta_A(x) and theta_A(x + e_B - e_A); phase (parity, A) reads theta_B at
// this parity only at x and x + e_A - e_B (the c and d angles of the staple,
// staple.h:85-92).  So along a diagonal x_j = x_0 + j (e_B - e_A), closed by
// the periodic boundary, the updates A(j) of theta_A(x_j) and B(j) of
// theta_B(x_j) may run in any order that has A(j) and A(j + 1) before B(j), and
// neither reads anything outside its diagonal that the launch writes.  A
// wavefront takes a segment j0 <= j < j1 of 64 diagonals, one per lane:
//     A(j0);  then A(j + 1), B(j) for j = j0 ... j1 - 2;  then B(j1 - 1),
// handing each new theta_A on in a register.  Only B(j1 - 1) needs an angle of
// another wavefront, theta_A(x_j1), from the first A of the next segment; a
// workgroup holds all segments of its diagonals, every wavefront leaves its
// first new theta_A in LDS, and one workgroup barrier after the first A covers
// that exchange and also keeps the store of B(j1 - 1) behind the next
// segment's read of the old theta_B(x_j1 - 1) in its A(j1).
//
// Loads.  With u_j = x_j + e_A = x_{j-1} + e_B and v_j = x_j - e_B = x_{j-1} -
// e_A, a step's links are a rung -- theta_A..D(u_j), theta_A,B(v_j),
// theta_C,D(x_j + e_A - e_C,D), read by A(j), B(j - 1) and A(j - 1) -- and a
// site -- theta_A..D(x_j), theta_A,B(x_j +- e_C,D), theta_C,D(x_j - e_C,D) --:
// 22 loads for two link updates, where two phase launches make 38.
#pragma once
#include <stdint.h>

#include <algorithm>
#include <vector>

#include "u1_device.h"

namespace u1d {

template <typename Real>
struct Rung {
  Real u[4];    // theta_A, theta_B, theta_C, theta_D at u_j
  Real va, vb;  // theta_A, theta_B at v_j
  Real w[2];    // theta_C, theta_D at x_j + e_A - e_C, x_j + e_A - e_D
};
template <typename Real>
struct RungSite {
  Real x[4];          // theta_A, theta_B, theta_C, theta_D at x_j
  Real ap[2], am[2];  // theta_A at x_j + e_C, e_D and x_j - e_C, e_D
  Real bp[2], bm[2];  // theta_B there
  Real f[2];          // theta_C at x_j - e_C, theta_D at x_j - e_D
};
// Place of x_j: byte offset base + off within the half of one direction's
// angles; base is wave-uniform.  t: its time slice.
struct WalkPos {
  uint32_t base, off;
  int32_t t;
};

__host__ __device__ __forceinline__ int32_t step_up(int32_t x, int32_t n) { return x + 1 == n ? 0 : x + 1; }
__host__ __device__ __forceinline__ int32_t step_dn(int32_t x, int32_t n) { return x == 0 ? n - 1 : x - 1; }

// Diagonals along e_t - e_z (A = 2, B = 3).  Diagonal c visits the planes
// (-j, c + j), j < len = lcm(Nz, Nt), c < gcd(Nz, Nt): at the same step all
// diagonals are in the same z, so what c and c + 1 share (the plane at t + 1)
// they read at the same time.  The in-plane index and its x and y neighbours
// stay the same all along (z + t keeps its parity).
//
// UNIFORM: one segment per wavefront, 64 consecutive in-plane sites on its
// lanes.  The walk then moves in the scalar unit only, and every access is a
// uniform offset plus one of five constant lane offsets.  Otherwise a
// wavefront holds several segments, 32 or 16 sites each, and plane offsets are
// kept per lane (about eight more vector instructions per link update, for
// more and smaller workgroups).  S: bytes of an angle.
template <int S, bool UNIFORM>
struct WalkZT {
  static constexpr int A = 2, B = 3, C = 0, D = 1;
  uint32_t same, opp;        // byte offset of the parity updated and of the other
  uint32_t Pb, Tb;           // bytes of a plane's, a time slice's angles of one parity and direction
  uint32_t Zlast, Tlast;     // offsets of the planes z = Nz - 1, t = Nt - 1
  uint32_t i, ip[2], im[2];  // lane: bytes to x, x + e_x, e_y, x - e_x, x - e_y in the plane
  uint32_t zb, tb;           // offset of the plane of x_j: z Pb, t Tb
  int32_t t;

  __host__ __device__ __forceinline__ uint32_t zup(uint32_t z) const { return z == Zlast ? 0 : z + Pb; }
  __host__ __device__ __forceinline__ uint32_t zdn(uint32_t z) const { return z == 0 ? Zlast : z - Pb; }
  __host__ __device__ __forceinline__ uint32_t tup(uint32_t x) const { return x == Tlast ? 0 : x + Tb; }
  __host__ __device__ __forceinline__ uint32_t tdn(uint32_t x) const { return x == 0 ? Tlast : x - Tb; }
  // lane: in-plane site (below P); diagonal c, first step j
  __host__ __device__ __forceinline__ void init(const RepDesc& r, int32_t parity, uint32_t lane, int32_t c, int32_t j) {
    init(r, parity, lane, c, j % r.N[2], (c + j) % r.N[3]);
  }
  // jz, jt: j modulo Nz, c + j modulo Nt
  __host__ __device__ __forceinline__ void init(const RepDesc& r, int32_t parity, uint32_t lane, int32_t c, int32_t jz,
                                                int32_t jt) {
    same = (uint32_t)(parity * r.HV) * S;
    opp = (uint32_t)((1 - parity) * r.HV) * S;
    Pb = (uint32_t)r.sz * S;
    Tb = (uint32_t)r.st * S;
    Zlast = (uint32_t)(r.N[2] - 1) * Pb;
    Tlast = (uint32_t)(r.N[3] - 1) * Tb;
    const uint32_t y = mdiv(lane, r.div_nxh_m, r.div_nxh_s);
    const int32_t xh = (int32_t)(lane - y * (uint32_t)r.nxh);
    const int32_t xodd = ((int32_t)y + c + parity) & 1;  // z + t = c modulo 2 all along
    i = lane * S;
    ip[0] = i + (uint32_t)(xodd ? (xh == r.nxh - 1 ? -(r.nxh - 1) : 1) : 0) * S;
    im[0] = i + (uint32_t)(xodd ? 0 : (xh == 0 ? r.nxh - 1 : -1)) * S;
    ip[1] = i + (uint32_t)((int32_t)y == r.N[1] - 1 ? -(r.N[1] - 1) * r.sy : r.sy) * S;
    im[1] = i + (uint32_t)(y == 0 ? (r.N[1] - 1) * r.sy : -r.sy) * S;
    t = jt;
    const int32_t z = jz == 0 ? 0 : r.N[2] - jz;
    zb = (uint32_t)z * Pb;
    tb = (uint32_t)t * Tb;
  }
  // angle of direction mu at lane offset k of the plane at offset p: the plane
  // belongs to the uniform part of the address if it is uniform
  template <typename L>
  __host__ __device__ __forceinline__ auto at(const L& ld, int mu, uint32_t half, uint32_t p, uint32_t k) const {
    return UNIFORM ? ld(mu, half + p, k) : ld(mu, half, p + k);
  }
  template <typename Real, typename L>
  __host__ __device__ __forceinline__ void rung(const L& ld, uint32_t pu, uint32_t pv, Rung<Real>& q) const {
    q.u[0] = at(ld, A, opp, pu, i);
    q.u[1] = at(ld, B, opp, pu, i);
    q.u[2] = at(ld, C, opp, pu, i);
    q.u[3] = at(ld, D, opp, pu, i);
    q.va = at(ld, A, opp, pv, i);
    q.vb = at(ld, B, opp, pv, i);
    q.w[0] = at(ld, C, same, pu, im[0]);
    q.w[1] = at(ld, D, same, pu, im[1]);
  }
  // rung j; returns theta_B(x_{j-1})
  template <typename Real, typename L>
  __host__ __device__ __forceinline__ Real start(const L& ld, Rung<Real>& q) const {
    const uint32_t zu = zup(zb), td = tdn(tb);
    rung(ld, zu + tb, zb + td, q);
    return at(ld, B, same, zu + td, i);
  }
  // site j and rung j + 1; moves on to j + 1
  template <typename Real, typename L>
  __host__ __device__ __forceinline__ WalkPos next(const L& ld, RungSite<Real>& q, Rung<Real>& r) {
    const uint32_t p = zb + tb;
    const WalkPos pos = {UNIFORM ? same + p : same, UNIFORM ? i : p + i, t};
    q.x[0] = at(ld, A, same, p, i);
    q.x[1] = at(ld, B, same, p, i);
    q.x[2] = at(ld, C, same, p, i);
    q.x[3] = at(ld, D, same, p, i);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      q.ap[k] = at(ld, A, opp, p, ip[k]);
      q.am[k] = at(ld, A, opp, p, im[k]);
      q.bp[k] = at(ld, B, opp, p, ip[k]);
      q.bm[k] = at(ld, B, opp, p, im[k]);
      q.f[k] = at(ld, k == 0 ? C : D, opp, p, im[k]);
    }
    const uint32_t zn = zdn(zb), tn = tup(tb);
    rung(ld, zb + tn, zn + tb, r);
    t = tb == Tlast ? 0 : t + 1;
    zb = zn;
    tb = tn;
    return pos;
  }
};

// One wavefront's segment of `steps` >= 1 steps.  ld(mu, base, off): the angle
// at byte base + off of direction mu.  update_a(site, pos, rung j, rung j + 1,
// old theta_B(x_{j-1})) returns the new theta_A(x_j); update_b(site, pos,
// theta_B(u_j), rung j + 1, new theta_A(x_j), new theta_A(x_{j+1})).  first()
// runs A(j0), rest(next) the others, next() giving the new theta_A(x_j1) that
// another wavefront (or this one) left after its first().  UNROLL: steps taken
// two at a time, so that the rungs and sites alternate between two sets of
// registers instead of being moved.
template <typename Real, typename Walk, typename L, typename UA, typename UB>
struct WalkSegment {
  Walk& wk;
  const L& ld;
  const UA& update_a;
  const UB& update_b;
  Rung<Real> ra, rb;
  RungSite<Real> sa, sb;
  WalkPos pa, pb;
  Real ub, na, nb;

  __host__ __device__ __forceinline__ Real first() {
    const Real before = wk.start(ld, rb);
    pa = wk.next(ld, sa, ra);
    na = update_a(sa, pa, rb, ra, before);
    ub = rb.u[1];
    return na;
  }
  // A(j + 1), B(j): r, s, p, n of step j; the other set receives j + 1's
  __host__ __device__ __forceinline__ void step(Rung<Real>& r, Rung<Real>& r2, RungSite<Real>& s, RungSite<Real>& s2,
                                                WalkPos& p, WalkPos& p2, Real& n, Real& n2) {
    p2 = wk.next(ld, s2, r2);
    n2 = update_a(s2, p2, r, r2, s.x[1]);
    update_b(s, p, ub, r, n, n2);
    ub = r.u[1];
  }
  template <bool UNROLL, typename N>
  __host__ __device__ __forceinline__ void rest(int32_t steps, const N& next) {
    int32_t k = steps - 1;
    if (UNROLL) {
      for (; k >= 2; k -= 2) {
        step(ra, rb, sa, sb, pa, pb, na, nb);
        step(rb, ra, sb, sa, pb, pa, nb, na);
      }
    }
    for (; k >= 1; --k) {
      step(ra, rb, sa, sb, pa, pb, na, nb);
      ra = rb;
      sa = sb;
      pa = pb;
      na = nb;
    }
    update_b(sa, pa, ub, ra, na, next());
  }
};

// Launch geometry.  A workgroup holds the segments of `width` (64, 32 or 16)
// consecutive in-plane sites of one diagonal: a strip.  Its wavefronts hold 64 /
// width segments each, seg steps long (the last ones shorter or empty; with
// width < 64 all equal).
//
// XCD x (workgroup index modulo 8) takes the strips of group x % sg and the
// diagonals of group x / sg, strips fastest: sg x (8 / sg) groups as even as the
// extents allow, every XCD with the same number of workgroups, some of them
// empty if the groups are not equal.  sg = 0: workgroups in plain order.
struct WalkArgs {
  int32_t orbits, len, seg, width;
  int32_t strips, sg;
  int32_t gs, go;  // strips and diagonals of a group (rounded up)
  int32_t row;     // first measurement row (batched replicas)
  uint32_t gs_m, gs_s;
  uint32_t nt_m, nt_s;  // magic division by Nt
};
// Batched replicas: workgroup b walks block map[b].y (walk_place, plain order)
// of replica map[b].x; map[b].x = kWalkNone: empty.
struct WalkBlock {
  uint32_t x, y;
};
constexpr uint32_t kWalkNone = 0xffffffffu;
struct WalkBatch {
  const WalkArgs* args;  // per replica, one width
  const WalkBlock* map;
};
inline int walk_gcd(int a, int b) {
  while (b != 0) {
    const int m = a % b;
    a = b;
    b = m;
  }
  return a;
}
inline WalkArgs walk_args(const RepDesc& r, int waves, int width, int sg) {
  WalkArgs w{};
  w.orbits = walk_gcd(r.N[2], r.N[3]);
  w.len = r.N[2] / w.orbits * r.N[3];
  const int segs = waves * (64 / width);
  w.seg = (w.len + segs - 1) / segs;
  w.width = width;
  w.strips = (r.nxh * r.N[1] + width - 1) / width;
  w.sg = sg;
  w.gs = sg == 0 ? w.strips : (w.strips + sg - 1) / sg;
  w.go = sg == 0 ? w.orbits : (w.orbits + 8 / sg - 1) / (8 / sg);
  const MagicDiv m = make_magic((uint32_t)w.gs);
  w.gs_m = m.m;
  w.gs_s = m.s;
  const MagicDiv t = make_magic((uint32_t)r.N[3]);
  w.nt_m = t.m;
  w.nt_s = t.s;
  return w;
}
inline int walk_blocks(const WalkArgs& w) { return w.sg == 0 ? w.strips * w.orbits : 8 * w.gs * w.go; }
inline int walk_rows(const RepDesc& r, int width) {
  const WalkArgs w = walk_args(r, 1, width, 0);
  return w.strips * w.orbits;
}
// Strip and diagonal of workgroup b; false if it is empty.
__host__ __device__ __forceinline__ bool walk_place(const WalkArgs& w, uint32_t b, uint32_t* strip, uint32_t* orbit) {
  const uint32_t x = w.sg == 0 ? 0u : b & 7u, k = w.sg == 0 ? b : b >> 3;
  const uint32_t gx = w.sg == 0 ? 0u : x & (uint32_t)(w.sg - 1), gy = w.sg == 0 ? 0u : x >> __builtin_ctz((uint32_t)w.sg);
  const uint32_t q = mdiv(k, w.gs_m, w.gs_s), s = k - q * (uint32_t)w.gs;
  *strip = gx * (uint32_t)w.gs + s;
  *orbit = gy * (uint32_t)w.go + q;
  return *strip < (uint32_t)w.strips && *orbit < (uint32_t)w.orbits;
}

// Workgroup order of a batch: replicas with the longest segments first, cut
// into eight lists of equal work (steps, and one for a segment's start), one
// per XCD (workgroup index modulo 8): a replica's planes then share one L2, no
// XCD is left with the long ones, and the short ones fill the end.
inline std::vector<WalkBlock> walk_batch_order(const std::vector<WalkArgs>& w) {
  std::vector<uint32_t> by(w.size());
  uint64_t total = 0;
  for (size_t i = 0; i < w.size(); ++i) {
    by[i] = (uint32_t)i;
    total += (uint64_t)walk_blocks(w[i]) * (uint64_t)(w[i].seg + 1);
  }
  std::stable_sort(by.begin(), by.end(), [&](uint32_t a, uint32_t b) { return w[a].seg > w[b].seg; });
  std::vector<WalkBlock> list[8];
  uint64_t done = 0;
  size_t longest = 0;
  for (const uint32_t i : by)
    for (int b = 0; b < walk_blocks(w[i]); ++b) {
      std::vector<WalkBlock>& l = list[8 * done / total];
      l.push_back({i, (uint32_t)b});
      longest = std::max(longest, l.size());
      done += (uint64_t)(w[i].seg + 1);
    }
  std::vector<WalkBlock> map(8 * longest, WalkBlock{kWalkNone, 0});
  for (int x = 0; x < 8; ++x)
    for (size_t k = 0; k < list[x].size(); ++k) map[8 * k + (size_t)x] = list[x][k];
  return map;
}

// Launch shapes the kernels take: whole wavefronts, none without a step.
constexpr int walk_max_waves(int elem_bytes) { return elem_bytes == 8 ? 8 : 16; }
inline bool walk_shape_ok(const RepDesc& r, int elem_bytes, int block, int width, int sg) {
  if (block < 64 || block > 64 * walk_max_waves(elem_bytes) || block % 64 != 0) return false;
  if (!(width == 64 || width == 32 || width == 16) || !(sg == 0 || sg == 1 || sg == 2 || sg == 4 || sg == 8)) return false;
  const WalkArgs w = walk_args(r, block / 64, width, sg);
  const int segs = block / width;
  return width == 64 ? w.seg * (segs - 1) < w.len : w.seg * segs == w.len;
}

}  // namespace u1d
