// CPU check of the diagonal walk (latticeu1_amd/csrc/u1_walk.h): the order of
// the updates and the addresses of every angle, on the kernels' own code.  The
// wavefronts' segments run in a random order that honours only the workgroup
// barrier (every first() of a workgroup before any of its rest()), lane by
// lane in a random order, with an update that mixes all nineteen angles; the
// lattice must come out exactly as from the two sequential phases, which read
// brute-force coordinates.  Every address must lie inside its direction's
// angles.  Also checks that the test sees a dropped barrier.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <functional>
#include <numeric>
#include <random>
#include <vector>

#include "../../latticeu1_amd/csrc/u1_walk.h"

using namespace u1d;
typedef uint64_t Word;  // "angles": exact integer mixing
constexpr int S = 8;

static Word mix(Word h, Word v) { return (h ^ (v + 0x9E3779B97F4A7C15ull + (h << 6) + (h >> 2))) * 0xD6E8FEB86659FD93ull; }
static Word mix6(int mu, int nu, Word a, Word b, Word c, Word d, Word e, Word f) {
  Word h = 0x51ED270B + 4 * mu + nu;
  for (Word w : {a, b, c, d, e, f}) h = mix(h, w);
  return h;
}

struct Lat {
  RepDesc r;
  std::vector<Word> w;  // [mu][parity][eo]
  bool ok = true;
  Word get(int mu, uint64_t byte) {
    if (byte % S || byte / S >= (uint64_t)r.V) { ok = false; return 0; }
    return w[(size_t)mu * r.V + byte / S];
  }
};
struct Load {
  Lat& l;
  Word operator()(int mu, uint32_t base, uint32_t off) const { return l.get(mu, (uint64_t)base + off); }
};

static RepDesc rep(const int* N) {
  RepDesc r{};
  for (int i = 0; i < 4; ++i) r.N[i] = N[i];
  r.nxh = N[0] / 2;
  r.V = N[0] * N[1] * N[2] * N[3];
  r.HV = r.V / 2;
  r.sy = r.nxh; r.sz = r.nxh * N[1]; r.st = r.sz * N[2];
  MagicDiv a = make_magic(r.nxh), b = make_magic(N[1]), c = make_magic(N[2]);
  r.div_nxh_m = a.m; r.div_nxh_s = a.s; r.div_ny_m = b.m; r.div_ny_s = b.s; r.div_nz_m = c.m; r.div_nz_s = c.s;
  return r;
}

// one sequential phase from coordinates
static void phase(Lat& l, int parity, int mu, int ml) {
  const RepDesc& r = l.r;
  const Lat old = l;
  auto at = [&](int nu, const int* x, int d1, int s1, int d2, int s2) {
    int y[4] = {x[0], x[1], x[2], x[3]};
    if (d1 >= 0) y[d1] = (y[d1] + s1 + r.N[d1]) % r.N[d1];
    if (d2 >= 0) y[d2] = (y[d2] + s2 + r.N[d2]) % r.N[d2];
    const int lex = y[0] + r.N[0] * (y[1] + r.N[1] * (y[2] + r.N[2] * y[3]));
    return (size_t)nu * r.V + ((y[0] + y[1] + y[2] + y[3]) & 1) * r.HV + (lex >> 1);
  };
  int x[4];
  for (x[3] = 0; x[3] < r.N[3]; ++x[3])
    for (x[2] = 0; x[2] < r.N[2]; ++x[2])
      for (x[1] = 0; x[1] < r.N[1]; ++x[1])
        for (x[0] = 0; x[0] < r.N[0]; ++x[0]) {
          if (((x[0] + x[1] + x[2] + x[3]) & 1) != parity) continue;
          if (mu != 3 && ml && x[3] % ml == 0) continue;
          Word h = old.w[at(mu, x, -1, 0, -1, 0)];
          for (int nu = 0; nu < 4; ++nu) {
            if (nu == mu) continue;
            h += mix6(mu, nu, old.w[at(nu, x, mu, 1, -1, 0)], old.w[at(mu, x, nu, 1, -1, 0)],
                      old.w[at(nu, x, -1, 0, -1, 0)], old.w[at(nu, x, mu, 1, nu, -1)],
                      old.w[at(mu, x, nu, -1, -1, 0)], old.w[at(nu, x, nu, -1, -1, 0)]);
          }
          l.w[at(mu, x, -1, 0, -1, 0)] = h;
        }
}

// One lane of one wavefront, suspended between first() and rest().
template <typename Walk>
struct Lane {
  Lat& l;
  Walk wk;
  int ml, steps;
  Load ld;
  std::function<Word(const RungSite<Word>&, const WalkPos&, const Rung<Word>&, const Rung<Word>&, Word)> ua;
  std::function<void(const RungSite<Word>&, const WalkPos&, Word, const Rung<Word>&, Word, Word)> ub;
  WalkSegment<Word, Walk, Load, decltype(ua), decltype(ub)> seg;
  Lane(Lat& lat, const Walk& w, int mask, int n)
      : l(lat), wk(w), ml(mask), steps(n), ld{lat}, seg{wk, ld, ua, ub} {
    constexpr int A = Walk::A, B = Walk::B, C = Walk::C, D = Walk::D;
    auto put = [this](int mu, const WalkPos& p, Word h) {
      if (((uint64_t)p.base + p.off) / S >= (uint64_t)l.r.V) { l.ok = false; return; }
      l.w[(size_t)mu * l.r.V + ((uint64_t)p.base + p.off) / S] = h;
    };
    ua = [this, put](const RungSite<Word>& q, const WalkPos& p, const Rung<Word>& r0, const Rung<Word>& r1, Word before) {
      if (ml && p.t % ml == 0) return q.x[0];
      const Word h = q.x[0] + mix6(A, B, r0.u[1], r1.u[0], q.x[1], before, r0.va, r0.vb) +
                     mix6(A, C, r0.u[2], q.ap[0], q.x[2], r0.w[0], q.am[0], q.f[0]) +
                     mix6(A, D, r0.u[3], q.ap[1], q.x[3], r0.w[1], q.am[1], q.f[1]);
      put(A, p, h);
      return h;
    };
    ub = [put](const RungSite<Word>& q, const WalkPos& p, Word u, const Rung<Word>& r1, Word n0, Word n1) {
      put(B, p, q.x[1] + mix6(B, A, r1.u[0], u, n0, n1, r1.vb, r1.va) +
                    mix6(B, C, r1.u[2], q.bp[0], q.x[2], r1.w[0], q.bm[0], q.f[0]) +
                    mix6(B, D, r1.u[3], q.bp[1], q.x[3], r1.w[1], q.bm[1], q.f[1]));
    };
  }
  Lane(const Lane&) = delete;
};

// Runs every lane's first(), then every rest(), each in random order (all
// workgroups together: no order between workgroups is assumed, and within one
// only the barrier).  drop: rest() of a lane right after its own first().
template <typename Walk>
static void run(std::vector<Lane<Walk>*>& lanes, const std::vector<int>& from, std::mt19937& rng, bool unroll,
                bool drop) {
  std::vector<Word> first(lanes.size());
  std::vector<size_t> order(lanes.size());
  std::iota(order.begin(), order.end(), 0);
  auto rest = [&](size_t k) {
    auto next = [&] { return first[(size_t)from[k]]; };
    if (unroll) lanes[k]->seg.template rest<true>(lanes[k]->steps, next);
    else lanes[k]->seg.template rest<false>(lanes[k]->steps, next);
  };
  std::shuffle(order.begin(), order.end(), rng);
  for (size_t k : order) {
    first[k] = lanes[k]->seg.first();
    if (drop) rest(k);
  }
  if (drop) return;
  std::shuffle(order.begin(), order.end(), rng);
  for (size_t k : order) rest(k);
}

template <bool UNIFORM>
static bool check(const int* N, int parity, int ml, int waves, int width, int sg, bool unroll, std::mt19937& rng,
                  bool drop) {
  using Walk = WalkZT<S, UNIFORM>;
  Lat l{rep(N), {}, true};
  l.w.resize(4 * (size_t)l.r.V);
  for (auto& w : l.w) w = rng();
  Lat ref = l;
  phase(ref, parity, 2, ml);
  phase(ref, parity, 3, ml);
  const WalkArgs w = walk_args(l.r, waves, width, sg);
  const int segs = waves * (64 / width), P = l.r.sz;
  std::vector<Lane<Walk>*> lanes;
  std::vector<int> from;
  std::vector<char> seen((size_t)w.strips * w.orbits, 0);
  for (int b = 0; b < walk_blocks(w); ++b) {
    uint32_t strip, c;
    if (!walk_place(w, (uint32_t)b, &strip, &c)) continue;
    if (seen[(size_t)c * w.strips + strip]++) return false;
    const int base = (int)lanes.size();
    const int used = (w.len + w.seg - 1) / w.seg, n = std::min(width, P - (int)strip * width);
    if (used > segs) return false;
    for (int k = 0; k < used; ++k)
      for (int i = 0; i < n; ++i) {
        Walk wk;
        wk.init(l.r, parity, strip * (uint32_t)width + (uint32_t)i, (int32_t)c, k * w.seg);
        lanes.push_back(new Lane<Walk>(l, wk, ml, std::min(w.seg, w.len - k * w.seg)));
        from.push_back(base + (k + 1 == used ? 0 : k + 1) * n + i);
      }
  }
  for (char k : seen)
    if (!k) return false;
  run(lanes, from, rng, unroll, drop);
  for (auto* p : lanes) delete p;
  return l.ok && l.w == ref.w;
}

int main() {
  const int geoms[][4] = {{2, 2, 2, 2}, {4, 4, 4, 4}, {4, 2, 6, 4}, {6, 4, 8, 12}, {4, 6, 4, 10}, {10, 6, 2, 8},
                          {4, 12, 12, 4}, {8, 4, 6, 8}, {6, 10, 4, 12}, {2, 6, 4, 2}, {18, 10, 4, 8}};
  std::mt19937 rng(11);
  long n = 0;
  for (const auto& N : geoms)
    for (int parity = 0; parity < 2; ++parity)
      for (int ml : {0, 2, 4})
        for (int waves = 1; waves <= 16; ++waves)
          for (int width : {64, 32, 16})
            for (int sg : {0, 1, 2, 4, 8}) {
              if (!walk_shape_ok(rep(N), 4, 64 * waves, width, sg)) continue;
              const bool u = (n & 1) != 0;
              if (!(width == 64 ? check<true>(N, parity, ml, waves, width, sg, u, rng, false)
                                : check<false>(N, parity, ml, waves, width, sg, u, rng, false))) {
                printf("walk wrong: %dx%dx%dx%d parity %d ml %d waves %d width %d sg %d\n", N[0], N[1], N[2], N[3],
                       parity, ml, waves, width, sg);
                return 1;
              }
              ++n;
            }
  int seen = 0;
  for (int k = 0; k < 8; ++k) seen += !check<true>(geoms[3], k & 1, 0, 4, 64, 1, false, rng, true);
  if (seen != 8) { printf("a dropped barrier went unseen (%d of 8 caught)\n", seen); return 1; }
  printf("walk ok: %ld walks\n", n);
  return 0;
}
