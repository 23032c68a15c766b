// u1_capi.hip -- implementation of the C ABI (include/latticeu1_amd.h):
// runtime context, argument checks, launch geometry, the autotuner, the
// multilevel driver and the batched-replica ensemble with its hipGraph.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <fstream>
#include <map>
#include <sstream>
#include <string>
#include <vector>

#include "../../include/latticeu1_amd.h"
#include "u1_chain.h"
#include "u1_kernels.h"

using u1d::PhaseArgs;
using u1d::RepDesc;

namespace {

thread_local std::string g_err;

// Scratch of u1_plaquette_noalloc: the reduction rows of the plaquette pass
// and the fold's second-level rows, in a file-scope device array (each GPU the
// library runs on holds its own copy until the process ends).  Host code never
// passes the array's name to a kernel: it uses the device address that
// hipGetSymbolAddress returns for the current device (kept per device in
// g_scratch_dev, set in u1_init).
constexpr size_t kNoAllocScratchDoubles = 1u << 20;  // 8 MiB
static __device__ __align__(256) double scratch[kNoAllocScratchDoubles];
constexpr int kMaxDevices = 64;
constexpr int kMaxHits = 8190;    // Metropolis hits per link and pass
constexpr int kMaxMetrop = 4095;  // Metropolis passes: 12 bits of Philox counter word 2
constexpr int kChainMaxMargin = 1024;  // fused-pass schedule margin accepted from a tune cache
// A fused pass must take under this fraction of the unfused pass's time:
// overrelaxation passes save bandwidth and ramps; Metropolis passes, bound by
// their arithmetic, only ramps, a gain the short tuning runs overstate (a
// binary32 Metropolis pass chosen at 5 % ahead ran no faster in full sweeps).
constexpr float kChainMinGainOR = 0.97f;
constexpr float kChainMinGainMetropolis = 0.90f;
// Multilevel: device memory for the two-slice products of level-2 steps that are
// accumulated together, and the largest workspace kept between calls.
constexpr size_t kMlSlotBytes = (size_t)256 << 20;
constexpr size_t kMlKeepBytes = (size_t)1 << 30;
// A walk must take under this fraction of the two phases' time.
constexpr float kWalkMinGain = 0.97f;
// While tuning, a shape is not timed again whose single launch takes this many times
// the two phases' time (it counts its event's microseconds), which then falls this
// far behind them, or this far behind the best shape.
constexpr float kWalkTooSlow = 3.0f;
constexpr float kWalkBehind = 1.5f;
constexpr float kWalkBehindBest = 1.1f;
double* g_scratch_dev[kMaxDevices] = {};

// Launch shape of an update phase kernel: workgroup size, even/odd sites per
// thread, XCD-aware workgroup order.
struct Cfg {
  int block, spt, xcd, tile = 0;  // tile: single-lattice planes in 2 x 4 tiles (set_phase_tiles)
  int margin = 0;                 // fused passes (tile: tiles along z): schedule margin (chain_schedule)
};

struct Ctx {
  bool init = false;
  int device = 0;
  hipStream_t st = nullptr;
  double* partials = nullptr;  // reduction scratch
  size_t partials_cap = 0;     // in doubles
  double* work = nullptr;      // Polyakov-volume and temporal-link scratch of u1_poly_volume / u1_poly2
  size_t work_cap = 0;         // in doubles
  void* ml = nullptr;          // multilevel workspace, kept between calls up to kMlKeepBytes
  size_t ml_cap = 0;           // in bytes
  unsigned long long* counter = nullptr;
  // results of a measurement (64 doubles): pinned host memory that the last
  // kernel of the fold writes through its device address (no copy afterwards)
  double* dres = nullptr;
  double* dres_dev = nullptr;
  bool tune = true;
  // fused (parity, 0) + (parity, 1) update launches on single lattices:
  // 0 never, 1 where the tuner measures them faster, 2 always
  int pair = 1;
  int verbosity = 0;                      // 0 silent, 1 summarize, 2 verbose (tuner output on stderr)
  // multilevel level-2 steps: replayed from one captured hipGraph (true) or
  // enqueued eagerly (false); the same kernels and counters either way
  bool graphs = true;
  // fused parity passes (k_chain) on single lattices: 0 never, 1 where the
  // tuner measures them faster, 2 always (where the geometry allows)
  int chain = 1;
  uint32_t* chain_cnt = nullptr;  // completion counters, 4 Nz Nt
  size_t chain_cnt_cap = 0;       // in counters
  uint32_t* chain_err = nullptr;  // wait-timeout flag (pinned host memory, written by the kernels)
  int chain_nz = 0, chain_nt = 0, chain_per = 0;  // layout of the counters' last use (per: wavefronts per plane)
  uint32_t chain_inc[4] = {};                     // launches that counted into each row since the last clear
  std::map<std::string, uint32_t*> chain_sched;   // "Nz Nt bpp" -> schedule list (device)
  std::map<std::string, int> chain_sched_len;
  uint32_t* die_ctl = nullptr;    // counters of one-launch sweeps (DIE_CTL words, zero between launches)
  std::map<std::string, Cfg> tunecache;  // key -> launch shape
  int tune_loaded = 0;
};
Ctx G;

int fail(int code, const std::string& msg) {
  g_err = msg;
  return code;
}

#define HIPCHK(expr)                                                                              \
  do {                                                                                            \
    hipError_t e_ = (expr);                                                                       \
    if (e_ != hipSuccess) return fail(U1_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)
#define REQ_INIT() \
  if (!G.init) return fail(U1_ERR_STATE, "u1_init has not been called")
// Pointers handed to kernels or written on the host are never null.
#define REQ_PTR(p) \
  if (!(p)) return fail(U1_ERR_ARG, "null pointer argument: " #p)
#define RET(expr)             \
  do {                        \
    int rc_ = (expr);         \
    if (rc_ != U1_OK) return rc_; \
  } while (0)

// Temporary device buffer, freed on every return path (after the library
// stream has drained, so no queued kernel still uses it).
struct DevBuf {
  void* p = nullptr;
  DevBuf() = default;
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  ~DevBuf() {
    if (p) {
      (void)hipStreamSynchronize(G.st);
      (void)hipFree(p);
    }
  }
  hipError_t alloc(size_t bytes) { return hipMalloc(&p, bytes ? bytes : 4); }
  template <typename T>
  T* as() const {
    return (T*)p;
  }
};

// HIP events owned by one call, destroyed on every return path.
struct EventSet {
  std::vector<hipEvent_t> ev;
  EventSet() = default;
  EventSet(const EventSet&) = delete;
  EventSet& operator=(const EventSet&) = delete;
  ~EventSet() {
    for (hipEvent_t e : ev) (void)hipEventDestroy(e);
  }
  hipError_t create(hipEvent_t* out) {
    const hipError_t e = hipEventCreate(out);
    if (e == hipSuccess) ev.push_back(*out);
    return e;
  }
};

// parameters.cu:163-168 rejects odd extents; the kernels here also need
// 4 * V < 2^31 (32-bit link index and Philox counter word).
int check_geom(const u1_geom* g) {
  if (!g) return fail(U1_ERR_ARG, "null geometry");
  int64_t v = 1;
  for (int i = 0; i < 4; ++i) {
    if (g->dims[i] < 2 || (g->dims[i] % 2) != 0)
      return fail(U1_ERR_ARG, "Number of points should be an even number >= 2 in every direction");
    v *= g->dims[i];
  }
  if (4 * v >= (int64_t)1 << 31) return fail(U1_ERR_ARG, "lattice too large: 4*V must be < 2^31");
  if (!(g->aniso > 0.0)) return fail(U1_ERR_ARG, "anisotropy must be > 0");
  return U1_OK;
}

int check_prec(int prec) {
  if (prec != U1_F64 && prec != U1_F32) return fail(U1_ERR_ARG, "precision must be U1_F64 or U1_F32");
  return U1_OK;
}

int check_metro(const u1_metro* m) {
  if (!m) return fail(U1_ERR_ARG, "null Metropolis settings");
  if (m->proposal != U1_PROPOSAL_INDEPENDENT && m->proposal != U1_PROPOSAL_DELTA)
    return fail(U1_ERR_ARG, "unknown proposal kind");
  if (m->nhit < 1 || m->nhit > kMaxHits) return fail(U1_ERR_ARG, "nhit must be in [1, 8190]");
  if (m->proposal == U1_PROPOSAL_DELTA && !(m->step >= 0.0 && m->step <= 3.141592653589793))
    return fail(U1_ERR_ARG, "the delta proposal needs 0 <= step <= pi");
  return U1_OK;
}

RepDesc make_rep(const u1_geom* g, uint64_t seed, uint32_t c3) {
  RepDesc r{};
  for (int i = 0; i < 4; ++i) r.N[i] = g->dims[i];
  r.nxh = r.N[0] / 2;
  r.V = r.N[0] * r.N[1] * r.N[2] * r.N[3];
  r.HV = r.V / 2;
  r.SV = r.N[0] * r.N[1] * r.N[2];
  r.sy = r.nxh;
  r.sz = r.nxh * r.N[1];
  r.st = r.nxh * r.N[1] * r.N[2];
  r.blk_begin = 0;
  r.nblk = 0;
  r.c3 = c3;
  const u1d::MagicDiv a = u1d::make_magic((uint32_t)r.nxh), b = u1d::make_magic((uint32_t)r.N[1]),
                     c = u1d::make_magic((uint32_t)r.N[2]);
  r.div_nxh_m = a.m;
  r.div_nxh_s = a.s;
  r.div_ny_m = b.m;
  r.div_ny_s = b.s;
  r.div_nz_m = c.m;
  r.div_nz_s = c.s;
  r.beta = g->beta;
  r.aniso = g->aniso;
  r.inv_aniso_f = (float)(1.0 / g->aniso);
  r.aniso_f = (float)g->aniso;
  r.bl2e_f = (float)(g->beta * 1.4426950408889634);  // beta log2(e)
  // |S| <= 6 xi (temporal links) or 4 / xi + 2 xi, so a weight's exponent
  // beta (Re' - Re) is at most 2 |beta| |S|
  const double smax = std::max(6.0 * g->aniso, 4.0 / g->aniso + 2.0 * g->aniso);
  r.exp_small = 2.0 * std::fabs(g->beta) * smax < 650.0 ? 1u : 0u;
  r.seed = seed;
  r.lat_off = 0;
  return r;
}

void set_blocks(RepDesc& r, int block) { u1d::set_phase_blocks(r, block); }
// Single-lattice update launches: plane decomposition of a launch shape,
// planes in 2 x 4 tiles (one per XCD) if the shape asks for it.
void set_update_blocks(RepDesc& r, const Cfg& c) {
  u1d::set_phase_blocks(r, c.block * c.spt);
  u1d::set_phase_tiles(r, c.tile != 0);
}

size_t elem_size(int prec) { return prec == U1_F64 ? sizeof(double) : sizeof(float); }

int ensure_partials(size_t n) {
  if (n <= G.partials_cap) return U1_OK;
  HIPCHK(hipStreamSynchronize(G.st));  // no queued kernel still reads the old buffer
  if (G.partials) HIPCHK(hipFree(G.partials));
  G.partials = nullptr;
  size_t cap = std::max<size_t>(n, 1 << 16);
  HIPCHK(hipMalloc((void**)&G.partials, cap * sizeof(double)));
  G.partials_cap = cap;
  return U1_OK;
}

// Kept between calls and grown on demand (the reference allocates these
// per call, polyakov.cu:443-508, 618-654).
int ensure_work(size_t n) {
  if (n <= G.work_cap) return U1_OK;
  HIPCHK(hipStreamSynchronize(G.st));
  if (G.work) HIPCHK(hipFree(G.work));
  G.work = nullptr;
  G.work_cap = 0;
  HIPCHK(hipMalloc((void**)&G.work, n * sizeof(double)));
  G.work_cap = n;
  return U1_OK;
}

int ensure_ml(size_t bytes) {
  if (bytes <= G.ml_cap) return U1_OK;
  HIPCHK(hipStreamSynchronize(G.st));
  if (G.ml) HIPCHK(hipFree(G.ml));
  G.ml = nullptr;
  G.ml_cap = 0;
  HIPCHK(hipMalloc(&G.ml, bytes));
  G.ml_cap = bytes;
  return U1_OK;
}

// Room for nblk rows of nv partial sums followed by the fold's scratch rows.
int ensure_fold(int nblk, int nv) { return ensure_partials((size_t)nv * nblk + u1d::fold_scratch(nblk, nv)); }
double* fold_scratch_ptr(int nblk, int nv) { return G.partials + (size_t)nv * nblk; }

// Launch shape of the plaquette: the (workgroup, sites per thread) pair whose
// chunks tile a (z, t) plane of P = Nx/2 * Ny sites with the fewest idle
// slots, then the most sites per workgroup (fewer partial rows).
void plaquette_shape(const RepDesc& r, int prec, int* block, int* spt) {
  const int P = r.nxh * r.N[1];
  long best_slots = -1;
  int bb = 64, bs = 1;
  for (int s : {1, 2, 4}) {
    if (s == 4 && prec == U1_F64) continue;
    for (int b : {64, 128, 192, 256}) {
      const long chunk = (long)b * s;
      const long slots = (P + chunk - 1) / chunk * chunk;
      if (best_slots < 0 || slots < best_slots || (slots == best_slots && chunk > (long)bb * bs)) {
        best_slots = slots;
        bb = b;
        bs = s;
      }
    }
  }
  *block = bb;
  *spt = bs;
}

// ------------------------------------------------------------------ autotuner
// Own tuner (replacing the QUDA-derived tune.cpp:306-416): launch shape per
// (kernel class, geometry, precision) -- workgroup size and even/odd sites per
// thread -- chosen by timing every candidate with HIP events on a scratch copy
// of the lattice, so tuning never perturbs the chain (the reference backs up
// and restores lattice and RNG instead, tune.h preTune/postTune).  Results do
// not depend on the launch shape.
const Cfg kShapes[] = {{64, 1, 0},  {128, 1, 0}, {192, 1, 0}, {256, 1, 0}, {384, 1, 0},
                       {512, 1, 0}, {64, 2, 0},  {128, 2, 0}, {192, 2, 0}, {256, 2, 0},
                       {384, 2, 0}, {64, 4, 0},  {128, 4, 0}, {192, 4, 0}, {256, 4, 0}};
// every shape is tried with and without the XCD-aware workgroup order and,
// for a single lattice, with lexicographic or 2 x 4 tiled planes: the tiles
// cut the halo between XCDs while the lattice lives in the MALL, and have
// measured slower on a lattice streamed from HBM (96^4)
std::vector<Cfg> candidates(bool tiles) {
  std::vector<Cfg> v;
  for (int t = 0; t < (tiles ? 2 : 1); ++t)
    for (int x = 0; x < 2; ++x)
      for (Cfg c : kShapes) {
        c.xcd = x;
        c.tile = t;
        v.push_back(c);
      }
  return v;
}
const Cfg kDefaultCfg = {256, 1, 1, 0};

std::string vol_str(const u1_geom* g) {
  std::ostringstream s;
  s << g->dims[0] << "x" << g->dims[1] << "x" << g->dims[2] << "x" << g->dims[3];
  return s.str();
}
std::string tune_key(const char* name, const u1_geom* g, int prec) {
  return vol_str(g) + "\t" + name + (prec == U1_F64 ? "_f64" : "_f32");
}

int time_phase(int prec, int kind, void* lat, const PhaseArgs& a, int nb, Cfg c, float* ms) {
  EventSet es;
  hipEvent_t e0, e1;
  HIPCHK(es.create(&e0));
  HIPCHK(es.create(&e1));
  HIPCHK(u1d::launch_phase(prec, kind, 0, lat, a, nb, c.block, c.spt, G.st));  // warm-up
  HIPCHK(hipEventRecord(e0, G.st));
  for (int rep = 0; rep < 2; ++rep)
    for (int mu = 0; mu < 4; ++mu) HIPCHK(u1d::launch_phase(prec, kind, mu, lat, a, nb, c.block, c.spt, G.st));
  HIPCHK(hipEventRecord(e1, G.st));
  HIPCHK(hipEventSynchronize(e1));
  HIPCHK(hipEventElapsedTime(ms, e0, e1));
  return U1_OK;
}

// Launch shape for the update phase kernel class `kind` on this geometry.
int phase_cfg(int prec, int kind, const u1_geom* g, const void* lat, const PhaseArgs& proto, Cfg* cfg) {
  const char* name = kind == u1d::KIND_METROPOLIS ? "Metropolis" : "OverRelaxation";
  const std::string key = tune_key(name, g, prec);
  auto it = G.tunecache.find(key);
  if (it != G.tunecache.end()) {
    *cfg = it->second;
    return U1_OK;
  }
  if (!G.tune) {
    *cfg = kDefaultCfg;
    return U1_OK;
  }
  const int64_t bytes = 4 * (int64_t)proto.single.V * (int64_t)elem_size(prec);
  DevBuf scratch;
  HIPCHK(scratch.alloc(bytes));
  HIPCHK(hipMemcpyAsync(scratch.p, lat, bytes, hipMemcpyDeviceToDevice, G.st));
  // Three rounds over all candidates, best time per candidate: a round-robin
  // order keeps clock ramp-up and neighbour noise from favouring one shape.
  std::vector<Cfg> cands;
  for (const Cfg c : candidates(true))
    if (!(c.spt == 4 && prec != U1_F32)) cands.push_back(c);
  std::vector<float> tbest(cands.size(), 1e30f);
  for (int round = 0; round < 3; ++round)
    for (size_t i = 0; i < cands.size(); ++i) {
      const Cfg c = cands[i];
      PhaseArgs a = proto;
      a.accepts = nullptr;
      a.meas = nullptr;
      a.xcd = (uint32_t)c.xcd;
      set_update_blocks(a.single, c);
      float ms = 0;
      RET(time_phase(prec, kind, scratch.p, a, a.single.nblk, c, &ms));
      tbest[i] = std::min(tbest[i], ms);
    }
  size_t ib = 0;
  for (size_t i = 1; i < cands.size(); ++i)
    if (tbest[i] < tbest[ib]) ib = i;
  if (G.verbosity >= 2)
    for (size_t i = 0; i < cands.size(); ++i)
      std::fprintf(stderr, "tune %s: block %d, %d site(s)/thread, %s order%s: %.2f us per launch%s\n", key.c_str(),
                   cands[i].block, cands[i].spt, cands[i].xcd ? "XCD" : "plain", cands[i].tile ? ", tiled planes" : "",
                   1e3 * tbest[i] / 8.0, i == ib ? "  <- chosen" : "");
  else if (G.verbosity >= 1)
    std::fprintf(stderr, "tune %s: block %d, %d site(s)/thread, %s order%s: %.2f us per launch\n", key.c_str(),
                 cands[ib].block, cands[ib].spt, cands[ib].xcd ? "XCD" : "plain", cands[ib].tile ? ", tiled planes" : "",
                 1e3 * tbest[ib] / 8.0);
  G.tunecache[key] = cands[ib];
  *cfg = cands[ib];
  return U1_OK;
}

// Fused pair shapes of a geometry: one step over the plane with 1, 2 or 3 sites
// per thread, where that fits a workgroup, and skewed steps (k_pair, PAIR_SKEW)
// of a few workgroup sizes: two, four and eight wavefronts (a barrier then joins
// few, and several workgroups share a CU) and 2, 3 or 4 even steps.
std::vector<Cfg> pair_candidates(int prec, const RepDesc& r) {
  const int P = r.nxh * r.N[1];
  std::vector<Cfg> v;
  auto add = [&v](int b, int spt) {
    for (const Cfg& c : v)
      if (c.block == b && c.spt == spt) return;
    for (int t = 0; t < 2; ++t)
      for (int x = 0; x < 2; ++x) v.push_back(Cfg{b, spt, x, t});
  };
  auto waves = [](int n) { return (n + 63) / 64 * 64; };
  const int maxb = u1d::pair_max_block((int)elem_size(prec), 1);
  for (int spt = 1; spt <= (prec == U1_F32 ? 3 : 2); ++spt) {
    const int b = waves((P + spt - 1) / spt);
    if (b <= u1d::pair_max_block((int)elem_size(prec), spt)) add(b, spt);
  }
  for (int b : {128, 256, 512, waves((P + 1) / 2), waves((P + 2) / 3), waves((P + 3) / 4)})
    if (b < P && b <= maxb && b >= 2 * r.nxh) add(b, 1);
  if (v.empty()) add(maxb, 1);  // rows of more than half a workgroup
  return v;
}
bool pair_shape_ok(int prec, const Cfg& c) {
  if (!(c.spt == 1 || c.spt == 2 || ((c.spt == 3 || c.spt == 4) && prec == U1_F32))) return false;
  const int maxb = u1d::pair_max_block((int)elem_size(prec), c.spt);
  return c.block >= 64 && c.block <= maxb && c.block % 64 == 0;
}
// Plane decomposition of the fused pair: one chunk (workgroup) per plane.
void set_pair_blocks(RepDesc& r, const Cfg& c) {
  u1d::set_phase_blocks(r, r.nxh * r.N[1]);
  u1d::set_phase_tiles(r, c.tile != 0);
}

int time_pair(int prec, int kind, void* lat, const PhaseArgs& a, const Cfg& c, float* ms) {
  EventSet es;
  hipEvent_t e0, e1;
  HIPCHK(es.create(&e0));
  HIPCHK(es.create(&e1));
  const int plane = a.single.nxh * a.single.N[1];
  HIPCHK(u1d::launch_pair(prec, kind, lat, a, a.single.nblk, c.block, c.spt, plane, G.st));  // warm-up
  HIPCHK(hipEventRecord(e0, G.st));
  for (int rep = 0; rep < 4; ++rep)
    HIPCHK(u1d::launch_pair(prec, kind, lat, a, a.single.nblk, c.block, c.spt, plane, G.st));
  HIPCHK(hipEventRecord(e1, G.st));
  HIPCHK(hipEventSynchronize(e1));
  HIPCHK(hipEventElapsedTime(ms, e0, e1));
  return U1_OK;
}

// Shape of the fused (parity, 0) + (parity, 1) launch for kernel class `kind`
// on this geometry, or block = 0 for two separate launches.  With tuning, the
// best pair shape is timed against the two phases in the single-phase shape
// `single` (tuned), on a scratch copy; the decision is cached with the shapes.
int pair_cfg(int prec, int kind, const u1_geom* g, const void* lat, const PhaseArgs& proto, const Cfg& single,
             Cfg* cfg) {
  *cfg = Cfg{0, 1, 0, 0};
  if (G.pair == 0) return U1_OK;
  if (proto.single.nxh * proto.single.N[1] > u1d::pair_max_plane((int)elem_size(prec)))
    return U1_OK;  // the plane's angles do not fit the pair kernel's LDS: two launches
  const char* name = kind == u1d::KIND_METROPOLIS ? "MetropolisPair" : "OverRelaxationPair";
  const std::string key = tune_key(name, g, prec);
  const std::vector<Cfg> cands = pair_candidates(prec, proto.single);
  // forced without a tuned pair shape: XCD order, lexicographic planes, 2
  // (binary32, one step) or 1 sites per thread
  auto forced_default = [&]() {
    for (const int spt : {1, prec == U1_F32 ? 2 : 1})
      for (const Cfg& c : cands)
        if (c.spt == spt && c.xcd == 1 && c.tile == 0) *cfg = c;
  };
  auto it = G.tunecache.find(key);
  if (it != G.tunecache.end()) {  // block 0: the tuner measured two launches faster
    if (it->second.block != 0) *cfg = it->second;
    else if (G.pair == 2) forced_default();
    return U1_OK;
  }
  if (!G.tune) {
    if (G.pair == 2) forced_default();
    return U1_OK;
  }
  const int64_t bytes = 4 * (int64_t)proto.single.V * (int64_t)elem_size(prec);
  DevBuf scratch;
  HIPCHK(scratch.alloc(bytes));
  HIPCHK(hipMemcpyAsync(scratch.p, lat, bytes, hipMemcpyDeviceToDevice, G.st));
  std::vector<float> tbest(cands.size(), 1e30f);
  float tsep = 1e30f;  // phases (parity, 0) and (parity, 1) as two launches each
  for (int round = 0; round < 3; ++round) {
    for (size_t i = 0; i < cands.size(); ++i) {
      PhaseArgs a = proto;
      a.accepts = nullptr;
      a.meas = nullptr;
      a.xcd = (uint32_t)cands[i].xcd;
      set_pair_blocks(a.single, cands[i]);
      float ms = 0;
      RET(time_pair(prec, kind, scratch.p, a, cands[i], &ms));
      tbest[i] = std::min(tbest[i], ms);
    }
    PhaseArgs a = proto;
    a.accepts = nullptr;
    a.meas = nullptr;
    a.xcd = (uint32_t)single.xcd;
    set_update_blocks(a.single, single);
    EventSet es;
    hipEvent_t e0, e1;
    HIPCHK(es.create(&e0));
    HIPCHK(es.create(&e1));
    HIPCHK(hipEventRecord(e0, G.st));
    for (int rep = 0; rep < 4; ++rep)
      for (int mu = 0; mu < 2; ++mu)
        HIPCHK(u1d::launch_phase(prec, kind, mu, scratch.p, a, a.single.nblk, single.block, single.spt, G.st));
    HIPCHK(hipEventRecord(e1, G.st));
    HIPCHK(hipEventSynchronize(e1));
    float ms = 0;
    HIPCHK(hipEventElapsedTime(&ms, e0, e1));
    tsep = std::min(tsep, ms);
  }
  size_t ib = 0;
  for (size_t i = 1; i < cands.size(); ++i)
    if (tbest[i] < tbest[ib]) ib = i;
  const bool use = G.pair == 2 || tbest[ib] < tsep;
  if (G.verbosity >= 2)
    for (size_t i = 0; i < cands.size(); ++i)
      std::fprintf(stderr, "tune %s: block %d, %d site(s)/thread, %s order%s: %.2f us per pair launch%s\n",
                   key.c_str(), cands[i].block, cands[i].spt, cands[i].xcd ? "XCD" : "plain",
                   cands[i].tile ? ", tiled planes" : "", 1e3 * tbest[i] / 4.0, i == ib ? "  <- best" : "");
  if (G.verbosity >= 1)
    std::fprintf(stderr, "tune %s: pair %.2f us (block %d, %d site(s)/thread) vs two launches %.2f us: %s\n",
                 key.c_str(), 1e3 * tbest[ib] / 4.0, cands[ib].block, cands[ib].spt, 1e3 * tsep / 4.0,
                 use ? "fused" : "separate");
  const Cfg chosen = use ? cands[ib] : Cfg{0, 1, 0, 0};
  G.tunecache[key] = tbest[ib] < tsep ? cands[ib] : Cfg{0, 1, 0, 0};
  *cfg = chosen;
  return U1_OK;
}

// Launch shapes of one kernel class on one geometry (block 0: not fused).
// walk: spt segments per wavefront (64 / width), tile the strip groups.
struct Shapes {
  Cfg phase = kDefaultCfg, pair{0, 1, 0, 0}, walk{0, 1, 0, 0}, chain{0, 1, 0, 0};
};
bool walk_cfg_ok(const RepDesc& r, int prec, const Cfg& c) {
  return c.spt >= 1 && 64 % c.spt == 0 &&
         u1d::walk_shape_ok(r, (int)elem_size(prec), c.block, 64 / c.spt, c.xcd ? 1 << c.tile : 0);
}

// The phases (a0.parity, mu0) and (a0.parity, mu0 + 1), mu0 = 0 or 2, in as many
// launches as sh has them.  rows(mu): measurement rows of the launch that starts
// with phase mu (null: not measuring).
template <typename Rows>
int launch_two_phases(int prec, int kind, void* lat, const PhaseArgs& a0, const Shapes& sh, int mu0, Rows rows) {
  PhaseArgs a = a0;
  if (mu0 == 2 && sh.walk.block != 0) {
    const Cfg& w = sh.walk;
    a.meas = rows(mu0);
    HIPCHK(u1d::launch_walk(prec, kind, lat, a, w.block, 64 / w.spt, w.xcd ? 1 << w.tile : 0, G.st));
    return U1_OK;
  }
  if (mu0 == 0 && sh.pair.block != 0) {
    a.xcd = (uint32_t)sh.pair.xcd;
    a.meas = rows(mu0);
    set_pair_blocks(a.single, sh.pair);
    HIPCHK(u1d::launch_pair(prec, kind, lat, a, a.single.nblk, sh.pair.block, sh.pair.spt,
                            a.single.nxh * a.single.N[1], G.st));
    return U1_OK;
  }
  a.xcd = (uint32_t)sh.phase.xcd;
  set_update_blocks(a.single, sh.phase);
  for (int mu = mu0; mu < mu0 + 2; ++mu) {
    a.meas = mu > 0 ? rows(mu) : nullptr;
    HIPCHK(u1d::launch_phase(prec, kind, mu, lat, a, a.single.nblk, sh.phase.block, sh.phase.spt, G.st));
  }
  return U1_OK;
}
const auto no_rows = [](int) -> double* { return nullptr; };

template <typename Rows>
int launch_parity(int prec, int kind, void* lat, const PhaseArgs& a, const Shapes& sh, Rows rows) {
  RET(launch_two_phases(prec, kind, lat, a, sh, 0, rows));
  return launch_two_phases(prec, kind, lat, a, sh, 2, rows);
}

// Shapes of the (parity, 2) + (parity, 3) walk: wavefronts and segments per
// wavefront in strip-grouped order (first tuning stage), then the orders of
// the best of them (second stage).
std::vector<Cfg> walk_shapes(const RepDesc& r, int prec) {
  std::vector<Cfg> v;
  for (int spt : {1, 2, 4})
    for (int w : {1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16}) {
      const Cfg c{64 * w, spt, 1, 1};
      if (walk_cfg_ok(r, prec, c)) v.push_back(c);
    }
  return v;
}
std::vector<Cfg> walk_orders(const std::vector<Cfg>& shapes, const std::vector<float>& t) {
  std::vector<size_t> by(shapes.size());
  for (size_t i = 0; i < by.size(); ++i) by[i] = i;
  std::sort(by.begin(), by.end(), [&](size_t a, size_t b) { return t[a] < t[b]; });
  std::vector<Cfg> v;
  for (size_t i = 0; i < by.size() && i < 3; ++i)
    for (int x = -1; x < 4; ++x) {
      Cfg c = shapes[by[i]];
      c.xcd = x >= 0;
      c.tile = std::max(x, 0);
      v.push_back(c);
    }
  return v;
}

// Shape of the walk for kernel class `kind`, or block = 0 for the two phases (sh:
// the shapes it would replace): where the tuner measures it faster, as pair_cfg;
// only with fused pairs left to the tuner (forced fusion means the plane pairs).
int walk_cfg(int prec, int kind, const u1_geom* g, const void* lat, const PhaseArgs& proto, const Shapes& sh,
             Cfg* cfg) {
  *cfg = Cfg{0, 1, 0, 0};
  if (G.pair != 1) return U1_OK;
  const char* name = kind == u1d::KIND_METROPOLIS ? "MetropolisWalk" : "OverRelaxationWalk";
  const std::string key = tune_key(name, g, prec);
  const std::vector<Cfg> shapes = walk_shapes(proto.single, prec);
  if (shapes.empty()) return U1_OK;
  auto it = G.tunecache.find(key);
  if (it != G.tunecache.end()) {  // block 0: the tuner measured the two phases faster
    if (it->second.block != 0 && walk_cfg_ok(proto.single, prec, it->second)) *cfg = it->second;
    return U1_OK;
  }
  if (!G.tune) return U1_OK;
  const int64_t bytes = 4 * (int64_t)proto.single.V * (int64_t)elem_size(prec);
  DevBuf scratch;
  HIPCHK(scratch.alloc(bytes));
  HIPCHK(hipMemcpyAsync(scratch.p, lat, bytes, hipMemcpyDeviceToDevice, G.st));
  EventSet es;
  hipEvent_t e0, e1;
  HIPCHK(es.create(&e0));
  HIPCHK(es.create(&e1));
  PhaseArgs a = proto;
  a.accepts = nullptr;
  a.meas = nullptr;
  Shapes s = sh;
  // mean time of reps launches after one to warm up
  auto timed = [&](const Cfg& c, float* best, int reps) -> int {
    s.walk = c;
    RET(launch_two_phases(prec, kind, scratch.p, a, s, 2, no_rows));
    HIPCHK(hipEventRecord(e0, G.st));
    for (int rep = 0; rep < reps; ++rep) RET(launch_two_phases(prec, kind, scratch.p, a, s, 2, no_rows));
    HIPCHK(hipEventRecord(e1, G.st));
    HIPCHK(hipEventSynchronize(e1));
    float ms = 0;
    HIPCHK(hipEventElapsedTime(&ms, e0, e1));
    *best = std::min(*best, ms / (float)reps);
    return U1_OK;
  };
  auto shape = [](const Cfg& c) {
    std::ostringstream o;
    o << c.block / 64 << " wavefronts of " << c.spt << " segment(s), ";
    if (c.xcd) o << (1 << c.tile) << " strip group(s)";
    else o << "plain order";
    return o.str();
  };
  const Cfg none{0, 1, 0, 0};
  float tsep = 1e30f;
  for (int round = 0; round < 3; ++round) RET(timed(none, &tsep, 4));
  const int reps = std::max(1, std::min(4, (int)(0.15f / tsep)));  // a tenth of a millisecond or so
  // three rounds over the candidates, but not over those that a launch shows to be
  // far behind the two phases, nor again over those behind the best (with few
  // diagonals all are, up to fifteen times: a first call at 28 x 20 x 36 x 22,
  // binary64, took 300 ms, 48 without walks)
  auto search = [&](const std::vector<Cfg>& cands, std::vector<float>& tbest) -> int {
    tbest.assign(cands.size(), 1e30f);
    std::vector<char> out(cands.size(), 0);
    for (size_t i = 0; i < cands.size(); ++i) {
      RET(timed(cands[i], &tbest[i], 1));
      out[i] = tbest[i] > kWalkTooSlow * tsep;
    }
    for (int round = 0; round < 3; ++round) {
      for (size_t i = 0; i < cands.size(); ++i)
        if (!out[i]) RET(timed(cands[i], &tbest[i], reps));
      const float most = std::min(kWalkBehind * tsep, kWalkBehindBest * *std::min_element(tbest.begin(), tbest.end()));
      for (size_t i = 0; i < cands.size(); ++i) out[i] = out[i] || tbest[i] > most;
    }
    if (G.verbosity >= 2)
      for (size_t i = 0; i < cands.size(); ++i)
        std::fprintf(stderr, "tune %s: %s: %.2f us per walk\n", key.c_str(), shape(cands[i]).c_str(), 1e3 * tbest[i]);
    return U1_OK;
  };
  std::vector<float> t1, t2;
  RET(search(shapes, t1));
  if (*std::min_element(t1.begin(), t1.end()) > kWalkBehindBest * tsep) {
    if (G.verbosity >= 1) std::fprintf(stderr, "tune %s: no walk near two launches %.2f us\n", key.c_str(), 1e3 * tsep);
    G.tunecache[key] = none;
    return U1_OK;
  }
  const std::vector<Cfg> orders = walk_orders(shapes, t1);
  RET(search(orders, t2));
  const Cfg best = orders[(size_t)(std::min_element(t2.begin(), t2.end()) - t2.begin())];
  // both sides timed afresh, alternating (chain_cfg), and a clear win asked for
  float tb = 1e30f;
  tsep = 1e30f;
  for (int round = 0; round < 5; ++round) {
    RET(timed(best, &tb, reps));
    RET(timed(none, &tsep, reps));
  }
  const bool use = tb < kWalkMinGain * tsep;
  if (G.verbosity >= 1)
    std::fprintf(stderr, "tune %s: walk %.2f us (%s) vs two launches %.2f us: %s\n", key.c_str(), 1e3 * tb,
                 shape(best).c_str(), 1e3 * tsep, use ? "walk" : "separate");
  *cfg = use ? best : none;
  G.tunecache[key] = *cfg;
  return U1_OK;
}

// Measurement rows of the phases (1, 1..3) of a pass launched by launch_parity:
// first row of the launch covering phase mu, and (mu = 4) their total.
int parity_row(const RepDesc& single, const Shapes& sh, int mu) {
  RepDesc r = single;
  set_update_blocks(r, sh.phase);
  const int n = r.nblk;
  set_pair_blocks(r, sh.pair);
  int row = 0;
  if (mu > 1) row += sh.pair.block != 0 ? r.nblk : n;
  if (mu > 2) row += sh.walk.block != 0 ? u1d::walk_rows(single, 64 / sh.walk.spt) : n;
  if (mu > 3 && sh.walk.block == 0) row += n;
  return row;
}

// ------------------------------------------------------------ fused passes
// Reports, and clears, a wait timeout of a fused pass (k_chain) since the
// last check; called after the library stream has been synchronised.
int chain_check() {
  if (G.chain_err && __atomic_load_n(G.chain_err, __ATOMIC_ACQUIRE) != 0) {
    __atomic_store_n(G.chain_err, 0u, __ATOMIC_RELEASE);
    return fail(U1_ERR_HIP, "fused parity pass: a dependency wait timed out; the updated lattice is not reliable");
  }
  return U1_OK;
}

int ensure_chain_err() {
  if (G.chain_err) return U1_OK;
  HIPCHK(hipHostMalloc((void**)&G.chain_err, sizeof(uint32_t), hipHostMallocMapped));
  *G.chain_err = 0;
  return U1_OK;
}

// Shapes of a fused pass: Cfg{block, spt, 1, tz, margin}, planes cut into
// chunks of block * spt sites, the (z, t) planes in tz x (8 / tz) tiles (one
// per XCD), dependencies at least margin + 1 schedule steps back.
void set_chain_blocks(RepDesc& r, const Cfg& c) { u1d::set_phase_blocks(r, c.block * c.spt); }
bool chain_shape_ok(const RepDesc& r0, const Cfg& c) {
  if (!(c.spt == 1 || c.spt == 2) || c.block < 64 || c.block > 512 || c.block % 64 != 0 || c.margin < 0 ||
      c.margin > kChainMaxMargin)
    return false;
  RepDesc r = r0;
  set_chain_blocks(r, c);
  return u1d::chain_possible(r.N[2], r.N[3], r.bpp, c.tile);
}
// Workgroup shapes (first tuning stage, default tiling and margin), then the
// tilings and margins of the best shape (second stage).
std::vector<Cfg> chain_shapes(const RepDesc& r) {
  std::vector<Cfg> v;
  for (int spt : {1, 2})
    for (int b : {64, 128, 192, 256, 384, 512}) {
      Cfg c{b, spt, 1, 2, 64};
      if (!chain_shape_ok(r, c)) c.tile = 1;
      if (chain_shape_ok(r, c)) v.push_back(c);
    }
  return v;
}
std::vector<Cfg> chain_layouts(const RepDesc& r, const Cfg& shape) {
  std::vector<Cfg> v;
  for (int tz : {1, 2, 4, 8})
    for (int margin : {16, 32, 64, 128, 256}) {
      Cfg c = shape;
      c.tile = tz;
      c.margin = margin;
      if (chain_shape_ok(r, c)) v.push_back(c);
    }
  return v;
}

// Schedule list, completion counters and counter targets of a fused pass over
// r (which carries set_chain_blocks) in workgroups of `block` threads;
// *nblocks: its workgroups.  Every wavefront adds 1 to its (mu, plane)
// counter, so a launch adds per = bpp * block / 64 to each.  The counters only
// grow: a launch waits for the value the previous launches with the same
// layout have brought them to plus per, and they are cleared (by a fill
// kernel on the library stream) when the layout changes or before they could
// overflow.
int chain_prepare(const RepDesc& r, const Cfg& cc, u1d::ChainArgs* c, int* nblocks) {
  const int nz = r.N[2], nt = r.N[3], bpp = r.bpp, per = r.bpp * (cc.block / 64), tz = cc.tile;
  const std::string key = std::to_string(nz) + " " + std::to_string(nt) + " " + std::to_string(bpp) + " " +
                          std::to_string(tz) + " " + std::to_string(cc.margin);
  auto it = G.chain_sched.find(key);
  if (it == G.chain_sched.end()) {
    const u1d::ChainSchedule s = u1d::chain_schedule(nz, nt, bpp, tz, cc.margin);
    uint32_t* d = nullptr;
    HIPCHK(hipMalloc((void**)&d, s.list.size() * sizeof(uint32_t)));
    const hipError_t e = hipMemcpy(d, s.list.data(), s.list.size() * sizeof(uint32_t), hipMemcpyHostToDevice);
    if (e != hipSuccess) {
      (void)hipFree(d);
      return fail(U1_ERR_HIP, std::string("chain schedule upload: ") + hipGetErrorString(e));
    }
    it = G.chain_sched.emplace(key, d).first;
    G.chain_sched_len[key] = (int)s.list.size();
  }
  const size_t need = 4 * (size_t)nz * (size_t)nt;
  bool clear = nz != G.chain_nz || nt != G.chain_nt || per != G.chain_per;
  for (int mu = 0; mu < 4; ++mu) clear = clear || (uint64_t)(G.chain_inc[mu] + 2) * (uint64_t)per >= (1ull << 31);
  if (need > G.chain_cnt_cap) {
    HIPCHK(hipStreamSynchronize(G.st));  // no queued launch still uses the old counters
    if (G.chain_cnt) HIPCHK(hipFree(G.chain_cnt));
    G.chain_cnt = nullptr;
    G.chain_cnt_cap = 0;
    HIPCHK(hipMalloc((void**)&G.chain_cnt, need * sizeof(uint32_t)));
    G.chain_cnt_cap = need;
    clear = true;
  }
  RET(ensure_chain_err());
  if (clear) {
    HIPCHK(u1d::launch_fill_zero(G.chain_cnt, (int64_t)(need * sizeof(uint32_t)), G.st));
    G.chain_nz = nz;
    G.chain_nt = nt;
    G.chain_per = per;
    for (int mu = 0; mu < 4; ++mu) G.chain_inc[mu] = 0;
  }
  void* err_dev = nullptr;
  HIPCHK(hipHostGetDevicePointer(&err_dev, G.chain_err, 0));
  c->sched = it->second;
  c->cnt = G.chain_cnt;
  c->err = (uint32_t*)err_dev;
  for (int mu = 0; mu < 4; ++mu) c->tgt[mu] = (G.chain_inc[mu] + 1) * (uint32_t)per;
  c->tz_log2 = tz == 8 ? 3 : tz == 4 ? 2 : tz == 2 ? 1 : 0;
  c->bz = (uint32_t)(nz / tz);
  c->bt = (uint32_t)(nt / (8 / tz));
  const u1d::MagicDiv md = u1d::make_magic(c->bz);
  c->bz_m = md.m;
  c->bz_s = md.s;
  *nblocks = 8 * G.chain_sched_len[key];
  return U1_OK;
}

// One fused pass (phases (a.parity, 0..3)) in shape cc; a.meas as for
// launch_chain.
int chain_launch(int prec, int kind, void* lat, const PhaseArgs& a0, const Cfg& cc) {
  PhaseArgs a = a0;
  a.xcd = 0;
  set_chain_blocks(a.single, cc);
  u1d::ChainArgs c{};
  int nb = 0;
  RET(chain_prepare(a.single, cc, &c, &nb));
  HIPCHK(u1d::launch_chain(prec, kind, lat, a, c, nb, cc.block, cc.spt, G.st));
  for (int mu = 0; mu < 4; ++mu) ++G.chain_inc[mu];
  return U1_OK;
}

// Shape of the fused parity pass for kernel class `kind` on this geometry, or
// block = 0 for the unfused launches.  With tuning, every fused shape is timed
// against the unfused pass (tuned shapes sh) on a scratch copy: four passes each (parities 0, 1, 0, 1); the decision is cached
// (MetropolisChain / OverRelaxationChain, block.x 0 = unfused).  Only for an
// unmasked single lattice whose (z, t) planes tile 2 x 4 (Nz even, Nt % 4 ==
// 0), and never during stream capture (the counter targets are per launch).
int chain_cfg(int prec, int kind, const u1_geom* g, const void* lat, const PhaseArgs& proto, const Shapes& sh,
              Cfg* cfg) {
  *cfg = Cfg{0, 1, 0, 0};
  if (G.chain == 0 || proto.ml != 0) return U1_OK;
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  HIPCHK(hipStreamIsCapturing(G.st, &cs));
  if (cs != hipStreamCaptureStatusNone) return U1_OK;
  const std::vector<Cfg> shapes = chain_shapes(proto.single);
  if (shapes.empty()) return U1_OK;
  const char* name = kind == u1d::KIND_METROPOLIS ? "MetropolisChain" : "OverRelaxationChain";
  const std::string key = tune_key(name, g, prec);
  auto forced_default = [&]() {
    *cfg = shapes[0];
    for (const Cfg& k : shapes)
      if (k.block == 256 && k.spt == 1) *cfg = k;
  };
  auto it = G.tunecache.find(key);
  if (it != G.tunecache.end()) {  // block 0: the tuner measured the unfused launches faster
    if (it->second.block != 0 && chain_shape_ok(proto.single, it->second)) *cfg = it->second;
    else if (G.chain == 2) forced_default();
    return U1_OK;
  }
  if (!G.tune) {
    if (G.chain == 2) forced_default();
    return U1_OK;
  }
  const int64_t bytes = 4 * (int64_t)proto.single.V * (int64_t)elem_size(prec);
  DevBuf scratch;
  HIPCHK(scratch.alloc(bytes));
  HIPCHK(hipMemcpyAsync(scratch.p, lat, bytes, hipMemcpyDeviceToDevice, G.st));
  EventSet es;
  hipEvent_t e0, e1;
  HIPCHK(es.create(&e0));
  HIPCHK(es.create(&e1));
  PhaseArgs a = proto;
  a.accepts = nullptr;
  a.meas = nullptr;
  auto timed = [&](bool fused, const Cfg& cc, float* ms) -> int {
    auto one = [&](int i) -> int {
      a.parity = i & 1;
      if (fused) return chain_launch(prec, kind, scratch.p, a, cc);
      return launch_parity(prec, kind, scratch.p, a, sh, no_rows);
    };
    RET(one(0));  // warm-up
    HIPCHK(hipEventRecord(e0, G.st));
    for (int i = 0; i < 4; ++i) RET(one(i));
    HIPCHK(hipEventRecord(e1, G.st));
    HIPCHK(hipEventSynchronize(e1));
    HIPCHK(hipEventElapsedTime(ms, e0, e1));
    return chain_check();
  };
  // three rounds over the candidates, best time per candidate; the unfused
  // pass timed in every round too
  float tsep = 1e30f;
  auto search = [&](const std::vector<Cfg>& cands, std::vector<float>& tbest) -> int {
    tbest.assign(cands.size(), 1e30f);
    for (int round = 0; round < 3; ++round) {
      for (size_t i = 0; i < cands.size(); ++i) {
        float ms = 0;
        RET(timed(true, cands[i], &ms));
        tbest[i] = std::min(tbest[i], ms);
      }
      float ms = 0;
      RET(timed(false, Cfg{0, 1, 0, 0}, &ms));
      tsep = std::min(tsep, ms);
    }
    return U1_OK;
  };
  auto report = [&](const std::vector<Cfg>& cands, const std::vector<float>& tbest, size_t ib) {
    if (G.verbosity >= 2)
      for (size_t i = 0; i < cands.size(); ++i)
        std::fprintf(stderr, "tune %s: block %d, %d site(s)/thread, %d z tiles, margin %d: %.2f us per fused pass%s\n",
                     key.c_str(), cands[i].block, cands[i].spt, cands[i].tile, cands[i].margin,
                     1e3 * tbest[i] / 4.0, i == ib ? "  <- best" : "");
  };
  auto argmin = [](const std::vector<float>& t) {
    size_t ib = 0;
    for (size_t i = 1; i < t.size(); ++i)
      if (t[i] < t[ib]) ib = i;
    return ib;
  };
  std::vector<float> t1, t2;
  RET(search(shapes, t1));
  const size_t i1 = argmin(t1);
  report(shapes, t1, i1);
  const std::vector<Cfg> layouts = chain_layouts(proto.single, shapes[i1]);
  RET(search(layouts, t2));
  const size_t i2 = argmin(t2);
  report(layouts, t2, i2);
  const Cfg best = layouts[i2];
  // the search's best time is the minimum over many candidates and rounds,
  // biased low against the unfused pass's few: both are timed afresh, the
  // same number of times, alternating, before they are compared
  float tb = 1e30f;
  tsep = 1e30f;
  for (int round = 0; round < 5; ++round) {
    float ms = 0;
    RET(timed(true, best, &ms));
    tb = std::min(tb, ms);
    RET(timed(false, Cfg{0, 1, 0, 0}, &ms));
    tsep = std::min(tsep, ms);
  }
  // chosen only on a clear win: the two paths' timings move by a few per cent
  // from one tuning run to the next
  const float gain = kind == u1d::KIND_METROPOLIS ? kChainMinGainMetropolis : kChainMinGainOR;
  const bool faster = tb < gain * tsep;
  const bool use = G.chain == 2 || faster;
  if (G.verbosity >= 1)
    std::fprintf(stderr,
                 "tune %s: fused pass %.2f us (block %d, %d site(s)/thread, %d z tiles, margin %d) vs unfused %.2f "
                 "us: %s\n",
                 key.c_str(), 1e3 * tb / 4.0, best.block, best.spt, best.tile, best.margin, 1e3 * tsep / 4.0,
                 use ? "fused" : "unfused");
  G.tunecache[key] = faster ? best : Cfg{0, 1, 0, 0};
  *cfg = use ? best : Cfg{0, 1, 0, 0};
  return U1_OK;
}

// Launch shapes of kernel class `kind` (tuned, if enabled).
int kind_shapes(int prec, int kind, const u1_geom* g, const void* lat, const PhaseArgs& proto, Shapes* sh) {
  RET(phase_cfg(prec, kind, g, lat, proto, &sh->phase));
  RET(pair_cfg(prec, kind, g, lat, proto, sh->phase, &sh->pair));
  RET(walk_cfg(prec, kind, g, lat, proto, *sh, &sh->walk));
  return chain_cfg(prec, kind, g, lat, proto, *sh, &sh->chain);
}

// Settles (tunes, if enabled) every launch shape a sweep of this geometry
// uses, and the fused passes' schedules and counters, so that a later sweep
// allocates and synchronises nothing (graph capture, timed regions).
int settle_update_cfgs(int prec, const u1_geom* g, const void* lat, const PhaseArgs& proto, int metrop, int ovrn) {
  Shapes sh;
  for (int kind = 0; kind < 2; ++kind) {
    if ((kind == u1d::KIND_METROPOLIS ? metrop : ovrn) <= 0) continue;
    RET(kind_shapes(prec, kind, g, lat, proto, &sh));
    if (sh.chain.block != 0) {
      RepDesc r = proto.single;
      set_chain_blocks(r, sh.chain);
      u1d::ChainArgs ca{};
      int nb = 0;
      RET(chain_prepare(r, sh.chain, &ca, &nb));
    }
  }
  return U1_OK;
}

// ------------------------------------------------------- one-launch sweeps
// Lattices that one XCD's share of the card may still run faster than the whole
// card does with a launch per one or two phases.  The tuner compares the two up
// to here: in binary32 they are level at 16^3 x 8 (2^14 sites per phase, 50 us per
// sweep), 16^4 takes 84 us against 56; in binary64 they meet near 2^13.
constexpr int kDieMaxHalfVolume = 1 << 14;
// With a multilevel mask every slab runs on an XCD by itself: sites of an XCD's
// slabs up to which the two are compared.
constexpr int kDieMaxSlabSites = 1 << 16;
// the accepted hits of a slab's four phases, counted by one wavefront (k_die)
static_assert(4ull * kDieMaxSlabSites * kMaxHits < 1ull << 32, "more than a 32-bit count holds");
// Passes of a one-launch sweep: its arrivals are counted in 32 bits, and beyond
// this many the launch itself is long.
constexpr int kDieMaxPasses = 1 << 13;
static_assert(8ull * u1d::kDieGroups * (kDieMaxPasses + 1) < 1ull << 32, "more arrivals than 32 bits count");
// A one-launch sweep must take under this fraction of the launches' time.
constexpr float kDieMinGain = 0.97f;

bool die_possible(const RepDesc& r, int ml, int metrop, int ovrn) {
  if (metrop < 0 || metrop > kMaxMetrop || ovrn < 0 || ovrn > kDieMaxPasses - metrop || metrop + ovrn == 0) return false;
  if (ml == 0) return r.HV <= kDieMaxHalfVolume;
  const int64_t rows = u1d::die_rows(u1d::die_slabs(ml, r.N[3]));
  return rows <= u1d::kDieGroups && rows * ml * r.st <= kDieMaxSlabSites;
}
// Workgroups of a slab.
uint32_t die_groups(const RepDesc& r, int ml, const Cfg& c) {
  const uint32_t rows = u1d::die_rows(u1d::die_slabs(ml, r.N[3]));
  const int sites = ml ? ml * r.st : r.HV;
  return std::min<uint32_t>((uint32_t)u1d::kDieGroups / rows, (uint32_t)((sites + c.block - 1) / c.block));
}

// What one-launch sweeps need allocated (counters for as many slabs as there can
// be).
int die_prepare() {
  RET(ensure_chain_err());
  if (G.die_ctl) return U1_OK;
  const size_t n = (size_t)u1d::DIE_CTL * 8 * u1d::kDieGroups;
  HIPCHK(hipMalloc((void**)&G.die_ctl, n * sizeof(uint32_t)));
  HIPCHK(u1d::launch_fill_zero(G.die_ctl, (int64_t)(n * sizeof(uint32_t)), G.st));
  return U1_OK;
}

int die_launch(int prec, void* lat, const PhaseArgs& a, int metrop, int ovrn, const Cfg& c, double* meas_dst,
               uint32_t patience = u1d::kDiePatience, bool in_order = false) {
  RET(die_prepare());
  u1d::DieArgs d{};
  void* err_dev = nullptr;
  HIPCHK(hipHostGetDevicePointer(&err_dev, G.chain_err, 0));
  d.ctl = G.die_ctl;
  d.err = (uint32_t*)err_dev;
  d.slabs = u1d::die_slabs(a.ml, a.single.N[3]);
  d.groups = die_groups(a.single, a.ml, c);
  d.metrop = metrop;
  d.ovrn = ovrn;
  d.patience = patience;
  d.in_order = in_order ? 1u : 0u;
  PhaseArgs b = a;
  b.meas = nullptr;
  if (meas_dst) {
    RET(ensure_partials(4 * u1d::kDieGroups));
    b.meas = G.partials;
    d.out = meas_dst;
    d.scale = 1.0 / (3.0 * (double)a.single.V);
  }
  HIPCHK(u1d::launch_die(prec, lat, b, d, c.block, G.st));
  return U1_OK;
}

int run_update(const u1_geom* g, int prec, void* lat, int metrop, int ovrn, const u1_metro* m, uint64_t seed,
               uint32_t stream, uint32_t sweep, uint32_t c3, int ml, unsigned long long* acc_dev,
               double* meas_dst = nullptr, const uint32_t* sweep_dev = nullptr, uint32_t sweep_mul = 0,
               bool one_launch = true);

// Workgroup size of the one-launch sweep of these passes, or block = 0: not
// with forced or forbidden fusion, large lattices or slabs, or where the tuner
// (on a scratch copy; cached per geometry and pass counts, block.x 0 =
// launches per phase) measures the launches faster.  meas: of the sweep with its
// plaquette, which costs the one launch about 10 us and the launches less; without
// tuning, and with no such entry loaded, as the plain sweep.
int die_cfg(const u1_geom* g, int prec, const void* lat, const PhaseArgs& a, int metrop, int ovrn, const u1_metro* m,
            bool meas, Cfg* cfg) {
  *cfg = Cfg{0, 1, 0, 0};
  if (G.chain != 1 || G.pair != 1 || !die_possible(a.single, a.ml, metrop, ovrn)) return U1_OK;
  const std::string name = "Sweep" + std::to_string(metrop) + "+" + std::to_string(ovrn) +
                           (a.ml ? "Mask" + std::to_string(a.ml) : "");
  const std::string plain = tune_key(name.c_str(), g, prec), key = meas ? tune_key((name + "Plaq").c_str(), g, prec) : plain;
  auto it = G.tunecache.find(key);
  if (it == G.tunecache.end() && meas && !G.tune) it = G.tunecache.find(plain);
  if (it != G.tunecache.end()) {
    *cfg = it->second;
    return U1_OK;
  }
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  HIPCHK(hipStreamIsCapturing(G.st, &cs));
  if (!G.tune || cs != hipStreamCaptureStatusNone) return U1_OK;
  const int64_t bytes = 4 * (int64_t)a.single.V * (int64_t)elem_size(prec);
  DevBuf scratch, plaq;
  HIPCHK(scratch.alloc(bytes));
  if (meas) HIPCHK(plaq.alloc(4 * sizeof(double)));
  HIPCHK(hipMemcpyAsync(scratch.p, lat, bytes, hipMemcpyDeviceToDevice, G.st));
  EventSet es;
  hipEvent_t e0, e1;
  HIPCHK(es.create(&e0));
  HIPCHK(es.create(&e1));
  PhaseArgs p = a;
  p.accepts = nullptr;
  p.sweep_dev = nullptr;
  // up to four passes of a kind: the others compare alike, and may be thousands
  // (4^3 x 6, binary64, 8000 passes: 4.5 s of tuning before a sweep of 0.11 s)
  const int mp = std::min(metrop, 4), op = std::min(ovrn, 4);
  auto one = [&](const Cfg& c) -> int {
    if (c.block != 0) return die_launch(prec, scratch.p, p, mp, op, c, plaq.as<double>());
    return run_update(g, prec, scratch.p, mp, op, m, a.single.seed, a.stream, a.sweep, a.single.c3, a.ml,
                      nullptr, plaq.as<double>(), nullptr, 0, false);
  };
  auto timed = [&](const Cfg& c, float* best) -> int {
    RET(one(c));  // warm-up
    HIPCHK(hipEventRecord(e0, G.st));
    for (int i = 0; i < 2; ++i) RET(one(c));
    HIPCHK(hipEventRecord(e1, G.st));
    HIPCHK(hipEventSynchronize(e1));
    float ms = 0;
    HIPCHK(hipEventElapsedTime(&ms, e0, e1));
    *best = std::min(*best, ms);
    return chain_check();
  };
  const Cfg none{0, 1, 0, 0};
  float tb = 1e30f, tsep = 1e30f;
  Cfg best = none;
  for (int b : {64, 128, 256, 512, 1024}) {
    if (b > u1d::die_max_block((int)elem_size(prec))) break;
    if (b > 64 && b / 2 >= (a.ml ? a.ml * a.single.st : a.single.HV)) break;
    float t = 1e30f;
    for (int round = 0; round < 2; ++round) RET(timed(Cfg{b, 1, 0, 0}, &t));
    if (t < tb) {
      tb = t;
      best = Cfg{b, 1, 0, 0};
    }
  }
  // both sides afresh, alternating
  tb = 1e30f;
  for (int round = 0; round < 3; ++round) {
    RET(timed(none, &tsep));
    RET(timed(best, &tb));
  }
  const bool use = tb < kDieMinGain * tsep;
  if (G.verbosity >= 1)
    std::fprintf(stderr, "tune %s: one launch %.2f us for %d+%d passes (block %d) vs %.2f us: %s\n", key.c_str(),
                 1e3 * tb / 2.0, mp, op, best.block, 1e3 * tsep / 2.0, use ? "one launch" : "separate");
  G.tunecache[key] = use ? best : none;
  *cfg = G.tunecache[key];
  return U1_OK;
}

// One UpdateLattice on a single lattice (update.cu:449-456 loop order).
// meas_dst (device, 4 doubles, nullable): the plaquette of the updated
// lattice, in u1_plaquette's normalisation, from the measuring variants of
// phases (parity 1, mu = 1, 2, 3) of the sweep's last pass.
// sweep_dev (nullable): the Philox sweep index is *sweep_dev * sweep_mul +
// sweep, read by the kernels (for graph capture; phase_cfg must have run).
// one_launch: the whole sweep may run as one launch (die_cfg).
int run_update(const u1_geom* g, int prec, void* lat, int metrop, int ovrn, const u1_metro* m, uint64_t seed,
               uint32_t stream, uint32_t sweep, uint32_t c3, int ml, unsigned long long* acc_dev,
               double* meas_dst, const uint32_t* sweep_dev, uint32_t sweep_mul, bool one_launch) {
  // the Metropolis pass index takes 12 bits of Philox counter word 2
  if (metrop < 0 || ovrn < 0 || metrop > kMaxMetrop) return fail(U1_ERR_ARG, "bad pass counts");
  PhaseArgs a{};
  a.single = make_rep(g, seed, c3);
  a.reps = nullptr;
  a.blockmap = nullptr;
  a.ml = ml;
  a.proposal = m->proposal;
  a.nhit = m->nhit;
  a.step = m->step;
  a.stream = stream;
  a.sweep = sweep;
  a.sweep_dev = sweep_dev;
  a.sweep_mul = sweep_mul;
  a.accepts = acc_dev;
  if (one_launch) {
    Cfg die;
    RET(die_cfg(g, prec, lat, a, metrop, ovrn, m, meas_dst != nullptr, &die));
    if (die.block != 0) return die_launch(prec, lat, a, metrop, ovrn, die, meas_dst);
  }
  Shapes sm, so;
  if (metrop > 0) RET(kind_shapes(prec, u1d::KIND_METROPOLIS, g, lat, a, &sm));
  if (ovrn > 0) RET(kind_shapes(prec, u1d::KIND_OVERRELAX, g, lat, a, &so));
  if (meas_dst && (ml != 0 || metrop + ovrn == 0)) return fail(U1_ERR_ARG, "no measuring pass");
  // measuring phases: parity 1, mu >= 1 of the last pass; one row per
  // workgroup of each launch that covers them, in launch order (a fused pass:
  // its own rows for phases 1-3, launch_chain)
  const Shapes& smeas = ovrn > 0 ? so : sm;
  int meas_rows_total = parity_row(a.single, smeas, 4);
  if (smeas.chain.block != 0) {
    RepDesc rc = a.single;
    set_chain_blocks(rc, smeas.chain);
    meas_rows_total = 3 * rc.N[2] * rc.N[3] * rc.bpp;
  }
  if (meas_dst) RET(ensure_fold(meas_rows_total, 4));
  // one pass of kind `kind`: per parity, one fused pass, or launch_parity
  auto pass = [&](int kind, uint32_t p, bool last, const Shapes& sh) -> int {
    a.pass = p;
    for (int parity = 0; parity < 2; ++parity) {
      const bool meas = meas_dst && last && parity == 1;
      a.parity = parity;
      if (sh.chain.block != 0) {
        PhaseArgs b = a;
        b.meas = meas ? G.partials : nullptr;
        RET(chain_launch(prec, kind, lat, b, sh.chain));
        continue;
      }
      RET(launch_parity(prec, kind, lat, a, sh, [&](int mu) -> double* {
        return meas ? G.partials + 4 * (size_t)parity_row(a.single, sh, std::max(mu, 1)) : nullptr;
      }));
    }
    return U1_OK;
  };
  for (int p = 0; p < metrop; ++p)
    RET(pass(u1d::KIND_METROPOLIS, (uint32_t)p, ovrn == 0 && p == metrop - 1, sm));
  for (int o = 0; o < ovrn; ++o) RET(pass(u1d::KIND_OVERRELAX, (uint32_t)o, o == ovrn - 1, so));
  if (meas_dst)
    HIPCHK(u1d::launch_finish_sums(G.partials, meas_rows_total, 4, 1.0 / (3.0 * (double)a.single.V), meas_dst,
                                   fold_scratch_ptr(meas_rows_total, 4), G.st));
  return U1_OK;
}

// Plaquette into a device result slot dst[4] (no synchronisation).
int plaquette_async(const u1_geom* g, int prec, const void* lat, double* dst) {
  RepDesc r = make_rep(g, 0, 0);
  int block, spt;
  plaquette_shape(r, prec, &block, &spt);
  set_blocks(r, block * spt);
  r.nblk *= 2;  // even sites, then odd sites
  const int nblk = r.nblk;
  RET(ensure_fold(nblk, 4));
  HIPCHK(u1d::launch_plaquette(prec, lat, r, G.partials, nblk, block, spt, G.st));
  HIPCHK(u1d::launch_finish_sums(G.partials, nblk, 4, 1.0 / (3.0 * (double)r.V), dst, fold_scratch_ptr(nblk, 4),
                                 G.st));
  return U1_OK;
}

// Doubles of the temporal-link field between links and product: the stochastic
// multihit, whose hits keep the card busy only with every link on its own, and the
// analytic one of more slices than k_poly_links takes.
size_t poly_field(const RepDesc& r, int mode) {
  const bool direct = mode == U1_POLY_PLAIN || (mode == U1_POLY_MULTIHIT && r.N[3] <= u1d::kPolyRows);
  return direct ? 0 : 2 * (size_t)r.V;
}
// Polyakov-loop volume P (polyakov.cu:415-508) into P (2 SV doubles, device);
// tl: poly_field doubles, if any.
int poly_volume_async(int prec, const void* lat, const RepDesc& r, int mode, const u1_metro* mh, uint32_t stream,
                      uint32_t c1, uint32_t c3, double* P, double* tl) {
  if (mode == U1_POLY_PLAIN) {
    HIPCHK(u1d::launch_poly_volume(prec, lat, r, P, G.st));
    return U1_OK;
  }
  if (poly_field(r, mode) == 0) {
    HIPCHK(u1d::launch_poly_links(prec, lat, r, P, G.st));
    return U1_OK;
  }
  HIPCHK(u1d::launch_temporal_links(prec, lat, r, mode, mh ? mh->proposal : 0, mh ? mh->nhit : 0,
                                    mh ? mh->step : 0.0, stream, c1, c3, tl, G.st));
  HIPCHK(u1d::launch_tprod(tl, r, P, G.st));
  return U1_OK;
}

// The n results the queued work leaves in G.dres, once it is done.
int take_results(double* host, size_t n) {
  HIPCHK(hipStreamSynchronize(G.st));
  std::memcpy(host, G.dres, n * sizeof(double));
  return chain_check();
}

int copy_back(double* host, const double* dev, size_t n) {
  HIPCHK(hipMemcpyAsync(host, dev, n * sizeof(double), hipMemcpyDeviceToHost, G.st));
  HIPCHK(hipStreamSynchronize(G.st));
  return chain_check();
}

}  // namespace

// Batched walks of one kernel class (u1d::WalkBatch; block 0: none).
struct EnsembleWalk {
  Cfg cfg = {0, 1, 0, 0};
  u1d::WalkArgs* args = nullptr;
  u1d::WalkBlock* map = nullptr;
  int blocks = 0;
};

struct u1_ensemble {
  int32_t nrep = 0;
  int prec = U1_F32;
  int32_t metrop = 1, ovrn = 3;
  u1_metro m{};
  std::vector<u1_geom> geoms;
  std::vector<RepDesc> upd_host, meas_host;  // per-replica descriptors (update / measurement launches)
  RepDesc* upd_dev = nullptr;
  RepDesc* meas_dev = nullptr;
  uint16_t* upd_map = nullptr;
  uint16_t* meas_map = nullptr;
  int upd_blocks = 0, meas_blocks = 0;
  void* lat = nullptr;
  int64_t total_links = 0;
  uint32_t* sweep_dev = nullptr;
  uint64_t sweeps_done = 0;
  double* res_dev = nullptr;
  double* partials = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  // sweep with the plaquette summed in its last pass (u1_ensemble_sweep_plaquette)
  double* mrows = nullptr;           // 4 doubles per row of the measuring launches
  u1d::RowSpan* mspans = nullptr;    // rows per launch and replica
  int mlaunches = 0;                 // measuring launches of a sweep
  int mfirst[4] = {0, 0, 0, 0};      // first row of the one that measures phase mu >= 1
  double* series_dev = nullptr;  // kEnsSeriesCap sweeps x nrep x 4 doubles
  uint32_t* base_dev = nullptr;  // sweep index of series row 0
  hipGraph_t mgraph = nullptr;
  hipGraphExec_t mexec = nullptr;
  Cfg cfg = {256, 1, 1, 0};  // launch shape of the update phases (tuned on first use)
  bool tuned = false;
  // fused (parity, 0) + (parity, 1) launches (block 0: none): per-replica
  // plane tables with one workgroup per (z, t) plane, or, where every plane
  // fits one (pair_packed), several planes to a workgroup
  Cfg pcfg = {0, 1, 0, 0};
  u1d::WalkBlock* pair_packed = nullptr;
  RepDesc* pair_dev = nullptr;
  uint16_t* pair_map = nullptr;
  int pair_blocks = 0;
  int pair_plane = 0;  // largest plane (Nx/2 * Ny sites) of the replicas: the pair kernel's LDS
  // walks over (parity, 2) + (parity, 3), one shape per kernel class
  EnsembleWalk walk[2];
};

namespace {

const int kEnsSeriesCap = 256;  // sweeps per device-side plaquette series chunk
const int kEnsBlock = 64;  // measurement launches: workgroup size and sites per thread
const int kEnsSpt = 1;     // (small plane chunks suit the small replicas of a batch)

// (Re)build the update-launch tables for launch shape c: per-replica plane
// decomposition and first workgroup, and the workgroup -> replica map.
int ensemble_build_update(u1_ensemble* e, Cfg c) {
  std::vector<uint16_t> umap;
  int nb = 0;
  for (int i = 0; i < e->nrep; ++i) {
    RepDesc& u = e->upd_host[i];
    set_blocks(u, c.block * c.spt);
    u.blk_begin = nb;
    nb += u.nblk;
    for (int b = 0; b < u.nblk; ++b) umap.push_back((uint16_t)i);
  }
  if (e->upd_map) HIPCHK(hipFree(e->upd_map));
  e->upd_map = nullptr;
  HIPCHK(hipMalloc((void**)&e->upd_map, umap.size() * sizeof(uint16_t)));
  HIPCHK(hipMemcpyAsync(e->upd_map, umap.data(), umap.size() * sizeof(uint16_t), hipMemcpyHostToDevice, G.st));
  HIPCHK(hipMemcpyAsync(e->upd_dev, e->upd_host.data(), e->nrep * sizeof(RepDesc), hipMemcpyHostToDevice, G.st));
  HIPCHK(hipStreamSynchronize(G.st));
  e->upd_blocks = nb;
  e->cfg = c;
  return U1_OK;
}

int ensemble_tune(u1_ensemble* e);
bool ensemble_pair_packs(const u1_ensemble* e, int plane);
int ensemble_build_pair(u1_ensemble* e, Cfg c);
int ensemble_build_walk(u1_ensemble* e, int kind, Cfg c);
// Settles the ensemble's launch shapes before either graph exists (they fix
// the launch layout): tuned, or, with tuning off and fused pairs forced
// (u1_set_pair_fusion(2)), default pair and walk shapes.
int ensemble_settle(u1_ensemble* e) {
  if (e->tuned || e->exec || e->mexec) return U1_OK;
  if (G.tune) return ensemble_tune(e);
  if (G.pair != 2 || e->pcfg.block != 0) return U1_OK;
  for (const int kind : {u1d::KIND_METROPOLIS, u1d::KIND_OVERRELAX})
    RET(ensemble_build_walk(e, kind, Cfg{128, 1, 0, 0}));  // two whole wavefronts: any extents
  int plane = 0;
  for (const RepDesc& r : e->upd_host) plane = std::max(plane, r.nxh * r.N[1]);
  return ensemble_build_pair(e, Cfg{ensemble_pair_packs(e, plane) ? (plane + 63) / 64 * 64 : 256, 1, 1, 0});
}

// Planes that fit a workgroup are packed (k_pair_packed): 64 replicas of 8^4 to
// 24^3 x 32, binary32, 970 us per sweep against 1136 us with one
// workgroup per plane.
bool ensemble_pair_packs(const u1_ensemble* e, int plane) {
  return (plane + 63) / 64 * 64 <= u1d::pair_max_block((int)elem_size(e->prec), 1);
}
// Workgroups of replica r's packed pairs (r.N, planes of 64-site chunks).
int ensemble_pair_groups(const RepDesc& r, const Cfg& c) {
  const int room = c.block / 64 / ((r.nxh * r.N[1] + 63) / 64);  // planes of a workgroup
  return (r.N[2] * r.N[3] + room - 1) / room;
}
int ensemble_launch_pair(u1_ensemble* e, int kind, void* lat, const PhaseArgs& a0) {
  PhaseArgs a = a0;
  a.reps = e->pair_dev;
  a.blockmap = e->pair_map;
  a.xcd = (uint32_t)e->pcfg.xcd;
  if (e->pair_packed)
    HIPCHK(u1d::launch_pair_packed(e->prec, kind, lat, a, e->pair_packed, e->pair_blocks, e->pcfg.block, G.st));
  else
    HIPCHK(u1d::launch_pair(e->prec, kind, lat, a, e->pair_blocks, e->pcfg.block, e->pcfg.spt, e->pair_plane, G.st));
  return U1_OK;
}

// Per-replica tables of the fused pair launches for shape c (block 0: none).
int ensemble_build_pair(u1_ensemble* e, Cfg c) {
  e->pcfg = Cfg{0, 1, 0, 0};  // set to c only once its tables are in place
  if (c.block == 0) return U1_OK;
  int plane = 0;
  for (const RepDesc& r : e->upd_host) plane = std::max(plane, r.nxh * r.N[1]);
  if (plane > u1d::pair_max_plane((int)elem_size(e->prec))) return U1_OK;  // planes too large for the LDS exchange
  std::vector<RepDesc> reps(e->upd_host);
  std::vector<uint16_t> pmap;
  int nb = 0;
  if (ensemble_pair_packs(e, plane)) {
    if (c.block < plane || c.spt != 1) return U1_OK;
    std::vector<u1d::WalkBlock> map;
    for (int i = 0; i < e->nrep; ++i) {
      RepDesc& p = reps[i];
      u1d::set_phase_blocks(p, 64);
      p.tile = 0;
      const int room = c.block / 64 / p.bpp;  // planes of a workgroup
      for (int b = 0; b < ensemble_pair_groups(p, c); ++b) map.push_back({(uint32_t)i, (uint32_t)(b * room * p.bpp)});
    }
    if (!e->pair_dev) HIPCHK(hipMalloc((void**)&e->pair_dev, e->nrep * sizeof(RepDesc)));
    if (e->pair_packed) HIPCHK(hipFree(e->pair_packed));
    e->pair_packed = nullptr;
    HIPCHK(hipMalloc((void**)&e->pair_packed, map.size() * sizeof(map[0])));
    HIPCHK(hipMemcpyAsync(e->pair_packed, map.data(), map.size() * sizeof(map[0]), hipMemcpyHostToDevice, G.st));
    HIPCHK(hipMemcpyAsync(e->pair_dev, reps.data(), e->nrep * sizeof(RepDesc), hipMemcpyHostToDevice, G.st));
    HIPCHK(hipStreamSynchronize(G.st));
    e->pair_blocks = (int)map.size();
    e->pcfg = c;
    return U1_OK;
  }
  for (int i = 0; i < e->nrep; ++i) {
    RepDesc& p = reps[i];
    u1d::set_phase_blocks(p, p.nxh * p.N[1]);  // one chunk per plane
    p.tile = 0;
    p.blk_begin = nb;
    nb += p.nblk;
    for (int b = 0; b < p.nblk; ++b) pmap.push_back((uint16_t)i);
  }
  if (!e->pair_dev) HIPCHK(hipMalloc((void**)&e->pair_dev, e->nrep * sizeof(RepDesc)));
  if (e->pair_map) HIPCHK(hipFree(e->pair_map));
  e->pair_map = nullptr;
  HIPCHK(hipMalloc((void**)&e->pair_map, pmap.size() * sizeof(uint16_t)));
  HIPCHK(hipMemcpyAsync(e->pair_map, pmap.data(), pmap.size() * sizeof(uint16_t), hipMemcpyHostToDevice, G.st));
  HIPCHK(hipMemcpyAsync(e->pair_dev, reps.data(), e->nrep * sizeof(RepDesc), hipMemcpyHostToDevice, G.st));
  HIPCHK(hipStreamSynchronize(G.st));
  e->pair_blocks = nb;
  e->pair_plane = plane;
  e->pcfg = c;
  return U1_OK;
}

void ensemble_drop_walk(EnsembleWalk& w) {
  if (w.args) (void)hipFree(w.args);
  if (w.map) (void)hipFree(w.map);
  w = EnsembleWalk{};
}
// Tables of kernel class `kind`'s walks for shape c (spt segments per
// wavefront; block 0, or a shape some replica cannot take: none).
int ensemble_build_walk(u1_ensemble* e, int kind, Cfg c) {
  EnsembleWalk& w = e->walk[kind];
  ensemble_drop_walk(w);
  if (c.block == 0) return U1_OK;
  std::vector<u1d::WalkArgs> args;
  int rows = 0;
  for (const RepDesc& r : e->upd_host) {
    if (!walk_cfg_ok(r, e->prec, c)) return U1_OK;
    args.push_back(u1d::walk_args(r, c.block / 64, 64 / c.spt, 0));
    args.back().row = rows;
    rows += u1d::walk_blocks(args.back());
  }
  const std::vector<u1d::WalkBlock> map = u1d::walk_batch_order(args);
  HIPCHK(hipMalloc((void**)&w.args, args.size() * sizeof(args[0])));
  HIPCHK(hipMalloc((void**)&w.map, map.size() * sizeof(map[0])));
  HIPCHK(hipMemcpyAsync(w.args, args.data(), args.size() * sizeof(args[0]), hipMemcpyHostToDevice, G.st));
  HIPCHK(hipMemcpyAsync(w.map, map.data(), map.size() * sizeof(map[0]), hipMemcpyHostToDevice, G.st));
  HIPCHK(hipStreamSynchronize(G.st));
  w.blocks = (int)map.size();
  w.cfg = c;
  return U1_OK;
}
int ensemble_launch_walk(u1_ensemble* e, int kind, void* lat, const PhaseArgs& a) {
  const EnsembleWalk& w = e->walk[kind];
  HIPCHK(u1d::launch_walk_batched(e->prec, kind, lat, a, u1d::WalkBatch{w.args, w.map}, w.blocks, w.cfg.block,
                                  64 / w.cfg.spt, G.st));
  return U1_OK;
}

// Measuring launches of a sweep -- parity 1 of its last pass: the pair (packed
// pairs only) or phase 1, the walk or phases 2 and 3 -- and their rows: spans,
// launch by launch, and e->mfirst.  Returns the number of rows.
int ensemble_meas_rows(u1_ensemble* e, std::vector<u1d::RowSpan>* spans) {
  const int kind = e->ovrn > 0 ? u1d::KIND_OVERRELAX : u1d::KIND_METROPOLIS;
  spans->clear();
  int rows = 0;
  for (int mu = 1; mu < 4; ++mu) {
    const bool pair = mu == 1 && e->pcfg.block != 0 && e->pair_packed, walk = mu >= 2 && e->walk[kind].cfg.block != 0;
    e->mfirst[mu] = mu == 3 && walk ? e->mfirst[2] : rows;
    if (mu == 3 && walk) continue;
    for (const RepDesc& r : e->upd_host) {
      int n = r.nblk;
      if (pair) n = ensemble_pair_groups(r, e->pcfg);
      if (walk) n = u1d::walk_rows(r, 64 / e->walk[kind].cfg.spt);
      spans->push_back({rows, n});
      rows += n;
    }
  }
  return rows;
}

// mrows (nullable): plaquette rows of the measuring launches (parity 1 of the
// last pass), laid out by ensemble_meas_rows.  With fused pairs (e->pcfg) the
// phases (parity, 0) + (parity, 1) of every pass, and with walks (e->walk) the
// phases (parity, 2) + (parity, 3), run as one launch; only a measuring pair
// that is not packed runs as two.
int ensemble_enqueue_phases(u1_ensemble* e, void* lat, double* mrows = nullptr) {
  PhaseArgs a{};
  a.reps = e->upd_dev;
  a.blockmap = e->upd_map;
  a.ml = 0;
  a.proposal = e->m.proposal;
  a.nhit = e->m.nhit;
  a.step = e->m.step;
  a.stream = u1r::STREAM_UPDATE;
  a.sweep = 0;
  a.sweep_dev = e->sweep_dev;
  a.sweep_mul = 1;
  a.accepts = nullptr;
  a.xcd = (uint32_t)e->cfg.xcd;
  auto pass = [&](int kind, uint32_t p, bool last) -> int {
    a.pass = p;
    for (int parity = 0; parity < 2; ++parity) {
      const bool measure = mrows && last && parity == 1;
      a.parity = parity;
      for (int mu = 0; mu < 4; ++mu) {
        if (mu == 0 && e->pcfg.block != 0 && (!measure || e->pair_packed)) {
          a.meas = measure ? mrows + 4 * (size_t)e->mfirst[1] : nullptr;
          RET(ensemble_launch_pair(e, kind, lat, a));
          ++mu;
          continue;
        }
        a.meas = measure && mu >= 1 ? mrows + 4 * (size_t)e->mfirst[mu] : nullptr;
        if (mu == 2 && e->walk[kind].cfg.block != 0) {
          RET(ensemble_launch_walk(e, kind, lat, a));
          ++mu;
          continue;
        }
        HIPCHK(u1d::launch_phase(e->prec, kind, mu, lat, a, e->upd_blocks, e->cfg.block, e->cfg.spt, G.st));
      }
    }
    return U1_OK;
  };
  for (int p = 0; p < e->metrop; ++p)
    RET(pass(u1d::KIND_METROPOLIS, (uint32_t)p, e->ovrn == 0 && p == e->metrop - 1));
  for (int o = 0; o < e->ovrn; ++o) RET(pass(u1d::KIND_OVERRELAX, (uint32_t)o, o == e->ovrn - 1));
  return U1_OK;
}

int ensemble_enqueue_sweep(u1_ensemble* e) {
  RET(ensemble_enqueue_phases(e, e->lat));
  HIPCHK(u1d::launch_increment(e->sweep_dev, G.st));
  return U1_OK;
}

// Time every launch-shape candidate over one full sweep of all replicas on a
// scratch copy of the packed lattice; keep the fastest.
int ensemble_tune(u1_ensemble* e) {
  const size_t bytes = (size_t)e->total_links * elem_size(e->prec);
  DevBuf scratch;
  HIPCHK(scratch.alloc(bytes));
  HIPCHK(hipMemcpyAsync(scratch.p, e->lat, bytes, hipMemcpyDeviceToDevice, G.st));
  EventSet es;
  hipEvent_t e0, e1;
  HIPCHK(es.create(&e0));
  HIPCHK(es.create(&e1));
  // m Metropolis and o overrelaxation passes, after one of each of them to warm up
  const int metrop = e->metrop, ovrn = e->ovrn;
  auto passes = [&](int m, int o) -> int {
    e->metrop = m;
    e->ovrn = o;
    const int rc = ensemble_enqueue_phases(e, scratch.p);
    e->metrop = metrop;
    e->ovrn = ovrn;
    return rc;
  };
  auto timed_passes = [&](int m, int o, float* t) -> int {
    RET(passes(std::min(m, 1), std::min(o, 1)));
    HIPCHK(hipEventRecord(e0, G.st));
    RET(passes(m, o));
    HIPCHK(hipEventRecord(e1, G.st));
    HIPCHK(hipEventSynchronize(e1));
    float ms = 0;
    HIPCHK(hipEventElapsedTime(&ms, e0, e1));
    *t = std::min(*t, ms);
    return U1_OK;
  };
  auto timed = [&](float* t) { return timed_passes(metrop, ovrn, t); };  // a whole sweep
  float best = 1e30f;
  Cfg bestc = e->cfg;
  for (const Cfg c : candidates(false)) {  // batched launches keep lexicographic planes
    if (c.spt == 4 && e->prec != U1_F32) continue;
    RET(ensemble_build_update(e, c));
    float t = 1e30f;
    RET(timed(&t));
    if (t < best) {
      best = t;
      bestc = c;
    }
  }
  RET(ensemble_build_update(e, bestc));
  // fused pairs: a few whole-plane shapes over full sweeps, against none
  if (G.pair != 0) {
    const Cfg none{0, 1, 0, 0};
    float tnone = best, tp = 1e30f;
    Cfg bestp = none;
    int plane = 0;
    for (const RepDesc& r : e->upd_host) plane = std::max(plane, r.nxh * r.N[1]);
    std::vector<Cfg> shapes = {{64, 1, 1, 0},  {128, 1, 1, 0}, {256, 1, 1, 0}, {512, 1, 1, 0},
                               {128, 2, 1, 0}, {256, 2, 1, 0}, {128, 1, 0, 0}, {256, 1, 0, 0}};
    if (ensemble_pair_packs(e, plane)) {
      // the largest plane's wavefronts, and up to twice as many
      shapes.clear();
      const int w = (plane + 63) / 64, most = u1d::pair_max_block((int)elem_size(e->prec), 1) / 64;
      for (int k = w; k <= std::min(2 * w, most); k += std::max(1, w / 4)) shapes.push_back({64 * k, 1, 1, 0});
      shapes.push_back({64 * w, 1, 0, 0});
    }
    for (const Cfg& pc : shapes) {
      RET(ensemble_build_pair(e, pc));
      float t = 1e30f;
      RET(timed(&t));
      if (t < tp) {
        tp = t;
        bestp = pc;
      }
    }
    const bool use = G.pair == 2 || tp < tnone;
    if (G.verbosity >= 1)
      std::fprintf(stderr, "tune ensemble (%d replicas): fused pairs %.1f us per sweep (block %d, %d site(s)/thread) "
                   "vs %.1f us without: %s\n", e->nrep, 1e3 * tp, bestp.block, bestp.spt, 1e3 * tnone,
                   use ? "fused" : "separate");
    RET(ensemble_build_pair(e, use ? bestp : none));
    if (use) best = tp;
    // walks of each class: shapes of a power of two segments per diagonal (the
    // others have more uneven ends or fit few extents) that all replicas
    // take, against none, over a pass of the class (over whole sweeps, creating
    // an ensemble of 64 replicas took 361 ms in binary64, 315 without walks)
    for (const int kind : {u1d::KIND_METROPOLIS, u1d::KIND_OVERRELAX}) {
      const bool metro = kind == u1d::KIND_METROPOLIS;
      if ((metro ? metrop : ovrn) == 0) continue;
      auto timed_pass = [&](float* t) { return timed_passes(metro ? 1 : 0, metro ? 0 : 1, t); };
      float tw = 1e30f;
      Cfg bestw = none;
      for (const Cfg& wc : walk_shapes(e->upd_host[0], e->prec)) {
        const int segs = wc.block / 64 * wc.spt;
        if (segs < 2 || (segs & (segs - 1)) != 0) continue;
        RET(ensemble_build_walk(e, kind, wc));
        if (e->walk[kind].cfg.block == 0) continue;
        float t = 1e30f;
        RET(timed_pass(&t));
        if (G.verbosity >= 2)
          std::fprintf(stderr, "tune ensemble, %s: %d wavefronts of %d segment(s): %.1f us per pass\n",
                       metro ? "Metropolis" : "OverRelaxation", wc.block / 64, wc.spt, 1e3 * t);
        if (t < tw) {
          tw = t;
          bestw = wc;
        }
      }
      if (bestw.block == 0) continue;
      // both sides afresh, alternating
      float tsep = 1e30f;
      tw = 1e30f;
      for (int round = 0; round < 3; ++round) {
        RET(ensemble_build_walk(e, kind, none));
        RET(timed_pass(&tsep));
        RET(ensemble_build_walk(e, kind, bestw));
        RET(timed_pass(&tw));
      }
      const bool usew = G.pair == 2 || tw < tsep;
      if (G.verbosity >= 1)
        std::fprintf(stderr, "tune ensemble (%d replicas), %s: walks %.1f us per pass (%d wavefronts of %d segment(s)) "
                     "vs %.1f us without: %s\n", e->nrep,
                     metro ? "Metropolis" : "OverRelaxation", 1e3 * tw, bestw.block / 64,
                     bestw.spt, 1e3 * tsep, usew ? "walks" : "separate");
      if (!usew) RET(ensemble_build_walk(e, kind, none));
    }
  }
  e->tuned = true;
  return U1_OK;
}

void ensemble_release(u1_ensemble* e) {
  if (e->exec) (void)hipGraphExecDestroy(e->exec);
  if (e->graph) (void)hipGraphDestroy(e->graph);
  if (e->mexec) (void)hipGraphExecDestroy(e->mexec);
  if (e->mgraph) (void)hipGraphDestroy(e->mgraph);
  if (e->mrows) (void)hipFree(e->mrows);
  if (e->mspans) (void)hipFree(e->mspans);
  if (e->series_dev) (void)hipFree(e->series_dev);
  if (e->base_dev) (void)hipFree(e->base_dev);
  if (e->upd_dev) (void)hipFree(e->upd_dev);
  if (e->meas_dev) (void)hipFree(e->meas_dev);
  if (e->upd_map) (void)hipFree(e->upd_map);
  if (e->pair_dev) (void)hipFree(e->pair_dev);
  if (e->pair_map) (void)hipFree(e->pair_map);
  if (e->pair_packed) (void)hipFree(e->pair_packed);
  for (EnsembleWalk& w : e->walk) ensemble_drop_walk(w);
  if (e->meas_map) (void)hipFree(e->meas_map);
  if (e->lat) (void)hipFree(e->lat);
  if (e->sweep_dev) (void)hipFree(e->sweep_dev);
  if (e->res_dev) (void)hipFree(e->res_dev);
  if (e->partials) (void)hipFree(e->partials);
}

// The measuring sweep graph (once per ensemble): phases with the plaquette
// summed in the last pass, the per-replica fold into the series row of the
// sweep, sweep index + 1.
int ensemble_build_mgraph(u1_ensemble* e) {
  if (e->mexec) return U1_OK;
  // (rebuilt by an attempt after a failed capture: the shapes may have changed)
  if (e->mrows) HIPCHK(hipFree(e->mrows));
  e->mrows = nullptr;
  if (e->mspans) HIPCHK(hipFree(e->mspans));
  e->mspans = nullptr;
  std::vector<u1d::RowSpan> spans;
  const int nrows = ensemble_meas_rows(e, &spans);
  e->mlaunches = (int)(spans.size() / (size_t)e->nrep);
  HIPCHK(hipMalloc((void**)&e->mrows, 4 * (size_t)nrows * sizeof(double)));
  HIPCHK(hipMalloc((void**)&e->mspans, spans.size() * sizeof(spans[0])));
  HIPCHK(hipMemcpyAsync(e->mspans, spans.data(), spans.size() * sizeof(spans[0]), hipMemcpyHostToDevice, G.st));
  HIPCHK(hipStreamSynchronize(G.st));
  if (!e->series_dev)
    HIPCHK(hipMalloc((void**)&e->series_dev, (size_t)kEnsSeriesCap * e->nrep * 4 * sizeof(double)));
  if (!e->base_dev) HIPCHK(hipMalloc((void**)&e->base_dev, sizeof(uint32_t)));
  HIPCHK(hipStreamBeginCapture(G.st, hipStreamCaptureModeThreadLocal));
  int rc = ensemble_enqueue_phases(e, e->lat, e->mrows);
  if (rc == U1_OK) {
    hipError_t f = u1d::launch_ensemble_plaquette_fold(e->mrows, e->mlaunches, e->mspans, e->upd_dev, e->nrep,
                                                       e->sweep_dev, e->base_dev, kEnsSeriesCap, e->series_dev, G.st);
    if (f == hipSuccess) f = u1d::launch_increment(e->sweep_dev, G.st);
    if (f != hipSuccess) rc = fail(U1_ERR_HIP, std::string("ensemble capture: ") + hipGetErrorString(f));
  }
  hipGraph_t gr = nullptr;
  const hipError_t ce = hipStreamEndCapture(G.st, &gr);
  if (rc != U1_OK) {
    if (gr) (void)hipGraphDestroy(gr);
    return rc;
  }
  HIPCHK(ce);
  e->mgraph = gr;
  HIPCHK(hipGraphInstantiate(&e->mexec, e->mgraph, nullptr, nullptr, 0));
  return U1_OK;
}

// nsweeps replays of the measuring graph, the series copied to the host in
// chunks of kEnsSeriesCap sweeps.  done_ev (optional) is recorded on the
// library stream after the last sweep's work, before the last chunk's copy.
int ensemble_measured_sweeps(u1_ensemble* e, int32_t nsweeps, double* series, hipEvent_t done_ev = nullptr) {
  for (int32_t done = 0; done < nsweeps;) {
    const int32_t n = std::min<int32_t>(kEnsSeriesCap, nsweeps - done);
    HIPCHK(hipMemcpyAsync(e->base_dev, e->sweep_dev, sizeof(uint32_t), hipMemcpyDeviceToDevice, G.st));
    for (int32_t s = 0; s < n; ++s) HIPCHK(hipGraphLaunch(e->mexec, G.st));
    if (done_ev && done + n == nsweeps) HIPCHK(hipEventRecord(done_ev, G.st));
    HIPCHK(hipMemcpyAsync(series + 4 * (size_t)e->nrep * done, e->series_dev, 4 * (size_t)e->nrep * n * sizeof(double),
                          hipMemcpyDeviceToHost, G.st));
    HIPCHK(hipStreamSynchronize(G.st));
    done += n;
    e->sweeps_done += (uint64_t)n;
  }
  return U1_OK;
}

// Launch classes of a sweep, for kernel timing.
enum LaunchClass {
  LC_METRO = 0,
  LC_OR,
  LC_OR_MEAS,
  LC_METRO_PAIR,
  LC_OR_PAIR,
  LC_OR_PAIR_MEAS,
  LC_METRO_CHAIN,   // fused parity passes (single lattices only)
  LC_OR_CHAIN,
  LC_OR_CHAIN_MEAS,
  LC_COUNT
};
constexpr int kTimingLaunches = 32;  // back-to-back launches per class

// Kernel timing of the ensemble's launch classes (shapes settled, ovrn >= 1):
// on a scratch copy of the packed lattice, kTimingLaunches back-to-back
// launches of each class over all replicas, in the sweep's launch tables, with
// (parity, mu) cycling over the phases the class covers in a pass.  ms[c]:
// mean launch duration; per_sweep[c]: launches per measuring sweep (the last
// overrelaxation pass measures in its parity-1 launches of mu >= 1; a measuring
// pair that is not packed runs as two phases).
int time_ensemble_classes(u1_ensemble* e, double* ms, double* per_sweep) {
  const size_t bytes = (size_t)e->total_links * elem_size(e->prec);
  std::vector<u1d::RowSpan> spans;
  const int nrows = ensemble_meas_rows(e, &spans);
  DevBuf scratch, rows;
  HIPCHK(scratch.alloc(bytes));
  HIPCHK(rows.alloc(4 * (size_t)nrows * sizeof(double)));
  HIPCHK(hipMemcpyAsync(scratch.p, e->lat, bytes, hipMemcpyDeviceToDevice, G.st));
  EventSet es;
  hipEvent_t e0, e1;
  HIPCHK(es.create(&e0));
  HIPCHK(es.create(&e1));
  PhaseArgs a{};
  a.reps = e->upd_dev;
  a.blockmap = e->upd_map;
  a.proposal = e->m.proposal;
  a.nhit = e->m.nhit;
  a.step = e->m.step;
  a.stream = u1r::STREAM_UPDATE;
  a.sweep = (uint32_t)e->sweeps_done;
  a.xcd = (uint32_t)e->cfg.xcd;
  // launches of a class in a sweep: (parity, first mu), with repetitions
  struct Launch {
    int parity, mu;
  };
  std::vector<Launch> list[LC_COUNT];
  auto add_pass = [&](int kind, bool measured) {
    for (int parity = 0; parity < 2; ++parity) {
      const bool measure = measured && parity == 1;
      const bool pair = e->pcfg.block != 0 && (!measure || e->pair_packed), walk = e->walk[kind].cfg.block != 0;
      for (int mu = 0; mu < 4; ++mu) {
        const bool fused = mu < 2 ? pair : walk;
        if (fused && mu % 2 == 1) continue;
        const int c = kind == u1d::KIND_METROPOLIS ? (fused ? LC_METRO_PAIR : LC_METRO)
                      : fused                      ? (measure ? LC_OR_PAIR_MEAS : LC_OR_PAIR)
                                                   : (measure && mu > 0 ? LC_OR_MEAS : LC_OR);
        list[c].push_back({parity, mu});
      }
    }
  };
  for (int p = 0; p < e->metrop; ++p) add_pass(u1d::KIND_METROPOLIS, false);
  for (int o = 0; o < e->ovrn; ++o) add_pass(u1d::KIND_OVERRELAX, o == e->ovrn - 1);
  for (int c = 0; c < LC_COUNT; ++c) {
    ms[c] = 0.0;
    per_sweep[c] = (double)list[c].size();
    if (list[c].empty()) continue;
    const int kind = (c == LC_METRO || c == LC_METRO_PAIR) ? u1d::KIND_METROPOLIS : u1d::KIND_OVERRELAX;
    const bool fused = c == LC_METRO_PAIR || c == LC_OR_PAIR || c == LC_OR_PAIR_MEAS;
    const bool meas = c == LC_OR_MEAS || c == LC_OR_PAIR_MEAS;
    PhaseArgs b = a;
    auto launch = [&](int i) -> int {
      const int mu = list[c][(size_t)i % list[c].size()].mu;
      b.parity = list[c][(size_t)i % list[c].size()].parity;
      b.pass = (uint32_t)(i / (int)list[c].size());
      b.meas = meas ? rows.as<double>() + 4 * (size_t)e->mfirst[std::max(mu, 1)] : nullptr;
      if (fused && mu == 0) return ensemble_launch_pair(e, kind, scratch.p, b);
      if (fused) return ensemble_launch_walk(e, kind, scratch.p, b);
      HIPCHK(u1d::launch_phase(e->prec, kind, mu, scratch.p, b, e->upd_blocks, e->cfg.block, e->cfg.spt, G.st));
      return U1_OK;
    };
    RET(launch(0));  // warm-up
    HIPCHK(hipEventRecord(e0, G.st));
    for (int i = 0; i < kTimingLaunches; ++i) RET(launch(i));
    HIPCHK(hipEventRecord(e1, G.st));
    HIPCHK(hipEventSynchronize(e1));
    float t = 0;
    HIPCHK(hipEventElapsedTime(&t, e0, e1));
    ms[c] = t / kTimingLaunches;
  }
  return U1_OK;
}

}  // namespace

extern "C" {

// ---------------------------------------------------------------- runtime
// Start (cuda_error_check.cpp:24-45): select the device, create the stream.
int u1_init(int device) {
  if (G.init) return U1_OK;
  int n = 0;
  HIPCHK(hipGetDeviceCount(&n));
  if (n == 0) return fail(U1_ERR_HIP, "no HIP device available");
  if (device < 0 || device >= n) return fail(U1_ERR_ARG, "GPU id out of range");
  HIPCHK(hipSetDevice(device));
  // non-blocking: no implicit synchronisation with the legacy default
  // stream, so default-stream work of other code in the process (another
  // thread, a profiler, a framework) neither waits on the library's launches
  // nor lands inside one of its stream captures
  HIPCHK(hipStreamCreateWithFlags(&G.st, hipStreamNonBlocking));
  HIPCHK(hipMalloc((void**)&G.counter, sizeof(unsigned long long)));
  HIPCHK(hipHostMalloc((void**)&G.dres, 64 * sizeof(double), hipHostMallocMapped));
  HIPCHK(hipHostGetDevicePointer((void**)&G.dres_dev, G.dres, 0));
  if (device < kMaxDevices && !g_scratch_dev[device]) {
    void* p = nullptr;
    HIPCHK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_scratch_dev[device] = (double*)p;
  }
  G.device = device;
  G.init = true;
  return U1_OK;
}

// Finalize (cuda_error_check.cpp:47-72) without the exit(): sync and release.
int u1_finalize(void) {
  if (!G.init) return U1_OK;
  HIPCHK(hipStreamSynchronize(G.st));
  if (G.partials) HIPCHK(hipFree(G.partials));
  if (G.work) HIPCHK(hipFree(G.work));
  G.work = nullptr;
  G.work_cap = 0;
  if (G.ml) HIPCHK(hipFree(G.ml));
  G.ml = nullptr;
  G.ml_cap = 0;
  if (G.counter) HIPCHK(hipFree(G.counter));
  if (G.dres) HIPCHK(hipHostFree(G.dres));
  for (auto& kv : G.chain_sched) HIPCHK(hipFree(kv.second));
  G.chain_sched.clear();
  G.chain_sched_len.clear();
  if (G.chain_cnt) HIPCHK(hipFree(G.chain_cnt));
  if (G.chain_err) HIPCHK(hipHostFree(G.chain_err));
  if (G.die_ctl) HIPCHK(hipFree(G.die_ctl));
  G.die_ctl = nullptr;
  G.chain_cnt = nullptr;
  G.chain_cnt_cap = 0;
  G.chain_err = nullptr;
  G.chain_nz = G.chain_nt = G.chain_per = 0;
  HIPCHK(hipStreamDestroy(G.st));
  G.partials = nullptr;
  G.partials_cap = 0;
  G.counter = nullptr;
  G.dres = G.dres_dev = nullptr;
  G.st = nullptr;
  G.init = false;
  return U1_OK;
}

int u1_sync(void) {
  REQ_INIT();
  HIPCHK(hipStreamSynchronize(G.st));
  return chain_check();
}

const char* u1_last_error(void) { return g_err.c_str(); }

int u1_device_name(char* buf, size_t len) {
  REQ_INIT();
  hipDeviceProp_t p;
  HIPCHK(hipGetDeviceProperties(&p, G.device));
  std::snprintf(buf, len, "%s (%s, %d CUs)", p.name, p.gcnArchName, p.multiProcessorCount);
  return U1_OK;
}

// ---------------------------------------------------------------- memory
int u1_malloc(void** ptr, size_t bytes) {
  REQ_INIT();
  if (!ptr) return fail(U1_ERR_ARG, "null pointer");
  *ptr = nullptr;
  HIPCHK(hipMalloc(ptr, bytes ? bytes : 4));
  HIPCHK(u1d::launch_fill_zero(*ptr, (int64_t)((bytes + 3) / 4 * 4), G.st));
  HIPCHK(hipStreamSynchronize(G.st));
  return U1_OK;
}

int u1_free(void* ptr) {
  REQ_INIT();
  if (!ptr) return U1_OK;
  HIPCHK(hipStreamSynchronize(G.st));
  HIPCHK(hipFree(ptr));
  return U1_OK;
}

int u1_memcpy(void* dst, const void* src, size_t bytes, int kind) {
  REQ_INIT();
  if ((!dst || !src) && bytes) return fail(U1_ERR_ARG, "null pointer");
  static const hipMemcpyKind kinds[4] = {hipMemcpyHostToHost, hipMemcpyHostToDevice, hipMemcpyDeviceToHost,
                                         hipMemcpyDeviceToDevice};
  if (kind < 0 || kind > 3) return fail(U1_ERR_ARG, "bad copy kind");
  HIPCHK(hipMemcpyAsync(dst, src, bytes, kinds[kind], G.st));
  HIPCHK(hipStreamSynchronize(G.st));
  return U1_OK;
}

int u1_zero(void* ptr, size_t bytes) {
  REQ_INIT();
  if (bytes) REQ_PTR(ptr);
  if (bytes % 4) return fail(U1_ERR_ARG, "u1_zero needs a multiple of 4 bytes");
  HIPCHK(u1d::launch_fill_zero(ptr, (int64_t)bytes, G.st));
  return U1_OK;
}

int u1_convert_precision(const void* src, int src_prec, void* dst, int dst_prec, int64_t n) {
  REQ_INIT();
  if (n < 0) return fail(U1_ERR_ARG, "negative element count");
  if (n) REQ_PTR(src);
  if (n) REQ_PTR(dst);
  RET(check_prec(src_prec));
  RET(check_prec(dst_prec));
  HIPCHK(u1d::launch_convert_precision(src, src_prec, dst, dst_prec, n, 256, G.st));
  return U1_OK;
}

// ---------------------------------------------------------------- updates
int u1_hotstart(const u1_geom* g, int prec, void* lat, uint64_t seed, uint32_t replica) {
  REQ_INIT();
  REQ_PTR(lat);
  RET(check_geom(g));
  RET(check_prec(prec));
  const RepDesc r = make_rep(g, seed, replica);
  HIPCHK(u1d::launch_hotstart(prec, lat, r, 256, G.st));
  return U1_OK;
}

int u1_update(const u1_geom* g, int prec, void* lat, int32_t metrop, int32_t ovrn, const u1_metro* m,
              uint64_t seed, uint32_t stream, uint32_t sweep, uint32_t c3, int32_t mask_ml, uint64_t* accepts) {
  REQ_INIT();
  RET(check_geom(g));
  RET(check_prec(prec));
  RET(check_metro(m));
  if (!lat) return fail(U1_ERR_ARG, "null lattice");
  if (metrop < 0 || ovrn < 0 || metrop > kMaxMetrop) return fail(U1_ERR_ARG, "bad pass counts");
  if (mask_ml != 0 && mask_ml != 2 && mask_ml != 4) return fail(U1_ERR_ARG, "mask_ml must be 0, 2 or 4");
  if (accepts) HIPCHK(u1d::launch_fill_zero(G.counter, sizeof(unsigned long long), G.st));
  RET(run_update(g, prec, lat, metrop, ovrn, m, seed, stream, sweep, c3, mask_ml, accepts ? G.counter : nullptr));
  if (accepts) {
    unsigned long long v = 0;
    HIPCHK(hipMemcpyAsync(&v, G.counter, sizeof(v), hipMemcpyDeviceToHost, G.st));
    HIPCHK(hipStreamSynchronize(G.st));
    RET(chain_check());
    *accepts += v;
  }
  return U1_OK;
}

int u1_update_plaquette(const u1_geom* g, int prec, void* lat, int32_t metrop, int32_t ovrn, const u1_metro* m,
                        uint64_t seed, uint32_t stream, uint32_t sweep, uint32_t c3, double out[4]) {
  REQ_INIT();
  RET(check_geom(g));
  RET(check_prec(prec));
  RET(check_metro(m));
  if (!lat || !out) return fail(U1_ERR_ARG, "null argument");
  if (metrop < 0 || ovrn < 0 || metrop > kMaxMetrop || metrop + ovrn == 0) return fail(U1_ERR_ARG, "bad pass counts");
  RET(run_update(g, prec, lat, metrop, ovrn, m, seed, stream, sweep, c3, 0, nullptr, G.dres_dev));
  return take_results(out, 4);
}

int u1_phase(const u1_geom* g, int prec, void* lat, int32_t kind, int32_t parity, int32_t mu, const u1_metro* m,
             uint64_t seed, uint32_t stream, uint32_t sweep, uint32_t pass, uint32_t c3, int32_t mask_ml) {
  REQ_INIT();
  RET(check_geom(g));
  RET(check_prec(prec));
  RET(check_metro(m));
  if (!lat) return fail(U1_ERR_ARG, "null lattice");
  if (kind != 0 && kind != 1) return fail(U1_ERR_ARG, "kind must be 0 (Metropolis) or 1 (overrelaxation)");
  if (parity < 0 || parity > 1 || mu < 0 || mu > 3) return fail(U1_ERR_ARG, "bad parity or direction");
  if (mask_ml != 0 && mask_ml != 2 && mask_ml != 4) return fail(U1_ERR_ARG, "mask_ml must be 0, 2 or 4");
  PhaseArgs a{};
  a.single = make_rep(g, seed, c3);
  a.ml = mask_ml;
  a.proposal = m->proposal;
  a.nhit = m->nhit;
  a.step = m->step;
  a.stream = stream;
  a.sweep = sweep;
  a.pass = pass;
  a.parity = parity;
  Cfg c = kDefaultCfg;
  RET(phase_cfg(prec, kind, g, lat, a, &c));
  set_update_blocks(a.single, c);
  a.xcd = (uint32_t)c.xcd;
  HIPCHK(u1d::launch_phase(prec, kind, mu, lat, a, a.single.nblk, c.block, c.spt, G.st));
  return U1_OK;
}

// ---------------------------------------------------------------- measurements
int u1_plaquette(const u1_geom* g, int prec, const void* lat, double out[4]) {
  REQ_INIT();
  REQ_PTR(lat);
  REQ_PTR(out);
  RET(check_geom(g));
  RET(check_prec(prec));
  RET(plaquette_async(g, prec, lat, G.dres_dev));
  return take_results(out, 4);
}

int u1_plaquette_noalloc(const u1_geom* g, int prec, const void* lat, double* out_dev) {
  REQ_INIT();
  REQ_PTR(lat);
  REQ_PTR(out_dev);
  RET(check_geom(g));
  RET(check_prec(prec));
  double* rows = G.device < kMaxDevices ? g_scratch_dev[G.device] : nullptr;
  if (!rows) return fail(U1_ERR_STATE, "no-alloc scratch is not available on this device");
  RepDesc r = make_rep(g, 0, 0);
  int block, spt;
  plaquette_shape(r, prec, &block, &spt);
  set_blocks(r, block * spt);
  r.nblk *= 2;  // even sites, then odd sites
  const int nblk = r.nblk;
  // rows, and a fold row for each 512 of them (more than the fold takes)
  const size_t need = 4 * ((size_t)nblk + ((size_t)nblk + 511) / 512);
  if (need > kNoAllocScratchDoubles)
    return fail(U1_ERR_ARG, "lattice too large for u1_plaquette_noalloc: needs " + std::to_string(need) +
                                " scratch doubles, the maximum is " + std::to_string(kNoAllocScratchDoubles));
  // every row and every fold row is written before it is read: nothing to clear
  HIPCHK(u1d::launch_plaquette(prec, lat, r, rows, nblk, block, spt, G.st));
  HIPCHK(u1d::launch_finish_sums(rows, nblk, 4, 1.0 / (3.0 * (double)r.V), out_dev, rows + 4 * (size_t)nblk, G.st));
  return U1_OK;
}

int u1_polyakov(const u1_geom* g, int prec, const void* lat, double out[2]) {
  REQ_INIT();
  REQ_PTR(lat);
  REQ_PTR(out);
  RET(check_geom(g));
  RET(check_prec(prec));
  const RepDesc r = make_rep(g, 0, 0);
  const int block = 256, nblk = (r.SV + block - 1) / block;
  RET(ensure_fold(nblk, 2));
  HIPCHK(u1d::launch_polyakov(prec, lat, r, G.partials, nblk, block, G.st));
  HIPCHK(u1d::launch_finish_sums(G.partials, nblk, 2, 1.0 / (double)r.SV, G.dres_dev, fold_scratch_ptr(nblk, 2), G.st));
  return take_results(out, 2);
}

int u1_poly_volume(const u1_geom* g, int prec, const void* lat, int32_t mode, const u1_metro* mh, uint64_t seed,
                   uint32_t stream, uint32_t c1, uint32_t c3, void* P_dev) {
  REQ_INIT();
  REQ_PTR(lat);
  REQ_PTR(P_dev);
  RET(check_geom(g));
  RET(check_prec(prec));
  if (mode < 0 || mode > 2) return fail(U1_ERR_ARG, "bad Polyakov mode");
  if (mode == U1_POLY_MULTIHIT_STOCHASTIC) RET(check_metro(mh));
  const RepDesc r = make_rep(g, seed, c3);
  RET(ensure_work(poly_field(r, mode)));
  return poly_volume_async(prec, lat, r, mode, mh, stream, c1, c3, (double*)P_dev, G.work);
}

int u1_temporal_links(const u1_geom* g, int prec, const void* lat, int32_t mode, const u1_metro* mh,
                      uint64_t seed, uint32_t stream, uint32_t c1, uint32_t c3, void* out_dev) {
  REQ_INIT();
  REQ_PTR(lat);
  REQ_PTR(out_dev);
  RET(check_geom(g));
  RET(check_prec(prec));
  if (mode < 0 || mode > 2) return fail(U1_ERR_ARG, "bad temporal-link mode");
  if (mode == U1_POLY_MULTIHIT_STOCHASTIC) RET(check_metro(mh));
  const RepDesc r = make_rep(g, seed, c3);
  HIPCHK(u1d::launch_temporal_links(prec, lat, r, mode, mh ? mh->proposal : 0, mh ? mh->nhit : 0,
                                    mh ? mh->step : 0.0, stream, c1, c3, (double*)out_dev, G.st));
  return U1_OK;
}

int u1_pp(const u1_geom* g, const void* P_dev, int32_t rmax, double* out) {
  REQ_INIT();
  REQ_PTR(P_dev);
  REQ_PTR(out);
  RET(check_geom(g));
  if (rmax < 1 || rmax > 32) return fail(U1_ERR_ARG, "rmax must be in [1, 32]");
  const RepDesc r = make_rep(g, 0, 0);
  const int block = 256, nblk = (r.SV + block - 1) / block;
  RET(ensure_fold(nblk, 2 * rmax));
  HIPCHK(u1d::launch_pp((const double*)P_dev, r, rmax, G.partials, nblk, block, G.st));
  HIPCHK(u1d::launch_finish_sums(G.partials, nblk, 2 * rmax, 1.0 / (3.0 * (double)r.SV), G.dres_dev,
                                 fold_scratch_ptr(nblk, 2 * rmax), G.st));
  return take_results(out, 2 * (size_t)rmax);
}

int u1_poly2(const u1_geom* g, int prec, const void* lat, int32_t mode, const u1_metro* mh, uint64_t seed,
             uint32_t c1, uint32_t c3, double* out) {
  REQ_INIT();
  REQ_PTR(lat);
  REQ_PTR(out);
  RET(check_geom(g));
  RET(check_prec(prec));
  if (mode < 0 || mode > 2) return fail(U1_ERR_ARG, "bad Polyakov mode");
  if (mode == U1_POLY_MULTIHIT_STOCHASTIC) RET(check_metro(mh));
  const RepDesc r = make_rep(g, seed, c3);
  // work: P (2 SV doubles), then the temporal links (2 V doubles, poly_field)
  RET(ensure_work(2 * (size_t)r.SV + poly_field(r, mode)));
  double* P = G.work;
  RET(poly_volume_async(prec, lat, r, mode, mh, U1_STREAM_MULTIHIT, c1, c3, P, G.work + 2 * (size_t)r.SV));
  return u1_pp(g, P, g->dims[0] / 2, out);
}

int u1_multilevel(const u1_geom* g, int prec, const void* lat, int32_t n4, int32_t k4, int32_t n2, int32_t k2,
                  int32_t metrop, int32_t ovrn, const u1_metro* m, int32_t mh_mode, const u1_metro* mh,
                  uint64_t seed, uint32_t call_id, double* out, void* ppspace_dev) {
  REQ_INIT();
  REQ_PTR(lat);
  REQ_PTR(out);
  RET(check_geom(g));
  RET(check_prec(prec));
  RET(check_metro(m));
  // multilevel.cu:641-644
  if (g->dims[3] % 4 != 0) return fail(U1_ERR_ARG, "Cannot apply MultiLevel algorithm: Nt is not a multiple of 4");
  if (n4 < 1 || n2 < 1 || k4 < 0 || k2 < 0) return fail(U1_ERR_ARG, "bad multilevel level counts");
  if (mh_mode != U1_POLY_PLAIN && mh_mode != U1_POLY_MULTIHIT && mh_mode != U1_POLY_MULTIHIT_STOCHASTIC)
    return fail(U1_ERR_ARG, "bad multihit mode");
  if (mh_mode == U1_POLY_MULTIHIT_STOCHASTIC) RET(check_metro(mh));
  const RepDesc r = make_rep(g, seed, call_id);
  const int rmax = r.N[0] / 2;
  if (rmax > 32) return fail(U1_ERR_ARG, "Nx/2 must be <= 32");
  const int64_t sz = (int64_t)r.SV * rmax * 3;
  const int64_t nl2 = r.N[3] / 2, nl4 = r.N[3] / 4;
  if (sz * nl2 >= ((int64_t)1 << 31)) return fail(U1_ERR_ARG, "lattice too large for the multilevel T2 tensor");
  const size_t latb = 4 * (size_t)r.V * elem_size(prec);
  // Workspace: the working lattice, the step counter, the two-slice products of
  // as many level-2 steps as fit kMlSlotBytes, the T4 tensor and, if the steps
  // of a level-4 step need more than one chunk of slots, the T2 tensor.
  const size_t slot = 16 * (size_t)r.SV * (size_t)nl2;
  const int slots = (int)std::min<size_t>((size_t)n2, std::max<size_t>(1, kMlSlotBytes / slot));
  const bool chunked = slots < n2;
  auto pad = [](size_t b) { return (b + 255) / 256 * 256; };
  const size_t o_ctr = pad(latb), o_p2 = o_ctr + 256, o_l4 = o_p2 + pad(slot * slots),
               o_l2 = o_l4 + pad(16 * (size_t)sz * nl4), total = o_l2 + (chunked ? pad(16 * (size_t)sz * nl2) : 0);
  RET(ensure_ml(total));
  char* ws = (char*)G.ml;
  void* wl = ws;
  uint32_t* ctr = (uint32_t*)(ws + o_ctr);  // level-2 step counter i * n2 + k, advanced by the device
  double *p2 = (double*)(ws + o_p2), *l4 = (double*)(ws + o_l4), *l2 = chunked ? (double*)(ws + o_l2) : nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  int rc = U1_OK;
  auto cleanup = [&]() {
    (void)hipStreamSynchronize(G.st);
    if (exec) (void)hipGraphExecDestroy(exec);
    if (graph) (void)hipGraphDestroy(graph);
    if (G.ml_cap > kMlKeepBytes) {
      (void)hipFree(G.ml);
      G.ml = nullptr;
      G.ml_cap = 0;
    }
  };
#define MLCHK(expr)                                                                          \
  do {                                                                                       \
    hipError_t e_ = (expr);                                                                  \
    if (e_ != hipSuccess) {                                                                  \
      cleanup();                                                                             \
      return fail(U1_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_));           \
    }                                                                                        \
  } while (0)
  MLCHK(hipMemcpyAsync(wl, lat, latb, hipMemcpyDeviceToDevice, G.st));
  MLCHK(u1d::launch_fill_zero(ctr, 2 * sizeof(uint32_t), G.st));
  const double l2norm = 1.0 / (double)n2, l4norm = 1.0 / (double)n4;
  const int mp = mh ? mh->proposal : 0, mn = mh ? mh->nhit : 0;
  const double ms = mh ? mh->step : 0.0;
  Cfg die{0, 1, 0, 0};
  {  // launch shapes are settled before capture (the tuner allocates and synchronises)
    PhaseArgs a{};
    a.single = r;
    a.nhit = m->nhit;
    a.proposal = m->proposal;
    a.step = m->step;
    rc = settle_update_cfgs(prec, g, wl, a, metrop, ovrn);
    a.ml = 2;
    if (rc == U1_OK && k2 > 0) rc = die_cfg(g, prec, wl, a, metrop, ovrn, m, false, &die);
    if (rc == U1_OK && die.block != 0) rc = die_prepare();
    if (rc != U1_OK) {
      cleanup();
      return rc;
    }
  }
  // One level-2 step -- k2 masked sweeps (Philox sweep index ctr * k2 + l) and
  // the two-slice products of the temporal links (c1 = ctr, then ctr += 1) --
  // captured once and replayed n4 * n2 times (multilevel.cu:680-700 order;
  // sweep and c1 indices equal to ((i n2 + k) k2 + l) and (i n2 + k)), or
  // enqueued eagerly with the same device counter when graphs are off.
  auto level2_step = [&]() -> int {
    for (int l = 0; l < k2; ++l)
      RET(run_update(g, prec, wl, metrop, ovrn, m, seed, u1r::STREAM_ML_L2, (uint32_t)l, call_id, 2, nullptr,
                     nullptr, ctr, (uint32_t)k2));
    HIPCHK(u1d::launch_temporal_pairs(prec, wl, r, mh_mode, mp, mn, ms, u1r::STREAM_ML_MULTIHIT, call_id, p2, ctr,
                                      (uint32_t)n2, (uint32_t)slots, G.st));
    return U1_OK;
  };
  // (nothing to gain from a graph where a sweep is one launch)
  if (G.graphs && die.block == 0) {
    MLCHK(hipStreamBeginCapture(G.st, hipStreamCaptureModeThreadLocal));
    rc = level2_step();
    const hipError_t ce = hipStreamEndCapture(G.st, &graph);
    if (rc != U1_OK) {
      cleanup();
      return rc;
    }
    MLCHK(ce);
    MLCHK(hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0));
  }
  for (int i = 0; i < n4 && rc == U1_OK; ++i) {
    for (int j = 0; j < k4 && rc == U1_OK; ++j)
      rc = run_update(g, prec, wl, metrop, ovrn, m, seed, u1r::STREAM_ML_L4, (uint32_t)(i * k4 + j), call_id, 4,
                      nullptr);
    for (int k = 0; k < n2 && rc == U1_OK; ++k) {
      if (exec)
        MLCHK(hipGraphLaunch(exec, G.st));
      else
        rc = level2_step();
      const bool last = k + 1 == n2;
      if (rc == U1_OK && (last || (k + 1) % slots == 0))
        MLCHK(u1d::launch_ml_accum(p2, k % slots + 1, l2, k >= slots, !last, l4, r, rmax, l2norm, i == 0, G.st));
    }
  }
  if (rc == U1_OK) {
    const int block = 256, nblk = (r.SV + block - 1) / block;
    rc = ensure_fold(nblk, 2 * rmax);
    if (rc == U1_OK) {
      MLCHK(u1d::launch_ml_final(l4, (double*)ppspace_dev, r, rmax, l4norm, G.partials, nblk, block, G.st));
      MLCHK(u1d::launch_finish_sums(G.partials, nblk, 2 * rmax, 1.0 / (3.0 * (double)r.SV), G.dres_dev,
                                    fold_scratch_ptr(nblk, 2 * rmax), G.st));
      rc = take_results(out, 2 * (size_t)rmax);
    }
  }
#undef MLCHK
  cleanup();
  return rc;
}

int u1_convert_layout(const u1_geom* g, int prec, const void* in, void* out, int32_t eo_to_no) {
  REQ_INIT();
  REQ_PTR(in);
  REQ_PTR(out);
  RET(check_geom(g));
  RET(check_prec(prec));
  if (in == out) return fail(U1_ERR_ARG, "in and out must differ");
  const RepDesc r = make_rep(g, 0, 0);
  HIPCHK(u1d::launch_convert_layout(prec, in, out, r, eo_to_no, 256, G.st));
  return U1_OK;
}

int u1_plaquette_fields(const u1_geom* g, int prec, const void* lat, int32_t spacetime, int32_t eo_order,
                        void* field_dev, double means[12]) {
  REQ_INIT();
  REQ_PTR(lat);
  REQ_PTR(field_dev);
  REQ_PTR(means);
  RET(check_geom(g));
  RET(check_prec(prec));
  const RepDesc r = make_rep(g, 0, 0);
  const int size = spacetime ? r.V : r.SV;
  const int block = 256, nblk = std::min((size + block - 1) / block, u1d::kFoldRows);
  RET(ensure_fold(nblk, 12));
  HIPCHK(u1d::launch_plaquette_fields(prec, lat, r, spacetime, eo_order, (double*)field_dev, G.partials, nblk, block,
                                      G.st));
  HIPCHK(u1d::launch_finish_sums(G.partials, nblk, 12, 1.0 / (double)size, G.dres_dev, fold_scratch_ptr(nblk, 12),
                                 G.st));
  return take_results(means, 12);
}

// ---------------------------------------------------------------- checkpoint
namespace {
struct CfgHeader {
  char magic[8];
  uint32_t version;
  int32_t dims[4];
  uint32_t reserved;
  double beta, aniso;
  uint64_t seed, sweep;
};
static_assert(sizeof(CfgHeader) == 64, "config header must be 64 bytes");
}  // namespace

int u1_config_save(const char* path, const u1_geom* g, int prec, const void* lat, uint64_t seed, uint64_t sweep) {
  REQ_INIT();
  RET(check_geom(g));
  RET(check_prec(prec));
  if (!path || !lat) return fail(U1_ERR_ARG, "null argument");
  const RepDesc r = make_rep(g, 0, 0);
  const size_t n = 4 * (size_t)r.V;
  std::vector<double> host(n);
  {
    DevBuf no, d64;
    HIPCHK(no.alloc(n * elem_size(prec)));
    HIPCHK(d64.alloc(n * sizeof(double)));
    HIPCHK(u1d::launch_convert_layout(prec, lat, no.p, r, 1, 256, G.st));
    HIPCHK(u1d::launch_convert_precision(no.p, prec, d64.p, U1_F64, (int64_t)n, 256, G.st));
    HIPCHK(hipMemcpyAsync(host.data(), d64.p, n * sizeof(double), hipMemcpyDeviceToHost, G.st));
    HIPCHK(hipStreamSynchronize(G.st));
  }
  CfgHeader h{};
  std::memcpy(h.magic, "U1AMDCFG", 8);
  h.version = 1;
  for (int i = 0; i < 4; ++i) h.dims[i] = g->dims[i];
  h.beta = g->beta;
  h.aniso = g->aniso;
  h.seed = seed;
  h.sweep = sweep;
  std::ofstream f(path, std::ios::binary);
  if (!f) return fail(U1_ERR_IO, std::string("cannot write ") + path);
  f.write((const char*)&h, sizeof(h));
  f.write((const char*)host.data(), n * sizeof(double));
  return f ? U1_OK : fail(U1_ERR_IO, std::string("write failed: ") + path);
}

int u1_config_load(const char* path, const u1_geom* g, int prec, void* lat, uint64_t* seed, uint64_t* sweep) {
  if (!path || !g) return fail(U1_ERR_ARG, "null argument");
  std::ifstream f(path, std::ios::binary);
  if (!f) return fail(U1_ERR_IO, std::string("cannot open ") + path);
  CfgHeader h{};
  f.read((char*)&h, sizeof(h));
  if (!f || std::memcmp(h.magic, "U1AMDCFG", 8) != 0 || h.version != 1)
    return fail(U1_ERR_IO, std::string("not a configuration file: ") + path);
  for (int i = 0; i < 4; ++i)
    if (h.dims[i] != g->dims[i]) return fail(U1_ERR_ARG, "configuration file geometry differs from the lattice");
  REQ_INIT();
  RET(check_geom(g));
  RET(check_prec(prec));
  if (!lat) return fail(U1_ERR_ARG, "null lattice");
  const RepDesc r = make_rep(g, 0, 0);
  const size_t n = 4 * (size_t)r.V;
  std::vector<double> host(n);
  f.read((char*)host.data(), n * sizeof(double));
  if (!f) return fail(U1_ERR_IO, std::string("truncated configuration file: ") + path);
  {
    DevBuf no, d64;
    HIPCHK(no.alloc(n * elem_size(prec)));
    HIPCHK(d64.alloc(n * sizeof(double)));
    HIPCHK(hipMemcpyAsync(d64.p, host.data(), n * sizeof(double), hipMemcpyHostToDevice, G.st));
    HIPCHK(u1d::launch_convert_precision(d64.p, U1_F64, no.p, prec, (int64_t)n, 256, G.st));
    HIPCHK(u1d::launch_convert_layout(prec, no.p, lat, r, 0, 256, G.st));
    HIPCHK(hipStreamSynchronize(G.st));
  }
  if (seed) *seed = h.seed;
  if (sweep) *sweep = h.sweep;
  return U1_OK;
}

// ---------------------------------------------------------------- ensemble
int u1_ensemble_create(u1_ensemble** out, int32_t nrep, const u1_geom* geoms, const uint64_t* seeds,
                       const int32_t* hot, int prec, int32_t metrop, int32_t ovrn, const u1_metro* m) {
  REQ_INIT();
  if (!out || !geoms || !seeds || nrep < 1 || nrep > 65535) return fail(U1_ERR_ARG, "bad ensemble arguments");
  if (metrop < 0 || ovrn < 0 || metrop > kMaxMetrop || ovrn > 4095) return fail(U1_ERR_ARG, "bad pass counts");
  RET(check_prec(prec));
  RET(check_metro(m));
  *out = nullptr;
  u1_ensemble* e = new u1_ensemble();
  e->nrep = nrep;
  e->prec = prec;
  e->metrop = metrop;
  e->ovrn = ovrn;
  e->m = *m;
  std::vector<uint16_t> mmap;
  int64_t off = 0;
  for (int i = 0; i < nrep; ++i) {
    int rc = check_geom(&geoms[i]);
    if (rc != U1_OK) {
      delete e;
      return rc;
    }
    e->geoms.push_back(geoms[i]);
    RepDesc r = make_rep(&geoms[i], seeds[i], (uint32_t)i);
    r.lat_off = (uint64_t)off;
    off += 4 * (int64_t)r.V;
    RepDesc u = r, q = r;
    set_blocks(q, kEnsBlock * kEnsSpt);
    q.nblk *= 2;  // even sites, then odd sites
    q.blk_begin = e->meas_blocks;
    e->meas_blocks += q.nblk;
    for (int b = 0; b < q.nblk; ++b) mmap.push_back((uint16_t)i);
    e->upd_host.push_back(u);
    e->meas_host.push_back(q);
  }
  e->total_links = off;
  auto bail = [&](const std::string& msg) {
    ensemble_release(e);
    delete e;
    return fail(U1_ERR_HIP, msg);
  };
#define ECHK(expr)                                                                       \
  do {                                                                                   \
    hipError_t e_ = (expr);                                                              \
    if (e_ != hipSuccess) return bail(std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)
  ECHK(hipMalloc(&e->lat, (size_t)off * elem_size(prec)));
  ECHK(u1d::launch_fill_zero(e->lat, off * (int64_t)elem_size(prec), G.st));
  ECHK(hipMalloc((void**)&e->upd_dev, nrep * sizeof(RepDesc)));
  ECHK(hipMalloc((void**)&e->meas_dev, nrep * sizeof(RepDesc)));
  ECHK(hipMalloc((void**)&e->meas_map, mmap.size() * sizeof(uint16_t)));
  ECHK(hipMalloc((void**)&e->sweep_dev, sizeof(uint32_t)));
  ECHK(hipMalloc((void**)&e->res_dev, 4 * (size_t)nrep * sizeof(double)));
  ECHK(hipMalloc((void**)&e->partials, 4 * (size_t)e->meas_blocks * sizeof(double)));
  ECHK(hipMemcpyAsync(e->meas_dev, e->meas_host.data(), nrep * sizeof(RepDesc), hipMemcpyHostToDevice, G.st));
  ECHK(hipMemcpyAsync(e->meas_map, mmap.data(), mmap.size() * sizeof(uint16_t), hipMemcpyHostToDevice, G.st));
  ECHK(u1d::launch_fill_zero(e->sweep_dev, sizeof(uint32_t), G.st));
  if (int rc = ensemble_build_update(e, e->cfg); rc != U1_OK) {
    ensemble_release(e);
    delete e;
    return rc;
  }
  for (int i = 0; i < nrep; ++i)
    if (hot && hot[i]) ECHK(u1d::launch_hotstart(prec, e->lat, e->upd_host[i], 256, G.st));
  ECHK(hipStreamSynchronize(G.st));
#undef ECHK
  *out = e;
  return U1_OK;
}

int u1_ensemble_sweep(u1_ensemble* e, int32_t nsweeps, int32_t use_graph) {
  REQ_INIT();
  if (!e) return fail(U1_ERR_ARG, "null ensemble");
  if (nsweeps < 0) return fail(U1_ERR_ARG, "nsweeps must be >= 0");
  // tuning changes the launch layout, so it only runs before either graph exists
  RET(ensemble_settle(e));
  if (use_graph && !e->exec) {
    HIPCHK(hipStreamBeginCapture(G.st, hipStreamCaptureModeThreadLocal));
    int rc = ensemble_enqueue_sweep(e);
    hipGraph_t gr = nullptr;
    hipError_t ce = hipStreamEndCapture(G.st, &gr);
    if (rc != U1_OK) {
      if (gr) (void)hipGraphDestroy(gr);
      return rc;
    }
    HIPCHK(ce);
    e->graph = gr;
    HIPCHK(hipGraphInstantiate(&e->exec, e->graph, nullptr, nullptr, 0));
  }
  for (int s = 0; s < nsweeps; ++s) {
    if (use_graph)
      HIPCHK(hipGraphLaunch(e->exec, G.st));
    else
      RET(ensemble_enqueue_sweep(e));
  }
  e->sweeps_done += (uint64_t)nsweeps;
  return U1_OK;
}

int u1_ensemble_sweep_plaquette(u1_ensemble* e, int32_t nsweeps, double* series) {
  REQ_INIT();
  if (!e || !series) return fail(U1_ERR_ARG, "null argument");
  if (nsweeps < 0) return fail(U1_ERR_ARG, "nsweeps must be >= 0");
  if (e->metrop + e->ovrn == 0) return fail(U1_ERR_ARG, "no measuring pass");
  if (nsweeps == 0) return U1_OK;
  RET(ensemble_settle(e));
  RET(ensemble_build_mgraph(e));
  return ensemble_measured_sweeps(e, nsweeps, series);
}

int u1_ensemble_bench(u1_ensemble* e, int32_t nsweeps, double* series, double* elapsed_ms, double* kernel_ms) {
  REQ_INIT();
  if (!e || !series || !elapsed_ms) return fail(U1_ERR_ARG, "null argument");
  if (nsweeps < 1) return fail(U1_ERR_ARG, "nsweeps must be >= 1");
  if (e->ovrn < 1) return fail(U1_ERR_ARG, "the ensemble timing needs an overrelaxation pass (ovrn >= 1)");
  RET(ensemble_settle(e));
  RET(ensemble_build_mgraph(e));
  EventSet es;
  hipEvent_t e0, e1;
  HIPCHK(es.create(&e0));
  HIPCHK(es.create(&e1));
  HIPCHK(hipStreamSynchronize(G.st));
  HIPCHK(hipEventRecord(e0, G.st));
  RET(ensemble_measured_sweeps(e, nsweeps, series, e1));
  float ms = 0;
  HIPCHK(hipEventElapsedTime(&ms, e0, e1));
  *elapsed_ms = ms;
  if (kernel_ms) {
    RET(time_ensemble_classes(e, kernel_ms, kernel_ms + LC_COUNT));
    kernel_ms[2 * LC_COUNT] = (double)ms / nsweeps;
    kernel_ms[2 * LC_COUNT + 1] = kTimingLaunches;
  }
  return U1_OK;
}

int u1_ensemble_plaquette(u1_ensemble* e, double* out) {
  REQ_INIT();
  if (!e || !out) return fail(U1_ERR_ARG, "null argument");
  HIPCHK(u1d::launch_plaquette_batched(e->prec, e->lat, e->meas_dev, e->meas_map, e->partials, e->meas_blocks,
                                       kEnsBlock, kEnsSpt, G.st));
  HIPCHK(u1d::launch_batched_finish(e->partials, e->meas_dev, e->nrep, e->res_dev, G.st));
  return copy_back(out, e->res_dev, 4 * (size_t)e->nrep);
}

int u1_ensemble_read(u1_ensemble* e, int32_t r, double* host) {
  REQ_INIT();
  if (!e || !host || r < 0 || r >= e->nrep) return fail(U1_ERR_ARG, "bad replica");
  const RepDesc& d = e->upd_host[r];
  const int64_t n = 4 * (int64_t)d.V;
  if (e->prec == U1_F64) {
    HIPCHK(hipMemcpyAsync(host, (double*)e->lat + d.lat_off, n * sizeof(double), hipMemcpyDeviceToHost, G.st));
  } else {
    std::vector<float> tmp(n);
    HIPCHK(hipMemcpyAsync(tmp.data(), (float*)e->lat + d.lat_off, n * sizeof(float), hipMemcpyDeviceToHost, G.st));
    HIPCHK(hipStreamSynchronize(G.st));
    for (int64_t i = 0; i < n; ++i) host[i] = (double)tmp[i];
  }
  HIPCHK(hipStreamSynchronize(G.st));
  return U1_OK;
}

int u1_ensemble_write(u1_ensemble* e, int32_t r, const double* host) {
  REQ_INIT();
  if (!e || !host || r < 0 || r >= e->nrep) return fail(U1_ERR_ARG, "bad replica");
  const RepDesc& d = e->upd_host[r];
  const int64_t n = 4 * (int64_t)d.V;
  if (e->prec == U1_F64) {
    HIPCHK(hipMemcpyAsync((double*)e->lat + d.lat_off, host, n * sizeof(double), hipMemcpyHostToDevice, G.st));
    HIPCHK(hipStreamSynchronize(G.st));
  } else {
    std::vector<float> tmp(n);
    for (int64_t i = 0; i < n; ++i) tmp[i] = (float)host[i];
    HIPCHK(hipMemcpyAsync((float*)e->lat + d.lat_off, tmp.data(), n * sizeof(float), hipMemcpyHostToDevice, G.st));
    HIPCHK(hipStreamSynchronize(G.st));
  }
  return U1_OK;
}

int u1_ensemble_info(u1_ensemble* e, uint64_t* sweeps_done, int64_t* total_links) {
  if (!e) return fail(U1_ERR_ARG, "null ensemble");
  if (sweeps_done) *sweeps_done = e->sweeps_done;
  if (total_links) *total_links = e->total_links;
  return U1_OK;
}

int u1_ensemble_destroy(u1_ensemble* e) {
  if (!e) return U1_OK;
  if (G.init) (void)hipStreamSynchronize(G.st);
  ensemble_release(e);
  delete e;
  return U1_OK;
}

// ---------------------------------------------------------------- autotuner
int u1_tune_enable(int32_t on) {
  G.tune = on != 0;
  return U1_OK;
}

int u1_set_graph_capture(int32_t on) {
  if (on != 0 && on != 1) return fail(U1_ERR_ARG, "graph capture switch must be 0 or 1");
  G.graphs = on != 0;
  return U1_OK;
}

int u1_set_pair_fusion(int32_t mode) {
  if (mode < 0 || mode > 2) return fail(U1_ERR_ARG, "pair fusion mode must be 0, 1 or 2");
  G.pair = mode;
  return U1_OK;
}

int u1_set_pass_fusion(int32_t mode) {
  if (mode < 0 || mode > 2) return fail(U1_ERR_ARG, "pass fusion mode must be 0, 1 or 2");
  G.chain = mode;
  return U1_OK;
}

int u1_set_verbosity(int32_t level) {
  if (level < 0 || level > 3) return fail(U1_ERR_ARG, "verbosity must be in [0, 3]");
  G.verbosity = level;
  return U1_OK;
}

// tunecache.csv format of the reference (tune.cpp:109-122, 238-295):
//   tunecache <version> <build hash>
//   volume name aux block.x block.y block.z grid.x grid.y grid.z shared_bytes comment
static const char* kTuneVersion = "latticeu1_amd-1";
static const char* kTuneHash = "gpu_arch=gfx950";

int u1_tune_load(const char* path) {
  if (!path) return fail(U1_ERR_ARG, "null path");
  std::ifstream f(path);
  if (!f) return fail(U1_ERR_IO, std::string("cannot open ") + path);
  std::string line, tok, ver, hash;
  if (!std::getline(f, line)) return fail(U1_ERR_IO, "empty tune cache");
  {
    std::istringstream ls(line);
    ls >> tok >> ver >> hash;
    if (tok != "tunecache") return fail(U1_ERR_IO, std::string("Bad format in ") + path);
    if (ver != kTuneVersion || hash != kTuneHash)
      return fail(U1_ERR_IO, std::string("Cache file ") + path + " does not match this build");
  }
  std::getline(f, line);  // column description
  std::vector<std::pair<std::string, Cfg>> parsed;  // applied only if every line is valid
  while (std::getline(f, line)) {
    if (line.empty()) continue;
    std::istringstream ls(line);
    std::string vol, name, aux;
    int bx, by, bz, gx, gy, gz, sh;
    if (!(std::getline(ls, vol, '\t') && std::getline(ls, name, '\t') && std::getline(ls, aux, '\t')))
      return fail(U1_ERR_IO, std::string("Bad format in ") + path);
    if (!(ls >> bx >> by >> bz >> gx >> gy >> gz >> sh)) return fail(U1_ERR_IO, std::string("Bad format in ") + path);
    // only the shapes the tuner itself tries are accepted: the kernels assume
    // whole wavefronts, at most 512 threads and 4 sites per thread (binary32)
    const bool f32 = name.size() > 4 && name.compare(name.size() - 4, 4, "_f32") == 0;
    bool known = false;
    if (name.compare(0, 5, "Sweep") == 0) {  // one-launch sweep: block 0 = launches per phase
      if (by != 1 || !(bx == 0 || (bx >= 64 && bx <= u1d::die_max_block(f32 ? 4 : 8) && bx % 64 == 0)))
        return fail(U1_ERR_IO, std::string("Bad launch shape in ") + path + ": " + line);
      parsed.push_back({vol + "\t" + name, Cfg{bx, 1, 0, 0}});
      continue;
    }
    if (name.find("Chain_") != std::string::npos) {
      // fused pass: block 0 = unfused, block.z = tiles along z, grid.x = schedule margin
      if (!((bx == 0 && by == 1) || ((by == 1 || by == 2) && bx >= 64 && bx <= 512 && bx % 64 == 0 &&
                                     (bz == 1 || bz == 2 || bz == 4 || bz == 8) && gx >= 0 && gx <= kChainMaxMargin)))
        return fail(U1_ERR_IO, std::string("Bad launch shape in ") + path + ": " + line);
      parsed.push_back({vol + "\t" + name, Cfg{bx, by, 1, bz, bx == 0 ? 0 : gx}});
      continue;
    }
    const bool walk = name.find("Walk_") != std::string::npos;
    if (walk)  // block 0 = two launches; block.y segments per wavefront
      known = (bx == 0 && by == 1) || (bx >= 64 && bx <= 64 * u1d::walk_max_waves(f32 ? 4 : 8) && bx % 64 == 0 &&
                                       (by == 1 || by == 2 || by == 4));
    else if (name.find("Pair_") != std::string::npos)  // fused pair: block 0 = two launches
      known = (bx == 0 && by == 1) || pair_shape_ok(f32 ? U1_F32 : U1_F64, Cfg{bx, by, 0, 0});
    else
      for (const Cfg& c : kShapes) known = known || (c.block == bx && c.spt == by);
    if (!known || (by == 4 && !f32 && !walk) || bz < 1 || bz > (walk ? 8 : 4))
      return fail(U1_ERR_IO, std::string("Bad launch shape in ") + path + ": " + line);
    parsed.push_back({vol + "\t" + name, Cfg{bx, by, (bz - 1) & 1, (bz - 1) >> 1}});
  }
  for (const auto& kv : parsed) G.tunecache[kv.first] = kv.second;
  G.tune_loaded = (int)parsed.size();
  return U1_OK;
}

int u1_tune_save(const char* path) {
  if (!path) return fail(U1_ERR_ARG, "null path");
  std::ofstream f(path);
  if (!f) return fail(U1_ERR_IO, std::string("cannot write ") + path);
  f << "tunecache\t" << kTuneVersion << "\t" << kTuneHash << "\n";
  f << "volume\tname\taux\tblock.x\tblock.y\tblock.z\tgrid.x\tgrid.y\tgrid.z\tshared_bytes\tcomment\n";
  for (const auto& kv : G.tunecache) {
    const std::string& key = kv.first;
    const size_t tab = key.find('\t');
    const std::string vol = key.substr(0, tab), name = key.substr(tab + 1);
    const bool chain = name.find("Chain_") != std::string::npos;
    f << vol << "\t" << name << "\tthreads=halfvolume\t" << kv.second.block << "\t" << kv.second.spt << "\t"
      << (chain ? kv.second.tile : 1 + kv.second.xcd + 2 * kv.second.tile) << "\t" << (chain ? kv.second.margin : 0)
      << "\t1\t1\t0\t# block.x = workgroup size, block.y = sites per thread, block.z - 1 = XCD-aware order (1) + "
         "tiled planes (2); Pair: fused (parity, 0) + (parity, 1) launch, block.x 0 = two launches; "
         "Walk: (parity, 2) + (parity, 3) in one launch along their diagonals, block.x 0 = two launches, block.y = "
         "segments per wavefront, block.z - 1 = XCD order (1) + 2 log2 strip groups; Chain: fused "
         "parity pass (phases 0-3) in one launch, block.x 0 = unfused, block.z = tiles along z, grid.x = schedule "
         "margin; Sweep: whole sweep in one launch, block.x 0 = launches per phase\n";
  }
  return f ? U1_OK : fail(U1_ERR_IO, "write failed");
}

int u1_tune_entries(int32_t* n) {
  if (!n) return fail(U1_ERR_ARG, "null pointer");
  *n = (int32_t)G.tunecache.size();
  return U1_OK;
}

// ---------------------------------------------------------------- timing helper

// Kernel timing of the launch classes of a sweep (1 <= metrop + ovrn, shapes
// already settled): on a scratch copy of the lattice, kTimingLaunches
// back-to-back launches of each class in the sweep's shapes (parity and mu
// cycling over the phases the class covers in a pass), bracketed by one event
// pair.  ms[c]: mean launch duration; per_sweep[c]: launches per sweep.
int time_launch_classes(const u1_geom* g, int prec, const void* lat, int metrop, int ovrn, const u1_metro* m,
                        uint64_t seed, uint32_t sweep, bool meas, double* ms, double* per_sweep) {
  PhaseArgs a{};
  a.single = make_rep(g, seed, 0);
  a.proposal = m->proposal;
  a.nhit = m->nhit;
  a.step = m->step;
  a.stream = U1_STREAM_UPDATE;
  a.sweep = sweep;
  Shapes shapes[2];
  const int passes[2] = {metrop, ovrn};
  for (int kind = 0; kind < 2; ++kind)
    if (passes[kind] > 0) RET(kind_shapes(prec, kind, g, lat, a, &shapes[kind]));
  const int64_t bytes = 4 * (int64_t)a.single.V * (int64_t)elem_size(prec);
  DevBuf scratch;
  HIPCHK(scratch.alloc(bytes));
  HIPCHK(hipMemcpyAsync(scratch.p, lat, bytes, hipMemcpyDeviceToDevice, G.st));
  EventSet es;
  hipEvent_t e0, e1;
  HIPCHK(es.create(&e0));
  HIPCHK(es.create(&e1));
  for (int c = 0; c < LC_COUNT; ++c) ms[c] = per_sweep[c] = 0.0;
  // with the plaquette, the last overrelaxation pass measures in its parity-1
  // launches of mu >= 1 (the parity-1 pair, when fused)
  const bool meas_or = meas && ovrn > 0;
  for (int c = 0; c < LC_COUNT; ++c) {
    const bool chain = c >= LC_METRO_CHAIN;
    const bool pair = c >= LC_METRO_PAIR && !chain;
    const int kind = (c == LC_METRO || c == LC_METRO_PAIR || c == LC_METRO_CHAIN) ? u1d::KIND_METROPOLIS
                                                                                  : u1d::KIND_OVERRELAX;
    const bool cmeas = c == LC_OR_MEAS || c == LC_OR_PAIR_MEAS || c == LC_OR_CHAIN_MEAS;
    const Shapes& sh = shapes[kind];
    const bool chained = sh.chain.block != 0;
    if (passes[kind] == 0 || (cmeas && !meas_or) || chain != chained) continue;
    if (chain) {
      // one launch per parity and pass; the parity-1 launch of the last pass measures
      per_sweep[c] = cmeas ? 1.0 : 2.0 * passes[kind] - (meas_or && kind == u1d::KIND_OVERRELAX ? 1 : 0);
      if (cmeas) {
        RepDesc rc = a.single;
        set_chain_blocks(rc, sh.chain);
        RET(ensure_fold(3 * rc.N[2] * rc.N[3] * rc.bpp, 4));
      }
      PhaseArgs b = a;
      auto launch = [&](int i) -> int {
        b.parity = cmeas ? 1 : i & 1;
        b.pass = (uint32_t)(i >> 1);
        b.meas = cmeas ? G.partials : nullptr;
        return chain_launch(prec, kind, scratch.p, b, sh.chain);
      };
      RET(launch(0));  // warm-up
      HIPCHK(hipEventRecord(e0, G.st));
      for (int i = 0; i < kTimingLaunches; ++i) RET(launch(i));
      HIPCHK(hipEventRecord(e1, G.st));
      HIPCHK(hipEventSynchronize(e1));
      RET(chain_check());
      float t = 0;
      HIPCHK(hipEventElapsedTime(&t, e0, e1));
      ms[c] = t / kTimingLaunches;
      continue;
    }
    // the (parity, mu) launches of one pass in this class (a fused pair is
    // listed by its first mu); launches per sweep without and with measurement
    std::vector<std::pair<int, int>> ph;
    int n_meas = 0;
    for (int parity = 0; parity < 2; ++parity)
      for (int mu = 0; mu < 4; ++mu) {
        const bool fused = (mu < 2 ? sh.pair : sh.walk).block != 0;
        if (fused != pair || (fused && mu % 2 != 0)) continue;
        const bool is_meas = parity == 1 && (pair || mu >= 1);
        n_meas += is_meas;
        if (!cmeas || is_meas) ph.push_back({parity, mu});
      }
    if (ph.empty()) continue;
    if (cmeas)
      per_sweep[c] = (double)ph.size();
    else
      per_sweep[c] = (double)ph.size() * passes[kind] - (meas_or && kind == u1d::KIND_OVERRELAX ? n_meas : 0);
    if (cmeas) RET(ensure_fold(parity_row(a.single, sh, 4), 4));
    auto launch = [&](int i) -> int {
      PhaseArgs b = a;
      const int mu = ph[(size_t)i % ph.size()].second;
      b.parity = ph[(size_t)i % ph.size()].first;
      b.pass = (uint32_t)(i / (int)ph.size());
      b.meas = cmeas ? G.partials : nullptr;
      if (pair) return launch_two_phases(prec, kind, scratch.p, b, sh, mu, [&](int) { return b.meas; });
      b.xcd = (uint32_t)sh.phase.xcd;
      set_update_blocks(b.single, sh.phase);
      HIPCHK(u1d::launch_phase(prec, kind, mu, scratch.p, b, b.single.nblk, sh.phase.block, sh.phase.spt, G.st));
      return U1_OK;
    };
    RET(launch(0));  // warm-up
    HIPCHK(hipEventRecord(e0, G.st));
    for (int i = 0; i < kTimingLaunches; ++i) RET(launch(i));
    HIPCHK(hipEventRecord(e1, G.st));
    HIPCHK(hipEventSynchronize(e1));
    float t = 0;
    HIPCHK(hipEventElapsedTime(&t, e0, e1));
    ms[c] = t / kTimingLaunches;
  }
  return U1_OK;
}

int u1_bench_updates(const u1_geom* g, int prec, void* lat, int32_t metrop, int32_t ovrn, const u1_metro* m,
                     uint64_t seed, uint32_t sweep0, int32_t nsweeps, int32_t measure_plaq, double* plaq_series,
                     double* elapsed_ms, double* kernel_ms) {
  REQ_INIT();
  REQ_PTR(lat);
  REQ_PTR(elapsed_ms);
  RET(check_geom(g));
  RET(check_prec(prec));
  RET(check_metro(m));
  if (nsweeps < 1) return fail(U1_ERR_ARG, "nsweeps must be >= 1");
  if (measure_plaq < 0 || measure_plaq > 2) return fail(U1_ERR_ARG, "measure_plaq must be 0, 1 or 2");
  if (measure_plaq == 1 && metrop + ovrn == 0) return fail(U1_ERR_ARG, "no measuring pass");
  DevBuf series_buf;
  if (measure_plaq) HIPCHK(series_buf.alloc(4 * (size_t)nsweeps * sizeof(double)));
  double* series = series_buf.as<double>();
  {  // tune outside the timed region
    PhaseArgs a{};
    a.single = make_rep(g, seed, 0);
    a.nhit = m->nhit;
    a.proposal = m->proposal;
    a.step = m->step;
    RET(settle_update_cfgs(prec, g, lat, a, metrop, ovrn));
  }
  // Timed region: one event pair around the whole region, nothing inside.
  EventSet es;
  hipEvent_t e0, e1;
  HIPCHK(es.create(&e0));
  HIPCHK(es.create(&e1));
  HIPCHK(hipStreamSynchronize(G.st));
  HIPCHK(hipEventRecord(e0, G.st));
  for (int s = 0; s < nsweeps; ++s) {
    // the launch classes of a sweep, which kernel_ms reports, at any size
    RET(run_update(g, prec, lat, metrop, ovrn, m, seed, U1_STREAM_UPDATE, sweep0 + (uint32_t)s, 0, 0, nullptr,
                   measure_plaq == 1 ? series + 4 * s : nullptr, nullptr, 0, false));
    if (measure_plaq == 2) RET(plaquette_async(g, prec, lat, series + 4 * s));
  }
  HIPCHK(hipEventRecord(e1, G.st));
  HIPCHK(hipEventSynchronize(e1));
  RET(chain_check());
  float ms = 0;
  HIPCHK(hipEventElapsedTime(&ms, e0, e1));
  *elapsed_ms = ms;
  if (kernel_ms) {
    RET(time_launch_classes(g, prec, lat, metrop, ovrn, m, seed, sweep0 + (uint32_t)nsweeps, measure_plaq == 1,
                            kernel_ms, kernel_ms + LC_COUNT));
    kernel_ms[2 * LC_COUNT] = (double)ms / nsweeps;
    kernel_ms[2 * LC_COUNT + 1] = kTimingLaunches;
  }
  if (measure_plaq && plaq_series)
    RET(copy_back(plaq_series, series, 4 * (size_t)nsweeps));
  return U1_OK;
}

// ---------------------------------------------------------------- self test
int u1_selftest_math(int32_t fn, const double* x, const double* y, double* out, int64_t n) {
  REQ_INIT();
  if (fn < 0 || fn > 10 || !x || !out || n < 0) return fail(U1_ERR_ARG, "bad self-test arguments");
  if (n == 0) return U1_OK;
  const int nout = (fn == 0 || fn == 3 || fn == 5 || fn == 7) ? 2 : 1;
  DevBuf dx, dy, dout;
  HIPCHK(dx.alloc(n * sizeof(double)));
  HIPCHK(dy.alloc(n * sizeof(double)));
  HIPCHK(dout.alloc(nout * n * sizeof(double)));
  HIPCHK(hipMemcpyAsync(dx.p, x, n * sizeof(double), hipMemcpyHostToDevice, G.st));
  HIPCHK(hipMemcpyAsync(dy.p, y ? y : x, n * sizeof(double), hipMemcpyHostToDevice, G.st));
  HIPCHK(u1d::launch_selftest_math(fn, dx.as<double>(), dy.as<double>(), dout.as<double>(), n, G.st));
  HIPCHK(hipMemcpyAsync(out, dout.p, nout * n * sizeof(double), hipMemcpyDeviceToHost, G.st));
  HIPCHK(hipStreamSynchronize(G.st));
  return U1_OK;
}

int u1_selftest_sweep(const u1_geom* g, int prec, void* lat, int32_t metrop, int32_t ovrn, const u1_metro* m,
                      uint64_t seed, uint32_t sweep, int32_t mask_ml, int32_t block, int32_t flags, uint64_t* accepts,
                      double* plaq) {
  REQ_INIT();
  REQ_PTR(lat);
  RET(check_geom(g));
  RET(check_prec(prec));
  RET(check_metro(m));
  if (metrop < 0 || ovrn < 0 || metrop > kMaxMetrop || metrop + ovrn == 0) return fail(U1_ERR_ARG, "bad pass counts");
  if (mask_ml != 0 && mask_ml != 2 && mask_ml != 4) return fail(U1_ERR_ARG, "mask_ml must be 0, 2 or 4");
  if (flags < 0 || flags > 3 || (plaq && mask_ml != 0)) return fail(U1_ERR_ARG, "bad self-test arguments");
  PhaseArgs a{};
  a.single = make_rep(g, seed, 0);
  a.ml = mask_ml;
  a.proposal = m->proposal;
  a.nhit = m->nhit;
  a.step = m->step;
  a.stream = U1_STREAM_UPDATE;
  a.sweep = sweep;
  if (!die_possible(a.single, mask_ml, metrop, ovrn) || block < 64 || block > u1d::die_max_block((int)elem_size(prec)) || block % 64)
    return fail(U1_ERR_ARG, "not a one-launch sweep");
  if (accepts) HIPCHK(u1d::launch_fill_zero(G.counter, sizeof(unsigned long long), G.st));
  a.accepts = accepts ? G.counter : nullptr;
  RET(die_launch(prec, lat, a, metrop, ovrn, Cfg{block, 1, 0, 0}, plaq ? G.dres_dev : nullptr,
                 flags & 1 ? 0u : u1d::kDiePatience, (flags & 2) != 0));
  unsigned long long v = 0;
  if (accepts) HIPCHK(hipMemcpyAsync(&v, G.counter, sizeof(v), hipMemcpyDeviceToHost, G.st));
  if (plaq) RET(take_results(plaq, 4));
  HIPCHK(hipStreamSynchronize(G.st));
  RET(chain_check());
  if (accepts) *accepts += v;
  return U1_OK;
}

int u1_selftest_stream(int32_t pattern, int64_t n, int32_t reps, double* gbs) {
  REQ_INIT();
  if (pattern < 0 || pattern > 2 || n < 8 || n % 8 != 0 || n > ((int64_t)1 << 30) || reps < 1 || !gbs)
    return fail(U1_ERR_ARG, "bad stream arguments");
  float *a = nullptr, *b = nullptr;
  HIPCHK(hipMalloc((void**)&a, 9 * (size_t)n * sizeof(float)));
  int rc = U1_OK;
  if (hipMalloc((void**)&b, 9 * (size_t)n * sizeof(float)) != hipSuccess) {
    (void)hipFree(a);
    return fail(U1_ERR_HIP, "hipMalloc failed");
  }
  hipEvent_t e0 = nullptr, e1 = nullptr;
  auto run = [&]() -> hipError_t {
    hipError_t e;
    if ((e = u1d::launch_fill_zero(a, 36 * n, G.st)) != hipSuccess) return e;
    if ((e = u1d::launch_stream(pattern, a, b, n, G.st)) != hipSuccess) return e;  // warm-up
    if ((e = hipEventCreate(&e0)) != hipSuccess || (e = hipEventCreate(&e1)) != hipSuccess) return e;
    if ((e = hipEventRecord(e0, G.st)) != hipSuccess) return e;
    for (int i = 0; i < reps; ++i)
      if ((e = u1d::launch_stream(pattern, a, b, n, G.st)) != hipSuccess) return e;
    if ((e = hipEventRecord(e1, G.st)) != hipSuccess) return e;
    if ((e = hipEventSynchronize(e1)) != hipSuccess) return e;
    float ms = 0;
    if ((e = hipEventElapsedTime(&ms, e0, e1)) != hipSuccess) return e;
    *gbs = 36.0 * (double)n * reps / (ms * 1e-3) / 1e9;
    return hipSuccess;
  };
  const hipError_t e = run();
  if (e != hipSuccess) rc = fail(U1_ERR_HIP, std::string("stream probe: ") + hipGetErrorString(e));
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  (void)hipStreamSynchronize(G.st);
  (void)hipFree(a);
  (void)hipFree(b);
  return rc;
}

int u1_selftest_philox(const uint32_t* ctr, const uint32_t* key, uint32_t* out, int64_t n) {
  REQ_INIT();
  if (!ctr || !key || !out || n < 0) return fail(U1_ERR_ARG, "bad self-test arguments");
  if (n == 0) return U1_OK;
  DevBuf dc, dk, dout;
  HIPCHK(dc.alloc(4 * n * sizeof(uint32_t)));
  HIPCHK(dk.alloc(2 * n * sizeof(uint32_t)));
  HIPCHK(dout.alloc(4 * n * sizeof(uint32_t)));
  HIPCHK(hipMemcpyAsync(dc.p, ctr, 4 * n * sizeof(uint32_t), hipMemcpyHostToDevice, G.st));
  HIPCHK(hipMemcpyAsync(dk.p, key, 2 * n * sizeof(uint32_t), hipMemcpyHostToDevice, G.st));
  HIPCHK(u1d::launch_selftest_philox(dc.as<uint32_t>(), dk.as<uint32_t>(), dout.as<uint32_t>(), n, G.st));
  HIPCHK(hipMemcpyAsync(out, dout.p, 4 * n * sizeof(uint32_t), hipMemcpyDeviceToHost, G.st));
  HIPCHK(hipStreamSynchronize(G.st));
  return U1_OK;
}

}  // extern "C"
