// CPU check of the control words of one-launch sweeps (u1_die_sync.h), on the
// kernel's own code: workgroups as fibers, every access a scheduling point, and
// every store and addition completed at a random later moment, in any order
// that the workgroup's drain() calls allow.  Launches follow each other on the
// same words.  At every barrier a workgroup must find what the others stored in
// the phase before, and after a launch every word must be zero again.  In some
// launches only a few of the workgroups can be resident at a time: the sweep must
// get done all the same, by one of them.
#include <ucontext.h>

#include <cstdio>
#include <cstdlib>
#include <memory>
#include <random>
#include <vector>

#include "../../latticeu1_amd/csrc/u1_die_sync.h"

using namespace u1d;

namespace {

std::mt19937 rng;
uint32_t pick(uint32_t n) { return (uint32_t)(rng() % n); }

struct Fiber {
  ucontext_t ctx;
  std::vector<char> stack;
  bool started = false, done = false;
};
struct Op {
  int fiber;
  enum { ADD, CAS, STORE, DATA } kind;
  int word;
  uint32_t v;
  uint32_t want;  // CAS
  uint32_t* got;  // where the old value goes; null: nobody waits for it
  bool* landed;
};

uint32_t ctl[DIE_CTL];
std::vector<uint32_t> slot;  // one per workgroup: phases it has stored
std::vector<Op> flying;
std::vector<std::unique_ptr<Fiber>> fibers;
ucontext_t scheduler;
int current, errors, timeouts;
bool spread;   // workgroups on two XCDs
bool patient;  // waits for the others before a workgroup goes on alone
int shared, alone;  // workgroups that took part: in a shared sweep, by themselves

void yield() { swapcontext(&fibers[current]->ctx, &scheduler); }

void land(size_t i) {
  // an older access of the same workgroup to the same word goes first
  for (size_t j = 0; j < i; ++j)
    if (flying[j].fiber == flying[i].fiber && flying[j].word == flying[i].word &&
        (flying[j].kind == Op::DATA) == (flying[i].kind == Op::DATA))
      i = j;
  const Op o = flying[i];
  flying.erase(flying.begin() + (long)i);
  if (o.kind == Op::DATA) {
    slot[(size_t)o.word] = o.v;
    return;
  }
  uint32_t& w = ctl[o.word];
  if (o.got) *o.got = w;
  if (o.kind == Op::CAS)
    w = w == o.want ? o.v : w;
  else
    w = o.kind == Op::ADD ? w + o.v : o.v;
  if (o.landed) *o.landed = true;
}

struct CpuMem {
  static constexpr uint32_t kSpin = 1u << 20;
  int id;
  bool leader() const { return true; }
  void barrier() const {}
  void pause() const {}
  uint32_t xcd() const { return spread ? (uint32_t)id % 8u : 3u; }
  uint32_t broadcast(uint32_t v) const { return v; }
  uint32_t patience() const { return patient ? 300u : 0u; }
  void fly(int kind, int word, uint32_t v, uint32_t want = 0, uint32_t* got = nullptr, bool* landed = nullptr) const {
    flying.push_back(Op{id, (decltype(Op::kind))kind, word, v, want, got, landed});
    yield();
  }
  uint32_t ask(int kind, int word, uint32_t v, uint32_t want = 0) const {
    uint32_t got = 0;
    bool landed = false;
    fly(kind, word, v, want, &got, &landed);
    while (!landed) yield();
    return got;
  }
  void drain() const {
    for (;;) {
      bool mine = false;
      for (const Op& o : flying) mine = mine || o.fiber == id;
      if (!mine) return;
      yield();
    }
  }
  uint32_t load(int word) const {
    yield();
    return ctl[word];
  }
  void store(int word, uint32_t v) const { fly(Op::STORE, word, v); }
  void add(int word, uint32_t v, bool) const { fly(Op::ADD, word, v); }
  uint32_t fetch_add(int word, uint32_t v) const { return ask(Op::ADD, word, v); }
  uint32_t cas(int word, uint32_t want, uint32_t v) const { return ask(Op::CAS, word, v, want); }
  void timed_out() const { ++timeouts; }
};

struct Launch {
  int n, phases;
  bool meas;
  uint32_t base;  // phases of the launches before
} launch;

void workgroup(int id) {
  DieSync<CpuMem> sync{{id}, (uint32_t)launch.n, (uint32_t)id, 0, 0, false, false};
  sync.start();
  sync.started();
  if (sync.n != 0) (sync.n == sync.all ? shared : alone) += 1;
  for (int p = 0; sync.n != 0 && p < launch.phases; ++p) {
    sync.wait();
    for (const uint32_t s : slot)
      if (s < launch.base + (uint32_t)p) ++errors;
    for (int i = 0; i < launch.n; ++i)
      if (i == id || sync.n != sync.all) sync.mem.fly(Op::DATA, i, launch.base + (uint32_t)p + 1);
    sync.arrive();
  }
  if (launch.meas && sync.n != 0) {
    sync.arrive();
    if (sync.wg == 0) {
      sync.wait();
      for (const uint32_t s : slot)
        if (s < launch.base + (uint32_t)launch.phases) ++errors;
    }
  }
  sync.leave();
  fibers[(size_t)id]->done = true;
  swapcontext(&fibers[(size_t)id]->ctx, &scheduler);
}

// One launch, at most `resident` workgroups at a time; false if it never ends.
bool run(const Launch& l, int resident) {
  launch = l;
  fibers.clear();
  for (int i = 0; i < l.n; ++i) fibers.push_back(std::make_unique<Fiber>());
  std::vector<int> in;
  int next = 0, left = l.n;
  shared = alone = 0;
  for (long step = 0; left > 0 || !flying.empty(); ++step) {
    if (step > 40000000) return false;
    while (next < l.n && (int)in.size() < resident) in.push_back(next++);
    // landings rarer than slices, so that accesses stay in flight for a while
    if (!flying.empty() && (in.empty() || pick(4) == 0)) {
      land(pick((uint32_t)flying.size()));
      continue;
    }
    if (in.empty()) continue;
    const size_t k = pick((uint32_t)in.size());
    current = in[k];
    Fiber& f = *fibers[(size_t)current];
    if (!f.started) {
      f.started = true;
      f.stack.resize(1 << 16);
      getcontext(&f.ctx);
      f.ctx.uc_stack.ss_sp = f.stack.data();
      f.ctx.uc_stack.ss_size = f.stack.size();
      f.ctx.uc_link = &scheduler;
      makecontext(&f.ctx, (void (*)())workgroup, 1, current);
    }
    swapcontext(&scheduler, &f.ctx);
    if (f.done) {
      in.erase(in.begin() + (long)k);
      --left;
    }
  }
  return true;
}

}  // namespace

int main() {
  int bad = 0, sweeps[2] = {0, 0};
  for (int seed = 0; seed < 400; ++seed) {
    rng.seed((unsigned)seed);
    const int ns[] = {1, 2, 3, 5, 8, 16};
    const int n = ns[pick(6)];
    spread = pick(2) != 0;
    slot.assign((size_t)n, 0);
    for (uint32_t& w : ctl) w = 0;
    errors = timeouts = 0;
    uint32_t base = 0;
    for (int k = 0; k < 4; ++k) {
      const Launch l = {n, (int)pick(4) + 1, pick(3) == 0, base};
      patient = pick(4) != 0;
      const int resident = pick(2) ? n : 1 + (int)pick((uint32_t)n);
      const bool ends = run(l, resident);
      // all or one (the only one of a launch counts as all)
      const bool fair = alone == 0 ? shared == l.n : alone == 1 && shared == 0;
      ++sweeps[alone];
      bool zero = true;
      for (const uint32_t w : ctl) zero = zero && w == 0;
      base += (uint32_t)l.phases;
      for (const uint32_t s : slot) errors += s != base;
      if (!ends || !zero || !fair || errors || timeouts) {
        std::printf("seed %d launch %d: %d workgroups, %d resident, %d phases%s: ended %d, words cleared %d, %d shared, %d "
                    "alone, stale reads %d, timeouts %d\n",
                    seed, k, l.n, resident, l.phases, l.meas ? ", measured" : "", ends, zero, shared, alone, errors,
                    timeouts);
        ++bad;
        break;
      }
    }
  }
  if (bad) {
    std::printf("%d of 400 sequences failed\n", bad);
    return 1;
  }
  if (sweeps[0] < 100 || sweeps[1] < 100) {
    std::printf("too few sweeps of a kind: %d shared, %d alone\n", sweeps[0], sweeps[1]);
    return 1;
  }
  std::printf("die sync ok: %d sweeps shared, %d alone\n", sweeps[0], sweeps[1]);
  return 0;
}
