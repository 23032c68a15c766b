// u1_die_sync.h -- the control words of a one-launch sweep (k_die in u1_die.hip)
// and the order in which its workgroups touch them.  Mem does the accesses: the
// kernel's are atomics in device memory; tests/cpu_checks/check_die_sync.cpp runs
// this code with accesses that complete late and in any order that drain() does
// not forbid.
//
// Every access is relaxed, and accesses to different words may complete in any
// order.  So a workgroup drains what it has issued wherever another one may act
// on the next word it touches.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace u1d {

// Words of a set of control words, each on a cache line of its own; all zero
// between launches.  DIE_HERE, which a workgroup touches once to begin: from bit 0
// on the workgroups that have begun, from bit 6 on one more than the number of the
// one that goes on alone, if any, from bit 12 on the sum of their XCDs' numbers
// and from bit 20 on of the numbers' squares (all on one XCD if and only if the
// squares' sum times the workgroups is the sum's square).
enum { DIE_HERE = 0, DIE_DONE = 32, DIE_LEFT = 64, DIE_CTL = 96 };
constexpr int kDieGroups = 32;  // workgroups at most
constexpr int kDieXcds = 8;
static_assert(kDieGroups < 1 << 6 && kDieGroups * (kDieXcds - 1) < 1 << 8 &&
                  kDieGroups * (kDieXcds - 1) * (kDieXcds - 1) < 1 << 12,
              "fields of DIE_HERE");

// Progress.  Workgroups may only wait for others that are resident, and other
// work on the card -- a one-launch sweep of another process, whose workgroups
// wait too -- may keep some from becoming so.  So the first wait, before the
// first store, is for all of them to have begun, and one that has waited long
// enough takes the whole sweep for itself: either the last arrival or its mark
// comes first on DIE_HERE, and every workgroup, whenever it begins, reads which.
// Later waits are for workgroups that have begun.
template <typename Mem>
struct DieSync {
  Mem mem;
  uint32_t all;     // workgroups of the launch
  uint32_t wg;      // this one
  uint32_t n;       // workgroups that share the sweep: all, or one
  uint32_t target;  // arrivals that complete the last barrier
  bool one;         // all on one XCD
  bool dead;        // a wait timed out: no more waiting

  __host__ __device__ __forceinline__ void start() {
    if (mem.leader()) {
      const uint32_t x = mem.xcd() % kDieXcds;
      mem.add(DIE_HERE, 1u | x << 12 | x * x << 20, false);
    }
    n = all;
    target = 0;
    one = false;
    dead = false;
  }
  // Before the first store.  n then is all, or 1 if this workgroup goes on alone
  // (as number 0), or 0 if another one does.
  __host__ __device__ __forceinline__ void started() {
    uint32_t v = 0;
    if (mem.leader()) {
      v = mem.load(DIE_HERE);
      for (uint32_t k = 0; (v & 0xfffu) < all; ++k) {
        if (k >= mem.patience()) {
          const uint32_t mark = v | (wg + 1u) << 6, old = mem.cas(DIE_HERE, v, mark);
          v = old == v ? mark : old;
        } else {
          mem.pause();
          v = mem.load(DIE_HERE);
        }
      }
    }
    v = mem.broadcast(v);
    const uint32_t mark = v >> 6 & 0x3fu, sum = v >> 12 & 0xffu;
    one = all * (v >> 20) == sum * sum;
    if (mark) {
      n = mark == wg + 1u ? 1u : 0u;
      wg = 0;
      one = true;
    }
  }
  // this workgroup's stores are visible to the others
  __host__ __device__ __forceinline__ void arrive() {
    mem.drain();
    mem.barrier();
    target += n;
    if (mem.leader()) mem.add(DIE_DONE, 1u, one);
  }
  __host__ __device__ __forceinline__ void wait() {
    if (mem.leader())
      for (uint32_t k = 0; !dead && mem.load(DIE_DONE) < target; ++k) {
        if (k == Mem::kSpin) {
          dead = true;
          mem.timed_out();
        }
        mem.pause();
      }
    mem.barrier();
  }
  // The last workgroup to leave clears the words for the next launch.  Each
  // counts itself only when its last arrival has completed: one still in flight
  // would land on the cleared word, and the next launch's barriers would all
  // open one arrival early.
  __host__ __device__ __forceinline__ void leave() {
    if (!mem.leader()) return;
    mem.drain();
    if (mem.fetch_add(DIE_LEFT, 1u) + 1 != all) return;
    for (int w : {DIE_HERE, DIE_DONE, DIE_LEFT}) mem.store(w, 0u);
  }
};

}  // namespace u1d
