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
// between launches.
enum { DIE_HERE = 0, DIE_XCDS = 32, DIE_DONE = 64, DIE_LEFT = 96, DIE_CTL = 128 };

template <typename Mem>
struct DieSync {
  Mem mem;
  uint32_t n;       // workgroups
  uint32_t target;  // arrivals that complete the last barrier
  bool one;         // all on one XCD
  bool dead;        // a wait timed out: no more waiting

  __host__ __device__ __forceinline__ void until(int word, uint32_t want) {
    if (mem.leader())
      for (uint32_t k = 0; !dead && mem.load(word) < want; ++k) {
        if (k == Mem::kSpin) {
          dead = true;
          mem.timed_out();
        }
        mem.pause();
      }
    mem.barrier();
  }
  __host__ __device__ __forceinline__ void start() {
    if (mem.leader()) {
      mem.set_bits(DIE_XCDS, 1u << mem.xcd());
      mem.drain();
      mem.add(DIE_HERE, 1u, false);
    }
    target = 0;
    one = false;
    dead = false;
  }
  // before the first store
  __host__ __device__ __forceinline__ void started() {
    until(DIE_HERE, n);
    const uint32_t m = mem.uniform(mem.load(DIE_XCDS));
    one = (m & (m - 1)) == 0;
  }
  // this workgroup's stores are visible to the others
  __host__ __device__ __forceinline__ void arrive() {
    mem.drain();
    mem.barrier();
    target += n;
    if (mem.leader()) mem.add(DIE_DONE, 1u, one);
  }
  __host__ __device__ __forceinline__ void wait() { until(DIE_DONE, target); }
  // The last workgroup to leave clears the words for the next launch.  Each
  // counts itself only when its last arrival has completed: one still in flight
  // would land on the cleared word, and the next launch's barriers would all
  // open one arrival early.
  __host__ __device__ __forceinline__ void leave() {
    if (!mem.leader()) return;
    mem.drain();
    if (mem.fetch_add(DIE_LEFT, 1u) + 1 != n) return;
    for (int w : {DIE_HERE, DIE_XCDS, DIE_DONE, DIE_LEFT}) mem.store(w, 0u);
  }
};

}  // namespace u1d
