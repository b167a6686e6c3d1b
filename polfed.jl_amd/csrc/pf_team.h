// Teams: groups of workgroups on one XCD that run many dependent steps in one
// launch.
//
// A multi-step driver with one launch per step pays the launch gap and, at
// every kernel boundary, the write-back and refetch of all vectors through the
// Infinity Fabric, because the eight XCDs share no L2.  The columns of a block
// (and the instances of a batch) never exchange data, so a team instead keeps
// one column on ONE XCD for all steps: its vectors stay in that XCD's L2, in
// LDS and in registers, and a step ends with a barrier among the team's blocks.
//
// Coherence.  Data that another block of the team wrote are stored and loaded
// at agent scope (sc1: the load misses the CU's vector L1), and a wave waits
// for its stores (vmcnt 0) before its block arrives at the barrier.  The L2 is
// shared by all CUs of an XCD, so it is the point where the team's stores and
// loads meet; the team is formed by the hardware's XCC id, never by the block
// index.  Blocks of different teams exchange nothing but job counters (agent
// scope atomics).
//
// Progress.  A block only ever waits for blocks that are already running: the
// members of an XCD check in on a counter, and the check-in is closed when the
// expected number has arrived or after kTeamJoinTicks, whichever comes first.
// Blocks that start later leave at once, and jobs (columns) are claimed from a
// counter by whichever teams exist.  So concurrent kernels on other streams can
// make a team smaller, but cannot make it wait for a block that never starts.
// Every spin also ends after kTeamSpinTicks with the abort flag set; the
// drivers' finishing kernel then writes NaN, never a partial result.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace pf {

constexpr int kTeamXcc = 16;         // XCC ids of the hardware register (4 bits)
constexpr int kTeamPerXcc = 32;      // most teams of one XCD
constexpr uint32_t kTeamClosed = 0x80000000u;
constexpr uint64_t kTeamJoinTicks = 3000;         // 30 us of the 100 MHz wall clock
constexpr uint64_t kTeamSpinTicks = 2000000000u;  // 20 s

// One check-in per XCD and one barrier per team, each on its own line.
struct TeamJoin {
  uint32_t arrive;  // members so far | kTeamClosed
  uint32_t size;    // members when the check-in was closed
  uint32_t pad[30];
};
struct TeamBar {
  uint32_t at[32];  // barriers each member has arrived at (one line)
  uint32_t job;     // the job its leader claimed
  uint32_t slot;    // its work space
  uint32_t pad[30];
};
struct TeamCtl {
  uint32_t next;   // next unclaimed job
  uint32_t slots;  // work-space slots handed out
  uint32_t done;   // finished jobs
  uint32_t abort;  // a bounded wait ran out
  uint32_t pad[28];
  TeamJoin join[kTeamXcc];
  TeamBar bar[kTeamXcc * kTeamPerXcc];
};

__device__ __forceinline__ uint32_t team_load(const uint32_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void team_store(uint32_t* p, uint32_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t team_add(uint32_t* p, uint32_t v) {
  return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// All earlier vector stores of this wave have reached the L2.
__device__ __forceinline__ void team_drain() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

__device__ __forceinline__ uint32_t team_xcc() {
  uint32_t x;
  asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(x));
  return x & (kTeamXcc - 1);
}

// This block's place: member `idx` of a team of `n`, whose barrier is `bar`.
struct TeamPlace {
  uint32_t idx, n;
  TeamBar* bar;
  uint32_t passed;  // barriers this block has passed
};

// Spins until cond() or the bound; false: the bound or the flag.
template <class F>
__device__ __forceinline__ bool team_spin(TeamCtl* c, F&& cond) {
  uint64_t t0 = 0;
  for (uint32_t i = 1;; ++i) {
    if (cond()) return true;
    if ((i & 1023u) == 0) {
      const uint64_t t = wall_clock64();
      if (t0 == 0) t0 = t;
      if (t - t0 > kTeamSpinTicks || team_load(&c->abort)) {
        team_store(&c->abort, 1u);
        return false;
      }
    }
  }
}

// Thread 0 of each block: join the check-in of this XCD and split its members
// into teams of `want` (one smaller team when fewer than `want` came).  False:
// this block has no team.
__device__ __forceinline__ bool team_join(TeamCtl* c, uint32_t expect, uint32_t want,
                                          TeamPlace& me) {
  const uint32_t x = team_xcc();
  TeamJoin* j = &c->join[x];
  const uint32_t v = team_add(&j->arrive, 1u);
  if (v & kTeamClosed) return false;
  const uint64_t t0 = wall_clock64();
  const bool ok = team_spin(c, [&] {
    const uint32_t cur = team_load(&j->arrive);
    if (cur & kTeamClosed) return true;
    if (cur < expect && wall_clock64() - t0 < kTeamJoinTicks) return false;
    const uint32_t old = __hip_atomic_fetch_or(&j->arrive, kTeamClosed, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT);
    if (!(old & kTeamClosed)) team_store(&j->size, old);  // members 0 .. old-1
    return true;
  });
  if (!ok) return false;
  uint32_t n = 0;
  if (!team_spin(c, [&] { return (n = team_load(&j->size)) != 0; })) return false;
  uint32_t t;
  if (n < want) {
    t = 0;
    me.idx = v;
    me.n = n;
  } else {
    t = v / want;
    if ((t + 1) * want > n || t >= (uint32_t)kTeamPerXcc) return false;
    me.idx = v - t * want;
    me.n = want;
  }
  me.bar = &c->bar[x * kTeamPerXcc + t];
  me.passed = 0;
  return true;
}

// The team barrier, in two halves, called by wave 0 after a __syncthreads()
// that follows team_drain() in every wave.  What the block does between the
// halves overlaps the other blocks' arrival.  Each member stores its own word
// and every member polls all words at once (one line): no atomics to serialize.
__device__ __forceinline__ void team_arrive(TeamPlace& me) {
  ++me.passed;
  if (me.n > 1 && threadIdx.x == 0) team_store(&me.bar->at[me.idx], me.passed);
}
__device__ __forceinline__ bool team_wait(TeamCtl* c, TeamPlace& me) {
  if (me.n == 1) return true;
  const uint32_t* at = &me.bar->at[threadIdx.x & 31u];
  const bool member = (threadIdx.x & 31u) < me.n;
  return team_spin(c, [&] {
    const uint32_t v = team_load(at);
    return __all(!member || (int32_t)(v - me.passed) >= 0) != 0;
  });
}

constexpr int kTeamWaves = 16;  // most waves of a block

// A value that is the same in all lanes, as a scalar.
__device__ __forceinline__ uint32_t uni(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
}


// Uniform read-only data through the scalar cache.
template <typename S>
__device__ __forceinline__ S cload(const S* p) {
  typedef const __attribute__((address_space(4))) S* cp;
  return *(cp)(uintptr_t)p;
}
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
constexpr int kAgent = 16;  // buffer instruction cache policy: sc1

// Loads of 4, 8 or 16 bytes at voff + soff bytes, at agent scope.  (Stores
// take the default policy: they pass the CU's L1 and stay in the L2, where a
// store at agent scope is written through to memory, at half the rate.)
template <typename V>
__device__ __forceinline__ V bload(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  if constexpr (sizeof(V) == 16)
    return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, kAgent));
  else if constexpr (sizeof(V) == 8)
    return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, kAgent));
  else
    return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, kAgent));
}
template <typename V>
__device__ __forceinline__ void bstore(V v, __amdgpu_buffer_rsrc_t r, uint32_t voff,
                                       uint32_t soff) {
  if constexpr (sizeof(V) == 16)
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, voff, soff, 0);
  else if constexpr (sizeof(V) == 4)
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r, voff, soff, 0);
  else
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, voff, soff, 0);
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_of(void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(p, 0, bytes, 0x00027000);
}

// LDS at a byte offset of the dynamic block.
extern __shared__ __align__(16) char team_lds[];
template <typename T>
__device__ __forceinline__ T lread(uint32_t off) {
  typedef const __attribute__((address_space(3))) T* lp;
  typedef const __attribute__((address_space(3))) char* lc;
  return *(lp)((lc)team_lds + off);
}
template <typename T>
__device__ __forceinline__ void lwrite(uint32_t off, T v) {
  typedef __attribute__((address_space(3))) T* lp;
  typedef __attribute__((address_space(3))) char* lc;
  *(lp)((lc)team_lds + off) = v;
}

// What the blocks of a team share about the job in hand.
struct TeamShared {
  uint32_t idx, n, bar, slot, ok, job, seg, pad[9];
  double red[2 * kTeamWaves];  // the waves' dots of a step
};

// Both halves of the barrier around `between` (this block's own LDS update).
template <class F>
__device__ __forceinline__ bool team_step_end(TeamCtl* ctl, TeamShared& sh, TeamPlace& me,
                                              bool read_job, F&& between) {
  team_drain();
  __syncthreads();
  if (threadIdx.x < 64) team_arrive(me);
  between();
  if (threadIdx.x < 64) {
    const bool ok = team_wait(ctl, me);
    if (threadIdx.x == 0) {
      if (ok && read_job && me.n > 1) sh.job = team_load(&me.bar->job);
      sh.ok = ok;
      sh.seg = 0;
    }
  }
  __syncthreads();
  return uni(sh.ok) != 0;
}

// Joins a team (wave 0 polls the barrier with all its lanes, so every thread gets
// the place); false: none, or the abort flag.  `between` runs before the team's
// first barrier.  sh.slot: the team's number among all teams.
template <class F>
__device__ __forceinline__ bool team_enter(TeamCtl* ctl, uint32_t expect, uint32_t want,
                                           TeamShared& sh, TeamPlace& me, F&& between) {
  if (threadIdx.x == 0) {
    sh.ok = team_join(ctl, expect, want, me);
    if (sh.ok) {
      sh.idx = me.idx;
      sh.n = me.n;
      sh.bar = (uint32_t)(me.bar - ctl->bar);
      if (me.idx == 0) {
        sh.slot = team_add(&ctl->slots, 1u);
        if (me.n > 1) team_store(&me.bar->slot, sh.slot);
      }
    }
  }
  __syncthreads();
  if (!uni(sh.ok)) return false;
  me.idx = uni(sh.idx);
  me.n = uni(sh.n);
  me.bar = &ctl->bar[uni(sh.bar)];
  me.passed = 0;
  between();
  if (!team_step_end(ctl, sh, me, false, [] {})) return false;
  if (threadIdx.x == 0 && me.n > 1) sh.slot = team_load(&me.bar->slot);
  __syncthreads();
  return true;
}

// Next column of this team, or >= ncols when none is left; false: abort.
__device__ __forceinline__ bool team_next(TeamCtl* ctl, TeamShared& sh, TeamPlace& me) {
  __syncthreads();  // the last job's readers of `sh` and of LDS are done
  if (threadIdx.x == 0 && me.idx == 0) {
    sh.job = team_add(&ctl->next, 1u);
    if (me.n > 1) team_store(&me.bar->job, sh.job);
  }
  return team_step_end(ctl, sh, me, true, [] {});
}

}  // namespace pf
