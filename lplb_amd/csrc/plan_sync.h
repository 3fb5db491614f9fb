// How the workgroups of the one-launch plan talk to each other through memory.
//
// Everything that crosses workgroups is written and read with agent-scope atomics.
// What that relies on, on gfx950 (MI355X: eight XCDs, each with its own L2 that is not
// coherent with the others'):
//   * an agent-scope atomic store or load carries the sc1 bit, which makes it write
//     through / miss in the issuing XCD's L2, so the value lives in memory where every
//     XCD sees it; an agent-scope atomic add is carried out by the atomic unit behind
//     the caches, so there is no cached copy that could go stale;
//   * an aligned 8-byte store is one piece: a word whose high half has the launch's tag has its low half too, so
//     nothing has to be acknowledged or announced before such a word is read, and words may arrive in any order;
//   * everything a workgroup reads of another's is read with such loads, never with plain
//     loads behind an acquire fence: the fence (buffer_inv sc1) would invalidate this XCD's
//     L2, which holds the batch's indices at that point, once per workgroup;
//   * a poll loads anew each time round (the atomic may not be taken out of the loop).
// tests/test_host.py compiles these helpers on their own and checks that the forms above are really what the
// compiler emits, and that no kernel of the plan invalidates or writes back a cache, so a toolchain change that
// lowers them differently fails a test instead of silently breaking the exchange.
// (Checked with ROCm 7.2.0, clang 20.)
#pragma once
#include <hip/hip_runtime.h>

namespace lplb {

__device__ inline int agent_load(const int *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline unsigned long long agent_load(const unsigned long long *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Four pairs of words, each 16-byte aligned, with one load past the caches for both (there is no 16-byte atomic to
// ask the compiler for; each of the two words arrives in one piece).  Returns when they are there.
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
__device__ inline void agent_load_pairs(u32x4 (&v)[4], const unsigned long long *const (&p)[4]) {
  asm volatile("global_load_dwordx4 %0, %4, off sc1\n\t"
               "global_load_dwordx4 %1, %5, off sc1\n\t"
               "global_load_dwordx4 %2, %6, off sc1\n\t"
               "global_load_dwordx4 %3, %7, off sc1\n\t"
               "s_waitcnt vmcnt(0)"
               : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3])
               : "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3])
               : "memory");
}
__device__ inline void agent_store(int *p, int v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void agent_store(unsigned long long *p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Two pairs of words side by side, 16-byte aligned, past the caches with one store for each pair (each word lands in one piece).
// The data registers of a store of more than 8 bytes may not be written by either of the next two instructions; the compiler sees to
// that behind its own stores only.  (As two statements with a wait each: [4096 x 8] at 32 ranks 19.3 -> 19.4 us.)
__device__ inline void agent_store_pairs(unsigned long long *p, u32x4 first, u32x4 second) {
  asm volatile("global_store_dwordx4 %0, %1, off sc1\n\t"
               "global_store_dwordx4 %0, %2, off offset:16 sc1\n\t"
               "s_nop 1" ::"v"(p), "v"(first), "v"(second) : "memory");
}
__device__ inline int agent_add(int *p, int v) {
  return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void agent_add(unsigned long long *p, unsigned long long v) {
  __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void agent_replace(int *p, int expected, int v) {
  __hip_atomic_compare_exchange_strong(p, &expected, v, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

} // namespace lplb
