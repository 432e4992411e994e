// Loads from global memory straight into LDS, and the barrier between stages that are filled by them.
#pragma once

#include <hip/hip_runtime.h>

// SHK_LOAD_TO_LDS(gptr, lptr): 16 bytes a lane: lane l's land at l * 16 behind lptr (the same for the whole wavefront)
#define SHK_LOAD_TO_LDS_PTR(gptr, lptr)                                                                    \
  __builtin_amdgcn_global_load_lds(                                                                       \
      reinterpret_cast<const __attribute__((address_space(1))) void*>(reinterpret_cast<uintptr_t>(gptr)), \
      (__attribute__((address_space(3))) void*)(lptr), 16, 0, 0)

// SHK_LOAD_TO_LDS(lds, offset, base): the same from base + offset to the byte `lds` of LDS.  Not the builtin: for that the
// compiler waits, before a read of LDS, for loads into any part of the same array; here the kernel waits by itself.
#define SHK_LOAD_TO_LDS_AT(lds, offset, base) shk::load_to_lds(lds, offset, base)

#define SHK_LOAD_TO_LDS_PICK(a, b, c, name, ...) name
#define SHK_LOAD_TO_LDS(...) \
  SHK_LOAD_TO_LDS_PICK(__VA_ARGS__, SHK_LOAD_TO_LDS_AT, SHK_LOAD_TO_LDS_PTR, )(__VA_ARGS__)

namespace shk {

// s_waitcnt's operand (gfx9 encoding): vmcnt in bits 3:0 and 15:14, expcnt in 6:4, lgkmcnt in 11:8; a counter at
// its maximum is not waited for.
constexpr int wait_counts(int vmcnt, int lgkmcnt) { return (vmcnt & 15) | (vmcnt >> 4) << 14 | 7 << 4 | lgkmcnt << 8; }

// (m0, the place in LDS, is an operand: written inside the statement, the builtin's next load would take what it had put
// there before, and a clobbered reserved register is no promise of the compiler's.  s_nop: m0 may be written right before.)
__device__ __forceinline__ void load_to_lds(unsigned lds, unsigned offset, const char* base) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"{m0}"(lds), "v"(offset), "s"(base) : "memory");
}

}  // namespace shk

// until at most n of the wavefront's loads from memory are in flight
#define SHK_WAIT_LOADS(n) __builtin_amdgcn_s_waitcnt(shk::wait_counts(n, 15))

// The workgroup's barrier between two stages.  Before it a wavefront waits until at most n of its loads are in flight, so
// that the older ones have landed in LDS for everybody behind the barrier, and until its own reads of LDS have
// returned: behind the barrier another wavefront's loads overwrite what they read, and neither the barrier nor the
// compiler, which sees no connection between those loads and these reads, waits for them.  (The multiplications that
// used them have nearly always waited already.)  Nothing that touches memory moves across.
#define SHK_MEET_WITH_LOADS(n)                               \
  asm volatile("" ::: "memory");                             \
  __builtin_amdgcn_s_waitcnt(shk::wait_counts(n, 0));        \
  asm volatile("" ::: "memory");                             \
  __builtin_amdgcn_s_barrier();                              \
  asm volatile("" ::: "memory")
