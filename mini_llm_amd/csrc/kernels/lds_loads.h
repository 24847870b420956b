// Loads from memory straight into LDS, and the waits for them.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

// One piece of a wavefront's loads straight into LDS: every lane's 16 bytes at base + offset go to lane-linear places from `lds` on. In
// assembly, because a load into LDS that the compiler knows of makes it wait for all of them in front of the next LDS read:
// whoever calls this waits (wait_loads_and_meet) and passes a barrier before the bytes are read. It has no result register. The compiler sees no
// instruction in here, so the wait state that gfx9 needs between a scalar write of m0 and a load into LDS (which would otherwise
// go to the place of the load before it) stands here too; m0 is ours for the length of the block only.
__device__ __forceinline__ void load_to_lds(const unsigned char* base, unsigned offset, unsigned lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" :: "s"(lds), "v"(offset), "s"(base) : "m0", "memory");
}
__device__ __forceinline__ void load_to_lds(const unsigned char* base, size_t offset, unsigned lds) {         // (for offsets of any size)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" :: "s"(lds), "v"(base + offset) : "m0", "memory");
}
// Waits until at most N of the wavefront's loads are under way (they end in their order) and its LDS reads are done, then for the others.
template <int N>
__device__ __forceinline__ void wait_loads_and_meet() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(N) : "memory");
}
// The same for a number of k tiles that may stay under way, at most MOST (all wavefronts of a workgroup pass the same).
template <int MOST, int LOADS>
__device__ __forceinline__ void wait_tiles_and_meet(int under_way) {
    if constexpr (MOST > 0) {
        if (under_way < MOST) return wait_tiles_and_meet<MOST - 1, LOADS>(under_way);
    }
    wait_loads_and_meet<MOST * LOADS>();
}
