// DMA from global memory into LDS with an address per lane.
#pragma once
#include "common.h"

namespace sp {

// One wave-wide DMA: every lane copies 16 bytes from its own global address to LDS byte m0 + 16 * lane; chunks that do
// not exist (past the end of a row) are fetched from a block of zeros instead.  Completion is tracked by vmcnt, which the
// compiler does not see.
__device__ __forceinline__ void dma_to_lds_addr(const unsigned char* addr, unsigned lds_addr) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(addr), "s"(lds_addr) : "memory", "m0");
}
__device__ __attribute__((aligned(16))) const unsigned kZeroChunk[4] = {0u, 0u, 0u, 0u};

}  // namespace sp
