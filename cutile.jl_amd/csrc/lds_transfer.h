// Transfers of one wave from global memory into LDS, without staging registers, for the kernels whose waves have LDS areas of their
// own (gemm_small.hip, gemm32_small.hip, moe_few.hip, fmha_few.hip).
#pragma once
#include "common.h"

#pragma clang diagnostic ignored "-Winline-asm"  // m0 is named as clobbered on purpose

namespace mi {

// One 1 KB transfer, 16 bytes per lane: to LDS byte address `lds` from sbase + voff / from a lane's own address.  (Inline
// assembly, so that the compiler does not tie reads of one stage to transfers into another; the waits are counted by hand.)
__device__ __forceinline__ void load_lds(unsigned lds, unsigned voff, const char* sbase) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds), "v"(voff), "s"(sbase) : "m0", "memory");
}
__device__ __forceinline__ void load_lds_at(unsigned lds, const char* p) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(lds), "v"(p) : "m0", "memory");
}

}  // namespace mi
