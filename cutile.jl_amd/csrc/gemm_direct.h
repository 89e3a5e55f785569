// Pieces shared by the direct-to-LDS GEMM kernels (gemm_big.hip and gemm_pc.hip: 16-bit operands, gemm32_big.hip: fp32,
// moe_dense.hip and moe_prefill.hip: grouped).
#pragma once
#include <cstdlib>

#include "gemm_common.h"

namespace mi {
namespace gemm {

// sched_group_barrier masks
#define SG_MFMA 0x008
#define SG_VMEM 0x010
#define SG_DSRD 0x100

__device__ __forceinline__ void gload_lds16(const void* g, void* lds_wave_base) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)g,
                                     (__attribute__((address_space(3))) void*)lds_wave_base, 16, 0, 0);
}

template <int VMCNT>
__device__ __forceinline__ void stage_barrier() {
    // My reads of the current stage are done (lgkmcnt(0)) and my transfers into the next stage
    // have landed (vmcnt leaves only the VMCNT youngest transfers in flight); then meet the
    // other waves.  The wait is the builtin, not inline asm, so that the compiler's own
    // wait-count bookkeeping sees it and does not add a full vmcnt(0) drain before the
    // following LDS reads.  gfx9 encoding: vmcnt[3:0] | expcnt[6:4] | lgkmcnt[11:8] | vmcnt[15:14].
    constexpr int imm = (VMCNT & 15) | (7 << 4) | (0 << 8) | ((VMCNT >> 4) << 14);
    __builtin_amdgcn_s_waitcnt(imm);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// waits until at most N transfers are in flight
template <int N>
__device__ __forceinline__ void wait_vm() {
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
    asm volatile("" ::: "memory");
}
__device__ __forceinline__ void wait_lds() { __builtin_amdgcn_s_waitcnt(0xc07f); }   // lgkmcnt(0)
__device__ __forceinline__ void meet() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Workgroup ids congruent mod 8 share an XCD and its L2: each XCD gets a contiguous run of the tiles, so that it works on
// neighbouring ones.  From 64 tiles on also where they are no multiple of 8 (2200 x 1100 x 4000 bf16 38.4 -> 36.8 us,
// 3667 x 407 x 384 10.0 -> 9.3); fewer are better spread (60 tiles, 1536 x 640 x 1280: 13.5 spread, 14.3 in runs).
__device__ __forceinline__ int xcd_tile(int id, int total) {
    const int x = id & 7, each = total >> 3, more = total & 7;
    if (more && total < 64) return id;
    return x * each + (x < more ? x : more) + (id >> 3);
}

// Stores a wave's (32*I) x (32*J) part (wm, wn) of the BTM x BTN tile at (m0, n0): the lane's column of an MFMA tile is m,
// its rows are n, so a half-wave stores 32 consecutive m of one column of C.  STREAM: see streamed_stores.
template <typename E, typename OutT, int I, int J, bool STREAM>
__device__ __forceinline__ void store_tile(const f32x16 (&acc)[I][J], OutT* C, int64_t ldc, int M, int N, int m0, int n0, int wm, int wn,
                                           int btm, int btn, int lane) {
    // The lane's own offset (m within the wave tile, plus its 4*hb rows of n) is a 32-bit element offset; the part of n
    // that is uniform across the wave goes into the base.
    const unsigned lane_off = (unsigned)((lane & 31) + (int64_t)(4 * (lane >> 5)) * ldc);
    OutT* Cw = C + (int64_t)m0 + wm + ((int64_t)n0 + wn) * ldc;
    if (m0 + btm <= M && n0 + btn <= N) {   // interior tile (same for the whole workgroup)
#pragma unroll
        for (int i = 0; i < I; ++i)
#pragma unroll
            for (int j = 0; j < J; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    OutT* cu = Cw + 32 * i + (int64_t)(32 * j + 8 * (r >> 2) + (r & 3)) * ldc;
                    st_global<STREAM>(cvt_out<E, OutT>(acc[i][j][r]), cu + lane_off);
                }
    } else {                                // edge tile: clip to the matrix
        int m_left = M - (m0 + wm + (lane & 31)), n_left = N - (n0 + wn + 4 * (lane >> 5));
#pragma unroll
        for (int i = 0; i < I; ++i)
#pragma unroll
            for (int j = 0; j < J; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    // the empty statement keeps each test next to its store (256 hoisted lane masks would
                    // not fit the scalar registers)
                    asm volatile("" : "+v"(m_left), "+v"(n_left));
                    const int dn = 32 * j + 8 * (r >> 2) + (r & 3);
                    if (32 * i < m_left && dn < n_left) {
                        float v = acc[i][j][r];
                        asm volatile("" : "+v"(v));   // convert after the test, not 256 values ahead of it
                        st_global<STREAM>(cvt_out<E, OutT>(v), Cw + 32 * i + (int64_t)dn * ldc + lane_off);
                    }
                }
    }
}

// Whether a product's results are stored past the L2.  The 32 lanes of a half-wave store 64 or 128 bytes of a column of C: whole
// segments where every column starts on a 64-byte boundary.  Off them a store ends inside a segment that the next one goes on
// with; streamed, each piece went to memory by itself, while ordinary stores meet in the L2 (us, streamed : ordinary, f16 3241 x 1985
// x 1723 to fp32 45.1 : 35.5, 2723 x 2496 x 704 25.2 : 20.9, 4095^3 151 : 140, bf16 2999 x 2100 x 3001 57.2 : 55.1, fp32 8 x 1021 x
// 2047 x 509 171 : 140).  On them the streamed ones are ahead (f16 1024 x 3072 x 961 to fp32 11.8 : 12.6, 320 x 1344 x 2944 13.4 : 14.4).
// A template parameter: with both kinds in one kernel the branches are made one, of ordinary stores, or the code is half as long again.
inline bool streamed_stores(const Problem& p) {
    const int64_t size = dtype_size(p.out_dtype);
    return !(((uintptr_t)p.C | (uintptr_t)(p.ldc * size) | (uintptr_t)(p.batch > 1 ? p.sc * size : 0)) & 63);
}

inline int64_t tiles_of(const Problem& p, int btm, int btn) {
    return (int64_t)((p.M + btm - 1) / btm) * ((p.N + btn - 1) / btn) * p.batch;
}

// Tile size: whichever needs least time by "rounds of workgroups x time of a round".  Measured time of
// one K step of a round (us): 256x256 0.63 (a quarter of the CUs busy) to 0.93 (all busy: the clock
// drops); 256x128 0.42 to 0.51; 128x128 0.33 with one workgroup per CU, 0.58 when CUs hold two.
// f16 examples (us, 256x256 / 256x128 / 128x128): 1024^3 23 / 15 / 10, 2048^3 40 / 27 / 21,
// 2560^3 51 / 37 / 46, 4096 x 2048 x 4096 77 / 65 / 74, 3072^3 64 / 83 / 77, 4096^3 119 / 128 / 144.
// `cost` (optional): the estimate for the tile chosen, in units of about 1 % of the 4096^3 product's time per 4096 of K.
inline int pick_direct_tile(const Problem& p, int64_t* cost = nullptr) {
    static const int force = [] { const char* e = getenv("MI_GEMM_BIG_TILE"); return e ? atoi(e) : 0; }();   // 44, 42 or 22
    const int64_t t44 = tiles_of(p, 256, 256), t42 = tiles_of(p, 256, 128), t22 = tiles_of(p, 128, 128);
    const int64_t c44 = (t44 + 255) / 256 * 90, c42 = (t42 + 255) / 256 * 50;
    const int64_t c22 = t22 <= 256 ? 33 : (t22 + 511) / 512 * 60;
    const int t = c22 <= c42 && c22 <= c44 ? 22 : c42 <= c44 ? 42 : 44;
    if (cost) *cost = t == 22 ? c22 : t == 42 ? c42 : c44;
    if (force == 44 || force == 42 || force == 22) return force;
    return t;
}

// gemm_pc.hip: the kernel whose transfers have waves of their own, with tiles of 256 x 128 (tile = 42) or 128 x 128 (22); kd: the
// extent of K that the transfers walk.
void pc16_launch(const Problem& p, int tile, int kd, hipStream_t s);
// gemm_small.hip: the kernel for few tiles, whose waves split K: the time (us) and the tile (11, 21, 22 or 42) that it would be
// launched with / the launch.
double small16_estimate(const Problem& p, bool misaligned, int* tile);
void small16_launch(const Problem& p, int tile, int kd, hipStream_t s);

}  // namespace gemm
}  // namespace mi
