// What the grouped GEMMs with 32 x 32 MFMA tiles (moe_dense.hip, moe_prefill.hip) share: how a tile is stored.
#pragma once
#include "gemm_common.h"
#include "moe_dense.h"

namespace mi {
namespace moe {

using namespace mi::gemm;

__device__ __forceinline__ float widen16(bool bf16, unsigned short h) {
    return bf16 ? __uint_as_float(((unsigned)h) << 16) : (float)__builtin_bit_cast(_Float16, h);
}

// Stores one 32-slot x 32-channel tile held slot-per-lane (o[r]: channel 8 * (r / 4) + 4 * hb + r % 4 of the lane's
// slot) as 16-byte pieces: four registers are four consecutive channels; the two half-waves of a lane pair (l, l + 32)
// hold the two halves of every group of eight, and two lane-half swaps per pair of groups leave every lane with eight
// consecutive channels of its slot's row.  `row`: the slot's output row at the tile's first channel; n_left: channels
// from there to the end of the row.
template <typename E>
__device__ __forceinline__ void store_tile_slot_lane(const float (&o)[16], unsigned short* row, bool valid, int n_left,
                                                     bool vec_ok, int hb) {
    unsigned P[4][2];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        P[q][0] = E::pack(o[4 * q], o[4 * q + 1]);
        P[q][1] = E::pack(o[4 * q + 2], o[4 * q + 3]);
    }
#pragma unroll
    for (int q = 0; q < 4; q += 2) {
        // lower half-wave: own group q, then the partner's half of it; upper: the partner's half of group q + 1, then own
        const auto s0 = __builtin_amdgcn_permlane32_swap(P[q][0], P[q + 1][0], false, false);
        const auto s1 = __builtin_amdgcn_permlane32_swap(P[q][1], P[q + 1][1], false, false);
        const u32x4 v = {s0[0], s1[0], s0[1], s1[1]};
        const int c = 8 * q + 8 * hb;   // first of this lane's eight channels
        if (valid) {
            if (vec_ok && c + 8 <= n_left) {
                // (an ordinary store: what is written here is read again by the next launch -- the down projection
                // or the sum over the slots -- and a streaming store would send it past the L2 it can be found in;
                // measured 1-7 % on both launches, most at 16 384 tokens)
                *reinterpret_cast<u32x4*>(row + c) = v;
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (c + e < n_left) row[c + e] = (unsigned short)(v[e >> 1] >> (16 * (e & 1)));
            }
        }
    }
}

// Adds a pair of 32-slot x 32-channel tiles held channel-per-lane (rows of a tile = slots 8 * (r / 4) + 4 * hb + r % 4) into
// the tokens' output columns.  Two neighbouring MFMA column tiles are 64 consecutive channels: swapping the upper half of
// the first one's register with the lower half of the second one's gives one register with all 64 channels of row R and
// one with those of row R + 4.  Column (token_id - 1) >> acc_shift receives the replica's value as rounded to the storage
// type, by a packed atomic add of two adjacent channels: even lanes send row R, odd lanes row R + 4, each row 128
// consecutive bytes.
// ch0: the pair's first channel; tok / wt (LDS): tokens (0 = none) and routed weights of the 32 slots; s0 / s1 (SCALED):
// scales of channels ch0 + lane % 32 and ch0 + 32 + lane % 32.
template <typename E, bool SCALED>
__device__ __forceinline__ void accumulate_tile(const DenseArgs& a, const f32x16& acc0, const f32x16& acc1, float s0, float s1, const int* tok,
                                                const float* wt, int ch0, int lane) {
    typedef int i32x4_ __attribute__((ext_vector_type(4)));
    const int hb = lane >> 5, gn = ch0 + lane;
    unsigned short* const col = a.C + (gn & ~1);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        // the slots that this lane sends (R + 4 from odd lanes), and the weights of those it holds
        const i32x4_ t4 = *reinterpret_cast<const i32x4_*>(tok + 8 * q + 4 * (lane & 1));
        f32x4 w4 = {1.f, 1.f, 1.f, 1.f};
        if (a.mul_routed_weight) w4 = *reinterpret_cast<const f32x4*>(wt + 8 * q + 4 * hb);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float v0 = acc0[4 * q + e], v1 = acc1[4 * q + e];
            if constexpr (SCALED) {
                v0 *= s0;
                v1 *= s1;
            }
            if (a.mul_routed_weight) {
                v0 *= w4[e];
                v1 *= w4[e];
            }
            const auto sw = __builtin_amdgcn_permlane32_swap((unsigned)E::from_f32(v0), (unsigned)E::from_f32(v1), false, false);
            const unsigned rowA = sw[0], rowB = sw[1];   // this lane's channel of row R / of row R + 4
            const unsigned nbrA = (unsigned)__shfl_xor((int)rowA, 1, 64), nbrB = (unsigned)__shfl_xor((int)rowB, 1, 64);
            const unsigned pair = (lane & 1) ? (nbrB | (rowB << 16)) : (rowA | (nbrA << 16));
            if (t4[e] && gn < a.N) atomic_add2(a.bf16, col + (int64_t)((t4[e] - 1) >> a.acc_shift) * a.ldc, pair);
        }
    }
}

}  // namespace moe
}  // namespace mi
