// Pieces shared by the GEMM kernels for few tiles, whose four waves split K (gemm_small.hip: 16-bit operands,
// gemm32_small.hip: fp32, moe_few.hip: grouped).
#pragma once
#include "gemm_direct.h"
#include "lds_transfer.h"

namespace mi {
namespace gemm {

constexpr int kSplitWaves = 4;

// The four waves' sums of a (32*I) x (32*J) tile, added through the LDS in the order of the waves; a wave stores a quarter of
// the tile, at (m0, n0) of C.  `areas`: one of AREA bytes per wave, at least 4096 * I * J, whose wave is done with it.
template <typename E, typename OutT, int I, int J, int AREA>
__device__ __forceinline__ void add_and_store(const f32x16 (&acc)[I][J], char* areas, int wave, int lane, OutT* C, int64_t ldc, int M, int N, int m0, int n0) {
    static_assert(AREA >= 4096 * I * J, "a wave's sums fit its area");
    char* sums = areas + wave * AREA;
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
        for (int j = 0; j < J; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *reinterpret_cast<f32x4*>(sums + ((4 * (i * J + j) + q) * 64 + lane) * 16) =
                    f32x4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
    __syncthreads();
#pragma unroll
    for (int u = 0; u < I * J; ++u) {
        const int q = wave * (I * J) + u, t = q >> 2;   // four rows of tile t = i * J + j
        f32x4 v = *reinterpret_cast<const f32x4*>(areas + (q * 64 + lane) * 16);
#pragma unroll
        for (int w = 1; w < kSplitWaves; ++w) v += *reinterpret_cast<const f32x4*>(areas + w * AREA + (q * 64 + lane) * 16);
        const int m = m0 + 32 * (t / J) + (lane & 31), n = n0 + 32 * (t % J) + 8 * (q & 3) + 4 * (lane >> 5);
        OutT* Cp = C + m + (int64_t)n * ldc;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (m < M && n + e < N) Cp[(int64_t)e * ldc] = cvt_out<E, OutT>(v[e]);
    }
}

// Workgroup -> batch entry and tile: XCDs get runs of neighbouring tiles, four tiles along M at a time.
struct TileAt {
    int bz, m, n;
};
__device__ __forceinline__ TileAt tile_at(int id, int tiles_m, int tiles_n, int batch) {
    const int total = tiles_m * tiles_n;
    int L = xcd_tile(id, total * batch);
    TileAt t;
    t.bz = L / total;
    L -= t.bz * total;
    constexpr int GM = 4;
    const int per_group = GM * tiles_n, first_m = (L / per_group) * GM;
    const int gsz = tiles_m - first_m < GM ? tiles_m - first_m : GM;
    t.m = first_m + (L % per_group) % gsz;
    t.n = (L % per_group) / gsz;
    return t;
}

}  // namespace gemm
}  // namespace mi
