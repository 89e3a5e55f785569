// Small f16/bf16 GEMM: C(M,N) = A(M,K) * B(K,N), column-major, fp32 accumulate, for products of up to 128 tiles of 128 x 128.
//
// What bounds a product that leaves most CUs idle is what one CU brings into its LDS, about 95 GB/s: a K step of 32 of a
// 128 x 128 tile is 16 KB, the 0.18 us that it takes on gemm_big.hip's kernel.  So the tiles here are as small as it takes to
// give every CU one -- 32 x 32, 64 x 32, 64 x 64 or 128 x 64, whichever small_estimate says is through first -- and the
// four waves of a workgroup do not share a tile's extent but its K: wave w takes the stages w, w + 4, ... of 64 k, with an LDS
// area and accumulators of its own.  Nothing is shared before the sums are, so there is no barrier in the walk: a wave waits
// for its own transfers, reads all fragments of the stage into registers, requests its next stage into the same place and
// multiplies meanwhile.  (A ring of two or three stages per wave is no faster; eight waves, and stages of 32 k, are slower.)
// Two or more workgroups of the two smaller tiles fit a CU, and one's transfers run under another's products; 64 x 64 tiles have 259
// registers a lane and 128 x 64 all 512 with four spilled, one workgroup to a CU.  A wave adds
// every second step of 16 k (fourth on 32 x 32 tiles) into a chain of its own, 8 (16) chains per element in all, so the sums are no further from
// exact than those of the split over K that this kernel replaces; the waves' sums are added through the LDS in their order.
//
// Layouts, edges and the register-fed step behind the last chunk of k are gemm_big.hip's; a stage's row of B is one 128-byte
// line, chunk c of row n at position c ^ ((n >> 1) & 7); a stage of A has rows of 64 bytes (32 m, as they come), 128 (64 m: chunk
// c of row k at c ^ 4 ((k >> 1) & 1)) or 256 (128 m: c ^ 4 (k & 3)), so that a transpose read's half-wave covers all banks.
//
// Measured (us, before -> now): bf16 256 x 320 x 704 to fp32 8.9 -> 3.6, f16 512 x 384 x 1152 to fp32 9.3 -> 4.2, 320 x 479 x 1227
// 13.5 -> 4.8, 704 x 691 x 1472 13.0 -> 5.7, 1472 x 832 x 1457 18.3 -> 13.0, 3648 x 375 x 3264 26.9 -> 20.1, 1536 x 735 x 576 8.9 -> 6.7; a launch
// that does next to nothing is 3.1.
#include "gemm_small.h"

namespace {

using namespace mi;
using namespace mi::gemm;

constexpr int BK = 64;   // k per stage
constexpr int NW = kSplitWaves;

// Source of every chunk that lies past K.
__device__ __attribute__((aligned(16))) const unsigned zeros16s[4] = {0u, 0u, 0u, 0u};

template <typename E, typename OutT, int I, int J>
__global__ __launch_bounds__(64 * NW) void gemm16_small(const unsigned short* __restrict__ A, int64_t lda, int64_t sa,
                                                        const unsigned short* __restrict__ B, int64_t ldb, int64_t sb, OutT* __restrict__ C,
                                                        int64_t ldc, int64_t sc, int M, int N, int K, int tiles_m, int tiles_n, int batch,
                                                        int kpeel) {
    // K: the extent the transfers walk (a multiple of 8); kpeel: values of k behind it for the register-fed step
    constexpr int TM = 32 * I, TN = 32 * J;
    constexpr int RA = 512 / TM, RB = 512 / BK;     // rows per transfer
    constexpr int TA = BK / RA, TB = TN / RB;       // transfers per stage
    constexpr int STAGE = BK * (TM + TN);           // elements
    constexpr int CH = I * J == 1 ? 4 : 2;          // chains of sums per wave and element
    constexpr int AREA = STAGE > 2048 * I * J ? STAGE : 2048 * I * J;   // a wave's stage, and later its sums
    __shared__ __attribute__((aligned(1024))) unsigned short areas[NW * AREA];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const TileAt at = tile_at(blockIdx.x, tiles_m, tiles_n, batch);
    const int bz = at.bz, m0 = at.m * TM, n0 = at.n * TN;

    // ---- transfers: lane -> row and position of its 16 bytes; swizzles as in the header ---------------------------------------
    const unsigned lda2 = (unsigned)lda * 2, ldb2 = (unsigned)ldb * 2;
    const int krow = lane / (TM / 8);
    int ca = (lane % (TM / 8)) ^ (I == 2 ? 4 * ((krow >> 1) & 1) : I == 4 ? 4 * (krow & 3) : 0);
    if (m0 + 8 * ca >= M) ca = (M - 1 - m0) / 8;
    const unsigned offA = (unsigned)krow * lda2 + 16 * ca;
    unsigned offB[TB];
    int cb[2];   // chunk of k of even / odd transfers
#pragma unroll
    for (int e = 0; e < 2; ++e) cb[e] = (lane & 7) ^ ((4 * e + (lane >> 4)) & 7);
#pragma unroll
    for (int t = 0; t < TB; ++t) {
        int row = RB * t + lane / (BK / 8);
        if (n0 + row > N - 1) row = N - 1 - n0;   // rows past the edge: the last one again (never stored)
        offB[t] = (unsigned)row * ldb2 + 16 * cb[t & 1];
    }
    const char* Ab = (const char*)(A + (int64_t)bz * sa + m0);
    const char* Bb = (const char*)(B + (int64_t)bz * sb + (int64_t)n0 * ldb);
    const unsigned lds0 = (unsigned)(size_t)LDS_PTR(unsigned short, areas) + wave * (AREA * 2);
    const int nk = (K + BK - 1) / BK;
    auto issue = [&](int c) __attribute__((always_inline)) {
        const char* ag = Ab + (int64_t)(BK * c) * lda2;
        const char* bg = Bb + (int64_t)(BK * c) * 2;
        if (BK * (c + 1) <= K) {
#pragma unroll
            for (int t = 0; t < TA; ++t) load_lds(lds0 + 1024 * t, offA, ag + (int64_t)(RA * t) * lda2);
#pragma unroll
            for (int t = 0; t < TB; ++t) load_lds(lds0 + 1024 * (TA + t), offB[t], bg);
        } else {
            const int left = K - BK * c;
#pragma unroll
            for (int t = 0; t < TA; ++t) load_lds_at(lds0 + 1024 * t, RA * t + krow < left ? ag + (int64_t)(RA * t) * lda2 + offA : (const char*)zeros16s);
#pragma unroll
            for (int t = 0; t < TB; ++t) load_lds_at(lds0 + 1024 * (TA + t), 8 * cb[t & 1] < left ? bg + offB[t] : (const char*)zeros16s);
        }
    };
    if (wave < nk) issue(wave);

    // ---- fragments: element offsets within a stage ------------------------------------------------------------------------------
    const int hb = lane >> 5, g = lane >> 4, r = lane & 15;
    unsigned fb[BK / 16], fa[I];
#pragma unroll
    for (int ks = 0; ks < BK / 16; ++ks) fb[ks] = BK * TM + (lane & 31) * BK + 8 * ((2 * ks + hb) ^ ((lane >> 1) & 7));
#pragma unroll
    for (int i = 0; i < I; ++i) {
        const int c = 4 * i + 2 * (g & 1) + ((r & 3) >> 1);
        fa[i] = (8 * (g >> 1) + (r >> 2)) * TM + 8 * (c ^ (I == 2 ? 4 * (r >> 3) : I == 4 ? 4 * (r >> 2) : 0)) + 4 * (r & 1);
    }
    f32x16 ch[CH][I][J];
#pragma unroll
    for (int h = 0; h < CH; ++h)
#pragma unroll
        for (int i = 0; i < I; ++i)
#pragma unroll
            for (int j = 0; j < J; ++j) ch[h][i][j] = f32x16{0};
    f32x16 (&acc)[I][J] = ch[0];

    if (kpeel > 0 && wave == (nk & (NW - 1))) {   // (the wave with the fewest stages)
        // k = K .. K + kpeel - 1 as the first values of one 16-wide MFMA step: the lower half-wave holds k 0..7 of its
        // row of B / column of A, the upper half-wave zeros.
        const unsigned short* Ap = A + (int64_t)bz * sa + (int64_t)K * lda;
        const unsigned short* Bp = B + (int64_t)bz * sb + K;
        const bool lower = lane < 32;
        s16x8 pa[I], pb[J];
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const int64_t n = n0 + 32 * j + (lane & 31);
#pragma unroll
            for (int q = 0; q < 8; ++q) pb[j][q] = lower && q < kpeel && n < N ? (short)Bp[n * ldb + q] : (short)0;
        }
#pragma unroll
        for (int i = 0; i < I; ++i) {
            const int64_t m = m0 + 32 * i + (lane & 31);
#pragma unroll
            for (int q = 0; q < 8; ++q) pa[i][q] = lower && q < kpeel && m < M ? (short)Ap[m + (int64_t)q * lda] : (short)0;
        }
#pragma unroll
        for (int i = 0; i < I; ++i)
#pragma unroll
            for (int j = 0; j < J; ++j) acc[i][j] = E::mfma32(pb[j], pa[i], acc[i][j]);
    }

    // ---- the walk: no barrier, a wave waits for its own transfers only ------------------------------------------------------------
    unsigned short* S = areas + wave * AREA;
    for (int c = wave; c < nk; c += NW) {
        wait_vm<0>();
        s16x8 a[BK / 16][I], b[BK / 16][J];
#pragma unroll
        for (int ks = 0; ks < BK / 16; ++ks) {
#pragma unroll
            for (int j = 0; j < J; ++j) b[ks][j] = *reinterpret_cast<const s16x8*>(S + fb[ks] + 32 * j * BK);
#pragma unroll
            for (int i = 0; i < I; ++i) {
                const unsigned short* p = S + fa[i] + 16 * ks * TM;
                const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(s16x4, p));
                const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(s16x4, p + 4 * TM));
                a[ks][i] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
            }
        }
        if (c + NW < nk) {
            wait_lds();          // every fragment of the stage is in registers: its place is free
            asm volatile("" ::: "memory");
            issue(c + NW);
        }
#pragma unroll
        for (int ks = 0; ks < BK / 16; ++ks)
#pragma unroll
            for (int i = 0; i < I; ++i)
#pragma unroll
                for (int j = 0; j < J; ++j) ch[ks % CH][i][j] = E::mfma32(b[ks][j], a[ks][i], ch[ks % CH][i][j]);
    }

    // ---- the four waves' sums, added in their order; a wave stores a quarter of the tile ---------------------------------------
#pragma unroll
    for (int h = 1; h < CH; ++h)
#pragma unroll
        for (int i = 0; i < I; ++i)
#pragma unroll
            for (int j = 0; j < J; ++j) acc[i][j] += ch[h][i][j];
    add_and_store<E, OutT, I, J, AREA * 2>(acc, (char*)areas, wave, lane, C + (int64_t)bz * sc, ldc, M, N, m0, n0);
}

template <typename E, typename OutT, int I, int J>
void launch(const Problem& p, int kd, hipStream_t s) {
    const int tiles_m = (p.M + 32 * I - 1) / (32 * I), tiles_n = (p.N + 32 * J - 1) / (32 * J);
    hipLaunchKernelGGL((gemm16_small<E, OutT, I, J>), dim3((unsigned)(tiles_m * tiles_n * p.batch)), dim3(64 * NW), 0, s,
                       (const unsigned short*)p.A, p.lda, p.sa, (const unsigned short*)p.B, p.ldb, p.sb, (OutT*)p.C, p.ldc, p.sc, p.M, p.N, kd,
                       tiles_m, tiles_n, p.batch, p.K - kd);
}

}  // namespace

namespace mi {
namespace gemm {

// The launch as such, and for every workgroup that a CU gets its ramp and its bytes, dearer where rows start off 16-byte
// boundaries.  Fitted to 420 shapes (256 to 4096 each way, up to 260 tiles of 128 x 128); the tile that it picks takes 1.007
// times the best tile's time in the mean, 1.12 at most.
double small16_estimate(const Problem& p, bool misaligned, int* tile) {
    static const struct { int tile, tm, tn; double launch, ramp, k, k_mis, k_once; } T[4] = {
        {11, 32, 32, 2.72, 0.13, 1.62e-3, 0.61e-3, -0.45e-3},
        {21, 64, 32, 2.67, 0.48, 1.83e-3, 0.86e-3, -0.26e-3},
        {22, 64, 64, 1.35, 3.03, 2.80e-3, 1.32e-3, -0.63e-3},
        {42, 128, 64, 1.04, 5.86, 3.82e-3, 1.48e-3, -0.09e-3}};
    double best = 1e30;
    for (const auto& t : T) {
        const double rounds = (double)((tiles_of(p, t.tm, t.tn) + 255) / 256);
        const double us = t.launch + t.k_once * p.K + rounds * (t.ramp + p.K * (t.k + (misaligned ? t.k_mis : 0.0)));
        if (us < best) {
            best = us;
            *tile = t.tile;
        }
    }
    return best;
}

void small16_launch(const Problem& p, int tile, int kd, hipStream_t s) {
    const bool f32out = p.out_dtype == MI_F32;
#define TILE(E, O) (tile == 11 ? launch<E, O, 1, 1>(p, kd, s) : tile == 21 ? launch<E, O, 2, 1>(p, kd, s) : tile == 22 ? launch<E, O, 2, 2>(p, kd, s) : launch<E, O, 4, 2>(p, kd, s))
    if (p.in_dtype == MI_F16) {
        if (f32out) TILE(F16, float);
        else TILE(F16, unsigned short);
    } else {
        if (f32out) TILE(BF16, float);
        else TILE(BF16, unsigned short);
    }
#undef TILE
    set_variant(tile == 11 ? "gemm16_small_32x32x64" : tile == 21 ? "gemm16_small_64x32x64" : tile == 22 ? "gemm16_small_64x64x64" : "gemm16_small_128x64x64");
}

}  // namespace gemm
}  // namespace mi
