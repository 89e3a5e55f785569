// fp32 GEMM for few tiles: C(M,N) = A(M,K) * B(K,N), column-major, v_mfma_f32_32x32x2_f32 -- the fp32 sibling of gemm_small.hip's
// kernel: the four waves of a workgroup split K, wave w takes the stages w, w + 4, ... of 32 k with an LDS area and accumulators of its
// own, no barrier in the walk, the sums added through the LDS at the end.
//
// What bounds a small fp32 product is the MFMA time of its busiest CU (32 x 32 x 1 k: 8 cycles), so tiles of 32 x 32 or 64 x 32, which
// spread it over two to four times the CUs of gemm32_big.hip's 64 x 64, win until every CU has one; from there on the larger tile's
// shorter transfers (256 bytes per k for 8 cycles here, 512 for 32 there) do.  64 x 64 and 128 x 64 split over the waves like this are
// behind the tiles of gemm32_big.hip, whose waves take a quarter of the tile each.
//
// Layouts, edges and the pairing of k with the MFMAs are gemm32_big.hip's; a stage's row of B is one 128-byte line, chunk c of row n at
// position c ^ ((n >> 1) & 7); the rows of a stage of A have 64 m (chunk c of row k at c ^ (8 * ((k >> 2) & 1))) or 32 m (row k in
// place of row k ^ ((k >> 2) & 1)), so that the two rows that the halves of a wave read, k and k + 4, are on different banks.
//
// Measured (us, before -> now): 2 x 128 x 525 x 448 9.5 -> 5.2, 4 x 256 x 215 x 273 8.1 -> 4.7, 6 x 151 x 320 x 352 9.3 -> 6.4, 3 x 723 x 128 x
// 499 11.1 -> 7.7; where gemm32_big.hip does not apply 2 x 192 x 128 x 320 42 -> 4.5, 4 x 165 x 543 x 128 19.9 -> 4.6.
#include "gemm_small.h"

namespace {

using namespace mi;
using namespace mi::gemm;

constexpr int BK = 32;   // k per stage
constexpr int NW = kSplitWaves;

// Source of every chunk that lies past K.
__device__ __attribute__((aligned(16))) const unsigned zeros32s[4] = {0u, 0u, 0u, 0u};

template <int I, int J>
__global__ __launch_bounds__(64 * NW) void gemm32_small(const float* __restrict__ A, int64_t lda, int64_t sa, const float* __restrict__ B,
                                                        int64_t ldb, int64_t sb, float* __restrict__ C, int64_t ldc, int64_t sc, int M, int N,
                                                        int K, int tiles_m, int tiles_n, int batch, int kpeel) {
    // K: the extent the transfers walk (a multiple of 4); kpeel: values of k behind it (up to 4) for the register-fed step
    constexpr int TM = 32 * I, TN = 32 * J;
    constexpr int RA = 256 / TM, RB = 256 / BK;     // rows per transfer
    constexpr int TA = BK / RA, TB = TN / RB;       // transfers per stage
    constexpr int STAGE = BK * (TM + TN);           // elements
    constexpr int AREA = STAGE > 1024 * I * J ? STAGE : 1024 * I * J;   // a wave's stage, and later its sums
    constexpr int CH = I * J == 1 ? 2 : 1;          // chains of sums per wave and element (one MFMA waits for the other)
    __shared__ __attribute__((aligned(1024))) float areas[NW * AREA];
    const int lane = threadIdx.x & 63, hb = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const TileAt at = tile_at(blockIdx.x, tiles_m, tiles_n, batch);
    const int bz = at.bz, m0 = at.m * TM, n0 = at.n * TN;

    // ---- transfers: lane -> row and position of its 16 bytes; swizzles as in the header ---------------------------------------
    const unsigned lda4 = (unsigned)lda * 4, ldb4 = (unsigned)ldb * 4;
    int krow[TA];   // row of k within a stage that the lane's part of transfer t holds
    unsigned offA[TA];
#pragma unroll
    for (int t = 0; t < TA; ++t) {
        const int p = RA * t + lane / (TM / 4);                      // LDS row
        krow[t] = I == 1 ? p ^ ((p >> 2) & 1) : p;
        int ca = (lane % (TM / 4)) ^ (I == 1 ? 0 : 8 * ((p >> 2) & 1));
        if (m0 + 4 * ca >= M) ca = (M - 1 - m0) / 4;
        offA[t] = (unsigned)krow[t] * lda4 + 16 * ca;
    }
    unsigned offB[TB];
    int cb[2];   // chunk of k of even / odd transfers
#pragma unroll
    for (int e = 0; e < 2; ++e) cb[e] = (lane & 7) ^ ((4 * e + (lane >> 4)) & 7);
#pragma unroll
    for (int t = 0; t < TB; ++t) {
        int row = RB * t + (lane >> 3);
        if (n0 + row > N - 1) row = N - 1 - n0;   // rows past the edge: the last one again (never stored)
        offB[t] = (unsigned)row * ldb4 + 16 * cb[t & 1];
    }
    const char* Ab = (const char*)(A + (int64_t)bz * sa + m0);
    const char* Bb = (const char*)(B + (int64_t)bz * sb + (int64_t)n0 * ldb);
    const unsigned lds0 = (unsigned)(size_t)LDS_PTR(float, areas) + wave * (AREA * 4);
    const int nk = (K + BK - 1) / BK;
    auto issue = [&](int c) __attribute__((always_inline)) {
        const char* ag = Ab + (int64_t)(BK * c) * lda4;
        const char* bg = Bb + (int64_t)(BK * c) * 4;
        if (BK * (c + 1) <= K) {
#pragma unroll
            for (int t = 0; t < TA; ++t) load_lds(lds0 + 1024 * t, offA[t], ag);
#pragma unroll
            for (int t = 0; t < TB; ++t) load_lds(lds0 + 1024 * (TA + t), offB[t], bg);
        } else {
            const int left = K - BK * c;
#pragma unroll
            for (int t = 0; t < TA; ++t) load_lds_at(lds0 + 1024 * t, krow[t] < left ? ag + offA[t] : (const char*)zeros32s);
#pragma unroll
            for (int t = 0; t < TB; ++t) load_lds_at(lds0 + 1024 * (TA + t), 4 * cb[t & 1] < left ? bg + offB[t] : (const char*)zeros32s);
        }
    };
    if (wave < nk) issue(wave);

    f32x16 ch[CH][I][J];
#pragma unroll
    for (int h = 0; h < CH; ++h)
#pragma unroll
        for (int i = 0; i < I; ++i)
#pragma unroll
            for (int j = 0; j < J; ++j) ch[h][i][j] = f32x16{0};
    f32x16 (&acc)[I][J] = ch[0];

    if (kpeel > 0 && wave == (nk & (NW - 1))) {   // (the wave with the fewest stages)
        const float* Ap = A + (int64_t)bz * sa + (int64_t)K * lda;
        const float* Bp = B + (int64_t)bz * sb + K;
        float pa[2][I], pb[2][J];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int q = 2 * s + hb;
#pragma unroll
            for (int j = 0; j < J; ++j) {
                const int64_t n = n0 + 32 * j + (lane & 31);
                pb[s][j] = q < kpeel && n < N ? Bp[n * ldb + q] : 0.f;
            }
#pragma unroll
            for (int i = 0; i < I; ++i) {
                const int64_t m = m0 + 32 * i + (lane & 31);
                pa[s][i] = q < kpeel && m < M ? Ap[m + (int64_t)q * lda] : 0.f;
            }
        }
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int i = 0; i < I; ++i)
#pragma unroll
                for (int j = 0; j < J; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(pb[s][j], pa[s][i], acc[i][j], 0, 0, 0);
    }

    // ---- the walk: no barrier, a wave waits for its own transfers only ------------------------------------------------------------
    // Lane half h carries k = 8 v + 4 h + q of the q-th of four MFMAs of a group v of 8 k.
    const float* const S = areas + wave * AREA;
    unsigned fb[BK / 8], fa[I == 1 ? 4 : I];
#pragma unroll
    for (int v = 0; v < BK / 8; ++v) fb[v] = BK * TM + (lane & 31) * BK + 4 * ((2 * v + hb) ^ ((lane >> 1) & 7));
#pragma unroll
    for (int x = 0; x < (I == 1 ? 4 : I); ++x)
        fa[x] = I == 1 ? (4 * hb + (x ^ hb)) * TM + (lane & 31) : 4 * hb * TM + ((32 * x + (lane & 31)) ^ (32 * hb));
    for (int c = wave; c < nk; c += NW) {
        wait_vm<0>();
        f32x4 b[BK / 8][J];
        float a[BK / 8][4][I];
#pragma unroll
        for (int v = 0; v < BK / 8; ++v) {
#pragma unroll
            for (int j = 0; j < J; ++j) b[v][j] = *reinterpret_cast<const f32x4*>(S + fb[v] + 32 * j * BK);
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int i = 0; i < I; ++i) a[v][q][i] = I == 1 ? S[fa[q] + 8 * v * TM] : S[fa[i] + (8 * v + q) * TM];
        }
        if (c + NW < nk) {
            wait_lds();          // every fragment of the stage is in registers: its place is free
            asm volatile("" ::: "memory");
            issue(c + NW);
        }
#pragma unroll
        for (int v = 0; v < BK / 8; ++v)
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int i = 0; i < I; ++i)
#pragma unroll
                    for (int j = 0; j < J; ++j) ch[q % CH][i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(b[v][j][q], a[v][q][i], ch[q % CH][i][j], 0, 0, 0);
    }
#pragma unroll
    for (int h = 1; h < CH; ++h)
#pragma unroll
        for (int i = 0; i < I; ++i)
#pragma unroll
            for (int j = 0; j < J; ++j) acc[i][j] += ch[h][i][j];
    add_and_store<F16, float, I, J, AREA * 4>(acc, (char*)areas, wave, lane, C + (int64_t)bz * sc, ldc, M, N, m0, n0);
}

template <int I, int J>
void launch(const Problem& p, int kd, hipStream_t s) {
    const int tiles_m = (p.M + 32 * I - 1) / (32 * I), tiles_n = (p.N + 32 * J - 1) / (32 * J);
    hipLaunchKernelGGL((gemm32_small<I, J>), dim3((unsigned)(tiles_m * tiles_n * p.batch)), dim3(64 * NW), 0, s, (const float*)p.A, p.lda, p.sa,
                       (const float*)p.B, p.ldb, p.sb, (float*)p.C, p.ldc, p.sc, p.M, p.N, kd, tiles_m, tiles_n, p.batch, p.K - kd);
}

}  // namespace

namespace mi {
namespace gemm {

// The kernel and tile that are estimated to be through first (us), for products of up to 2048 tiles of 64 x 64 and a K of 64 to 1024:
// this one's, gemm32_big.hip's 64 x 64, 128 x 128 or 256 x 128, or where that does not apply the register-staged kernel.  A launch,
// and per round of the CUs a ramp and the walk, in whole stages for each wave, dearer with rows off 16-byte boundaries; fitted to 420
// shapes of 2 to 12 times 128..1024 x 128..2048 x 128..512, each with all of the tiles, off by 5 to 9 % (standard deviation).  Five
// workgroups of the 32 x 32 tile fit a CU by their LDS, three of the 64 x 32 one: what comes sixth runs by itself, and there the 64 x 64 tile,
// which has 1.3 to 1.5 rounds then, is the quicker one (8 x 765 x 256 x 384 16.5 : 19.8, of 67 such shapes 38 by more than 2 %); with three
// rounds of 64 x 32 tiles likewise, and with five of 32 x 32 ones the estimate has to promise 12 %.  Of 5000 shapes that this rule sends elsewhere
// than the rule by rounds alone (1 to 40 times 4..2048 x 1..4096 x 64..1024, three sets of operands in turn) 25 take 1.02 to 1.15 of the time; without
// these lines 50 of 4500, up to 1.24.  The mean is 0.66 within the 128..1024 x 128..2048 x 128..512 of 1 to 12 entries, 0.38 of the others.  (7 x 832 x
// 384 x 489: 128 x 128 36, 64 x 64 31, 32 x 32 29.)  MI_GEMM_SMALL=0, read at every call, leaves all to that rule, and so does a forced tile.
bool small32_try(const Problem& p, int* big_tile, hipStream_t s) {
    static const bool forced = getenv("MI_GEMM_KERNEL") || getenv("MI_GEMM_BIG_TILE");
    if (forced || p.out_dtype != MI_F32 || p.M < 4 || p.K < 64 || p.K > 1024 || tiles_of(p, 64, 64) > 2048) return false;
    // (32-bit lane offsets within 64 rows, of rows that follow each other upwards in memory)
    if (p.lda < p.M || p.ldb < p.K || p.ldc < p.M || p.sa < 0 || p.sb < 0 || p.sc < 0 || p.lda >= (1 << 23) || p.ldb >= (1 << 23)) return false;
    const char* e = getenv("MI_GEMM_SMALL");
    if (e && atoi(e) == 0) return false;
    const bool mis = p.lda % 4 || p.ldb % 4 || (p.batch > 1 && (p.sa % 4 || p.sb % 4)) || !aligned(p.A, 16) || !aligned(p.B, 16);
    auto rounds = [&](int tm, int tn) { return (double)((tiles_of(p, tm, tn) + 255) / 256); };
    auto us = [&](double launch, double r, double ramp, double walked, double per_k, double k_mis) {
        return launch + r * (ramp + walked * per_k + (mis ? p.K * k_mis : 0.0));
    };
    const double k4 = (p.K + 4 * BK - 1) / (4 * BK) * (4.0 * BK), k64 = (p.K + 63) / 64 * 64.0;
    const double t11 = us(2.37 + 0.58e-3 * k4, rounds(32, 32), 0.56, k4, 3.40e-3, 0.63e-3);
    const double t21 = us(2.42 + 0.11e-3 * k4, rounds(64, 32), 0.77, k4, 7.77e-3, 1.45e-3);
    double other = 1e30, margin = 0.94;
    if (big32_applicable(p)) {
        const double b11 = us(2.40, rounds(64, 64), 0.77, k64, 14.46e-3, 1.86e-3);
        const double b22 = us(0.76, rounds(128, 128), 4.59, k64, 54.9e-3, 5.2e-3);
        const double b42 = us(1.55, rounds(256, 128), 7.36, k64, 107.3e-3, 7.4e-3);
        other = b11 < b22 && b11 < b42 ? b11 : b22 < b42 ? b22 : b42;
        *big_tile = other == b11 ? 11 : other == b22 ? 22 : 42;
        if (*big_tile == 11) margin = t11 > t21 ? (rounds(64, 32) == 3 ? 0.0 : 0.94) : rounds(32, 32) == 6 ? 0.0 : rounds(32, 32) == 5 ? 0.88 : 0.94;
    } else {
        other = us(2.5, rounds(128, 128), 2.8, p.K, 115e-3, 0.0);
    }
    if ((t11 < t21 ? t11 : t21) > margin * other) return false;
    const int kd = p.M % 4 ? (p.K - 1) / 4 * 4 : p.K / 4 * 4;
    if (t11 <= t21) launch<1, 1>(p, kd, s);
    else launch<2, 1>(p, kd, s);
    set_variant(t11 <= t21 ? "gemm32_small_32x32x32" : "gemm32_small_64x32x32");
    return true;
}

}  // namespace gemm
}  // namespace mi
