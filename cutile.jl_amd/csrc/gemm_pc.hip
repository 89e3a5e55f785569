// f16/bf16 GEMM whose transfers have waves of their own: C(M,N) = A(M,K) * B(K,N), column-major, fp32 accumulate, for
// operands whose rows start off 16-byte boundaries (an odd M or K).
//
// What bounds those products is the path into LDS, not the matrix cores: a CU brings 103-118 GB/s of aligned 16-byte chunks,
// 77 of chunks on 4-byte boundaries, 57 of any others, less where the lines come from memory, whatever is in flight.  On the
// kernel of gemm_big.hip a wave that asks for more than the path takes stands at the instruction and multiplies nothing
// meanwhile.  Here four waves only transfer and four only multiply, one of each per SIMD, which meet once per stage of 64 k;
// a stage's row of B is one 128-byte line where stages of 32 k ask for every line twice (64-byte runs: 70 GB/s against 94 on
// the mix of a 256 x 256 tile).  2999 x 2100 x 3001: transfers alone 55 us (56 with the fragments' reads as well: LDS itself is
// not short), products alone 33, together 61.
//
//   tile 128 x 128 (three stages of 32 KB) or 256 x 128 (of 48 KB), one workgroup per CU; a multiplying wave has 64 x 64 or
//   128 x 64 of it.  Layouts, fragments, edges and the register-fed step behind the last chunk of k are gemm_big.hip's, with
//   chunk c of row n of B at position c ^ ((n >> 1) & 7).
//
// Measured (us, gemm_big.hip -> this, one session): 2496 x 825 x 3247 35.4 -> 30.0, 3776 x 768 x 1459 18.6 -> 17.3, 2432 x 1536 x
// 2313 27.5 -> 25.4, 965 x 2048 x 3859 49.0 -> 42.3; 256 x 128 tiles 1946 x 2255 x 2995 45.8 -> 41.6, 2999 x 2100 x 3000 61.3 ->
// 58.1, 3000 x 2100 x 3001 52.9 -> 50.8, 2999 x 2100 x 3001, with both operands on 2-byte boundaries, 64.2 either way.  The rule
// stands in gemm_big.hip.  With aligned rows it is ahead or behind by up to 10 % without a pattern and is not used.
//
// Tried and not kept: A read straight into registers (4 bytes per lane and row of k, transposed by v_perm; no LDS for A): the
// 256 x 128 tile as fast as before, the 128 x 128 tile 15-20 % slower, as 4-byte requests take the path's time of 16-byte ones.
#include "gemm_direct.h"

namespace {

using namespace mi;
using namespace mi::gemm;

constexpr int BK = 64;        // k per stage: a row of B is one 128-byte line
constexpr int kStages = 3;

// Source of every chunk that lies past K.
__device__ __attribute__((aligned(16))) const unsigned zeros16c[4] = {0u, 0u, 0u, 0u};

// Tile (64*I) m x (64*J) n, a multiplying wave's part (32*I) x (32*J).
template <typename E, typename OutT, int I, int J>
__global__ __launch_bounds__(512) void gemm16_pc(const unsigned short* __restrict__ A, int64_t lda, int64_t sa, const unsigned short* __restrict__ B,
                                                 int64_t ldb, int64_t sb, OutT* __restrict__ C, int64_t ldc, int64_t sc, int M, int N, int K,
                                                 int tiles_m, int tiles_n, int batch, int kpeel) {
    // K: the extent the transfers walk (a multiple of 8); kpeel: values of k behind it for the register-fed step
    constexpr int BTM = 64 * I, BTN = 64 * J, kStageA = BTM * BK, kStage = kStageA + BTN * BK;
    __shared__ __attribute__((aligned(1024))) unsigned short ring[kStages * kStage];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int total = tiles_m * tiles_n, total_all = total * batch;
    int L = xcd_tile(blockIdx.x, total_all);
    const int bz = L / total;
    L -= bz * total;
    constexpr int GM = 4;
    const int per_group = GM * tiles_n;
    const int first_m = (L / per_group) * GM;
    const int gsz = tiles_m - first_m < GM ? tiles_m - first_m : GM;
    const int bm = first_m + (L % per_group) % gsz, bn = (L % per_group) / gsz;
    const int KD = (K + BK - 1) / BK;   // stages, >= 3 (checked on the host)
    A += (int64_t)bz * sa;
    B += (int64_t)bz * sb;

    if (wave >= 4) {
        // ---- transfers ----
        // A: 64 rows of 128*I bytes, 8*I transfers of 8/I rows, 2*I per wave; B: 64*J rows of 128 bytes, 8*J transfers of 8
        // rows, 2*J per wave.  Chunks of 8 m that start past the edge re-read the last chunk that starts inside, rows of B
        // past the edge the last row: what they bring reaches elements of C only that are never stored.
        const int w = wave - 4;
        const char *pA[2 * I], *pB[2 * J];
        int kA[2 * I], kB[2 * J];
#pragma unroll
        for (int j = 0; j < 2 * I; ++j) {
            const int k = (w + 4 * j) * (8 / I) + lane / (8 * I);
            int c = (lane % (8 * I)) ^ (4 * (k & 3));
            if (bm * BTM + 8 * c >= M) c = (M - 1 - bm * BTM) / 8;
            kA[j] = k;
            pA[j] = (const char*)(A + (int64_t)bm * BTM + 8 * c + k * lda);
        }
#pragma unroll
        for (int j = 0; j < 2 * J; ++j) {
            const int r = (w + 4 * j) * 8 + (lane >> 3);
            const int64_t n = (int64_t)bn * BTN + r < N ? (int64_t)bn * BTN + r : N - 1;
            const int c = (lane & 7) ^ ((r >> 1) & 7);
            kB[j] = 8 * c;
            pB[j] = (const char*)(B + n * ldb + 8 * c);
        }
        auto issue = [&](int d, int slot) {
            unsigned short* As = ring + slot * kStage + w * 512;
            unsigned short* Bs = As + kStageA;
            const int left = K - d * BK;
            if (left >= BK) {
#pragma unroll
                for (int j = 0; j < 2 * J; ++j) {
                    gload_lds16(pB[j], Bs + 2048 * j);
                    pB[j] += 2 * BK;
                }
#pragma unroll
                for (int j = 0; j < 2 * I; ++j) {
                    gload_lds16(pA[j], As + 2048 * j);
                    pA[j] += 2 * BK * lda;
                }
            } else {   // (the last stage)
#pragma unroll
                for (int j = 0; j < 2 * J; ++j) gload_lds16(kB[j] < left ? pB[j] : (const char*)zeros16c, Bs + 2048 * j);
#pragma unroll
                for (int j = 0; j < 2 * I; ++j) gload_lds16(kA[j] < left ? pA[j] : (const char*)zeros16c, As + 2048 * j);
            }
        };
        constexpr int PER = 2 * (I + J);   // transfers per wave and stage
        issue(0, 0);
        issue(1, 1);
        issue(2, 2);
        wait_vm<2 * PER>();
        meet();
        int slot = 0;
        for (int d = 0; d < KD; ++d) {
            // stage d + 1 has landed; stage d + 2 may be on its way
            if (d + 2 < KD) wait_vm<PER>();
            else wait_vm<0>();
            meet();
            if (d + 3 < KD) issue(d + 3, slot);
            slot = slot == kStages - 1 ? 0 : slot + 1;
        }
        return;
    }

    // ---- products ----
    struct Frag {
        s16x8 a[I], b[J];
    };
    const int wm = (wave & 1) * (32 * I), wn = (wave >> 1) * (32 * J);
    unsigned fb[4], fa[I];   // LDS element offsets of the fragments: B of sub-step u, A of m tile i (+ 16*u*BTM)
    {
        const int hb = lane >> 5, g = lane >> 4, r = lane & 15, n = wn + (lane & 31);
#pragma unroll
        for (int u = 0; u < 4; ++u) fb[u] = kStageA + n * BK + 8 * ((2 * u + hb) ^ ((n >> 1) & 7));
#pragma unroll
        for (int i = 0; i < I; ++i) {
            const int k = 8 * (g >> 1) + (r >> 2), m = wm + 32 * i + 16 * (g & 1) + 4 * (r & 3);
            fa[i] = k * BTM + 8 * ((m >> 3) ^ (4 * (r >> 2))) + (m & 7);
        }
    }
    f32x16 acc[I][J];
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
        for (int j = 0; j < J; ++j) acc[i][j] = f32x16{0};
    auto frags = [&](const unsigned short* S, int u, Frag& f) {
#pragma unroll
        for (int j = 0; j < J; ++j) f.b[j] = *reinterpret_cast<const s16x8*>(S + fb[u] + 32 * j * BK);
#pragma unroll
        for (int i = 0; i < I; ++i) {
            const unsigned short* p = S + fa[i] + 16 * u * BTM;
            const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(s16x4, p));
            const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(s16x4, p + 4 * BTM));
            f.a[i] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        }
    };
    auto mma = [&](const Frag& f) {
#pragma unroll
        for (int i = 0; i < I; ++i)
#pragma unroll
            for (int j = 0; j < J; ++j) acc[i][j] = E::mfma32(f.b[j], f.a[i], acc[i][j]);
    };
    auto spread = [&] {   // the 2*I + J reads of the next sub-step between the I*J MFMAs of this one
#pragma unroll
        for (int i = 0; i < I * J; ++i) {
            __builtin_amdgcn_sched_group_barrier(SG_MFMA, 1, 0);
            __builtin_amdgcn_sched_group_barrier(SG_DSRD, 1, 0);
            if (i < 2 * I + J - I * J) __builtin_amdgcn_sched_group_barrier(SG_DSRD, 1, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    Frag f0, f1;
    meet();
    frags(ring, 0, f0);
    int slot = 0;
    for (int d = 0; d < KD; ++d) {
        const unsigned short* S = ring + slot * kStage;
        slot = slot == kStages - 1 ? 0 : slot + 1;
        frags(S, 1, f1);
        mma(f0);
        spread();
        frags(S, 2, f0);
        mma(f1);
        spread();
        frags(S, 3, f1);
        mma(f0);
        spread();
        wait_lds();
        meet();
        frags(ring + slot * kStage, 0, f0);   // (behind the last stage: in bounds, unused)
        mma(f1);
        spread();
    }

    if (kpeel > 0) {   // (same for the whole grid)
        // k = K .. K + kpeel - 1 as the first values of one 16-wide MFMA step: the lower half-wave holds k 0..7 of its
        // row of B / column of A, the upper half-wave zeros.
        const unsigned short *Ap = A + (int64_t)K * lda, *Bp = B + K;
        Frag fp;
        const bool lower = lane < 32;
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const int64_t n = (int64_t)bn * BTN + wn + 32 * j + (lane & 31);
#pragma unroll
            for (int q = 0; q < 8; ++q) fp.b[j][q] = lower && q < kpeel && n < N ? (short)Bp[n * ldb + q] : (short)0;
        }
#pragma unroll
        for (int i = 0; i < I; ++i) {
            const int64_t m = (int64_t)bm * BTM + wm + 32 * i + (lane & 31);
#pragma unroll
            for (int q = 0; q < 8; ++q) fp.a[i][q] = lower && q < kpeel && m < M ? (short)Ap[m + (int64_t)q * lda] : (short)0;
        }
        mma(fp);
    }
    C += (int64_t)bz * sc;
    store_tile<E, OutT, I, J>(acc, C, ldc, M, N, bm * BTM, bn * BTN, wm, wn, BTM, BTN, lane);
}

}  // namespace

namespace mi {
namespace gemm {

void pc16_launch(const Problem& p, int tile, int kd, hipStream_t s) {
    const int btm = tile == 42 ? 256 : 128, tiles_m = (p.M + btm - 1) / btm, tiles_n = (p.N + 127) / 128;
    const dim3 grid((unsigned)(tiles_m * tiles_n * p.batch));
#define PC(E, O, I, J)                                                                                                                     \
    hipLaunchKernelGGL((gemm16_pc<E, O, I, J>), grid, dim3(512), 0, s, (const unsigned short*)p.A, p.lda, p.sa, (const unsigned short*)p.B, p.ldb, \
                       p.sb, (O*)p.C, p.ldc, p.sc, p.M, p.N, kd, tiles_m, tiles_n, p.batch, p.K - kd)
#define TILE(E, O)                         \
    do {                                   \
        if (tile == 42) PC(E, O, 4, 2);    \
        else PC(E, O, 2, 2);               \
    } while (0)
    const bool f32out = p.out_dtype == MI_F32;
    if (p.in_dtype == MI_F16) {
        if (f32out) TILE(F16, float);
        else TILE(F16, unsigned short);
    } else {
        if (f32out) TILE(BF16, float);
        else TILE(BF16, unsigned short);
    }
#undef TILE
#undef PC
}

}  // namespace gemm
}  // namespace mi
