// Token-gather grouped GEMM of the MoE for few tokens per expert (fused_moe_kernel, examples/moe.jl:45-105): the structure of
// gemm_small.hip on 32 sorted slots of an expert x 64 of its weight rows.  The four waves of a workgroup split K: wave w takes the
// stages w, w + 4, ... of 64 k (a stage row is a whole 128-byte line, 64 bytes of e4m3 weights), with an LDS area and accumulators of
// its own, reads a stage into registers, requests its next one into the same place and multiplies; no barrier before the sums
// are added in the order of the waves.
//
// What bounds these launches is a weight stream that no workgroup waits for: the streaming kernel (moe.hip) brings it through
// registers, one K step of all its waves in flight per workgroup and a barrier on either side of it; here every wave has 12 KB (e4m3: 8)
// under way on its own, three to four workgroups to a CU.  What it costs is a ramp per workgroup (ids, tokens, first stage): which
// launches are worth it stands at few_launch.
//
// e4m3 weights stay bytes in LDS and are widened, exactly, in front of their MFMAs.  Epilogues: plain, SiLU(gate) * up (tile 0 gate
// channels, tile 1 the up channels that go with them) with the slot in the lane, and accumulating with the channel pair in the lane
// (tile 0 even, tile 1 odd channels: one packed atomic per lane, a slot's 64 channels are 128 consecutive bytes).
//
// Measured (cutile_moe in us, weights from memory, before -> now): 256 tokens top-2 of 32 experts, 1024 x 2048 e4m3 52.0 -> 48.5 (the down
// projection alone), 768 top-2 of 64, 1024 x 1408 e4m3 91 -> 80, 64 top-2 of 8, 1024 x 1024 26.2 -> 23, 75 top-4 of 8, 1024 x 512 32 -> 24, 320 top-2 of
// 8, 512 x 512 e4m3 26 -> 19.  Tried and not kept: eight waves (1.0-1.8 of the time), non-temporal weights (1.04).
#include "gemm_small.h"
#include "moe_dense.h"
#include "moe_tiles.h"

namespace {

using namespace mi;
using namespace mi::gemm;
using mi::moe::DenseArgs;

constexpr int BK = 64;     // k per stage
constexpr int kTS = 32;    // slots per workgroup
constexpr int kTW = 64;    // weight rows per workgroup
constexpr int NW = kSplitWaves;
constexpr int MODE_PLAIN = 0, MODE_SILU = 1, MODE_ACC = 2;

// Source of every chunk that lies past K.
__device__ __attribute__((aligned(16))) const unsigned zeros16f[4] = {0u, 0u, 0u, 0u};

template <typename E, int MODE, bool W8>
__global__ __launch_bounds__(64 * NW) void moe_few_kernel(const DenseArgs a, int strips, int blocks) {
    constexpr int STAGE_T = kTS * BK * 2, STAGE_W = kTW * BK * (W8 ? 1 : 2), AREA = STAGE_T + STAGE_W;   // bytes
    constexpr int TT = STAGE_T / 1024, TW = STAGE_W / 1024;                                             // transfers per stage
    static_assert(AREA >= 8192, "a wave's sums fit its area");
    __shared__ __attribute__((aligned(1024))) char areas[NW * AREA];                                    // a wave's stage, and later its sums
    const int lane = threadIdx.x & 63, hb = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // Workgroup -> 32-slot tile and strip: the first tile of every block, then the second of every block, ... (those of a block behind
    // its last token are over at once), a tile's strips one after the other.
    const int per = blocks * strips, sub = blockIdx.x / per, r = blockIdx.x - sub * per, block = r / strips, strip = r - block * strips;
    const int slot0 = block * a.TILE_M + kTS * sub;
    const int expert = a.sorted_expert_ids[block] - 1;
    if (expert < 0 || expert >= a.num_experts || slot0 >= a.num_slots) return;
    int tok = 0;   // (1-based, 0 = none) of slot lane % 32
    if (slot0 + (lane & 31) < a.num_slots) tok = a.sorted_token_ids[slot0 + (lane & 31)];
    if (tok < 1 || tok > a.total_tokens) tok = 0;
    if (__ballot(tok != 0) == 0) return;

    // ---- transfers ---------------------------------------------------------------------------------------------------------
    const int half_n = a.N / 2, row0 = strip * (MODE == MODE_SILU ? kTW / 2 : kTW);
    const char* pT[TT];
    const char* pW[TW];
    int cT[2], cW;   // chunk of k: of even / odd token transfers (and 16-bit weight transfers) / of e4m3 weight transfers
#pragma unroll
    for (int e = 0; e < 2; ++e) cT[e] = (lane & 7) ^ ((4 * e + (lane >> 4)) & 7);
    cW = (lane & 3) ^ ((lane >> 4) & 3);
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        const int q = __shfl(tok, 8 * t + (lane >> 3), 64);
        const int col = q ? (q - 1) / a.replicas : 0;   // slots without a token read column 0
        pT[t] = (const char*)a.A + ((int64_t)col * a.lda + 8 * cT[t & 1]) * 2;
    }
    const char* const Bx = (const char*)a.B + (int64_t)expert * a.sbe * (W8 ? 1 : 2);
#pragma unroll
    for (int t = 0; t < TW; ++t) {
        const int R = W8 ? 16 * t + (lane >> 2) : 8 * t + (lane >> 3);   // row of the tile
        int row;
        if (MODE == MODE_SILU) {          // tile 0: gate channels, tile 1: the up channels that go with them
            int ch = row0 + (R & 31);
            if (ch > half_n - 1) ch = half_n - 1;
            row = R >= 32 ? half_n + ch : ch;
        } else {                          // accumulating: tile 0 the even channels of 64, tile 1 the odd ones
            row = row0 + (MODE == MODE_ACC ? 2 * (R & 31) + (R >> 5) : R);
            if (row > a.N - 1) row = a.N - 1;
        }
        pW[t] = W8 ? Bx + (int64_t)row * a.ldb + 16 * cW : Bx + ((int64_t)row * a.ldb + 8 * cT[t & 1]) * 2;
    }
    const unsigned lds0 = (unsigned)(size_t)LDS_PTR(char, areas) + wave * AREA;
    const int nk = (a.K + BK - 1) / BK;
    auto issue = [&](int c) __attribute__((always_inline)) {
        const int64_t ko = (int64_t)c * BK;
        const bool whole = BK * (c + 1) <= a.K;
        const int left = a.K - BK * c;
#pragma unroll
        for (int t = 0; t < TW; ++t) {
            const char* p = pW[t] + ko * (W8 ? 1 : 2);
            if (!whole && (W8 ? 16 * cW : 8 * cT[t & 1]) >= left) p = (const char*)zeros16f;
            load_lds_at(lds0 + STAGE_T + 1024 * t, p);
        }
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            const char* p = pT[t] + ko * 2;
            if (!whole && 8 * cT[t & 1] >= left) p = (const char*)zeros16f;
            load_lds_at(lds0 + 1024 * t, p);
        }
    };
    if (wave < nk) issue(wave);

    unsigned ft[4], fw[4];   // byte offsets of the fragments within a stage
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int row = lane & 31;
        ft[u] = row * (BK * 2) + 16 * ((2 * u + hb) ^ ((row >> 1) & 7));
        fw[u] = W8 ? STAGE_T + row * BK + 16 * (u ^ ((row >> 2) & 3)) + 8 * hb : STAGE_T + ft[u];
    }
    f32x16 acc[2] = {f32x16{0}, f32x16{0}};
    const char* const S = areas + wave * AREA;
    for (int c = wave; c < nk; c += NW) {
        wait_vm<0>();
        s16x8 t[4], w[4][2];
        u32x2 w8[4][2];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            t[u] = *reinterpret_cast<const s16x8*>(S + ft[u]);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                if constexpr (W8) w8[u][j] = *reinterpret_cast<const u32x2*>(S + fw[u] + 32 * j * BK);
                else w[u][j] = *reinterpret_cast<const s16x8*>(S + fw[u] + 32 * j * BK * 2);
            }
        }
        if (c + NW < nk) {
            wait_lds();
            asm volatile("" ::: "memory");
            issue(c + NW);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const s16x8 wf = W8 ? mi::moe::widen_e4m3<E>(w8[u][j]) : w[u][j];
                acc[j] = MODE == MODE_ACC ? E::mfma32(t[u], wf, acc[j]) : E::mfma32(wf, t[u], acc[j]);
            }
    }

    // ---- the waves' sums, added in their order; wave q takes register group q of both tiles -------------------------------------
    char* const mine = areas + wave * AREA;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            *reinterpret_cast<f32x4*>(mine + ((4 * j + q) * 64 + lane) * 16) = f32x4{acc[j][4 * q], acc[j][4 * q + 1], acc[j][4 * q + 2], acc[j][4 * q + 3]};
    __syncthreads();
    f32x4 v[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        v[j] = *reinterpret_cast<const f32x4*>(areas + ((4 * j + wave) * 64 + lane) * 16);
#pragma unroll
        for (int x = 1; x < NW; ++x) v[j] += *reinterpret_cast<const f32x4*>(areas + x * AREA + ((4 * j + wave) * 64 + lane) * 16);
    }
    auto weight_of = [&](int tk) {
        float wt = 1.f;
        if (a.mul_routed_weight && tk) {
            const int q = tk - 1, t = q / a.w_topk;
            wt = mi::moe::widen16(a.bf16, a.topk_weights[t * a.w_s0 + (q - t * a.w_topk) * a.w_s1]);
        }
        return wt;
    };
    const float* const scale = W8 ? a.b_scale + (int64_t)expert * a.ld_scale : nullptr;
    if constexpr (MODE == MODE_ACC) {
        // lane = channel pair, rows = slots 8 * wave + 4 * hb + e: a half-wave adds a slot's 64 channels, 128 consecutive bytes
        const int gn = row0 + 2 * (lane & 31);
        const float s0 = W8 && gn < a.N ? scale[gn] : 1.f, s1 = W8 && gn + 1 < a.N ? scale[gn + 1] : 1.f;
        const float wt = weight_of(tok);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int slot = 8 * wave + 4 * hb + e;
            const int tk = __shfl(tok, slot, 64);
            const float wl = __shfl(wt, slot, 64);
            float x = v[0][e], y = v[1][e];
            if (W8) {
                x *= s0;
                y *= s1;
            }
            if (a.mul_routed_weight) {
                x *= wl;
                y *= wl;
            }
            if (tk && gn < a.N) mi::moe::atomic_add2(a.bf16, a.C + gn + (int64_t)((tk - 1) >> a.acc_shift) * a.ldc, E::pack(x, y));
        }
    } else {
        // lane = slot, channels 8 * wave + 4 * hb + e of the tile
        const float wt = weight_of(tok);
        const int ch = 8 * wave + 4 * hb;
        unsigned short* const rowp = a.C + (int64_t)(tok ? tok - 1 : 0) * a.ldc;
        auto put = [&](const float (&o)[4], int n0, int n) {
            if (!tok) return;
            if (n0 + 4 <= n && a.ldc % 4 == 0 && ((uintptr_t)a.C & 7) == 0) {
                *reinterpret_cast<u32x2*>(rowp + n0) = u32x2{E::pack(o[0], o[1]), E::pack(o[2], o[3])};
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n0 + e < n) rowp[n0 + e] = E::from_f32(o[e]);
            }
        };
        if constexpr (MODE == MODE_SILU) {
            const int n0 = row0 + ch;
            float o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float g = v[0][e], u = v[1][e];
                if (W8 && n0 + e < half_n) {
                    g *= scale[n0 + e];
                    u *= scale[half_n + n0 + e];
                }
                g *= wt;
                u *= wt;
                o[e] = mi::moe::silu_mul(E::round(g), E::round(u));
            }
            put(o, n0, half_n);
        } else {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int n0 = row0 + 32 * j + ch;
                float o[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    o[e] = v[j][e];
                    if (W8 && n0 + e < a.N) o[e] *= scale[n0 + e];
                    o[e] *= wt;
                }
                put(o, n0, a.N);
            }
        }
    }
}

}  // namespace

namespace mi {
namespace moe {

// True where this kernel is the one to take; launches it.  `live`: tiles of 32 slots that hold tokens, about; with their strips of 64
// rows they are the workgroups that do something (`work`).  Measured as whole calls of cutile_moe with weights that come from memory, this
// kernel : the ones that take the launch otherwise, f16 and bf16 and e4m3, 500 shapes of 8 to 64 experts, 512 or 1024 hidden and 512 to 2048
// inter and 340 of up to 256 experts, 7168 hidden and 4096 inter.  Below 32 tokens per expert a weight row is read once, and
//  * the first projection runs otherwise on the streaming kernel's wide strips, which are ahead from about 700 workgroups on, as the ramp
//    of a second round is: up to 512 of them -1.1 us in the mean (-3.5 to +1.3), 1024 +2.1, 2048 and more +6 (16-bit weights of 1024 hidden
//    in just 512: 31.4 : 34.4, e4m3 of 7168 106 : 102);
//  * the second one (the launch that multiplies by the routed weights) on 32- or 64-channel strips whose waves split K between two barriers:
//    -1.8 us in the mean up to 1024 workgroups (1312 56 : 64 and 1536 80 : 83 with less than a token per expert), and behind from
//    1800 on (2048 and more 1.02-1.17 of the call, 28672, 256 experts of 7168, 975 : 909).  Where its lines lie is measured and no more:
//    16-bit rows of 4 KB pay from 192 to 511 workgroups (32 experts, 1024 of 2048, 512 of them +4.5; 256 -0.9 to -1.8; 8 experts, 128 of
//    them, 12 and 18 tokens each +0.3 and +0.7), rows of 8 KB never (256 workgroups 75 : 70 and 97 : 91); e4m3 rows of 4 KB below 512 (64
//    experts, 1024 of them, 172 : 157), of 2 KB where the other kernel runs on its 64-channel strips below 1024 (87 : 84).
// From 32 tokens per expert on a strip is read once per 32 slots and not per 128: up to 450 workgroups with e4m3 weights, 352 with others (432
// tokens top-2 of 16, K = 1408 e4m3 33 : 29, 224 top-2 of 8 35 : 28, 512 top-2 of 16, 320 workgroups, 46 : 37; but 256 top-4 of 32, 384
// workgroups, K = 1024 and 1408 37.2 : 38.0 and 46.2 : 47.5, K = 512 and 2048 30.2 : 29.3 and 63.6 : 59.6; 283 top-4, 816, 93 : 103), 320 with
// rows of 4 KB (8 experts, 70 to 75 tokens each, 336 and 352 workgroups 42.7 : 41).
// With these lines no shape of the 500 takes more than 1.02 of what it took without this kernel, of the 340 none more than 1.025.
// The line is the same for every epilogue of a projection, so fused and separate launches of a call add in the same order.  MI_MOE_FEW=0,
// read at every call, and the settings that force another kernel or a shape of one (MI_MOE_DENSE*, MI_MOE_PREFILL) switch it off.
bool few_launch(const DenseArgs& a, hipStream_t s) {
    const char* env = getenv("MI_MOE_FEW");
    if (a.a8 || (env && atoi(env) == 0)) return false;
    for (const char* forced : {"MI_MOE_DENSE", "MI_MOE_PREFILL", "MI_MOE_DENSE_J", "MI_MOE_DENSE_WIDE", "MI_MOE_DENSE_STREAM"})
        if (getenv(forced)) return false;
    const int per16 = a.w8 ? 16 : 8;   // weights per 16-byte chunk
    if (a.TILE_M % kTS || a.K % per16 || a.K < 256 || a.N < 1 || (a.silu && a.N % 2)) return false;
    if (!aligned(a.A, 16) || !aligned(a.B, 16) || a.lda % 8 || a.ldb % per16 || a.sbe % per16 || a.lda < 0 || a.ldb < 0) return false;
    if (cld((int64_t)a.total_tokens, (int64_t)a.replicas) > a.num_a_cols) return false;   // (a replica without a column of A: the streaming kernel feeds it zeros)
    const int strips = a.silu ? (int)cld((int64_t)a.N / 2, (int64_t)32) : (int)cld((int64_t)a.N, (int64_t)64);
    const int64_t wgs = (int64_t)a.num_blocks * (a.TILE_M / kTS) * strips;
    if (wgs > MI_MAX_GRID_DIM) return false;
    const bool once = a.total_tokens < 32ll * a.num_experts;
    const int64_t live = !once ? a.total_tokens / 32 + a.num_experts / 2 : a.total_tokens < a.num_experts ? a.total_tokens : a.num_experts;
    const int64_t work = live * strips;
    const int64_t row = a.ldb * (a.w8 ? 1 : 2);   // bytes
    if (!once) {
        if (work > (a.w8 ? 450 : row >= 4096 ? 320 : 352)) return false;
    } else if (!a.mul_routed_weight) {
        if (work > (a.w8 && row < 4096 ? 512 : 480)) return false;
    } else {
        if (work > 1280 || (row >= 4096 && work >= 512)) return false;
        if (a.w8 ? row >= 2048 && a.K % 256 == 0 && work >= 1024 : row >= 8192 || (row >= 4096 && work < 192)) return false;
    }
#define LAUNCH(ET, MODE)                                                                                                                     \
    do {                                                                                                                                     \
        if (a.w8) hipLaunchKernelGGL((moe_few_kernel<ET, MODE, true>), dim3((unsigned)wgs), dim3(64 * NW), 0, s, a, strips, a.num_blocks);   \
        else hipLaunchKernelGGL((moe_few_kernel<ET, MODE, false>), dim3((unsigned)wgs), dim3(64 * NW), 0, s, a, strips, a.num_blocks);       \
    } while (0)
    if (a.silu) {
        if (a.bf16) LAUNCH(BF16, MODE_SILU);
        else LAUNCH(F16, MODE_SILU);
        set_variant(a.w8 ? "fused_moe_few_silu_t32_n32x2_k64_ksplit4_w8a16" : "fused_moe_few_silu_t32_n32x2_k64_ksplit4");
    } else if (a.acc_shift >= 0) {
        if (a.bf16) LAUNCH(BF16, MODE_ACC);
        else LAUNCH(F16, MODE_ACC);
        set_variant(a.w8 ? "fused_moe_few_acc_t32_n64_k64_ksplit4_w8a16" : "fused_moe_few_acc_t32_n64_k64_ksplit4");
    } else {
        if (a.bf16) LAUNCH(BF16, MODE_PLAIN);
        else LAUNCH(F16, MODE_PLAIN);
        set_variant(a.w8 ? "fused_moe_few_t32_n64_k64_ksplit4_w8a16" : "fused_moe_few_t32_n64_k64_ksplit4");
    }
#undef LAUNCH
    return true;
}

}  // namespace moe
}  // namespace mi
