// Token-gather grouped GEMM of the MoE for prefill sizes (fused_moe_kernel, examples/moe.jl:45-105): the products of
// moe_dense.hip with waves of their own for the transfers.
//
// What bounds it: the transfers into LDS at the latency of memory.  A CU brings 118 GB/s of whole, aligned 128-byte lines from
// the L2 (50-70 in runs of 64 bytes), but requests are answered in order, and token rows that the L2 has wait behind weight
// lines that it has not: 40-46 GB/s here.  On the ring kernel of moe_dense.hip, whose waves multiply and transfer, a wave that
// asks for more than the path takes stands at the instruction, and that time is lost to the matrix cores.  Here a workgroup
// (one per CU, persistent) is four waves that only transfer and four that only multiply, one of each per SIMD, which meet once
// per stage of 64 k, so a stage's rows are whole lines.  4096 tokens top-2 of 32 experts, evenly routed (1024 hidden, 2048 inter,
// gate / up + down projection): without products 78 + 41 us, 7 of the latter the packed atomics of the one round's
// end, without transfers 70 + 42, together 93 + 51.  The ring kernel takes 115 + 66.
//
//   tile = up to 160 slots x 256 weight rows, a wave all slots x 64 rows (10 MFMA 32x32x16 tiles), or up to 192 slots x 128
//   rows, a wave every second 32-slot sub-tile x 64 rows; three stages of 52 / 40 KB.  A launch picks one of the two from the table
//   of runs below.
//
// Slots are dealt in 32-slot sub-tiles and not in blocks of 128: an expert's run of blocks is cut evenly into as few tiles as
// hold its sub-tiles with tokens (a table of runs that every workgroup makes at its start, 2.4 us).  At 256 +- 16 slots per
// expert that is two tiles of 4 or 5 sub-tiles where blocks of 128 make two or three.  The tiles of a run are numbered
// strip-major, so the workgroups of an XCD share weight strips and token rows in its L2.
//
// A stage: rows of 128 bytes, 16-byte chunk c of row r at position c ^ ((r >> 1) & 7), fragments are plain 16-byte reads
// without conflicts; chunks past K come from a block of zeros.  The transfer waves run up to three stages ahead, into the
// next tile while this one is stored.  At the barrier of stage s the products of its last quarter are all that is left of
// it, stage s + 1 has landed, and stage s + 3 may be requested into its place.
// k is walked in ascending order with the k <-> lane map of the other kernels: the same bits.
//
// Tried and not kept: four stages of 36 KB, fragments two quarters ahead, one copy of the epilogue's code in a loop (all
// without effect); 128 weight rows and at most 128 slots (slower wherever the ring kernel is not the better one).
#include "gemm_direct.h"
#include "moe_dense.h"
#include "moe_tiles.h"

namespace {

using namespace mi;
using namespace mi::gemm;
using mi::moe::DenseArgs;

constexpr int BK = 64;                       // k per stage: a stage row is one 128-byte line
constexpr int kStages = 3;
constexpr int kMaxRuns = 112;                // runs of blocks of one expert that the table holds
constexpr int kMaxBlocks = 4096;             // blocks of TILE_M slots that the setup looks at
constexpr int kBlock = 128;                  // slots per tile where there are more runs than that
constexpr int MODE_PLAIN = 0, MODE_SILU = 1, MODE_ACC = 2;

// Source of every chunk that lies past K.
__device__ __attribute__((aligned(16))) const unsigned zeros16p[4] = {0u, 0u, 0u, 0u};

// waits until at most the transfers of the youngest STAGES stages, W + live sub-tiles each, are in flight
template <int STAGES, int W>
__device__ __forceinline__ void wait_transfers(int live) {
    if (live == 6) wait_vm<(W + 6) * STAGES>();
    else if (live == 5) wait_vm<(W + 5) * STAGES>();
    else if (live == 4) wait_vm<(W + 4) * STAGES>();
    else if (live == 3) wait_vm<(W + 3) * STAGES>();
    else if (live == 2) wait_vm<(W + 2) * STAGES>();
    else if (live == 1) wait_vm<(W + 1) * STAGES>();
    else wait_vm<0>();
}

struct Tile {
    int slot0, live, strip, expert;   // first slot, 32-slot sub-tiles, strip of weight rows, expert (0-based)
};

constexpr int max_live(int wc) { return wc == 4 ? 5 : 6; }          // sub-tiles of 32 slots per tile at most
constexpr int stage_of(int wc) { return (32 * max_live(wc) + 64 * wc) * BK; }   // elements of a stage
constexpr int kSlotsMax = 32 * max_live(2);

// The runs of blocks of one expert.
struct Runs {
    const int *first, *slot, *live;   // (LDS) of every run: its first tile, its first slot, its 32-slot sub-tiles up to its last token | expert << 16
    int runs, tiles;                  // their number (-1: one tile per 128 slots), and the tiles of all
};

// WC: groups of 64 weight rows, one or two waves each (WS slot groups).
template <typename E, int MODE, int WC>
__device__ __forceinline__ void walk_tiles(const DenseArgs& a, int strips, const Runs& table, unsigned short* ring, int (*s_tok)[kSlotsMax], float* s_wt) {
    constexpr int WS = 4 / WC, kMaxL = max_live(WC), kRows = (kMaxL + WS - 1) / WS;      // sub-tiles of 32 slots per tile / per wave at most
    constexpr int kW = 64 * WC;                                                          // weight rows per tile
    constexpr int kSlots = 32 * kMaxL;
    constexpr int kStageT = kSlots * BK, kStage = kStageT + kW * BK;   // elements of a stage's token part / of a stage
    static_assert(kStage == stage_of(WC), "the ring holds the stages");
    struct Frags {
        s16x8 t[kRows], w[2];
    };
    const int tid = threadIdx.x, lane = tid & 63, hb = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int runs = table.runs, tiles_all = table.tiles;
    const int *const r_first = table.first, *const r_slot = table.slot, *const r_live = table.live;
    const int first0 = lane < runs ? r_first[lane] : 0x7fffffff, first1 = lane + 64 < runs ? r_first[lane + 64] : 0x7fffffff;

    // Workgroup ids congruent mod 8 share an XCD; XCD x takes tiles [x * per, (x + 1) * per), its workgroups with a stride.
    const int per = (tiles_all + 7) >> 3, stride = gridDim.x >> 3;
    const int lo = (blockIdx.x & 7) * per, hi = lo + per < tiles_all ? lo + per : tiles_all;
    const int it0 = lo + (int)(blockIdx.x >> 3);
    if (it0 >= hi) return;

    // Tile idx: the tiles of a run are numbered strip-major, so the workgroups of an XCD work on a few strips of all of an
    // expert's slots at a time.  A run's sub-tiles are dealt to its tiles evenly.
    auto decode = [&](int idx) {
        Tile t;
        if (runs >= 0) {
            const int r = __popcll(__ballot(first0 <= idx)) + __popcll(__ballot(first1 <= idx)) - 1;
            const int le = __builtin_amdgcn_readfirstlane(r_live[r]), live = le & 0xffff;
            const int nt = (live + kMaxL - 1) / kMaxL;
            const int x = idx - __builtin_amdgcn_readfirstlane(r_first[r]);
            t.strip = x / nt;
            const int i = x - t.strip * nt, each = live / nt, more = live - each * nt;
            t.live = each + (i < more ? 1 : 0);
            t.slot0 = __builtin_amdgcn_readfirstlane(r_slot[r]) + 32 * (i * each + (i < more ? i : more));
            t.expert = le >> 16;
        } else {
            const int b = idx / strips;
            t.strip = idx - b * strips;
            t.live = kBlock / 32;
            t.slot0 = b * kBlock;
            t.expert = __builtin_amdgcn_readfirstlane(a.sorted_expert_ids[t.slot0 / a.TILE_M]) - 1;
        }
        return t;
    };
    const int KD = (a.K + BK - 1) / BK;   // stages per tile, >= 4 (K >= 256 is checked on the host)
    // token (1-based, 0 = none) of slot `i` of a tile, from what sorted_token_ids holds there
    auto fix = [&](const Tile& t, int i, int raw) {
        return (i < 32 * t.live && t.expert >= 0 && t.expert < a.num_experts && t.slot0 + i < a.num_slots && raw >= 1 && raw <= a.total_tokens) ? raw : 0;
    };
    auto raw_token = [&](const Tile& t, int i) {
        const int s = t.slot0 + (i < 32 * t.live ? i : 0);
        return a.sorted_token_ids[s < a.num_slots ? s : a.num_slots - 1];
    };

    Tile cur = decode(it0);
    if (tid < kSlots) s_tok[0][tid] = fix(cur, tid, raw_token(cur, tid));
    __syncthreads();

    if (wave >= 4) {
        // ---- transfers ----
        const int w = wave - 4;
        const int row = 8 * w + (lane >> 3);                                  // of every 32 rows
        const int chunk = (lane & 7) ^ ((4 * w + (lane >> 4)) & 7);           // 16-byte chunk that belongs at this lane's position
        constexpr int NW = 2 * WC;                                            // weight transfers per wave and stage
        const int ntiles = (hi - 1 - it0) / stride + 1, total = ntiles * KD;
        int it = it0, d = 0, slot = 0, p = 0;
        Tile t = cur;
        const unsigned lda2 = (unsigned)a.lda * 2, ldb2 = (unsigned)a.ldb * 2, half_n = a.N / 2;
        const int shift = (a.replicas & (a.replicas - 1)) == 0 ? __builtin_ctz(a.replicas) : -1;
        // byte offsets of the lane's chunks: of its slots' columns of A, of its rows of a strip (constant but for the rows
        // of a last strip that lie past the edge and re-read the last row)
        unsigned oT[kMaxL], oW[NW];
        const char* Bx = nullptr;
        int clipped = 1;
        auto setup = [&] {
#pragma unroll
            for (int j = 0; j < kMaxL; ++j) {
                const int tok = s_tok[p][32 * j + row];
                const unsigned q = tok ? tok - 1 : 0;                         // slots without a token read column 0
                oT[j] = (shift >= 0 ? q >> shift : q / (unsigned)a.replicas) * lda2 + 16 * chunk;
            }
            const int e = t.expert >= 0 && t.expert < a.num_experts ? t.expert : 0;
            const int row0 = t.strip * (MODE == MODE_SILU ? kW / 2 : kW), rows = MODE == MODE_SILU ? half_n : a.N;
            Bx = (const char*)a.B + (int64_t)e * a.sbe * 2 + (int64_t)row0 * ldb2;
            const int clip = row0 + (MODE == MODE_SILU ? kW / 2 : kW) > rows;
            if (clip | clipped) {
#pragma unroll
                for (int j = 0; j < NW; ++j) {
                    // tile row R: channel group R / 64, MFMA tile (R / 32) % 2 of it, channel R % 32 of that; with the SiLU
                    // epilogue a group's tile 0 is 32 gate channels and its tile 1 the up channels that go with them
                    const int R = 32 * j + row;
                    // (accumulating: tile 0 is the even and tile 1 the odd channels of 64, so that a lane holds adjacent pairs)
                    int r = MODE == MODE_SILU ? 32 * (R >> 6) + (R & 31) : MODE == MODE_ACC ? (R & ~63) + 2 * (R & 31) + ((R >> 5) & 1) : R;
                    if (row0 + r > rows - 1) r = rows - 1 - row0;
                    if (MODE == MODE_SILU && ((R >> 5) & 1)) r += half_n;
                    oW[j] = (unsigned)r * ldb2 + 16 * chunk;
                }
            }
            clipped = clip;
        };
        setup();
        auto issue = [&] {   // the next stage; returns its live sub-tiles
            unsigned short* S = ring + slot * kStage + w * 512;
            const int live = t.live;
            if ((d + 1) * BK <= a.K) {
                const int64_t ko = (int64_t)d * (BK * 2);
#pragma unroll
                for (int j = 0; j < NW; ++j) gload_lds16(Bx + ko + oW[j], S + kStageT + 2048 * j);
#pragma unroll
                for (int j = 0; j < kMaxL; ++j)
                    if (j < live) gload_lds16((const char*)a.A + ko + oT[j], S + 2048 * j);
            } else {
                const int64_t ko = (int64_t)d * (BK * 2);
                const bool in = d * BK + 8 * chunk < a.K;
#pragma unroll
                for (int j = 0; j < NW; ++j) gload_lds16(in ? Bx + ko + oW[j] : (const char*)zeros16p, S + kStageT + 2048 * j);
#pragma unroll
                for (int j = 0; j < kMaxL; ++j)
                    if (j < live) gload_lds16(in ? (const char*)a.A + ko + oT[j] : (const char*)zeros16p, S + 2048 * j);
            }
            slot = slot == kStages - 1 ? 0 : slot + 1;
            if (++d == KD) {
                d = 0;
                it += stride;
                p ^= 1;
                if (it < hi) t = decode(it);
            }
            return live;
        };
        issue();
        issue();
        int youngest = issue();   // (KD >= 4: three stages of one tile)
        wait_transfers<2, NW>(youngest);
        meet();
        for (int q = 0; q < total; ++q) {
            wait_transfers<1, NW>(q + 2 < total ? youngest : 0);
            meet();
            if (q + kStages < total) {
                if (d == 0) setup();
                youngest = issue();
            }
        }
        return;
    }

    // ---- products ----
    constexpr bool SL = MODE != MODE_ACC;
    unsigned fo[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) fo[u] = (lane & 31) * BK + 8 * ((2 * u + hb) ^ (((lane & 31) >> 1) & 7));
    const int wc = wave % WC, ws = wave / WC;   // the wave's channel group; its sub-tiles are ws, ws + WS, ...
    const unsigned short* const ringW = ring + kStageT + 64 * wc * BK;
    const unsigned short* const ringT = ring + 32 * ws * BK;
    const bool vec_ok = ((uintptr_t)a.C % 16) == 0 && a.ldc % 8 == 0;
    int slot = 0, p = 0;
    meet();
    for (int it = it0;; it += stride) {
        f32x16 acc[kRows][2];
#pragma unroll
        for (int i = 0; i < kRows; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] = f32x16{0};
        const bool have_next = it + stride < hi;
        Tile nxt = cur;
        int rawN = 0;
        float wt = 1.f;
        if (have_next) nxt = decode(it + stride);
        if (tid < kSlots) {
            if (have_next) rawN = raw_token(nxt, tid);
            const int tm = s_tok[p][tid];
            if (a.mul_routed_weight && tm) {
                // weight of replica q = token * w_topk + slot: element (token, slot) of the (num_tokens, topk) matrix
                const int q = tm - 1, tk = q / a.w_topk;
                wt = mi::moe::widen16(a.bf16, a.topk_weights[tk * a.w_s0 + (q - tk * a.w_topk) * a.w_s1]);
            }
        }
        auto walk = [&](auto LV) {
            constexpr int L = decltype(LV)::value;
            Frags f0, f1;
            auto frags = [&](int s, int u, Frags& f) {
                const unsigned short* T = ringT + s * kStage + fo[u];
                const unsigned short* W = ringW + s * kStage + fo[u];
#pragma unroll
                for (int j = 0; j < 2; ++j) f.w[j] = *reinterpret_cast<const s16x8*>(W + 32 * j * BK);
#pragma unroll
                for (int i = 0; i < L; ++i) f.t[i] = *reinterpret_cast<const s16x8*>(T + 32 * WS * i * BK);
            };
            auto mma = [&](const Frags& f) {
#pragma unroll
                for (int i = 0; i < L; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) acc[i][j] = SL ? E::mfma32(f.w[j], f.t[i], acc[i][j]) : E::mfma32(f.t[i], f.w[j], acc[i][j]);
#pragma unroll
                for (int i = 0; i < 2 * L; ++i) {
                    __builtin_amdgcn_sched_group_barrier(SG_MFMA, 1, 0);
                    if (i < L + 2) __builtin_amdgcn_sched_group_barrier(SG_DSRD, 1, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            };
            frags(slot, 0, f0);
            for (int d = 0; d < KD; ++d) {
                const int s = slot;
                slot = slot == kStages - 1 ? 0 : slot + 1;
                frags(s, 1, f1);
                mma(f0);
                frags(s, 2, f0);
                mma(f1);
                frags(s, 3, f1);
                mma(f0);
                if (d == KD - 3 && have_next && tid < kSlots) s_tok[p ^ 1][tid] = fix(nxt, tid, rawN);
                if (d == KD - 2 && tid < kSlots) s_wt[tid] = wt;
                wait_lds();
                meet();
                frags(slot, 0, f0);   // (behind the last stage: in bounds, unused)
                mma(f1);
            }
        };
        const int rows = (cur.live - ws + WS - 1) / WS;
        switch (rows) {
            case 0: walk(std::integral_constant<int, 0>{}); break;
            case 1: walk(std::integral_constant<int, 1>{}); break;
            case 2: walk(std::integral_constant<int, 2>{}); break;
            case 3: walk(std::integral_constant<int, 3>{}); break;
            case 4: if constexpr (kRows > 3) walk(std::integral_constant<int, 4>{}); break;
            default: if constexpr (kRows > 3) walk(std::integral_constant<int, 5>{}); break;
        }
#pragma unroll
        for (int i = 0; i < kRows; ++i) {
            if (i >= rows) break;
            const int first = 32 * (ws + WS * i);   // slot of the tile
            const int tokv = MODE != MODE_ACC ? s_tok[p][first + (lane & 31)] : 0;
            const float wtv = MODE != MODE_ACC ? s_wt[first + (lane & 31)] : 1.f;
            if (MODE != MODE_ACC && a.mul_routed_weight) {
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[i][j][r] *= wtv;
            }
            if constexpr (MODE == MODE_SILU) {
                const int ch0 = cur.strip * (kW / 2) + 32 * wc;
                float o[16];
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    // (both halves rounded as the unfused GEMM stores them)
                    o[r] = mi::moe::silu_mul(E::round(acc[i][0][r]), E::round(acc[i][1][r]));
                }
                mi::moe::store_tile_slot_lane<E>(o, a.C + (int64_t)(tokv ? tokv - 1 : 0) * a.ldc + ch0, tokv != 0, a.N / 2 - ch0, vec_ok, hb);
            } else if constexpr (MODE == MODE_PLAIN) {
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const int ch0 = cur.strip * kW + 64 * wc + 32 * j;
                    float o[16];
#pragma unroll
                    for (int r = 0; r < 16; ++r) o[r] = acc[i][j][r];
                    mi::moe::store_tile_slot_lane<E>(o, a.C + (int64_t)(tokv ? tokv - 1 : 0) * a.ldc + ch0, tokv != 0, a.N - ch0, vec_ok, hb);
                }
            } else {
                // lane = channel pair; rows of a tile = slots 8 * (r / 4) + 4 * hb + r % 4: a half-wave adds a slot's 64 channels,
                // 128 consecutive bytes, with one packed atomic per lane
                typedef int i32x4_ __attribute__((ext_vector_type(4)));
                const int gn = cur.strip * kW + 64 * wc + 2 * (lane & 31);
                unsigned short* const col = a.C + gn;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const i32x4_ t4 = *reinterpret_cast<const i32x4_*>(&s_tok[p][first + 8 * q + 4 * hb]);
                    const f32x4 w4 = *reinterpret_cast<const f32x4*>(&s_wt[first + 8 * q + 4 * hb]);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        float v0 = acc[i][0][4 * q + e], v1 = acc[i][1][4 * q + e];
                        if (a.mul_routed_weight) {
                            v0 *= w4[e];
                            v1 *= w4[e];
                        }
                        if (t4[e] && gn < a.N) mi::moe::atomic_add2(a.bf16, col + (int64_t)((t4[e] - 1) >> a.acc_shift) * a.ldc, E::pack(v0, v1));
                    }
                }
            }
        }
        if (!have_next) break;
        cur = nxt;
        p ^= 1;
    }
}

// `rows`: 256 or 128 weight rows per tile, or 0 for whichever is the quicker with the routing at hand, which is known here only:
// 128 where they make no more rounds of the CUs than 256 (as many rounds: 0.82 of the time of 256; two for one: 1.23; 3600 launches
// of 360 shapes, from even to very uneven routing).  A few tiles more than CUs are a second round, and uneven routing has them
// where even routing has not: 32 experts of 256, 2048 -> 1024, take 50 us with 256 rows, one round; with experts of 150 to 540
// they are 270 tiles and take 73, with 128 rows 56.
template <typename E, int MODE>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void moe_prefill_kernel(const DenseArgs a, int strips4, int strips2, int rows) {
    constexpr int kRing = kStages * (stage_of(4) > stage_of(2) ? stage_of(4) : stage_of(2));
    __shared__ __attribute__((aligned(1024))) unsigned short ring[kRing];
    __shared__ __attribute__((aligned(16))) int s_tok[2][kSlotsMax];   // 1-based replica id of every slot of the tile (two tiles), 0 = no token
    __shared__ __attribute__((aligned(16))) float s_wt[kSlotsMax];     // its routed weight
    __shared__ int r_first[kMaxRuns], r_slot[kMaxRuns], r_live[kMaxRuns];
    __shared__ int s_runs, s_tiles, s_wide, s_cnt[8];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    auto rounds = [](int tiles) { return (((tiles + 7) >> 3) + 31) >> 5; };
    auto choose = [&](int tiles4, int tiles2) { return rows ? rows == 256 : rounds(tiles2) > rounds(tiles4); };

    // ---- the runs of blocks of one expert, and how many of a run's sub-tiles hold tokens ----
    const int nb = a.num_blocks;
    {
        int* ids = (int*)ring;                        // [nb] expert of every block, 0 = none
        int* r_end = (int*)ring + kMaxBlocks;         // [kMaxRuns] last block of a run
        for (int b = tid; b < nb; b += 512) {
            const int e = a.sorted_expert_ids[b];
            ids[b] = e >= 1 && e <= a.num_experts ? e : 0;
        }
        if (tid < kMaxRuns) r_live[tid] = 0;
        __syncthreads();
        int base = 0;
        for (int c = 0; c < nb; c += 512) {
            const int b = c + tid;
            const int e = b < nb ? ids[b] : 0;
            const bool start = e && (b == 0 || ids[b - 1] != e);
            const bool end = e && (b == nb - 1 || ids[b + 1] != e);
            const unsigned long long m = __ballot(start);
            if (lane == 0) s_cnt[wave] = __popcll(m);
            __syncthreads();
            int before = base;
            for (int w = 0; w < 8; ++w) {
                if (w < wave) before += s_cnt[w];
                base += s_cnt[w];
            }
            const int upto = before + __popcll(m & ((2ull << lane) - 1ull));   // starts up to and including this block
            if (start && upto - 1 < kMaxRuns) r_slot[upto - 1] = b;
            if (end && upto - 1 < kMaxRuns) r_end[upto - 1] = b;
            __syncthreads();
        }
        const int runs = base;
        if (runs <= kMaxRuns) {
            // last sub-tile of a run's last block with a token in it (the blocks before it count as full)
            const int per = a.TILE_M / 4;   // groups of four slots in a block
            for (int g = tid; g < runs * per; g += 512) {
                const int r = g / per, q = g - r * per;
                const int slot = r_end[r] * a.TILE_M + 4 * q;
                bool any = false;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int t = slot + i < a.num_slots ? a.sorted_token_ids[slot + i] : 0;
                    any = any || (t >= 1 && t <= a.total_tokens);
                }
                if (any) atomicMax(&r_live[r], q / 8 + 1);
            }
            __syncthreads();
            if (wave == 0) {
                int tiles = 0, tiles4 = 0, tiles2 = 0;
                for (int r = lane; r < runs; r += 64) {
                    const int live = r_live[r] + (r_end[r] - r_slot[r]) * (a.TILE_M / 32);
                    tiles4 += (live + max_live(4) - 1) / max_live(4) * strips4;
                    tiles2 += (live + max_live(2) - 1) / max_live(2) * strips2;
                    r_live[r] = live;
                }
#pragma unroll
                for (int o = 32; o; o >>= 1) {
                    tiles4 += __shfl_xor(tiles4, o, 64);
                    tiles2 += __shfl_xor(tiles2, o, 64);
                }
                const bool wide = choose(tiles4, tiles2);
                const int most = wide ? max_live(4) : max_live(2), strips = wide ? strips4 : strips2;
                for (int r0 = 0; r0 < runs; r0 += 64) {
                    const int r = r0 + lane;
                    int n = 0;
                    if (r < runs) {
                        const int b = r_slot[r], e = ids[b], live = r_live[r];
                        n = (live + most - 1) / most * strips;
                        r_live[r] = live | (e - 1) << 16;
                        r_slot[r] = b * a.TILE_M;
                    }
                    int pre = n;
#pragma unroll
                    for (int o = 1; o < 64; o <<= 1) {
                        const int v = __shfl_up(pre, o, 64);
                        if (lane >= o) pre += v;
                    }
                    if (r < runs) r_first[r] = tiles + pre - n;
                    tiles += __shfl(pre, 63, 64);
                }
                if (lane == 0) {
                    s_runs = runs;
                    s_tiles = tiles;
                    s_wide = wide;
                }
            }
        } else if (tid == 0) {   // one tile per 128 slots and strip
            const int blocks = nb * (a.TILE_M / kBlock);
            const bool wide = choose(blocks * strips4, blocks * strips2);
            s_runs = -1;
            s_tiles = blocks * (wide ? strips4 : strips2);
            s_wide = wide;
        }
        __syncthreads();
    }
    // (the ring's memory is free from here on; the same for all lanes, and known to be, as there are barriers in either branch)
    const Runs table = {r_first, r_slot, r_live, __builtin_amdgcn_readfirstlane(s_runs), __builtin_amdgcn_readfirstlane(s_tiles)};
    if (__builtin_amdgcn_readfirstlane(s_wide)) walk_tiles<E, MODE, 4>(a, strips4, table, ring, s_tok, s_wt);
    else walk_tiles<E, MODE, 2>(a, strips2, table, ring, s_tok, s_wt);
}

}  // namespace

namespace mi {
namespace moe {

static bool prefill_applicable(const DenseArgs& a) {
    return !a.a8 && !a.w8 && a.num_blocks > 0 && a.num_blocks <= kMaxBlocks && (int64_t)a.num_blocks * (a.TILE_M / 32) < 65536 && a.num_experts < 32768 &&
           // (32-bit byte offsets of a token's column and of a weight row within its expert)
           (int64_t)a.num_a_cols * a.lda * 2 <= 0xffffffffll && (int64_t)a.N * a.ldb * 2 <= 0xffffffffll;
}

// True where this kernel is the one to take.  The host knows the replicas per expert n only, not how evenly they are dealt,
// so the line lies where the kernel is the quicker one for even and for uneven routing alike (router logits ~ N(0, 1) with
// an offset per expert of 0, 0.25, 0.5, 1 or 2 deviations).  `w`: rounds of the CUs that tiles of 160 x 256 make, an expert's last
// tile half full; the kernel wins where the last round is well filled, or where there are many, the sooner the longer K is (with
// K = 512 a tile is over before its transfers are spread: 1.0-1.1 of the ring kernel's time at 3 to 5 rounds), and below 112
// replicas the blocks of 128 slots are as good (90: 1.0-1.5).
// 300 shapes (8 to 64 experts, 112 to 1100 replicas each, hidden 512 / 1024, inter 512 to 2048) at the five degrees of
// unevenness: 0.90-0.91 (gate / up, 97 shapes taken) and 0.83-0.84 (down, 68) of the ring kernel's time at each degree, 1.02 at worst
// in a shape's mean over them, 1.09 in one launch.  A line drawn for even routing alone was off by up to 1.65.
static bool pays(double n, int K, double w) {
    if (n < 112) return false;
    if (K >= 2048) return w >= 1.28 || (w >= 0.48 && w <= 1.15);
    if (K >= 1024) return w >= 2.45 || (n >= 200 && ((w >= 1.37 && w <= 1.9) || (w >= 0.84 && w <= 1.05)));
    return K >= 512 && w >= 5.1;
}

// MI_MOE_PREFILL = 0 | 2 | 4: never / with 128 / with 256 weight rows per tile wherever possible (read at every call).
bool prefill_launch(const DenseArgs& a, hipStream_t s) {
    if (!prefill_applicable(a)) return false;
    const char* env = getenv("MI_MOE_PREFILL");
    const int force = env ? atoi(env) : -1, rows = force == 4 ? 256 : force == 2 ? 128 : 0;
    const int64_t half = a.silu ? 2 : 1;
    const int strips4 = (int)cld((int64_t)a.N / half, 256 / half), strips2 = (int)cld((int64_t)a.N / half, 128 / half);
    const double n = (double)a.total_tokens / a.num_experts;
    if (!rows && (force == 0 || !pays(n, a.K, a.num_experts * (n / 160 + 0.5) * strips4 / 256.0))) return false;
    const int64_t tiles = (int64_t)a.num_blocks * (a.TILE_M / 32) * strips2;   // (at most)
    const int64_t per_xcd = cld(tiles, (int64_t)8) < 32 ? cld(tiles, (int64_t)8) : 32;
    const dim3 grid((unsigned)(per_xcd * 8));
#define LAUNCH(ET, MODE) hipLaunchKernelGGL((moe_prefill_kernel<ET, MODE>), grid, dim3(512), 0, s, a, strips4, strips2, rows)
#define NAME(P, WIDE, NARROW) set_variant(rows == 256 ? P "_t128_to160_" WIDE "_k64_ring3" : rows == 128 ? P "_t128_to192_" NARROW "_k64_ring3" : P "_t128_to160_" WIDE "_or_to192_" NARROW "_k64_ring3")
    if (a.silu) {
        if (a.bf16) LAUNCH(BF16, MODE_SILU);
        else LAUNCH(F16, MODE_SILU);
        NAME("fused_moe_dense_silu", "n128x2", "n64x2");
    } else if (a.acc_shift >= 0) {
        if (a.bf16) LAUNCH(BF16, MODE_ACC);
        else LAUNCH(F16, MODE_ACC);
        NAME("fused_moe_dense_acc", "n256", "n128");
    } else {
        if (a.bf16) LAUNCH(BF16, MODE_PLAIN);
        else LAUNCH(F16, MODE_PLAIN);
        NAME("fused_moe_dense", "n256", "n128");
    }
#undef NAME
#undef LAUNCH
    return true;
}

}  // namespace moe
}  // namespace mi
