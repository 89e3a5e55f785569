// Fused multi-head attention forward, software-pipelined kernel for head dimension 128: stand-in for fmha_kernel of the
// reference's examples/fmha.jl:20-139 on prompts (any Sq, Skv, decode offset and head grouping; rows 16-byte aligned).
//
// What bounds attention at D = 128 is the LDS pipe, not the softmax: per key a wave reads twice the fragments of D = 64
// while the exponentials stay the same.  With 32 queries per wave (fmha_fwd_dma_kernel) the eight waves of a CU read
// 3072 LDS cycles of K and V fragments per 64 keys for 2048 cycles of MFMA.  So a wave takes two 32-query column tiles
// ("streams") that share every fragment: half the LDS reads per MFMA, at the price of one wave per SIMD with all of its
// 512 registers (O 128, Q 64, two score tiles per stream 64, fragments and weights 80).  Nothing else runs on the SIMD, so
// everything that is not an MFMA has to ride in the shadow of one: the walk is software-pipelined over halves of 32 keys
// and laid out by hand in issue slots of one MFMA (32 cycles of the matrix pipe) plus up to that much of other work:
//     slots  0..15  S(j+1) = K(j+1) . Q, k-step major over the streams;
//     slots 16..31  O += V(j) . P(j), 16-key chunk major;
//     weights P(j) = exp2(S(j) * scale - m) one score at a time, spread over slots 0..27;
//     V(j) fragments (LDS transpose reads) in slots 1..8, K(j+2) fragments in slots 18..25, the row maxima of S(j+1) in
//     slots 18..31, the requests for halves K(j+5) and V(j+3) in every third slot, the barrier in slot 1.
// K and V travel through two rings of four 8 KB LDS slots filled by direct global->LDS loads three steps ahead.  The loop
// over unmasked halves is unrolled by four so that ring slots are immediate offsets.
//
// The running maximum is the true one at every half, as in the general kernel: the row's largest weight is exactly 1, and
// the weights' rounding costs no more than there (error against float64, 2 x 32 heads, S = 2000 causal bf16: 1.746e-3 of the
// result, the general kernel 1.756e-3).  A stream's sums are rescaled when any of its 32 rows has a new maximum, which is
// most halves: 64 multiplies that nothing hides, a fifth of the time in all.  Raising only what had outgrown its maximum
// by 2^8 (P in (0, 2^8]) took 75 instead of 86 us and was off by 1.831e-3 (scores of three times the spread: 2.15e-3
// against 1.75e-3); the multiplies spread over slots 0..15 behind a branch each took 91 us, and maxima raised once per two
// halves 90 us: half the multiplies, but a third set of scores, which with O takes 224 of the 256 registers that vector
// instructions reach, and what else is there moves to and fro.  Scores are scaled in fp32.
//
// Measured (2 x 32 heads in groups of 4, bf16, against the general kernel): S = 2048 causal 120 -> 86 us (0.57 -> 0.80
// PFLOP/s), not causal 153 -> 142 us (0.90 -> 0.97), S = 2000 causal 117 -> 87 us.  What bounds it is the issue of one wave per
// SIMD: one barrier per two halves, four waves per K / V ring (256 queries) and row sums by the matrix cores (ones times P:
// 40 instructions less per step, 4 MFMAs more) were tried and did not help.  Causal pays for its diagonals and for the
// last, unequal workgroups.
#include "fmha_common.h"
#include "fmha_pipe128_map.h"

#include <utility>

namespace mi {
namespace fmha {
namespace {

constexpr int kD = 128;           // head dimension
constexpr int NW = 2;             // waves of a workgroup
constexpr int kHK = 32;           // keys per half
constexpr int kSlot = kHK * kD;   // elements per ring slot
constexpr int kSlotBytes = kSlot * 2;
constexpr int kKS = kD / 16;      // k-steps of a score tile
constexpr int kDT = kD / 32;      // 32-channel tiles of the output
constexpr int T = kSlotBytes / 1024 / NW;   // 1 KB transfers per wave and half, for K and for V each
constexpr int KO = 2;             // distinct K lane offsets: transfers 16 keys apart share theirs
constexpr int kPre = 1;           // the slot that waits for the transfers and for the other waves

// f(0), f(1), ... f(N - 1) with the argument a constant: the slots of a step are laid out at compile time.
template <typename F, int... I>
__device__ __forceinline__ void static_for(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    static_for(f, std::make_integer_sequence<int, N>{});
}

// gfx9 s_waitcnt: vmcnt(n), lgkmcnt(0)
constexpr int wait_vm(int n) { return 0x0070 | (n & 15) | ((n >> 4) << 14); }

struct Lane {
    // wave-uniform
    const char *kbase[T], *vbase[T];        // first key of transfer i in half 0, less what the lane and instruction offsets hold
    unsigned k_half, v_half;                // bytes per half
    unsigned ks_base, vs_base;              // LDS byte addresses of the rings, this wave's first transfer
    int nh;                                 // halves walked by the workgroup
    int back;                               // rows by which the last half starts early (see below)
    // per lane
    unsigned koff[KO], voff;                // byte offsets of the lane in the next half to be requested ...
    unsigned kend[KO], vend;                // ... and in the last one: past the end the last half is sent again, which
                                            // keeps the number of transfers in flight the same at every step
    unsigned kfo[kKS];                      // fragment element offsets inside a slot
    unsigned vfo[kDT];
    int hb4;                                // 4 in the upper half-wave
    int lim[2];                             // last visible key of the lane's query
};

// When the walk reaches the end of a key range that is not a multiple of 32, its last half is the last 32 keys that
// exist: no transfer passes the end, and the `back` leading rows, which the half before has already covered, are masked
// (that half is never one of the unmasked steps).

struct Acc {
    s16x8 qf[2][kKS];
    f32x16 o[2][kDT];
    float l[2];         // row sums of the weights over the lane's half of the keys
    float top[2];       // running maximum
    float m[2];         // the same, scaled (exp2 domain)
};

// Transfer d = 0 .. 2T-1 of a half's worth: d < T is transfer d of the next K half, the others of the next V half.  The
// LDS destination is m0 plus the instruction's offset, which covers the T transfers of a half around one value of m0
// (and is taken off the base addresses, as it counts for the global side as well); `dest` sets m0, at least one
// instruction before the load that follows it.
constexpr int inst_offset(int i) { return 1024 * NW * (i - T / 2); }
__device__ __forceinline__ void dest(unsigned base, int slot) {
    asm volatile("s_mov_b32 m0, %0" : : "s"(base + slot * kSlotBytes) : "m0");
}
template <int OFF>
__device__ __forceinline__ void load_lds(unsigned voff, const char* sbase) {
    asm volatile("global_load_lds_dwordx4 %0, %1 offset:%2" : : "v"(voff), "s"(sbase), "n"(OFF) : "memory");
}
template <int D>
__device__ __forceinline__ void load_of(Lane& c) {
    if constexpr (D < T) {
        load_lds<inst_offset(D)>(c.koff[D % KO], c.kbase[D]);
        if constexpr (D >= T - KO) {
            const unsigned n = c.koff[D % KO] + c.k_half;
            c.koff[D % KO] = n < c.kend[D % KO] ? n : c.kend[D % KO];
        }
    } else {
        load_lds<inst_offset(D - T)>(c.voff, c.vbase[D - T]);
        if constexpr (D == 2 * T - 1) {
            const unsigned n = c.voff + c.v_half;
            c.voff = n < c.vend ? n : c.vend;
        }
    }
}
// The next K half into ring slot `slot`, the next V half likewise.
__device__ __forceinline__ void fill_k(Lane& c, int slot) {
    dest(c.ks_base, slot);
    asm volatile("s_nop 0");
    static_for<T>([&](auto I) __attribute__((always_inline)) { load_of<I>(c); });
}
__device__ __forceinline__ void fill_v(Lane& c, int slot) {
    dest(c.vs_base, slot);
    asm volatile("s_nop 0");
    static_for<T>([&](auto I) __attribute__((always_inline)) { load_of<T + I>(c); });
}

__device__ __forceinline__ void read_k(const unsigned short* Ks, const Lane& c, int slot, int ks, s16x8 (&kf)[kKS]) {
    kf[ks] = *reinterpret_cast<const s16x8*>(Ks + slot * kSlot + c.kfo[ks]);
}

// Operation i = 0..7 of a stream's row maximum over its sixteen scores of the lane's half of the keys; MASK: rows past
// `lim` of the half, counted from the lane's first row, are not visible.
template <bool MASK>
__device__ __forceinline__ void row_max(f32x16& s, int i, int lim, float& mx) {
    auto mask = [&](int r) {
        if (MASK) s[r] = 8 * (r >> 2) + (r & 3) <= lim ? s[r] : -INFINITY;
    };
    if (i == 0) {
        mask(0); mask(1); mask(2);
        mx = max3(s[0], s[1], s[2]);
    } else if (i < 7) {
        mask(2 * i + 1); mask(2 * i + 2);
        mx = max3(mx, s[2 * i + 1], s[2 * i + 2]);
    } else {
        mask(15);
        mx = max3(mx, s[15], s[15]);
    }
}

// The query fragments stay in the accumulator half of the register file, which no vector instruction needs to read them
// from: the other half is for what they work on.
__device__ __forceinline__ void pin(Acc& a) {
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int s = 0; s < kKS; ++s) asm volatile("" : "+a"(a.qf[q][s]));
}

// The slots of a step, one MFMA each: S(j+1) in 0..15, then the tiles of O per 16-key chunk and stream.
constexpr int kSlots = 32;
// The weights of a step are made in 32 units, the exponential of one score each -- piece x = 0..15 (chunk x / 8, stream
// (x / 4) % 2, pair x % 4) is units 2x and 2x + 1 -- and a pair is rounded, packed and added to the row sum one unit after
// its second exponential.  This is the number of units done before slot sl; slots 16, 20, 24 and 28 are the first that
// need the pieces of (chunk, stream) 0 to 3.
constexpr int units_before(int sl) { return sl <= 8 ? sl : 8 + (5 * (sl - 8) + 3) / 4 > 33 ? 33 : 8 + (5 * (sl - 8) + 3) / 4; }
static_assert(units_before(16) >= 9 && units_before(20) >= 17 && units_before(24) >= 25 && units_before(28) == 33, "the weights of a chunk exist before its MFMAs");
// Operations of the row maxima done before slot sl (those of stream 0 first; S(j+1) is complete behind slot 15).
constexpr int max_before(int sl) { return sl <= 18 ? 0 : sl <= 28 ? sl - 18 : 10 + 2 * (sl - 28) > 16 ? 16 : 10 + 2 * (sl - 28); }

// One half j: P(j) and O += V(j) P(j); with NEXT also S(j+1) and its row maxima (MASK: against c.lim).  The step waits for
// what was requested three steps ago -- K(j+2) and V(j) --, meets the other waves, which are done with the step before, and
// requests K(j+5) and V(j+3) into the slots that this freed.  SLOT: j % 4 when it is a constant of the unrolled loop, -1
// otherwise.
template <typename E, bool NEXT, bool MASK, int SLOT>
__device__ __forceinline__ void step(const unsigned short* Ks, const unsigned short* Vs, Lane& c, Acc& a, int j, float scale2,
                                     f32x16 (&s_cur)[2], f32x16 (&s_next)[2], s16x8 (&kf)[kKS], float (&cand)[2]) {
    const int s0 = SLOT >= 0 ? SLOT : j & 3;
    // ---- raise the running maxima of a stream if some row has a new one (every row sees key 0 in the first half) ----
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        if (__any(cand[q] > a.top[q])) {
            a.top[q] = fmaxf(a.top[q], xhalf_max(cand[q]));
            const float m_new = a.top[q] * scale2;
            const float alpha = __builtin_amdgcn_exp2f(a.m[q] - m_new);   // (0 at the first half: l and O are zero)
            a.l[q] *= alpha;
#pragma unroll
            for (int dt = 0; dt < kDT; ++dt)
#pragma unroll
                for (int r = 0; r < 16; ++r) a.o[q][dt][r] *= alpha;
            a.m[q] = m_new;
        }
    }
    pin(a);
    unsigned pf[2][2][4];     // [stream][chunk][pair]
    s16x8 vf[2][kDT];         // [chunk][d tile]
    float p[2][2];            // exponentials of two pieces in flight
    auto unit = [&](auto UI) __attribute__((always_inline)) {
        constexpr int u = UI, x = u / 2, e = u % 2, q = (x / 4) % 2, h = 4 * (x / 8) + x % 4;
        if constexpr (u < 32) p[x & 1][e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s_cur[q][2 * h + e], scale2, -a.m[q]));
        if constexpr (e == 0 && x > 0) {
            constexpr int y = x - 1, qy = (y / 4) % 2, hy = 4 * (y / 8) + y % 4;
            const unsigned pk = Pack<E>::pack(p[y & 1][0], p[y & 1][1]);
            pf[qy][hy >> 2][hy & 3] = pk;
            a.l[qy] = Pack<E>::sum2(pk, p[y & 1][0], p[y & 1][1], a.l[qy]);   // (not the f16 chunk sums: they round)
        }
    };
    auto vread = [&](int f) {
        const int ch = f / kDT, dt = f % kDT;
        const unsigned short* q = Vs + s0 * kSlot + c.vfo[dt] + 16 * ch * kD;
        s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(s16x4, q));
        s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(s16x4, q + 8 * kD));
        vf[ch][dt] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    };
    auto pv = [&](auto KI) __attribute__((always_inline)) {   // k = 0..15: chunk k / 8, stream (k / 4) % 2, d tile k % 4
        constexpr int k = KI, ch = k / 8, q = (k / 4) % 2, dt = k % 4;
        const u32x4 pw = {pf[q][ch][0], pf[q][ch][1], pf[q][ch][2], pf[q][ch][3]};
        a.o[q][dt] = E::mfma32(vf[ch][dt], __builtin_bit_cast(s16x8, pw), a.o[q][dt]);
    };
    slot_end();
    if constexpr (NEXT) {
        const int back = MASK && j + 2 == c.nh ? c.back : 0;   // (of the half whose scores are masked)
        const int first = kHK * (j + 1) - back + c.hb4;        // key in the lane's first row of that half
        static_for<kSlots>([&](auto SL) __attribute__((always_inline)) {
            constexpr int sl = SL, u0 = units_before(sl), nu = units_before(sl + 1) - u0, m0 = max_before(sl), nm = max_before(sl + 1) - m0;
            // one transfer in every 32 / 2T slots: the CU moves 64 bytes a cycle, and its four waves walk in step
            constexpr int every = (kSlots - 2) / (2 * T), d = (sl - 2) / every;
            constexpr bool dma = sl >= 2 && (sl - 2) % every == 0 && d < 2 * T;
            if constexpr (sl == 0 || sl == 16) __builtin_amdgcn_s_waitcnt(0xc07f);   // the fragments (read eight slots ago): lgkmcnt(0)
            if constexpr (dma && d == 0) dest(c.ks_base, (s0 + 1) & 3);
            if constexpr (dma && d == T) dest(c.vs_base, (s0 + 3) & 3);
            slot_end();
            if constexpr (sl < 16) s_next[sl % 2] = E::mfma32(kf[sl / 2], a.qf[sl % 2][sl / 2], sl < 2 ? f32x16{0} : s_next[sl % 2]);
            else pv(std::integral_constant<int, sl - 16>{});
            slot_end();
            if constexpr (sl == kPre) wait_and_barrier<wait_vm(4 * T)>();
            if constexpr (dma) load_of<d>(c);
            if constexpr (sl >= 1 && sl <= 8) vread(sl - 1);
            if constexpr (sl >= 18 && sl < 26) read_k(Ks, c, (s0 + 2) & 3, sl - 18, kf);
            if constexpr (MASK && sl == 17) {
                if (back > 0) {   // rows that the half before has covered
#pragma unroll
                    for (int q = 0; q < 2; ++q)
#pragma unroll
                        for (int r = 0; r < 16; ++r) s_next[q][r] = 8 * (r >> 2) + (r & 3) + c.hb4 >= back ? s_next[q][r] : -INFINITY;
                }
            }
            static_for<nu>([&](auto I) __attribute__((always_inline)) { unit(std::integral_constant<int, u0 + I>{}); });
            static_for<nm>([&](auto I) __attribute__((always_inline)) {
                constexpr int q = (m0 + I) / 8;
                row_max<MASK>(s_next[q], (m0 + I) % 8, MASK ? c.lim[q] - first : 0, cand[q]);
            });
            slot_end();
        });
    } else {
        wait_and_barrier<wait_vm(4 * T)>();
#pragma unroll
        for (int f = 0; f < 2 * kDT; ++f) vread(f);
        fill_k(c, (s0 + 1) & 3);
        fill_v(c, (s0 + 3) & 3);
        static_for<9>([&](auto U) __attribute__((always_inline)) { unit(U); });
        static_for<16>([&](auto KI) __attribute__((always_inline)) {
            constexpr int u0 = 9 + 2 * KI;
            pv(KI);
            static_for<(u0 + 2 <= 33 ? 2 : u0 < 33 ? 33 - u0 : 0)>([&](auto I) __attribute__((always_inline)) { unit(std::integral_constant<int, u0 + I>{}); });
            slot_end();
        });
    }
}

template <typename E, bool CAUSAL>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(1, 1))) void fmha_pipe128_kernel(
    const unsigned short* __restrict__ Q, Strides qs, const unsigned short* __restrict__ K, Strides ks,
    const unsigned short* __restrict__ V, Strides vs, unsigned short* __restrict__ O, Strides os, int Sq, int Skv, int H,
    float scale2, int input_pos, int nqb, Map mp) {
    __shared__ __attribute__((aligned(1024))) unsigned short Ks[4 * kSlot];
    __shared__ __attribute__((aligned(1024))) unsigned short Vs[4 * kSlot];

    const int tid = threadIdx.x, lane = tid & 63, hb = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // Workgroup id -> (query block, head): fmha_pipe128_map.h.
    int qb, bh;
    mp.at(blockIdx.x, nqb, CAUSAL, &qb, &bh);
    const int batch = (int)mp.H.div((unsigned)bh), head = bh - batch * H, kvh = (int)mp.group.div((unsigned)head);
    Q += (int64_t)head * qs.s2 + (int64_t)batch * qs.s3;
    O += (int64_t)head * os.s2 + (int64_t)batch * os.s3;

    const int q_wg = 64 * NW * qb, q_wave = q_wg + 64 * wave;   // first query of the workgroup / of the wave
    // Halves walked by the workgroup and by the wave; leading halves that every query of the wave sees whole.
    auto keys_for = [&](int last_q) {
        if (!CAUSAL) return Skv;
        const int lim = input_pos + (last_q < Sq - 1 ? last_q : Sq - 1) + 1;
        return lim < Skv ? lim : Skv;
    };
    const int nh = (keys_for(q_wg + 64 * NW - 1) + kHK - 1) / kHK;
    const int nw = q_wave < Sq ? (keys_for(q_wave + 63) + kHK - 1) / kHK : 0;
    const int open = (keys_for(q_wave)) / kHK;

    Lane c;
    {
        const char* kg = (const char*)(K + (int64_t)kvh * ks.s2 + (int64_t)batch * ks.s3);
        const char* vg = (const char*)(V + (int64_t)kvh * vs.s2 + (int64_t)batch * vs.s3);
#pragma unroll
        for (int i = 0; i < T; ++i) {
            c.kbase[i] = kg + 16 * (i / KO) * ks.s1 * 2 - inst_offset(i);
            c.vbase[i] = vg + 4 * NW * i * vs.s1 * 2 - inst_offset(i);
        }
        const unsigned kp = (unsigned)ks.s1 * 2, vp = (unsigned)vs.s1 * 2;   // bytes per key
        c.k_half = kHK * kp;
        c.v_half = kHK * vp;
        c.ks_base = (unsigned)(size_t)Ks + wave * 1024 - inst_offset(0);
        c.vs_base = (unsigned)(size_t)Vs + wave * 1024 - inst_offset(0);
        c.nh = nh;
        c.back = nh * kHK > Skv ? nh * kHK - Skv : 0;
        c.hb4 = 4 * hb;
        // Transfer t = wave + NW i of a half moves the four keys 4 t ..; a lane 16 bytes of one.  K chunks stand at
        // chunk ^ (key % 16), V chunks at chunk ^ 4 (key % 4): see ksw in fmha.hip.
        const unsigned r4 = lane >> 4, pos = lane & 15, last = (unsigned)(kHK * (nh - 1) - c.back);
#pragma unroll
        for (int i = 0; i < KO; ++i) {
            const unsigned key = 4 * (wave + NW * i) + r4;
            c.koff[i] = key * kp + 16 * (pos ^ (key & 15));
            c.kend[i] = c.koff[i] + last * kp;
        }
        const unsigned key4 = 4 * wave + r4;
        c.voff = key4 * vp + 16 * (pos ^ (4 * (key4 & 3)));
        c.vend = c.voff + last * vp;
    }
    {
        const int key = lane & 31;
#pragma unroll
        for (int s = 0; s < kKS; ++s) c.kfo[s] = key * kD + 8 * ((2 * s + hb) ^ (key & 15));
        const int g = lane >> 4, r = lane & 15;
#pragma unroll
        for (int dt = 0; dt < kDT; ++dt) {
            const int row = 4 * (g >> 1) + (r >> 2);
            const int col = 32 * dt + 16 * (g & 1) + 4 * (r & 3);
            c.vfo[dt] = row * kD + 8 * ((col >> 3) ^ (4 * (r >> 2))) + (col & 7);
        }
    }

    // Q first, then the ring fill in the order of need.  All of it is inline assembly, so the waits are counted by hand.
    int my_q[2];
    u32x4 qraw[2][kKS];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        my_q[q] = q_wave + 32 * q + (lane & 31);
        const int row = my_q[q] < Sq ? my_q[q] : Sq - 1;   // (queries past the end: any row, never stored)
        c.lim[q] = Skv - 1;
        if (CAUSAL && input_pos + my_q[q] < c.lim[q]) c.lim[q] = input_pos + my_q[q];
        const unsigned short* qp = Q + (int64_t)row * qs.s1 + 8 * hb;
#pragma unroll
        for (int s = 0; s < kKS; ++s)
            asm volatile("global_load_dwordx4 %0, %1, off offset:%2" : "=v"(qraw[q][s]) : "v"(qp), "n"(32 * s) : "memory");
    }
    fill_k(c, 0);
    fill_k(c, 1);
    fill_k(c, 2);
    fill_v(c, 0);
    fill_k(c, 3);
    fill_v(c, 1);
    // (the registers are operands of the wait, so nothing that reads them is scheduled above it)
#define QW(q) "+v"(qraw[q][0]), "+v"(qraw[q][1]), "+v"(qraw[q][2]), "+v"(qraw[q][3]), "+v"(qraw[q][4]), "+v"(qraw[q][5]), "+v"(qraw[q][6]), "+v"(qraw[q][7])
    asm volatile("s_waitcnt vmcnt(%8)" : QW(0) : "n"(6 * T) : "memory");
    asm volatile("" : QW(1) : : "memory");
#undef QW

    Acc a;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
#pragma unroll
        for (int s = 0; s < kKS; ++s) a.qf[q][s] = __builtin_bit_cast(s16x8, qraw[q][s]);
#pragma unroll
        for (int dt = 0; dt < kDT; ++dt) a.o[q][dt] = f32x16{0};
        a.l[q] = 0.f;
        a.m[q] = a.top[q] = -INFINITY;
    }

    // ---- prologue: S(0), its row maxima, the K(1) fragments -----------------------------------------------------
    f32x16 sa[2], sb[2];
    s16x8 kf[kKS];
    float cand[2];
    wait_and_barrier<wait_vm(5 * T)>();   // K(0)
#pragma unroll
    for (int s = 0; s < kKS; ++s) read_k(Ks, c, 0, s, kf);
#pragma unroll
    for (int s = 0; s < kKS; ++s)
#pragma unroll
        for (int q = 0; q < 2; ++q) sa[q] = E::mfma32(kf[s], a.qf[q][s], s == 0 ? f32x16{0} : sa[q]);
    wait_and_barrier<wait_vm(4 * T)>();   // K(1); every wave has read K(0)
#pragma unroll
    for (int s = 0; s < kKS; ++s) read_k(Ks, c, 1, s, kf);
    fill_k(c, 0);   // K(4)
    fill_v(c, 2);
    {
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                if (open < 1) row_max<true>(sa[q], i, c.lim[q] - c.hb4, cand[q]);
                else row_max<false>(sa[q], i, 0, cand[q]);
            }
    }

    // ---- the walk ---------------------------------------------------------------------------------------------------
#define STEP(NEXT, MASK, SLOT, jx, s0, s1) step<E, NEXT, MASK, SLOT>(Ks, Vs, c, a, jx, scale2, s0, s1, kf, cand)
    int j = 0;
    if (nw > 0) {
        const int plain = open - 1 < nw - 1 ? open - 1 : nw - 1;   // steps whose S(j+1) needs no mask
        for (; j + 4 <= plain; j += 4) {
            STEP(true, false, 0, j, sa, sb);
            STEP(true, false, 1, j + 1, sb, sa);
            STEP(true, false, 2, j + 2, sa, sb);
            STEP(true, false, 3, j + 3, sb, sa);
        }
        for (; j + 2 <= plain; j += 2) {   // (at most one trip)
            STEP(true, false, -1, j, sa, sb);
            STEP(true, false, -1, j + 1, sb, sa);
        }
        for (; j + 2 <= nw - 1; j += 2) {
            STEP(true, true, -1, j, sa, sb);
            STEP(true, true, -1, j + 1, sb, sa);
        }
        if (j < nw - 1) {
            STEP(true, true, -1, j, sa, sb);
            ++j;
            STEP(false, false, -1, j, sb, sa);
        } else {
            STEP(false, false, -1, j, sa, sb);
        }
        ++j;
    }
#undef STEP
    for (; j < nh; ++j) {   // the other waves' diagonals: this wave moves its share of the halves and keeps the barriers
        wait_and_barrier<wait_vm(4 * T)>();
        fill_k(c, (j + 1) & 3);
        fill_v(c, (j + 3) & 3);
    }
    // Transfers for halves past the end are still in flight: let them land before the LDS goes to another workgroup.
    __builtin_amdgcn_s_waitcnt(wait_vm(0));

    // ---- epilogue: O / l (approximate reciprocal, fmha.jl:132-134), round, store ------------------------------------
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const float inv = __builtin_amdgcn_rcpf(xhalf_sum(a.l[q]));
        // (two lane halves hold four channels of every eight: an exchange makes each store 16 bytes)
        unsigned short* op = O + (int64_t)my_q[q] * os.s1 + 8 * hb;
#pragma unroll
        for (int dt = 0; dt < kDT; ++dt)
#pragma unroll
            for (int g = 0; g < 4; g += 2) {
                const f32x16& v = a.o[q][dt];
                u32x4 w;
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const unsigned x = Pack<E>::pack(v[4 * g + 2 * e] * inv, v[4 * g + 2 * e + 1] * inv);
                    const unsigned y = Pack<E>::pack(v[4 * g + 4 + 2 * e] * inv, v[4 * g + 5 + 2 * e] * inv);
                    const auto r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
                    w[e] = r[0];
                    w[2 + e] = r[1];
                }
                if (my_q[q] < Sq) *reinterpret_cast<u32x4*>(op + 32 * dt + 8 * g) = w;
            }
    }
}

template <typename E>
void launch_e(const Problem& p, hipStream_t stream) {
    const mi_tile_array *Q = p.Q, *K = p.K, *V = p.V, *O = p.O;
    Strides qs{Q->strides[1], Q->strides[2], Q->strides[3]}, ks{K->strides[1], K->strides[2], K->strides[3]},
        vs{V->strides[1], V->strides[2], V->strides[3]}, os{O->strides[1], O->strides[2], O->strides[3]};
    const int Sq = (int)Q->sizes[1], Skv = (int)K->sizes[1];
    const int nqb = (Sq + 64 * NW - 1) / (64 * NW), nbh = (int)(Q->sizes[2] * Q->sizes[3]);
    const Map mp = make_map(nqb, nbh, p.H, p.group, p.causal);
    if (p.causal)
        hipLaunchKernelGGL((fmha_pipe128_kernel<E, true>), dim3((unsigned)(nqb * nbh)), dim3(64 * NW), 0, stream,
                           (const unsigned short*)Q->ptr, qs, (const unsigned short*)K->ptr, ks, (const unsigned short*)V->ptr, vs,
                           (unsigned short*)O->ptr, os, Sq, Skv, p.H, p.scale2, p.input_pos, nqb, mp);
    else
        hipLaunchKernelGGL((fmha_pipe128_kernel<E, false>), dim3((unsigned)(nqb * nbh)), dim3(64 * NW), 0, stream,
                           (const unsigned short*)Q->ptr, qs, (const unsigned short*)K->ptr, ks, (const unsigned short*)V->ptr, vs,
                           (unsigned short*)O->ptr, os, Sq, Skv, p.H, p.scale2, p.input_pos, nqb, mp);
}

}  // namespace

bool pipe128_applicable(const Problem& p) {
    const mi_tile_array *Q = p.Q, *K = p.K, *V = p.V, *O = p.O;
    if (Q->sizes[0] != kD || V->sizes[0] != kD) return false;
    if (!(p.scale2 > 0.f)) return false;
    if (!vec16(Q) || !vec16(K) || !vec16(V) || !vec16(O)) return false;
    // 32-bit byte offsets within a head's keys
    const int64_t rows = K->sizes[1] + 2 * kHK;
    if (K->strides[1] < 0 || V->strides[1] < 0 || rows * K->strides[1] >= (1ll << 31) || rows * V->strides[1] >= (1ll << 31)) return false;
    if (!map_exact((Q->sizes[1] + 127) / 128, Q->sizes[2] * Q->sizes[3], p.H)) return false;   // (its numbering's divisions)
    if (K->sizes[1] < kHK) return false;   // (the last half is the last 32 keys)
    return Q->sizes[1] > 64;               // (few queries: a group's heads are stacked in one tile, fmha.hip)
}

bool pipe128_pays(const Problem& p, int parts) {
    const int64_t Sq = p.Q->sizes[1], Skv = p.K->sizes[1], nqb = (Sq + 127) / 128, wgs = nqb * p.Q->sizes[2] * p.Q->sizes[3];
    int64_t longest = Skv, shortest = Skv;   // keys walked by the last / by the first workgroup of a head
    if (p.causal) {
        longest = p.input_pos + Sq < Skv ? p.input_pos + Sq : Skv;
        shortest = p.input_pos + 128 < longest ? p.input_pos + 128 : longest;
    }
    const double halves = (double)((longest + kHK - 1) / kHK), all = (double)(longest + shortest) / (2 * kHK) * (double)wgs;
    // Times of both kernels on 950 shapes (1 to 8 batches of 1 to 64 heads, 65 to 4096 queries, up to 16384 keys, bf16):
    // against the kernel that is split over the keys this one is quicker where its longest walk, 9 us + 0.8 us per half,
    // ends before the split one's 18 us + 2.8 ns per half of all walks together.  (Quicker / slower, this kernel : the split
    // one: 1 x 32 heads, 996 queries and keys, causal 34 : 42 us, 1200 of them not causal 45 : 58; 2 heads, 2034 causal 57 : 28,
    // 16 heads, 1024 of 8192 causal 191 : 117.)
    if (parts > 1) return 0.8 * halves <= 9.0 + 0.0028 * all;
    // Where the other kernel walks the keys alone as well, the grid has to fill most of its last round of 512 workgroups
    // (two per CU) and the walks be long enough to pay for the ramp: 2 x 32 heads, S = 2000 causal 82 : 115 us, 8 x 32 heads,
    // S = 506 causal 38 : 45, 1 x 32 heads, S = 2048 causal 64 : 70; but 640 workgroups of 19 halves, not causal, 54 : 45, 4 x
    // 32 heads, S = 1171 causal (1280 workgroups) 90 : 81, and 8 x 16 heads, S = 173 12.1 : 11.3.  On 700 further shapes,
    // 220 of them taken, the times were 0.49 to 1.11 of the other kernel's, 0.76 in the mean.  Since the other kernel starts
    // its long causal walks first, launches of three rounds and more are worth it from 48 halves only (4 x 64 heads, S = 653
    // causal 62 : 57, 6 x 64, 712 102 : 93, 7 x 32, 1079 106 : 99; 5 x 16, 3766 347 : 362, 6 x 40, 1955 323 : 358).
    const int64_t rounds = (wgs + 511) / 512;
    return wgs >= 448 && wgs * 100 >= rounds * 512 * (rounds <= 2 ? 78 : 90) && halves >= (wgs < 800 ? 32 : rounds <= 2 ? 8 : 48) && (p.causal || rounds <= 2);
}

void pipe128_launch(const Problem& p, hipStream_t stream) {
    if (p.bf16) launch_e<BF16>(p, stream);
    else launch_e<F16>(p, stream);
    set_variant("fmha_pipe_d128_q128_kv32_ring4");
}

}  // namespace fmha
}  // namespace mi
