// Fused multi-head attention forward for prompts that give the chip few queries: stand-in for fmha_kernel of the reference's
// examples/fmha.jl:20-139 (heads of 64 and 128, more than 64 queries, any Sq, Skv, decode offset and head grouping; rows 16-byte
// aligned).
//
// A workgroup of the pipelined kernels has 128 queries of a head and walks their keys one half of 32 after the other; with fewer of
// them than it takes to fill the SIMDs the launch lasts as long as that chain (0.2-0.4 us a half) while most SIMDs idle.  Here a
// workgroup has 32 queries, and its four (or two) waves share their keys: wave w takes the halves w, w + 4, ... with an LDS area,
// accumulators, maxima and row sums of its own, so there is no barrier before the parts are added at the end.  A wave waits for its
// half of K and V, reads all fragments into registers, requests its next half into the same place and computes; what it waits
// for, other waves of the SIMD fill (heads of 64: four per SIMD, 128: two).
//
// What bounds it: with few workgroups a step's own latency (transfer, S, maxima, weights, O), with many the path into LDS, which brings
// a half of K and V per 32 queries and not per 128 -- 8 KB (heads of 64) for 0.2 us of a SIMD's issue, at about 100 GB/s per CU for
// its four SIMDs 0.32 us; from there on the pipelined kernels are ahead.  Tried and not kept: 64 queries per wave (half the bytes, but
// half the waves: slower up to where the pipelined kernels win), a ring of two halves per wave (fewer waves per CU), eight waves.
//
// Heads of 128: the weights of a half refer to that half's own maximum (at most 2^8 below the running one), heads of 64: to the
// running maximum.  Either way each wave's largest weights are exact, and error against float64 is below that of every kernel that
// took these launches before (260 shapes each, of its error in the mean: heads of 128 0.91-0.98, at most 0.984; heads of 64 0.70-0.75).
//
// Measured (us, before -> now): heads of 64 2 x 8, S = 384 causal 8.3 -> 6.1, 2 x 4, 1408 17.7 -> 9.9, 2 x 8, 1088 15.6 -> 9.6, 7 x 4, 1472
// 28 -> 18, 2 x 8, 2688 not causal 69 -> 52; heads of 128 4 x 4, 512 causal 15.0 -> 7.6, 1 x 4, 3328 47 -> 27, 3 x 4, 1408 28.8 -> 16.4, 1 x 8, 3520
// 60 -> 42, 6 x 8, 817 28.8 -> 20.7.
#include "fmha_common.h"
#include "lds_transfer.h"

namespace mi {
namespace fmha {
namespace {

constexpr int kHK = 32;   // keys per half
constexpr int kQT = 32;   // queries per workgroup

template <typename E, int D, bool CAUSAL, int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(D == 64 ? 4 : 2))) void fmha_few_kernel(
    const unsigned short* __restrict__ Q, Strides qs, const unsigned short* __restrict__ K, Strides ks, const unsigned short* __restrict__ V, Strides vs,
    unsigned short* __restrict__ O, Strides os, int Sq, int Skv, int H, int group, float scale2, int input_pos, int nqt, int nbh) {
    constexpr bool OWN = D == 128;
    constexpr int KS = D / 16, DT = D / 32;            // k-steps of a score tile, 32-channel tiles of the output
    constexpr int HALF = kHK * D;                      // elements of a half of K or V
    constexpr int T = HALF * 2 / 1024, KT = 512 / D;   // transfers per half, keys per transfer
    constexpr int P = 16 / KT;                         // distinct K lane offsets: transfers 16 keys apart share theirs
    constexpr int AREA = 2 * HALF;                     // elements of a wave's half of K and V; at the end its sums
    static_assert(AREA * 2 >= D * 128, "a wave's sums fit its area");
    __shared__ __attribute__((aligned(1024))) unsigned short areas[NW * AREA];
    __shared__ float s_m[NW][kQT], s_l[NW][kQT];
    const int lane = threadIdx.x & 63, hb = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // Workgroup -> query tile and head: an XCD (ids congruent mod 8) gets neighbouring heads, which share keys; long walks first.
    int qt, bh;
    {
        const int L = blockIdx.x;
        if (nbh % 8 == 0) {
            const int each = nbh >> 3, i = L >> 3, r = i / each;
            bh = (L & 7) * each + (i - r * each);
            qt = r;
        } else {
            qt = L / nbh;
            bh = L - qt * nbh;
        }
        if (CAUSAL) qt = nqt - 1 - qt;
    }
    const int batch = bh / H, head = bh - batch * H, kvh = head / group;
    const int q0 = kQT * qt;
    const int my_q = q0 + (lane & 31);   // the lane's query
    int lim;                             // the last key that it sees
    s16x8 qf[KS];
    {
        const int row = my_q < Sq ? my_q : Sq - 1;   // (queries past the end: the last one again, never stored)
        lim = CAUSAL && input_pos + row < Skv - 1 ? input_pos + row : Skv - 1;
        const unsigned short* qp = Q + (int64_t)head * qs.s2 + (int64_t)batch * qs.s3 + (int64_t)row * qs.s1 + 8 * hb;
#pragma unroll
        for (int s = 0; s < KS; ++s) qf[s] = *reinterpret_cast<const s16x8*>(qp + 16 * s);
    }

    // Halves that the tile's last query sees; leading halves that its first query sees whole.
    int nh = (Skv + kHK - 1) / kHK, open = Skv / kHK;
    if (CAUSAL) {
        const int last = input_pos + (q0 + kQT - 1 < Sq ? q0 + kQT - 1 : Sq - 1);
        if (last < Skv - 1) nh = last / kHK + 1;
        const int o = (input_pos + q0 + 1) / kHK;
        open = o < open ? o : open;
    }

    // ---- transfers: lane -> key and position of its 16 bytes; chunk c of key k stands at c ^ swizzle(k) (see fmha.hip) ------------
    const unsigned kp = (unsigned)ks.s1 * 2, vp = (unsigned)vs.s1 * 2;   // bytes per key
    const int lr = lane / (D / 8), pos = lane % (D / 8);
    auto ksw = [](int key) { return D == 64 ? (key >> 1) & 7 : key & 15; };
    auto vsw = [](int key) { return D == 64 ? 2 * (key & 3) : 4 * (key & 3); };
    unsigned koff[P];
#pragma unroll
    for (int t = 0; t < P; ++t) koff[t] = (unsigned)(KT * t + lr) * kp + 16 * (pos ^ ksw(KT * t + lr));
    const unsigned voff = (unsigned)lr * vp + 16 * (pos ^ vsw(lr));
    const char* const kg = (const char*)(K + (int64_t)kvh * ks.s2 + (int64_t)batch * ks.s3);
    const char* const vg = (const char*)(V + (int64_t)kvh * vs.s2 + (int64_t)batch * vs.s3);
    const unsigned lds0 = (unsigned)(size_t)LDS_PTR(unsigned short, areas) + wave * (AREA * 2);
    auto issue = [&](int j) __attribute__((always_inline)) {
        const char* kj = kg + (int64_t)(kHK * j) * kp;
        const char* vj = vg + (int64_t)(kHK * j) * vp;
        if (kHK * (j + 1) <= Skv) {
#pragma unroll
            for (int t = 0; t < T; ++t) load_lds(lds0 + 1024 * t, koff[t % P], kj + (int64_t)(16 * (t / P)) * kp);
#pragma unroll
            for (int t = 0; t < T; ++t) load_lds(lds0 + 1024 * (T + t), voff, vj + (int64_t)(KT * t) * vp);
        } else {   // keys past the end: the last one again, masked below
            const int last = Skv - 1 - kHK * j;
#pragma unroll
            for (int t = 0; t < T; ++t) {
                const int key = KT * t + lr, k = key < last ? key : last;
                load_lds_at(lds0 + 1024 * t, kj + (int64_t)k * kp + 16 * (pos ^ ksw(key)));
            }
#pragma unroll
            for (int t = 0; t < T; ++t) {
                const int key = KT * t + lr, k = key < last ? key : last;
                load_lds_at(lds0 + 1024 * (T + t), vj + (int64_t)k * vp + 16 * (pos ^ vsw(key)));
            }
        }
    };
    if (wave < nh) issue(wave);

    unsigned kfo[KS], vfo[DT];
    {
        const int key = lane & 31, g = lane >> 4, r = lane & 15;
#pragma unroll
        for (int s = 0; s < KS; ++s) kfo[s] = key * D + 8 * ((2 * s + hb) ^ ksw(key));
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            const int vrow = 4 * (g >> 1) + (r >> 2), col = 32 * dt + 16 * (g & 1) + 4 * (r & 3);
            vfo[dt] = HALF + vrow * D + 8 * ((col >> 3) ^ vsw(r >> 2)) + (col & 7);
        }
    }
    f32x16 o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[dt] = f32x16{0};
    float top = -INFINITY;          // OWN: the running maximum; m is then the latest half's, at most 8 below it
    float m = -INFINITY, l = 0.f;   // running maximum (scaled, exp2 domain) and the sum over the lane's half of the keys
    // (the compiler's own wait for Q, here and not in every trip)
#pragma unroll
    for (int s = 0; s < KS; ++s) asm volatile("" : "+v"(qf[s]));

    for (int j = wave; j < nh; j += NW) {
        __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0)
        fence();
        const unsigned short* S = areas + wave * AREA;
        s16x8 kf[KS], vf[2][DT];
#pragma unroll
        for (int s = 0; s < KS; ++s) kf[s] = *reinterpret_cast<const s16x8*>(S + kfo[s]);
#pragma unroll
        for (int ch = 0; ch < 2; ++ch)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                const unsigned short* p = S + vfo[dt] + 16 * ch * D;
                const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(s16x4, p));
                const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(s16x4, p + 8 * D));
                vf[ch][dt] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
            }
        f32x16 s;
#pragma unroll
        for (int x = 0; x < KS; ++x) s = E::mfma32(kf[x], qf[x], x == 0 ? f32x16{0} : s);
        if (j + NW < nh) {
            __builtin_amdgcn_s_waitcnt(0xc07f);   // every fragment is in registers: the half's place is free
            fence();
            issue(j + NW);
        }
        if (j >= open) {
            const int left = lim - kHK * j - 4 * hb;
#pragma unroll
            for (int r = 0; r < 16; ++r) s[r] = 8 * (r >> 2) + (r & 3) <= left ? s[r] : -INFINITY;
        }
        float mx = max3(s[0], s[1], s[2]);
#pragma unroll
        for (int r = 3; r < 15; r += 2) mx = max3(mx, s[r], s[r + 1]);
        mx = xhalf_max(max3(mx, s[15], s[15])) * scale2;
        float mn;
        if constexpr (OWN) {
            top = fmaxf(top, mx);
            mn = fmaxf(mx, top - 8.f);
        } else {
            mn = fmaxf(m, mx);
        }
        if (__any(mn != m)) {
            const float alpha = mn == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m - mn);   // (nothing seen yet: all is zero)
            l *= alpha;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
            m = mn;
        }
        const float mu = m == -INFINITY ? 0.f : m;
#pragma unroll
        for (int ch = 0; ch < 2; ++ch) {
            u32x4 pw;
#pragma unroll
            for (int h = 0; h < 4; ++h) {
                const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[8 * ch + 2 * h], scale2, -mu));
                const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[8 * ch + 2 * h + 1], scale2, -mu));
                pw[h] = Pack<E>::pack(p0, p1);
                l = Pack<E>::sum2(pw[h], p0, p1, l);
            }
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) o[dt] = E::mfma32(vf[ch][dt], __builtin_bit_cast(s16x8, pw), o[dt]);
        }
    }

    // ---- the waves' parts, added in their order; a wave stores a quarter of the channels ----------------------------------------
    l = xhalf_sum(l);
    if (hb == 0) {
        s_m[wave][lane] = m;
        s_l[wave][lane] = l;
    }
    __syncthreads();
    float most = -INFINITY, sum = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) most = fmaxf(most, s_m[w][lane & 31]);
#pragma unroll
    for (int w = 0; w < NW; ++w) {   // (a wave whose halves the row does not see has m = -inf, l = 0 and o = 0)
        const float mw = s_m[w][lane & 31];
        sum += mw == -INFINITY ? 0.f : s_l[w][lane & 31] * __builtin_amdgcn_exp2f(mw - most);
    }
    const float f = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - most);
    char* const mine = (char*)areas + wave * (AREA * 2);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int g = 0; g < 4; ++g)
            *reinterpret_cast<f32x4*>(mine + ((4 * dt + g) * 64 + lane) * 16) =
                f32x4{o[dt][4 * g] * f, o[dt][4 * g + 1] * f, o[dt][4 * g + 2] * f, o[dt][4 * g + 3] * f};
    __syncthreads();
    const float inv = __builtin_amdgcn_rcpf(sum);   // (approximate reciprocal, fmha.jl:132-134)
    unsigned short* op = O + (int64_t)head * os.s2 + (int64_t)batch * os.s3 + (int64_t)my_q * os.s1 + 8 * hb;
    constexpr int G = 4 * DT / NW;   // groups of four channels per wave
    static_assert(G % 2 == 0, "groups are stored in pairs");
#pragma unroll
    for (int u = 0; u < G; u += 2) {
        const int q = wave * G + u;
        unsigned w[2][2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            f32x4 v = *reinterpret_cast<const f32x4*>((const char*)areas + ((q + e) * 64 + lane) * 16);
#pragma unroll
            for (int x = 1; x < NW; ++x) v += *reinterpret_cast<const f32x4*>((const char*)areas + x * (AREA * 2) + ((q + e) * 64 + lane) * 16);
            w[e][0] = Pack<E>::pack(v[0] * inv, v[1] * inv);
            w[e][1] = Pack<E>::pack(v[2] * inv, v[3] * inv);
        }
        // (two lane halves hold four channels of every eight: an exchange makes each store 16 bytes)
        const auto a = __builtin_amdgcn_permlane32_swap(w[0][0], w[1][0], false, false);
        const auto b = __builtin_amdgcn_permlane32_swap(w[0][1], w[1][1], false, false);
        if (my_q < Sq) *reinterpret_cast<u32x4*>(op + 8 * q) = u32x4{a[0], b[0], a[1], b[1]};
    }
}

template <typename E, int D, int NW>
void launch_t(const Problem& p, hipStream_t stream) {
    const mi_tile_array *Q = p.Q, *K = p.K, *V = p.V, *O = p.O;
    Strides qs{Q->strides[1], Q->strides[2], Q->strides[3]}, ks{K->strides[1], K->strides[2], K->strides[3]},
        vs{V->strides[1], V->strides[2], V->strides[3]}, os{O->strides[1], O->strides[2], O->strides[3]};
    const int Sq = (int)Q->sizes[1], Skv = (int)K->sizes[1], nqt = (Sq + kQT - 1) / kQT, nbh = (int)(Q->sizes[2] * Q->sizes[3]);
    const dim3 grid((unsigned)nqt * nbh), blk(64 * NW);
    if (p.causal)
        hipLaunchKernelGGL((fmha_few_kernel<E, D, true, NW>), grid, blk, 0, stream, (const unsigned short*)Q->ptr, qs, (const unsigned short*)K->ptr, ks,
                           (const unsigned short*)V->ptr, vs, (unsigned short*)O->ptr, os, Sq, Skv, p.H, p.group, p.scale2, p.input_pos, nqt, nbh);
    else
        hipLaunchKernelGGL((fmha_few_kernel<E, D, false, NW>), grid, blk, 0, stream, (const unsigned short*)Q->ptr, qs, (const unsigned short*)K->ptr, ks,
                           (const unsigned short*)V->ptr, vs, (unsigned short*)O->ptr, os, Sq, Skv, p.H, p.group, p.scale2, p.input_pos, nqt, nbh);
}

}  // namespace

Walks walks_of(const Problem& p) {
    const int64_t Sq = p.Q->sizes[1], Skv = p.K->sizes[1], tiles = (Sq + kQT - 1) / kQT, heads = p.Q->sizes[2] * p.Q->sizes[3];
    int64_t last = Skv, first = Skv;   // keys that the last / the first tile of a head sees
    if (p.causal) {
        last = p.input_pos + Sq < Skv ? p.input_pos + Sq : Skv;
        first = p.input_pos + kQT < last ? p.input_pos + kQT : last;
    }
    Walks w;
    w.longest = (double)((last + kHK - 1) / kHK);
    w.tiles = (double)(tiles * heads) / 1024.0;
    w.halves = w.tiles * (w.longest + (double)((first + kHK - 1) / kHK)) / 2.0;
    return w;
}

bool few_applicable(const Problem& p) {
    // MI_FMHA_FEW=0, read at every call: never
    const char* e = getenv("MI_FMHA_FEW");
    if ((e && atoi(e) == 0) || !(p.scale2 > 0.f) || p.Q->sizes[1] <= 64) return false;   // (few queries: a group's heads are stacked in one tile, fmha.hip)
    if (!vec16(p.Q) || !vec16(p.K) || !vec16(p.V) || !vec16(p.O)) return false;
    // (32-bit byte offsets within a half)
    if (p.K->strides[1] < 0 || p.V->strides[1] < 0 || p.K->strides[1] >= (1 << 20) || p.V->strides[1] >= (1 << 20)) return false;
    return (p.Q->sizes[1] + kQT - 1) / kQT * p.Q->sizes[2] * p.Q->sizes[3] <= MI_MAX_GRID_DIM;
}

// Fitted to 198 (heads of 64) and 237 shapes (128): a launch, the longest walk of a wave, and what every SIMD has to do.
double few_estimate(const Problem& p, const Walks& w, int* waves) {
    const double c4 = ceil(w.longest / 4), c2 = ceil(w.longest / 2);
    const bool d64 = p.Q->sizes[0] == 64;
    const double t4 = d64 ? 5.35 + 0.060 * c4 + 0.366 * w.halves + 1.41 * w.tiles : 4.47 + 0.241 * c4 + 0.630 * w.halves + 6.38 * w.tiles;
    const double t2 = d64 ? 4.67 + 0.254 * c2 + 0.318 * w.halves + 0.38 * w.tiles : 4.73 + 0.391 * c2 + 0.527 * w.halves + 2.64 * w.tiles;
    *waves = t4 <= t2 ? 4 : 2;
    // Walks of one length in a last round that is nearly empty (heads of 128, two resp. four workgroups per CU): 1 x 8 heads, 2282 of 1619 keys,
    // 576 workgroups, 29.3 estimated and 35.7 us, 4 x 8, 523 of 4075, 544, 58 : 80, 2 x 16, 608 of 2554, 608, 43 : 52 (slower than two groups
    // by up to 8 %).  The longest walks of a causal launch start first and leave no such tail.
    const double rounds = w.tiles * (*waves == 4 ? 2.0 : 1.0);
    const double tail = d64 || p.causal || rounds <= 1.0 ? 1.0 : 1.0 + 0.45 * (ceil(rounds) / rounds - 1.0);
    // A half of a wave's walk takes 0.8 us by itself, from its request to its products (1 x 8 heads, 136 of 2396 keys 19.7, 4 x 4, 134 of 1384 13.7,
    // 1 x 4, 160 of 637 8.5), with heads of 64 0.55 (1 x 1 to 1 x 16, 65 to 512 of 3300 keys 17, 4000 20, 5120 24: a split takes 15 to 17 there).
    const double alone = (d64 ? 2.2 : 4.0) + (d64 ? 0.545 : 0.8) * (*waves == 4 ? c4 : c2);
    return fmax(tail * (*waves == 4 ? t4 : t2), alone);
}

void few_launch(const Problem& p, int waves, hipStream_t stream) {
#define GO(E, D) (waves == 4 ? launch_t<E, D, 4>(p, stream) : launch_t<E, D, 2>(p, stream))
    if (p.Q->sizes[0] == 64) {
        if (p.bf16) GO(BF16, 64);
        else GO(F16, 64);
        set_variant(waves == 4 ? "fmha_few_d64_q32_keys4" : "fmha_few_d64_q32_keys2");
    } else {
        if (p.bf16) GO(BF16, 128);
        else GO(F16, 128);
        set_variant(waves == 4 ? "fmha_few_d128_q32_keys4" : "fmha_few_d128_q32_keys2");
    }
#undef GO
}

}  // namespace fmha
}  // namespace mi
