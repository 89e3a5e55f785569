// Column softmax: stand-ins for softmax_tma_kernel (examples/softmax.jl:18-42) and
// softmax_chunked_kernel (examples/softmax.jl:48-100) of the reference.
//
// input/output are (N, M) with the softmax dimension N contiguous.  One workgroup owns one
// column at a time.  The single-tile kernel keeps the whole column in registers, so HBM is
// touched exactly once per element each way (algorithmic traffic 2*M*N*sizeof(T)): 16-byte
// loads, wave64 shuffle reductions, one LDS exchange per reduction across the waves of the
// workgroup.  Columns of more than 65536 elements take the reference's three passes (max, denominator,
// normalise), re-reading the column from L2; softmax_chunked_kernel uses the register kernel too whenever
// its column fits.
//
// Numerics follow the reference: fp32 math, max ignores NaN, the exponential of x - max, one correctly rounded
// reciprocal of the sum per column, padding rows read as -Inf and are never written.  The exponential is the library's
// for fp32 columns of up to 16384 elements, else the hardware's 2^x (struct Exp2).
#include "common.h"
#include <math.h>

namespace {

using namespace mi;

template <typename T> struct Raw;  // 16-byte vectors of the storage type
template <> struct Raw<float> {
    typedef float V __attribute__((ext_vector_type(4)));
    static constexpr int EV = 4;
};
template <> struct Raw<__half> {
    typedef _Float16 V __attribute__((ext_vector_type(8)));
    static constexpr int EV = 8;
};
template <> struct Raw<__hip_bfloat16> {
    typedef unsigned short V __attribute__((ext_vector_type(8)));
    static constexpr int EV = 8;
};

template <typename T> __device__ __forceinline__ float vget(const typename Raw<T>::V& v, int q);
template <> __device__ __forceinline__ float vget<float>(const Raw<float>::V& v, int q) { return v[q]; }
template <> __device__ __forceinline__ float vget<__half>(const Raw<__half>::V& v, int q) {
    return (float)v[q];
}
template <> __device__ __forceinline__ float vget<__hip_bfloat16>(const Raw<__hip_bfloat16>::V& v, int q) {
    return __uint_as_float(((unsigned)v[q]) << 16);
}
template <typename T> __device__ __forceinline__ void vset(typename Raw<T>::V& v, int q, float f);
template <> __device__ __forceinline__ void vset<float>(Raw<float>::V& v, int q, float f) { v[q] = f; }
template <> __device__ __forceinline__ void vset<__half>(Raw<__half>::V& v, int q, float f) {
    v[q] = (_Float16)f;
}
template <> __device__ __forceinline__ void vset<__hip_bfloat16>(Raw<__hip_bfloat16>::V& v, int q, float f) {
    v[q] = to_bf16(f);
}

// A 16-byte vector at an address that is aligned for its elements only: global memory takes such accesses, in one
// instruction (a column of 50257 floats starts anywhere).
template <bool STREAM, typename V, typename T>
__device__ __forceinline__ V ld_vec(const T* p) {
    typedef V U __attribute__((aligned(alignof(T))));
    const U* q = reinterpret_cast<const U*>(p);
    return STREAM ? __builtin_nontemporal_load(q) : *q;
}
template <typename V, typename T>
__device__ __forceinline__ void st_vec(V v, T* p) {
    typedef V U __attribute__((aligned(alignof(T))));
    __builtin_nontemporal_store(v, reinterpret_cast<U*>(p));
}

// Barrier that waits for this wave's LDS accesses only: loads and stores stay in flight across it.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
// All-reduce over the workgroup, one barrier: `red` (NW floats) has to be another array than the reduction's before.
template <int NW, typename Op>
__device__ __forceinline__ float reduce(float v, float* red, Op op) {
    v = wave_reduce(v, op);
    if constexpr (NW == 1) return v;
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    lds_barrier();
    v = red[threadIdx.x & (NW - 1)];
#pragma unroll
    for (int off = NW / 2; off >= 1; off >>= 1) v = op(v, __shfl_xor(v, off, 64));
    return v;
}

// exp(x - max) as the hardware's 2^x on (x - max) * log2(e), the product formed by one fma: an error of the argument's
// rounding, |x - max| * 2^-24 relative (3e-6 at 50 below the maximum, where the value is 2e-22).  The rounding of
// max * log2(e) is a factor that every element and their sum share; it is a power of two of at most 1/16 while |max| is
// below 2^20.  A larger maximum (a mask value, an offset) is subtracted first, or that factor would overflow.  The
// subtraction in every column and the multiply by 1 / sum, where 16-bit results once took 2^(x log2 e - (max log2 e +
// log2 sum)) -- off by the rounding of max log2 e, a factor of 2^31 at -1e9 --, cost 1 us of 40 (bf16 1024 x 50257).  (Two
// copies of what follows the maximum, one without the subtraction, spill: 48 us.)  Values below 2^-126 come out as 0.
struct Exp2 {
    float base, shift;
    __device__ __forceinline__ explicit Exp2(float mx) {
        base = fabsf(mx) <= 0x1p20f ? 0.f : mx;   // (an infinite maximum makes the whole column NaN, as x - max does)
        shift = (mx - base) * kLog2e;
    }
    __device__ __forceinline__ float operator()(float x) const {
        return __builtin_amdgcn_exp2f(__builtin_fmaf(x - base, kLog2e, -shift));
    }
    static constexpr float kLog2e = 1.4426950408889634f;
};

// ---- single-tile kernel: column cached in registers -----------------------------------
// Capacity BLOCK*VPT*EV elements.  A column is a scalar head up to its first 16-byte boundary, whole vectors, and a scalar
// tail; head and tail are one element in each of the first lanes.  (Where input and output do not sit at the same
// offset from such a boundary there is no head and the vectors move unaligned.)
// What bounds it is HBM, so everything is about keeping loads in flight:
//   - a lane's vectors are requested together, from addresses clamped to the last vector of the column (its value
//     again changes no maximum, and is left out of the sum and of the stores); behind a per-vector bounds branch each
//     load was waited for before the next was sent;
//   - 16-bit columns stay packed in the registers and their exponentials are made twice, for the sum and for the result:
//     at 1024 lanes a column of 65536 takes 32 of a lane's 64 registers, so two workgroups share a CU;
// Before / now, in three rotating buffers: bf16 1024 x 50257 57 -> 41 us (5.0 TB/s), 4096 x 32768 239 -> 93, 1682 x 28672
// 102 -> 35; f16 2048 x 8191 18.7 -> 11.7, 4096 x 4096 13.1 -> 11.3; fp32 1024 x 50257 92 -> 85, 3000 x 20000 93 -> 82.
// Workgroups that walk the columns and request the next one while they store were no faster (1024 lanes, fp32
// 4096 x 32768: 190 us against 179 with a workgroup per column).
template <typename T, int BLOCK, int VPT, bool STREAM>
__global__ __launch_bounds__(BLOCK, BLOCK == 1024 && VPT <= 8 ? 8 : 1) void softmax_regs_kernel(
    T* __restrict__ out, int64_t ldo, const T* __restrict__ in, int64_t ldi, int L) {
    constexpr int EV = Raw<T>::EV;
    constexpr bool PACKED = sizeof(T) == 2;
    using V = typename Raw<T>::V;
    constexpr int NW = BLOCK / 64;
    __shared__ float red_max[NW], red_sum[NW];
    const float NEG_INF = -INFINITY;
    const int t = threadIdx.x;

    const T* ip = in + blockIdx.x * ldi;
    T* op = out + blockIdx.x * ldo;
    int head = 0;
    {
        const uintptr_t ai = (uintptr_t)ip, ao = (uintptr_t)op;
        if ((ai & 15) == (ao & 15)) head = (int)(((16 - (ai & 15)) & 15) / sizeof(T));
        if (head > L) head = L;
    }
    const int nv = (L - head) / EV;                        // whole vectors
    const bool has1 = t < L - nv * EV;                     // the lane holds an element of head or tail, this one:
    const int e1 = t < head ? t : nv * EV + t;
    V x[VPT];
    if (nv > 0) {
#pragma unroll
        for (int v = 0; v < VPT; ++v) {
            const int i = t + v * BLOCK;
            x[v] = ld_vec<STREAM, V>(ip + head + (i < nv ? i : nv - 1) * EV);
        }
    } else {
#pragma unroll
        for (int v = 0; v < VPT; ++v)
#pragma unroll
            for (int q = 0; q < EV; ++q) vset<T>(x[v], q, NEG_INF);
    }
    float x1 = has1 ? to_f32<T>(ip[e1]) : NEG_INF;
    auto keep_packed = [&]() {   // (or the widened elements of one pass would be kept for the next)
        if constexpr (PACKED)
#pragma unroll
            for (int v = 0; v < VPT; ++v) asm volatile("" : "+v"(x[v]));
    };
    float mx = x1;
#pragma unroll
    for (int v = 0; v < VPT; ++v)
#pragma unroll
        for (int q = 0; q < EV; ++q) mx = fmaxf(mx, vget<T>(x[v], q));
    mx = reduce<NW>(mx, red_max, MaxOp{});
    keep_packed();
    // exp(x - max): where a lane makes many of them and little else runs under them (1024 lanes, or exponentials made
    // twice) by Exp2, three instructions where the library's takes about twenty.
    const Exp2 ex2(mx);
    auto ex = [&](float v) {
        if constexpr (BLOCK == 1024 || PACKED) return ex2(v);
        else return expf(v - mx);
    };
    x1 = ex(x1);
    float sum = has1 ? x1 : 0.f;
#pragma unroll
    for (int v = 0; v < VPT; ++v) {
        float s = 0.f;
#pragma unroll
        for (int q = 0; q < EV; ++q) {
            const float e = ex(vget<T>(x[v], q));
            if constexpr (!PACKED) vset<T>(x[v], q, e);
            s += e;
        }
        sum += t + v * BLOCK < nv ? s : 0.f;
    }
    sum = reduce<NW>(sum, red_sum, SumOp{});
    keep_packed();
    // one correctly rounded reciprocal per column, then multiplies: within 1.5 ulp of the
    // element-wise quotient, at a tenth of the instructions
    const float rsum = 1.0f / sum;
#pragma unroll
    for (int v = 0; v < VPT; ++v) {
        V y;
#pragma unroll
        for (int q = 0; q < EV; ++q) {
            const float e = vget<T>(x[v], q);
            vset<T>(y, q, (PACKED ? ex(e) : e) * rsum);
        }
        const int i = t + v * BLOCK;
        if (i < nv) st_vec<V>(y, op + head + i * EV);
    }
    if (has1) op[e1] = from_f32<T>(x1 * rsum);
}

// ---- three-pass kernel: any column length ---------------------------------------------
// ALIGNED: every column starts on a 16-byte boundary.  Otherwise a column whose input and output sit at the same
// offset from such a boundary (the usual case: equal leading dimensions) is walked as a scalar head up to the
// boundary, 16-byte vectors, and a scalar tail; columns that do not, element by element.
template <typename T, int BLOCK, bool ALIGNED>
__global__ __launch_bounds__(BLOCK) void softmax_3pass_kernel(T* __restrict__ out, int64_t ldo,
                                                              const T* __restrict__ in, int64_t ldi,
                                                              int64_t L, int64_t M) {
    constexpr int EV = Raw<T>::EV;
    using V = typename Raw<T>::V;
    constexpr int NW = BLOCK / 64;
    __shared__ float red[NW];
    const float NEG_INF = -INFINITY;

    for (int64_t col = blockIdx.x; col < M; col += gridDim.x) {
        const T* ip = in + col * ldi;
        T* op = out + col * ldo;
        int64_t head = 0, nvec = L / EV;
        if (!ALIGNED) {
            const uintptr_t ai = (uintptr_t)ip, ao = (uintptr_t)op;
            if ((ai & 15) == (ao & 15) && ai % sizeof(T) == 0) {
                head = (int64_t)(((16 - (ai & 15)) & 15) / sizeof(T));
                if (head > L) head = L;
                nvec = (L - head) / EV;
            } else {
                head = L;
                nvec = 0;
            }
        }
        const T* ipv = ip + head;
        T* opv = op + head;
        const int64_t nscalar = L - nvec * EV;                       // head and tail elements
        auto at = [&](int64_t e) { return e < head ? e : e + nvec * EV; };   // their positions in the column
        // pass 1: running maximum
        float mx = NEG_INF;
#pragma unroll 4
        for (int64_t v = threadIdx.x; v < nvec; v += BLOCK) {
            V raw = *reinterpret_cast<const V*>(ipv + v * EV);
#pragma unroll
            for (int q = 0; q < EV; ++q) mx = fmaxf(mx, vget<T>(raw, q));
        }
        for (int64_t e = threadIdx.x; e < nscalar; e += BLOCK) mx = fmaxf(mx, to_f32<T>(ip[at(e)]));
        mx = block_reduce<NW>(mx, red, MaxOp{}, NEG_INF);
        // (a column this long is walked by one workgroup per CU: the library exponential was most of passes 2 and 3)
        const Exp2 ex(mx);
        // pass 2: per-lane partial denominators, one reduction at the end
        float den = 0.f;
#pragma unroll 4
        for (int64_t v = threadIdx.x; v < nvec; v += BLOCK) {
            V raw = *reinterpret_cast<const V*>(ipv + v * EV);
#pragma unroll
            for (int q = 0; q < EV; ++q) den += ex(vget<T>(raw, q));
        }
        for (int64_t e = threadIdx.x; e < nscalar; e += BLOCK) den += ex(to_f32<T>(ip[at(e)]));
        den = block_reduce<NW>(den, red, SumOp{}, 0.f);
        const float rden = 1.0f / den;   // (one reciprocal per column, then multiplies, as in the register kernel)
        // pass 3: normalise and store
#pragma unroll 4
        for (int64_t v = threadIdx.x; v < nvec; v += BLOCK) {
            V raw = *reinterpret_cast<const V*>(ipv + v * EV);
            V res;
#pragma unroll
            for (int q = 0; q < EV; ++q) vset<T>(res, q, ex(vget<T>(raw, q)) * rden);
            st_global<true>(res, reinterpret_cast<V*>(opv + v * EV));
        }
        for (int64_t e = threadIdx.x; e < nscalar; e += BLOCK)
            op[at(e)] = from_f32<T>(ex(to_f32<T>(ip[at(e)])) * rden);
    }
}

int check(const mi_tile_array* output, const mi_tile_array* input, int TILE_SIZE, int num_programs) {
    MI_CHECK(check_array(output, 2));
    MI_CHECK(check_array(input, 2));
    if (output->dtype != input->dtype) return MI_E_DTYPE;
    if (input->dtype != MI_F32 && input->dtype != MI_F16 && input->dtype != MI_BF16) return MI_E_DTYPE;
    if (!same_shape(output, input)) return MI_E_SHAPE;
    if (!is_pow2(TILE_SIZE)) return MI_E_TILE;
    if (num_programs < 1 || num_programs > MI_MAX_GRID_DIM) return MI_E_GRID;
    if (input->sizes[0] > 1 && (input->strides[0] != 1 || output->strides[0] != 1)) return MI_E_STRIDE;
    return MI_OK;
}

template <typename T>
bool vec_ok(const mi_tile_array* output, const mi_tile_array* input) {
    constexpr int EV = Raw<T>::EV;
    return aligned(input->ptr, 16) && aligned(output->ptr, 16) &&
           (input->sizes[1] <= 1 || (input->strides[1] % EV == 0 && output->strides[1] % EV == 0));
}

template <typename T, int BLOCK, int VPT>
void launch_regs(const mi_tile_array* output, const mi_tile_array* input, int L, bool al,
                 hipStream_t s) {
    const int64_t M = input->sizes[1], ldi = input->strides[1], ldo = output->strides[1];
    const bool stream = al && stream_hint(2 * M * (int64_t)L * (int64_t)sizeof(T));
    constexpr int64_t kMost = 0xffffffffll / BLOCK;   // workgroups of a launch: fewer than 2^32 lanes
    for (int64_t c = 0; c < M; c += kMost) {
        const dim3 grid((unsigned)(M - c < kMost ? M - c : kMost)), block(BLOCK);
        T* op = (T*)output->ptr + c * ldo;
        const T* ip = (const T*)input->ptr + c * ldi;
        if (stream) hipLaunchKernelGGL((softmax_regs_kernel<T, BLOCK, VPT, true>), grid, block, 0, s, op, ldo, ip, ldi, L);
        else hipLaunchKernelGGL((softmax_regs_kernel<T, BLOCK, VPT, false>), grid, block, 0, s, op, ldo, ip, ldi, L);
    }
}

template <typename T>
int launch_3pass(const mi_tile_array* output, const mi_tile_array* input, int64_t L, hipStream_t s) {
    const int64_t M = input->sizes[1];
    const bool al = vec_ok<T>(output, input);
    // (few columns: 1024 lanes each, so that a column has sixteen 16-byte loads per lane-slot in flight, not four)
    const bool wide = M < 1024;
    dim3 grid((unsigned)M), block(wide ? 1024 : 256);
#define GO(B, AL)                                                                                          \
    hipLaunchKernelGGL((softmax_3pass_kernel<T, B, AL>), grid, block, 0, s, (T*)output->ptr, output->strides[1], \
                       (const T*)input->ptr, input->strides[1], L, M)
    if (wide && al) GO(1024, true);
    else if (wide) GO(1024, false);
    else if (al) GO(256, true);
    else GO(256, false);
#undef GO
    set_variant(wide ? "softmax_3pass_b1024" : "softmax_3pass_b256");
    return launch_status();
}

// Softmax over the first L64 rows of every column: the register kernel when the column fits
// (one HBM pass), otherwise three passes.
template <typename T>
int launch_len(const mi_tile_array* output, const mi_tile_array* input, int64_t L64, hipStream_t s) {
    constexpr int EV = Raw<T>::EV;
    if (L64 > 65536) return launch_3pass<T>(output, input, L64, s);
    const int L = (int)L64;
    // (a column that is aligned as a whole: its last vector may still cross the end, which the kernel handles)
    const bool al = vec_ok<T>(output, input);
    const int vecs = (int)cld(L, EV);
    if (vecs > 256 * 16) {
        // Up to 65536 elements in the registers of 1024 lanes: one pass over HBM where the three-pass kernel re-reads the
        // column twice (1024 x 50257 fp32: 121 us).  As many vectors per lane as the column needs: a lane past the end
        // requests the last vector again, which costs an access all the same (2000 x 40000 bf16: 5 per lane 56.3 us, 8
        // per lane 59.1).
        const int per = (int)cld(vecs, 1024);
#define WIDE(V) launch_regs<T, 1024, V>(output, input, L, al, s)
        if (per <= 5) WIDE(5);
        else if (per <= 6) WIDE(6);
        else if (per <= 7) WIDE(7);
        else if (per <= 8) WIDE(8);
        if constexpr (EV == 4) {
            if (per > 12) WIDE(16);
            else if (per > 10) WIDE(12);
            else if (per > 8) WIDE(10);
        }
#undef WIDE
        set_variant(L > 32768 ? "softmax_regs_b1024_e64" : "softmax_regs_b1024_e32");   // (at most 64 / 32 elements per lane)
        return launch_status();
    }
    if (vecs <= 64) { launch_regs<T, 64, 1>(output, input, L, al, s); set_variant("softmax_regs_b64_v1"); }
    else if (vecs <= 128) { launch_regs<T, 64, 2>(output, input, L, al, s); set_variant("softmax_regs_b64_v2"); }
    else if (vecs <= 256) { launch_regs<T, 64, 4>(output, input, L, al, s); set_variant("softmax_regs_b64_v4"); }   // one wave per column: no barriers
    else if (vecs <= 512) { launch_regs<T, 256, 2>(output, input, L, al, s); set_variant("softmax_regs_b256_v2"); }
    else if (vecs <= 1024) { launch_regs<T, 256, 4>(output, input, L, al, s); set_variant("softmax_regs_b256_v4"); }
    else if (vecs <= 2048) { launch_regs<T, 256, 8>(output, input, L, al, s); set_variant("softmax_regs_b256_v8"); }
    else { launch_regs<T, 256, 16>(output, input, L, al, s); set_variant("softmax_regs_b256_v16"); }
    return launch_status();
}

}  // namespace

extern "C" int mi_softmax_tma_kernel(const mi_tile_array* output, const mi_tile_array* input,
                                     int TILE_SIZE, int num_programs, void* stream) {
    MI_CHECK(check(output, input, TILE_SIZE, num_programs));
    if (input->sizes[0] == 0 || input->sizes[1] == 0) return MI_OK;
    if (input->sizes[1] > 0x7fffffffLL) return MI_E_GRID;
    hipStream_t s = (hipStream_t)stream;
    const int64_t L = input->sizes[0] < TILE_SIZE ? input->sizes[0] : (int64_t)TILE_SIZE;  // one tile per column
    switch (input->dtype) {
        case MI_F32: return launch_len<float>(output, input, L, s);
        case MI_F16: return launch_len<__half>(output, input, L, s);
        default: return launch_len<__hip_bfloat16>(output, input, L, s);
    }
}

extern "C" int mi_softmax_chunked_kernel(const mi_tile_array* output, const mi_tile_array* input,
                                         int n_elems, int TILE_SIZE, int num_programs, void* stream) {
    MI_CHECK(check(output, input, TILE_SIZE, num_programs));
    if (n_elems < 0) return MI_E_ARG;
    if (input->sizes[0] == 0 || input->sizes[1] == 0) return MI_OK;
    if (input->sizes[1] > 0x7fffffffLL) return MI_E_GRID;
    // The chunk loop visits rows 1 .. cld(n_elems, TILE_SIZE)*TILE_SIZE; rows past the
    // array's end are padding (softmax.jl:58, 65-69).
    int64_t L = cld((int64_t)n_elems, (int64_t)TILE_SIZE) * TILE_SIZE;
    if (L > input->sizes[0]) L = input->sizes[0];
    if (L == 0) return MI_OK;
    hipStream_t s = (hipStream_t)stream;
    switch (input->dtype) {
        // Same function of the column as the reference's three chunked passes; a column that
        // fits in registers is read from HBM once instead.
        case MI_F32: return launch_len<float>(output, input, L, s);
        case MI_F16: return launch_len<__half>(output, input, L, s);
        default: return launch_len<__hip_bfloat16>(output, input, L, s);
    }
}
