// Numbering of the pipelined attention kernel's workgroups (fmha_pipe128.hip): which query block of which head a workgroup
// id is.  Plain C++, so that it is checked on the CPU as well.
//
// Workgroup ids congruent mod 8 share an XCD: an XCD gets whole key / value heads (all query heads of a group with
// theirs) where their number allows it.  Within an XCD the ids walk `chunk` heads at a time, the query blocks with the
// longest key ranges first: as many heads as fill the XCD's 64 slots (two workgroups per CU), so that few K / V share
// its L2 at a time (4 x 32 ungrouped heads, S = 2048: 154 us, 158 with all heads at once, 163 with half as many).
// The last group of a causal launch takes up to two chunks, so that the walks that start last are short ones (us, all
// chunks alike -> so: 4 x 12 heads, 2054 87 -> 74, 4 x 6, 4944 210 -> 181, 8 x 8, 1716 76 -> 67, 8 x 16, 673 40 -> 34; heads that
// no XCD has to itself, 512 slots: 4 x 7, 3433 149 -> 108, 5 x 6, 3755 164 -> 135).
#pragma once
#include <stdint.h>

#ifdef __HIPCC__
#define MI_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define MI_HOST_DEVICE inline
#endif

namespace mi {
namespace fmha {

// Division by a launch constant: a multiply-high with floor(2^32 / d) + 1, exact while x * d < 2^32 (make_map sees to it).
struct Magic {
    unsigned d, m;
    MI_HOST_DEVICE unsigned div(unsigned x) const { return m ? (unsigned)(((uint64_t)x * m) >> 32) : x; }   // (m = 0: d = 1)
};
inline Magic magic(int d) { return Magic{(unsigned)d, d <= 1 ? 0u : (unsigned)((1ull << 32) / (unsigned)d) + 1u}; }

struct Map {
    Magic span, heads, heads_last, gm, H, group;
    int nx, nfull;   // XCDs told apart; groups of `heads` heads, the rest is the last group

    MI_HOST_DEVICE void at(unsigned id, int nqb, bool causal, int* qb, int* bh) const {
        const unsigned x = nx == 8 ? id & 7u : 0u, idx = nx == 8 ? id >> 3 : id;
        unsigned cg = span.div(idx);
        if (cg > (unsigned)nfull) cg = nfull;
        const unsigned r = idx - cg * span.d, h0 = cg * heads.d;
        const bool last = cg == (unsigned)nfull;
        const unsigned qi = last ? heads_last.div(r) : heads.div(r);
        const unsigned b = h0 + r - qi * (last ? heads_last.d : heads.d), bg = gm.div(b);
        *qb = causal ? nqb - 1 - (int)qi : (int)qi;
        *bh = (int)((x + nx * bg) * gm.d + b - bg * gm.d);
    }
};

// True where every division of the workgroup id is exact with chunks for an XCD's 64 slots, which every launch can take.
inline bool map_exact(int64_t nqb, int64_t nbh, int64_t H) {
    return nqb * nbh * (128 + 2 * nqb) < (1ll << 32) && nbh * (H > 128 ? H : 128) < (1ll << 32);
}

inline Map make_map(int nqb, int nbh, int H, int group, bool causal) {
    const int nkv = nbh / group;
    const int nx = nkv % 8 == 0 || nbh % 8 == 0 ? 8 : 1, gm = nkv % 8 == 0 ? group : 1, nloc = nbh / nx;
    // (ids times the span of a chunk, at most 511 + nqb or 63 + nqb, stay below 2^32; every other division is of fewer ids)
    const bool spread = nx == 1 && causal && (int64_t)nqb * nbh * (511 + nqb) < (1ll << 32);
    int chunk = ((spread ? 512 : 64) + nqb - 1) / nqb;
    if (chunk > nloc) chunk = nloc;
    int nfull = (nloc + chunk - 1) / chunk - 1;
    if (causal && nfull > 0) --nfull;
    const int rest = nloc - nfull * chunk;
    return Map{magic(chunk * nqb), magic(chunk), magic(rest), magic(gm), magic(H), magic(group), nx, nfull};
}

}  // namespace fmha
}  // namespace mi
