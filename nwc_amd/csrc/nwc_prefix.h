// nwc_prefix.h -- parts that the kernels of the prefix-coded layouts 0 and 1 share: staging of a tile's lane streams and of
// the decode table in LDS, the cursor's steps over one row, and layout 1's block coordinates.
#pragma once
#include "nwc_device.h"

namespace nwc {

// Bit position where part j (0-3) of block b starts in lane L's stream: 0 for the first part, else row-index entry
// j - 1.  The entry is loaded for every part (the first part's load reads entry 0 and drops it): a load inside a branch
// makes the compiler wait at the branch's end for it and for every request before it, which would hold back the
// stream copy by a whole round trip.  Callers request it after their other prologue loads (the compiler may read its
// register as the don't-care high half of a 64-bit multiply-add operand, which would wait for it).
__device__ __forceinline__ uint32_t part_start(const BlockArgs &a, uint32_t b, uint32_t j, uint32_t L) {
    const uint32_t v = a.aux[((uint64_t)b * kRowIndexSplits + (j ? j - 1u : 0u)) * kLanes + L];
    return j ? v : 0u;
}

// ---- workgroup staging of the streams of a run of consecutive blocks ----
// The blocks of a workgroup's tile are consecutive in `data`, so a round of H blocks (one per half-wave) is one
// contiguous byte range: [bases[b_lo], bases[b_hi]) -- for the matrix's last block, its base plus four bytes per header
// word.  All threads copy it into LDS with 16-byte loads; no half-wave needs its own header scan before the copy.
// With fixed slots (stride != 0) the range is [b_lo * stride, b_hi * stride) and nothing is read to find it.
struct Region {
    uint32_t lo16, n16;         // 16-byte aligned start (byte offset into data), 16-byte chunks
};

// One past the last stream byte of the matrix (block nb - 1: its base plus four bytes per header word).
__device__ __forceinline__ uint32_t matrix_end(const BlockArgs &a, uint32_t nb) {
    const uint32_t *h = (const uint32_t *)(a.hdr + (uint64_t)(nb - 1u) * kHdrBytes);
    uint32_t words = 0;
#pragma unroll
    for (int i = 0; i < (int)kHdrBytes / 4; i++) words = __builtin_amdgcn_udot4(h[i], 0x01010101u, words, false);
    return a.bases[nb - 1u] + 4u * words;
}

// Blocks [b_lo, b_hi) plus the 16 bytes the last lane's window reads past its stream (inside the 64 slack bytes that
// follow the matrix's last block, or the 128 after its last slot).  stride: a.stride (fixed slots) or 0 (bases[]).
__device__ __forceinline__ Region region_of(const BlockArgs &a, uint32_t b_lo, uint32_t b_hi, uint32_t nb, uint32_t mend,
                                            uint32_t stride) {
    Region r;
    if (stride) {
        r.lo16 = b_lo * stride;                                 // a multiple of 16
        r.n16 = ((b_hi > b_lo ? b_hi - b_lo : 0u) * stride + 31u) >> 4;
        return r;
    }
    const uint32_t s = a.bases[b_lo], e = a.bases[min(b_hi, nb - 1u)];
    r.lo16 = s & ~15u;
    r.n16 = ((b_hi < nb ? e : mend) + 16u - r.lo16 + 15u) >> 4;
    return r;
}

// Four 16-byte chunks per thread cover a region buffer of up to 512 words per half-wave; native vectors keep the
// words in registers.  Only chunks inside the region are requested (a wave wholly past it issues nothing): the
// prologue's vector-memory instructions all pass through the CU's address unit, so a workgroup that requested its
// full four chunks per thread would delay the other workgroup on its CU (o_proj: 9.3 -> 8.7 us).
struct Bulk {
    u32x4_t v0, v1, v2, v3;
};
__device__ __forceinline__ void bulk_issue(Bulk &B, const uint8_t *__restrict__ data, const Region &r, uint32_t tid, uint32_t nth) {
    const uint8_t *p = data + r.lo16;
    if (tid < r.n16) B.v0 = *(const u32x4_t *)(p + 16u * tid);
    if (tid + nth < r.n16) B.v1 = *(const u32x4_t *)(p + 16u * (tid + nth));
    if (tid + 2u * nth < r.n16) B.v2 = *(const u32x4_t *)(p + 16u * (tid + 2u * nth));
    if (tid + 3u * nth < r.n16) B.v3 = *(const u32x4_t *)(p + 16u * (tid + 3u * nth));
}
__device__ __forceinline__ void bulk_commit(const Bulk &B, uint32_t *buf, const Region &r, uint32_t tid, uint32_t nth) {
    if (tid < r.n16) *(u32x4_t *)(buf + 4u * tid) = B.v0;
    if (tid + nth < r.n16) *(u32x4_t *)(buf + 4u * (tid + nth)) = B.v1;
    if (tid + 2u * nth < r.n16) *(u32x4_t *)(buf + 4u * (tid + 2u * nth)) = B.v2;
    if (tid + 3u * nth < r.n16) *(u32x4_t *)(buf + 4u * (tid + 3u * nth)) = B.v3;
}

// The table entries of one row's 16 weights for one lane (four steps of the cursor; a step that was not fast in some
// lane is redone code by code by the whole wave), kept apart from their use so that a row can be decoded before its
// raw bytes have arrived.
template <int ELEM, class Tab>
__device__ __forceinline__ void row_codes(Seq<ELEM> &S, const Tab &s, uint32_t (&e1)[4], uint32_t (&e2)[4]) {
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const uint32_t s0 = S.s;
        const uint32_t *wp0 = S.wp;
        if (__builtin_expect(__any(S.fast_quad(s, e1[k], e2[k]) >= kSeqSlowTest), 0)) {
            S.s = s0;
            S.wp = wp0;
            S.reload();
            S.slow_quad(s, e1[k], e2[k]);
        }
    }
}
// Staging of the decode table: the stored 12-bit LUT, re-encoded (PEEK 12), or the prepared 13-bit table (PEEK 13).
template <int PEEK> struct TabStage;
// issue: the first chunks of the decode table; commit: store them; finish: the chunks a small workgroup has left,
// called after every request that must not wait for the streams (lut_finish says why)
template <> struct TabStage<kPeek> {
    LutLoad Q;
    __device__ __forceinline__ void issue(const BlockArgs &a, uint32_t nth = blockDim.x) { lut_issue(Q, a.lut, nth); }
    __device__ __forceinline__ void commit(LutLds &s, uint32_t nth = blockDim.x) { lut_commit<kLutSeq>(s, Q, nth); }
    __device__ __forceinline__ void finish(LutLds &s, const BlockArgs &a, uint32_t nth = blockDim.x) {
        lut_finish<kLutSeq>(s, a.lut, nth);
    }
};
template <> struct TabStage<kPeekSeq> {
    SeqLoad Q;
    __device__ __forceinline__ void issue(const BlockArgs &a, uint32_t nth = blockDim.x) { seq_issue(Q, a.seq, nth); }
    __device__ __forceinline__ void commit(LutLds13 &s, uint32_t nth = blockDim.x) { seq_commit(s, Q, nth); }
    __device__ __forceinline__ void finish(LutLds13 &s, const BlockArgs &a, uint32_t nth = blockDim.x) {
        seq_finish(s, a.seq, nth);
    }
};

// ---- layout 1 ----
template <int ELEM>
__device__ __forceinline__ uint4 raw_slot1(const uint8_t *__restrict__ p) {
    if (ELEM == kElemFp8) return expand_nibbles(ldnt2(p));
    return ldnt4(p);
}

struct Coord1 {
    uint32_t g, cb, b, rb, nsc;
    uint32_t ro;                // byte offset in `low` of the lane's raw bytes of super-chunk 0 of the block
};
template <int ELEM>
__device__ __forceinline__ Coord1 coord1(uint32_t t, uint32_t rg0, const Shape &f, uint32_t L) {
    constexpr uint32_t RB = ELEM == kElemFp8 ? 8u : 16u;
    Coord1 c;
    c.g = t / f.CB;
    c.cb = t - c.g * f.CB;
    c.rb = rg0 + c.g;
    c.b = c.rb * f.CB + c.cb;
    c.nsc = c.cb == f.CB - 1u ? f.nsl : 16u;
    c.ro = ((c.rb * f.spr + c.cb * 16u) * kLanes + L) * RB;
    return c;
}
// Raw super-chunk sc of a block; past the block's last super-chunk it re-reads the last, so loads stay unconditional.
// 32-bit offsets (the plane is below 4 GB: M * K16 < 2^32) keep one address register per load.
template <int ELEM>
__device__ __forceinline__ uint4 raw1(const uint8_t *__restrict__ low, const Coord1 &c, uint32_t sc) {
    constexpr uint32_t RB = ELEM == kElemFp8 ? 8u : 16u;
    return raw_slot1<ELEM>(low + (c.ro + min(sc, c.nsc - 1u) * (kLanes * RB)));
}
}  // namespace nwc
