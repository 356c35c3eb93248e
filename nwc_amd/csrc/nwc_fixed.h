// nwc_fixed.h -- the decode of layout 2's fixed-width ranks and exception lists, shared by its kernels.
#pragma once
#include "nwc_device.h"

namespace nwc {

struct RankTab { uint32_t T0, T1, U0, U1; };   // table byte of ranks 0..7; low-byte bit 7 of ranks 0..7 (fp8)

// 8 positions (one nibble word) -> the high bytes of positions 0..3 and 4..7 of the word, BF16 byte order
__device__ __forceinline__ void ranks8(const RankTab &t, uint32_t nw, uint32_t &h03, uint32_t &h47, uint32_t &l03, uint32_t &l47, bool fp8) {
    const uint32_t a = nw & 0x0F0F0F0Fu;                 // nibbles of positions 0, 2, 4, 6
    const uint32_t b = (nw >> 4) & 0x0F0F0F0Fu;          // positions 1, 3, 5, 7
    const uint32_t ra = a & 0x07070707u, rb = b & 0x07070707u;
    const uint32_t ha = perm(t.T1, t.T0, ra) | ((a << 4) & 0x80808080u);
    const uint32_t hb = perm(t.T1, t.T0, rb) | ((b << 4) & 0x80808080u);
    h03 = perm(hb, ha, 0x05010400u);
    h47 = perm(hb, ha, 0x07030602u);
    if (fp8) {
        const uint32_t la = perm(t.U1, t.U0, ra), lb = perm(t.U1, t.U0, rb);
        l03 = perm(lb, la, 0x05010400u);
        l47 = perm(lb, la, 0x07030602u);
    } else {
        l03 = l47 = 0u;
    }
}
// BF16 pairs of positions (0,1) and (2,3) of a 4-position group: [low0 | high0][low1 | high1]
constexpr uint32_t kSelLoHi01 = 0x05010400u;
constexpr uint32_t kSelLoHi23 = 0x07030602u;

// bits 12G .. 12G+11 (and what follows them above) of the 96-bit little-endian integer w2:w1:w0 (G a compile-time constant after unrolling)
__device__ __forceinline__ uint32_t bits12(uint32_t w0, uint32_t w1, uint32_t w2, int G) {
    const int bit = 12 * G, k = bit >> 5, sh = bit & 31;
    const uint32_t lo = k == 0 ? w0 : k == 1 ? w1 : w2, hi = k == 0 ? w1 : k == 1 ? w2 : 0u;
    return __builtin_amdgcn_alignbit(hi, lo, (uint32_t)sh);
}

__device__ __forceinline__ float e4m3_to_f32(uint32_t b) {
    const uint32_t e = (b >> 3) & 15u, m = b & 7u;
    const float v = e ? __uint_as_float(((e + 120u) << 23) | (m << 20)) : (float)m * 0.001953125f;
    return (b & 0x80u) ? -v : v;
}

template <int ELEM>
__device__ __forceinline__ float exc_value(const uint8_t *e) {
    if (ELEM == kElemFp8) return e4m3_to_f32(e[1]);
    return __uint_as_float(((uint32_t)e[1] | ((uint32_t)e[2] << 8)) << 16);
}

// fp8: the four 3-bit fields of a 12-bit value, each in bits 4..6 of its byte (six operations; a 4096-entry LDS table
// instead cost a random read per four weights and its staging: k_layout2s, 6144 x 2560 fp8, 17.5 us with it)
__device__ __forceinline__ uint32_t mant4(uint32_t v) {
    const uint32_t y = (v & 0x3Fu) | ((v << 10) & 0x3F0000u);
    return ((y << 4) | (y << 9)) & 0x70707070u;
}

// Decodes one super-chunk of a lane: p[k] = BF16 pair of row r (positions 4k, 4k+1), q[k] = pair of row r+8.
template <int ELEM, int G0>
__device__ __forceinline__ void decode_sc(const RankTab &t, uint2 nib, uint4 raw, uint32_t c0, uint32_t c1, uint32_t c2,
                                          uint32_t p[4], uint32_t q[4]) {
#pragma unroll
    for (int h = 0; h < 2; h++) {
        uint32_t h03, h47, l03, l47;
        ranks8(t, h ? nib.y : nib.x, h03, h47, l03, l47, ELEM == kElemFp8);
        uint32_t r0, r1;                                          // low bytes of positions 8h+0..3 and 8h+4..7
        if (ELEM == kElemFp8) {
            r0 = mant4(bits12(c0, c1, c2, G0 + 2 * h)) | l03;
            r1 = mant4(bits12(c0, c1, c2, G0 + 2 * h + 1)) | l47;
        } else {
            r0 = h ? raw.z : raw.x;
            r1 = h ? raw.w : raw.y;
        }
        p[2 * h] = perm(h03, r0, kSelLoHi01);
        q[2 * h] = perm(h03, r0, kSelLoHi23);
        p[2 * h + 1] = perm(h47, r1, kSelLoHi01);
        q[2 * h + 1] = perm(h47, r1, kSelLoHi23);
    }
}

// start of this lane's exception entries in block b (prefix over the half's counts)
__device__ __forceinline__ const uint8_t *exc_start(const BlockArgs &a, uint32_t b, uint32_t L, uint32_t esz, uint32_t &cnt) {
    cnt = a.hdr[(uint64_t)b * kHdrBytes + L];
    const uint32_t incl = half_scan_incl(cnt, L);
    return a.data + a.bases[b] + (uint64_t)(incl - cnt) * esz;
}

}  // namespace nwc
