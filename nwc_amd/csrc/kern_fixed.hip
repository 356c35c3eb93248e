// kern_fixed.hip -- gfx950 kernels for layout 2 (format v11): fixed-width [sign | rank] nibbles, a raw plane and
// per-lane exception lists, in layout 1's 16 x 512 blocks and fragment order (docs/format.md section 4d).
//
// No bit window: per lane and 32-column super-chunk one 8-byte nibble load, one 16-byte raw load (fp8: three words
// per super-chunk pair) and one 16-byte activation load.  Eight ranks at a time go through v_perm_b32 against the
// 8-byte rank table held in two registers; signs come from bit 3 of the nibbles; BF16 pairs for v_dot2_f32_bf16
// are assembled with two more v_perm_b32.  Exceptions (rank 7, planes zero) are added after the super-chunks.
#include "nwc_fixed.h"
#include "nwc_launch.h"

namespace nwc {

template <int ELEM, int MODE, bool XBF16>
__global__ void __launch_bounds__(1024) k_layout2(BlockArgs a) {
    extern __shared__ float part[];
    const RankTab tab{a.lut[0], a.lut[1], a.lut[2], a.lut[3]};
    constexpr uint32_t esz = ELEM == kElemFp8 ? 2u : 3u;
    const uint32_t tid = threadIdx.x, L = tid & 31, r = L >> 2, q = L & 3;
    const uint32_t hw = tid >> 5, nhw = blockDim.x >> 5;
    const Shape f(a.M, a.K, 2);
    const uint8_t *rplane = a.low + f.nib2_bytes();
    const uint32_t rg0 = blockIdx.x * a.G;
    const uint32_t ng = min(a.G, f.groups() - rg0);
    const RowFinish fin = row_finish_load<MODE, ELEM == kElemFp8>(a, rg0 * kRows12, ng * kRows12);
    const uint32_t nt = ng * f.CB;

    for (uint32_t t = hw; t < nt; t += nhw) {
        const uint32_t g = t / f.CB, cb = t - g * f.CB, rb = rg0 + g, b = rb * f.CB + cb;
        const uint32_t row0 = rb * kRows12;
        const uint32_t nsc = ((cb == f.CB - 1 ? f.nl : 32u) + 1) / 2, slot0 = rb * f.spr + cb * 16;
        const uint8_t *np = a.low + ((uint64_t)slot0 * kLanes + L) * 8;
        const uint8_t *rp = ELEM == kElemFp8 ? rplane + (((uint64_t)rb * f.spr2 + cb * 8) * 3 * kLanes + L) * 4
                                             : rplane + ((uint64_t)slot0 * kLanes + L) * 16;
        float accA = 0.f, accB = 0.f;

        auto consume = [&](uint32_t sc, const uint32_t p[4], const uint32_t qq[4]) {
            const uint32_t kc = cb * kCols + sc * 32 + 8 * q;
            if (MODE == kDequant) {
                if (kc < f.K16) {
                    uint16_t *o = (uint16_t *)a.out + (uint64_t)row0 * f.K16 + kc;
                    if (row0 + r < f.M) *(uint4 *)(o + (uint64_t)r * f.K16) = make_uint4(p[0], p[1], p[2], p[3]);
                    if (row0 + r + 8 < f.M) *(uint4 *)(o + (uint64_t)(r + 8) * f.K16) = make_uint4(qq[0], qq[1], qq[2], qq[3]);
                }
            } else if (XBF16) {
                const uint4 xv = kc + 8u <= f.K || f.K < 16u ? *(const uint4 *)((const uint16_t *)a.x + kc)
                                                             : x8_tail((const uint16_t *)a.x, kc, f.K);
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    accA = dot2_bf16(p[k], u4_get(xv, k), accA);
                    accB = dot2_bf16(qq[k], u4_get(xv, k), accB);
                }
            } else {
                const float4 x0 = ((const float4 *)((const float *)a.x + kc))[0], x1 = ((const float4 *)((const float *)a.x + kc))[1];
                const float xf[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    accA = fmaf(bf16_lo(p[k]), xf[2 * k], accA); accA = fmaf(bf16_hi(p[k]), xf[2 * k + 1], accA);
                    accB = fmaf(bf16_lo(qq[k]), xf[2 * k], accB); accB = fmaf(bf16_hi(qq[k]), xf[2 * k + 1], accB);
                }
            }
        };

        if (ELEM == kElemFp8) {
            const uint32_t nsp = (nsc + 1) / 2;
            for (uint32_t sp = 0; sp < nsp; sp++) {
                const uint8_t *pp = rp + (uint64_t)sp * 3 * kLanes * 4;
                const uint32_t c0 = ldnt1(pp);
                const uint32_t c1 = ldnt1((pp + kLanes * 4));
                const uint32_t c2 = ldnt1((pp + 2 * kLanes * 4));
                uint32_t p[4], qq[4];
                const uint2 n0 = ldnt2((np + (uint64_t)(2 * sp) * kLanes * 8));
                decode_sc<ELEM, 0>(tab, n0, make_uint4(0, 0, 0, 0), c0, c1, c2, p, qq);
                consume(2 * sp, p, qq);
                if (2 * sp + 1 < nsc) {
                    const uint2 n1 = ldnt2((np + (uint64_t)(2 * sp + 1) * kLanes * 8));
                    decode_sc<ELEM, 4>(tab, n1, make_uint4(0, 0, 0, 0), c0, c1, c2, p, qq);
                    consume(2 * sp + 1, p, qq);
                }
            }
        } else {
            uint2 nn = ldnt2(np);
            uint4 rr = ldnt4(rp);
            for (uint32_t sc = 0; sc < nsc; sc++) {
                const uint2 nib = nn;
                const uint4 raw = rr;
                if (sc + 1 < nsc) {
                    nn = ldnt2((np + (uint64_t)(sc + 1) * kLanes * 8));
                    rr = ldnt4((rp + (uint64_t)(sc + 1) * kLanes * 16));
                }
                uint32_t p[4], qq[4];
                decode_sc<ELEM, 0>(tab, nib, raw, 0u, 0u, 0u, p, qq);
                consume(sc, p, qq);
            }
        }

        // exceptions: planes decoded to +-0, the entries carry the value
        uint32_t cnt;
        const uint8_t *ep = exc_start(a, b, L, esz, cnt);
        float eA = 0.f, eB = 0.f;
        for (uint32_t k = 0; k < cnt; k++, ep += esz) {
            const uint32_t i = ep[0], j = i & 15;
            const uint32_t col = cb * kCols + (i >> 4) * 32 + frag_col(L, j), upper = (j >> 1) & 1u;
            const float w = exc_value<ELEM>(ep);
            if (MODE == kDequant) {
                ((uint16_t *)a.out)[(uint64_t)(row0 + r + 8 * upper) * f.K16 + col] = (uint16_t)f32_to_bf16_rne(w);
                continue;
            }
            const float xv = XBF16 ? __uint_as_float((uint32_t)((const uint16_t *)a.x)[col] << 16) : ((const float *)a.x)[col];
            if (upper) eB = fmaf(w, xv, eB); else eA = fmaf(w, xv, eA);
        }
        if (MODE != kDequant) {
            accA += eA; accB += eB;
            accA += xor_f<1>(accA); accA += xor_f<2>(accA);
            accB += xor_f<1>(accB); accB += xor_f<2>(accB);
            if (q == 0) {
                part[(g * kRows12 + r) * f.CB + cb] = accA;
                part[(g * kRows12 + r + 8) * f.CB + cb] = accB;
            }
        }
    }
    if (MODE != kDequant) finish_rows<MODE>(a, part, rg0 * kRows12, ng * kRows12, f.CB, ELEM == kElemFp8 ? &fin : nullptr);
}

// A lane's exceptions, entries first, first + SP, ... (the SP half-waves of a block share them out: any of them can add any
// entry, so each meets a quarter of the longest list of its lanes instead of reading all of it), N at a time.  The first
// batch is in flight while the super-chunks decode; one dependent load per entry after them cost a memory round trip each.
template <int ELEM, int SP>
struct Exceptions {
    static constexpr uint32_t N = (ELEM == kElemFp8 ? 4 : 2) * (SP == 4 ? 1 : 2), SIZE = ELEM == kElemFp8 ? 2 : 3;
    typedef __attribute__((address_space(1))) const uint8_t byte_t;
    typedef __attribute__((address_space(1), aligned(1))) const uint16_t any16_t;
    byte_t *ep;
    uint32_t cnt, next, v[N], top[N];
    // a lane without entries reads bytes that are there (its block's header), never past `data`; the pointer is kept
    // from the compiler, which would branch around the loads and wait inside the branch
    __device__ __forceinline__ void init(const BlockArgs &a, uint32_t L, uint32_t n, uint32_t base, uint32_t first) {
        cnt = n;
        next = first;
        const uint32_t incl = half_scan_incl(n, L);
        uint64_t e = (uint64_t)(n ? a.data + base + (incl - n) * SIZE : a.hdr);
        asm volatile("" : "+v"(e));
        ep = (byte_t *)e;
    }
    __device__ __forceinline__ void request() {                  // past the last entry: the last again
        const uint32_t last = max(cnt, 1u) - 1u;
#pragma unroll
        for (uint32_t k = 0; k < N; k++) {
            byte_t *e = ep + min(next + k * SP, last) * SIZE;
            v[k] = *(any16_t *)e;
            if constexpr (ELEM != kElemFp8) top[k] = e[2];
        }
    }
    __device__ __forceinline__ bool has(uint32_t k) const { return next + k * SP < cnt; }
    __device__ __forceinline__ float value(uint32_t k) const {
        if constexpr (ELEM == kElemFp8) return e4m3_to_f32((v[k] >> 8) & 0xFFu);
        return __uint_as_float(top[k] << 24 | (v[k] & 0xFF00u) << 8);
    }
};

// Token path: a workgroup owns G whole 16-row groups; each half-wave decodes super-chunks sc0 .. sc0 + NS - 1 of a block
// (SP = 16 / NS half-waves per block, so small matrices still fill the CUs; several blocks in turn when the tile has more
// than fit), with its nibble and raw loads four super-chunks ahead, the BF16 activations staged once per workgroup in
// LDS, and its share of its lane's exceptions (the fp32 path keeps k_layout2 and its fp32
// products).  Partial row sums per (row, column block, part), summed in a fixed order by the workgroup.  The fixed-width
// format needs no index to start inside a block.
template <int ELEM, int NS>
__global__ void __launch_bounds__(1024) k_layout2s(BlockArgs a) {
    static_assert(NS == 4 || NS == 8 || NS == 16, "four, two or one half-wave per block");
    constexpr uint32_t SP = 16u / NS, R = 4;
    constexpr bool FP8 = ELEM == kElemFp8;
    extern __shared__ uint32_t dyn[];
    const RankTab tab{a.lut[0], a.lut[1], a.lut[2], a.lut[3]};
    const uint32_t tid = threadIdx.x, nth = blockDim.x, L = tid & 31, r = L >> 2, q = L & 3;
    const uint32_t hw = tid >> 5, H = nth >> 5;
    const Shape f(a.M, a.K, 2);
    const uint32_t n8 = (f.K16 + 31u) / 32u * 4u;                   // x: K32 BF16 values, in chunks of eight
    uint4 *xs = (uint4 *)dyn;
    float *part = (float *)(xs + n8);
    const uint8_t *rplane = a.low + f.nib2_bytes();
    const uint32_t rg0 = blockIdx.x * a.G;
    const uint32_t ng = min(a.G, f.groups() - rg0);
    const uint32_t nt = ng * f.CB;
    const RowFinish fin = row_finish_load<kToken, FP8>(a, rg0 * kRows12, ng * kRows12);
    for (uint32_t i = tid; i < n8; i += nth) xs[i] = x8_settle<true>(x8_at<true>(a.x, 8u * i, f.K), 8u * i, f.K);
    __syncthreads();
    for (uint32_t it = hw; it < nt * SP; it += H) {
        const uint32_t t = it / SP, p = it - t * SP;
        const uint32_t g = t / f.CB, cb = t - g * f.CB, rb = rg0 + g, b = rb * f.CB + cb;
        const uint32_t nsc = ((cb == f.CB - 1 ? f.nl : 32u) + 1) / 2, slot0 = rb * f.spr + cb * 16;
        const uint32_t sc0 = p * NS, ns = sc0 < nsc ? min(NS, nsc - sc0) : 0u;
        const uint32_t cnt = a.hdr[(uint64_t)b * kHdrBytes + L], base = a.bases[b];
        const uint8_t *np = a.low + ((uint64_t)(slot0 + sc0) * kLanes + L) * 8;
        const uint8_t *rp = FP8 ? rplane + (((uint64_t)rb * f.spr2 + cb * 8 + sc0 / 2) * 3 * kLanes + L) * 4
                                : rplane + ((uint64_t)(slot0 + sc0) * kLanes + L) * 16;
        // the ring: super-chunk i of the range in slot i % R (fp8: the three words of chunks i, i + 1 in slot i % R, i
        // even); loads past the range re-read its last super-chunk
        uint2 nr[R];
        uint4 rr[R];
        const uint32_t last = ns ? ns - 1u : 0u;
        auto request = [&](uint32_t i) {
            const uint32_t c = min(i, last);
            nr[i % R] = ldnt2(np + (uint64_t)c * kLanes * 8);
            if constexpr (FP8) {
                if (i % 2u == 0u) {
                    const uint8_t *pp = rp + (uint64_t)(c / 2u) * 3 * kLanes * 4;
                    rr[i % R].x = ldnt1(pp);
                    rr[i % R].y = ldnt1(pp + kLanes * 4);
                    rr[i % R].z = ldnt1(pp + 2 * kLanes * 4);
                }
            } else {
                rr[i % R] = ldnt4(rp + (uint64_t)c * kLanes * 16);
            }
        };
#pragma unroll
        for (uint32_t i = 0; i < R; i++) request(i);
        Exceptions<ELEM, SP> X;
        X.init(a, L, cnt, base, p);
        X.request();
        float accA = 0.f, accB = 0.f;
#pragma unroll
        for (uint32_t i = 0; i < NS; i++) {
            if (i >= ns) continue;                               // a last column block's missing super-chunks
            uint32_t pa[4], qa[4];
            if constexpr (FP8) {
                const uint4 c = rr[(i % R) & ~1u];
                if (i % 2u) decode_sc<ELEM, 4>(tab, nr[i % R], c, c.x, c.y, c.z, pa, qa);
                else decode_sc<ELEM, 0>(tab, nr[i % R], c, c.x, c.y, c.z, pa, qa);
            } else {
                decode_sc<ELEM, 0>(tab, nr[i % R], rr[i % R], 0u, 0u, 0u, pa, qa);
            }
            if constexpr (FP8) {
                if (i % 2u && i + R - 1u < NS) {
                    request(i + R - 1u);
                    request(i + R);
                }
            } else {
                if (i + R < NS) request(i + R);
            }
            const uint4 xv = xs[(cb * kCols + (sc0 + i) * 32u + 8u * q) >> 3];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                accA = dot2_bf16(pa[k], u4_get(xv, k), accA);
                accB = dot2_bf16(qa[k], u4_get(xv, k), accB);
            }
            asm volatile("" : "+v"(accA), "+v"(accB));
        }
        // this half-wave's share of the lane's exceptions (planes decoded to +-0, the entries carry the value)
        while (__any(X.has(0u))) {
#pragma unroll
            for (uint32_t k = 0; k < X.N; k++) {
                if (!X.has(k)) continue;
                const uint32_t i = X.v[k] & 0xFFu, j = i & 15;
                const uint32_t col = cb * kCols + (i >> 4) * 32 + frag_col(L, j), upper = (j >> 1) & 1u;
                const float xv = __uint_as_float((uint32_t)((const uint16_t *)xs)[col] << 16), w = X.value(k);
                if (upper) accB = fmaf(w, xv, accB);
                else accA = fmaf(w, xv, accA);
            }
            X.next += X.N * SP;
            if (__any(X.has(0u))) X.request();
        }
        accA += xor_f<1>(accA); accA += xor_f<2>(accA);
        accB += xor_f<1>(accB); accB += xor_f<2>(accB);
        if (q == 0) {
            const uint32_t pi = ((g * kRows12 + r) * f.CB + cb) * SP + p;
            part[pi] = accA;
            part[pi + 8u * f.CB * SP] = accB;
        }
    }
    finish_rows<kToken>(a, part, rg0 * kRows12, ng * kRows12, f.CB * SP, FP8 ? &fin : nullptr);
}

// Row gather: one half-wave per requested row; the row's lanes store their columns, then patch their exceptions.
template <int ELEM>
__global__ void __launch_bounds__(256) k_gather2(GatherArgs a) {
    const RankTab tab{a.lut[0], a.lut[1], a.lut[2], a.lut[3]};
    constexpr uint32_t esz = ELEM == kElemFp8 ? 2u : 3u;
    const uint32_t L = threadIdx.x & 31, r = L >> 2, q = L & 3;
    const Shape f(a.M, a.K, 2);
    // four half-waves per (id, column block), each a quarter of its super-chunks (4p .. 4p + 3): the fixed-width planes
    // need no cursor, so every super-chunk's loads go out together and a lookup waits one round trip, not sixteen
    const uint32_t item = blockIdx.x * (blockDim.x >> 5) + (threadIdx.x >> 5), pair = item >> 2, p = item & 3u;
    const uint32_t id = pair / f.CB, cb = pair - id * f.CB;
    if (id >= a.n_ids) return;
    const int64_t R = a.ids[id];
    if (R < 0 || R >= (int64_t)a.M) return;
    const uint32_t nsc = ((cb == f.CB - 1 ? f.nl : 32u) + 1) / 2, sc0 = 4u * p;
    if (sc0 >= nsc) return;
    const uint32_t last = min(4u, nsc - sc0) - 1u;            // super-chunks past the block's last re-read it
    const uint8_t *rplane = a.low + f.nib2_bytes();
    const uint32_t rb = (uint32_t)R / kRows12, rr = (uint32_t)R % kRows12;
    const bool mine = (rr & 7u) == r, upper = rr >= 8;
    uint16_t *o = a.out + (uint64_t)id * f.K16;
    const uint32_t slot0 = rb * f.spr + cb * 16;
    const uint8_t *np = a.low + ((uint64_t)(slot0 + sc0) * kLanes + L) * 8;
    uint2 nib[4];
    uint4 raw[4];
    uint32_t c[2][3];
#pragma unroll
    for (uint32_t i = 0; i < 4; i++) nib[i] = *(const uint2 *)(np + (uint64_t)min(i, last) * kLanes * 8);
    if constexpr (ELEM == kElemFp8) {                          // 3-bit fields per pair of super-chunks (sc0 is even)
        const uint8_t *rp = rplane + (((uint64_t)rb * f.spr2 + cb * 8 + sc0 / 2u) * 3 * kLanes + L) * 4;
#pragma unroll
        for (uint32_t h = 0; h < 2; h++) {
            const uint8_t *pp = rp + (uint64_t)min(h, last / 2u) * 3 * kLanes * 4;
#pragma unroll
            for (uint32_t w = 0; w < 3; w++) c[h][w] = *(const uint32_t *)(pp + w * kLanes * 4);
        }
    } else {
        const uint8_t *rp = rplane + ((uint64_t)(slot0 + sc0) * kLanes + L) * 16;
#pragma unroll
        for (uint32_t i = 0; i < 4; i++) raw[i] = *(const uint4 *)(rp + (uint64_t)min(i, last) * kLanes * 16);
    }
#pragma unroll
    for (uint32_t i = 0; i < 4; i++) {
        if (i > last) break;
        uint32_t pv[4], qv[4];
        if constexpr (ELEM == kElemFp8) {
            if (i & 1u) decode_sc<ELEM, 4>(tab, nib[i], make_uint4(0, 0, 0, 0), c[i / 2][0], c[i / 2][1], c[i / 2][2], pv, qv);
            else decode_sc<ELEM, 0>(tab, nib[i], make_uint4(0, 0, 0, 0), c[i / 2][0], c[i / 2][1], c[i / 2][2], pv, qv);
        } else {
            decode_sc<ELEM, 0>(tab, nib[i], raw[i], 0u, 0u, 0u, pv, qv);
        }
        const uint32_t kc = cb * kCols + (sc0 + i) * 32 + 8 * q;
        if (mine && kc < f.K16) {
            const uint32_t *v = upper ? qv : pv;
            *(uint4 *)(o + kc) = make_uint4(v[0], v[1], v[2], v[3]);
        }
    }
    // exceptions of this lane in this quarter's super-chunks, after its plane values (the planes decode them to +-0);
    // the whole half computes the prefix over the lanes' counts, only the row's lanes use it
    const uint32_t b = rb * f.CB + cb;
    const uint32_t cnt = a.hdr[(uint64_t)b * kHdrBytes + L];
    const uint32_t incl = half_scan_incl(cnt, L);
    const uint8_t *ep = a.data + a.bases[b] + (uint64_t)(incl - cnt) * esz;
    if (mine) {
        for (uint32_t k = 0; k < cnt; k++, ep += esz) {
            const uint32_t i = ep[0], j = i & 15, sc = i >> 4;
            if (sc - sc0 > last || (((j >> 1) & 1u) != 0) != upper) continue;
            o[cb * kCols + sc * 32 + frag_col(L, j)] = (uint16_t)f32_to_bf16_rne(exc_value<ELEM>(ep));
        }
    }
}

template <int ELEM, int MODE, bool XBF16>
static int launch_fixed_t(const LaunchPlan &p, const BlockArgs &a, hipStream_t st) {
    if constexpr (MODE == kToken && XBF16) {
        if (p.split) {
            if (p.split == 4) hipLaunchKernelGGL((k_layout2s<ELEM, 4>), dim3(p.grid), dim3(p.threads), p.lds, st, a);
            else if (p.split == 2) hipLaunchKernelGGL((k_layout2s<ELEM, 8>), dim3(p.grid), dim3(p.threads), p.lds, st, a);
            else hipLaunchKernelGGL((k_layout2s<ELEM, 16>), dim3(p.grid), dim3(p.threads), p.lds, st, a);
            return (int)hipGetLastError();
        }
    }
    hipLaunchKernelGGL((k_layout2<ELEM, MODE, XBF16>), dim3(p.grid), dim3(p.threads), p.lds, st, a);
    return (int)hipGetLastError();
}

int launch_fixed(const LaunchPlan &p, int elem_t, int mode, bool xbf16, const BlockArgs &a, hipStream_t st) {
    if (elem_t == kElemFp8) {
        if (mode == kDequant) return launch_fixed_t<kElemFp8, kDequant, true>(p, a, st);
        if (mode == kF32) return launch_fixed_t<kElemFp8, kF32, false>(p, a, st);
        return xbf16 ? launch_fixed_t<kElemFp8, kToken, true>(p, a, st) : launch_fixed_t<kElemFp8, kToken, false>(p, a, st);
    }
    if (mode == kDequant) return launch_fixed_t<kElemBf16, kDequant, true>(p, a, st);
    if (mode == kF32) return launch_fixed_t<kElemBf16, kF32, false>(p, a, st);
    return xbf16 ? launch_fixed_t<kElemBf16, kToken, true>(p, a, st) : launch_fixed_t<kElemBf16, kToken, false>(p, a, st);
}

int launch_gather_fixed(int elem_t, const GatherArgs &a, hipStream_t st) {
    const uint32_t per = 8;                                        // half-wave items per workgroup
    const uint64_t items = (uint64_t)a.n_ids * Shape(a.M, a.K, 2).CB * 4u;
    const dim3 grid((uint32_t)((items + per - 1) / per));
    if (elem_t == kElemFp8) hipLaunchKernelGGL(k_gather2<kElemFp8>, grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL(k_gather2<kElemBf16>, grid, dim3(256), 0, st, a);
    return (int)hipGetLastError();
}

}  // namespace nwc
