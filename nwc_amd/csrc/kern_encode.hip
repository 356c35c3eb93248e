// kern_encode.hip -- the encoder on the GPU: the stored tensors of a matrix that is (or is about to be) in GPU memory, byte
// for byte those of the host encoder (encode.cpp).  Three passes with the caller's small host steps between them: a
// histogram of the symbols (the host ranks them), the size of every lane stream or exception list, and the write of
// streams and planes to their places.  A half-wave takes one block, its lanes the block's lanes, so the loads are whole
// row pieces; each lane packs its own stream.
// 2560 x 9728 BF16, layout 0: host encoder on 16 threads 20.4 ms; the three passes here read 100 MB and write 34 MB.
#include "nwc_fixed.h"
#include "nwc_launch.h"
#include "nwc_private.h"

namespace nwc {

// Eight weights of a row from a column on, as their codes need them: `hi` = sign << 7 | symbol, `lo` = raw byte (BF16),
// nibble (fp8, layouts 0/1) or 3-bit field (fp8, layout 2), `src` = the source bits.  n: how many lie in the matrix.
struct Eight {
    uint32_t hi[8], lo[8], src[8], n;
};

// Symbol and raw bits of an fp8 e4m3 byte: the decoder rebuilds an fp32 value from the exponent's upper seven bits (the
// coded symbol) and the raw bits (the exponent's low bit and three mantissa bits; layout 2: the mantissa bits).
__device__ __forceinline__ void split_fp8(uint32_t b, bool l2, uint32_t &sym, uint32_t &raw) {
    const uint32_t u = __float_as_uint(e4m3_to_f32(b & 0x7Fu)), ex = u >> 23, top3 = (u >> 20) & 7u, b3 = ex >> 1;
    if (l2) {
        const uint32_t e = (b >> 3) & 15u, m = b & 7u;
        sym = e ? e : m >= 4u ? 16u : m >= 2u ? 17u : m == 1u ? 18u : 19u;
        raw = top3;
    } else {
        sym = b3 >= 60u ? b3 - 60u : b3 == 59u ? 8u : 9u;        // table bytes 60..67, 59, zero
        raw = (ex & 1u) << 3 | top3;
    }
}

template <int ELEM, bool L2>
__device__ __forceinline__ void load8(Eight &o, const void *w, uint32_t M, uint32_t K, uint32_t row, uint32_t col) {
    typedef __attribute__((aligned(1))) uint64_t any64;
    o.n = row < M && col < K ? min(K - col, 8u) : 0u;
    const uint64_t at = (uint64_t)row * K + col;
#pragma unroll
    for (int i = 0; i < 8; i++) o.src[i] = 0u;
    if constexpr (ELEM == kElemFp8) {
        const uint8_t *p = (const uint8_t *)w + at;
        if (o.n == 8u) {
            const uint64_t v = *(const any64 *)p;
#pragma unroll
            for (int i = 0; i < 8; i++) o.src[i] = (uint32_t)(v >> (8 * i)) & 0xFFu;
        } else {
#pragma unroll
            for (int i = 0; i < 8; i++)
                if ((uint32_t)i < o.n) o.src[i] = p[i];
        }
#pragma unroll
        for (int i = 0; i < 8; i++) {
            uint32_t sym, raw;
            split_fp8(o.src[i], L2, sym, raw);
            o.hi[i] = (o.src[i] & 0x80u) | sym;
            o.lo[i] = raw;
        }
    } else {
        const uint16_t *p = (const uint16_t *)w + at;
        if (o.n == 8u) {
            const uint4 v = ld_any4(p);
#pragma unroll
            for (int i = 0; i < 8; i++) o.src[i] = (u4_get(v, i / 2) >> (16 * (i & 1))) & 0xFFFFu;
        } else {
#pragma unroll
            for (int i = 0; i < 8; i++)
                if ((uint32_t)i < o.n) o.src[i] = p[i];
        }
#pragma unroll
        for (int i = 0; i < 8; i++) {
            o.hi[i] = o.src[i] >> 8;
            o.lo[i] = o.src[i] & 0xFFu;
        }
    }
}

// ---- pass 1: symbol counts (count[128]: NaN among fp8 input) ----
// 32 copies of the bins, one per bank: neighbouring weights share a few exponents, so a single copy would serialise.
template <int ELEM, bool L2>
__global__ void __launch_bounds__(256) k_enc_hist(const void *w, uint64_t n, unsigned long long *count) {
    __shared__ uint32_t bins[128 * 32], nan;
    for (uint32_t i = threadIdx.x; i < 128u * 32u; i += 256u) bins[i] = 0u;
    if (threadIdx.x == 0) nan = 0u;
    __syncthreads();
    const uint32_t copy = threadIdx.x & 31u;
    bool bad = false;
    const uint64_t n8 = (n + 7u) / 8u;
    for (uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x; i < n8; i += (uint64_t)gridDim.x * 256u) {
        Eight e;                                               // the matrix as one row of up to 2^32 - 1 columns at a time
        const uint64_t left = n - 8u * i;
        const uint8_t *p = (const uint8_t *)w + 8u * i * (ELEM == kElemFp8 ? 1u : 2u);
        load8<ELEM, L2>(e, p, 1u, left < 8u ? (uint32_t)left : 8u, 0u, 0u);
#pragma unroll
        for (uint32_t k = 0; k < 8; k++) {
            if (k >= e.n) break;
            if (ELEM == kElemFp8 && (e.src[k] & 0x7Fu) == 0x7Fu) bad = true;
            else atomicAdd(&bins[(e.hi[k] & 0x7Fu) * 32u + copy], 1u);
        }
    }
    if (bad) nan = 1u;
    __syncthreads();
    if (threadIdx.x < 128u) {
        uint32_t sum = 0;
        for (uint32_t c = 0; c < 32u; c++) sum += bins[threadIdx.x * 32u + (c + threadIdx.x) % 32u];
        if (sum) atomicAdd(&count[threadIdx.x], (unsigned long long)sum);
    } else if (threadIdx.x == 128u && nan) {
        atomicAdd(&count[128], 1ull);
    }
}

// ---- passes 2 and 3 ----
struct EncArgs {
    const void *w;
    const uint8_t *rank;         // of each symbol (layout 2: 7 = exception)
    uint8_t *hdr, *data, *low;
    uint32_t *size;              // pass 2: bytes of each block's streams or exceptions
    uint32_t *over;              // pass 2: set where a lane has more than its header byte can say
    const uint32_t *bases;       // pass 3
    uint32_t M, K;
};

// MSB-first code words of one lane; without a destination it only counts.
struct WordSink {
    uint32_t *dst;
    uint64_t acc;
    uint32_t n, words;
    __device__ __forceinline__ void put(uint32_t v, uint32_t len) {
        acc = acc << len | v;
        n += len;
        if (n >= 32u) {
            n -= 32u;
            dst[words++] = (uint32_t)(acc >> n);
        }
    }
    __device__ __forceinline__ void close() {
        if (n) dst[words++] = (uint32_t)(acc << (32u - n));
    }
};

// the code of one weight: value and length (filler outside the matrix: rank 0, sign 0)
template <int ELEM>
__device__ __forceinline__ void code_of(uint32_t hi, bool in, const uint8_t *rank, uint32_t &v, uint32_t &len) {
    constexpr uint32_t maxr = ELEM == kElemFp8 ? kMaxRankFp8 : kMaxRankBf16;
    const uint32_t r = in ? rank[hi & 0x7Fu] : 0u;
    const bool esc = r >= maxr;
    v = esc ? 0x100u | hi : 2u | (in ? hi >> 7 : 0u);
    len = esc ? 24u : r + 2u;
}

// 16 raw values of a lane in stream order as stored: BF16 bytes, fp8 nibbles (value j in byte (j & 3) + 4 (j >> 3), high half
// for j & 4)
template <int ELEM>
__device__ __forceinline__ void store_raw16(uint8_t *p, const uint32_t (&v)[16]) {
    if constexpr (ELEM == kElemFp8) {
        uint32_t o[2];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            o[h] = 0u;
#pragma unroll
            for (int j = 0; j < 8; j++) o[h] |= v[8 * h + j] << (8 * (j & 3) + 4 * (j >> 2));
        }
        *(uint2 *)p = make_uint2(o[0], o[1]);
    } else {
        uint32_t o[4];
#pragma unroll
        for (int k = 0; k < 4; k++) o[k] = v[4 * k] | v[4 * k + 1] << 8 | v[4 * k + 2] << 16 | v[4 * k + 3] << 24;
        *(uint4 *)p = make_uint4(o[0], o[1], o[2], o[3]);
    }
}

// Layouts 0 and 1, sizes (WRITE false) or streams and raw plane.
template <int ELEM, int LAYOUT, bool WRITE>
__global__ void __launch_bounds__(256) k_enc_prefix(EncArgs a) {
    constexpr uint32_t RB = ELEM == kElemFp8 ? 8u : 16u;          // raw bytes of 16 weights
    __shared__ uint8_t rank[128];
    if (threadIdx.x < 128u) rank[threadIdx.x] = a.rank[threadIdx.x];
    __syncthreads();
    const Shape f(a.M, a.K, LAYOUT);
    const uint32_t b = blockIdx.x * 8u + (threadIdx.x >> 5), L = threadIdx.x & 31u;
    if (b >= f.nb) return;
    const uint32_t rb = b / f.CB, cb = b - rb * f.CB;
    WordSink s{nullptr, 0u, 0u, 0u};
    if (WRITE) {
        const uint32_t n = a.hdr[(uint64_t)b * kHdrBytes + L];
        s.dst = (uint32_t *)(a.data + a.bases[b]) + (half_scan_incl(n, L) - n);
    }
    uint32_t bits = 0;
    auto code = [&](const Eight &e, int i) {
        uint32_t v, len;
        code_of<ELEM>(e.hi[i], (uint32_t)i < e.n, rank, v, len);
        if (WRITE) s.put(v, len);
        else bits += len;
    };
    const uint32_t r = L >> 2, q = L & 3u;
    const uint32_t steps = LAYOUT == 0 ? kRows0 : cb == f.CB - 1u ? f.nsl : 16u;
    for (uint32_t i = 0; i < steps; i++) {                         // a row's 16 columns, or a super-chunk's two rows of eight
        Eight x, y;
        const uint32_t row = LAYOUT == 0 ? rb * kRows0 + i : rb * kRows12 + r;
        const uint32_t col = LAYOUT == 0 ? cb * kCols + 16u * L : cb * kCols + 32u * i + 8u * q;
        load8<ELEM, false>(x, a.w, a.M, a.K, row, col);
        if (LAYOUT == 0) load8<ELEM, false>(y, a.w, a.M, a.K, row, col + 8u);
        else load8<ELEM, false>(y, a.w, a.M, a.K, row + 8u, col);
        uint32_t raw[16];
#pragma unroll
        for (int j = 0; j < 16; j++) {                             // stream order
            const bool second = LAYOUT == 0 ? j >= 8 : (j >> 1) & 1;
            const int at = LAYOUT == 0 ? j & 7 : 2 * (j >> 2) + (j & 1);
            const Eight &e = second ? y : x;
            code(e, at);
            raw[j] = (uint32_t)at < e.n ? e.lo[at] : 0u;
        }
        if (WRITE) {
            if (LAYOUT == 0) {
                if (row < a.M && col < f.K16) store_raw16<ELEM>(a.low + ((uint64_t)row * f.K16 + col) / 16u * RB, raw);
            } else {
                store_raw16<ELEM>(a.low + ((uint64_t)(rb * f.spr + cb * 16u + i) * kLanes + L) * RB, raw);
            }
        }
    }
    if (WRITE) {
        s.close();
        return;
    }
    const uint32_t words = (bits + 31u) / 32u;
    if (words > 255u) *a.over = 1u;
    a.hdr[(uint64_t)b * kHdrBytes + L] = (uint8_t)words;
    const uint32_t total = half_scan_incl(words, L);
    if (L == 31u) a.size[b] = 4u * total;
}

// Layout 2: exception counts, or the nibble and raw planes and the exception entries (position, value), whose planes are zero.
template <int ELEM, bool WRITE>
__global__ void __launch_bounds__(256) k_enc_fixed(EncArgs a) {
    constexpr uint32_t SIZE = ELEM == kElemFp8 ? 2u : 3u;
    __shared__ uint8_t rank[128];
    if (threadIdx.x < 128u) rank[threadIdx.x] = a.rank[threadIdx.x];
    __syncthreads();
    const Shape f(a.M, a.K, 2);
    const uint32_t b = blockIdx.x * 8u + (threadIdx.x >> 5), L = threadIdx.x & 31u;
    if (b >= f.nb) return;
    const uint32_t rb = b / f.CB, cb = b - rb * f.CB, r = L >> 2, q = L & 3u;
    const uint32_t nsc = cb == f.CB - 1u ? f.nsl : 16u;
    uint32_t cnt = 0;
    uint8_t *ep = nullptr, *rplane = a.low + f.nib2_bytes();
    if (WRITE) {
        const uint32_t n = a.hdr[(uint64_t)b * kHdrBytes + L];
        ep = a.data + a.bases[b] + (half_scan_incl(n, L) - n) * SIZE;
    }
    uint64_t first = 0;                                            // fp8: the 48 raw bits of a pair's first super-chunk
    for (uint32_t sc = 0; sc < nsc; sc++) {
        Eight x, y;
        const uint32_t row = rb * kRows12 + r, col = cb * kCols + 32u * sc + 8u * q;
        load8<ELEM, true>(x, a.w, a.M, a.K, row, col);
        load8<ELEM, true>(y, a.w, a.M, a.K, row + 8u, col);
        uint32_t raw[16], nib[2] = {0u, 0u};
#pragma unroll
        for (int j = 0; j < 16; j++) {
            const Eight &e = (j >> 1) & 1 ? y : x;
            const int at = 2 * (j >> 2) + (j & 1);
            const bool in = (uint32_t)at < e.n;
            const uint32_t rk = in ? rank[e.hi[at] & 0x7Fu] : 0u;
            const bool exc = rk == 7u;
            if (WRITE) {
                if (exc) {
                    ep[0] = (uint8_t)(16u * sc + j);
                    ep[1] = (uint8_t)e.src[at];
                    if (ELEM != kElemFp8) ep[2] = (uint8_t)(e.src[at] >> 8);
                    ep += SIZE;
                }
                raw[j] = in && !exc ? e.lo[at] : 0u;
                nib[j >> 3] |= (in ? (e.hi[at] >> 7) << 3 | rk : 0u) << (4 * (j & 7));
            }
            cnt += exc ? 1u : 0u;
        }
        if (!WRITE) continue;
        const uint64_t slot = (uint64_t)(rb * f.spr + cb * 16u + sc) * kLanes + L;
        *(uint2 *)(a.low + slot * 8u) = make_uint2(nib[0], nib[1]);
        if constexpr (ELEM == kElemFp8) {
            uint64_t bits = 0;
#pragma unroll
            for (int j = 0; j < 16; j++) bits |= (uint64_t)raw[j] << (3 * j);
            if ((sc & 1u) == 0u) first = bits;
            if ((sc & 1u) != 0u || sc + 1u == nsc) {
                const uint64_t second = sc & 1u ? bits : 0u;
                uint32_t *p = (uint32_t *)(rplane + (((uint64_t)rb * f.spr2 + cb * 8u + (sc >> 1)) * 3u * kLanes + L) * 4u);
                p[0] = (uint32_t)first;
                p[kLanes] = (uint32_t)(first >> 32) | (uint32_t)(second << 16);
                p[2u * kLanes] = (uint32_t)(second >> 16);
            }
        } else {
            store_raw16<kElemBf16>(rplane + slot * 16u, raw);
        }
    }
    if (WRITE) return;
    if (cnt > 255u) *a.over = 1u;
    a.hdr[(uint64_t)b * kHdrBytes + L] = (uint8_t)cnt;
    const uint32_t total = half_scan_incl(cnt, L);
    if (L == 31u) a.size[b] = SIZE * total;
}

// dst[to[b] + j] = src[from[b] + j], j < size[b]: 4-byte words, one wave per block.
__global__ void __launch_bounds__(256) k_copy_spans(const uint8_t *src, const int64_t *from, uint8_t *dst, const int64_t *to,
                                                    const int64_t *size, uint32_t nb) {
    const uint32_t b = blockIdx.x * 4u + (threadIdx.x >> 6);
    if (b >= nb) return;
    const uint32_t *s = (const uint32_t *)(src + from[b]);
    uint32_t *d = (uint32_t *)(dst + to[b]);
    const uint32_t n = (uint32_t)(size[b] / 4);
    for (uint32_t i = threadIdx.x & 63u; i < n; i += 64u) d[i] = s[i];
}

template <int ELEM, bool WRITE>
static int launch_enc(int layout, const EncArgs &a, hipStream_t st) {
    const dim3 g((Shape(a.M, a.K, layout).nb + 7u) / 8u), t(256);
    if (layout == 0) hipLaunchKernelGGL((k_enc_prefix<ELEM, 0, WRITE>), g, t, 0, st, a);
    else if (layout == 1) hipLaunchKernelGGL((k_enc_prefix<ELEM, 1, WRITE>), g, t, 0, st, a);
    else hipLaunchKernelGGL((k_enc_fixed<ELEM, WRITE>), g, t, 0, st, a);
    return (int)hipGetLastError();
}

// The shapes whose planes 32-bit arithmetic and the kernels can address (as abi.cpp's device entry points).
static bool enc_ok(uint64_t M, uint32_t K, int elem) {
    if (M == 0 || K == 0 || M > 0xFFFFFFFFull || elem_type(elem) > 1 || elem_layout(elem) > 2 || (elem & ~0xFF) != 0) return false;
    const uint64_t K16 = ((uint64_t)K + 15u) & ~15ull, rows = elem_layout(elem) ? kRows12 : kRows0;
    return (M + rows) * (K16 + kCols) < (1ull << 32);
}

}  // namespace nwc

using namespace nwc;

extern "C" int nwc_encode_supported(uint64_t M, uint32_t K, int elem) { return enc_ok(M, K, elem) ? 1 : 0; }

extern "C" int nwc_encode_hist(void *stream, const void *w, uint64_t n, int elem, uint64_t *count) {
    if (n == 0 || elem_type(elem) > 1 || elem_layout(elem) > 2) return -1;
    const dim3 g((uint32_t)std::min<uint64_t>((n / 8u + 255u) / 256u + 1u, 1024u)), t(256);
    hipStream_t st = (hipStream_t)stream;
    unsigned long long *c = (unsigned long long *)count;
    if (elem_type(elem) != kElemFp8) hipLaunchKernelGGL((k_enc_hist<kElemBf16, false>), g, t, 0, st, w, n, c);
    else if (elem_layout(elem) == 2) hipLaunchKernelGGL((k_enc_hist<kElemFp8, true>), g, t, 0, st, w, n, c);
    else hipLaunchKernelGGL((k_enc_hist<kElemFp8, false>), g, t, 0, st, w, n, c);
    return (int)hipGetLastError();
}

extern "C" int nwc_encode_sizes(void *stream, const void *w, uint64_t M, uint32_t K, int elem, const uint8_t *rank,
                                uint8_t *hdr, uint32_t *size, uint32_t *over) {
    if (!enc_ok(M, K, elem)) return -1;
    const EncArgs a{w, rank, hdr, nullptr, nullptr, size, over, nullptr, (uint32_t)M, K};
    return elem_type(elem) == kElemFp8 ? launch_enc<kElemFp8, false>(elem_layout(elem), a, (hipStream_t)stream)
                                       : launch_enc<kElemBf16, false>(elem_layout(elem), a, (hipStream_t)stream);
}

extern "C" int nwc_encode_write(void *stream, const void *w, uint64_t M, uint32_t K, int elem, const uint8_t *rank,
                                const uint8_t *hdr, const uint32_t *bases, uint8_t *data, uint8_t *low) {
    if (!enc_ok(M, K, elem)) return -1;
    const EncArgs a{w, rank, (uint8_t *)hdr, data, low, nullptr, nullptr, bases, (uint32_t)M, K};
    return elem_type(elem) == kElemFp8 ? launch_enc<kElemFp8, true>(elem_layout(elem), a, (hipStream_t)stream)
                                       : launch_enc<kElemBf16, true>(elem_layout(elem), a, (hipStream_t)stream);
}

extern "C" int nwc_copy_spans(void *stream, const uint8_t *src, const int64_t *from, uint8_t *dst, const int64_t *to,
                              const int64_t *size, uint32_t nb) {
    if (nb == 0) return 0;
    hipLaunchKernelGGL(k_copy_spans, dim3((nb + 3u) / 4u), dim3(256), 0, (hipStream_t)stream, src, from, dst, to, size, nb);
    return (int)hipGetLastError();
}
