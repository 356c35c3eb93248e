// kern_tokens.hip -- a compressed matrix times a small batch of BF16 activation vectors (2 to 64) on the matrix cores,
// without a BF16 copy of the matrix: y[t] = W x[t] (fp8: times the row scale) + bias, all layouts, fp32 accumulation,
// one rounding to BF16.
//
// A workgroup keeps the decode table and activations in LDS for its whole life, and its waves work through blocks, one
// task (row group, column block) at a time: a wave decodes a block on its two halves (layout 0: rows 0-3 and 4-7; layouts
// 1/2: super-chunks 0-7 and 8-15; from the row index) and multiplies it by v_mfma_f32_16x16x32_bf16 (A: 16 rows x 32
// columns, lane l row l & 15, columns 8 (l >> 4) .. + 7; B: the same columns of 16 tokens).  Decoded weights reach the
// operand's lanes through LDS that belongs to the wave alone (layout 0: the block's exponent bytes; layout 2: one
// super-chunk a half) or through lane permutes (layout 1); a wave requests its next task's streams and raw bytes while it
// decodes, so after the first barrier no wave waits for another.
// Two ways of sharing the matrix out (abi.cpp plan_tokens): a workgroup has one column block of a run of row groups and
// its sums go to a workspace [column block][token][row], which k_tokens_finish adds in order; or, where the activations
// fit, all column blocks of its rows, whose sums it adds in LDS in order.  Either way equal inputs give equal bits.
//
// What bounds it: the LDS pipe (the decode's table reads, about 24k of 60k cycles a CU on 19456 x 2560) and the latency
// of its chain, so the split aims at waves: a task of one block a wave keeps the LDS share of a wave at 6 KB (layout 0),
// which lets 16 waves share a CU (8-9 with two row groups a wave: 19456 x 2560 at 16 tokens 34.6 us, now 28.6; two
// interleaved cursors a lane instead 34.0; activations from L2 instead of LDS 38.4, at 64 tokens 82 instead of 43).
// Against the temporary BF16 matrix and hipBLASLt, graph-timed with matrices out of the caches, 32 tokens (4 tokens),
// layout 0: 6144 x 2560 18.1 (14.2) against 34 us, 2560 x 4096 15.4 (13.6) against 31, 19456 x 2560 31.8 (24.6) against 87,
// 2560 x 9728 23.0 (20.3) against 43; layout 1 17.9 / 18.2 / 31.6 / 23.7 against 36 / 32 / 100 / 48; layout 2 15.6 / 14.3 /
// 29.3 / 21.6 against 40 / 37 / 104 / 48.  The second kernel is 3.3 us of a split product.
#include "nwc_fixed.h"
#include "nwc_launch.h"
#include "nwc_prefix.h"

namespace nwc {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;

__device__ __forceinline__ bf16x8_t operand(uint32_t w0, uint32_t w1, uint32_t w2, uint32_t w3) {
    return __builtin_bit_cast(bf16x8_t, make_uint4(w0, w1, w2, w3));
}
__device__ __forceinline__ bf16x8_t operand(const uint4 &v) { return __builtin_bit_cast(bf16x8_t, v); }
__device__ __forceinline__ f32x4_t mfma(bf16x8_t w, bf16x8_t x, f32x4_t acc) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, x, acc, 0, 0, 0);
}

// lanes 32-63 of x against lanes 0-31 of y
__device__ __forceinline__ void swap32(uint32_t &x, uint32_t &y) {
    const u32x2_t v = __builtin_amdgcn_permlane32_swap(x, y, false, false);
    x = v.x;
    y = v.y;
}

// Orders a wave's LDS writes before its later LDS reads of other lanes' words (LDS serves one wave's requests in order;
// only the compiler has to keep them so).
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The activations in LDS: token t's columns (512 of one column block, or all of them) from xs + t * p.xrow, zero past K.
// Rows 4 banks apart, so that an operand read (16 tokens) meets no bank twice.  The first N chunks of 8 columns per thread
// are requested early (issue); commit stores them and copies the rest.  Rows that begin anywhere and end inside a chunk are
// read as they are (x8_tail's way), which costs less than the two launches of a padded copy.
struct StageX {
    static constexpr uint32_t N = 4;
    u32x4_t v[N];
    uint32_t per, total, col0;                                   // chunks a row and in all, first column
    __device__ __forceinline__ void load(const TokensArgs &p, uint32_t i0) {
        const uint32_t K = p.a.K;
#pragma unroll
        for (uint32_t k = 0; k < N; k++) {
            const uint32_t i = min(i0 + k * blockDim.x, total - 1u), t = i / per, col = col0 + 8u * (i - t * per);
            v[k] = *(const u32x4_any *)(p.x + (uint64_t)t * p.ldx + min(col, K - 8u));
        }
    }
    __device__ __forceinline__ void store(uint32_t *xs, const TokensArgs &p, uint32_t i0) const {
#pragma unroll
        for (uint32_t k = 0; k < N; k++) {
            const uint32_t i = i0 + k * blockDim.x, t = i / per, K = p.a.K, col = col0 + 8u * (i - t * per);
            if (i >= total) continue;
            uint32_t w[4] = {v[k].x, v[k].y, v[k].z, v[k].w};
            if (K & 7u) shift_down<4>(w, col - min(col, K - 8u));
            const uint32_t keep = col < K ? ~0u : 0u;
            *(uint4 *)(xs + t * p.xrow + 4u * (i - t * per)) = make_uint4(w[0] & keep, w[1] & keep, w[2] & keep, w[3] & keep);
        }
    }
    __device__ __forceinline__ void issue(const TokensArgs &p, uint32_t cb, uint32_t blocks) {
        per = 64u * blocks;
        total = p.T * per;
        col0 = cb * kCols;
        load(p, threadIdx.x);
    }
    __device__ __forceinline__ void commit(uint32_t *xs, const TokensArgs &p) {
        store(xs, p, threadIdx.x);
        for (uint32_t i0 = threadIdx.x + N * blockDim.x; i0 < total; i0 += N * blockDim.x) {
            load(p, i0);
            store(xs, p, i0);
        }
    }
};

// A wave's tasks: t = wave, wave + waves, ... < n of its workgroup's.  A workgroup has a run of row groups ("units"), and
// either one column block of them (blockIdx = part * CB + cb), its sums going to the workspace, or, `direct`, all of their
// column blocks, whose sums it adds in LDS and finishes itself.
struct TokensTasks {
    uint32_t CB, u0, cb0, n, step, t;
    bool direct;
    __device__ __forceinline__ void init(const TokensArgs &p, const Shape &f) {
        CB = f.CB;
        direct = p.direct;
        const uint32_t part = direct ? blockIdx.x : blockIdx.x / CB, units = f.groups();
        cb0 = direct ? 0u : blockIdx.x - part * CB;
        u0 = (uint32_t)((uint64_t)part * units / p.parts);
        n = ((uint32_t)((uint64_t)(part + 1u) * units / p.parts) - u0) * (direct ? CB : 1u);
        step = blockDim.x >> 6;
        t = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    }
    // task i's unit and column block (past the last: the last again)
    __device__ __forceinline__ void at(uint32_t i, uint32_t &unit, uint32_t &cb) const {
        i = min(i, n - 1u);
        const uint32_t q = direct ? i / CB : i;
        unit = u0 + q;
        cb = direct ? i - q * CB : cb0;
    }
};

// A task's sums: lane l holds rows 4 (l >> 4) .. + 3 of the R rows of its unit for tokens 16 j + (l & 15).
template <int NT, int R>
__device__ __forceinline__ void store_part(const TokensArgs &p, const TokensTasks &w, uint32_t unit, float *sums,
                                           const f32x4_t (&acc)[NT]) {
    const uint32_t lane = threadIdx.x & 63u, m = 4u * (lane >> 4);
    if (m >= (uint32_t)R) return;
#pragma unroll
    for (int j = 0; j < NT; j++) {
        const uint32_t t = 16u * j + (lane & 15u);
        if (t >= p.T) break;
        if (w.direct) *(f32x4_t *)(sums + (w.t * p.T + t) * R + m) = acc[j];
        else *(f32x4_t *)(p.part + ((uint64_t)w.cb0 * p.T + t) * p.Mu + unit * R + m) = acc[j];
    }
}

// Rows m .. m + 3 of token t: scale, bias, one rounding.
__device__ __forceinline__ void finish4(const BlockArgs &a, uint32_t t, uint32_t m, const f32x4_t &v) {
    uint32_t h[4];
#pragma unroll
    for (uint32_t e = 0; e < 4; e++) {
        const uint32_t row = min(m + e, a.M - 1u);
        float u = v[e];
        if (a.scale) u *= a.scale[row];
        if (a.bias) u += bf16_lo(a.bias[row]);
        h[e] = f32_to_bf16_rne(u);
    }
    uint16_t *o = (uint16_t *)a.out + (uint64_t)t * a.M + m;
    if ((a.M & 3u) == 0u) {
        *(uint2 *)o = make_uint2(h[0] | h[1] << 16, h[2] | h[3] << 16);
    } else {
#pragma unroll
        for (uint32_t e = 0; e < 4; e++)
            if (m + e < a.M) o[e] = (uint16_t)h[e];
    }
}

// The direct workgroup's rows from its tasks' sums in LDS, column blocks in order.
template <int R>
__device__ __forceinline__ void finish_direct(const TokensArgs &p, const TokensTasks &w, const float *sums) {
    __syncthreads();
    const uint32_t units = w.n / w.CB, q = R / 4u;
    for (uint32_t i = threadIdx.x; i < units * p.T * q; i += blockDim.x) {
        const uint32_t ut = i / q, u = ut / p.T, t = ut - u * p.T, m = 4u * (i - ut * q);
        if ((w.u0 + u) * R + m >= p.a.M) continue;
        const float *src = sums + (u * w.CB * p.T + t) * R + m;
        f32x4_t v = *(const f32x4_t *)src;
        for (uint32_t c = 1; c < w.CB; c++) v += *(const f32x4_t *)(src + c * p.T * R);
        finish4(p.a, t, (w.u0 + u) * R + m, v);
    }
}

// y from the column blocks' sums, in order.
__global__ void __launch_bounds__(256) k_tokens_finish(TokensArgs p, uint32_t CB) {
    const uint32_t q = p.Mu / 4u, i = blockIdx.x * 256u + threadIdx.x;
    if (i >= p.T * q) return;
    const uint32_t t = i / q, m = 4u * (i - t * q);
    if (m >= p.a.M) return;
    const float *src = p.part + (uint64_t)t * p.Mu + m;
    const uint64_t step = (uint64_t)p.T * p.Mu;
    f32x4_t v = *(const f32x4_t *)src;
#pragma unroll 4
    for (uint32_t s = 1; s < CB; s++) v += *(const f32x4_t *)(src + s * step);
    finish4(p.a, t, m, v);
}

// ---------------------------------------------------------------------------------------------------------------
// Streams of one block on their way into a wave's slot, N 16-byte chunks a lane: requested a task ahead, stored once the
// slot is free.  `start`: the lane's first word in the slot; `fits`: else the block is decoded from memory (packed
// streams longer than the slot).
template <uint32_t N>
struct BlockStream {
    u32x4_t v[N];
    uint32_t n16, start, base;
    bool fits;
    // n: the lane's header byte; cap: the slot's words
    __device__ __forceinline__ void request(const BlockArgs &a, uint32_t b, uint32_t n, uint32_t cap) {
        const uint32_t lane = threadIdx.x & 63u, incl = half_scan_incl(n, lane & 31u);
        base = block_base(a, b);
        const uint32_t sh = (base & 15u) >> 2, total = __builtin_amdgcn_readlane(incl, 31);
        start = sh + incl - n;
        // with the 12 bytes the cursor reads past the last lane's stream (inside the slack after the last block)
        n16 = a.stride ? a.stride / 16u + 1u : (sh + total + 3u + 3u) / 4u;
        fits = n16 * 4u <= cap && n16 <= 64u * N;
        const uint8_t *src = a.data + (base & ~15u);
#pragma unroll
        for (uint32_t i = 0; i < N; i++)
            if (lane + 64u * i < n16) v[i] = *(const u32x4_t *)(src + 16u * (lane + 64u * i));
    }
    __device__ __forceinline__ void store(uint32_t *slot) const {
        if (!fits) return;
        const uint32_t lane = threadIdx.x & 63u;
#pragma unroll
        for (uint32_t i = 0; i < N; i++)
            if (lane + 64u * i < n16) *(u32x4_t *)(slot + 4u * (lane + 64u * i)) = v[i];
    }
};

// ---------------------------------------------------------------------------------------------------------------
// Layout 0: a wave decodes one block of eight rows, rows 0-3 and 4-7 (from the row index) a half; lane L the columns
// 16 L .. + 15.  The block's exponent bytes (8 rows x 512 columns) go to the wave's LDS tile and are read back by row,
// next to the raw bytes, which come from memory in the operand's arrangement.  Eight rows fill half of an operand; the
// other half takes the same rows 128 columns on (lane l: row l & 7, columns + 128 for l & 8), and each operand meets
// both columns' activations: the first product's rows 0-7 and the second's rows 8-15 are the block's.
template <int ELEM, class Tab>
__device__ __forceinline__ void tokens_decode0(const Tab &s, const uint32_t *lane_words, uint32_t P, uint32_t keep, uint32_t *tile) {
    Seq<ELEM> S;
    S.init_at(lane_words, P);
#pragma unroll
    for (uint32_t r = 0; r < 4; r++) {
        uint32_t e1[4], e2[4], b[4];
        row_codes(S, s, e1, e2);
#pragma unroll
        for (int k = 0; k < 4; k++) b[k] = perm(e2[k], e1[k], 0x06050201u) & keep;
        *(uint4 *)(tile + r * kTokensTileRow) = make_uint4(b[0], b[1], b[2], b[3]);
    }
}

template <int ELEM, int NT, int PEEK>
__global__ void __launch_bounds__(kTokensMaxWaves * 64) k_tokens0(TokensArgs p) {
    const BlockArgs &a = p.a;
    __shared__ LutT<PEEK> s;
    extern __shared__ __attribute__((aligned(16))) uint32_t dyn[];
    const uint32_t lane = threadIdx.x & 63u, L = threadIdx.x & 31u, h = lane >> 5;
    const uint32_t r8 = lane & 7u, far = (lane >> 3) & 1u, i16 = lane & 15u, c4 = lane >> 4;
    const Shape f(a.M, a.K, 0);
    TokensTasks w;
    w.init(p, f);
    const uint32_t tcol = 128u * far + 16u * c4;                  // operand columns of step j: + 64 (j & 1) + 256 (j >> 1)
    auto step_col = [](uint32_t j) { return 64u * (j & 1u) + 256u * (j >> 1); };
    auto cols_of = [&](uint32_t cb) { return min(kCols, f.K16 - cb * kCols); };      // coded columns of a block
    // lanes past the coded columns have no stream: they decode the block's first lane's rows, for nothing
    auto part_at = [&](uint32_t unit, uint32_t cb) {
        const uint32_t P = part_start(a, unit * f.CB + cb, 2u * h, L);
        return 16u * L < cols_of(cb) ? P : 0u;
    };
    auto raw_at = [&](uint32_t unit, uint32_t cb, uint32_t j) {
        const uint32_t row = min(unit * 8u + r8, a.M - 1u), col = min(cb * kCols + tcol + step_col(j), f.K16 - 16u);
        if constexpr (ELEM == kElemFp8) {
            const uint2 v = ldnt2(a.low + (row * (f.K16 / 2u) + col / 2u));
            return make_uint4(v.x, v.y, 0u, 0u);
        } else {
            return ldnt4(a.low + (row * f.K16 + col));
        }
    };
    uint32_t *xs = dyn, *tile = dyn + p.xwords + w.t * (kTokensTileWords + p.cap), *slot = tile + kTokensTileWords;
    float *sums = (float *)(dyn + p.xwords + w.step * (kTokensTileWords + p.cap));
    TabStage<PEEK> Q;
    Q.issue(a);
    uint32_t unit, cb, un, cn;
    w.at(w.t, unit, cb);
    w.at(w.t + w.step, un, cn);
    const uint32_t n = a.hdr[(uint64_t)(unit * f.CB + cb) * kHdrBytes + L];
    StageX X;
    X.issue(p, w.cb0, w.direct ? f.CB : 1u);
    BlockStream<2> B;
    B.request(a, unit * f.CB + cb, n, p.cap);
    uint32_t nn = a.hdr[(uint64_t)(un * f.CB + cn) * kHdrBytes + L], P = part_at(unit, cb);
    Q.commit(s);
    X.commit(xs, p);
    Q.finish(s, a);
    B.store(slot);
    __syncthreads();
    // the first task's raw bytes only now: nothing needs them before its decode is done
    uint4 raw[4];
#pragma unroll
    for (uint32_t j = 0; j < 4; j++) raw[j] = raw_at(unit, cb, j);
    uint32_t *mine = tile + 4u * h * kTokensTileRow + 4u * L;
    const uint32_t *er = tile + r8 * kTokensTileRow + tcol / 4u;
    uint32_t xr[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) xr[t] = min(16u * t + i16, p.T - 1u) * p.xrow + 8u * c4;
    for (; w.t < w.n; w.t += w.step) {
        const uint32_t cols = cols_of(cb), base = B.base, from = P;
        const bool fits = B.fits, col_ok = 16u * L < cols;
        const uint32_t start = col_ok ? B.start : (B.base & 15u) >> 2, keep = col_ok ? ~0u : 0u;
        uint32_t u2, c2;
        w.at(w.t + 2u * w.step, u2, c2);
        B.request(a, un * f.CB + cn, nn, p.cap);
        P = part_at(un, cn);
        nn = a.hdr[(uint64_t)(u2 * f.CB + c2) * kHdrBytes + L];
        if (fits) tokens_decode0<ELEM>(s, slot + start, from, keep, mine);
        else tokens_decode0<ELEM>(s, (const uint32_t *)(a.data + (base & ~15u)) + start, from, keep, mine);
        wave_lds_order();
        B.store(slot);
        f32x4_t acc[NT], acc_far[NT];
#pragma unroll
        for (int t = 0; t < NT; t++) acc[t] = acc_far[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        const uint32_t *xc = xs + (w.direct ? cb * (kCols / 2u) : 0u);
        // all steps, also where the block has fewer columns: x is zero there and the weights are masked to +0
#pragma unroll
        for (uint32_t j = 0; j < 4; j++) {
            const uint4 e = *(const uint4 *)(er + step_col(j) / 4u);
            const uint4 rw = ELEM == kElemFp8 ? expand_nibbles(make_uint2(raw[j].x, raw[j].y)) : raw[j];
            const uint32_t in = tcol + step_col(j) < cols ? ~0u : 0u;
            const bf16x8_t w0 = operand(perm(e.x, rw.x, 0x05010400u) & in, perm(e.x, rw.x, 0x07030602u) & in,
                                        perm(e.y, rw.y, 0x05010400u) & in, perm(e.y, rw.y, 0x07030602u) & in);
            const bf16x8_t w1 = operand(perm(e.z, rw.z, 0x05010400u) & in, perm(e.z, rw.z, 0x07030602u) & in,
                                        perm(e.w, rw.w, 0x05010400u) & in, perm(e.w, rw.w, 0x07030602u) & in);
            raw[j] = raw_at(un, cn, j);
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const uint32_t *x = xc + xr[t] + step_col(j) / 2u;
                acc[t] = mfma(w0, operand(*(const uint4 *)x), acc[t]);
                acc_far[t] = mfma(w0, operand(*(const uint4 *)(x + 64)), acc_far[t]);
                acc[t] = mfma(w1, operand(*(const uint4 *)(x + 4)), acc[t]);
                acc_far[t] = mfma(w1, operand(*(const uint4 *)(x + 68)), acc_far[t]);
            }
        }
        wave_lds_order();                                        // the tile's reads before the next task's writes
        // rows 0-7 (lanes 0-31) of acc plus rows 8-15 (lanes 32-63) of acc_far
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                uint32_t u = __float_as_uint(acc_far[t][e]), v = __float_as_uint(acc[t][e]);
                swap32(u, v);                                    // v, lanes 0-31: acc_far's lanes 32-63
                acc[t][e] += __uint_as_float(v);
            }
        store_part<NT, 8>(p, w, unit, sums, acc);
        unit = un;
        cb = cn;
        un = u2;
        cn = c2;
    }
    if (w.direct) finish_direct<8>(p, w, sums);
}

// ---------------------------------------------------------------------------------------------------------------
// Layout 1: a half-wave's lane (r = L >> 2, q = L & 3) holds columns 8q .. + 7 of rows r and r + 8 of a super-chunk.
// v_permlane32_swap gathers one super-chunk's 16 rows in the wave's 64 lanes (lane 4 row + q) and four ds_bpermute a
// super-chunk put them in the operand's lanes (row + 16 q).
__device__ __forceinline__ uint32_t from_lane(uint32_t idx4, uint32_t v) {
    return (uint32_t)__builtin_amdgcn_ds_bpermute((int)idx4, (int)v);
}
// products of one super-chunk pair (half 0's chunk i, half 1's chunk 8 + i of the column block); xr: the lane's place in
// each 16 tokens' rows
template <int NT>
__device__ __forceinline__ void chunk_products(bf16x8_t w0, bf16x8_t w1, bool two, const uint32_t *xc, const uint32_t (&xr)[NT],
                                               uint32_t i, f32x4_t (&acc)[NT]) {
#pragma unroll
    for (int j = 0; j < NT; j++) acc[j] = mfma(w0, operand(*(const uint4 *)(xc + xr[j] + 16u * i)), acc[j]);
    if (two) {
#pragma unroll
        for (int j = 0; j < NT; j++) acc[j] = mfma(w1, operand(*(const uint4 *)(xc + xr[j] + 16u * (i + 8u))), acc[j]);
    }
}

// The operands of one super-chunk pair from its table entries and raw bytes.
__device__ __forceinline__ void chunk_operands(const uint32_t (&e1)[4], const uint32_t (&e2)[4], const uint4 &raw, uint32_t from,
                                               bf16x8_t &w0, bf16x8_t &w1) {
    uint32_t pa[4], pb[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const uint32_t rk = u4_get(raw, k);
        pa[k] = perm(e1[k], rk, kSelPair0);
        pb[k] = perm(e2[k], rk, kSelPair2);
        swap32(pa[k], pb[k]);                                    // pa: half 0's chunk, pb: half 1's, lane 4 row + q
        pa[k] = from_lane(from, pa[k]);
        pb[k] = from_lane(from, pb[k]);
    }
    w0 = operand(pa[0], pa[1], pa[2], pa[3]);
    w1 = operand(pb[0], pb[1], pb[2], pb[3]);
}

// One task of layout 1.  nsc: the block's super-chunks (uniform); FULL: all 16, straight-line code.  In LDS a half may
// walk past its lanes' streams where the other half has more super-chunks (its weights are then not used); GLOBAL, the
// streams read from memory, it does not.  ring: the raw bytes of the next four chunks, then the next task's first four.
template <int ELEM, int NT, bool FULL, bool GLOBAL, class Tab>
__device__ __forceinline__ void tokens_chunks1(const Tab &s, const uint32_t *lane_words, uint32_t P0, const uint8_t *low,
                                               uint32_t nsc, const Coord1 &c, const Coord1 &cn, uint32_t sc0, uint4 (&ring)[4],
                                               const uint32_t *xc, const uint32_t (&xr)[NT], f32x4_t (&acc)[NT]) {
    const uint32_t lane = threadIdx.x & 63u, from = 4u * (4u * (lane & 15u) + (lane >> 4));
    Seq<ELEM> S;
    S.init_at(lane_words, P0);
#pragma unroll
    for (uint32_t i = 0; i < 8; i++) {
        if (FULL || i < nsc) {
            uint32_t e1[4] = {0u, 0u, 0u, 0u}, e2[4] = {0u, 0u, 0u, 0u};
            bf16x8_t w0, w1;
            if (!GLOBAL || sc0 + i < nsc) row_codes(S, s, e1, e2);
            chunk_operands(e1, e2, ring[i & 3u], from, w0, w1);
            chunk_products<NT>(w0, w1, FULL || i + 8u < nsc, xc, xr, i, acc);
        }
        ring[i & 3u] = i < 4u ? raw1<ELEM>(low, c, sc0 + i + 4u) : raw1<ELEM>(low, cn, sc0 + i - 4u);
    }
}

template <int ELEM, int NT, int PEEK>
__global__ void __launch_bounds__(kTokensMaxWaves * 64) k_tokens1(TokensArgs p) {
    const BlockArgs &a = p.a;
    __shared__ LutT<PEEK> s;
    extern __shared__ __attribute__((aligned(16))) uint32_t dyn[];
    const uint32_t lane = threadIdx.x & 63u, L = threadIdx.x & 31u, h = lane >> 5;
    const Shape f(a.M, a.K, 1);
    TokensTasks w;
    w.init(p, f);
    auto coord = [&](uint32_t unit, uint32_t cb) { return coord1<ELEM>(unit * f.CB + cb, 0u, f, L); };
    auto nsc_of = [&](uint32_t cb) { return cb == f.CB - 1u ? f.nsl : 16u; };
    // a half without super-chunks of its own decodes the block's first ones again, for nothing
    auto part_at = [&](uint32_t b, uint32_t cb) { return part_start(a, b, 8u * h < nsc_of(cb) ? 2u * h : 0u, L); };
    uint32_t *xs = dyn, *slot = dyn + p.xwords + w.t * p.cap;
    float *sums = (float *)(dyn + p.xwords + w.step * p.cap + kTokensOverrun);
    TabStage<PEEK> Q;
    Q.issue(a);
    uint32_t unit, cb, un, nb;
    w.at(w.t, unit, cb);
    w.at(w.t + w.step, un, nb);
    Coord1 c = coord(unit, cb);
    const uint32_t n = a.hdr[(uint64_t)c.b * kHdrBytes + L];
    StageX X;
    X.issue(p, w.cb0, w.direct ? f.CB : 1u);
    BlockStream<4> B;
    B.request(a, c.b, n, p.cap);
    uint32_t P0 = part_at(c.b, cb), nn = a.hdr[(uint64_t)(un * f.CB + nb) * kHdrBytes + L];
    Q.commit(s);
    X.commit(xs, p);
    Q.finish(s, a);
    B.store(slot);
    uint4 ring[4];
#pragma unroll
    for (uint32_t i = 0; i < 4; i++) ring[i] = raw1<ELEM>(a.low, c, 8u * h + i);
    __syncthreads();
    uint32_t xr[NT];
#pragma unroll
    for (int j = 0; j < NT; j++) xr[j] = min(16u * j + (lane & 15u), p.T - 1u) * p.xrow + 4u * (lane >> 4);
    for (; w.t < w.n; w.t += w.step) {
        const uint32_t start = B.start, base = B.base, P = P0, nsc = nsc_of(cb);
        const bool fits = B.fits;
        const Coord1 cn = coord(un, nb);
        uint32_t u2, b2;
        w.at(w.t + 2u * w.step, u2, b2);
        B.request(a, cn.b, nn, p.cap);
        P0 = part_at(cn.b, nb);
        nn = a.hdr[(uint64_t)(u2 * f.CB + b2) * kHdrBytes + L];
        f32x4_t acc[NT];
#pragma unroll
        for (int j = 0; j < NT; j++) acc[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        const uint32_t *xc = xs + (w.direct ? cb * (kCols / 2u) : 0u);
        if (fits && nsc == 16u)
            tokens_chunks1<ELEM, NT, true, false>(s, slot + start, P, a.low, nsc, c, cn, 8u * h, ring, xc, xr, acc);
        else if (fits)
            tokens_chunks1<ELEM, NT, false, false>(s, slot + start, P, a.low, nsc, c, cn, 8u * h, ring, xc, xr, acc);
        else
            tokens_chunks1<ELEM, NT, false, true>(s, (const uint32_t *)(a.data + (base & ~15u)) + start, P, a.low, nsc, c, cn,
                                                  8u * h, ring, xc, xr, acc);
        wave_lds_order();
        B.store(slot);
        wave_lds_order();
        store_part<NT, 16>(p, w, unit, sums, acc);
        c = cn;
        unit = un;
        cb = nb;
        un = u2;
        nb = b2;
    }
    if (w.direct) finish_direct<16>(p, w, sums);
}

// ---------------------------------------------------------------------------------------------------------------
// Layout 2: the same fragment order without streams.  A super-chunk pair's 2 x 16 rows x 32 columns go through the
// wave's LDS patch (row r's 16-byte piece q at place q ^ (r >> 2), so that neither the writes by lane nor the reads by
// row meet in a bank), where the lanes' exceptions replace the planes' zeros before the operands are read.
// A block's exception entries on their way into the wave's LDS, a task ahead; `fits`: else they are read from memory.
template <int ELEM>
struct ExcStream {
    static constexpr uint32_t N = kTokensExcWords / 64u, SIZE = ELEM == kElemFp8 ? 2 : 3;
    typedef __attribute__((aligned(1))) uint32_t any32;
    uint32_t v[N], n, first, bytes, base;                        // of the lane: entries, the first one's byte
    bool fits;
    __device__ __forceinline__ void request(const BlockArgs &a, uint32_t b, uint32_t cnt) {
        const uint32_t lane = threadIdx.x & 63u, incl = half_scan_incl(cnt, lane & 31u);
        n = cnt;
        first = (incl - cnt) * SIZE;
        bytes = __builtin_amdgcn_readlane(incl, 31) * SIZE;
        base = a.bases[b];
        fits = bytes <= kTokensExcWords * 4u && bytes >= 4u;
        // a word that would pass the last entry is read up to three bytes early and moved down: nothing past it is read
        if (fits) {
#pragma unroll
            for (uint32_t k = 0; k < N; k++)
                if (256u * k < bytes) v[k] = *(const any32 *)(a.data + base + min(4u * (lane + 64u * k), bytes - 4u));
        }
    }
    __device__ __forceinline__ void store(uint32_t *slot) const {
        if (!fits) return;
        const uint32_t lane = threadIdx.x & 63u;
#pragma unroll
        for (uint32_t k = 0; k < N; k++) {
            const uint32_t at = 4u * (lane + 64u * k);
            if (at < bytes) slot[at / 4u] = v[k] >> (8u * (at - min(at, bytes - 4u)));
        }
    }
};
// A lane's next exception: position (0..255; 0xFFFF: none) and BF16 bits, from LDS or, `mem` set, from memory.
template <int ELEM>
struct ExcCursor {
    const uint8_t *lds, *mem;
    uint32_t at, left, pos, bits;
    __device__ __forceinline__ void load() {
        constexpr uint32_t SIZE = ExcStream<ELEM>::SIZE;
        pos = 0xFFFFu;
        if (left == 0u) return;
        uint32_t e[3];
#pragma unroll
        for (uint32_t i = 0; i < SIZE; i++) e[i] = mem ? mem[at + i] : lds[at + i];
        pos = e[0];
        if constexpr (ELEM == kElemFp8) bits = __float_as_uint(e4m3_to_f32(e[1])) >> 16;     // exact
        else bits = e[1] | e[2] << 8;
    }
    __device__ __forceinline__ void next() {
        at += ExcStream<ELEM>::SIZE;
        left--;
        load();
    }
};

template <int ELEM, int NT>
__global__ void __launch_bounds__(kTokensMaxWaves * 64) k_tokens2(TokensArgs p) {
    const BlockArgs &a = p.a;
    extern __shared__ __attribute__((aligned(16))) uint32_t dyn[];
    const uint32_t lane = threadIdx.x & 63u, L = threadIdx.x & 31u, h = lane >> 5;
    const uint32_t i16 = lane & 15u, c4 = lane >> 4;
    const Shape f(a.M, a.K, 2);
    TokensTasks w;
    w.init(p, f);
    const RankTab tab{a.lut[0], a.lut[1], a.lut[2], a.lut[3]};
    const uint8_t *rplane = a.low + f.nib2_bytes();
    auto nsc_of = [&](uint32_t cb) { return cb == f.CB - 1u ? f.nsl : 16u; };
    uint2 nib[8];
    uint4 raw[8];                                                // fp8: the three words of chunks i, i + 1 in raw[i]
    // chunk 8h + i of a unit's block (past the block's last it re-reads that one)
    auto request = [&](uint32_t rb, uint32_t cb, uint32_t i) {
        const uint32_t sc = min(8u * h + i, nsc_of(cb) - 1u);
        nib[i] = ldnt2(a.low + ((uint64_t)(rb * f.spr + cb * 16u + sc) * kLanes + L) * 8u);
        if constexpr (ELEM == kElemFp8) {
            if ((i & 1u) == 0u) {
                const uint8_t *pp = rplane + (((uint64_t)rb * f.spr2 + cb * 8u + (sc >> 1)) * 3u * kLanes + L) * 4u;
                raw[i].x = ldnt1(pp);
                raw[i].y = ldnt1(pp + kLanes * 4u);
                raw[i].z = ldnt1(pp + 2u * kLanes * 4u);
            }
        } else {
            raw[i] = ldnt4(rplane + ((uint64_t)(rb * f.spr + cb * 16u + sc) * kLanes + L) * 16u);
        }
    };
    uint32_t unit, cb;
    w.at(w.t, unit, cb);
    StageX S;
    S.issue(p, w.cb0, w.direct ? f.CB : 1u);
#pragma unroll
    for (uint32_t i = 0; i < 8; i++) request(unit, cb, i);
    constexpr uint32_t own = kTokensPatchWords + kTokensExcWords;
    uint32_t *xs = dyn, *patch = dyn + p.xwords + w.t * own, *slot = patch + kTokensPatchWords;
    float *sums = (float *)(dyn + p.xwords + w.step * own);
    ExcStream<ELEM> E;
    E.request(a, unit * f.CB + cb, a.hdr[(uint64_t)(unit * f.CB + cb) * kHdrBytes + L]);
    uint32_t un, cn;
    w.at(w.t + w.step, un, cn);
    uint32_t nn = a.hdr[(uint64_t)(un * f.CB + cn) * kHdrBytes + L];
    S.commit(xs, p);
    E.store(slot);
    __syncthreads();
    const uint32_t r = L >> 2, q = L & 3u;
    uint32_t *wa = patch + 256u * h + 16u * r + 4u * ((q ^ (r >> 2)) & 3u);
    uint32_t *wb = patch + 256u * h + 16u * (r + 8u) + 4u * ((q ^ ((r + 8u) >> 2)) & 3u);
    const uint32_t *ra = patch + 16u * i16 + 4u * ((c4 ^ (i16 >> 2)) & 3u);
    uint32_t xr[NT];
#pragma unroll
    for (int j = 0; j < NT; j++) xr[j] = min(16u * j + i16, p.T - 1u) * p.xrow + 4u * c4;
    for (; w.t < w.n; w.t += w.step) {
        const uint32_t nsc = nsc_of(cb), *xc = xs + (w.direct ? cb * (kCols / 2u) : 0u);
        ExcCursor<ELEM> X{(const uint8_t *)slot, E.fits ? nullptr : a.data + E.base, E.first, E.n, 0u, 0u};
        uint32_t u2, c2;
        w.at(w.t + 2u * w.step, u2, c2);
        E.request(a, un * f.CB + cn, nn);
        nn = a.hdr[(uint64_t)(u2 * f.CB + c2) * kHdrBytes + L];
        X.load();
        while (X.pos < 128u * h) X.next();                       // half 1: past the exceptions of chunks 0-7
        f32x4_t acc[NT];
#pragma unroll
        for (int j = 0; j < NT; j++) acc[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (uint32_t i = 0; i < 8; i++) {
            if (i < nsc) {
                uint32_t pa[4], pb[4];
                if constexpr (ELEM == kElemFp8) {
                    const uint4 c = raw[i & ~1u];
                    if (i & 1u) decode_sc<ELEM, 4>(tab, nib[i], c, c.x, c.y, c.z, pa, pb);
                    else decode_sc<ELEM, 0>(tab, nib[i], c, c.x, c.y, c.z, pa, pb);
                } else {
                    decode_sc<ELEM, 0>(tab, nib[i], raw[i], 0u, 0u, 0u, pa, pb);
                }
                *(uint4 *)wa = make_uint4(pa[0], pa[1], pa[2], pa[3]);
                *(uint4 *)wb = make_uint4(pb[0], pb[1], pb[2], pb[3]);
                const uint32_t end = 128u * h + 16u * (i + 1u);
                while (X.pos < end) {                            // this super-chunk's exceptions of the lane
                    const uint32_t j = X.pos & 15u;
                    uint16_t *o = (uint16_t *)((j >> 1) & 1u ? wb : wa);
                    o[4u * ((j >> 3) & 1u) + 2u * ((j >> 2) & 1u) + (j & 1u)] = (uint16_t)X.bits;
                    X.next();
                }
                wave_lds_order();
                const bf16x8_t w0 = operand(*(const uint4 *)ra), w1 = operand(*(const uint4 *)(ra + 256));
                wave_lds_order();
                chunk_products<NT>(w0, w1, i + 8u < nsc, xc, xr, i, acc);
            }
            if (ELEM != kElemFp8) request(un, cn, i);
            else if (i & 1u) {
                request(un, cn, i - 1u);
                request(un, cn, i);
            }
        }
        wave_lds_order();
        E.store(slot);
        wave_lds_order();
        store_part<NT, 16>(p, w, unit, sums, acc);
        unit = un;
        cb = cn;
        un = u2;
        cn = c2;
    }
    if (w.direct) finish_direct<16>(p, w, sums);
}

// ---------------------------------------------------------------------------------------------------------------
template <int ELEM, int NT>
static int launch_tokens_t(int layout, const TokensPlan &q, const TokensArgs &p, hipStream_t st) {
    void (*const kernel)(TokensArgs) = layout == 2   ? k_tokens2<ELEM, NT>
                                       : layout == 1 ? (q.seq13 ? k_tokens1<ELEM, NT, kPeekSeq> : k_tokens1<ELEM, NT, kPeek>)
                                                     : (q.seq13 ? k_tokens0<ELEM, NT, kPeekSeq> : k_tokens0<ELEM, NT, kPeek>);
    hipError_t e;
    // more than 64 KB of LDS: raise the kernel's limit (idempotent, so concurrent first calls are fine)
    if (q.lds > 64u * 1024u) {
        e = hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)q.lds);
        if (e != hipSuccess) return (int)e;
    }
    hipLaunchKernelGGL(kernel, dim3(q.grid), dim3(q.threads), q.lds, st, p);
    e = hipGetLastError();
    if (e != hipSuccess || p.direct) return (int)e;
    const uint64_t items = (uint64_t)p.T * (p.Mu / 4u);
    hipLaunchKernelGGL(k_tokens_finish, dim3((uint32_t)((items + 255u) / 256u)), dim3(256), 0, st, p, Shape(p.a.M, p.a.K, layout).CB);
    return (int)hipGetLastError();
}

int launch_tokens(int layout, int elem_t, const TokensPlan &q, const TokensArgs &p, hipStream_t st) {
    const bool fp8 = elem_t == kElemFp8;
    if (p.T <= 16u) return fp8 ? launch_tokens_t<kElemFp8, 1>(layout, q, p, st) : launch_tokens_t<kElemBf16, 1>(layout, q, p, st);
    if (p.T <= 32u) return fp8 ? launch_tokens_t<kElemFp8, 2>(layout, q, p, st) : launch_tokens_t<kElemBf16, 2>(layout, q, p, st);
    return fp8 ? launch_tokens_t<kElemFp8, 4>(layout, q, p, st) : launch_tokens_t<kElemBf16, 4>(layout, q, p, st);
}

}  // namespace nwc
