// nwc_launch.h -- launch plans and the launchers each kernel file exports to the C ABI layer (abi.cpp).
#pragma once
#include "nwc_device.h"

#include <algorithm>

namespace nwc {

struct LaunchPlan {
    int layout;
    bool pipe;              // layout 0: rounds through two region buffers, the next round prefetched
    uint32_t split;         // layout 0: half-waves per block (1, or 2 or 4 with the row index)
    bool seq13;             // layout 0 token path: the 13-bit decode table (a larger static LDS share)
    bool multi;             // layout 1: several items (block, quarter) per half-wave, one 16-row group per workgroup
    uint32_t tail;          // layout 0 token path: k_layout0t, G whole row groups then the rest split tail-ways (2, 4)
    uint32_t grid, threads, lds, G;
    uint32_t slot_words;    // layout 0: region-buffer words per block
};

int launch_prefix(const LaunchPlan &p, int elem_t, int mode, bool xbf16, const BlockArgs &a, hipStream_t st);
int launch_fixed(const LaunchPlan &p, int elem_t, int mode, bool xbf16, const BlockArgs &a, hipStream_t st);
int launch_gather_prefix(int layout, int elem_t, const GatherArgs &a, hipStream_t st);
// layouts 0/1 gather with the row index (k_gather0x / k_gather1x); seq: the 13-bit table or null
int launch_gather0x(int layout, int elem_t, const GatherArgs &a, const uint16_t *aux, const uint32_t *seq, hipStream_t st);
// layout-0 token path for ntok (2..4) activation vectors at once (k_layout0_batch); plan from plan_layout0_batch
int launch_layout0_batch(const LaunchPlan &p, int elem_t, const BlockArgs &a, uint32_t ntok, hipStream_t st);
// A small batch of tokens on the matrix cores (kern_tokens.hip).
struct TokensArgs {
    BlockArgs a;            // out: y BF16 [T x M]; aux: the row index (layout 1); seq: the 13-bit table
    const uint16_t *x;      // BF16 [T][ldx]
    float *part;            // sums of each column block [CB][T][Mu]
    uint32_t T, ldx, Mu;    // Mu: rows of all row groups
    uint32_t parts;         // runs of row groups: workgroups in all (direct) or per column block
    bool direct;            // a workgroup has all column blocks of its rows and finishes them; else `part` and a second kernel
    uint32_t xrow, xwords;  // LDS words of a token's activations (4 banks past a whole number of bank rows) and of all
    uint32_t cap;           // LDS words of a block's streams in a wave's share (layouts 0/1)
};
struct TokensPlan {
    uint32_t grid, threads, lds;
    bool seq13;
};
constexpr uint32_t kTokensMaxWaves = 16;
// LDS words of a wave: layout 0's tile of exponent bytes (8 rows, 4 banks apart), layout 2's super-chunk pair
constexpr uint32_t kTokensTileRow = 132, kTokensTileWords = 8 * kTokensTileRow, kTokensPatchWords = 512;
constexpr uint32_t kTokensExcWords = 256;   // a block's exceptions (fp8: 32 lanes x 7 x 2 bytes on average for Gaussian weights)
constexpr uint32_t kTokensOverrun = 128;   // 7 super-chunks x 16 codes of at most 24 bits, and the cursor's words
int launch_tokens(int layout, int elem_t, const TokensPlan &q, const TokensArgs &p, hipStream_t st);
int launch_gather_fixed(int elem_t, const GatherArgs &a, hipStream_t st);
// layout-0 prefill (k_prefill0): tt tokens per workgroup tile (64, 128, 256 or 512)
int launch_prefill0(int elem_t, uint32_t tt, const PrefillArgs &p, hipStream_t st);
// Y[T x N] = X[T x K] W[N x K]^T (+ bias), BF16 (k_gemm_xwt); the launcher fills nT, S, stages, cnt and part
struct GemmArgs {
    const uint16_t *x, *w, *bias;
    uint16_t *y;
    float *part;            // S partial tiles per output tile (split products)
    uint32_t *cnt;          // per output tile: workgroups of its splits that have finished
    uint32_t ldx, ldw, T, N, K, nT, S, stages;
};
constexpr uint32_t kGemmCounters = 1024;
constexpr uint64_t kGemmScratchBytes = 24ull << 20;     // nwc_gemm_xbf16_noalloc's workspace per GPU
uint32_t gemm_splits(uint32_t T, uint32_t N, uint32_t K, int ncu);
uint64_t gemm_workspace_bytes(uint32_t T, uint32_t N, uint32_t K, int ncu);
int launch_gemm_xwt(GemmArgs g, void *ws, int ncu, hipStream_t st);
// the current device's copy of the library's static workspace (its counters cleared on `st` by the first call on
// the device outside graph capture, and by every captured call before that), or null with *err set
void *gemm_scratch(hipStream_t st, int *err);
int launch_ref_fp8(const uint8_t *w, const float *scale, const float *x, uint16_t *y, uint32_t M, uint32_t K, int ncu,
                   hipStream_t st);
int launch_ref_bf16(const uint16_t *w, const uint16_t *x, uint16_t *y, uint32_t M, uint32_t K, int ncu, hipStream_t st);
int launch_stream_read(const void *p, uint64_t bytes, uint32_t *out, uint32_t grid, hipStream_t st);

}  // namespace nwc
