/* nwc_private.h -- entry points of nwc_ops.so that only this package's Python side calls (nwc_amd/_abi.py PRIVATE).  They
 * are not part of the C ABI of include/nwc_ops.h and may change with any build. */
#ifndef NWC_PRIVATE_H
#define NWC_PRIVATE_H
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* A small batch on the matrix cores, every layout and element type: y BF16 [ntok][M] = RNE_bf16(scale * (W x[t]) + bias)
 * for 2 <= ntok <= 64 and K >= 8, fp32 accumulation in a fixed order.  x BF16 [ntok][ldx], ldx at least K; bias BF16 [M] or null;
 * scale fp32 [M] or null; row_index (required for layouts 0 and 1) and seq_table (null: the stored LUT) as
 * nwc_linear_xbf16.  `ws`: 4 * ntok * Mp * CB bytes (Mp * CB: nwc_layout's out[2]) of device memory, 16-byte aligned,
 * that no other call in flight uses; its contents do not matter.  0, -1 for arguments it does not take, or a HIP error. */
int nwc_tokens(void *stream, const uint8_t *data, const uint32_t *bases, const uint8_t *hdr, const uint32_t *tab,
               const uint8_t *low, const uint16_t *row_index, const uint32_t *seq_table, const uint16_t *x, uint32_t ldx,
               const uint16_t *bias, const float *scale, uint16_t *y, void *ws, uint64_t ws_bytes, uint64_t n, uint32_t K,
               int elem, uint32_t ntok);

/* The encoder on the GPU (kern_encode.hip), in the order a caller runs them; w: the row-major source on the device.
 * nwc_encode_supported: whether it takes the shape (else the host's nwc_encode).
 * nwc_encode_hist adds the symbol counts of n weights to count[0..127] and, where fp8 input holds NaN, to count[128].
 * nwc_encode_rank (host) turns the counts into psym[0..1023] (as nwc_encode) and rank[0..127].
 * nwc_encode_sizes writes hdr[32 nb] and each block's bytes, and sets *over where a lane passes 255 words or exceptions.
 * nwc_encode_write writes streams (block b at bases[b], a multiple of 8) and the raw plane; what it does not write of
 * `data` and `low` (gaps, slack) the caller has zeroed.  0, -1, or a HIP error. */
int nwc_encode_supported(uint64_t M, uint32_t K, int elem);
int nwc_encode_hist(void *stream, const void *w, uint64_t n, int elem, uint64_t *count);
int nwc_encode_rank(const uint64_t *count, int elem, uint16_t *psym, uint8_t *rank);
int nwc_encode_sizes(void *stream, const void *w, uint64_t M, uint32_t K, int elem, const uint8_t *rank, uint8_t *hdr,
                     uint32_t *size, uint32_t *over);
int nwc_encode_write(void *stream, const void *w, uint64_t M, uint32_t K, int elem, const uint8_t *rank,
                     const uint8_t *hdr, const uint32_t *bases, uint8_t *data, uint8_t *low);

/* dst[to[b] + j] = src[from[b] + j] for every block b and j < size[b]; all multiples of 4. */
int nwc_copy_spans(void *stream, const uint8_t *src, const int64_t *from, uint8_t *dst, const int64_t *to,
                   const int64_t *size, uint32_t nb);

#ifdef __cplusplus
}
#endif
#endif
