/* nwc_private.h -- entry points of nwc_ops.so that only this package's Python side calls (nwc_amd/_abi.py PRIVATE).  They
 * are not part of the C ABI of include/nwc_ops.h and may change with any build. */
#ifndef NWC_PRIVATE_H
#define NWC_PRIVATE_H
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* A small batch on the matrix cores, every layout and element type: y BF16 [ntok][M] = RNE_bf16(scale * (W x[t]) + bias)
 * for 2 <= ntok <= 64, fp32 accumulation in a fixed order.  x BF16 [ntok][ldx], ldx at least K; bias BF16 [M] or null;
 * scale fp32 [M] or null; row_index (required for layouts 0 and 1) and seq_table (null: the stored LUT) as
 * nwc_linear_xbf16.  `ws`: 4 * ntok * Mp * CB bytes (Mp * CB: nwc_layout's out[2]) of device memory, 16-byte aligned,
 * that no other call in flight uses; its contents do not matter.  0, -1 for arguments it does not take, or a HIP error. */
int nwc_tokens(void *stream, const uint8_t *data, const uint32_t *bases, const uint8_t *hdr, const uint32_t *tab,
               const uint8_t *low, const uint16_t *row_index, const uint32_t *seq_table, const uint16_t *x, uint32_t ldx,
               const uint16_t *bias, const float *scale, uint16_t *y, void *ws, uint64_t ws_bytes, uint64_t n, uint32_t K,
               int elem, uint32_t ntok);

#ifdef __cplusplus
}
#endif
#endif
