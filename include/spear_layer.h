/*
 * spear_layer.h -- C ABI of the MI355X (gfx950) kernels that run parts of a whole Phalanx layer for the package's own
 * Python classes. The operator's boundary is spear_btp.h, whose conventions (dtype tags, error codes, streams,
 * spear_btp_last_error) hold here too. None of these has a counterpart function in the reference.
 */
#ifndef SPEAR_LAYER_H_
#define SPEAR_LAYER_H_

#ifdef __cplusplus
extern "C" {
#endif

/* The mixing stage on a whole prompt of any length L >= 1, and the streaming state that decoding continues from
 * (spear_phalanx_mix_step): what spear_phalanx_mix_prefill does, for lengths that end inside a block too.
 *     a_logit [B, L, H]   b_logit, c [B, L, kv_heads * 16]   v, out [B, L, H * 16]      16-bit, `dtype`
 *     h, c_prev [B, H, 16] fp32    r [B, H] fp32    pos [B] int32      every element is written
 * Tensor pointers 16-byte aligned; r and pos 4-byte. */
int spear_layer_prefill(const void* a_logit, const void* b_logit, const void* c, const void* v, void* out, float* h,
                        float* r, float* c_prev, int* pos, int B, int L, int H, int kv_heads, int dtype, void* stream);

#ifdef __cplusplus
}
#endif
#endif /* SPEAR_LAYER_H_ */
