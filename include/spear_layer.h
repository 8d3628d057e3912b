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
 * L < 1 is refused. Tensor pointers 16-byte aligned; r and pos 4-byte. */
int spear_layer_prefill(const void* a_logit, const void* b_logit, const void* c, const void* v, void* out, float* h,
                        float* r, float* c_prev, int* pos, int B, int L, int H, int kv_heads, int dtype, void* stream);

/* One token of B sequences through the layer's four input projections and the mixing stage's step (spear_phalanx_mix_step
 * with positions on the device), bf16 operands, fp32 sums and state:
 *     x [B, K], rows ldx elements apart   w_a [H, K]   w_b, w_c [kv_heads * 16, K]   w_v [H * 16, K]   b_a, b_b, b_c biases
 *     out [B, H * 16]    h, c_prev [B, H, 16] fp32    r [B, H] fp32    pos [B] int32       state updated in place
 * With advance == 0 pos is read only, and is to be moved by spear_layer_linear on the results.
 * K and ldx multiples of 8; x, weights, out, h and c_prev 16-byte aligned, b_b and b_c 8-byte, b_a 2-byte, r and pos 4-byte. */
int spear_layer_token(const void* x, long long ldx, const void* w_a, const void* b_a, const void* w_b, const void* b_b,
                      const void* w_c, const void* b_c, const void* w_v, void* out, float* h, float* r, float* c_prev, int* pos,
                      int block_len, int advance, int B, int K, int H, int kv_heads, void* stream);

/* Column sums of n (1 .. 5) dense fp32 arrays, rounded to `dtype` (16-bit), in one launch:
 *     out[i][c] = sum over r of in[i][r * cols[i] + c]
 * in[i] 16-byte and out[i] 8-byte aligned. An array without rows gives zeros. */
int spear_layer_sums(int n, const float* const* in, void* const* out, const long long* rows, const long long* cols, int dtype,
                     void* stream);

/* The four projections' weights one under the other in the order b, c, v, a, and the padding of the gradient buffer they meet:
 *     stacked [ld, K]: w_b [Fkv, K], w_c [Fkv, K], w_v [F, K], w_a [H, K], zero rows       packed [M, ld]: columns 2 Fkv + F + H .. ld <- 0
 * 16-bit elements, dense, 16-byte aligned; ld and K multiples of 8. */
int spear_layer_stack(const void* w_a, const void* w_b, const void* w_c, const void* w_v, void* stacked, void* packed, long long M,
                      int ld, int K, int H, int Fkv, int F, void* stream);

/* The same weights transposed, as spear_layer_linear takes them for the input gradients, and proj_out's, and the same padding:
 *     stacked [K, ld]: columns w_b^T, w_c^T, w_v^T, w_a^T, zeros       out_t [F, K]: w_out^T, w_out [K, F]
 *     packed [M, ld]: columns 2 Fkv + F + H .. ld <- 0
 * 16-bit elements, dense, 16-byte aligned; ld, K, Fkv and F multiples of 8. */
int spear_layer_transpose(const void* w_a, const void* w_b, const void* w_c, const void* w_v, const void* w_out, void* stacked, void* out_t,
                          void* packed, long long M, int ld, int K, int H, int Fkv, int F, void* stream);

/* n (1 .. 4) linear layers on the same rows, bf16 with fp32 sums:  out[i] [M, N[i]] = x [M, K] w[i]^T + bias[i] (null: none). x has
 * rows ldx elements apart, the rest is dense; K and ldx multiples of 8; x and w 16-byte, out 8-byte, bias 2-byte aligned.
 * pos: NULL, or int32 [M] block positions that are moved on by one, to 0 from block_len - 1. */
int spear_layer_linear(int n, const void* x, long long ldx, int M, int K, const void* const* w, const void* const* bias,
                       void* const* out, const int* N, int* pos, int block_len, void* stream);

/* Which of its kernels spear_layer_linear takes for such a call (without positions): 0 the one for few rows, 1 tiles of 128 x 128, 2 of 256 x 256;
 * -1 for a shape that it refuses. */
int spear_layer_linear_choice(int n, long long ldx, int M, int K, const int* N);

/* n (1 .. 2) products over M tokens, bf16, as fp32 parts:  dy[i]^T x[i], [N[i], K[i]], cut into splits[i] runs of tokens.
 *     dy[i] [M, N[i]], rows ld_dy[i] elements apart, cols_dy[i] >= N[i] of which may be read       x[i] [M, K[i]] dense
 *     parts  fp32, 65536 * sum of splits[i] ceil(N[i] / 256) ceil(K[i] / 256) elements; written in the order that
 *            spear_layer_wgrad_sums reads
 * ld_dy, cols_dy and K multiples of 8; pointers 16-byte aligned; 1 <= splits[i] <= ceil(M / 32). */
int spear_layer_wgrad(int n, const void* const* dy, const int* ld_dy, const int* cols_dy, const int* N, const void* const* x, const int* K,
                      const int* splits, long long M, float* parts, void* stream);

/* The same with results that need no parts: dw[i] NULL, or with splits[i] = 1 and K[i] below 2^21 the product itself, [N[i], K[i]] dense, rounded to bf16
 * (8-byte aligned). Such a product takes no room in `parts`, which may be NULL if none does; spear_layer_wgrad_sums is for the others. */
int spear_layer_wgrad_to(int n, const void* const* dy, const int* ld_dy, const int* cols_dy, const int* N, const void* const* x, const int* K,
                         const int* splits, long long M, float* parts, void* const* dw, void* stream);

/* The number of splits for one of these products that the library's model of it expects to be fastest. */
int spear_layer_wgrad_splits(long long M, int N, int K);
/* The same of `atleast` splits and more, for parts that are sums over fewer tokens. */
int spear_layer_wgrad_splits_from(long long M, int N, int K, int atleast);

/* The parts added up and rounded to `dtype` (16-bit), dw[i] [N[i], K[i]] dense, and m (0 .. 3) column sums of dense fp32 arrays as
 * spear_layer_sums makes them, in one launch. dw[i] 8-byte aligned. */
int spear_layer_wgrad_sums(int n, const float* parts, const int* N, const int* K, const int* splits, void* const* dw, int m,
                           const float* const* in, void* const* out, const long long* rows, const long long* cols, int dtype, void* stream);

#ifdef __cplusplus
}
#endif
#endif /* SPEAR_LAYER_H_ */
