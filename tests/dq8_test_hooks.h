/*
 * dq8_test_hooks.h -- entry points of libdisc_q8_ral.so that exist for the tests and for
 * tuning only: they force one kernel variant where the library would choose, and expose the
 * MFMA register layouts to a brute-force check.  Not part of the product ABI (include/).
 */
#ifndef DQ8_TEST_HOOKS_H_
#define DQ8_TEST_HOOKS_H_

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* dq8_qgemm (include/disc_q8.h), forcing one kernel variant:
 *  -1 heuristic, 0 generic scalar kernel, 1.. MFMA tile configurations
 *  (dq8_qgemm_num_variants() of them, names from dq8_qgemm_variant_name()).  A problem
 *  an MFMA variant cannot take (unaligned rows; K % 16 != 0 without scratch) runs on the
 *  generic kernel whatever the variant; non-zero zx / zw with a forced MFMA variant is an error
 *  (they need the heuristic or the generic variant), and so is a persistent variant with result
 *  rows off 16 bytes or, of the 256-row ones, with 4-byte results. */
int dq8_qgemm_variant(int variant, const int8_t* A, int64_t lda,
                      const int8_t* W, int64_t ldw, void* out, int64_t ldo,
                      int64_t M, int64_t N, int64_t K, int tp_a, int tp_b,
                      int epilogue, const void* bias, int bias_kind,
                      const float* sx, int64_t n_sx, const float* sw,
                      int64_t n_sw, const float* so, int64_t n_so, int32_t zx,
                      int32_t zw, int32_t zo, void* workspace,
                      size_t workspace_bytes, void* stream);
int dq8_qgemm_num_variants(void);
const char* dq8_qgemm_variant_name(int variant);


/* dq8_qconv2d_ws (include/disc_q8.h), forcing one kernel variant (numbering as above). */
int dq8_qconv2d_variant(int variant, const int8_t* in,
                        const int64_t in_sizes[4], const int8_t* w,
                        const int64_t w_sizes[4], const int32_t padding[4],
                        const int32_t metadata[17], void* out,
                        const int64_t out_sizes[4], int epilogue,
                        const void* bias, int bias_kind, const float* sx,
                        const float* sw, int64_t n_sw, const float* so,
                        int32_t zo, void* workspace, size_t workspace_bytes,
                        void* stream);

/* Runs one v_mfma_i32_32x32x32_i8 and one v_mfma_i32_16x16x64_i8 on device
 * buffers: a[32*32] (row i, k contiguous), b[32*32] (column j, k contiguous) ->
 * d32[32*32] row-major; a16[16*64], b16[16*64] -> d16[16*16].  Lets a test pin
 * the operand and result register layouts against brute force. */
int dq8_mfma_probe(const int8_t* a, const int8_t* b, int32_t* d32,
                   const int8_t* a16, const int8_t* b16, int32_t* d16,
                   void* stream);

/* Whether dq8_observe_fake_quant (include/disc_q8.h) of a tensor with 16-byte aligned pointers folds
 * the observed range in its last kernel (two launches); otherwise a kernel of its own does. */
int dq8_observe_folds_range(int64_t outer, int64_t channels, int64_t inner);

/* What dq8_weight_only_qgemm (include/disc_q8.h) plans for a problem when it has all the scratch it
 * wants: plan[0] the tile form (numbered as in weight_only.hip; -1 where a kernel for few rows runs),
 * plan[1] the k ranges, plan[2], plan[3] the rows and channels of a tile.  ragged: rows that are not
 * 16-byte aligned multiples of 16 bytes. */
void dq8_weight_only_plan(int64_t M, int64_t N, int64_t K, int x_dtype, int ragged, int plan[4]);

/* What dq8_qgemm runs for A [M, K] and W [N, K], k-contiguous rows that are not all 16-byte aligned multiples
 * of 16 bytes, K at least 64: the kernel's name, and form[0] = 1 tiles on rows of whole words, 2 the small-M
 * kernel, 3 the 64 x 64 tiles through registers, 0 (name "") a copy to aligned rows first.  a_at, w_at: the
 * operands' addresses modulo 16; zw: the weights' zero point; out_bytes: of a result element, 1 or 4. */
const char* dq8_qgemm_rows_kernel(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldw, int a_at,
                                  int w_at, int zw, int out_bytes, int* form);

#ifdef __cplusplus
}
#endif
#endif /* DQ8_TEST_HOOKS_H_ */
