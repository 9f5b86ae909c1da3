/*
 * mls_ext.h — entry points of libmls_hip.so for this package's own Python modules.
 *
 * They follow mls.h's conventions (host-side validation, status codes, the caller owns
 * every buffer, work enqueued on `stream`) and carry no ABI version of their own: the
 * modules and the library are built together.
 */
#ifndef MLS_EXT_H
#define MLS_EXT_H

#include "mls.h"

#ifdef __cplusplus
extern "C" {
#endif

/* ---------------------------------------------------------------- weight-only GEMMs */

/* mls_int8_gemm_ws / mls_int4_gemm_ws with a workspace of mlsx_wq_workspace bytes (256-byte
 * aligned; 0: none): shapes whose tiles would not fill the GPU, or whose K is a multiple of
 * 32 but not of 64, run with the reduction axis split over blocks and fp32 partial products
 * in the workspace (gemm_ksplit.hip; at most 384 MiB of them, and of x as three parts, whatever
 * the rows); every other call is the _ws one. */
/* The number of ranges that K is split into for such a call, 1: these kernels unsplit, 0: the _ws entry
 * point's kernels (faster there by the models of both). */
int mlsx_wq_ksplit(int wbits, int64_t M, int64_t N, int64_t K, int a_dt, int group);
int64_t mlsx_wq_workspace(int wbits, int64_t M, int64_t N, int64_t K, int a_dt, int group);
int mlsx_int8_gemm(const void* a, int a_dt, int64_t lda, const int8_t* w, int64_t ldw, const void* s, int s_dt,
                   void* c, int c_dt, int64_t ldc, int64_t M, int64_t N, int64_t K, void* workspace,
                   int64_t ws_bytes, mls_stream_t stream);
int mlsx_int4_gemm(const void* a, int a_dt, int64_t lda, const uint8_t* w, int64_t ldw, const void* s, int s_dt,
                   int64_t ld_sn, int64_t ld_sg, int group, void* c, int c_dt, int64_t ldc, int64_t M, int64_t N,
                   int64_t K, void* workspace, int64_t ws_bytes, mls_stream_t stream);

/* ---------------------------------------------------------------- paged attention */

/* mls_paged_attention_decode with the contexts cut into pieces of equal length instead of as
 * many splits a sequence, so that a batch of unequal lengths keeps the GPU even; the length comes
 * from the batch's contexts, on the device, whatever the tables' width. Arguments as there; the
 * workspace holds mlsx_paged_attention_workspace floats (0: none). */
int64_t mlsx_paged_attention_workspace(int64_t n_seqs, int64_t H, int64_t D, int64_t block_size, int64_t max_blocks);
int mlsx_paged_attention_decode(const void* q, int q_dt, int64_t q_ss, int64_t q_sh, const void* k_pool,
                                const void* v_pool, int kv_dt, int64_t kv_sb, int64_t kv_sh, int64_t kv_st,
                                int64_t num_blocks, const int32_t* block_tables, int64_t bt_ss, int64_t max_blocks,
                                const int32_t* context_lens, void* out, int64_t o_ss, int64_t o_sh, int64_t n_seqs,
                                int64_t H, int64_t D, int64_t block_size, float scale, float* workspace,
                                int64_t workspace_floats, mls_stream_t stream);

/* ---------------------------------------------------------------- grouped INT4 GEMMs */

/* 1 where the grouped INT4 entry points of mls.h take a call of M_total rows on the kernel for
 * few rows an expert (grouped_skinny.hip), 0: on the chunk kernel, whose results it repeats bit
 * for bit. splits: K ranges (1 but for the partial products). */
int mlsx_int4_grouped_few_rows(int64_t M_total, int E, int64_t K, int group, int splits);

/* ---------------------------------------------------------------- MoE routing */

/* Top-k of softmax(logits[t]) in fp32, largest first, divided by their sum (train/model.py:
 * 158-162): weights fp32 [tokens][k], experts int64 [tokens][k]. logits: dt [tokens][ld]. At most
 * 256 experts and k = 8 (MLS_ERR_UNSUPPORTED above). */
int mlsx_route_topk(const void* logits, int dt, int64_t ld, int64_t tokens, int E, int k, float* weights,
                    int64_t* experts, mls_stream_t stream);

/* The expert-sorted order of n = tokens * k assignments (kernels/moe_routing.py:116-130), stable:
 * token_of_slot[p] (int32 [n]) the token of sorted row p, seg_off (int32 [E + 1]) the segments,
 * pos[i] (int64 [n]) the sorted row of assignment i. An id outside [0, E) joins no segment (pos
 * -1; rows past the last segment hold token -1) and sets *bad (1, or 2 where one is negative; 0
 * otherwise), which may be pinned host memory. At most 256 experts and MLSX_ROUTE_MAX
 * assignments. */
#define MLSX_ROUTE_MAX 32768
int mlsx_route_sort(const int64_t* experts, int64_t n, int k, int E, int32_t* token_of_slot, int32_t* seg_off,
                    int64_t* pos, int32_t* bad, mls_stream_t stream);

/* ---------------------------------------------------------------- weight gradient */

/* dw[N][K] = dy[M][N]^T x[M][K], all fp32 row-major (kernels/autograd_ops.py:132), as bf16 parts
 * that add up to the fp32 values. M >= 1. The 16-byte aligned workspace holds
 * mlsx_dw_fp32_workspace bytes (0: sizes it does not take, MLS_ERR_UNSUPPORTED). */
int64_t mlsx_dw_fp32_workspace(int64_t M, int64_t N, int64_t K);
/* 1 where mlsx_dw_fp32 is faster than an fp32 library product and its workspace at most 4 GiB. */
int mlsx_dw_fp32_pays(int64_t M, int64_t N, int64_t K);
int mlsx_dw_fp32(const float* dy, int64_t lddy, const float* x, int64_t ldx, float* dw, int64_t lddw, int64_t M,
                 int64_t N, int64_t K, void* ws, int64_t ws_bytes, mls_stream_t stream);

/* ---------------------------------------------------------------- FP8 training */

/* The fp8 operands of train/fp8.py:62-95 padded for the K-contiguous GEMM:
 * out[r][c] = fp8(x[r][c] / scale[r]) as [rows][Cp], and, when out_t is not null, its
 * transpose [cols][Rp], where Cp and Rp are cols and rows rounded up to 64 and every
 * padding byte is 0 (a zero in both formats). e5m2: 1 for e5m2, 0 for e4m3. e4m3 NaN codes
 * are written as zeros into a copy whose reduction axis is padded (cols % 64 != 0: out;
 * rows % 64 != 0: out_t): mls_fp8_gemm decodes them to 0 at such a K
 * (kernels/fp8_matmul.py:46). out, out_t: 16-byte aligned. */
int mlsx_fp8_encode_pad(int e5m2, const void* x, int x_dt, int64_t rows, int64_t cols, int64_t ldx, float scale,
                        const float* scale_ptr, int64_t scale_stride, uint8_t* out, uint8_t* out_t,
                        mls_stream_t stream);

/* max |x| of n contiguous values in two steps (train/fp8.py:33-48, 86-87: the amax behind
 * a per-tensor scale; NaN wins over every number, as in torch's amax). mlsx_absmax_parts
 * writes MLSX_ABSMAX_PARTS partial maxima; mlsx_absmax_scales takes those of `tensors`
 * tensors one after another and writes amax[t] and scale[t] = max(amax[t] / fp8_max, 1e-12)
 * (one IEEE division; a NaN stays). */
#define MLSX_ABSMAX_PARTS 1024
int mlsx_absmax_parts(const void* x, int x_dt, int64_t n, float* parts, mls_stream_t stream);
int mlsx_absmax_scales(const float* parts, int tensors, float fp8_max, float* amax, float* scale,
                       mls_stream_t stream);

#ifdef __cplusplus
}
#endif

#endif /* MLS_EXT_H */
