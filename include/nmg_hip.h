/*
 * nmg_hip.h -- C ABI of libnmg_hip.so: the grouped n:m ("nmg") sparse path for MI355X (gfx950).
 *
 * Conventions
 *   - Every pointer named d_* is a device pointer owned by the caller; outputs are allocated by
 *     the caller and fully overwritten.  The library allocates no device memory.  The only
 *     device state it owns is a small file-scope table of pattern orders (one 8 KiB slot per
 *     distinct (n, m), filled on first use with a blocking copy).
 *   - `stream` is a hipStream_t passed as void* (NULL = the default stream).  Calls are
 *     stream-ordered and return without waiting for the GPU.
 *   - Return value: 0 on success, otherwise one of NMG_ERR_*; nmg_last_error() gives a message
 *     for the calling thread.  Nothing aborts the process.
 *   - dtype codes: NMG_F32, NMG_F16, NMG_BF16, NMG_F64 (sparsify / to_dense / gather only).
 *
 * Each entry point cites the reference interface it replaces (paths relative to the reference
 * repository root).  In the reference these are per-shape `extern "C" func(...)` symbols that
 * are generated, compiled and dlopen'ed at run time; here shapes are run-time arguments.
 */
#ifndef NMG_HIP_H
#define NMG_HIP_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

enum { NMG_F32 = 0, NMG_F16 = 1, NMG_BF16 = 2, NMG_F64 = 3 };

enum {
    NMG_OK = 0,
    NMG_ERR_ARG = 1,         /* invalid argument (shape, n/m/g, dtype, null pointer) */
    NMG_ERR_UNSUPPORTED = 2, /* valid request the kernels cannot serve (e.g. tile too large for LDS) */
    NMG_ERR_HIP = 3,         /* a HIP runtime call failed; see nmg_last_error() */
    NMG_ERR_NO_DEVICE = 4
};

/* spmm kernel selection (for measurement); NMG_KERNEL_AUTO picks by shape. */
enum {
    NMG_KERNEL_AUTO = 0,
    NMG_KERNEL_MFMA = 1,   /* dense MFMA on tiles decompressed into LDS */
    NMG_KERNEL_SMFMAC = 2, /* sparse MFMA (2:4-compatible patterns, reduction along the sparse dim) */
    NMG_KERNEL_SKINNY = 3  /* bandwidth-bound wavefront-reduction kernel for few tokens */
};

int nmg_version(void);
const char *nmg_last_error(void);

/* Pattern order table of make_n_m(n, m): out[C(m,n)][n] (host memory).  Returns C(m,n) or -1.
 * Replaces: src/sten/grouped_nm/grouped_nm_tensor.py:37-50 (make_n_m), whose result the
 * reference pastes into every generated kernel as `nnz_order` (:254, :741, :814). */
int64_t nmg_order(int n, int m, int8_t *out);
int64_t nmg_chunk(int n, int m);

/* Geometry of a strided view that is read or written tile by tile.
 * Logical view: [batch, G, S] (group dim extent G, sparse dim extent S), element strides given
 * in elements.  Tile t = (b * num_chunks + kc) * num_blocks + mb covers group indices
 * kc*c*g .. +c*g and sparse indices mb*m .. +m; indices beyond G / S read as zero and are not
 * written.  The reference builds the same tiles with pad -> reshape -> permute -> reshape on
 * the host (grouped_nm_tensor.py:701-710, layout from :71-217); the "merged" [outer,c,g,m]
 * tensor it hands to its kernels is the special case batch=outer, G=c*g, S=m. */
typedef struct nmg_view {
    int64_t batch, G, S;
    int64_t stride_b, stride_g, stride_s;
} nmg_view;

/* Dense -> grouped n:m.  val: [outer, c, g, n] (dtype of the input), idx: [outer, c, g] int16,
 * outer = batch * ceil(G/(c*g)) * ceil(S/m).  Bit-exact with the reference CPU sparsifier.
 * Replaces: `extern "C" void func(T* dense, T* sparse, int16_t* idx)` generated by
 * grouped_nm_tensor.py:244-299 (driver :636-685). */
int nmg_sparsify(const void *d_dense, const nmg_view *view, void *d_val, int16_t *d_idx, int n,
                 int m, int g, int dtype, void *stream);

/* Grouped n:m -> dense (scatter through idx and the pattern order); every element of the view
 * is written (zeros where nothing is kept).
 * Replaces: `extern "C" void func(T* sparse, T* dense, int16_t* idx)` generated by
 * grouped_nm_tensor.py:735-760 (CPU) / :800-839 (CUDA), driver :848-874. */
int nmg_to_dense(const void *d_val, const int16_t *d_idx, void *d_dense, const nmg_view *view,
                 int n, int m, int g, int dtype, void *stream);

/* Re-compress a dense tensor with an existing pattern: val[t,s,j] = dense[idx[t,s], order[s/g][j]].
 * This is the SameFormatSparsifier implementation for the format.
 * Replaces: the intended behaviour of GroupedNMTensor.clone_layout, grouped_nm_tensor.py:908-951
 * (disabled upstream). */
int nmg_gather(const void *d_dense, const nmg_view *view, const int16_t *d_idx, void *d_val, int n,
               int m, int g, int dtype, void *stream);

/* ---- matmul operand ("rowpack"): a GPU-private re-ordering of val/idx for a 2-D weight.
 * For each line q of the group dim and each block b of the sparse dim: the n kept values and
 * the pattern number.  pk_val: [G, nb, n] (dtype), pk_pat: [G, nb] uint8 (C(m,n) <= 256) or
 * uint16.  Derived from the canonical val/idx, which stay the interchange format.
 * No counterpart in the reference (its CPU kernel consumes val/idx directly,
 * dace_gnm_mult.py:200-213). */
int64_t nmg_rowpack_pat_bytes(int n, int m); /* 1 or 2 */
int nmg_rowpack(const void *d_val, const int16_t *d_idx, int64_t G, int64_t S, void *d_pk_val,
                void *d_pk_pat, int n, int m, int g, int dtype, void *stream);

/* Dense copy of a 2-D weight from its rowpack operand: out[q, s] (transpose = 0, G rows, ld_out >=
 * S) or out[s, q] (transpose = 1, S rows, ld_out >= G); dropped positions are written as zeros.
 * Same result as nmg_to_dense on the canonical val/idx, with contiguous reads and writes.
 * Replaces: grouped_n_m_to_dense for a 2-D weight, grouped_nm_tensor.py:848-874. */
int nmg_rowpack_expand(const void *d_pk_val, const void *d_pk_pat, int64_t G, int64_t S, void *d_out,
                       int64_t ld_out, int transpose, int n, int m, int dtype, void *stream);

/* Y[T, G] = X[T, S] * W2^T      (reduce_sparse = 1)   W2 = the [G, S] weight view
 * Y[T, S] = X[T, G] * W2        (reduce_sparse = 0)
 * X, Y row-major with leading dimensions ldx, ldy (elements).  X/Y/pk_val share `dtype`
 * (F32, F16 or BF16); accumulation is fp32, the bias
 * included, and a 16-bit result is rounded once (so in every product below).  `bias` (length = output features, same dtype) may be
 * NULL.  `kernel` is one of NMG_KERNEL_*.
 * Replaces: `__program_<name>(state, A_idx, A_val, B, C, groups)` produced by
 * dace_gnm_mult.py:572-1007 and called from sten_impls.py:111-138, plus the bias add of
 * sten_impls.py:172-173. */
int nmg_spmm(const void *d_pk_val, const void *d_pk_pat, int64_t G, int64_t S, const void *d_x,
             int64_t ldx, void *d_y, int64_t ldy, const void *d_bias, int64_t T, int reduce_sparse,
             int n, int m, int dtype, int kernel, void *stream);

/* ---- sparse-matrix-core operand ("fragpack") for 2-of-4 compatible patterns (2:4, 1:4, 1:8,
 * 2:8, ...) when the reduction runs along the sparse dim: the kept values and their 2-bit
 * positions in the register order of V_SMFMAC_F32_32X32X32, for blocks of 32 lines x 32 dense
 * positions.  fp_val: val_elems 16-bit elements, fp_idx: idx_words uint32 (sizes from
 * nmg_fragpack_sizes; lines padded to 32, positions to 64, with zeros).  Built from the rowpack
 * operand.  No counterpart in the reference. */
int nmg_fragpack_supported(int n, int m); /* 1 if every aligned group of 4 keeps <= 2 values */
int nmg_fragpack_sizes(int64_t G, int64_t S, int64_t *val_elems, int64_t *idx_words);
int nmg_fragpack(const void *d_pk_val, const void *d_pk_pat, int64_t G, int64_t S, void *d_fp_val,
                 void *d_fp_idx, int n, int m, int dtype, void *stream);

/* Both operands from the canonical val/idx in one pass (same results as nmg_rowpack followed by
 * nmg_fragpack, bit for bit).  d_fp_val / d_fp_idx may be NULL: rowpack only (any n:m, f32 too).
 * No counterpart in the reference. */
int nmg_pack_operands(const void *d_val, const int16_t *d_idx, int64_t G, int64_t S, void *d_pk_val,
                      void *d_pk_pat, void *d_fp_val, void *d_fp_idx, int n, int m, int g, int dtype,
                      void *stream);

/* Y[T, M] = X[T, K] * W^T (+ bias) on the sparse matrix cores; W given as its fragpack operand
 * (M = lines of the group dim, K = extent of the sparse dim).  dtype F16 or BF16, fp32
 * accumulation.  X must be 16-byte aligned with K and ldx multiples of 8.  `variant` selects the
 * kernel: 0 = register-prefetch kernel, workgroup tile 256 lines x 128 tokens (any K);
 * 5 = bandwidth-bound streaming kernel for T <= 16, and up to 32 where K % 128 == 0 (one workgroup
 * per 32 lines, K split over its wavefronts; above that the call runs variant 0); 6 = the weight fragments go from global memory straight into the registers of the
 * wavefront that multiplies them and only the activations pass through LDS, by DMA (4 wavefronts
 * stacked on the lines, 256 x 128); 8 = 6 with a 256 x 256 tile; -1 = the default for large
 * batches (6).  6 and 8 need K % 64 == 0 and X below 2 GiB, else variant 0 runs.
 * Replaces the same reference interface as nmg_spmm (sten_impls.py:111-138, :172-173). */
int nmg_spmm_smfmac(const void *d_fp_val, const void *d_fp_idx, int64_t M, int64_t K,
                    const void *d_x, int64_t ldx, void *d_y, int64_t ldy, const void *d_bias,
                    int64_t T, int dtype, int variant, void *stream);

/* The product with both dense operands transposed, C[M, T] = W * B (+ bias[M] added to every
 * column), B [K, T] and C [M, T] row-major with leading dimensions ldb / ldc: what
 * torch.mm(W, B) asks for, without a transposing copy on either side (the tile of B is fetched as
 * it lies in memory and transposed by the LDS transpose reads of gfx950).  Large-batch kernel,
 * 128 lines x 128 columns per workgroup, 256 x 128 or 256 x 256 by the extents, any T; K % 64 == 0, ldb % 8 == 0,
 * B 16-byte aligned.  Every row of B is read in whole pieces of 8 columns, the last one too.
 * Replaces: nmg_mult(..., transpose_b=True, transpose_c=True), dace_gnm_mult.py:572-627, whose
 * generated code makes the transposing copies of :813-915. */
int nmg_spmm_smfmac_tt(const void *d_fp_val, const void *d_fp_idx, int64_t M, int64_t K, const void *d_b,
                       int64_t ldb, void *d_c, int64_t ldc, const void *d_bias, int64_t T, int dtype,
                       void *stream);
/* The same result from activations X [T, K] (B transposed beforehand, nmg_transpose16): C [M, T] = W * X^T. */
int nmg_spmm_smfmac_ct(const void *d_fp_val, const void *d_fp_idx, int64_t M, int64_t K, const void *d_x, int64_t ldx,
                       void *d_c, int64_t ldc, const void *d_bias, int64_t T, int dtype, void *stream);

/* The same product with the reduction cut into slices, for token counts between the decode shapes
 * and a batch that fills the chip (a 4096 x 11008 weight x 17..512 tokens is 16..64 tiles of
 * 256 x 128 on 256 CUs, each walking the whole reduction).  Slice s of a tile sums its share of
 * K in single precision into workspace[s][token][feature]; a second kernel adds the slices in
 * order (+ bias) and rounds once.  nmg_splitk_plan gives the number of slices for a product of M
 * outputs, reduction K and T tokens (1 = do not split) and the workspace in bytes; the workspace
 * is caller-owned device memory, 16-byte aligned, written and read inside the call only.
 * nmg_smfmac_plan gives the number that is fastest with the tiles that the kernels choose for it (1024 x 1024 x 1024 tokens: 16.8 us
 * in two slices, 9.7 whole); nmg_splitk_plan brings the workgroups of 256 x 128 towards one per CU.
 * slices <= 1 is the unsplit entry point with its default tile.  K % 64 == 0, T > 16.
 * nmg_spmm_densefrag_splitk (declared with the densefrag entry points) is the same for the
 * dense-matrix-core route, its slices from nmg_densefrag_plan.
 * No counterpart in the reference (sten_impls.py:44-140 calls one generated loop nest). */
int nmg_splitk_plan(int64_t M, int64_t K, int64_t T, int *slices, int64_t *workspace_bytes);
int nmg_smfmac_plan(int64_t M, int64_t K, int64_t T, int *slices, int64_t *workspace_bytes);
int nmg_spmm_smfmac_splitk(const void *d_fp_val, const void *d_fp_idx, int64_t M, int64_t K,
                           const void *d_x, int64_t ldx, void *d_y, int64_t ldy, const void *d_bias,
                           int64_t T, int dtype, int slices, void *d_workspace, int64_t workspace_bytes,
                           void *stream);

/* The product for a K that is a multiple of 8 only, activations as they lie: pieces of the last step of 64 that lie behind the row
 * are cleared on the way in.  `slices` and the workspace (none for one slice) are those of nmg_smfmac_plan for K in whole steps of 64.
 * nmg_spmm_densefrag_ragged is the same for the dense-matrix-core route and nmg_densefrag_plan. */
int nmg_spmm_smfmac_ragged(const void *d_fp_val, const void *d_fp_idx, int64_t M, int64_t K, const void *d_x, int64_t ldx, void *d_y,
                           int64_t ldy, const void *d_bias, int64_t T, int dtype, int slices, void *d_workspace,
                           int64_t workspace_bytes, void *stream);

/* nmg_spmm_smfmac_splitk without the workspace argument, for callers that cannot allocate device
 * memory or carry a workspace around: code under HIP graph capture, tight serving loops, harnesses
 * that forbid hipMalloc.  The partial sums go to a 32 MiB array inside the library (one copy per
 * GPU, held until the process ends); the call allocates nothing, on the device or through any
 * library.  A product whose partial sums (slices * T * ceil(M/256)*256 * 4 bytes) exceed
 * nmg_noalloc_scratch_bytes() is refused with NMG_ERR_UNSUPPORTED.  All calls on one GPU share that
 * GPU's array: calls that overlap there (two streams) race; calls in stream order may follow each
 * other in any sizes.  nmg_noalloc_prepare() looks the array up on the current device ahead of
 * time (optional; the first call on a device does it otherwise -- do it before a graph capture).
 * This entry point has no counterpart in the reference. */
int64_t nmg_noalloc_scratch_bytes(void);
int nmg_noalloc_prepare(void);
int nmg_spmm_smfmac_splitk_noalloc(const void *d_fp_val, const void *d_fp_idx, int64_t M, int64_t K,
                                   const void *d_x, int64_t ldx, void *d_y, int64_t ldy, const void *d_bias,
                                   int64_t T, int dtype, int slices, void *stream);

/* Plain dense product Y[T, O] = X[T, K] * A[O, K]^T (+ bias), both operands row-major with the
 * reduction contiguous, on the same pipelined dense-MFMA kernel as nmg_spmm.  It is the second
 * half of the "expand, then multiply" route: nmg_to_dense writes the weight (or its transpose,
 * through the strides of nmg_view) into caller-owned scratch, nmg_gemm_nt multiplies.  Used for
 * the transposed product of the backward pass (reduction along the group dim) and for n:m
 * patterns the sparse matrix cores cannot take, where it runs at the dense library's speed.
 * dtype F16 / BF16: K % 64 == 0, rows 16-byte aligned, operands < 2 GiB.
 * dtype F32: any K > 0 and any row pitch, on V_MFMA_F32_32X32X2_F32 or, products of many tiles, on the
 * bf16 matrix cores with every number in three parts (no larger an error against 64 bits, for numbers of
 * any size; what operands beyond 2^104 or sums beyond 2^80 are part of is computed on the fp32 instruction);
 * nmg_gemm_nn and nmg_gemm_tn too.  It is what single-precision products run on, after nmg_to_dense.
 * No counterpart in the reference (its nmg path has no backward, sten.py:1690-1693). */
int nmg_gemm_nt(const void *d_a, int64_t lda, const void *d_x, int64_t ldx, void *d_y, int64_t ldy,
                const void *d_bias, int64_t O, int64_t K, int64_t T, int dtype, void *stream);

/* The same single-precision product with the weight-side operand reduction-major:
 * Y[T, O] = X[T, K] * A[K, O] (+ bias[o]).  It is how torch.mm(W_nmg, B) and its gradient with
 * respect to B run in fp32 without transposing copies: X is the expanded weight (or its transpose,
 * both from nmg_to_dense), A is B as it lies in memory, Y is the result as torch.mm lays it
 * out (the reference's transpose_b / transpose_c, dace_gnm_mult.py:572-627).  dtype F32 only; any
 * extents and pitches, 128-bit loads where rows are 16-byte aligned and O % 4 == 0. */
int nmg_gemm_nn(const void *d_a, int64_t lda, const void *d_x, int64_t ldx, void *d_y, int64_t ldy,
                const void *d_bias, int64_t O, int64_t K, int64_t T, int dtype, void *stream);

/* And with both operands reduction-major: Y[T, O] = X[K, T]^T * A[K, O] (+ bias[o]).  The dense
 * weight gradient of a linear layer, grad_W[R, C] = dY[tokens, R]^T * X[tokens, C], from the operands
 * as the backward pass holds them (the training shape of tests/test_training.py:45-72: a dense
 * grad_w beside the sparse forward and grad_input); for fp32 nmg_gather then keeps the entries of
 * the pattern (the compressed gradient of examples/rosa.py:216-221 in the reference's dtype; 16-bit
 * types have the fused nmg_sddmm).  F32: any extents and pitches, 128-bit loads where rows are
 * 16-byte aligned and O % 4 == 0, T % 4 == 0.  F16 / BF16 (the kernel of nmg_sddmm without its
 * mask, fp32 accumulation): O, T and the pitches multiples of 8, 16-byte aligned bases, else
 * NMG_ERR_UNSUPPORTED.  No counterpart in the reference (no backward, sten.py:1690-1693). */
int nmg_gemm_tn(const void *d_a, int64_t lda, const void *d_x, int64_t ldx, void *d_y, int64_t ldy,
                const void *d_bias, int64_t O, int64_t K, int64_t T, int dtype, void *stream);

/* The single-precision product (`form` 0: nmg_gemm_nt, 1: nmg_gemm_nn, 2: nmg_gemm_tn) on the bf16 matrix cores with the reduction cut into
 * slices, which a second kernel adds up in order: products whose results are too few tiles for the chip (1021 x 1999
 * results over 2047: 85 us whole, 66 in two slices).  nmg_gemm_f32_plan gives the number of slices (1: the entry points
 * above) and the bytes of its workspace. */
int nmg_gemm_f32_plan(int64_t lda, int64_t ldx, int64_t O, int64_t K, int64_t T, int form, int *slices, int64_t *workspace_bytes);
int nmg_gemm_f32_splitk(const void *d_a, int64_t lda, const void *d_x, int64_t ldx, void *d_y, int64_t ldy, const void *d_bias,
                        int64_t O, int64_t K, int64_t T, int form, int slices, void *d_workspace, int64_t workspace_bytes,
                        void *stream);

/* dst [dst_rows, dst_cols] = src [rows, cols] in a 16-bit type, zeros beyond the source; any pitches and
 * alignments.  Brings operands into the shape of the matrix-core products (row starts, K steps), or a padded
 * result back.  No counterpart in the reference. */
int nmg_copy_rows16(const void *d_src, int64_t rows, int64_t cols, int64_t ld_src, void *d_dst, int64_t dst_rows,
                    int64_t dst_cols, int64_t ld_dst, void *stream);
/* dst [cols, dst_cols] = src [rows, cols] transposed in a 16-bit type, zeros from `rows` on; dst_cols a multiple of 8. */
int nmg_transpose16(const void *d_src, int64_t rows, int64_t cols, int64_t ld_src, void *d_dst, int64_t dst_cols,
                    int64_t ld_dst, void *stream);
/* y [cols] = sum of the rows of x [rows, cols] (row pitch ld), single-precision sums (f32, f16, bf16). */
int nmg_colsum(const void *d_x, int64_t rows, int64_t cols, int64_t ld, void *d_y, int dtype, void *stream);

/* ---- "densefrag": the weight expanded into the register order of V_MFMA_F32_32X32X16, for the
 * products the sparse matrix cores cannot do: patterns that do not fit 2-of-4 groups, and the
 * reduction along the group dim (gradient with respect to the activations).
 * densefrag [OB][K/16][64][8] (dtype F16/BF16): outputs O = G lines (transpose = 0) or S positions
 * (transpose = 1), padded to OB*32 = a multiple of 256; reduction K = the other extent, padded
 * with zeros to a multiple of 64; m must be a power of two or three times one (3, 6, 12, 24, 48).  Built from the rowpack operand per call or
 * cached by the caller.  No counterpart in the reference. */
int nmg_densefrag_supported(int n, int m);
int nmg_densefrag_elems(int64_t O, int64_t K, int64_t *elems);
int nmg_densefrag(const void *d_pk_val, const void *d_pk_pat, int64_t G, int64_t S, int transpose,
                  void *d_df, int n, int m, int dtype, void *stream);

/* Y[T, O] = X[T, K] * A^T (+ bias), A given as densefrag.  variant 0 = 256 outputs x 128 tokens
 * per workgroup, 1 = 256 x 256, -1 = the fastest of these, 128 x 128 and the kernel for few tokens for the extents.  X must be
 * 16-byte aligned with ldx a multiple of 8 and smaller than 2 GiB.
 * Replaces: the forward of sten_impls.py:143-174 for patterns outside 2-of-4, and supplies the
 * grad_input product the reference leaves to the dense fallback (sten.py:1586-1601). */
int nmg_spmm_densefrag(const void *d_df, int64_t O, int64_t K, const void *d_x, int64_t ldx, void *d_y,
                       int64_t ldy, const void *d_bias, int64_t T, int dtype, int variant, void *stream);
/* C[O, T] = A * B (+ bias[o] on row o) for B [K, T] and C as they lie in memory (row pitches ldb,
 * ldc), A given as densefrag: the dense-matrix-core product with both dense operands transposed.
 * K % 64 == 0, ldb % 8 == 0, B 16-byte aligned, ldb < 2^24; tiles and reads of B as nmg_spmm_smfmac_tt.
 * No counterpart in the reference (its operators have no backward): this is the gradient with
 * respect to B of torch.mm(W, B), W^T * grad_out, taken without transposing copies; same
 * transpose_b / transpose_c meaning as dace_gnm_mult.py:572-627. */
int nmg_spmm_densefrag_tt(const void *d_df, int64_t O, int64_t K, const void *d_b, int64_t ldb, void *d_c,
                          int64_t ldc, const void *d_bias, int64_t T, int dtype, void *stream);
/* The same result from activations X [T, K]: C [O, T] = A * X^T. */
int nmg_spmm_densefrag_ct(const void *d_df, int64_t O, int64_t K, const void *d_x, int64_t ldx, void *d_c, int64_t ldc,
                          const void *d_bias, int64_t T, int dtype, void *stream);
/* Few tokens: the same product on a kernel that deals the reduction out inside the workgroups (one launch, no workspace; at most 64
 * tokens) and takes any K that is a multiple of 8.  nmg_densefrag_few: 1 where it is the one to take; nmg_spmm_densefrag with variant -1
 * takes it there by itself, and nmg_densefrag_plan then answers one slice. */
int nmg_densefrag_few(int64_t O, int64_t K, int64_t T);
int nmg_spmm_densefrag_few(const void *d_df, int64_t O, int64_t K, const void *d_x, int64_t ldx, void *d_y, int64_t ldy,
                           const void *d_bias, int64_t T, int dtype, void *stream);

/* nmg_spmm_densefrag with the reduction cut into slices.  nmg_densefrag_plan gives the number of slices for a product of O
 * outputs, reduction K and T tokens (1: nmg_spmm_densefrag as it is) and the bytes of its workspace. */
int nmg_densefrag_plan(int64_t O, int64_t K, int64_t T, int *slices, int64_t *workspace_bytes);
int nmg_spmm_densefrag_splitk(const void *d_df, int64_t O, int64_t K, const void *d_x, int64_t ldx,
                              void *d_y, int64_t ldy, const void *d_bias, int64_t T, int dtype, int slices,
                              void *d_workspace, int64_t workspace_bytes, void *stream);
int nmg_spmm_densefrag_ragged(const void *d_df, int64_t O, int64_t K, const void *d_x, int64_t ldx, void *d_y, int64_t ldy,
                              const void *d_bias, int64_t T, int dtype, int slices, void *d_workspace, int64_t workspace_bytes,
                              void *stream);

/* ---- masked weight gradient, written straight into the `val` layout (no dense [G, S] product
 * is stored): val[t, s, j] = sum over tokens of L[tok, line] * P[tok, position], for the line
 * (group-dim index) and the n kept positions (sparse-dim indices) that slot s of tile t names.
 * L [T, G] and P [T, S] are row-major with leading dimensions ld_lines / ld_pos (elements); for a
 * Linear weight [out, in] that is n:m along `in`, L is the upstream gradient [T, out] and P the
 * activations [T, in].  dtype F16 / BF16 (val has the same type), fp32 accumulation, one rounding.
 * G, S and the leading dimensions must be multiples of 8 and the operands 16-byte aligned.
 * Every element of val is written (padded lines and positions get zeros).
 *
 * d_slot is the slot map of the pattern, the inverse of idx: int16 [ceil(S/m)][Gpad],
 * Gpad = ceil(G/(c*g))*c*g, slot[b][q] = the s with idx[(q/(c*g))*nb + b][s] == q % (c*g).
 * nmg_slotmap builds it from idx (2-D weight); it depends on the pattern only, not on val.
 *
 * The reference has no nmg backward (sten.py:1690-1693 installs a failing one); this is the
 * weight-gradient half of the training step of tests/test_training.py:45-72,98-104
 * (dense grad_w = dY^T X) fused with the same-pattern re-compression that
 * grouped_nm_tensor.py:908-951 (clone_layout) describes; the compressed-gradient registration
 * pattern is examples/rosa.py:216-221,382-386. */
int nmg_slotmap(const int16_t *d_idx, int64_t G, int64_t S, int16_t *d_slot, int n, int m, int g,
                void *stream);
int nmg_sddmm(const void *d_lines, int64_t ld_lines, const void *d_pos, int64_t ld_pos, int64_t T,
              const int16_t *d_slot, int64_t G, int64_t S, void *d_val, int n, int m, int g, int dtype,
              void *stream);
/* The same for any G and S: the rows of both operands are readable, with zeros behind G and S, up to the next
 * multiple of 8. */
int nmg_sddmm_padded(const void *d_lines, int64_t ld_lines, const void *d_pos, int64_t ld_pos, int64_t T,
                     const int16_t *d_slot, int64_t G, int64_t S, void *d_val, int n, int m, int g, int dtype,
                     void *stream);
/* The same with the operands given reduction-contiguous: L^T [G, T] and P^T [S, T] (leading
 * dimensions >= T), as the operands of the weight gradient of torch.mm(W, B) lie in memory
 * (grad_out [R, N] and B [C, N]); T % 8 == 0, any G and S.  Replaces the transposing copies the
 * reference makes around its kernel (dace_gnm_mult.py:813-915). */
int nmg_sddmm_nt(const void *d_lines_t, int64_t ld_lines, const void *d_pos_t, int64_t ld_pos, int64_t T,
                 const int16_t *d_slot, int64_t G, int64_t S, void *d_val, int n, int m, int g, int dtype,
                 void *stream);

/* ---- ungrouped n:m: every block of m consecutive indices of the sparse dim keeps its n largest
 * magnitudes (no constraint across the group dim).  The dense tensor is seen as
 * [outer, S, inner]: the dims before / at / after the sparse dim of a contiguous tensor.
 * val [outer, nb, n, inner] (dtype of the input), idx [outer, nb, n, inner] int64 = position inside
 * the block, nb = ceil(S/m), kept values in descending magnitude (equal magnitudes: lower position
 * first; NaN counts as largest); positions beyond S are zero padding.  m <= 64.
 * nmg_perfect_nm_to_dense writes every element of the dense tensor.
 * Replaces: PerfectNMTensor.from_dense / to_dense, grouped_nm_tensor.py:1010-1065 (pad, reshape,
 * argsort of the magnitudes, gather / scatter with torch operators). */
int nmg_perfect_nm(const void *d_dense, int64_t outer, int64_t S, int64_t inner, void *d_val, int64_t *d_idx,
                   int n, int m, int dtype, void *stream);
int nmg_perfect_nm_to_dense(const void *d_val, const int64_t *d_idx, int64_t outer, int64_t S, int64_t inner,
                            void *d_dense, int n, int m, int dtype, void *stream);

/* ---- few tokens with the reduction along the group dim (F.linear with a weight in the reference's
 * default orientation, n:m blocks along the outputs: sten_impls.py:24-31; the reference kernel
 * gathers g rows of B per pattern there, dace_gnm_mult.py:200-213).
 * Y[T, S] = X[T, G] * W (+ bias) for T <= 16.  The operand ("gpack", nmg_gpack from the rowpack
 * operand, once per weight version; nmg_gpack_bytes gives its size) holds the compressed lines in
 * tiles of 32 lines of the group dim (= the reduction) x 256 outputs, every tile one contiguous run
 * in the order in which the lanes of the kernel take it: the kept values and one pattern number per
 * block (4 bits where the pattern has at most 16 numbers, else 8) -- 1.125 bytes per dense weight
 * at 2:4.  The kernel streams it once, expands the blocks in registers and multiplies on the dense
 * matrix cores; the reduction is cut into slices whose single-precision sums go to the caller's
 * workspace and are added in order by a second kernel.  16-bit types, m = 4 or 8 with n = 1 or 2
 * (nmg_spmm_gstream_supported), G % 8 == 0, ldx % 8 == 0, 16-byte aligned X and operand.
 * nmg_spmm_gstream_plan gives the number of slices and the workspace size in bytes. */
int nmg_spmm_gstream_supported(int n, int m);
int nmg_gpack_bytes(int64_t G, int64_t S, int n, int m, int64_t *bytes);
int nmg_gpack(const void *d_pk_val, const void *d_pk_pat, int64_t G, int64_t S, int n, int m, void *d_gp,
              int dtype, void *stream);
int nmg_spmm_gstream_plan(int64_t G, int64_t S, int64_t T, int n, int m, int *slices, int64_t *ws_bytes);
int nmg_spmm_gstream(const void *d_gp, int64_t G, int64_t S, const void *d_x, int64_t ldx, void *d_y,
                     int64_t ldy, const void *d_bias, int64_t T, int n, int m, int dtype, void *d_ws,
                     int64_t ws_bytes, void *stream);

/* ---- a handful of tokens with the reduction along the group dim at 2:4 (same product and
 * reference as nmg_spmm_gstream above): every workgroup owns 16 outputs over the whole reduction, so
 * the sums never leave it -- one kernel, no workspace -- at the price that every workgroup reads the
 * token rows over the whole reduction.  Y[T, S] = X[T, G] * W (+ bias), T <= 4.  No matrix
 * instruction: per pair of lines one byte permute per output and one two-element dot product per
 * output and token.  The operand ("opack", nmg_opack from the rowpack operand, once per weight
 * version; size from nmg_opack_bytes) holds, per span of 16 outputs and set of 256 lines, the kept
 * values and 4-bit pattern numbers in the order in which the lanes of the kernel fetch them: 1.125
 * bytes per dense weight.  16-bit types, n:m = 2:4 (nmg_spmm_ostream_supported), G % 8 == 0,
 * ldx % 8 == 0, 16-byte aligned X and operand. */
int nmg_spmm_ostream_supported(int n, int m);
int nmg_opack_bytes(int64_t G, int64_t S, int n, int m, int64_t *bytes);
int nmg_opack(const void *d_pk_val, const void *d_pk_pat, int64_t G, int64_t S, int n, int m, void *d_op,
              int dtype, void *stream);
int nmg_spmm_ostream(const void *d_op, int64_t G, int64_t S, const void *d_x, int64_t ldx, void *d_y,
                     int64_t ldy, const void *d_bias, int64_t T, int n, int m, int dtype, void *stream);

/* ---- few tokens on a weight with blocks of 8 along the reduction (1:8, 2:8, 4:8; the reference's
 * kernel walks val / idx with one gathered FMA per kept value, dace_gnm_mult.py:185-253).
 * Y[T, G] = X[T, S] * W^T (+ bias) for T <= 16.  The operand ("lanepack8", nmg_lanepack8 from the
 * rowpack operand, once per weight version: the kept values and one pattern number per block -- 5
 * bits at 1:8 and 2:8, a byte at 4:8 -- in the order in which the lanes of the kernel take them, 32
 * lines x 32 blocks per set; sizes from nmg_lanepack8_sizes in elements / bytes) holds 0.594 bytes
 * per dense weight at 2:8 where the operand of the sparse matrix cores holds 1.125.  One kernel: the
 * operand is streamed once, expanded in registers and multiplied on the dense matrix cores; the
 * wavefronts of a workgroup split the reduction and add their sums in LDS.  16-bit types,
 * S % 256 == 0, ldx % 8 == 0, 16-byte aligned X. */
int nmg_spmm_sstream_supported(int n, int m);
int nmg_lanepack8_sizes(int64_t G, int64_t S, int n, int64_t *val_elems, int64_t *pat_bytes);
int nmg_lanepack8(const void *d_pk_val, const void *d_pk_pat, int64_t G, int64_t S, int n, void *d_lp_val,
                  void *d_lp_pat, int dtype, void *stream);
int nmg_spmm_sstream(const void *d_lp_val, const void *d_lp_pat, int64_t G, int64_t S, const void *d_x,
                     int64_t ldx, void *d_y, int64_t ldy, const void *d_bias, int64_t T, int n, int m,
                     int dtype, void *stream);

/* ---- 2:4 + int4 decode path (the benchmark's "sparse-marlin" configuration).
 * A row-major fp16 weight [M, K] (K % 128 == 0) is pruned to 2:4 along K by magnitude, quantised
 * to symmetric int4 with one fp16 scale per row and 128 positions, and stored in the register
 * order of the sparse matrix cores: B (nibbles), meta (2-bit positions), s (scales); sizes from
 * nmg_w4_sizes (bytes, 32-bit words, fp16 elements).  nmg_w4_linear: Y[T, M] = X[T, K] * W^T (+
 * bias), fp16 in / out, fp32 accumulation, T <= 16.  nmg_w4_to_dense writes the dequantised
 * weight.  Stands where the reference calls marlin.mul_2_4 (tests/test_sparse_marlin.py:95-114);
 * the packing is this library's own, not Sparse-Marlin's. */
int nmg_w4_sizes(int64_t M, int64_t K, int64_t *b_bytes, int64_t *meta_words, int64_t *scales);
int nmg_w4_pack(const void *d_w, int64_t ldw, int64_t M, int64_t K, void *d_B, void *d_meta, void *d_s,
                void *stream);
int nmg_w4_to_dense(const void *d_B, const void *d_meta, const void *d_s, int64_t M, int64_t K,
                    void *d_out, int64_t ldo, void *stream);
int nmg_w4_linear(const void *d_B, const void *d_meta, const void *d_s, int64_t M, int64_t K,
                  const void *d_x, int64_t ldx, void *d_y, int64_t ldy, const void *d_bias, int64_t T,
                  void *stream);

#ifdef __cplusplus
}
#endif
#endif /* NMG_HIP_H */
