// lq_linear: y[M, N] = x[M, K] . W[N, K]^T, dispatch over the kernels.
#include "common.h"

int lq_gemm_generic(const void* x, const void* w, void* out, int in_dtype, int out_dtype, int M,
                    int N, int K, int lda, int ldw, int ldc, hipStream_t stream);
bool lq_gemm_mfma_accepts(const void* x, const void* w, int in_dtype, int K, int lda, int ldw);
int lq_gemm_mfma(const void* x, const void* w, void* out, int out_dtype, int M, int N, int K, int lda,
                 int ldw, int ldc, int epilogue, int splits, long long split_stride, int packed, hipStream_t stream);
bool lq_gemm_packable(int N, int K);
int lq_gemm_mfma_splits(int M, int N, int K);
int lq_gemm_narrow_splits(int M, int N, int K);
bool lq_gemm_few_and_narrow(int M, int N, int K);
int lq_gemm_fused_parts(int M, int N, int K);
int lq_gemm_residual(const void* act, const void* w, float* x, float* sq_out, const float* gain, void* scaled,
                     int ld_scaled, int M, int N, int K, int lda, int ldw, int ldx, int packed, hipStream_t stream);
int lq_gemm_scaled(const void* h, int ldh, const float* sq_parts, int n_parts, int width, float eps, const void* w,
                   void* out, int out_dtype, int M, int N, int K, int ldw, int ldc, int swiglu, int packed,
                   hipStream_t stream);

// In how many shares of K lq_linear wants to compute this product (1: whole).  With s > 1 shares the
// caller passes an output of s pieces, `split_stride` elements apart; their sum is the product, and
// whoever consumes it adds the pieces in ascending order.
extern "C" int lq_linear_splits(int in_dtype, int M, int N, int K, int force_generic) {
  if (force_generic || in_dtype != LQ_BF16 || K % 8 != 0) return 1;
  return lq_gemm_mfma_splits(M, N, K);
}

// The same for a caller that adds the pieces up right away, by a kernel of its own: a few rows of a weight with few rows
// and a long K are then shared out as well.
extern "C" int lq_linear_narrow_splits(int in_dtype, int M, int N, int K, int force_generic) {
  const int usual = lq_linear_splits(in_dtype, M, N, K, force_generic);
  if (usual > 1 || force_generic || in_dtype != LQ_BF16 || K % 8 != 0) return usual;
  return lq_gemm_narrow_splits(M, N, K);
}

// Whether that caller is better off without pieces: at most 8 rows, whose kernels share K over the waves of a block, up to four pieces.
// Microseconds in pieces with the launch that adds them up, and whole: 128 x 2 048 in two, 1 row 4.6 and 3.1, 8 rows 5.5 and 4.0; 8
// rows in four of 64 x 4 096 5.7 and 5.4, of 288 x 4 096 6.3 and 5.5; 288 x 8 192 in eight, 1 row 6.5 and 6.9, 8 rows 7.7 and 8.9.
extern "C" int lq_linear_whole(int in_dtype, int M, int N, int K, int force_generic) {
  return !force_generic && in_dtype == LQ_BF16 && K % 8 == 0 && lq_gemm_mfma_splits(M, N, K) <= 1 && lq_gemm_few_and_narrow(M, N, K) &&
         lq_gemm_narrow_splits(M, N, K) <= 4;
}

// Whether a bfloat16 weight [N, K] may be handed to the products packed (lq_pack_weight): only where every
// kernel that can meet it reads that layout.  `w_packed` below says that w is; its ldw is then the whole matrix's K.
extern "C" int lq_weight_packable(int dtype, int N, int K) { return dtype == LQ_BF16 && lq_gemm_packable(N, K); }

extern "C" int lq_linear(const void* x, const void* w, void* out, int in_dtype, int out_dtype,
                         int M, int N, int K, int lda, int ldw, int ldc, int splits, long long split_stride,
                         int force_generic, int w_packed, hipStream_t stream) {
  LQ_REQUIRE(M > 0 && N > 0 && K > 0, "linear: sizes M=%d N=%d K=%d must be positive", M, N, K);
  LQ_REQUIRE(lda >= K && ldw >= K && ldc >= N, "linear: a row stride is smaller than its row");
  LQ_REQUIRE(x && w && out, "linear: null pointer");
  LQ_REQUIRE(splits >= 1 && (splits == 1 || split_stride >= (long long)M * ldc), "linear: bad split arguments");
  // (a packed weight's ldw is the whole matrix's K, a multiple of 64, where w is a run of its columns)
  LQ_REQUIRE(!w_packed || (ldw % 64 == 0 && lq_weight_packable(in_dtype, N, K)), "linear: this weight cannot be packed");
  if (!force_generic && lq_gemm_mfma_accepts(x, w, in_dtype, K, lda, ldw))
    return lq_gemm_mfma(x, w, out, out_dtype, M, N, K, lda, ldw, ldc, 0, splits, split_stride, w_packed, stream);
  LQ_REQUIRE(splits == 1, "linear: only the matrix-core kernels split K");
  LQ_REQUIRE(!w_packed, "linear: only the matrix-core kernels read a packed weight (x must be 16-byte aligned rows)");
  return lq_gemm_generic(x, w, out, in_dtype, out_dtype, M, N, K, lda, ldw, ldc, stream);
}

int lq_gemm_grouped(const void* x, const void* w, void* out, int M, int N, int K, int lda, int ldw, int ldc,
                    const int* counts, int groups, long long w_step, int packed, hipStream_t stream);

// Whether lq_linear_grouped takes weights [N, K] of a mixture of `groups` experts (else: a product an expert).
extern "C" int lq_linear_grouped_supported(int in_dtype, int groups, int N, int K, int force_generic) {
  return !force_generic && in_dtype == LQ_BF16 && groups >= 1 && groups <= 64 && K % 64 == 0 && K >= 512 && N > 0;
}

// out (32-bit) = x . W_i^T for x's rows in runs, counts[i] rows (on the device) for expert i, whose weight lies i * w_step
// entries behind the first's.  Rows of x beyond the counts' sum are not read, and their rows of out not written.
extern "C" int lq_linear_grouped(const void* x, const void* w, void* out, int in_dtype, int M, int N, int K, int lda, int ldw,
                                 int ldc, const int* counts, int groups, long long w_step, int w_packed, hipStream_t stream) {
  LQ_REQUIRE(M > 0 && lda >= K && ldw >= K && ldc >= N && w_step >= 0, "linear_grouped: bad sizes or strides");
  LQ_REQUIRE(x && w && out && counts, "linear_grouped: null pointer");
  LQ_REQUIRE(lq_linear_grouped_supported(in_dtype, groups, N, K, 0) && lq_gemm_mfma_accepts(x, w, in_dtype, K, lda, ldw) &&
                 w_step % 8 == 0,
             "linear_grouped: %d experts of [%d, %d] are not taken", groups, N, K);
  // (packed rows of one matrix, or packed columns: runs of 64 of them lie 512 entries apart)
  LQ_REQUIRE(!w_packed || (N % 8 == 0 && ldw % 64 == 0 && (ldw == K ? w_step % (8ll * K) == 0 : w_step % 512 == 0)),
             "linear_grouped: these weights are not packed rows in eights or columns in 64s");
  return lq_gemm_grouped(x, w, out, M, N, K, lda, ldw, ldc, counts, groups, w_step, w_packed, stream);
}

// Whether lq_linear_swiglu takes this problem (else: lq_linear into [M, 2I] and lq_swiglu).
extern "C" int lq_linear_swiglu_supported(int in_dtype, int N, int K) {
  return in_dtype == LQ_BF16 && N % 16 == 0 && K % 8 == 0;
}

// out[M, N/2] = silu(gate) * up where [gate | up] = x . W^T and W's N rows hold gate and up rows
// interleaved in groups of 8 (rows 16j..16j+7 gate 8j..8j+7, rows 16j+8..16j+15 up 8j..8j+7).  `act`: 1 the tanh form of
// gelu, 2 relu in silu's place (bfloat16 out).
extern "C" int lq_linear_swiglu(const void* x, const void* w, void* out, int in_dtype, int out_dtype, int M,
                                int N, int K, int lda, int ldw, int ldc, int w_packed, int act, hipStream_t stream) {
  LQ_REQUIRE(act >= 0 && act <= 2 && (act == 0 || out_dtype == LQ_BF16), "linear+swiglu: the gelu and relu forms leave bfloat16");
  LQ_REQUIRE(M > 0 && N > 0 && K > 0, "linear+swiglu: sizes M=%d N=%d K=%d must be positive", M, N, K);
  LQ_REQUIRE(lda >= K && ldw >= K && ldc >= N / 2, "linear+swiglu: a row stride is smaller than its row");
  LQ_REQUIRE(x && w && out, "linear+swiglu: null pointer");
  LQ_REQUIRE(lq_linear_swiglu_supported(in_dtype, N, K) && lq_gemm_mfma_accepts(x, w, in_dtype, K, lda, ldw),
             "linear+swiglu: needs bfloat16, 16-byte aligned rows, K %% 8 == 0 and N %% 16 == 0");
  LQ_REQUIRE(!w_packed || (ldw == K && lq_weight_packable(in_dtype, N, K)), "linear+swiglu: this weight cannot be packed");
  return lq_gemm_mfma(x, w, out, out_dtype, M, N, K, lda, ldw, ldc, act == 2 ? 4 : act == 1 ? 3 : 1, 1, 0, w_packed, stream);
}

int lq_gemm_unit(const void* x, const void* w, void* out, int M, int N, int K, int lda, int ldw, int ldc, const float* bias, int tail,
                 int act, int packed, hipStream_t stream);

// Whether lq_linear_unit takes weights [N, K]: with a bias (gated) for any number of rows, without one for up to 16.
extern "C" int lq_linear_unit_supported(int in_dtype, int rows, int N, int K, int biased, int force_generic) {
  return !force_generic && in_dtype == LQ_BF16 && rows >= 1 && lq_gemm_packable(N, K) && (biased ? N % 16 == 0 : rows <= 16);
}

// `bias` [N]: out[M, N / 2 + tail] = silu(gate + its bias) (up + its bias) where W's rows, and the bias' entries, are gate's and up's interleaved
// in groups of 8 as lq_linear_swiglu has them; the last `tail` columns become a one and zeros.  No bias: out[M, N] = act(x . W^T), `act`
// 1 silu, 2 relu, 3 and 4 the tanh and the exact form of gelu, 5 the square of relu.  bfloat16 in and out, 32-bit in between.
extern "C" int lq_linear_unit(const void* x, const void* w, void* out, int M, int N, int K, int lda, int ldw, int ldc, const float* bias,
                              int tail, int act, int w_packed, hipStream_t stream) {
  LQ_REQUIRE(x && w && out, "linear_unit: null pointer");
  LQ_REQUIRE(lq_linear_unit_supported(LQ_BF16, M, N, K, bias != nullptr, 0), "linear_unit: M=%d N=%d K=%d is not taken", M, N, K);
  LQ_REQUIRE(tail >= 0 && (bias != nullptr ? act == 1 && (uintptr_t)bias % 16 == 0 : tail == 0 && act >= 1 && act <= 5), "linear_unit: bad bias, tail or activation");
  LQ_REQUIRE(lda >= K && ldw >= K && ldc >= (bias != nullptr ? N / 2 + tail : N), "linear_unit: a row stride is smaller than its row");
  LQ_REQUIRE(lq_gemm_mfma_accepts(x, w, LQ_BF16, K, lda, ldw), "linear_unit: operands are not aligned");
  LQ_REQUIRE(!w_packed || ldw == K, "linear_unit: a packed weight is whole");
  return lq_gemm_unit(x, w, out, M, N, K, lda, ldw, ldc, bias, tail, act, w_packed, stream);
}

// ------------------------------------------------------------------ the products around a norm (decoding)
// A pre-norm block's x += act . w^T; out = rmsnorm(x) . w2^T in two kernels instead of three.  The first
// adds into the float32 stream, leaves per-row sums of squares, a part per block, and the rows times the
// norm's gain in bfloat16; the second multiplies those rows with w2 and scales each output row by
// 1 / sqrt(mean(x^2) + eps) from the parts.  (The rows are rounded to bfloat16 before the division by the
// root mean square, not after: the same relative rounding.)  lq_linear_fused_parts: the number of parts
// the first leaves for [M, K] x [N, K]^T, or 0 when these kernels do not take the size (then the caller
// uses the separate kernels).
extern "C" int lq_linear_fused_parts(int dtype, int M, int N, int K) {
  if (dtype != LQ_BF16) return 0;
  return lq_gemm_fused_parts(M, N, K);
}

extern "C" int lq_linear_residual(const void* act, const void* w, float* x, float* sq_out, const float* gain,
                                  void* scaled, int ld_scaled, int dtype, int M, int N, int K, int lda, int ldw,
                                  int ldx, int parts, int w_packed, hipStream_t stream) {
  LQ_REQUIRE(act && w && x && sq_out, "linear_residual: null pointer");
  LQ_REQUIRE((gain == nullptr) == (scaled == nullptr) && (scaled == nullptr || ld_scaled >= N),
             "linear_residual: a gain and a place for the scaled rows come together");
  LQ_REQUIRE(lda >= K && ldw >= K && ldx >= N, "linear_residual: a row stride is smaller than its row");
  LQ_REQUIRE(parts > 0 && parts == lq_linear_fused_parts(dtype, M, N, K),
             "linear_residual: M=%d N=%d K=%d leaves %d parts, not %d", M, N, K, lq_linear_fused_parts(dtype, M, N, K),
             parts);
  LQ_REQUIRE(lq_gemm_mfma_accepts(act, w, dtype, K, lda, ldw), "linear_residual: operands are not aligned");
  LQ_REQUIRE(!w_packed || (ldw == K && lq_weight_packable(dtype, N, K)), "linear_residual: this weight cannot be packed");
  return lq_gemm_residual(act, w, x, sq_out, gain, scaled, ld_scaled, M, N, K, lda, ldw, ldx, w_packed, stream);
}

extern "C" int lq_linear_scaled(const void* h, int ldh, const float* sq_parts, int parts, float eps, const void* w,
                                void* out, int dtype, int out_dtype, int M, int N, int K, int ldw, int ldc,
                                int swiglu, int w_packed, hipStream_t stream) {
  LQ_REQUIRE(h && sq_parts && w && out, "linear_scaled: null pointer");
  LQ_REQUIRE(parts > 0 && ldh >= K && ldw >= K && ldc >= (swiglu ? N / 2 : N), "linear_scaled: bad sizes");
  LQ_REQUIRE(lq_linear_fused_parts(dtype, M, N, K) > 0 && (!swiglu || N % 16 == 0),
             "linear_scaled: M=%d N=%d K=%d is not taken", M, N, K);
  LQ_REQUIRE(lq_gemm_mfma_accepts(h, w, dtype, K, ldh, ldw), "linear_scaled: operands are not aligned");
  LQ_REQUIRE(!w_packed || (ldw == K && lq_weight_packable(dtype, N, K)), "linear_scaled: this weight cannot be packed");
  return lq_gemm_scaled(h, ldh, sq_parts, parts, K, eps, w, out, out_dtype, M, N, K, ldw, ldc, swiglu, w_packed, stream);
}
