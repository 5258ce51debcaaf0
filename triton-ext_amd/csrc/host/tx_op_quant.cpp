// absmax + fp8 quantiser entry points (MX block scales, row-wise scales)
// and their table registrations: the producer step in front of the fp8 and
// MX-scaled GEMMs.
//
// Reference: the MX quantiser is _compute_scale_and_quantize /
// _to_mxfp8_block (extensions/utlx/python/utlx_plugin/mxfp8_utils.py:10-56),
// emitted into TLX kernels; the row-wise form is the per-row absmax scaling
// the fp8 scaled dot consumes (one fp32 scale per row of A / column of B).
#include <algorithm>
#include <climits>
#include <cstdio>

#include "tx_kernel_args.h"
#include "tx_ops.h"

namespace tx {
namespace {

const char *q_name(tx_dtype t) {
  return t == TX_FP8E4M3FN ? "e4m3fn" : (t == TX_FP8E5M2 ? "e5m2" : nullptr);
}
const char *x_name(tx_dtype t) {
  return t == TX_F32 ? "f32" : (t == TX_BF16 ? "bf16" : nullptr);
}

tx_status check_quant(const char *what, const void *x, tx_dtype x_type, int64_t ldx, const void *q,
                      tx_dtype q_type, int64_t ldq, const void *scales, int64_t rows, int64_t K) {
  if (!x_name(x_type))
    return fail(TX_INVALID_ARGUMENT, "%s: x must be fp32 or bf16 (got %d)", what, int(x_type));
  if (!q_name(q_type))
    return fail(TX_INVALID_ARGUMENT, "%s: q must be an fp8 type (got %d)", what, int(q_type));
  if (rows < 0 || K < 0)
    return fail(TX_INVALID_ARGUMENT, "%s: negative size (rows=%lld K=%lld)", what, (long long)rows,
                (long long)K);
  if (rows == 0 || K == 0) return TX_SUCCESS;
  if (!x || !q || !scales) return fail(TX_INVALID_ARGUMENT, "%s: NULL buffer", what);
  if (ldx < K || ldq < K)
    return fail(TX_INVALID_ARGUMENT, "%s: stride smaller than the row (ldx=%lld ldq=%lld)", what,
                (long long)ldx, (long long)ldq);
  const size_t xs = x_type == TX_F32 ? 4 : 2;
  if (!aligned(x, xs)) return fail(TX_INVALID_ARGUMENT, "%s: x not %zu-byte aligned", what, xs);
  return TX_SUCCESS;
}

// The vector paths: 16-byte x loads (fp32: 4, bf16: 8 elements), q stores
// of `qbytes` (4 or 8) bytes, so rows and pitches must keep that alignment.
bool quant_vec(const void *x, tx_dtype x_type, int64_t ldx, const void *q, int64_t ldq,
               int64_t K, int64_t qbytes) {
  const int64_t ve = x_type == TX_F32 ? 4 : 8;
  return aligned(x, 16) && ldx % ve == 0 && K % ve == 0 && aligned(q, size_t(qbytes)) &&
         ldq % qbytes == 0;
}

tx_status quantize_mx(const void *x, tx_dtype x_type, int64_t ldx, void *q, tx_dtype q_type,
                      int64_t ldq, uint8_t *scales, int64_t ld_scales, int64_t rows, int64_t K,
                      tx_stream_t stream) {
  const char *what = "tx_quantize_mx";
  TX_TRY(check_quant(what, x, x_type, ldx, q, q_type, ldq, scales, rows, K));
  if (rows == 0 || K == 0) return TX_SUCCESS;
  if (K % 32)
    return fail(TX_INVALID_ARGUMENT, "%s: K = %lld is not a multiple of the 32-element block", what,
                (long long)K);
  if (ld_scales < K / 32)
    return fail(TX_INVALID_ARGUMENT, "%s: scale stride %lld < K / 32", what, (long long)ld_scales);
  char kname[64];
  std::snprintf(kname, sizeof kname, "tx_quant_mx_%s_%s", q_name(q_type), x_name(x_type));
  hipFunction_t fn;
  TX_TRY(get_kernel(CodeObject::Fp8Codec, kname, &fn));
  // 8-byte q stores at multiples of 8 elements; x loads as for the row path
  tx_quant_args a{x, static_cast<uint8_t *>(q), scales, ldx, ldq, ld_scales, rows, K,
                  quant_vec(x, x_type, ldx, q, ldq, K, 8) ? 1 : 0, 0};
  const int64_t threads = rows * (K / 32) * (x_type == TX_F32 ? 4 : 2);  // lanes per 32-element block
  const int64_t grid = std::min<int64_t>((threads + 255) / 256, int64_t(cu_count()) * 32);
  return launch(fn, unsigned(grid), 1, 256, static_cast<hipStream_t>(stream), &a, sizeof a, kname);
}

// Whether a row gets 1024 threads (kWideRow in fp8_codec.hip) instead of 256:
// from a length on that grows with the rows.  With a workgroup per CU or
// fewer, the row's own latency counts, and 1024 threads hold it in registers in
// fewer steps; past one (two at 256 threads) per CU the larger workgroups wait
// for each other, and pay where 256 threads read a row twice (K > 8192) and most
// of their own second vectors are there.  Time of a launch, 256 -> 1024
// threads, bf16: 16 x 4096 3.16 -> 3.23 us, 256 x 4096 3.33 -> 3.50, 256 x 8192 4.06
// -> 3.95, 256 x 16384 6.9 -> 4.8, 511 x 8192 4.7 -> 5.4, 511 x 8200 5.8 -> 5.7, 600 x
// 12288 7.9 -> 8.3, 1024 x 14336 12.2 -> 11.7, 4096 x 8200 26.0 -> 30.9, 4096 x 11264 34.3
// -> 33.9, 8192 x 16384 104 -> 83; fp32: 256 x 2056 3.60 -> 3.37, 256 x 8192 5.6 -> 4.2,
// 511 x 4096 4.2 -> 4.7, 511 x 8192 5.9 -> 5.6, 600 x 9216 7.7 -> 8.0, 600 x 10240 9.6 ->
// 8.5, 1024 x 9216 12.3 -> 12.0, 4096 x 14336 78 -> 59.
bool quant_row_wide(bool f32, int64_t rows, int64_t K, int64_t cus) {
  int64_t from;
  if (rows <= cus) from = f32 ? 2048 : 6144;
  else if (rows < 2 * cus) from = f32 ? 6144 : 8193;
  else if (rows < (f32 ? 4 : 8) * cus) from = f32 ? 10240 : 13312;
  else from = f32 ? 8193 : 11264;
  return K >= from && K <= 16384;
}

tx_status quantize_rowwise(const void *x, tx_dtype x_type, int64_t ldx, void *q, tx_dtype q_type,
                           int64_t ldq, float *scales, int64_t rows, int64_t K,
                           tx_stream_t stream) {
  const char *what = "tx_quantize_rowwise";
  TX_TRY(check_quant(what, x, x_type, ldx, q, q_type, ldq, scales, rows, K));
  if (rows == 0 || K == 0) return TX_SUCCESS;
  if (!aligned(scales, 4)) return fail(TX_INVALID_ARGUMENT, "%s: scales not 4-byte aligned", what);
  char kname[64];
  const int64_t ve = x_type == TX_F32 ? 4 : 8;  // elements per 16-byte vector
  tx_quant_args a{x, static_cast<uint8_t *>(q), scales, ldx, ldq, 0, rows, K,
                  quant_vec(x, x_type, ldx, q, ldq, K, int(ve)) ? 1 : 0, 0};
  const bool wide = a.vec && K % ve == 0 && quant_row_wide(x_type == TX_F32, rows, K, cu_count());
  std::snprintf(kname, sizeof kname, "tx_quant_row_%s%s_%s", wide ? "wide_" : "", q_name(q_type), x_name(x_type));
  hipFunction_t fn;
  TX_TRY(get_kernel(CodeObject::Fp8Codec, kname, &fn));
  const int64_t grid = std::min<int64_t>(rows, int64_t(cu_count()) * 16);
  return launch(fn, unsigned(grid), 1, wide ? 1024 : 256, static_cast<hipStream_t>(stream), &a, sizeof a, kname);
}

// tx.quantize_mx: {q (result), scales (result), x, rows, K, ldx, ldq, ld_scales, x_type, q_type}
tx_status quant_mx_op(tx_value *v, size_t count, tx_stream_t stream) {
  Operands o{v, count, "tx.quantize_mx"};
  TX_TRY(o.need(10));
  void *q, *s, *x;
  int64_t rows, K, ldx, ldq, lds, xt, qt;
  TX_TRY(o.ptr(0, &q));
  TX_TRY(o.ptr(1, &s));
  TX_TRY(o.ptr(2, &x));
  TX_TRY(o.integer(3, &rows));
  TX_TRY(o.integer(4, &K));
  TX_TRY(o.integer(5, &ldx));
  TX_TRY(o.integer(6, &ldq));
  TX_TRY(o.integer(7, &lds));
  TX_TRY(o.integer(8, &xt));
  TX_TRY(o.integer(9, &qt));
  return quantize_mx(x, tx_dtype(xt), ldx, q, tx_dtype(qt), ldq, static_cast<uint8_t *>(s), lds,
                     rows, K, stream);
}

// tx.quantize_rowwise: {q (result), scales (result), x, rows, K, ldx, ldq, x_type, q_type}
tx_status quant_row_op(tx_value *v, size_t count, tx_stream_t stream) {
  Operands o{v, count, "tx.quantize_rowwise"};
  TX_TRY(o.need(9));
  void *q, *s, *x;
  int64_t rows, K, ldx, ldq, xt, qt;
  TX_TRY(o.ptr(0, &q));
  TX_TRY(o.ptr(1, &s));
  TX_TRY(o.ptr(2, &x));
  TX_TRY(o.integer(3, &rows));
  TX_TRY(o.integer(4, &K));
  TX_TRY(o.integer(5, &ldx));
  TX_TRY(o.integer(6, &ldq));
  TX_TRY(o.integer(7, &xt));
  TX_TRY(o.integer(8, &qt));
  return quantize_rowwise(x, tx_dtype(xt), ldx, q, tx_dtype(qt), ldq, static_cast<float *>(s), rows,
                          K, stream);
}

const bool reg_quant_mx = register_op(
    "tx.quantize_mx", quant_mx_op,
    "q:fp8*(result), scales:e8m0*(result, rows x K/32), x:f32|bf16*, rows, K, ldx, ldq, "
    "ld_scales, x_type:i32, q_type:i32");
const bool reg_quant_row = register_op(
    "tx.quantize_rowwise", quant_row_op,
    "q:fp8*(result), scales:f32*(result, rows), x:f32|bf16*, rows, K, ldx, ldq, x_type:i32, "
    "q_type:i32");

}  // namespace
}  // namespace tx

extern "C" {

TX_API tx_status tx_quantize_mx(const void *x, tx_dtype x_type, int64_t ldx, void *q,
                                tx_dtype q_type, int64_t ldq, uint8_t *scales, int64_t ld_scales,
                                int64_t rows, int64_t K, tx_stream_t stream) {
  tx::clear_error();
  return tx::quantize_mx(x, x_type, ldx, q, q_type, ldq, scales, ld_scales, rows, K, stream);
}

TX_API tx_status tx_quantize_rowwise(const void *x, tx_dtype x_type, int64_t ldx, void *q,
                                     tx_dtype q_type, int64_t ldq, float *scales, int64_t rows,
                                     int64_t K, tx_stream_t stream) {
  tx::clear_error();
  return tx::quantize_rowwise(x, x_type, ldx, q, q_type, ldq, scales, rows, K, stream);
}

}  // extern "C"
