// Host launchers of the VAEChunkedMHA kernels (mha_kernels.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace s2 {

// rows of x (element type kind: 0 fp32, 1 bf16, 2 fp16; row width qdim) ->
// bf16 xp [rows_padded][qdim], zero rows from `rows` on
hipError_t launch_mha_stage(const void* x, int kind, int rows, int rows_padded, int qdim,
                            uint16_t* xp, hipStream_t stream);
// out[i] = bf16(w[i] * scale), i < n
hipError_t launch_mha_weight(const float* w, long n, float scale, uint16_t* out,
                             hipStream_t stream);
// out[i] = b[i] * scale, i < n
hipError_t launch_mha_bias(const float* b, int n, float scale, float* out, hipStream_t stream);
// P[r][c] = softmax over c < cols of S[r] (row stride ld_s), bf16, row
// stride ld_p, zero for cols <= c < ld_p; with a gate, only when *gate != 0
hipError_t launch_mha_softmax(const float* s, long ld_s, int rows, int cols, int ld_p,
                              uint16_t* p, const int* gate, hipStream_t stream);
// The exponentials' reference of each row of q k^T (bf16 rows of width d and
// pitch ld, multiples of 8): ref[0, pitch), pitch >= rows a multiple of 256,
// and *general = 1 when it does not cover every row or the values vt [d][lp]
// (rows rounded up to 64; rows >= 64), else 0; stats: 3 * pitch floats of
// scratch, 16-byte aligned
hipError_t launch_mha_reference(const uint16_t* q, const uint16_t* k, int ld, const uint16_t* vt,
                                int lp, int rows, int d, int pitch, float* stats, float* ref,
                                int* general, hipStream_t stream);
// scale[0, pitch): 1 / sum over parts of sums[part][row], or 1 when *general;
// pitch % 64 == 0
hipError_t launch_mha_row_scale(const float* sums, int parts, int pitch, const int* general,
                                float* scale, int rows, hipStream_t stream);
// oh [rows][d] -> columns [h*d, (h+1)*d) of o [rows][embed]
hipError_t launch_mha_interleave(const uint16_t* oh, int rows, int d, int embed, int h,
                                 uint16_t* o, hipStream_t stream);

}  // namespace s2
