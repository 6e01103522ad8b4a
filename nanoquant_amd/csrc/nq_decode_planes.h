// Decode calls of several tokens on fp6 planes (nq_decode_planes.hip).
#pragma once

#include "nq_common.h"
#include "nq_decode.h"

namespace nq {

// Scratch bytes one linear needs: less than decode_scratch_bytes (60.5 bytes a
// column of x and of the rank against 64), which callers size buffers by.
int64_t decode_planes_bytes(const nq_linear_desc* d);

// Planes of x * s_in, GEMM 1, GEMM 2 for 1..8 linears sharing the token count
// (at most 16) and dtypes; scratch[i] (16-byte aligned) holds
// decode_planes_bytes(descs[i]). The caller checked the descriptions.
int launch_decode_planes(const nq_linear_desc* const* descs, int count, const void* const* xs, int x_dtype,
                         int64_t tokens, void* const* ys, int y_dtype, void* const* scratch, hipStream_t stream);

}  // namespace nq
