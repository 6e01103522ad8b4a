// Prefill path (token counts above the decode kernel's 16) on the tile layout.
#pragma once

#include "nq_common.h"
#include "nq_decode.h"

namespace nq {

// Workspace bytes of a call above the decode kernel's token counts, the general
// path's fp32 rank intermediate among them (all of it without tiles).
int64_t prefill_scratch_bytes(const nq_linear_desc* d, int64_t tokens);

// The size that nq_linear_static's limit is held against (at most
// prefill_scratch_bytes, and at least 1 / kPrefillOverReserve of it).
int64_t prefill_reserved_bytes(const nq_linear_desc* d, int64_t tokens);
constexpr int kPrefillOverReserve = 3;

// The whole call's reserved bytes (nq_linear_workspace_bytes with
// prefill_reserved_bytes in place of prefill_scratch_bytes), or -1.
int64_t linear_reserved_bytes(const nq_linear_desc* d, int64_t tokens);

// True when desc->tiles is set and tokens exceed the decode kernel's range.
bool prefill_path_applies(const nq_linear_desc* d, int64_t tokens);

// Launch prep -> GEMM(V) -> GEMM(U); scratch is prefill_scratch_bytes bytes.
int launch_prefill(const nq_linear_desc* d, const void* x, int x_dtype, int64_t tokens, void* y, int y_dtype,
                   void* scratch, hipStream_t stream);

// The same for 1..8 linears with one token count: one launch per phase (row
// passes, GEMM 1, its reductions, GEMM 2, its reductions) for all members;
// scratch[i] is prefill_scratch_bytes(descs[i], tokens) bytes.
int launch_prefill_batch(const nq_linear_desc* const* descs, int count, const void* const* xs, int x_dtype,
                         int64_t tokens, void* const* ys, int y_dtype, void* const* scratch, hipStream_t stream);

}  // namespace nq
