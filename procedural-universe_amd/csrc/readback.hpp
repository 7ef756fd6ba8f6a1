// Read-back of float4 state records as packed (x, y, z) floats, shared by the
// single-system handle and the batch.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

#include "../../include/nbody.h"

namespace nbody {

constexpr int kReadFields = 3;

// A handle's staging memory for reads, allocated on the first one and kept.
struct ReadStage {
    float* pinned = nullptr;  // host memory the device writes to (at most kPinnedReadBytes)
    size_t pinned_floats = 0;
    float* dev = nullptr;     // device memory, one field
    size_t dev_floats = 0;
};

// Reads up to this many bytes of packed fields go through pinned memory: a host
// copy out of it costs less there than three copies by the DMA engines into
// pageable memory (all three fields of 200,000 particles: 0.38 ms against 0.47;
// of 400,000, 0.92 against 0.86).
constexpr size_t kPinnedReadBytes = size_t(8) << 20;

// Pack the fields' n records (src[f] with a non-null dst[f]) behind whatever is
// queued on the stream, and wait for them.  dst[f]: 3n floats each.
nbody_status read_packed(ReadStage& st, const float4* const (&src)[kReadFields], float* const (&dst)[kReadFields],
                         size_t n, hipStream_t stream);

// The same, but a small read stays where the device wrote it: out[f] points to
// field f's 3n floats in the pinned memory (valid until the next read).  Returns
// NBODY_ERR_CAPACITY, with nothing done, when the fields do not fit it.
nbody_status read_pinned(ReadStage& st, const float4* const (&src)[kReadFields], const bool (&want)[kReadFields],
                         size_t n, hipStream_t stream, const float* (&out)[kReadFields]);

void release_stage(ReadStage& st);

}  // namespace nbody
