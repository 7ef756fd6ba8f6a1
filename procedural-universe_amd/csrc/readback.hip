// Read-back: the device packs the records, so that 12 bytes a particle and
// field cross the bus instead of 16 and the host copies nothing twice.
//
// A small read is one kernel that writes the packed fields into pinned host
// memory, one wait and a memcpy; a large one packs a field into a device buffer
// and copies that straight into the caller's memory.  Against a copy of the
// whole records, a wait and a host loop per field, into the caller's own
// buffers: 1,000 particles 89 -> 18 us, 50,000 187 -> 90 us, 10^6 4.9 -> 2.1 ms,
// 4 x 10^6 30 -> 8.2 ms.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <memory>
#include <new>

#include "common.hpp"
#include "readback.hpp"

namespace nbody {

namespace {

constexpr int kPackThreads = 256;

struct PackArgs {
    const float4* src[kReadFields];
    float* dst[kReadFields];
    int n;
};

// Field blockIdx.y, 256 records a workgroup, through LDS so that the writes are
// whole lines in order (they may go to host memory).
__global__ __launch_bounds__(kPackThreads) void pack_fields_kernel(PackArgs A) {
    __shared__ float s[3 * kPackThreads];
    const int t = threadIdx.x, base = blockIdx.x * kPackThreads;
    const float4* src = A.src[blockIdx.y];
    if (base + t < A.n) {
        const float4 p = src[base + t];
        s[3 * t] = p.x;
        s[3 * t + 1] = p.y;
        s[3 * t + 2] = p.z;
    }
    __syncthreads();
    float* dst = A.dst[blockIdx.y] + 3 * static_cast<size_t>(base);
    const int count = 3 * min(kPackThreads, A.n - base);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int i = k * kPackThreads + t;
        if (i < count) dst[i] = s[i];
    }
}

nbody_status pack(const PackArgs& A, int fields, hipStream_t stream) {
    hipLaunchKernelGGL(pack_fields_kernel, dim3((A.n + kPackThreads - 1) / kPackThreads, fields), dim3(kPackThreads), 0,
                       stream, A);
    NB_HIP(hipGetLastError());
    return NBODY_OK;
}

}  // namespace

nbody_status read_pinned(ReadStage& st, const float4* const (&src)[kReadFields], const bool (&want)[kReadFields],
                         size_t n, hipStream_t stream, const float* (&out)[kReadFields]) {
    PackArgs A{};
    int fields = 0;
    for (int f = 0; f < kReadFields; ++f)
        if (want[f]) A.src[fields++] = src[f];
    const size_t floats = 3 * n * static_cast<size_t>(fields);
    if (floats * sizeof(float) > kPinnedReadBytes) return NBODY_ERR_CAPACITY;
    if (floats > st.pinned_floats) {
        if (st.pinned) (void)hipHostFree(st.pinned);
        st.pinned = nullptr;
        st.pinned_floats = 0;
        // in powers of two from 64 KiB on: a batch reads systems of many sizes,
        // and an allocation takes some 350 us
        size_t bytes = size_t(1) << 16;
        while (bytes < floats * sizeof(float)) bytes *= 2;
        if (hipHostMalloc(reinterpret_cast<void**>(&st.pinned), bytes, hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();
            st.pinned = nullptr;
            return NBODY_ERR_CAPACITY;
        }
        st.pinned_floats = bytes / sizeof(float);
    }
    A.n = static_cast<int>(n);
    int at = 0;
    for (int f = 0; f < kReadFields; ++f) {
        out[f] = nullptr;
        if (!want[f]) continue;
        A.dst[at] = st.pinned + 3 * n * static_cast<size_t>(at);
        out[f] = A.dst[at++];
    }
    if (n > 0 && fields > 0) NB_TRY(pack(A, fields, stream));
    NB_HIP(hipStreamSynchronize(stream));
    return NBODY_OK;
}

nbody_status read_packed(ReadStage& st, const float4* const (&src)[kReadFields], float* const (&dst)[kReadFields],
                         size_t n, hipStream_t stream) {
    const bool want[kReadFields] = {dst[0] != nullptr, dst[1] != nullptr, dst[2] != nullptr};
    const float* from[kReadFields];
    const nbody_status small = read_pinned(st, src, want, n, stream, from);
    if (small == NBODY_OK) {
        for (int f = 0; f < kReadFields; ++f)
            if (want[f]) std::memcpy(dst[f], from[f], 3 * n * sizeof(float));
        return NBODY_OK;
    }
    if (small != NBODY_ERR_CAPACITY) return small;
    if (3 * n > st.dev_floats) {
        if (st.dev) {
            NB_HIP(hipStreamSynchronize(stream));
            (void)hipFree(st.dev);
        }
        const size_t floats = std::max(3 * n, st.dev_floats + st.dev_floats / 2);
        st.dev = nullptr;
        st.dev_floats = 0;
        if (hipMalloc(reinterpret_cast<void**>(&st.dev), floats * sizeof(float)) == hipSuccess) {
            st.dev_floats = floats;
        } else {
            (void)hipGetLastError();
            st.dev = nullptr;
        }
    }
    std::unique_ptr<float4[]> tmp;  // a device too full for one packed field: whole records
    if (!st.dev) {
        tmp.reset(new (std::nothrow) float4[n]);
        NB_CHECK(tmp, NBODY_ERR_OUT_OF_MEMORY, "no host memory to read %zu records", n);
    }
    for (int f = 0; f < kReadFields; ++f) {
        if (!want[f]) continue;
        if (st.dev) {
            PackArgs A{};
            A.src[0] = src[f];
            A.dst[0] = st.dev;
            A.n = static_cast<int>(n);
            NB_TRY(pack(A, 1, stream));
            NB_HIP(hipMemcpyAsync(dst[f], st.dev, 3 * n * sizeof(float), hipMemcpyDeviceToHost, stream));
        } else {
            NB_HIP(hipMemcpyAsync(tmp.get(), src[f], n * sizeof(float4), hipMemcpyDeviceToHost, stream));
            NB_HIP(hipStreamSynchronize(stream));
            for (size_t i = 0; i < n; ++i) {
                dst[f][3 * i] = tmp[i].x;
                dst[f][3 * i + 1] = tmp[i].y;
                dst[f][3 * i + 2] = tmp[i].z;
            }
        }
    }
    NB_HIP(hipStreamSynchronize(stream));
    return NBODY_OK;
}

void release_stage(ReadStage& st) {
    if (st.pinned) (void)hipHostFree(st.pinned);
    if (st.dev) (void)hipFree(st.dev);
    st = ReadStage{};
}

}  // namespace nbody
