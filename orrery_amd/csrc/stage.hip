// Host arrays to and from the device, several rows of one length at a time.
//
// A copy from or to pageable memory costs some ten microseconds of its own
// whatever its size, and a force evaluation from host arrays makes seven of
// them, a batch's read-back nine a system. Small transfers go through one
// pinned buffer a context instead: the rows are copied into it by the host (or
// out of it), and one launch moves them all, reading or writing the pinned
// memory directly. Longer transfers are bound by the link, not by their number,
// and are copied row by row as they are.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <mutex>

#include "engine.hpp"

namespace orr {
namespace {

constexpr int kBlock = 256;

struct Rows {
    double* device[kStageRows];
};

__global__ __launch_bounds__(kBlock) void rows_to_host(Rows rows, double* __restrict__ host, std::uint64_t count) {
    const std::uint64_t i = static_cast<std::uint64_t>(blockIdx.x) * kBlock + threadIdx.x;
    if (i < count) host[blockIdx.y * count + i] = rows.device[blockIdx.y][i];
}

__global__ __launch_bounds__(kBlock) void rows_to_device(Rows rows, const double* __restrict__ host,
                                                         std::uint64_t count) {
    const std::uint64_t i = static_cast<std::uint64_t>(blockIdx.x) * kBlock + threadIdx.x;
    if (i < count) rows.device[blockIdx.y][i] = host[blockIdx.y * count + i];
}

dim3 row_grid(int rows, std::uint64_t count) {
    return dim3(static_cast<std::uint32_t>((count + kBlock - 1) / kBlock), static_cast<std::uint32_t>(rows));
}

// The context's pinned buffer with room for `bytes` and nothing in flight
// through it. The caller holds the stage's lock.
double* pinned(orr_ctx* ctx, std::size_t bytes) {
    auto& s = ctx->staging;
    if (s.busy) {
        ORR_HIP(hipStreamSynchronize(ctx->stream));
        s.busy = false;
    }
    if (bytes > s.bytes) {
        s.release();
        const std::size_t grown = std::min(kStageBytes, std::max<std::size_t>(bytes * 2, 1u << 16));
        ORR_HIP(hipHostMalloc(&s.ptr, grown, hipHostMallocDefault));
        s.bytes = grown;
    }
    return static_cast<double*>(s.ptr);
}

}  // namespace

void stage_upload(orr_ctx* ctx, double* const* device, const double* const* host, int rows,
                  std::uint64_t count) {
    if (rows == 0 || count == 0) return;
    const std::size_t row = sizeof(double) * count;
    if (row * rows > kStageBytes) {
        for (int k = 0; k < rows; ++k) {
            ORR_HIP(hipMemcpyAsync(device[k], host[k], row, hipMemcpyHostToDevice, ctx->stream));
        }
        ORR_HIP(hipStreamSynchronize(ctx->stream));
        return;
    }
    std::lock_guard<std::mutex> lock(ctx->staging.lock);
    double* p = pinned(ctx, row * rows);
    Rows r{};
    for (int k = 0; k < rows; ++k) {
        std::memcpy(p + k * count, host[k], row);
        r.device[k] = device[k];
    }
    hipLaunchKernelGGL(rows_to_device, row_grid(rows, count), dim3(kBlock), 0, ctx->stream, r, p, count);
    ORR_LAUNCHED("rows_to_device");
    ctx->staging.busy = true;
}

void stage_download(orr_ctx* ctx, double* const* host, double* const* device, int rows, std::uint64_t count) {
    if (rows == 0 || count == 0) {
        ctx->sync();
        return;
    }
    const std::size_t row = sizeof(double) * count;
    if (row * rows > kStageBytes) {
        for (int k = 0; k < rows; ++k) {
            ORR_HIP(hipMemcpyAsync(host[k], device[k], row, hipMemcpyDeviceToHost, ctx->stream));
        }
        ctx->sync();
        return;
    }
    std::lock_guard<std::mutex> lock(ctx->staging.lock);
    double* p = pinned(ctx, row * rows);
    Rows r{};
    for (int k = 0; k < rows; ++k) r.device[k] = device[k];
    hipLaunchKernelGGL(rows_to_host, row_grid(rows, count), dim3(kBlock), 0, ctx->stream, r, p, count);
    ORR_LAUNCHED("rows_to_host");
    ctx->sync();
    for (int k = 0; k < rows; ++k) std::memcpy(host[k], p + k * count, row);
}

}  // namespace orr
