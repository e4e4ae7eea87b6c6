// The bounding cube and the Morton codes of positions, bit for bit the reference's
// (src/solvers/morton.cpp:87-164): shared by the ordering launches and the
// kernels that order a small system themselves.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace orr {

constexpr unsigned kGrid = 1u << 21;

// The cube arithmetic of morton.cpp:87-103 from exact extrema: cube = {origin, size}.
__device__ inline void make_cube(const double lo[3], const double hi[3], double* cube) {
#pragma clang fp contract(off)
    const double ex = hi[0] - lo[0], ey = hi[1] - lo[1], ez = hi[2] - lo[2];
    // std::max({ex, ey, ez}) keeps the first of equals; the value is what matters.
    double size = ex;
    if (size < ey) size = ey;
    if (size < ez) size = ez;
    if (!(size > 0)) size = 1;
    for (int c = 0; c < 3; ++c) {
        const double centre = (lo[c] + hi[c]) / 2;
        cube[c] = centre - size / 2;
    }
    cube[3] = size;
}

__device__ inline std::uint64_t spread_bits(std::uint32_t v) {
    std::uint64_t s = v & 0x1fffffu;
    s = (s | (s << 32)) & 0x1f00000000ffffull;
    s = (s | (s << 16)) & 0x1f0000ff0000ffull;
    s = (s | (s << 8)) & 0x100f00f00f00f00full;
    s = (s | (s << 4)) & 0x10c30c30c30c30c3ull;
    s = (s | (s << 2)) & 0x1249249249249249ull;
    return s;
}

__device__ inline std::uint32_t to_grid(double coordinate, double origin, double scale) {
#pragma clang fp contract(off)
    const double cell = (coordinate - origin) * scale;
    if (!(cell > 0)) return 0;
    if (cell >= static_cast<double>(kGrid)) return kGrid - 1;
    return static_cast<std::uint32_t>(cell);
}

// The 32 bits of a position's code from digit 4 up, as encode computes them.
__device__ __forceinline__ std::uint32_t top_code(double px, double py, double pz, const double* cube,
                                                  double scale) {
    if (!(cube[3] > 0)) return 0;
    const std::uint64_t code = (spread_bits(to_grid(px, cube[0], scale)) << 2) |
                               (spread_bits(to_grid(py, cube[1], scale)) << 1) |
                               spread_bits(to_grid(pz, cube[2], scale));
    return static_cast<std::uint32_t>(code >> 32);
}

}  // namespace orr
