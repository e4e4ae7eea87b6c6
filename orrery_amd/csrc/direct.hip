// Direct O(N^2) softened gravity on gfx950.
//
// Replaces the reference's CUDA direct kernel (src/solvers/cuda_direct_kernel.cu:87-214),
// which gives one thread one target and stages j-tiles of positions through
// shared memory with two barriers per tile. Here:
//
//   * Sources are packed once per evaluation into 64-particle tiles: a float4
//     {ox, oy, oz, m} per particle, the offset o taken in FP64 from the tile's
//     FP64 centre (midpoint of its bounding box) and rounded to FP32, plus the
//     rounding residual o_lo = (x - c) - o as a second float4. In Morton order
//     a tile is spatially compact, so o carries the precision of the tile's
//     size rather than of the system's.
//   * A wave reads a source tile through the scalar unit: the address is
//     wave-uniform, so each {ox, oy, oz, m} arrives in SGPRs and is broadcast
//     to all 64 lanes as an instruction operand. No LDS, no barriers.
//   * Each lane owns R targets. Per target and source tile the target is
//     re-expressed against the source tile's centre as one FP64 difference
//     rounded once; far tiles use the separation o_j - t_hi (one rounding of
//     the separation), 12 VALU operations and one v_rsq_f32 of (r^2+eps^2)^3
//     per interaction.
//   * Near tiles -- boxes whose gap is at most a tenth of their summed
//     half-widths (near_tiles) -- use the double-float separation (o_j - t) +
//     (o_lo_j - t_lo). Pairs among them closer than a quarter of the wider tile's
//     half-width are marked and evaluated afterwards in FP64 (close_pair.hpp):
//     their single term can be many times the net force on either particle.
//   * Far tiles' terms are summed in FP32 in runs of 16, near tiles' in runs
//     of 8, each run Kahan-added into the target's running sum.
//   * The source range is split over gridDim.y; a fixed-order FP64 reduction
//     kernel folds the splits, multiplies by G and scatters to particle order.
//   * By default (direct_pairs, below) each far pair of tiles is evaluated
//     once and applied to both tiles, with the same packing, near test, close
//     pairs and compensation; the one-sided kernel above then covers what the
//     pairs path does not take (configured off, too few tiles, or slots beyond
//     16 GiB).
//
// The reference counts 20 flop per interaction (docs/performance.md:103-109).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <mutex>
#include <type_traits>
#include <utility>

#include "close_pair.hpp"
#include "engine.hpp"
#include "morton_code.hpp"

namespace orr {
namespace {

constexpr int kTile = 64;    // sources per tile = one wave of the prepare kernel
constexpr int kBlock = 256;  // four waves
constexpr float kNearGap = 0.1f;

__device__ inline double wave_min(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmin(v, __shfl_xor(v, off, 64));
    return v;
}
__device__ inline double wave_max(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off, 64));
    return v;
}

// One wave packs one tile: centre its (valid) particles, split each offset
// into an FP32 value and its FP32 residual. centres[tile] = {cx, cy, cz,
// largest half-extent}; extents[tile] = {hx, hy, hz, w}.
__device__ __forceinline__ void pack_tile(double px, double py, double pz, double pm, bool valid,
                                          std::uint64_t k, std::uint32_t tile,
                                          float4* __restrict__ packed,
                                          float4* __restrict__ packed_lo,
                                          double4* __restrict__ centres,
                                          float4* __restrict__ extents,
                                          float2* __restrict__ mass_range = nullptr) {
    const double inf = __builtin_huge_val();
    const double lx = wave_min(valid ? px : inf), hx = wave_max(valid ? px : -inf);
    const double ly = wave_min(valid ? py : inf), hy = wave_max(valid ? py : -inf);
    const double lz = wave_min(valid ? pz : inf), hz = wave_max(valid ? pz : -inf);
    const double cx = 0.5 * (lx + hx), cy = 0.5 * (ly + hy), cz = 0.5 * (lz + hz);
    const double w = 0.5 * fmax(hx - lx, fmax(hy - ly, hz - lz));
    if (valid) {
        const double dx = px - cx, dy = py - cy, dz = pz - cz;
        const float ox = static_cast<float>(dx), oy = static_cast<float>(dy), oz = static_cast<float>(dz);
        packed[k] = make_float4(ox, oy, oz, static_cast<float>(pm));
        packed_lo[k] = make_float4(static_cast<float>(dx - ox), static_cast<float>(dy - oy),
                                   static_cast<float>(dz - oz), 0.f);
    } else {
        packed[k] = make_float4(0.f, 0.f, 0.f, 0.f);
        packed_lo[k] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    if (mass_range != nullptr) {
        // The tile's smallest and largest packed mass, its massless pads
        // included: a system with pads never counts as one of equal masses.
        const double fm = valid ? static_cast<double>(static_cast<float>(pm)) : 0.0;
        const double lo = wave_min(fm), hi = wave_max(fm);
        if ((threadIdx.x & (kTile - 1)) == 0) {
            mass_range[tile] = make_float2(static_cast<float>(lo), static_cast<float>(hi));
        }
    }
    if ((threadIdx.x & (kTile - 1)) == 0) {
        centres[tile] = make_double4(cx, cy, cz, w);
        extents[tile] = make_float4(static_cast<float>(0.5 * (hx - lx)), static_cast<float>(0.5 * (hy - ly)),
                                    static_cast<float>(0.5 * (hz - lz)), static_cast<float>(w));
    }
}

// One wave per tile of one system: gather (optionally through `order`) and pack.
__global__ __launch_bounds__(64) void direct_prepare(const double* __restrict__ x,
                                                     const double* __restrict__ y,
                                                     const double* __restrict__ z,
                                                     const double* __restrict__ m,
                                                     const std::uint32_t* __restrict__ order,
                                                     std::uint64_t n, float4* __restrict__ packed,
                                                     float4* __restrict__ packed_lo,
                                                     double4* __restrict__ centres,
                                                     float4* __restrict__ extents,
                                                     float2* __restrict__ mass_range) {
    const std::uint64_t k = static_cast<std::uint64_t>(blockIdx.x) * kTile + threadIdx.x;
    const bool valid = k < n;
    const std::uint64_t src = valid ? (order != nullptr ? order[k] : k) : 0;
    pack_tile(valid ? x[src] : 0.0, valid ? y[src] : 0.0, valid ? z[src] : 0.0,
              valid ? m[src] : 0.0, valid, k, blockIdx.x, packed, packed_lo, centres, extents,
              mass_range);
}

// uniform[0] = the common packed mass when every particle has the same
// positive mass, else 0 (one block over the tiles' ranges).
__global__ __launch_bounds__(256) void mass_uniform(const float2* __restrict__ mass_range,
                                                    std::uint32_t tiles, int enabled,
                                                    float* __restrict__ uniform) {
    __shared__ float lo_s[256], hi_s[256];
    float lo = __builtin_huge_valf(), hi = -__builtin_huge_valf();
    for (std::uint32_t t = threadIdx.x; t < tiles; t += blockDim.x) {
        const float2 r = mass_range[t];
        lo = fminf(lo, r.x);
        hi = fmaxf(hi, r.y);
    }
    lo_s[threadIdx.x] = lo;
    hi_s[threadIdx.x] = hi;
    __syncthreads();
    for (unsigned half = 128; half > 0; half >>= 1) {
        if (threadIdx.x < half) {
            lo_s[threadIdx.x] = fminf(lo_s[threadIdx.x], lo_s[threadIdx.x + half]);
            hi_s[threadIdx.x] = fmaxf(hi_s[threadIdx.x], hi_s[threadIdx.x + half]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) uniform[0] = (enabled && lo_s[0] == hi_s[0] && lo_s[0] > 0.f) ? lo_s[0] : 0.f;
}

// One pairwise term accumulated into (px, py, pz). kSafe masks r^2 == 0 (zero
// softening): the self term and coincident pads then contribute m * finite * 0
// = 0 instead of NaN, as the reference's CUDA kernel masks self and tail terms
// (cuda_direct_kernel.cu:134-159). kRefine applies one Newton-Raphson step to
// the hardware reciprocal square root y0 before cubing: with e = 1 - x y0^2
// (one rounding, via FMA), y^3 = y0^3 (1 + 3e/2) to second order in e.
template<bool kSafe, bool kRefine>
__device__ __forceinline__ float inv_cubed(float r2) {
    if constexpr (kSafe) r2 = r2 > 0.f ? r2 : 1.f;
    if constexpr (!kSafe && !kRefine) {
        return __builtin_amdgcn_rsqf((r2 * r2) * r2);
    } else {
        const float inv = __builtin_amdgcn_rsqf(r2);
        float inv3 = (inv * inv) * inv;
        if constexpr (kRefine) {
            const float e = __builtin_fmaf(-(r2 * inv), inv, 1.f);
            inv3 = inv3 * __builtin_fmaf(1.5f, e, 1.f);
        }
        return inv3;
    }
}

template<bool kSafe, bool kRefine>
__device__ __forceinline__ void term(float dx, float dy, float dz, float m, float eps2, float& px,
                                     float& py, float& pz) {
    float r2 = __builtin_fmaf(dx, dx, eps2);
    r2 = __builtin_fmaf(dy, dy, r2);
    r2 = __builtin_fmaf(dz, dz, r2);
    const float f = m * inv_cubed<kSafe, kRefine>(r2);
    px = __builtin_fmaf(f, dx, px);
    py = __builtin_fmaf(f, dy, py);
    pz = __builtin_fmaf(f, dz, pz);
}

__device__ __forceinline__ void kahan(float p, float& s, float& c) {
    const float y = p - c;
    const float t = s + y;
    c = (t - s) - y;
    s = t;
}

// Near: the gap between the two tiles' boxes (centre c, half-extents e; the
// source tile's C, E) is at most kNearGap of their summed half-widths. Outside
// it every separation exceeds that gap, so the FP32 offsets round it to
// O(epsilon) relative error. One definition, without contraction, so the mask
// pass and the kernels classify every tile pair alike.
__device__ __forceinline__ bool near_tiles(const double4& C, const float4& E, double cx, double cy,
                                           double cz, const float4& e) {
#pragma clang fp contract(off)
    const float gx = fmaxf(0.f, fabsf(static_cast<float>(C.x - cx)) - e.x - E.x);
    const float gy = fmaxf(0.f, fabsf(static_cast<float>(C.y - cy)) - e.y - E.y);
    const float gz = fmaxf(0.f, fabsf(static_cast<float>(C.z - cz)) - e.z - E.z);
    const float reach = kNearGap * (e.w + E.w);
    return gx * gx + gy * gy + gz * gz <= reach * reach;
}

// Close pairs: closer than kClose times the wider tile's largest half-extent.
// Their terms are evaluated in FP64 (close_pair.hpp); about
// one step in twenty of a near pass has such a pair on some lane.
constexpr float kClose = 0.25f;

// The FP32 r^2 below which a near pair is close (r^2 includes eps^2).
__device__ __forceinline__ float close_limit(double w_target, double w_source, float eps2) {
    const float rc = kClose * static_cast<float>(fmax(w_target, w_source));
    return __builtin_fmaf(rc, rc, eps2);
}

// Adds the double-float value (h, l) to the Kahan pair (s, c) (value s - c).
__device__ __forceinline__ void kahan_df(float h, float l, float& s, float& c) {
    kahan(h, s, c);
    c = c - l;
}

// Targets' sums against one 64-source tile J.
//
//   * Far tiles: each target is re-expressed against the source tile's centre
//     with one rounding (the FP64 difference of its (hi, lo) offset and the
//     centres, rounded once); the terms are summed plainly in FP32 in runs of
//     kRun and each run is Kahan-added per component into (s, k).
//   * Near tiles: double-float separations, runs of kNearRun terms summed in
//     FP32 and Kahan-added into the tile's own pair, close pairs evaluated in
//     FP64 and added to it as (hi, lo); the tile's pair then joins (s, k).
//
// kUnroll sets how many far-path sources are in flight (their SGPR loads
// included). `sources` of the tile are particles and the rest massless pads at
// its centre, and `live` says which targets are particles: pads lie on top of
// one another, so the near path leaves them out -- their zero terms change no
// sum, and as close pairs they would take up to 64 FP64 evaluations a lane.
constexpr int kRun = 16;
// Terms of a near tile summed plainly in FP32 before each Kahan addition.
constexpr int kNearRun = 8;

//
// source_tile_to hands each far run's sums, or the near tile's pair, to its
// caller; source_tile adds them.
template<int R, bool kSafe, bool kRefine, bool kGivenNear, int kUnroll, class Far, class Near>
__device__ __forceinline__ void source_tile_to(
    const float4* __restrict__ packed, const float4* __restrict__ packed_lo,
    const double4* __restrict__ centres, const float4* __restrict__ extents, std::uint32_t J,
    bool given_near, std::uint32_t sources, const bool (&live)[R], float eps2,
    const float (&ox)[R], const float (&oy)[R], const float (&oz)[R], const float (&lx)[R], const float (&ly)[R], const float (&lz)[R], const double (&cx)[R],
    const double (&cy)[R], const double (&cz)[R], const float4 (&ce)[R], Far&& far_run, Near&& near_pair_sums) {
    const double4 C = centres[J];
    const float4 E = extents[J];
    const float4* __restrict__ src = packed + static_cast<std::size_t>(J) * kTile;
    // eps^2 enters every term: a vector register, since a scalar operand
    // halves an FP32 instruction's issue rate.
    asm volatile("" : "+v"(eps2));
    // All lanes of a wave share one target tile per r, so the branch is
    // uniform. With kGivenNear the caller read the pair's flag from the mask.
    bool near = false;
    if constexpr (kGivenNear) {
        near = given_near;
    } else {
#pragma unroll
        for (int r = 0; r < R; ++r) near = near || near_tiles(C, E, cx[r], cy[r], cz[r], ce[r]);
    }
    // Each target's position relative to the source tile's centre: FP64 from
    // its (hi, lo) offset, split into (hi, lo) floats.
    float th[R][3], tl[R][3];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const double t[3] = {(static_cast<double>(ox[r]) + lx[r]) - (C.x - cx[r]),
                             (static_cast<double>(oy[r]) + ly[r]) - (C.y - cy[r]),
                             (static_cast<double>(oz[r]) + lz[r]) - (C.z - cz[r])};
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            th[r][c] = static_cast<float>(t[c]);
            tl[r][c] = static_cast<float>(t[c] - th[r][c]);
        }
    }
    if (!near) {
#pragma unroll
        for (int run = 0; run < kTile / kRun; ++run) {
            float px[R], py[R], pz[R];
#pragma unroll
            for (int r = 0; r < R; ++r) px[r] = py[r] = pz[r] = 0.f;
#pragma unroll (kUnroll < kRun ? kUnroll : kRun)
            for (int j = run * kRun; j < (run + 1) * kRun; ++j) {
                const float4 q = src[j];
#pragma unroll
                for (int r = 0; r < R; ++r)
                    term<kSafe, kRefine>(q.x - th[r][0], q.y - th[r][1], q.z - th[r][2], q.w, eps2,
                                         px[r], py[r], pz[r]);
            }
#pragma unroll
            for (int r = 0; r < R; ++r) far_run(r, run, px[r], py[r], pz[r]);
        }
        return;
    }
    const float4* __restrict__ src_lo = packed_lo + static_cast<std::size_t>(J) * kTile;
    float px[R], py[R], pz[R], pkx[R], pky[R], pkz[R], lim[R];
    // Per lane, the sources that are close pairs: the flags of 32 sources in a
    // word, shifted in from the right (one add with carry a source).
    std::uint32_t close[R][2];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        px[r] = py[r] = pz[r] = pkx[r] = pky[r] = pkz[r] = 0.f;
        lim[r] = live[r] ? close_limit(ce[r].w, E.w, eps2) : -1.f;
        close[r][0] = close[r][1] = 0;
    }
#pragma unroll 1
    for (int j0 = 0; j0 < static_cast<int>(sources); j0 += kNearRun) {
        if (j0 == kTile / 2) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                close[r][0] = close[r][1];
                close[r][1] = 0;
            }
        }
        float qx[R], qy[R], qz[R];
#pragma unroll
        for (int r = 0; r < R; ++r) qx[r] = qy[r] = qz[r] = 0.f;
#pragma unroll
        for (int j = j0; j < j0 + kNearRun; ++j) {
            const float4 q = src[j];
            const float4 ql = src_lo[j];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const float dx = (q.x - th[r][0]) + (ql.x - tl[r][0]);
                const float dy = (q.y - th[r][1]) + (ql.y - tl[r][1]);
                const float dz = (q.z - th[r][2]) + (ql.z - tl[r][2]);
                float r2 = __builtin_fmaf(dx, dx, eps2);
                r2 = __builtin_fmaf(dy, dy, r2);
                r2 = __builtin_fmaf(dz, dz, r2);
                // A close pair's FP32 term is left out here and added in
                // FP64 below (r^2 holds eps^2, so it is zero only without
                // softening).
                const bool near_pair = r2 < lim[r] && (!kSafe || r2 > 0.f);
                close[r][1] = close[r][1] + close[r][1] + (near_pair ? 1u : 0u);
                const float f = near_pair ? 0.f : q.w * inv_cubed<kSafe, kRefine>(r2);
                qx[r] = __builtin_fmaf(f, dx, qx[r]);
                qy[r] = __builtin_fmaf(f, dy, qy[r]);
                qz[r] = __builtin_fmaf(f, dz, qz[r]);
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            kahan(qx[r], px[r], pkx[r]);
            kahan(qy[r], py[r], pky[r]);
            kahan(qz[r], pz[r], pkz[r]);
        }
    }
    // What the pads' runs of zero terms would do: one addition of zero moves a
    // compensation into its sum where it is large enough to show, more change
    // nothing.
    auto add_zero = [&](int r) {
        kahan(0.f, px[r], pkx[r]);
        kahan(0.f, py[r], pky[r]);
        kahan(0.f, pz[r], pkz[r]);
    };
    if (sources + kNearRun <= kTile) {
#pragma unroll
        for (int r = 0; r < R; ++r) add_zero(r);
    }
    // The close pairs, each lane over its own (few): sources read by index.
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const double t[3] = {static_cast<double>(th[r][0]) + static_cast<double>(tl[r][0]),
                             static_cast<double>(th[r][1]) + static_cast<double>(tl[r][1]),
                             static_cast<double>(th[r][2]) + static_cast<double>(tl[r][2])};
        // The first source to the highest bit (the runs taken fill `taken` bits,
        // the last 32 of them or fewer in close[1]), and no pads.
        const std::uint32_t taken = (sources + kNearRun - 1) / kNearRun * kNearRun;
        std::uint64_t bits = static_cast<std::uint64_t>(close[r][0]) << 32 |
                             static_cast<std::uint64_t>(close[r][1]) << (taken > 32 ? 64 - taken : 32 - taken);
        if (taken <= 32) bits <<= 32;
        bits &= ~std::uint64_t{0} << (kTile - sources);
        while (bits != 0) {
            const int j = __builtin_clzll(bits);
            bits &= ~(std::uint64_t{1} << (63 - j));
            const float4 q = src[j];
            const float4 ql = src_lo[j];
            const float bh[3] = {q.x, q.y, q.z}, bl[3] = {ql.x, ql.y, ql.z};
            double G[3];
            close_pair(t, bh, bl, eps2, G);
            const double mq = q.w;
            float h, l;
            split(mq * G[0], h, l);
            kahan_df(h, l, px[r], pkx[r]);
            split(mq * G[1], h, l);
            kahan_df(h, l, py[r], pky[r]);
            split(mq * G[2], h, l);
            kahan_df(h, l, pz[r], pkz[r]);
        }
        if (sources < kTile) {
            // The pads, at the tile's centre, are close pairs or none of them is.
            const float dx = -th[r][0] - tl[r][0], dy = -th[r][1] - tl[r][1], dz = -th[r][2] - tl[r][2];
            const float r2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, __builtin_fmaf(dx, dx, eps2)));
            if (r2 < lim[r] && (!kSafe || r2 > 0.f)) add_zero(r);
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) near_pair_sums(r, px[r], py[r], pz[r], pkx[r], pky[r], pkz[r]);
}

template<int R, bool kSafe, bool kRefine, bool kGivenNear = false, int kUnroll = 16>
__device__ __forceinline__ void source_tile(
    const float4* __restrict__ packed, const float4* __restrict__ packed_lo,
    const double4* __restrict__ centres, const float4* __restrict__ extents, std::uint32_t J,
    bool given_near, std::uint32_t sources, const bool (&live)[R], float eps2,
    const float (&ox)[R], const float (&oy)[R], const float (&oz)[R], const float (&lx)[R], const float (&ly)[R], const float (&lz)[R], const double (&cx)[R],
    const double (&cy)[R], const double (&cz)[R], const float4 (&ce)[R], float (&sx)[R],
    float (&sy)[R], float (&sz)[R], float (&kx)[R], float (&ky)[R], float (&kz)[R]) {
    source_tile_to<R, kSafe, kRefine, kGivenNear, kUnroll>(
        packed, packed_lo, centres, extents, J, given_near, sources, live, eps2, ox, oy, oz, lx, ly, lz, cx, cy,
        cz, ce,
        [&](int r, int, float x, float y, float z) {
            kahan(x, sx[r], kx[r]);
            kahan(y, sy[r], ky[r]);
            kahan(z, sz[r], kz[r]);
        },
        [&](int r, float x, float y, float z, float cx_, float cy_, float cz_) {
            kahan_df(x, -cx_, sx[r], kx[r]);
            kahan_df(y, -cy_, sy[r], ky[r]);
            kahan_df(z, -cz_, sz[r], kz[r]);
        });
}

// For the pairs path: the near flags of every (target tile, source tile) pair,
// one bit each, rows of ceil(tiles / 32) words, computed once per evaluation so
// that its kernels read one word per 32 source tiles through the scalar unit
// instead of each wave repeating the (wave-uniform) box test on its vector lanes.
constexpr int kMaskRows = 8;  // target tiles per block of the mask pass

__global__ __launch_bounds__(256) void near_mask(const double4* __restrict__ centres,
                                                 const float4* __restrict__ extents,
                                                 std::uint32_t tiles, std::uint32_t words,
                                                 std::uint32_t* __restrict__ mask) {
    // kMaskRows target tiles per block (wave-uniform: scalar loads); each
    // thread loads one source tile per chunk and tests it against all of them;
    // a wave's 64 results become two words by ballot.
    const std::uint32_t row0 = blockIdx.x * kMaskRows;
    const int lane = threadIdx.x & 63;
    for (std::uint32_t chunk = 0; chunk < tiles; chunk += blockDim.x) {
        const std::uint32_t J = chunk + threadIdx.x;
        const bool valid = J < tiles;
        const double4 C = valid ? centres[J] : make_double4(0, 0, 0, 0);
        const float4 E = valid ? extents[J] : make_float4(0, 0, 0, 0);
        const std::uint32_t first_word = (chunk + (threadIdx.x & ~63u)) / 32;
#pragma unroll
        for (int r = 0; r < kMaskRows; ++r) {
            const std::uint32_t row = row0 + r;
            if (row >= tiles) break;
            const double4 c = centres[row];
            const float4 e = extents[row];
            const std::uint64_t bits = __ballot(valid && near_tiles(C, E, c.x, c.y, c.z, e));
            if (lane == 0) {
                std::uint32_t* out = mask + static_cast<std::size_t>(row) * words;
                if (first_word < words) out[first_word] = static_cast<std::uint32_t>(bits);
                if (first_word + 1 < words) out[first_word + 1] = static_cast<std::uint32_t>(bits >> 32);
            }
        }
    }
}

// Where a one-sided evaluation's sums go: the fold's arguments.
struct FieldOut {
    std::uint64_t n = 0;
    const std::uint32_t* order = nullptr;
    double G = 1.0;
    double* ax = nullptr;
    double* ay = nullptr;
    double* az = nullptr;
    FusedKick kick;
};

// The fold's output: a, and the fused kick's v += s a when there is one.
__device__ __forceinline__ void store_field(std::uint64_t dst, double gx, double gy, double gz,
                                            double* __restrict__ ax, double* __restrict__ ay,
                                            double* __restrict__ az, const FusedKick& kick) {
    ax[dst] = gx;
    ay[dst] = gy;
    az[dst] = gz;
    if (kick.vx != nullptr) {
        kick.vx[dst] = kick_update(kick.vx[dst], kick.s, gx);
        kick.vy[dst] = kick_update(kick.vy[dst], kick.s, gy);
        kick.vz[dst] = kick_update(kick.vz[dst], kick.s, gz);
    }
}

// One-sided sums. A wave owns R target tiles (R lanes' worth of whole tiles, so
// a tile's centre and extents are wave-uniform) and takes groups of
// `per_group` source tiles; a group's sums start fresh in FP32 with their Kahan
// compensations and are added to the wave's FP64 sums as sum - compensation, so
// a wave leaves 24 bytes a target whatever number of groups it took (it used to
// leave them a group: 150 MB and 0.1 ms of an evaluation at N = 20,001).
//
// The groups are dealt to the blocks of a target (gridDim.y) in turn: near
// source tiles, which cost several times a far one, lie together around the
// target in Morton order and would otherwise all fall to one block. A wave
// finds which of its next 64 source tiles are near with one test a lane.
//
// The four waves of a block have target tiles of their own and meet the same
// source tiles at about the same time, so the scalar cache serves three of the
// four (four waves of one target on different source tiles took 1.6 times as
// long at N = 20,001). With one block a target (gridDim.y == 1) the field is
// written here.
//
// kPerSimd 8 asks the compiler for eight waves a SIMD, and it then takes one
// source's term after another where it otherwise interleaves four: faster from
// kFoldEightTiles tiles on, slower while a launch's own latency counts.
// Evaluations with kPerSimd 1 and 8: 1000 particles 56.9 and 58.0 us, 4096 66.9 and
// 67.7, 8192 118.6 and 117.6, 20,001 275 and 259, 131,072 6.44 and 5.55 ms,
// 262,144 23.6 and 19.9, 900,000, where the pairs path's slots no longer fit,
// 269.7 and 223.7 (before the groups' FP64 sums 375 us at 20,001, 23.3 and 265.7
// ms). It is that sequence that does it: with eight waves by fewer scalar registers
// alone 23.7 ms at 262,144. Near tiles lose by it, so particles taken in the
// caller's order, whose tiles may all be near, keep kPerSimd 1 (unsorted: 16,384
// 433 and 443 us, 40,000 2.18 and 2.23 ms).
constexpr std::uint32_t kFoldEightTiles = 128;

template<int R, bool kSafe, bool kRefine, int kPerSimd>
__global__ __launch_bounds__(kBlock, kPerSimd) void direct_fold(
    const float4* __restrict__ packed, const float4* __restrict__ packed_lo,
    const double4* __restrict__ centres, const float4* __restrict__ extents, std::uint32_t tiles,
    std::uint32_t per_group, std::uint32_t groups, float eps2, double* __restrict__ partial, FieldOut out) {
    constexpr int kWaves = kBlock / kTile;
    __shared__ double sums[kWaves][3 * R][kTile];
    const unsigned lane = threadIdx.x & (kTile - 1);
    const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kTile);
    // Target tile r of the wave (one past the last is worked on as the last and writes nothing).
    auto target_tile = [&](int r) { return (blockIdx.x * R + r) * kWaves + wave; };
    float ox[R], oy[R], oz[R], lx[R], ly[R], lz[R];
    double cx[R], cy[R], cz[R];
    float4 ce[R];
    bool live[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const std::uint32_t tile = min(target_tile(r), tiles - 1);
        live[r] = static_cast<std::uint64_t>(tile) * kTile + lane < out.n;
        const float4 o = packed[static_cast<std::size_t>(tile) * kTile + lane];
        const float4 l = packed_lo[static_cast<std::size_t>(tile) * kTile + lane];
        const double4 c = centres[tile];
        ox[r] = o.x;
        oy[r] = o.y;
        oz[r] = o.z;
        lx[r] = l.x;
        ly[r] = l.y;
        lz[r] = l.z;
        cx[r] = c.x;
        cy[r] = c.y;
        cz[r] = c.z;
        ce[r] = extents[tile];
    }
    // The lane's own FP64 sums, in LDS: touched once a group, and six registers
    // more a target would cost the eighth wave of a SIMD.
#pragma unroll
    for (int c = 0; c < 3 * R; ++c) sums[wave][c][lane] = 0.0;
    const std::uint32_t stride = gridDim.y;
    const std::uint32_t last = static_cast<std::uint32_t>(out.n - (static_cast<std::uint64_t>(tiles) - 1) * kTile);
    std::uint32_t met = 0;        // source tiles taken so far
    std::uint64_t near_bits = 0;  // of the 64 from met & ~63
    for (std::uint32_t g = blockIdx.y; g < groups; g += stride) {
        float sx[R], sy[R], sz[R], kx[R], ky[R], kz[R];
#pragma unroll
        for (int r = 0; r < R; ++r) sx[r] = sy[r] = sz[r] = kx[r] = ky[r] = kz[r] = 0.f;
        for (std::uint32_t o = 0; o < per_group && g * per_group + o < tiles; ++o, ++met) {
            if (met % 64 == 0) {
                const std::uint32_t gg = g + (o + lane) / per_group * stride;
                const std::uint32_t J = gg * per_group + (o + lane) % per_group;
                const bool valid = gg < groups && J < tiles;
                const double4 C = centres[valid ? J : 0];
                const float4 E = extents[valid ? J : 0];
                bool near = false;
#pragma unroll
                for (int r = 0; r < R; ++r) near = near || near_tiles(C, E, cx[r], cy[r], cz[r], ce[r]);
                near_bits = __ballot(valid && near);
            }
            const bool near = ((near_bits >> (met % 64)) & 1u) != 0;
            const std::uint32_t J = g * per_group + o;
            const std::uint32_t sources = J + 1 < tiles ? kTile : last;
            source_tile<R, kSafe, kRefine, true>(packed, packed_lo, centres, extents, J, near, sources, live,
                                                 eps2, ox, oy, oz, lx, ly, lz, cx, cy, cz, ce, sx, sy, sz, kx,
                                                 ky, kz);
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            sums[wave][3 * r][lane] += static_cast<double>(sx[r]) - static_cast<double>(kx[r]);
            sums[wave][3 * r + 1][lane] += static_cast<double>(sy[r]) - static_cast<double>(ky[r]);
            sums[wave][3 * r + 2][lane] += static_cast<double>(sz[r]) - static_cast<double>(kz[r]);
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const std::uint32_t tile = target_tile(r);
        if (tile >= tiles) continue;
        const double a[3] = {sums[wave][3 * r][lane], sums[wave][3 * r + 1][lane], sums[wave][3 * r + 2][lane]};
        const std::size_t k = static_cast<std::size_t>(tile) * kTile + lane;
        if (gridDim.y == 1) {
            if (k >= out.n) continue;
            const std::uint64_t dst = out.order != nullptr ? out.order[k] : k;
            store_field(dst, out.G * a[0], out.G * a[1], out.G * a[2], out.ax, out.ay, out.az, out.kick);
            continue;
        }
        // Component c of target k from block y at partial[(3 y + c) npad + k].
        const std::size_t np = static_cast<std::size_t>(tiles) * kTile;
        double* const to = partial + static_cast<std::size_t>(blockIdx.y) * 3 * np + k;
        to[0] = a[0];
        to[np] = a[1];
        to[2 * np] = a[2];
    }
}

// The blocks' FP64 sums of a target, in block order.
__global__ __launch_bounds__(kTile) void direct_reduce(const double* __restrict__ partial,
                                                       std::uint32_t blocks, std::uint32_t tiles,
                                                       FieldOut out) {
    const std::uint64_t k = static_cast<std::uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k >= out.n) return;
    const std::size_t np = static_cast<std::size_t>(tiles) * kTile;
    double a0 = 0.0, a1 = 0.0, a2 = 0.0;
#pragma unroll 8
    for (std::uint32_t s = 0; s < blocks; ++s) {
        const double* p = partial + static_cast<std::size_t>(s) * 3 * np + k;
        a0 += p[0];
        a1 += p[np];
        a2 += p[2 * np];
    }
    const std::uint64_t dst = out.order != nullptr ? out.order[k] : k;
    store_field(dst, out.G * a0, out.G * a1, out.G * a2, out.ax, out.ay, out.az, out.kick);
}

// ---- tiny systems: whole steps in one workgroup ----------------------------------
//
// Up to kTinyTiles tiles a step is five or six launches of a few microseconds
// each, 16 to 43 us that no launch fills. One workgroup does it all instead, any
// number of steps in one launch: wave (t, J) of tiles^2 waves takes the pairs of
// target tile t and source tile J, thread i < n holds particle i's state in
// registers, and the ordered, packed tiles live in LDS. Every piece of
// arithmetic is the launches' own -- the cube, codes and order (morton_code.hpp),
// pack_tile, near_tiles, source_tile, the FP64 addition of the tiles' sums in
// order, the unfused kicks and drifts -- so the steps are the same bits.
// Bound by one workgroup's latency: a velocity Verlet step of two bodies 33 ->
// 2.8 us, of 64 particles 33 -> 11, of 128 65 -> 18, of 256 72 -> 29.
constexpr int kTinyTiles = 4;
constexpr std::uint32_t kTinyMax = kTinyTiles * kTile;

struct TinyArgs {
    double *x[3] = {}, *v[3] = {}, *a[3] = {};
    const double* m = nullptr;
    std::uint32_t n = 0, steps = 0;
    int mode = 0;      // 0: the field only, 1: kick-drift-kick substeps, 2: Runge-Kutta 4
    int substeps = 1;  // mode 1
    bool ordered = false;
    float eps2 = 0.f;
    double G = 1.0;
    double kick[3] = {}, drift[3] = {};  // mode 1, per substep
    double dt = 0.0;                     // mode 2
};

__device__ __forceinline__ double unfused(double a, double s, double b) {
#pragma clang fp contract(off)
    return a + s * b;
}

template<bool kSafe, bool kRefine, bool kRk4>
__global__ __launch_bounds__(kTinyTiles * kTinyTiles * kTile) void direct_tiny(TinyArgs A) {
    __shared__ float4 packed[kTinyMax], packed_lo[kTinyMax];
    __shared__ double4 centres[kTinyTiles];
    __shared__ float4 extents[kTinyTiles];
    __shared__ double pos[4][kTinyMax];               // x y z m in tile order
    __shared__ double sums[kTinyTiles][3][kTinyMax];  // [source tile][component][target]
    __shared__ double wave_ext[kTinyTiles][6];
    __shared__ std::uint32_t codes[kTinyMax], ranks[kTinyMax];
    const std::uint32_t n = A.n, tiles = (n + kTile - 1) / kTile;
    const std::uint32_t i = threadIdx.x, lane = i & (kTile - 1);
    const std::uint32_t wave = __builtin_amdgcn_readfirstlane(i / kTile);
    const bool mine = i < n;
    double x[3] = {0, 0, 0}, v[3] = {0, 0, 0}, a[3] = {0, 0, 0};
    const double m = mine ? A.m[i] : 0.0;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        if (mine) x[c] = A.x[c][i];
        if (mine && A.mode != 0) {
            v[c] = A.v[c][i];
            a[c] = A.a[c][i];
        }
    }
    // a = the field of the positions x.
    auto field = [&] {
        std::uint32_t at = i;  // the particle's place in tile order
        if (A.ordered) {
            if (wave < tiles) {
                const double inf = __builtin_huge_val();
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const double lo = wave_min(mine ? x[c] : inf), hi = wave_max(mine ? x[c] : -inf);
                    if (lane == 0) {
                        wave_ext[wave][c] = lo;
                        wave_ext[wave][3 + c] = hi;
                    }
                }
            }
            if (i < kTinyMax) ranks[i] = 0;
            __syncthreads();
            double lo[3], hi[3], cube[4];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                lo[c] = wave_ext[0][c];
                hi[c] = wave_ext[0][3 + c];
                for (std::uint32_t w = 1; w < tiles; ++w) {
                    lo[c] = wave_ext[w][c] < lo[c] ? wave_ext[w][c] : lo[c];
                    hi[c] = wave_ext[w][3 + c] > hi[c] ? wave_ext[w][3 + c] : hi[c];
                }
            }
            make_cube(lo, hi, cube);
            if (i < tiles * kTile) {
                codes[i] = mine ? top_code(x[0], x[1], x[2], cube, static_cast<double>(kGrid) / cube[3]) : ~0u;
            }
            __syncthreads();
            // Rank: keys (code, index) before particle k's, the waves of one tile
            // of particles taking a tile of codes each.
            const std::uint32_t k = wave % tiles * kTile + lane, j0 = wave / tiles * kTile;
            if (k < n) {
                const std::uint32_t key = codes[k];
                std::uint32_t before = 0;
#pragma unroll 8
                for (std::uint32_t j = j0; j < j0 + kTile; ++j) {
                    const std::uint32_t c = codes[j];
                    before += c < key || (c == key && j < k) ? 1u : 0u;
                }
                atomicAdd(&ranks[k], before);
            }
            __syncthreads();
            if (mine) at = ranks[i];
        }
        if (mine) {
            pos[0][at] = x[0];
            pos[1][at] = x[1];
            pos[2][at] = x[2];
            pos[3][at] = m;
        }
        __syncthreads();
        if (wave < tiles) {
            pack_tile(mine ? pos[0][i] : 0.0, mine ? pos[1][i] : 0.0, mine ? pos[2][i] : 0.0,
                      mine ? pos[3][i] : 0.0, mine, i, wave, packed, packed_lo, centres, extents);
        }
        __syncthreads();
        const std::uint32_t t = wave / tiles, J = wave % tiles, k = t * kTile + lane;
        const float4 o = packed[k], l = packed_lo[k];
        const double4 C = centres[t];
        const float ox[1] = {o.x}, oy[1] = {o.y}, oz[1] = {o.z};
        const float lx[1] = {l.x}, ly[1] = {l.y}, lz[1] = {l.z};
        const double cx[1] = {C.x}, cy[1] = {C.y}, cz[1] = {C.z};
        const float4 ce[1] = {extents[t]};
        const bool live[1] = {k < n};
        float sx[1] = {0.f}, sy[1] = {0.f}, sz[1] = {0.f}, kx[1] = {0.f}, ky[1] = {0.f}, kz[1] = {0.f};
        const std::uint32_t sources = J + 1 < tiles ? kTile : n - (tiles - 1) * kTile;
        source_tile<1, kSafe, kRefine, false, 8>(packed, packed_lo, centres, extents, J, false, sources, live,
                                                 A.eps2, ox, oy, oz, lx, ly, lz, cx, cy, cz, ce, sx, sy, sz, kx,
                                                 ky, kz);
        sums[J][0][k] = static_cast<double>(sx[0]) - static_cast<double>(kx[0]);
        sums[J][1][k] = static_cast<double>(sy[0]) - static_cast<double>(ky[0]);
        sums[J][2][k] = static_cast<double>(sz[0]) - static_cast<double>(kz[0]);
        __syncthreads();
        if (mine) {
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                double total = 0.0;
                for (std::uint32_t w = 0; w < tiles; ++w) total += sums[w][c][at];
                a[c] = A.G * total;
            }
        }
    };
    // One evaluation a turn: what comes before it and after it by the turn's
    // place in its step.
    double x0[3], v0[3], slope_x[3], slope_v[3];
    const std::uint32_t per_step = kRk4 ? 4 : A.substeps, turns = A.mode == 0 ? 1 : A.steps * per_step;
    std::uint32_t p = 0;
#pragma unroll 1
    for (std::uint32_t turn = 0; turn < turns; ++turn) {
        if constexpr (kRk4) {
            // runge_kutta4.cpp:64-139, as rk4_kernel's four operations.
            const double scale = p < 2 ? A.dt / 2 : p == 2 ? A.dt : A.dt / 6;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                if (p == 0) {
                    x0[c] = x[c];
                    v0[c] = slope_x[c] = v[c];
                    slope_v[c] = a[c];
                }
                x[c] = unfused(x0[c], scale, p == 3 ? slope_x[c] : v[c]);
                v[c] = unfused(v0[c], scale, p == 3 ? slope_v[c] : a[c]);
            }
        } else if (A.mode != 0) {
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                v[c] = unfused(v[c], A.kick[p], a[c]);
                x[c] = unfused(x[c], A.drift[p], v[c]);
            }
        }
        field();
        if constexpr (kRk4) {
            const double weight = p < 2 ? 2.0 : 1.0;
            if (p < 3) {
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    slope_x[c] = unfused(slope_x[c], weight, v[c]);
                    slope_v[c] = unfused(slope_v[c], weight, a[c]);
                }
            }
        } else if (A.mode != 0) {
#pragma unroll
            for (int c = 0; c < 3; ++c) v[c] = unfused(v[c], A.kick[p], a[c]);
        }
        p = p + 1 == per_step ? 0 : p + 1;
    }
    if (!mine) return;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        A.a[c][i] = a[c];
        if (A.mode != 0) {
            A.x[c][i] = x[c];
            A.v[c][i] = v[c];
        }
    }
}

// ---- batches: many independent systems in one launch ---------------------
//
// Each system of a batch owns whole tiles (its last tile padded with massless
// lanes), so a tile never mixes systems. tile[t] = {first particle, valid
// count, system, first partial slot}. A work item {target tile, first source
// tile, end source tile, partial slot} is one wave's job; the split of a
// system's source range depends on that system's size only, so its result does
// not depend on which other systems share the batch.

// One wave per tile of the batch.
__global__ __launch_bounds__(64) void batch_prepare(const double* __restrict__ x,
                                                    const double* __restrict__ y,
                                                    const double* __restrict__ z,
                                                    const double* __restrict__ m,
                                                    const std::uint32_t* __restrict__ order,
                                                    const uint4* __restrict__ tile,
                                                    float4* __restrict__ packed,
                                                    float4* __restrict__ packed_lo,
                                                    double4* __restrict__ centres,
                                                    float4* __restrict__ extents) {
    const uint4 T = tile[blockIdx.x];
    const bool valid = threadIdx.x < T.y;
    const std::uint64_t k = static_cast<std::uint64_t>(T.x) + threadIdx.x;
    const std::uint64_t src = valid ? (order != nullptr ? order[k] : k) : 0;
    pack_tile(valid ? x[src] : 0.0, valid ? y[src] : 0.0, valid ? z[src] : 0.0,
              valid ? m[src] : 0.0, valid,
              static_cast<std::uint64_t>(blockIdx.x) * kTile + threadIdx.x, blockIdx.x, packed,
              packed_lo, centres, extents);
}

// Persistent: the grid's W waves take the item list (sorted longest first) in
// strides -- wave w runs items w, w + W, w + 2W, ... -- so every wave starts on a
// long item and finishes on short ones, with no shared counter to contend on.
// Each item writes its own partial slot: the result does not depend on which
// wave ran it.
constexpr int kItemUnroll = 8;

// Eight waves per SIMD: without the hint the scheduler spends registers on
// instruction-level parallelism (87 VGPRs, SGPRs spilled to VGPR lanes).
template<bool kSafe, bool kRefine>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(8, 8))) void direct_items(const float4* __restrict__ packed,
                                                       const float4* __restrict__ packed_lo,
                                                       const double4* __restrict__ centres,
                                                       const float4* __restrict__ extents,
                                                       const uint4* __restrict__ tile,
                                                       const uint4* __restrict__ item,
                                                       std::uint32_t items,
                                                       const float* __restrict__ eps2_of,
                                                       float* __restrict__ partial) {
    const unsigned lane = threadIdx.x & (kTile - 1);
    const std::uint32_t waves = gridDim.x * (kBlock / kTile);
    const std::uint32_t first = __builtin_amdgcn_readfirstlane(blockIdx.x * (kBlock / kTile) + threadIdx.x / kTile);
    for (std::uint32_t next = first; next < items; next += waves) {
        const uint4 it = item[next];
        const uint4 own = tile[it.x];
        const float eps2 = eps2_of[own.z];
        const bool live[1] = {lane < own.y};
        const std::uint32_t k = it.x * kTile + lane;
        const float4 o = packed[k];
        const float4 l = packed_lo[k];
        const double4 c = centres[it.x];
        const float ox[1] = {o.x}, oy[1] = {o.y}, oz[1] = {o.z};
        const float lx[1] = {l.x}, ly[1] = {l.y}, lz[1] = {l.z};
        const double cx[1] = {c.x}, cy[1] = {c.y}, cz[1] = {c.z};
        const float4 ce[1] = {extents[it.x]};
        float sx[1] = {0.f}, sy[1] = {0.f}, sz[1] = {0.f}, kx[1] = {0.f}, ky[1] = {0.f},
              kz[1] = {0.f};
        for (std::uint32_t J = it.y; J < it.z; ++J)
            source_tile<1, kSafe, kRefine, false, kItemUnroll>(packed, packed_lo, centres, extents, J, false,
                                                        tile[J].y, live, eps2,
                                                        ox, oy, oz, lx, ly, lz, cx, cy, cz, ce, sx,
                                                        sy, sz, kx, ky, kz);
        float* out = partial + static_cast<std::size_t>(it.w) * 6 * kTile;
        out[lane] = sx[0];
        out[kTile + lane] = sy[0];
        out[2 * kTile + lane] = sz[0];
        out[3 * kTile + lane] = kx[0];
        out[4 * kTile + lane] = ky[0];
        out[5 * kTile + lane] = kz[0];
    }
}

// The same, kWaves waves an item, for batches of direct systems alone with fewer
// items than the chip holds waves (beside a tree branch that is the longer one and
// then has fewer waves of its own running, a 48-system batch went from 19.7 to
// 20.2 ms; a batch with any tree system, also a small one, takes one wave an
// item): each wave takes every kWaves-th source tile and leaves the tile's run sums in LDS; after each round of kWaves tiles a wave a component
// adds them in tile order, so the sums are the same bits. Alone on its
// SIMD, a wave took some 17 us a source tile, sixteen in a row. Whole
// evaluations of batches of systems of 256 to 4096 particles with one, four and
// eight waves an item, us: 197 items 207, 128, 107; 1212 items 244, 157, 147;
// 1770 items 246, 177, 178; 5023 items 340, 323, 337; 13,720 items 649, 725, 777.
constexpr std::uint32_t kEightWaveItems = 1536;
constexpr std::uint32_t kFourWaveItems = 5120;

template<bool kSafe, bool kRefine, int kWaves>
__global__ __launch_bounds__(64 * kWaves) void direct_items_wide(
    const float4* __restrict__ packed, const float4* __restrict__ packed_lo,
    const double4* __restrict__ centres, const float4* __restrict__ extents,
    const uint4* __restrict__ tile, const uint4* __restrict__ item, std::uint32_t items,
    const float* __restrict__ eps2_of, float* __restrict__ partial) {
    constexpr int kRuns = kTile / kRun;
    static_assert(3 * kRuns >= 6 && kWaves >= 3);
    __shared__ float s_sums[kWaves][3 * kRuns][kTile];  // far: run by run; near: the pair, sums then compensations
    __shared__ std::uint32_t s_near[kWaves];
    const unsigned lane = threadIdx.x & (kTile - 1);
    const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kTile);
    for (std::uint32_t next = blockIdx.x; next < items; next += gridDim.x) {
        const uint4 it = item[next];
        const uint4 own = tile[it.x];
        const float eps2 = eps2_of[own.z];
        const bool live[1] = {lane < own.y};
        const std::uint32_t k = it.x * kTile + lane;
        const float4 o = packed[k];
        const float4 l = packed_lo[k];
        const double4 c = centres[it.x];
        const float ox[1] = {o.x}, oy[1] = {o.y}, oz[1] = {o.z};
        const float lx[1] = {l.x}, ly[1] = {l.y}, lz[1] = {l.z};
        const double cx[1] = {c.x}, cy[1] = {c.y}, cz[1] = {c.z};
        const float4 ce[1] = {extents[it.x]};
        float sum = 0.f, compensation = 0.f;  // component `wave`
        for (std::uint32_t J0 = it.y; J0 < it.z; J0 += kWaves) {
            const std::uint32_t J = J0 + wave;
            if (J < it.z) {
                if (lane == 0) s_near[wave] = 0;
                source_tile_to<1, kSafe, kRefine, false, kItemUnroll>(
                    packed, packed_lo, centres, extents, J, false, tile[J].y, live, eps2, ox, oy, oz, lx, ly, lz,
                    cx, cy, cz, ce,
                    [&](int, int run, float x, float y, float z) {
                        s_sums[wave][3 * run][lane] = x;
                        s_sums[wave][3 * run + 1][lane] = y;
                        s_sums[wave][3 * run + 2][lane] = z;
                    },
                    [&](int, float x, float y, float z, float kx, float ky, float kz) {
                        const float v[6] = {x, y, z, kx, ky, kz};
#pragma unroll
                        for (int u = 0; u < 6; ++u) s_sums[wave][u][lane] = v[u];
                        if (lane == 0) s_near[wave] = 1;
                    });
            }
            __syncthreads();
            if (wave < 3) {
                const std::uint32_t met = min(it.z - J0, static_cast<std::uint32_t>(kWaves));
                for (std::uint32_t w = 0; w < met; ++w) {
                    if (s_near[w] != 0) {
                        kahan_df(s_sums[w][wave][lane], -s_sums[w][3 + wave][lane], sum, compensation);
                    } else {
#pragma unroll
                        for (int run = 0; run < kRuns; ++run) kahan(s_sums[w][3 * run + wave][lane], sum, compensation);
                    }
                }
            }
            __syncthreads();
        }
        if (wave < 3) {
            float* out = partial + static_cast<std::size_t>(it.w) * 6 * kTile;
            out[wave * kTile + lane] = sum;
            out[(3 + wave) * kTile + lane] = compensation;
        }
    }
}

// One thread per particle of the batch (sorted position k): fold its tile's
// slots in split order in FP64, multiply by the system's G, scatter through
// `order`. sys[s] = {first particle, count, first tile, splits}.
__global__ __launch_bounds__(256) void batch_reduce(const float* __restrict__ partial,
                                                    const uint4* __restrict__ sys,
                                                    const uint4* __restrict__ tile,
                                                    const std::uint32_t* __restrict__ seg_of,
                                                    const double* __restrict__ G_of,
                                                    std::uint64_t n,
                                                    const std::uint32_t* __restrict__ order,
                                                    double* __restrict__ ax,
                                                    double* __restrict__ ay,
                                                    double* __restrict__ az) {
    const std::uint64_t k = static_cast<std::uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const std::uint32_t s = seg_of[k];
    const uint4 S = sys[s];
    const std::uint32_t local = static_cast<std::uint32_t>(k) - S.x;
    const std::uint32_t lane = local & (kTile - 1);
    const std::uint32_t first_slot = tile[S.z + local / kTile].w;
    double a0 = 0.0, a1 = 0.0, a2 = 0.0;
    for (std::uint32_t i = 0; i < S.w; ++i) {
        const float* p = partial + static_cast<std::size_t>(first_slot + i) * 6 * kTile + lane;
        a0 += static_cast<double>(p[0]) - static_cast<double>(p[3 * kTile]);
        a1 += static_cast<double>(p[kTile]) - static_cast<double>(p[4 * kTile]);
        a2 += static_cast<double>(p[2 * kTile]) - static_cast<double>(p[5 * kTile]);
    }
    const double G = G_of[s];
    const std::uint64_t dst = order != nullptr ? order[k] : k;
    ax[dst] = G * a0;
    ay[dst] = G * a1;
    az[dst] = G * a2;
}

// ---- pairs: each far tile pair once, applied to both tiles ---------------
//
// The one-sided kernel above spends 12 VALU operations and one v_rsq_f32 on
// every interaction. Gravity is symmetric: the term that pulls target i toward
// source j, scaled by m_i / m_j, pulls j toward i. Evaluating each tile pair
// once for both sides costs 16 VALU and one v_rsq_f32 per PAIR, i.e. 8 VALU and
// half a v_rsq_f32 per interaction:
//
//   * Tiles are grouped into blocks of kStay. A wave owns one block: each lane
//     holds one particle of each of its kStay tiles (the stationary side),
//     with their sums and Kahan compensations in registers.
//   * The wave streams the tiles I before its block (a chunk of them per
//     wave). Lane l loads particle l of I; after every step the streamed
//     particles and their force accumulators move one lane around the wave
//     (DPP wave rotate), so in 64 steps every stationary particle meets every
//     streamed one, and the accumulator of each streamed particle comes home
//     holding its sum over the block's 64 kStay particles.
//   * Separations are FP32 offsets from the tile centres, the stationary
//     offset re-expressed against the streamed tile's centre once per tile
//     (as the one-sided kernel re-expresses its target). Near tile pairs
//     (the mask) are skipped in that pass and get a pass of their own with the
//     one-sided kernel's double-float separation. The pairs inside a block are
//     left to the complement kernel, one-sided.
//   * Stationary side: the 64 terms of one streamed tile summed in FP32, then
//     Kahan-added (compensations in LDS), per item written to its own slot.
//     Streamed side: per step the kStay terms summed, then added to the
//     travelling accumulator, which is flushed every kFlush steps into the
//     particle's FP64 sum in LDS; after the block's 64 steps (and the near
//     passes, which flush the same way) the sums are written per (particle,
//     block) to their own FP64 slots. A fixed-order FP64 fold (pairs_reduce)
//     sums a particle's slots.
//   * Close pairs of the near passes are evaluated in FP64 (close_pair.hpp)
//     and applied to both sides.
//
// Items: block Q >= 1 streams tiles [0, Q kStay) in chunks of S tiles, S a
// divisor of kStay (kStay Q / S chunks) or a multiple of it (s = S / kStay:
// ceil(Q / s) chunks); items are numbered block by block, items_before(Q) of
// them before block Q.
constexpr int kStay = 8;
// Steps between flushes of the streamed side's travelling sums (to LDS).
constexpr int kFlush = 8;

__host__ __device__ inline std::uint32_t pair_chunks(std::uint32_t Q, std::uint32_t S) {
    return (kStay * Q + S - 1) / S;
}

__host__ __device__ inline std::uint64_t pair_items_before(std::uint32_t Q, std::uint32_t S) {
    if (Q == 0) return 0;
    const std::uint64_t q = Q;
    if (S < kStay) return (kStay / S) * q * (q - 1) / 2;
    // sum over q' < Q of ceil(q' / s): q' = a s + r
    const std::uint64_t s = S / kStay, m = q - 1, a = m / s, r = m % s;
    return s * a * (a + 1) / 2 + (a + 1) * r;
}

__host__ __device__ inline std::uint64_t pair_slot(std::uint32_t Q, std::uint32_t tile) {
    // Block Q's streamed tiles [0, Q kStay) after those of blocks 1 .. Q - 1.
    return static_cast<std::uint64_t>(kStay) * Q * (Q - 1) / 2 + tile;
}

// Every lane takes the value of its neighbour, around the whole wave (DPP
// wave_ror:1); 64 rotations bring every value home. wave_rotate moves in
// place; rotate_add(a, t) = rotate(a) + t folds the move into the add.
__device__ __forceinline__ float wave_rotate(float v) {
    const int u = __builtin_bit_cast(int, v);
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(u, u, 0x13C, 0xf, 0xf, false));
}
__device__ __forceinline__ float rotate_add(float a, float t) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, a), 0x13C,
                                                                 0xf, 0xf, false)) + t;
}

// Four waves per SIMD (128 VGPRs): the stationary side holds 13 values per
// tile per lane (offset re-expressed against the streamed tile, mass, the
// streamed tile's partial sums, Kahan sums and compensations), 104 in all.
//
// kEqual: every particle has one mass (the flag the mass pass leaves). The
// masses then leave the pair term -- both sides add inv^3 d, two multiplies
// fewer per pair and no travelling mass -- and the fold multiplies the pairs'
// slots by the common mass.
template<bool kSafe, bool kRefine, bool kEqual>
__device__ __forceinline__ void pairs_item(const float4* __restrict__ packed,
                                           const float4* __restrict__ packed_lo,
                                           const double4* __restrict__ centres,
                                           const std::uint32_t* __restrict__ mask,
                                           std::uint32_t tiles, std::uint32_t words,
                                           std::uint32_t blocks, std::uint32_t S,
                                           std::uint32_t item, float eps2,
                                           float* __restrict__ jpart,
                                           double* __restrict__ ipart,
                                           double* __restrict__ home,
                                           float* __restrict__ comp) {
    // The item's block: the largest Q with pair_items_before(Q) <= item.
    std::uint32_t lo = 1, hi = blocks - 1;
    while (lo < hi) {
        const std::uint32_t mid = (lo + hi + 1) / 2;
        if (pair_items_before(mid, S) <= item) lo = mid;
        else hi = mid - 1;
    }
    const std::uint32_t Q = lo;
    const std::uint32_t chunk = item - static_cast<std::uint32_t>(pair_items_before(Q, S));
    const std::uint32_t t0 = Q * kStay;
    const std::uint32_t i0 = chunk * S;
    const std::uint32_t i1 = min(i0 + S, t0);
    const unsigned lane = threadIdx.x & (kTile - 1);

    // Stationary tiles past the last (a partial last block) repeat the last
    // tile massless: they pull nothing and their sums are never read.
    // home: the wave's streamed-side sums by particle, in FP64 (LDS); the
    // travelling accumulators are added there every kFlush steps (each lane to
    // the slot of the particle it holds then), so no FP32 sum runs longer than
    // kFlush steps of kStay terms. comp: this lane's stationary-side Kahan
    // compensations (LDS, [(3 r + c) kTile]), touched once per streamed tile,
    // so that the far loop keeps its registers.

    // An FP32 instruction with a scalar operand issues at half the rate of one
    // that reads only vector registers (measured: 4.1 against 2.4 cycles a
    // wave), and eps^2 enters every pair: keep it in a vector register.
    asm volatile("" : "+v"(eps2));
    float m[kStay], sx[kStay], sy[kStay], sz[kStay];
#pragma unroll
    for (int r = 0; r < kStay; ++r) {
        if constexpr (kEqual) {
            m[r] = 1.f;
        } else {
            m[r] = t0 + r < tiles ? packed[static_cast<std::size_t>(min(t0 + r, tiles - 1)) * kTile + lane].w : 0.f;
        }
        sx[r] = sy[r] = sz[r] = 0.f;
        comp[(3 * r) * kTile] = comp[(3 * r + 1) * kTile] = comp[(3 * r + 2) * kTile] = 0.f;
    }
    // Adds (h, l) to stationary sum (s, compensation of component c of tile r).
    auto stay_add = [&](int r, int c, float h, float l, float& sum) {
        float k = comp[(3 * r + c) * kTile];
        kahan_df(h, l, sum, k);
        comp[(3 * r + c) * kTile] = k;
    };

    for (std::uint32_t I = i0; I < i1; ++I) {
        const double4 CI = centres[I];
        const float4 qi = packed[static_cast<std::size_t>(I) * kTile + lane];
        float xi = qi.x, yi = qi.y, zi = qi.z, mi = kEqual ? 1.f : qi.w;
        std::uint32_t near = 0;
        float wx[kStay], wy[kStay], wz[kStay];
        // The stationary offsets and centres are re-read for every streamed
        // tile (cache hits) rather than held: the index is hidden from the
        // compiler, which would otherwise keep 9 kStay more VGPRs live.
        std::uint32_t first = t0;
        asm volatile("" : "+s"(first));
#pragma unroll
        for (int r = 0; r < kStay; ++r) {
            const std::uint32_t tile = min(first + r, tiles - 1);
            near |= ((mask[static_cast<std::size_t>(tile) * words + I / 32] >> (I & 31u)) & 1u) << r;
            const double4 C = centres[tile];
            const float4 o = packed[static_cast<std::size_t>(tile) * kTile + lane];
            // The stationary offset re-expressed relative to the streamed
            // tile's centre: the FP64 difference rounded once.
            wx[r] = static_cast<float>(static_cast<double>(o.x) - (CI.x - C.x));
            wy[r] = static_cast<float>(static_cast<double>(o.y) - (CI.y - C.y));
            wz[r] = static_cast<float>(static_cast<double>(o.z) - (CI.z - C.z));
        }
        float px[kStay], py[kStay], pz[kStay];
#pragma unroll
        for (int r = 0; r < kStay; ++r) px[r] = py[r] = pz[r] = 0.f;
        float ax = 0.f, ay = 0.f, az = 0.f;
        // d = x_i - x_j; j gains m_i d / r^3, i gains -m_j d / r^3 (the
        // travelling sums hold its negative until they are flushed: the same
        // bits, and the two-operand accumulate encoding for both sides).
        auto pair = [&](int r, float& tx, float& ty, float& tz) {
            const float dx = xi - wx[r], dy = yi - wy[r], dz = zi - wz[r];
            float r2 = __builtin_fmaf(dx, dx, eps2);
            r2 = __builtin_fmaf(dy, dy, r2);
            r2 = __builtin_fmaf(dz, dz, r2);
            const float inv3 = inv_cubed<kSafe, kRefine>(r2);
            const float fj = kEqual ? inv3 : mi * inv3, fi = kEqual ? inv3 : m[r] * inv3;
            px[r] = __builtin_fmaf(fj, dx, px[r]);
            py[r] = __builtin_fmaf(fj, dy, py[r]);
            pz[r] = __builtin_fmaf(fj, dz, pz[r]);
            tx = __builtin_fmaf(fi, dx, tx);
            ty = __builtin_fmaf(fi, dy, ty);
            tz = __builtin_fmaf(fi, dz, tz);
        };
        auto advance = [&](float tx, float ty, float tz) {
            ax = rotate_add(ax, tx);
            ay = rotate_add(ay, ty);
            az = rotate_add(az, tz);
            xi = wave_rotate(xi);
            yi = wave_rotate(yi);
            zi = wave_rotate(zi);
            if constexpr (!kEqual) mi = wave_rotate(mi);
        };
        // After step s the accumulator on lane l belongs to streamed particle
        // (l - s) mod 64. Flushes after steps kFlush - 1, 2 kFlush - 1, ...
        auto flush_streamed = [&](std::uint32_t last_step) {
            const unsigned slot = (lane - last_step) & (kTile - 1);
            if (last_step == kFlush - 1) {
                home[slot] = -ax;
                home[kTile + slot] = -ay;
                home[2 * kTile + slot] = -az;
            } else {
                atomicAdd(&home[slot], static_cast<double>(-ax));
                atomicAdd(&home[kTile + slot], static_cast<double>(-ay));
                atomicAdd(&home[2 * kTile + slot], static_cast<double>(-az));
            }
            ax = ay = az = 0.f;
        };
        // Runs of kFlush steps, each followed by a flush of the streamed sums.
#pragma unroll 1
        for (std::uint32_t run = 0; run < kTile; run += kFlush) {
            if (near == 0) {
#pragma unroll 4
                for (int u = 0; u < kFlush; ++u) {
                    float tx = 0.f, ty = 0.f, tz = 0.f;
#pragma unroll
                    for (int r = 0; r < kStay; ++r) pair(r, tx, ty, tz);
                    advance(tx, ty, tz);
                }
            } else {
#pragma unroll 4
                for (int u = 0; u < kFlush; ++u) {
                    float tx = 0.f, ty = 0.f, tz = 0.f;
                    // The flags as bits of one scalar, hidden from the compiler,
                    // which would otherwise keep each as a lane mask and spend
                    // two vector instructions a pair on testing it.
                    std::uint32_t flags = near;
                    asm volatile("" : "+s"(flags));
#pragma unroll
                    for (int r = 0; r < kStay; ++r) {
                        if (((flags >> r) & 1u) == 0) pair(r, tx, ty, tz);
                    }
                    advance(tx, ty, tz);
                }
            }
            flush_streamed(run + kFlush - 1);
        }
#pragma unroll
        for (int r = 0; r < kStay; ++r) {
            stay_add(r, 0, px[r], 0.f, sx[r]);
            stay_add(r, 1, py[r], 0.f, sy[r]);
            stay_add(r, 2, pz[r], 0.f, sz[r]);
        }
        if (near != 0) {
            // Near stationary tiles, one pass of 64 steps each: the one-sided
            // kernel's double-float separation (the streamed offset (hi, lo)
            // against the stationary position taken relative to the streamed
            // tile's centre in FP64 and split into (hi, lo)); both sides sum
            // runs of kFlush terms, the stationary runs Kahan-added, the
            // streamed runs added to the FP64 slots. Close pairs are marked
            // and evaluated afterwards in FP64.
            const float4 il = packed_lo[static_cast<std::size_t>(I) * kTile + lane];
            float xl = il.x, yl = il.y, zl = il.z;
            // The stationary tiles' centres and offsets are read again here
            // (cache hits), from an index hidden afresh: otherwise the
            // compiler keeps the far pass's FP64 centre differences alive
            // through the far loop, and they spill on every streamed tile.
            std::uint32_t again = t0;
            asm volatile("" : "+s"(again));
#pragma unroll
            for (int r = 0; r < kStay; ++r) {
                if (((near >> r) & 1u) == 0) continue;
                const std::uint32_t tile = min(again + r, tiles - 1);
                const double4 C = centres[tile];
                const float4 o = packed[static_cast<std::size_t>(tile) * kTile + lane];
                const float4 l = packed_lo[static_cast<std::size_t>(tile) * kTile + lane];
                const double t[3] = {(static_cast<double>(o.x) + l.x) - (CI.x - C.x),
                                     (static_cast<double>(o.y) + l.y) - (CI.y - C.y),
                                     (static_cast<double>(o.z) + l.z) - (CI.z - C.z)};
                float th[3], tl[3];
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    th[c] = static_cast<float>(t[c]);
                    tl[c] = static_cast<float>(t[c] - th[c]);
                }
                const float lim = close_limit(C.w, CI.w, eps2);
                const float mr = m[r];
                std::uint64_t close = 0;  // bit s: this lane's pair at step s is close
                float qx = 0.f, qy = 0.f, qz = 0.f;  // stationary run
                ax = ay = az = 0.f;                  // streamed run (travelling)
#pragma unroll 1
                for (std::uint32_t run = 0; run < kTile; run += kFlush) {
#pragma unroll 2
                    for (std::uint32_t u = 0; u < kFlush; ++u) {
                        const std::uint32_t step = run + u;
                        const float dx = (xi - th[0]) + (xl - tl[0]);
                        const float dy = (yi - th[1]) + (yl - tl[1]);
                        const float dz = (zi - th[2]) + (zl - tl[2]);
                        float r2 = __builtin_fmaf(dx, dx, eps2);
                        r2 = __builtin_fmaf(dy, dy, r2);
                        r2 = __builtin_fmaf(dz, dz, r2);
                        const bool near_pair = r2 < lim && (!kSafe || r2 > 0.f);
                        close |= near_pair ? std::uint64_t{1} << step : std::uint64_t{0};
                        const float inv3 = near_pair ? 0.f : inv_cubed<kSafe, kRefine>(r2);
                        const float fj = kEqual ? inv3 : mi * inv3, fi = kEqual ? inv3 : mr * inv3;
                        qx = __builtin_fmaf(fj, dx, qx);
                        qy = __builtin_fmaf(fj, dy, qy);
                        qz = __builtin_fmaf(fj, dz, qz);
                        ax = rotate_add(ax, -fi * dx);
                        ay = rotate_add(ay, -fi * dy);
                        az = rotate_add(az, -fi * dz);
                        xi = wave_rotate(xi);
                        yi = wave_rotate(yi);
                        zi = wave_rotate(zi);
                        if constexpr (!kEqual) mi = wave_rotate(mi);
                        xl = wave_rotate(xl);
                        yl = wave_rotate(yl);
                        zl = wave_rotate(zl);
                    }
                    const unsigned slot = (lane - (run + kFlush - 1)) & (kTile - 1);
                    atomicAdd(&home[slot], static_cast<double>(ax));
                    atomicAdd(&home[kTile + slot], static_cast<double>(ay));
                    atomicAdd(&home[2 * kTile + slot], static_cast<double>(az));
                    ax = ay = az = 0.f;
                    stay_add(r, 0, qx, 0.f, sx[r]);
                    stay_add(r, 1, qy, 0.f, sy[r]);
                    stay_add(r, 2, qz, 0.f, sz[r]);
                    qx = qy = qz = 0.f;
                }
                // Close pairs: at step s this lane met streamed particle
                // (lane - s) mod 64, read back here by index.
                const double ah[3] = {static_cast<double>(th[0]) + static_cast<double>(tl[0]),
                                      static_cast<double>(th[1]) + static_cast<double>(tl[1]),
                                      static_cast<double>(th[2]) + static_cast<double>(tl[2])};
                while (close != 0) {
                    const unsigned step = __builtin_ctzll(close);
                    close &= close - 1;
                    const unsigned p = (lane - step) & (kTile - 1);
                    const std::size_t k = static_cast<std::size_t>(I) * kTile + p;
                    const float4 b = packed[k];
                    const float4 bl4 = packed_lo[k];
                    const float bh[3] = {b.x, b.y, b.z}, bl[3] = {bl4.x, bl4.y, bl4.z};
                    double G[3];
                    close_pair(ah, bh, bl, eps2, G);
                    const double mb = kEqual ? 1.0 : static_cast<double>(b.w);
                    const double ms = static_cast<double>(mr);
                    float h, l;
                    split(mb * G[0], h, l);
                    stay_add(r, 0, h, l, sx[r]);
                    split(mb * G[1], h, l);
                    stay_add(r, 1, h, l, sy[r]);
                    split(mb * G[2], h, l);
                    stay_add(r, 2, h, l, sz[r]);
                    atomicAdd(&home[p], -(ms * G[0]));
                    atomicAdd(&home[kTile + p], -(ms * G[1]));
                    atomicAdd(&home[2 * kTile + p], -(ms * G[2]));
                }
            }
        }
        // The streamed particles are home: each lane's sum over the block is in
        // its FP64 slot.
        double* out = ipart + pair_slot(Q, I) * 3 * kTile;
        out[lane] = home[lane];
        out[kTile + lane] = home[kTile + lane];
        out[2 * kTile + lane] = home[2 * kTile + lane];
    }
    float* out = jpart + static_cast<std::size_t>(item) * 6 * kStay * kTile;
    constexpr int kRow = kStay * kTile;
#pragma unroll
    for (int r = 0; r < kStay; ++r) {
        const unsigned k = r * kTile + lane;
        out[k] = sx[r];
        out[kRow + k] = sy[r];
        out[2 * kRow + k] = sz[r];
        out[3 * kRow + k] = comp[(3 * r) * kTile];
        out[4 * kRow + k] = comp[(3 * r + 1) * kTile];
        out[5 * kRow + k] = comp[(3 * r + 2) * kTile];
    }
}

// One launch per mass case, both enqueued; the mass pass's flag (uniform[0] >
// 0: every particle's mass) lets one of them run and the other exit at once,
// so the host never waits for the flag and each case keeps its own registers.
template<bool kSafe, bool kRefine, bool kEqual>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4, 4))) void direct_pairs(const float4* __restrict__ packed,
                                                       const float4* __restrict__ packed_lo,
                                                       const double4* __restrict__ centres,
                                                       const std::uint32_t* __restrict__ mask,
                                                       std::uint32_t tiles, std::uint32_t words,
                                                       std::uint32_t blocks, std::uint32_t S,
                                                       std::uint32_t items, float eps2,
                                                       const float* __restrict__ uniform,
                                                       float* __restrict__ jpart,
                                                       double* __restrict__ ipart) {
    if ((uniform[0] > 0.f) != kEqual) return;
    const std::uint32_t item =
        __builtin_amdgcn_readfirstlane(blockIdx.x * (kBlock / kTile) + threadIdx.x / kTile);
    if (item >= items) return;
    __shared__ double flushed[kBlock / kTile][3][kTile];
    __shared__ float compensation[kBlock / kTile][3 * kStay][kTile];
    const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kTile);
    double* const home = &flushed[wave][0][0];
    float* const comp = &compensation[wave][0][threadIdx.x & (kTile - 1)];
    pairs_item<kSafe, kRefine, kEqual>(packed, packed_lo, centres, mask, tiles, words, blocks, S,
                                       item, eps2, jpart, ipart, home, comp);
}

// What the pairs kernel leaves out: the pairs inside each block, one-sided.
// One wave per target tile over the tiles of its own block (near flags from
// the mask); sums and compensations to cpart[6][npad].
template<bool kSafe, bool kRefine>
__global__ __launch_bounds__(kBlock) void direct_complement(const float4* __restrict__ packed,
                                                            const float4* __restrict__ packed_lo,
                                                            const double4* __restrict__ centres,
                                                            const float4* __restrict__ extents,
                                                            const std::uint32_t* __restrict__ mask,
                                                            std::uint32_t tiles, std::uint32_t words,
                                                            float eps2, float* __restrict__ cpart) {
    const std::uint32_t t =
        __builtin_amdgcn_readfirstlane(blockIdx.x * (kBlock / kTile) + threadIdx.x / kTile);
    if (t >= tiles) return;
    const unsigned lane = threadIdx.x & (kTile - 1);
    const std::size_t k = static_cast<std::size_t>(t) * kTile + lane;
    const float4 o = packed[k];
    const float4 l = packed_lo[k];
    const double4 c = centres[t];
    const float ox[1] = {o.x}, oy[1] = {o.y}, oz[1] = {o.z};
    const float lx[1] = {l.x}, ly[1] = {l.y}, lz[1] = {l.z};
    const double cx[1] = {c.x}, cy[1] = {c.y}, cz[1] = {c.z};
    const float4 ce[1] = {extents[t]};
    const bool live[1] = {true};
    float sx[1] = {0.f}, sy[1] = {0.f}, sz[1] = {0.f}, kx[1] = {0.f}, ky[1] = {0.f}, kz[1] = {0.f};
    const std::uint32_t* row = mask + static_cast<std::size_t>(t) * words;
    const std::uint32_t b0 = t / kStay * kStay, b1 = min(b0 + kStay, tiles);
    for (std::uint32_t J = b0; J < b1; ++J) {
        const bool near = ((row[J / 32] >> (J & 31u)) & 1u) != 0;
        source_tile<1, kSafe, kRefine, true>(packed, packed_lo, centres, extents, J, near, kTile, live, eps2, ox,
                                             oy, oz, lx, ly, lz, cx, cy, cz, ce, sx, sy, sz, kx, ky, kz);
    }
    const std::size_t np = static_cast<std::size_t>(tiles) * kTile;
    cpart[k] = sx[0];
    cpart[np + k] = sy[0];
    cpart[2 * np + k] = sz[0];
    cpart[3 * np + k] = kx[0];
    cpart[4 * np + k] = ky[0];
    cpart[5 * np + k] = kz[0];
}

// A particle's slots in a fixed order, in FP64: its block's items (sum minus
// compensation), its tile's streamed sums for every later block, the
// complement; times G, scattered through `order`.
__global__ __launch_bounds__(256) void pairs_reduce(const float* __restrict__ jpart,
                                                    const double* __restrict__ ipart,
                                                    const float* __restrict__ cpart,
                                                    const float* __restrict__ uniform,
                                                    std::uint32_t tiles, std::uint32_t blocks,
                                                    std::uint32_t S, std::uint64_t n,
                                                    const std::uint32_t* __restrict__ order,
                                                    double G, double* __restrict__ ax,
                                                    double* __restrict__ ay,
                                                    double* __restrict__ az, FusedKick kick) {
    const std::uint64_t k = static_cast<std::uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const std::uint32_t t = static_cast<std::uint32_t>(k / kTile), lane = static_cast<std::uint32_t>(k % kTile);
    const std::uint32_t P = t / kStay, r = t % kStay;
    constexpr std::size_t kRow = kStay * kTile;
    double a0 = 0.0, a1 = 0.0, a2 = 0.0;
    const std::uint64_t first = pair_items_before(P, S);
    const std::uint32_t count = pair_chunks(P, S);
#pragma unroll 4
    for (std::uint32_t u = 0; u < count; ++u) {
        const float* p = jpart + (first + u) * 6 * kRow + r * kTile + lane;
        a0 += static_cast<double>(p[0]) - static_cast<double>(p[3 * kRow]);
        a1 += static_cast<double>(p[kRow]) - static_cast<double>(p[4 * kRow]);
        a2 += static_cast<double>(p[2 * kRow]) - static_cast<double>(p[5 * kRow]);
    }
#pragma unroll 4
    for (std::uint32_t Q = P + 1; Q < blocks; ++Q) {
        const double* p = ipart + pair_slot(Q, t) * 3 * kTile + lane;
        a0 += p[0];
        a1 += p[kTile];
        a2 += p[2 * kTile];
    }
    // The pairs kernel's slots leave out a common mass; the complement's not.
    const double scale = uniform[0] > 0.f ? static_cast<double>(uniform[0]) : 1.0;
    a0 *= scale;
    a1 *= scale;
    a2 *= scale;
    const std::size_t np = static_cast<std::size_t>(tiles) * kTile;
    a0 += static_cast<double>(cpart[k]) - static_cast<double>(cpart[3 * np + k]);
    a1 += static_cast<double>(cpart[np + k]) - static_cast<double>(cpart[4 * np + k]);
    a2 += static_cast<double>(cpart[2 * np + k]) - static_cast<double>(cpart[5 * np + k]);
    const std::uint64_t dst = order != nullptr ? order[k] : k;
    store_field(dst, G * a0, G * a1, G * a2, ax, ay, az, kick);
}

template<int R, int kPerSimd>
void launch_fold(orr_ctx* ctx, bool safe, bool refine, dim3 grid, const float4* packed,
                 const float4* packed_lo, const double4* centres, const float4* extents,
                 std::uint32_t tiles, std::uint32_t per_group, std::uint32_t groups, float eps2,
                 double* partial, const FieldOut& out) {
    auto kernel = safe ? (refine ? direct_fold<R, true, true, kPerSimd> : direct_fold<R, true, false, kPerSimd>)
                       : (refine ? direct_fold<R, false, true, kPerSimd> : direct_fold<R, false, false, kPerSimd>);
    hipLaunchKernelGGL(kernel, grid, dim3(kBlock), 0, ctx->stream, packed, packed_lo, centres, extents, tiles, per_group, groups, eps2, partial, out);
    ORR_LAUNCHED("direct_fold");
}

// The pairs path's mask of near tile pairs holds up to this many tiles (128 MiB).
constexpr std::uint32_t kMaskTiles = 32768;

// The pairs path: blocks of kStay tiles, chunks of S tiles per item, slot
// counts. Taken when the mask exists, there are at least four blocks (pair
// mode 1: at least kPairMinTiles tiles) and the streamed-side slots (3 doubles
// per particle and later block) fit in 16 GiB; otherwise, or when configured
// off, the one-sided kernel runs.
struct PairPlan {
    bool use = false;
    std::uint32_t blocks = 0, S = kStay;  // S: streamed tiles per item
    std::uint64_t items = 0, slots = 0;
    std::size_t jpart_floats = 0, ipart_doubles = 0;
};

// The streamed-side slots grow as N^2 (one per tile and later block), and so
// does the kernel's work: their write and fold cost a fixed few per cent of an
// evaluation at any N. 16 GiB of the 288 GB HBM takes the pairs path to
// 856,064 particles.
constexpr std::size_t kPairSlotBytes = std::size_t{1} << 34;
// Items wanted per evaluation: some sixteen rounds of the 4096 resident waves.
// Short items balance the items that carry near passes (measured at
// N = 262,144: 16384 items 14.8 ms, 32768 14.0, 65536 13.7, 131072 13.5 ms,
// the last with twice the stationary-side slots).
constexpr std::uint64_t kPairItems = 65536;

// From this many tiles on pair mode 1 takes the pairs path, pair mode 3 wherever
// it applies. Evaluations one-sided and in pairs, us, Plummer spheres of equal
// masses (and of spread ones in pairs; one-sided they are the same): 16,384 225 and 305
// (323), 24,576 366 and 372 (418), 32,768 539 and 489 (542), 36,000 544 and 612
// (607), 40,960 735 and 636 (684), 44,992 788 and 704 (763), 49,152 966 and 809
// (877), 65,536 1602 and 1223 (1348). Two-disc collisions of 30,000 427 and 617,
// 40,960 975 and 763, 49,152 1213 and 889. The two cross between 32,768 and 40,960
// particles, depending on the masses and on how the count falls on whole waves;
// the line, set for an earlier one-sided kernel, lies somewhat above.
constexpr std::uint32_t kPairMinTiles = 704;

PairPlan pair_plan(std::uint32_t tiles, bool masked, int mode) {
    PairPlan p;
    if ((mode != 1 && mode != 3) || !masked) return p;
    if (mode == 1 && tiles < kPairMinTiles) return p;
    p.blocks = (tiles + kStay - 1) / kStay;
    if (p.blocks < 4) return p;
    p.slots = pair_slot(p.blocks, 0);
    p.ipart_doubles = static_cast<std::size_t>(p.slots) * 3 * kTile;
    if (p.ipart_doubles * sizeof(double) > kPairSlotBytes) return p;
    // About B^2 kStay / (2 S) items: S = kStay s for large systems, down to
    // kStay / 4 for small ones (more, shorter items; below that the
    // stationary-side slots outgrow the work).
    const std::uint64_t B = p.blocks;
    const std::uint64_t s = B * B / (2 * kPairItems);
    p.S = s >= 1 ? static_cast<std::uint32_t>(s) * kStay
                 : (B * B * 2 >= kPairItems ? kStay / 2 : kStay / 4);
    p.items = pair_items_before(p.blocks, p.S);
    p.jpart_floats = static_cast<std::size_t>(p.items) * 6 * kStay * kTile;
    p.use = true;
    return p;
}

// The complement (one wave per tile: too few waves to fill the device below a
// few hundred thousand particles, and latency-bound there) runs on the
// context's second stream, beside the pairs kernel; the main stream waits for
// it before the fold.
template<bool kSafe, bool kRefine>
void launch_pairs(orr_ctx* ctx, const PairPlan& plan, const float4* packed, const float4* packed_lo,
                  const double4* centres, const float4* extents, const std::uint32_t* mask,
                  std::uint32_t tiles, std::uint32_t words, float eps2, const float* uniform,
                  float* jpart, double* ipart, float* cpart) {
    constexpr std::uint32_t kWaves = kBlock / kTile;
    const std::uint32_t items = static_cast<std::uint32_t>(plan.items);
    ensure_aux(ctx);
    ORR_HIP(hipEventRecord(ctx->aux_fork, ctx->stream));
    ORR_HIP(hipStreamWaitEvent(ctx->aux, ctx->aux_fork, 0));
    hipLaunchKernelGGL((direct_complement<kSafe, kRefine>), dim3((tiles + kWaves - 1) / kWaves),
                       dim3(kBlock), 0, ctx->aux, packed, packed_lo, centres, extents, mask, tiles,
                       words, eps2, cpart);
    ORR_LAUNCHED("direct_complement");
    ORR_HIP(hipEventRecord(ctx->aux_join, ctx->aux));
    hipLaunchKernelGGL((direct_pairs<kSafe, kRefine, true>), dim3((items + kWaves - 1) / kWaves),
                       dim3(kBlock), 0, ctx->stream, packed, packed_lo, centres, mask, tiles, words, plan.blocks,
                       plan.S, items, eps2, uniform, jpart, ipart);
    ORR_LAUNCHED("direct_pairs");
    hipLaunchKernelGGL((direct_pairs<kSafe, kRefine, false>), dim3((items + kWaves - 1) / kWaves),
                       dim3(kBlock), 0, ctx->stream, packed, packed_lo, centres, mask, tiles, words, plan.blocks,
                       plan.S, items, eps2, uniform, jpart, ipart);
    ORR_LAUNCHED("direct_pairs");
    ORR_HIP(hipStreamWaitEvent(ctx->stream, ctx->aux_join, 0));
}

}  // namespace

namespace {

// The shape of one single-system evaluation: tiles, one-sided launch grid,
// near mask and pairs plan, as direct_enqueue chooses them for the context's
// configuration.
struct DirectShape {
    std::uint32_t tiles = 0, npad = 0, words = 0;
    // One-sided: target tiles a wave, blocks of targets, source tiles a group
    // (summed in FP32 with one compensation) and groups, blocks a target.
    int R = 1;
    std::uint32_t blocks_i = 0, per_split = 0, splits = 0, blocks_j = 1;
    bool masked = false;  // pairs: the near mask fits
    PairPlan plan;
};

// One-sided launch: blocks of four targets, kFoldWaves waves while every block
// has a group. Near tiles make waves uneven, so many rounds of waves: kernel and
// fold at N = 20,001 279 us at 8192 waves, 206 at 32,768, 204 at 65,536, 213 at
// 131,072; at 32,768 745, 596, 554 and 567 us.
constexpr std::uint32_t kFoldWaves = 65536;

void one_sided_shape(DirectShape& d) {
    const std::uint32_t waves = d.blocks_i * (kBlock / kTile);
    d.blocks_j = std::max(1u, std::min((kFoldWaves + waves - 1) / waves, d.splits));
}

DirectShape direct_shape(const orr_ctx* ctx, std::uint64_t n) {
    if (n > (std::uint64_t{1} << 31)) fail(ORR_ERR_LENGTH, "direct: more than 2^31 particles");
    DirectShape d;
    d.tiles = static_cast<std::uint32_t>((n + kTile - 1) / kTile);
    d.npad = d.tiles * kTile;
    // Up to four tiles a block has a wave for each: more targets a lane would be the
    // last tile over again (64 particles, evaluation: four a lane 47.6 us, one 23.8;
    // 256: 72.6 and 43.4).
    d.R = d.tiles <= kBlock / kTile ? 1 : ctx->direct_targets_per_lane;
    d.blocks_i = (d.npad + kBlock * d.R - 1) / (kBlock * d.R);
    // Source tiles summed together in FP32: `block_target` blocks of four target
    // tiles times groups, each group at least one tile.
    const std::uint32_t want = ctx->direct_block_target;
    std::uint32_t splits = std::max<std::uint32_t>(1, (want + d.blocks_i - 1) / d.blocks_i);
    splits = std::min(splits, d.tiles);
    d.per_split = (d.tiles + splits - 1) / splits;
    d.splits = (d.tiles + d.per_split - 1) / d.per_split;
    d.masked = d.tiles <= kMaskTiles;
    d.words = (d.tiles + 31) / 32;
    d.plan = pair_plan(d.tiles, d.masked, ctx->direct_pair_mode);
    one_sided_shape(d);
    return d;
}

// Device buffers of one evaluation (DirectShape's sizes).
struct DirectBuffers {
    float4* packed = nullptr;     // [npad] {o, m}, then [npad] residuals
    double4* centres = nullptr;   // [tiles], then extents [tiles], mass ranges [tiles], uniform
    void* partials = nullptr;     // one-sided: FP64 [blocks_j][3][npad]; pairs: slots
    std::uint32_t* mask = nullptr;  // [tiles][words] when masked
};

std::size_t packed_buffer_bytes(const DirectShape& d) { return 2 * sizeof(float4) * d.npad; }
std::size_t centre_buffer_bytes(const DirectShape& d) {
    return (sizeof(double4) + sizeof(float4) + sizeof(float2)) * d.tiles + 16;
}
std::size_t partial_buffer_bytes(const DirectShape& d) {
    const std::size_t cpart_floats = 6 * static_cast<std::size_t>(d.npad);
    return d.plan.use ? sizeof(double) * d.plan.ipart_doubles +
                            sizeof(float) * (d.plan.jpart_floats + cpart_floats)
                      : (d.blocks_j > 1 ? sizeof(double) * 3 * static_cast<std::size_t>(d.npad) * d.blocks_j : 0);
}
std::size_t mask_buffer_bytes(const DirectShape& d) {
    return d.plan.use ? sizeof(std::uint32_t) * static_cast<std::size_t>(d.words) * d.tiles : 0;
}

// Every launch of one evaluation on given buffers; phases timed when `timed`.
void direct_launch(orr_ctx* ctx, const orr_direct_args& a, const std::uint32_t* order,
                   const DirectShape& d, const DirectBuffers& buf, bool timed,
                   const FusedKick& kick = FusedKick{}) {
    const std::uint64_t n = a.count;
    const std::uint32_t tiles = d.tiles, npad = d.npad, words = d.words;
    const PairPlan& plan = d.plan;
    float4* packed = buf.packed;
    float4* packed_lo = packed + npad;
    double4* centres = buf.centres;
    float4* extents = reinterpret_cast<float4*>(centres + tiles);
    float2* mass_range = reinterpret_cast<float2*>(extents + tiles);
    float* uniform = reinterpret_cast<float*>(mass_range + tiles);
    std::uint32_t* mask = buf.mask;
    {
        PhaseTimer t(ctx, kDirectPrepare, timed);
        hipLaunchKernelGGL(direct_prepare, dim3(tiles), dim3(kTile), 0, ctx->stream, a.x, a.y, a.z,
                           a.m, order, n, packed, packed_lo, centres, extents, mass_range);
        ORR_LAUNCHED("direct_prepare");
        if (plan.use) {
            hipLaunchKernelGGL(mass_uniform, dim3(1), dim3(256), 0, ctx->stream, mass_range, tiles,
                               ctx->direct_equal_masses == 1 ? 1 : 0, uniform);
            ORR_LAUNCHED("mass_uniform");
            hipLaunchKernelGGL(near_mask, dim3((tiles + kMaskRows - 1) / kMaskRows), dim3(256), 0,
                               ctx->stream, centres, extents, tiles, words, mask);
            ORR_LAUNCHED("near_mask");
        }
    }
    const float eps2 = static_cast<float>(a.softening_squared);
    const bool safe = !(a.softening_squared > 0);
    const bool refine = ctx->direct_refine != 0;
    if (plan.use) {
        // Doubles first: every part stays aligned to its type.
        double* ipart = static_cast<double*>(buf.partials);
        float* jpart = reinterpret_cast<float*>(ipart + plan.ipart_doubles);
        float* cpart = jpart + plan.jpart_floats;
        {
            PhaseTimer t(ctx, kDirectKernel, timed);
            auto launch = safe ? (refine ? launch_pairs<true, true> : launch_pairs<true, false>)
                               : (refine ? launch_pairs<false, true> : launch_pairs<false, false>);
            launch(ctx, plan, packed, packed_lo, centres, extents, mask, tiles, words, eps2, uniform,
                   jpart, ipart, cpart);
        }
        {
            PhaseTimer t(ctx, kDirectReduce, timed);
            const std::uint32_t blocks = static_cast<std::uint32_t>((n + 255) / 256);
            hipLaunchKernelGGL(pairs_reduce, dim3(blocks), dim3(256), 0, ctx->stream, jpart, ipart,
                               cpart, uniform, tiles, plan.blocks, plan.S, n, order,
                               a.gravitational_constant, a.ax, a.ay, a.az, kick);
            ORR_LAUNCHED("pairs_reduce");
        }
        return;
    }
    FieldOut out;
    out.n = n;
    out.order = order;
    out.G = a.gravitational_constant;
    out.ax = a.ax;
    out.ay = a.ay;
    out.az = a.az;
    out.kick = kick;
    double* const partial = static_cast<double*>(buf.partials);
    {
        PhaseTimer t(ctx, kDirectKernel, timed);
        const dim3 grid(d.blocks_i, d.blocks_j);
        auto launch = d.R == 4   ? launch_fold<4, 1>
                      : d.R == 2 ? launch_fold<2, 1>
                      : order != nullptr && d.tiles >= kFoldEightTiles ? launch_fold<1, 8> : launch_fold<1, 1>;
        launch(ctx, safe, refine, grid, packed, packed_lo, centres, extents, tiles, d.per_split, d.splits,
               eps2, partial, out);
    }
    if (d.blocks_j > 1) {
        PhaseTimer t(ctx, kDirectReduce, timed);
        hipLaunchKernelGGL(direct_reduce, dim3(tiles), dim3(kTile), 0, ctx->stream, partial, d.blocks_j,
                           tiles, out);
        ORR_LAUNCHED("direct_reduce");
    }
}

}  // namespace

void direct_enqueue(orr_ctx* ctx, const orr_direct_args& a, const std::uint32_t* order,
                    const FusedKick& kick) {
    if (a.count == 0) return;
    const DirectShape d = direct_shape(ctx, a.count);
    ctx->direct_packed.reserve(packed_buffer_bytes(d));
    ctx->direct_centres.reserve(centre_buffer_bytes(d));
    ctx->direct_partials.reserve(partial_buffer_bytes(d));
    ctx->direct_near.reserve(mask_buffer_bytes(d));
    DirectBuffers buf;
    buf.packed = ctx->direct_packed.as<float4>();
    buf.centres = ctx->direct_centres.as<double4>();
    buf.partials = ctx->direct_partials.ptr;
    buf.mask = ctx->direct_near.as<std::uint32_t>();
    direct_launch(ctx, a, order, d, buf, true, kick);
}

namespace {
std::size_t packed_bytes(std::uint64_t tiles) { return 2 * sizeof(float4) * kTile * tiles; }
std::size_t centre_bytes(std::uint64_t tiles) { return (sizeof(double4) + sizeof(float4)) * tiles; }
std::size_t slot_bytes(std::uint64_t slots) { return sizeof(float) * 6 * kTile * slots; }
}  // namespace

std::size_t direct_batch_bytes(std::uint64_t tiles, std::uint64_t slots) {
    return packed_bytes(tiles) + centre_bytes(tiles) + slot_bytes(slots);
}

namespace {

// Whether a system's evaluations are direct_tiny's: one source tile a group and
// one target tile a wave, as the launches would take them, and no phase to time.
bool tiny_applies(const orr_ctx* ctx, std::uint64_t n) {
    if (n == 0 || n > kTinyMax || ctx->timing || ctx->direct_small_order != 1) return false;
    const DirectShape d = direct_shape(ctx, n);
    return d.R == 1 && d.per_split == 1 && !d.plan.use;
}

void tiny_launch(orr_ctx* ctx, const TinyArgs& args, double softening_squared) {
    const std::uint32_t tiles = (args.n + kTile - 1) / kTile;
    const bool safe = !(softening_squared > 0), refine = ctx->direct_refine != 0;
    auto pick = [&](auto rk4) {
        constexpr bool kRk4 = decltype(rk4)::value;
        return safe ? (refine ? direct_tiny<true, true, kRk4> : direct_tiny<true, false, kRk4>)
                    : (refine ? direct_tiny<false, true, kRk4> : direct_tiny<false, false, kRk4>);
    };
    auto kernel = args.mode == 2 ? pick(std::true_type{}) : pick(std::false_type{});
    hipLaunchKernelGGL(kernel, dim3(1), dim3(tiles * tiles * kTile), 0, ctx->stream, args);
    ORR_LAUNCHED("direct_tiny");
}

}  // namespace

bool direct_tiny_steps(orr_ctx* ctx, const SystemArrays& s, std::uint64_t n, const orr_step_config& c,
                       double dt, std::uint64_t steps) {
    if (!tiny_applies(ctx, n)) return false;
    TinyArgs t;
    for (int k = 0; k < 3; ++k) {
        t.x[k] = s.x[k];
        t.v[k] = s.v[k];
        t.a[k] = s.a[k];
    }
    t.m = s.m;
    t.n = static_cast<std::uint32_t>(n);
    t.ordered = n > kTile;
    t.eps2 = static_cast<float>(c.softening_squared);
    t.G = c.gravitational_constant;
    t.dt = dt;
    if (c.integrator == 2) {
        t.mode = 2;
    } else {
        t.mode = 1;
        t.substeps = c.integrator == 1 ? 3 : 1;
        const double w[3] = {kOuterWeight, kInnerWeight, kOuterWeight};
        for (int p = 0; p < t.substeps; ++p) {
            t.drift[p] = c.integrator == 1 ? w[p] * dt : dt;
            t.kick[p] = t.drift[p] / 2;
        }
    }
    // A launch of so many steps lasts up to some 30 ms (Runge-Kutta, 256 particles; velocity
    // Verlet 7 ms): no kernel holds the device for long.
    constexpr std::uint64_t kStepsPerLaunch = 256;
    while (steps > 0) {
        t.steps = static_cast<std::uint32_t>(std::min(steps, kStepsPerLaunch));
        tiny_launch(ctx, t, c.softening_squared);
        steps -= t.steps;
    }
    return true;
}

void direct_evaluate(orr_ctx* ctx, const orr_direct_args& a, const FusedKick& kick) {
    if (a.count == 0) return;
    const bool ordered = a.spatial_order != 0 && a.count > 64;
    // Without an order the launches are two or three, and from the fourth tile on
    // faster than one workgroup (192 particles 30.9 us against 30.4, 193 31.5
    // against 34.2, 256 31.6 against 38.4; with an order 42.4 here and 45.6 by
    // launches at 257).
    if (kick.vx == nullptr && tiny_applies(ctx, a.count) && (ordered || a.count <= 3 * kTile)) {
        TinyArgs t;
        t.x[0] = const_cast<double*>(a.x);
        t.x[1] = const_cast<double*>(a.y);
        t.x[2] = const_cast<double*>(a.z);
        t.a[0] = a.ax;
        t.a[1] = a.ay;
        t.a[2] = a.az;
        t.m = a.m;
        t.n = static_cast<std::uint32_t>(a.count);
        t.ordered = ordered;
        t.eps2 = static_cast<float>(a.softening_squared);
        t.G = a.gravitational_constant;
        tiny_launch(ctx, t, a.softening_squared);
        return;
    }
    // Compact tiles need only the top 32 bits of the 63-bit codes: the four
    // upper radix passes of eight, or for a small system the same order by
    // counting ranks.
    const bool small = ctx->direct_small_order == 1 && a.count <= kRankOrder;
    auto enqueue_order = [&] {
        if (small) {
            morton_enqueue_small(ctx, a.x, a.y, a.z, a.count);
        } else {
            morton_enqueue(ctx, a.x, a.y, a.z, a.count, 4);
        }
    };
    auto order = [&]() -> const std::uint32_t* {
        return ordered ? ctx->order_index.as<std::uint32_t>() : nullptr;
    };
    std::vector<unsigned char> key;
    key_add(key, a.x);
    key_add(key, a.y);
    key_add(key, a.z);
    key_add(key, a.count);
    key_add(key, small);
    if (ctx->timing) {
        // The order's short launches as one replayed graph, untimed; the direct
        // launches eager and timed.
        if (ordered) run_captured(ctx, ctx->direct_graph, std::move(key), enqueue_order, true);
        direct_enqueue(ctx, a, order(), kick);
        return;
    }
    // A small system's launches outrun the host: the whole evaluation as one
    // graph (N = 1000: 56 us, 66 with the order alone as a graph). Without an
    // order there are two launches, cheaper than a graph; beyond kSmallOrder
    // the launches are long enough for the host to stay ahead of them.
    if (!ordered || a.count > kSmallOrder) {
        if (ordered) enqueue_order();
        direct_enqueue(ctx, a, order(), kick);
        return;
    }
    key_add(key, a.m);
    key_add(key, a.ax);
    key_add(key, a.ay);
    key_add(key, a.az);
    key_add(key, a.softening_squared);
    key_add(key, a.gravitational_constant);
    key_add(key, ordered);
    key_add(key, kick.vx);
    key_add(key, kick.vy);
    key_add(key, kick.vz);
    key_add(key, kick.s);
    key_add(key, ctx->direct_targets_per_lane);
    key_add(key, ctx->direct_refine);
    key_add(key, ctx->direct_block_target);
    key_add(key, ctx->direct_pair_mode);
    key_add(key, ctx->direct_equal_masses);
    run_captured(ctx, ctx->direct_graph, std::move(key), [&] {
        if (ordered) enqueue_order();
        direct_enqueue(ctx, a, order(), kick);
    });
}

void direct_batch_enqueue(orr_ctx* ctx, const double* x, const double* y, const double* z,
                          const double* m, const std::uint32_t* order, const DirectBatchView& b,
                          double* ax, double* ay, double* az) {
    if (b.count == 0 || b.tiles == 0) return;
    const std::size_t npad = static_cast<std::size_t>(b.tiles) * kTile;
    ctx->direct_packed.reserve(packed_bytes(b.tiles));
    ctx->direct_centres.reserve(centre_bytes(b.tiles));
    ctx->direct_partials.reserve(slot_bytes(b.slots));
    float4* packed = ctx->direct_packed.as<float4>();
    float4* packed_lo = packed + npad;
    double4* centres = ctx->direct_centres.as<double4>();
    float4* extents = reinterpret_cast<float4*>(centres + b.tiles);
    float* partials = ctx->direct_partials.as<float>();
    {
        PhaseTimer t(ctx, kDirectPrepare);
        hipLaunchKernelGGL(batch_prepare, dim3(b.tiles), dim3(kTile), 0, ctx->stream, x, y, z, m,
                           order, b.tile, packed, packed_lo, centres, extents);
        ORR_LAUNCHED("batch_prepare");
    }
    {
        PhaseTimer t(ctx, kDirectKernel);
        // Eight blocks of four waves per CU; never more waves than items.
        const std::uint32_t cap = static_cast<std::uint32_t>(std::max(1, ctx->compute_units)) * 8;
        const bool refine = ctx->direct_refine != 0;
        auto pick = [&](auto safe, auto refined) {
            constexpr bool kS = decltype(safe)::value, kF = decltype(refined)::value;
            if (b.alone && b.items <= kEightWaveItems) return std::make_pair(&direct_items_wide<kS, kF, 8>, 8);
            if (b.alone && b.items <= kFourWaveItems) return std::make_pair(&direct_items_wide<kS, kF, 4>, 4);
            return std::make_pair(&direct_items<kS, kF>, 1);
        };
        const auto [kernel, waves] =
            b.safe ? (refine ? pick(std::true_type{}, std::true_type{}) : pick(std::true_type{}, std::false_type{}))
                   : (refine ? pick(std::false_type{}, std::true_type{}) : pick(std::false_type{}, std::false_type{}));
        const std::uint32_t blocks = std::max<std::uint32_t>(
            1, waves == 1 ? std::min(cap, (b.items + 3) / 4) : std::min(cap * 4 / waves, b.items));
        hipLaunchKernelGGL(kernel, dim3(blocks), dim3(waves == 1 ? kBlock : 64 * waves), 0, ctx->stream, packed,
                           packed_lo, centres, extents, b.tile, b.item, b.items, b.eps2, partials);
        ORR_LAUNCHED("direct_items");
    }
    {
        PhaseTimer t(ctx, kDirectReduce);
        const std::uint32_t blocks = static_cast<std::uint32_t>((b.count + 255) / 256);
        hipLaunchKernelGGL(batch_reduce, dim3(blocks), dim3(256), 0, ctx->stream, partials, b.sys,
                           b.tile, b.seg_of, b.G, b.count, order, ax, ay, az);
        ORR_LAUNCHED("batch_reduce");
    }
}

// ---- the direct sum on the library's static scratch ----------------------
//
// For callers that cannot allocate device memory: every buffer of the
// evaluation -- packed tiles, centres, the Morton order's codes, index and
// histograms, the one-sided kernel's FP64 sums a block -- is carved out
// of `scratch` below, a fixed array each device holds from the first call
// until the process ends. Limits: at most kStaticMaxCount particles; the
// one-sided kernel always (the pairs path's slots do not fit); the groups of
// direct_shape, fewer where a sum and compensation a target and group would not
// fit (the same bits as direct_evaluate with the one-sided kernel whenever they
// do, else the same terms in fewer Kahan-summed groups). Nothing in the scratch has to
// start at zero: every launch writes what the next reads. Calls on one device
// share the array, so calls that overlap on one device (two contexts, two
// host threads) race.

constexpr std::size_t kStaticScratchBytes = std::size_t{16} << 20;
constexpr std::uint64_t kStaticMaxCount = 32768;

}  // namespace orr

static __device__ __align__(256) unsigned char scratch[orr::kStaticScratchBytes];

namespace {

using orr::kStaticMaxCount;
using orr::kStaticScratchBytes;
constexpr int kMaxDevices = 64;

// The array's device address on each device, looked up once per device with
// that device current (host code must never use the symbol itself as an
// address).
std::mutex g_scratch_lock;
void* g_scratch_ptr[kMaxDevices] = {};

void* scratch_on(int device) {
    if (device < 0 || device >= kMaxDevices) orr::fail(ORR_ERR_INVALID_ARGUMENT, "device index out of range");
    std::lock_guard<std::mutex> lock(g_scratch_lock);
    if (g_scratch_ptr[device] == nullptr) {
        void* ptr = nullptr;
        ORR_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        if (ptr == nullptr) orr::fail(ORR_ERR_RUNTIME, "static scratch: no device address");
        g_scratch_ptr[device] = ptr;
    }
    return g_scratch_ptr[device];
}

// Bump allocation inside the scratch, 256-byte aligned.
struct Carver {
    unsigned char* base;
    std::size_t used = 0;
    template<typename T> T* take(std::size_t bytes) {
        T* p = reinterpret_cast<T*>(base + used);
        used += (bytes + 255) & ~std::size_t{255};
        return p;
    }
};

std::size_t aligned(std::size_t bytes) { return (bytes + 255) & ~std::size_t{255}; }

}  // namespace

namespace orr {

std::size_t direct_static_scratch_bytes() { return kStaticScratchBytes; }
std::uint64_t direct_static_max_count() { return kStaticMaxCount; }

void direct_evaluate_static(orr_ctx* ctx, const orr_direct_args& a) {
    if (a.count == 0) return;
    if (a.count > kStaticMaxCount) {
        fail(ORR_ERR_LENGTH, "direct (static scratch): more than 32768 particles; use orr_direct_eval");
    }
    const std::uint64_t n = a.count;
    DirectShape d = direct_shape(ctx, n);
    d.plan = PairPlan{};  // the one-sided kernel
    const bool ordered = a.spatial_order != 0 && n > 64;
    const OrderSizes oz = order_sizes(n, 1, 0, false);
    // What the groups of source tiles are sized by: room beside the other
    // buffers for one FP32 sum and compensation a target and group and for a near
    // mask. Neither is carved (the FP64 sums of a block need less); counting
    // them keeps the groups, and so the bits.
    const std::size_t fixed = aligned(packed_buffer_bytes(d)) + aligned(centre_buffer_bytes(d)) +
                              aligned(sizeof(std::uint32_t) * static_cast<std::size_t>(d.words) * d.tiles) +
                              (ordered ? aligned(oz.bbox) + 2 * aligned(oz.codes) +
                                             2 * aligned(oz.index) + aligned(oz.hist)
                                       : 0);
    const std::size_t split_bytes = aligned(sizeof(float) * 6 * static_cast<std::size_t>(d.npad));
    if (fixed + split_bytes > kStaticScratchBytes) {
        fail(ORR_ERR_LENGTH, "direct (static scratch): the evaluation does not fit the scratch");
    }
    const std::uint32_t fit = static_cast<std::uint32_t>((kStaticScratchBytes - fixed) / split_bytes);
    if (d.splits > fit) {
        d.per_split = (d.tiles + fit - 1) / fit;
        d.splits = (d.tiles + d.per_split - 1) / d.per_split;
    }
    one_sided_shape(d);
    Carver c{static_cast<unsigned char*>(scratch_on(ctx->device))};
    DirectBuffers buf;
    buf.packed = c.take<float4>(packed_buffer_bytes(d));
    buf.centres = c.take<double4>(centre_buffer_bytes(d));
    const std::uint32_t* order = nullptr;
    if (ordered) {
        OrderScratch ob;
        ob.bbox = c.take<double>(oz.bbox);
        ob.codes[0] = c.take<std::uint64_t>(oz.codes);
        ob.codes[1] = c.take<std::uint64_t>(oz.codes);
        ob.index[0] = c.take<std::uint32_t>(oz.index);
        ob.index[1] = c.take<std::uint32_t>(oz.index);
        ob.hist = c.take<std::uint32_t>(oz.hist);
        // The order direct_evaluate uses: by the upper half of the codes.
        const int cur = morton_enqueue_into(ctx, a.x, a.y, a.z, n, SegmentView{}, nullptr, 4, ob, false);
        order = ob.index[cur];
    }
    buf.partials = c.take<double>(partial_buffer_bytes(d));
    if (c.used > kStaticScratchBytes) fail(ORR_ERR_RUNTIME, "direct (static scratch): layout overflow");
    direct_launch(ctx, a, order, d, buf, false);
}

}  // namespace orr
