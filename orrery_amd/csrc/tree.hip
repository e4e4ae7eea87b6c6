// Barnes-Hut on gfx950: octree build from sorted Morton keys, FP64 monopole
// moments, and a wave-coherent theta-criterion walk.
//
// The tree is the reference's (src/solvers/octree.cpp:196-468): cells split in
// octant order, empty cells skipped, a leaf when a cell holds <= leaf_capacity
// particles or sits at level 21, nodes in depth-first order with `next` the
// index just past the subtree. The reference builds it by recursion; here every
// node is derived independently from the sorted keys:
//
//   d(k)   the first level at which key k differs from key k-1 (d(0) = 0, 22
//          for a duplicate key): a cell of level l starts at particle k exactly
//          when d(k) <= l.
//   chain  the cells that start at k form a chain of levels d(k), d(k)+1, ...
//          Its first cell is a node iff its parent (level d(k)-1) holds more
//          than leaf_capacity particles (found by scanning +-leaf_capacity keys
//          around k); every deeper cell of the chain is a node while the one
//          above it holds more than leaf_capacity, i.e. down to level
//          min(21, max(d(k), min d over the next leaf_capacity keys)), a leaf.
//   DFS    depth-first order sorts nodes by (first particle, level), so an
//          exclusive scan of chain lengths numbers the nodes, and the node
//          after a subtree is the first node starting at the cell's end:
//          next = first_node[end].
//
// Moments follow octree.cpp:91-185 operation for operation in FP64 (leaf: sums
// over particles in index order; internal: over children in DFS order), with
// contraction disabled, so masses, centres of mass and acceptance radii
// (octree.cpp:374-387) are the reference's bit for bit.
//
// The walk (tree_walk.cpp:20-83 per target) runs waves over groups of up to 64
// consecutive sorted targets. A wave goes through the nodes that any of its
// targets visits -- each target still takes part in exactly its own walk, as in the
// reference's coherent CUDA walk (ADR-0029) -- with the node read through the
// scalar unit. Accepted cells
// use FP32 positions relative to the root centre; leaf particles are stored as
// FP32 offsets from their leaf's geometric centre and a lane interacting with a
// leaf re-expresses its own offset against that centre in FP64, so close pairs
// keep the precision of the leaf size. Per-lane partial sums are Kahan-folded
// after each leaf.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <limits>
#include <type_traits>
#include <vector>

#include "engine.hpp"

#pragma clang fp contract(off)

namespace orr {
namespace {

constexpr int kBlock = 256;
constexpr unsigned kLevels = 21;
constexpr std::uint8_t kNoBoundary = 22;
constexpr int kMaxChildren = 8;                 // octants
constexpr std::uint32_t kNoChild = 0xffffffffu;
// Spare float4 entries past the last particle of leaf_rel: a leaf's sources are
// read in rounds of four, one round ahead.
constexpr std::size_t kLeafPad = 4;
// The fewest targets a walk wave holds.
constexpr std::uint64_t kMinLanes = 16;

struct WalkNode {
    float4 a;  // centre of mass relative to the root centre (FP32), mass
    uint4 b;   // acceptance radius^2 (FP32 bits), next, first particle, particle count
};

struct QuadF {
    float4 a;  // xx, xy, xz, yy
    float4 b;  // yz, zz, 0, 0
};

// Device counters, uint32: [0] nodes, [1] leaves, [2] depth.
// Device statistics, uint64: [0] particle-particle, [1] particle-cell, [2] lane visits,
// [3] wave steps.

__device__ inline std::uint32_t grid_stride_start() { return blockIdx.x * blockDim.x + threadIdx.x; }
__device__ inline std::uint32_t grid_stride_step() { return gridDim.x * blockDim.x; }

// d(k) from adjacent sorted codes; 0 where a system starts (each system of a
// batch is its own tree, and a level-0 boundary ends every window at it). The
// first block also clears the counters of the launches to come.
__global__ __launch_bounds__(kBlock) void tree_levels(const std::uint64_t* __restrict__ codes,
                                                      const std::uint32_t* __restrict__ seg_of,
                                                      std::uint32_t n, std::uint8_t* __restrict__ d,
                                                      std::uint32_t* __restrict__ c32,
                                                      unsigned long long* __restrict__ c64,
                                                      std::uint32_t count64) {
    if (blockIdx.x == 0) {
        if (threadIdx.x < 4) c32[threadIdx.x] = 0;
        if (c64 != nullptr) {
            for (std::uint32_t k = threadIdx.x; k < count64; k += kBlock) c64[k] = 0;
        }
    }
    const std::uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= n) return;
    if (k == 0 || (seg_of != nullptr && seg_of[k] != seg_of[k - 1])) {
        d[k] = 0;
        return;
    }
    const std::uint64_t x = codes[k] ^ codes[k - 1];
    if (x == 0) {
        d[k] = kNoBoundary;
        return;
    }
    const unsigned h = 63u - static_cast<unsigned>(__clzll(x));  // highest differing bit
    d[k] = static_cast<std::uint8_t>(kLevels - h / 3u);
}

// Chain length of the nodes that start at particle k; leaf level in `leaf_level`.
// The searches read kAhead levels at once: one at a time, each waits for the
// one before (16,384 particles 10.8 -> 5.5 us, 2,097,152 37 -> 22).
constexpr int kAhead = 8;
__global__ __launch_bounds__(kBlock) void tree_chain(const std::uint8_t* __restrict__ d,
                                                     std::uint32_t n, std::uint32_t cap,
                                                     std::uint32_t* __restrict__ chain,
                                                     std::uint8_t* __restrict__ leaf_level) {
    const std::uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= n) return;
    const unsigned dk = d[k];
    std::uint32_t len = 0;
    unsigned lleaf = dk;
    if (dk <= kLevels) {
        bool head = true;
        if (dk > 0) {  // d = 0: the root of its system
            // Parent cell of level dk-1 spans [p, q) around k; it is a leaf (so
            // no node starts at k) iff q - p <= cap.
            const unsigned P = dk - 1;
            const std::uint32_t lo = k + 1 > cap ? k + 1 - cap : 0;
            std::int64_t p = -1;
            for (std::int64_t j = static_cast<std::int64_t>(k) - 1; j >= static_cast<std::int64_t>(lo) && p < 0;
                 j -= kAhead) {
                std::uint8_t level[kAhead];
                // Past the end of the search, its last element again.
#pragma unroll
                for (int u = 0; u < kAhead; ++u) level[u] = d[std::max<std::int64_t>(j - u, lo)];
#pragma unroll
                for (int u = kAhead - 1; u >= 0; --u) {
                    if (level[u] <= P) p = std::max<std::int64_t>(j - u, lo);
                }
            }
            if (p >= 0) {
                const std::uint64_t limit = static_cast<std::uint64_t>(p) + cap;  // q must be <= limit
                std::uint64_t q = n;
                const std::uint64_t stop = limit < n - 1 ? limit : n - 1;
                for (std::uint64_t j = k + 1; j <= stop && q == n; j += kAhead) {
                    std::uint8_t level[kAhead];
#pragma unroll
                    for (int u = 0; u < kAhead; ++u) level[u] = d[std::min<std::uint64_t>(j + u, stop)];
#pragma unroll
                    for (int u = kAhead - 1; u >= 0; --u) {
                        if (level[u] <= P) q = std::min<std::uint64_t>(j + u, stop);
                    }
                }
                head = !(q <= limit);
            }
        }
        if (head) {
            if (n - k <= cap) {
                lleaf = dk;
            } else {
                unsigned w = kNoBoundary;
                for (std::uint32_t j = k + 1; j <= k + cap; j += kAhead) {
#pragma unroll
                    for (std::uint32_t u = 0; u < kAhead; ++u) {
                        w = min(w, static_cast<unsigned>(d[min(j + u, k + cap)]));
                    }
                }
                lleaf = min(kLevels, max(dk, w));
            }
            len = lleaf - dk + 1;
        }
    }
    chain[k] = len;
    leaf_level[k] = static_cast<std::uint8_t>(lleaf);
}

// First index j >= lo whose code prefix of `level` exceeds that of `key`.
__device__ std::uint32_t prefix_end(const std::uint64_t* __restrict__ codes, std::uint32_t n,
                                    std::uint32_t lo, std::uint64_t key, unsigned level) {
    if (level == 0) return n;
    const unsigned s = 3u * (kLevels - level);
    const std::uint64_t want = key >> s;
    if (lo >= n || (codes[lo] >> s) != want) return lo;
    // Gallop, then narrow down: codes[lo] shares the prefix. Four probes at once:
    // one at a time, each waits for the one before, 27 in a row for a root of
    // 16,384 particles (tree_node_fill of 60,000 particles 11.6 -> 9.3 us, of
    // 262,144 12.4 -> 9.8).
    constexpr unsigned kProbes = 4;
    auto matches = [&](std::uint64_t at) { return (codes[at] >> s) == want; };
    std::uint32_t good = lo, bad = n;
    bool found = false;
    for (unsigned power = 0; !found; power += kProbes) {
        bool match[kProbes];
#pragma unroll
        for (unsigned u = 0; u < kProbes; ++u) {
            match[u] = matches(std::min<std::uint64_t>(lo + (std::uint64_t{1} << (power + u)), n - 1));
        }
#pragma unroll
        for (unsigned u = 0; u < kProbes; ++u) {
            const std::uint64_t at = lo + (std::uint64_t{1} << (power + u));
            if (found) continue;
            found = at >= n || !match[u];
            if (at < n) (match[u] ? good : bad) = static_cast<std::uint32_t>(at);
        }
    }
    while (bad - good > 1) {
        const std::uint32_t step = (bad - good + kProbes) / (kProbes + 1);
        const std::uint32_t from = good, to = bad;
        bool match[kProbes];
#pragma unroll
        for (unsigned u = 0; u < kProbes; ++u) {
            match[u] = matches(std::min<std::uint64_t>(from + std::uint64_t{step} * (u + 1), to - 1));
        }
        // The probes that match come first.
#pragma unroll
        for (unsigned u = 0; u < kProbes; ++u) {
            const std::uint64_t at = std::min<std::uint64_t>(from + std::uint64_t{step} * (u + 1), to - 1);
            if (match[u]) {
                good = static_cast<std::uint32_t>(at);
            } else if (at < bad) {
                bad = static_cast<std::uint32_t>(at);
            }
        }
    }
    return bad;
}

// Each chain's nodes: start particle and level (one thread per chain start; no
// searches here, so no thread waits on another's).
__global__ __launch_bounds__(kBlock) void tree_chains(
    const std::uint8_t* __restrict__ d, const std::uint8_t* __restrict__ leaf_level,
    const std::uint32_t* __restrict__ chain, const std::uint32_t* __restrict__ first_node,
    std::uint32_t n, uint2* __restrict__ block_counts, std::uint32_t* __restrict__ node_begin,
    std::uint8_t* __restrict__ node_level) {
    __shared__ unsigned s_leaves[kBlock / 64], s_depth[kBlock / 64];
    const std::uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    const bool owns = k < n && chain[k] != 0;
    unsigned depth = 0;
    if (owns) {
        const unsigned dk = d[k], lleaf = leaf_level[k];
        const std::uint32_t base = first_node[k];
        for (unsigned l = dk; l <= lleaf; ++l) {
            node_begin[base + (l - dk)] = k;
            node_level[base + (l - dk)] = static_cast<std::uint8_t>(l);
        }
        depth = lleaf;
    }
    // One leaf per chain: each block writes its leaf count and deepest level to
    // its own slot (atomics on one address would serialise every wave).
    const unsigned long long leaves = __ballot(owns);
    unsigned deepest = depth;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) deepest = max(deepest, static_cast<unsigned>(__shfl_xor(static_cast<int>(deepest), off, 64)));
    if ((threadIdx.x & 63) == 0) {
        s_leaves[threadIdx.x / 64] = static_cast<unsigned>(__popcll(leaves));
        s_depth[threadIdx.x / 64] = deepest;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned total = 0, deep = 0;
        for (int w = 0; w < kBlock / 64; ++w) {
            total += s_leaves[w];
            deep = max(deep, s_depth[w]);
        }
        block_counts[blockIdx.x] = make_uint2(total, deep);
    }
}

// One block: leaf count and depth from the per-block slots.
__device__ void tree_counts(const uint2* __restrict__ block_counts, std::uint32_t blocks,
                            std::uint32_t* __restrict__ counters) {
    __shared__ unsigned s_total[kBlock], s_deep[kBlock];
    unsigned total = 0, deep = 0;
    for (std::uint32_t b = threadIdx.x; b < blocks; b += kBlock) {
        total += block_counts[b].x;
        deep = max(deep, block_counts[b].y);
    }
    s_total[threadIdx.x] = total;
    s_deep[threadIdx.x] = deep;
    __syncthreads();
    for (int w = kBlock / 2; w > 0; w >>= 1) {
        if (static_cast<int>(threadIdx.x) < w) {
            s_total[threadIdx.x] += s_total[threadIdx.x + w];
            s_deep[threadIdx.x] = max(s_deep[threadIdx.x], s_deep[threadIdx.x + w]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        counters[1] = s_total[0];
        counters[2] = s_deep[0];
    }
}

// One thread per node: its cell's end (a prefix search from its start, so a
// node never waits on another), escape index, geometric centre (octree.cpp:41-47:
// one halving per level from the root centre of morton.hpp:93-95) and, for a
// leaf, the leaf id of its particles.
__global__ __launch_bounds__(kBlock) void tree_node_fill(
    const std::uint64_t* __restrict__ codes, const std::uint8_t* __restrict__ leaf_level,
    const std::uint32_t* __restrict__ first_node, std::uint32_t n,
    const std::uint32_t* __restrict__ seg_of, const std::uint32_t* __restrict__ seg_start,
    const double* __restrict__ cubes, const std::uint32_t* __restrict__ counters,
    const std::uint32_t* __restrict__ node_begin, const std::uint8_t* __restrict__ node_level,
    std::uint32_t* __restrict__ node_count, std::uint32_t* __restrict__ node_next,
    double4* __restrict__ node_geo, std::uint32_t* __restrict__ leaf_of) {
    const std::uint32_t M = counters[0];
    for (std::uint32_t node = grid_stride_start(); node < M; node += grid_stride_step()) {
        const std::uint32_t k = node_begin[node];
        const unsigned l = node_level[node];
        const std::uint64_t key = codes[k];
        const std::uint32_t seg = seg_of != nullptr ? seg_of[k] : 0u;
        const std::uint32_t seg_end = seg_start != nullptr ? seg_start[seg + 1] : n;
        const double* cube = cubes + 4 * static_cast<std::size_t>(seg);
        const std::uint32_t end = prefix_end(codes, seg_end, k + 1, key, l);
        node_count[node] = end - k;
        node_next[node] = end >= n ? M : first_node[end];
        double size = cube[3];
        double c[3] = {cube[0] + size / 2, cube[1] + size / 2, cube[2] + size / 2};
        for (unsigned s = 1; s <= l; ++s) {
            const unsigned oct = static_cast<unsigned>((key >> (3u * (kLevels - s))) & 7u);
            const double q = size / 4;
            c[0] = c[0] + ((oct & 4u) != 0 ? q : -q);
            c[1] = c[1] + ((oct & 2u) != 0 ? q : -q);
            c[2] = c[2] + ((oct & 1u) != 0 ? q : -q);
            size = size / 2;
        }
        node_geo[node] = make_double4(c[0], c[1], c[2], size);
        if (l == leaf_level[k]) {
            for (std::uint32_t j = k; j < end; ++j) leaf_of[j] = node;
        }
    }
}

// Sorted FP64 particles for the moments; FP32 walk data: position relative to
// the root centre, and offset from the particle's leaf centre.
__global__ __launch_bounds__(kBlock) void tree_gather(
    const double4* __restrict__ aos, const std::uint32_t* __restrict__ index, std::uint32_t n,
    const double* __restrict__ cubes, const std::uint32_t* __restrict__ seg_of,
    const std::uint32_t* __restrict__ leaf_of,
    const double4* __restrict__ node_geo, double4* __restrict__ sorted,
    float4* __restrict__ root_rel, float4* __restrict__ leaf_rel) {
    const std::uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    // One 32-byte record per particle ({x, y, z, m} written in index order by
    // the encode pass) rather than four scattered FP64 loads.
    const double4 p = aos[index[i]];
    const double px = p.x, py = p.y, pz = p.z, pm = p.w;
    sorted[i] = p;
    const double* cube = cubes + (seg_of != nullptr ? 4 * static_cast<std::size_t>(seg_of[i]) : 0);
    const double half = cube[3] / 2;
    const double c0x = cube[0] + half, c0y = cube[1] + half, c0z = cube[2] + half;
    root_rel[i] = make_float4(static_cast<float>(px - c0x), static_cast<float>(py - c0y),
                              static_cast<float>(pz - c0z), static_cast<float>(pm));
    const double4 g = node_geo[leaf_of[i]];
    leaf_rel[i] = make_float4(static_cast<float>(px - g.x), static_cast<float>(py - g.y),
                              static_cast<float>(pz - g.z), static_cast<float>(pm));
}

// The walk's escape index: the DFS successor, or "done" when the node's cell
// ends its system (the successor then belongs to the next system or past M).
__device__ inline std::uint32_t walk_escape(std::uint32_t next, std::uint32_t cell_end,
                                            std::uint32_t system_end) {
    return cell_end >= system_end ? 0xffffffffu : next;
}

// A value that another workgroup of the same launch reads (on any XCD): stored
// past this XCD's L2, and loaded past the reader's.
__device__ __forceinline__ void share(double* p, double v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double shared_value(const double* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ inline void finish_node(std::uint32_t node, double mass, double cx, double cy, double cz,
                                   const double4 geo, double theta, const double* __restrict__ cube,
                                   bool leaf, std::uint32_t begin, std::uint32_t count,
                                   std::uint32_t next, double4* __restrict__ moment,
                                   WalkNode* __restrict__ walk) {
    share(&moment[node].x, cx);
    share(&moment[node].y, cy);
    share(&moment[node].z, cz);
    share(&moment[node].w, mass);
    // octree.cpp:370-371 and :374-387.
    const double ox = cx - geo.x, oy = cy - geo.y, oz = cz - geo.z;
    const double offset = sqrt((ox * ox) + (oy * oy) + (oz * oz));
    double acc;
    if (!(theta > 0)) {
        acc = __builtin_huge_val();
    } else {
        const double r = (geo.w / theta) + offset;
        acc = r * r;
    }
    const double half = cube[3] / 2;
    WalkNode w;
    w.a = make_float4(static_cast<float>(cx - (cube[0] + half)), static_cast<float>(cy - (cube[1] + half)),
                      static_cast<float>(cz - (cube[2] + half)), static_cast<float>(mass));
    float accf = static_cast<float>(acc);
    std::uint32_t bits;
    std::memcpy(&bits, &accf, sizeof(bits));
    w.b = make_uint4(bits, next, leaf ? begin : 0u, leaf ? count : 0u);
    walk[node] = w;
}

// octree.cpp:75-84: traceless second moment of a point mass displaced by d.
__device__ inline void add_displaced(double q[6], double mass, double dx, double dy, double dz) {
    const double trace = mass * (((dx * dx) + (dy * dy)) + (dz * dz));
    q[0] += (3 * mass * dx * dx) - trace;
    q[1] += 3 * mass * dx * dy;
    q[2] += 3 * mass * dx * dz;
    q[3] += (3 * mass * dy * dy) - trace;
    q[4] += 3 * mass * dy * dz;
    q[5] += (3 * mass * dz * dz) - trace;
}

__device__ inline void store_quad(std::uint32_t node, const double q[6], double* __restrict__ quad64,
                                  QuadF* __restrict__ quadf) {
    for (int k = 0; k < 6; ++k) share(&quad64[6 * static_cast<std::size_t>(node) + k], q[k]);
    QuadF f;
    f.a = make_float4(static_cast<float>(q[0]), static_cast<float>(q[1]), static_cast<float>(q[2]),
                      static_cast<float>(q[3]));
    f.b = make_float4(static_cast<float>(q[4]), static_cast<float>(q[5]), 0.f, 0.f);
    quadf[node] = f;
}

// Every internal node's children in DFS order (the next chain from node + 1 to
// the node's own next), side by side for the moments, and what the climb
// needs: the parent of every node, and how many children an internal node
// still waits for. These two lie in memory nothing else uses yet: an internal
// node's moment (the parent in the first word, the count in the second), a
// leaf's row of `children`. The last block sums the leaf counts meanwhile.
__device__ __forceinline__ std::uint32_t* link_words(double4* moment, std::uint32_t node) {
    return reinterpret_cast<std::uint32_t*>(&moment[node]);
}
__global__ __launch_bounds__(kBlock) void tree_links(
    std::uint32_t* __restrict__ counters, const std::uint8_t* __restrict__ node_level,
    const std::uint8_t* __restrict__ leaf_level_of_first, const std::uint32_t* __restrict__ node_begin,
    const std::uint32_t* __restrict__ node_next, const uint2* __restrict__ block_counts,
    std::uint32_t blocks, std::uint32_t* __restrict__ children, double4* __restrict__ moment) {
    if (blockIdx.x + 1 == gridDim.x) {
        tree_counts(block_counts, blocks, counters);
        return;
    }
    const std::uint32_t M = counters[0];
    const std::uint32_t stride = (gridDim.x - 1) * kBlock;
    for (std::uint32_t node = grid_stride_start(); node < M; node += stride) {
        const unsigned level = node_level[node];
        const bool leaf = level == leaf_level_of_first[node_begin[node]];
        std::uint32_t* const row = children + static_cast<std::size_t>(kMaxChildren) * node;
        if (level == 0) *(leaf ? row : link_words(moment, node)) = kNoChild;
        if (leaf) continue;
        const std::uint32_t end = node_next[node];
        std::uint32_t k = 0;
        for (std::uint32_t c = node + 1; c < end && k < kMaxChildren; c = max(node_next[c], c + 1)) {
            row[k++] = c;
            const bool leaf_child = node_level[c] == leaf_level_of_first[node_begin[c]];
            *(leaf_child ? children + static_cast<std::size_t>(kMaxChildren) * c : link_words(moment, c)) = node;
        }
        link_words(moment, node)[1] = k;
        for (; k < kMaxChildren; ++k) row[k] = kNoChild;
    }
}

// octree.cpp:142-185 (internal): children in DFS order; quadrupoles by the
// parallel-axis theorem, children's moments first.
__device__ void internal_moments(
    std::uint32_t node, const std::uint32_t* __restrict__ node_begin,
    const std::uint32_t* __restrict__ node_count, const std::uint32_t* __restrict__ node_next,
    const std::uint32_t* __restrict__ children, const double4* __restrict__ node_geo, double theta,
    const double* __restrict__ cube, std::uint32_t system_end, double4* __restrict__ moment,
    WalkNode* __restrict__ walk, double* __restrict__ quad64, QuadF* __restrict__ quadf) {
    // The children's indices, then their moments, loaded side by side; the
    // sums below still run in DFS order.
    const std::uint32_t* list = children + static_cast<std::size_t>(kMaxChildren) * node;
    std::uint32_t child[kMaxChildren];
    double4 cms[kMaxChildren];
#pragma unroll
    for (int k = 0; k < kMaxChildren; ++k) child[k] = list[k];
#pragma unroll
    for (int k = 0; k < kMaxChildren; ++k) {
        const double* m = &moment[child[k] == kNoChild ? node : child[k]].x;
        cms[k] = make_double4(shared_value(m), shared_value(m + 1), shared_value(m + 2), shared_value(m + 3));
    }
    double mass = 0, wx = 0, wy = 0, wz = 0, mx = 0, my = 0, mz = 0;
    std::uint32_t count = 0;
#pragma unroll
    for (int k = 0; k < kMaxChildren; ++k) {
        if (child[k] == kNoChild) continue;
        const double4 cm = cms[k];
        mass += cm.w;
        wx += cm.x * cm.w;
        wy += cm.y * cm.w;
        wz += cm.z * cm.w;
        mx += cm.x;
        my += cm.y;
        mz += cm.z;
        ++count;
    }
    double cx, cy, cz;
    if (mass > 0) {
        cx = wx / mass;
        cy = wy / mass;
        cz = wz / mass;
    } else {
        const double k = static_cast<double>(count == 0 ? 1 : count);
        cx = mx / k;
        cy = my / k;
        cz = mz / k;
    }
    const std::uint32_t b = node_begin[node];
    finish_node(node, mass, cx, cy, cz, node_geo[node], theta, cube, false, b, 0,
                walk_escape(node_next[node], b + node_count[node], system_end), moment, walk);
    if (quad64 != nullptr) {
        double q[6] = {0, 0, 0, 0, 0, 0};
        // Four children's moments on their way together: one latency, not four.
#pragma unroll
        for (int k = 0; k < kMaxChildren; k += 4) {
            double cq[4][6];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const std::uint32_t c = child[k + u] == kNoChild ? node : child[k + u];
#pragma unroll
                for (int j = 0; j < 6; ++j) cq[u][j] = shared_value(quad64 + 6 * static_cast<std::size_t>(c) + j);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                if (child[k + u] == kNoChild) continue;
                for (int j = 0; j < 6; ++j) q[j] += cq[u][j];
                const double4 cm = cms[k + u];
                add_displaced(q, cm.w, cm.x - cx, cm.y - cy, cm.z - cz);
            }
        }
        store_quad(node, q, quad64, quadf);
    }
}

// All moments in one launch. One thread a leaf, octree.cpp:91-135: index-order
// sums, fallback to the first particle; with quadrupoles, the displaced
// moments of the particles about the centre of mass. Then up the tree: the
// thread whose child was the last one a node waited for computes the node and
// goes on to its parent; the others are done, and no thread waits. Which
// thread comes last does not change what it computes. A launch a level, 21 of
// them, cost 3 to 10 us each, most over levels that have no nodes: all
// moments of 16,384 particles 70 -> 33 us, of 65,536 72 -> 34, with
// quadrupoles of 262,144 126 -> 71 and of 2,097,152 264 -> 225. Plain stores
// between agent-scope fences instead of stores and loads past the L2: 33 -> 35
// and 225 -> 1120 us.
__global__ __launch_bounds__(kBlock) void tree_moments(
    const std::uint32_t* __restrict__ counters, const std::uint8_t* __restrict__ node_level,
    const std::uint8_t* __restrict__ leaf_level_of_first, const std::uint32_t* __restrict__ node_begin,
    const std::uint32_t* __restrict__ node_count, const std::uint32_t* __restrict__ node_next,
    const std::uint32_t* __restrict__ children, const double4* __restrict__ node_geo,
    const double4* __restrict__ sorted, double theta,
    const double* __restrict__ cubes, const std::uint32_t* __restrict__ seg_of,
    const std::uint32_t* __restrict__ seg_start, std::uint32_t n,
    double4* moment, WalkNode* __restrict__ walk, double* quad64, QuadF* __restrict__ quadf) {
    const std::uint32_t M = counters[0];
    for (std::uint32_t node = grid_stride_start(); node < M; node += grid_stride_step()) {
        const std::uint32_t b = node_begin[node];
        if (node_level[node] != leaf_level_of_first[b]) continue;  // internal
        const std::uint32_t seg = seg_of != nullptr ? seg_of[b] : 0u;
        const double* cube = cubes + 4 * static_cast<std::size_t>(seg);
        const std::uint32_t system_end = seg_start != nullptr ? seg_start[seg + 1] : n;
        const std::uint32_t e = b + node_count[node];
        double mass = 0, wx = 0, wy = 0, wz = 0;
#pragma unroll 4
        for (std::uint32_t i = b; i < e; ++i) {
            const double4 p = sorted[i];
            mass += p.w;
            wx += p.x * p.w;
            wy += p.y * p.w;
            wz += p.z * p.w;
        }
        double cx, cy, cz;
        if (mass > 0) {
            cx = wx / mass;
            cy = wy / mass;
            cz = wz / mass;
        } else {
            cx = sorted[b].x;
            cy = sorted[b].y;
            cz = sorted[b].z;
        }
        finish_node(node, mass, cx, cy, cz, node_geo[node], theta, cube, true, b, e - b,
                    walk_escape(node_next[node], e, system_end), moment, walk);
        if (quad64 != nullptr) {
            double q[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll 4
            for (std::uint32_t i = b; i < e; ++i) {
                const double4 p = sorted[i];
                add_displaced(q, p.w, p.x - cx, p.y - cy, p.z - cz);
            }
            store_quad(node, q, quad64, quadf);
        }
        std::uint32_t up = children[static_cast<std::size_t>(kMaxChildren) * node];
        while (up != kNoChild) {
            std::uint32_t* const link = link_words(moment, up);
            const std::uint32_t above = __hip_atomic_load(link, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            // The child's moments are in memory before the count says so (the
            // stores above go past the L2; this waits for them), and the
            // siblings' are read after it.
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            if (__hip_atomic_fetch_sub(link + 1, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 1) break;
            asm volatile("" ::: "memory");
            internal_moments(up, node_begin, node_count, node_next, children, node_geo, theta, cube, system_end,
                             moment, walk, quad64, quadf);
            up = above;
        }
    }
}

__device__ __forceinline__ void kahan(float p, float& s, float& c) {
    const float y = p - c;
    const float t = s + y;
    c = (t - s) - y;
    s = t;
}

// Targets a wave, and waves that share the walk of a group of targets (parts),
// by the launch's full (64-lane) waves. Walk in ms, Plummer spheres (P) and
// two-disc collisions (D), opening angle 0.5 or 0.6, monopoles (m) or quadrupoles (q),
// as {16 targets, 1 part}, {32, 1}, {16, 8}, {16, 4}, {32, 2}, and from 65,536 on
// {32, 1}, {64, 1}, {32, 2}:
//   1000 Pq  0.145 0.153 0.049 0.065           28,000 Pq 0.690 0.727   -   0.676 0.582
//   4096 Pq  0.336 0.372 0.125 0.156           49,152 Pq 0.828 0.828   -   1.153 0.690
//   8192 Dm  0.263 0.277 0.118 0.167           60,000 Dm 0.505 0.492   -   0.837 0.418
//   8192 Pq  0.490 0.539 0.231 0.221           65,536 Dq 0.822 0.896 0.758
//   10,240 Pm 0.392 0.427 0.243 0.188          73,728 Pq 0.974 1.013 0.922
//   16,384 Pm 0.447 0.483 0.417 0.259          81,920 Dq 0.863 0.912 0.892
//   24,576 Pq 0.678 0.705   -   0.505 0.534    98,304 Pq 1.026 1.062 1.140
//   24,576 Dm 0.473 0.493   -   0.358 0.373    106,496 Pq 1.062 1.017 1.151
// More parts pay while the launch leaves the SIMDs short of waves; past that
// the nodes walked twice, and the room in LDS, cost more than they hide.
//
// A small opening angle visits thousands of leaves a target where a part has
// room for a few dozen runs, and each part ends up waiting for the one before:
// from kOnePartFrom particles a system on, angles up to kOnePartAngle take one
// part. Whole evaluations of Plummer spheres, us, in parts and in one: 10,000
// at angle 0.1 (leaves of 4) 3423 and 3038; 16,384 at 0.1 (4) 5517 and 4402,
// at 0.15 (8) 3587 and 3132, at 0.2 (8) 2751 and 2643, at 0.3 (8) 1578 and 1776;
// 24,576 at 0.1 (4) 7937 and 6161; 60,000 at 0.15 (16) 6961 and 5687, at 0.5
// (16) 812 and 861.
struct WalkShape {
    int lanes, parts;
};
constexpr std::uint64_t kEightPartWaves = 128;
constexpr std::uint64_t kFourPartWaves = 384;
constexpr std::uint64_t kTwoPartWaves = 1152;
constexpr std::uint64_t kHalfLaneWaves = 1600;
constexpr double kOnePartAngle = 0.15;
constexpr std::uint64_t kOnePartFrom = 10240;
// `longest`: particles of the launch's largest system.
WalkShape walk_shape(std::uint64_t full_waves, std::uint64_t longest, double theta) {
    const bool one_part = theta <= kOnePartAngle && longest > kOnePartFrom;
    if (full_waves <= kEightPartWaves && !one_part) return {16, 8};
    if (full_waves <= kFourPartWaves && !one_part) return {16, 4};
    if (full_waves <= kTwoPartWaves && !one_part) return {32, 2};
    return {full_waves <= kHalfLaneWaves ? 32 : 64, 1};
}

// Runs a part of a split walk has room for: as many as let all groups of the
// launch be on the chip at once (the 160 KB of LDS of a CU over its share of
// the groups, less 4 KB for the kernel's own), within a block's 64 KB.
// Too few make a part wait for the one before it (4096 particles, eight parts,
// quadrupoles: 24 runs 0.243, 32 runs 0.169 ms), too many make a group wait for a
// place (49,152 particles, two parts of 32 targets: 48 runs 0.762, 64 runs,
// which leave room for five groups of six on a CU, 0.926 ms).
std::uint32_t split_runs(std::uint32_t groups, std::uint32_t run_bytes) {
    constexpr std::uint32_t kLds = 160 << 10, kBlockLds = 64 << 10, kOwn = 4 << 10, kCus = 256;
    const std::uint32_t share = std::min(kLds / ((groups + kCus - 1) / kCus), kBlockLds) - kOwn;
    return std::max(share / run_bytes, 4u);
}

// Workgroups are dispatched to the 8 XCDs in turn (block b to XCD b mod 8),
// and each XCD has its own L2. Neighbouring targets in Morton order visit the
// same deep nodes and leaves, so block b walks the logical block that gives
// each XCD runs of kXcdRun consecutive logical blocks, the runs dealt to the
// XCDs in turn: the nodes a wave pulls into an L2 are the ones its
// neighbours on that XCD need, while every XCD still sees all parts of the
// system (one contiguous eighth each would leave the XCD with the densest part
// finishing last). A bijection of [0, blocks): blocks past the last whole
// round of runs keep their own index.
constexpr std::uint32_t kXcds = 8;
constexpr std::uint32_t kXcdRun = 16;
__device__ __forceinline__ std::uint32_t xcd_block(std::uint32_t b, std::uint32_t blocks) {
    const std::uint32_t whole = blocks / (kXcds * kXcdRun) * (kXcds * kXcdRun);
    if (b >= whole) return b;
    const std::uint32_t x = b % kXcds, k = b / kXcds;
    return ((k / kXcdRun) * kXcds + x) * kXcdRun + k % kXcdRun;
}

// One target's walk state: FP32 position relative to the root centre and
// offset from its leaf centre, its leaf, Kahan sums and the running partial.
struct WalkTarget {
    float4 xi, oi;
    std::uint32_t own;
    float sx, sy, sz, kx, ky, kz, px, py, pz;
    // Accepted nodes and particle-particle terms: at most M and n.
    std::uint32_t pc, pp;
};

// Separation of the target from a node's centre of mass, and its square.
__device__ __forceinline__ float separation(const WalkTarget& t, const float4& com, float& dx,
                                            float& dy, float& dz) {
    dx = com.x - t.xi.x;
    dy = com.y - t.xi.y;
    dz = com.z - t.xi.z;
    return __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
}

// An accepted node's term (tree_walk.cpp:20-83): monopole, optionally quadrupole.
template<bool kSafe, bool kQuad>
__device__ __forceinline__ void accept(WalkTarget& t, float mass, const float4& Qa, const float4& Qb,
                                       float dx, float dy, float dz, float r2, float eps2) {
    // tree_walk.hpp:129-139 monopole.
    float r2e = r2 + eps2;
    if constexpr (kSafe) r2e = r2e > 0.f ? r2e : 1.f;
    const float inv = __builtin_amdgcn_rsqf(r2e);
    if constexpr (!kQuad) {
        const float f = (mass * inv) * (inv * inv);
        t.px = __builtin_fmaf(f, dx, t.px);
        t.py = __builtin_fmaf(f, dy, t.py);
        t.pz = __builtin_fmaf(f, dz, t.pz);
    } else {
        // Monopole plus tree_walk.hpp:156-181 in one update:
        // d (m inv^3 + 2.5 (d.Q d) inv^7) - (Q d) inv^5.
        const float i2 = inv * inv;
        const float i3 = i2 * inv;
        const float i5 = i3 * i2;
        const float i7 = i5 * i2;
        const float qx = __builtin_fmaf(Qa.z, dz, __builtin_fmaf(Qa.y, dy, Qa.x * dx));
        const float qy = __builtin_fmaf(Qb.x, dz, __builtin_fmaf(Qa.w, dy, Qa.y * dx));
        const float qz = __builtin_fmaf(Qb.y, dz, __builtin_fmaf(Qb.x, dy, Qa.z * dx));
        const float quadratic = __builtin_fmaf(dz, qz, __builtin_fmaf(dy, qy, dx * qx));
        const float g = __builtin_fmaf(2.5f * quadratic, i7, mass * i3);
        t.px = __builtin_fmaf(dx, g, __builtin_fmaf(qx, -i5, t.px));
        t.py = __builtin_fmaf(dy, g, __builtin_fmaf(qy, -i5, t.py));
        t.pz = __builtin_fmaf(dz, g, __builtin_fmaf(qz, -i5, t.pz));
    }
}

// Four consecutive leaf particles. The last round of a leaf still loads four
// (leaf_rel holds kLeafPad spare entries past the last particle).
struct LeafRound {
    float4 q[4];
};
__device__ __forceinline__ LeafRound load_round(const float4* __restrict__ leaf_rel, std::uint32_t j) {
    const float4* const q = leaf_rel + j;
    return LeafRound{{q[0], q[1], q[2], q[3]}};
}

// Particle-particle terms of leaf [b, e) for one target. The target is
// re-expressed against the leaf's centre cb in FP64 (ca: the centre of the
// target's own leaf).
template<bool kSafe>
__device__ __forceinline__ void leaf_pairs(WalkTarget& t, const double4& cb, double cax, double cay,
                                           double caz, const float4* __restrict__ leaf_rel,
                                           std::uint32_t b, std::uint32_t e, float eps2, std::uint32_t lane0) {
    const float tx = t.oi.x - static_cast<float>(cb.x - cax);
    const float ty = t.oi.y - static_cast<float>(cb.y - cay);
    const float tz = t.oi.z - static_cast<float>(cb.z - caz);
    auto pair = [&](const float4& q) {
        const float dx = q.x - tx, dy = q.y - ty, dz = q.z - tz;
        float r2 = __builtin_fmaf(dx, dx, eps2);
        r2 = __builtin_fmaf(dy, dy, r2);
        r2 = __builtin_fmaf(dz, dz, r2);
        if constexpr (kSafe) r2 = r2 > 0.f ? r2 : 1.f;
        const float inv = __builtin_amdgcn_rsqf(r2);
        const float f = (q.w * inv) * (inv * inv);
        t.px = __builtin_fmaf(f, dx, t.px);
        t.py = __builtin_fmaf(f, dy, t.py);
        t.pz = __builtin_fmaf(f, dz, t.pz);
    };
    // Whole rounds without a branch between the four terms, whose chains then
    // overlap; the sums still take them in index order. `lane0` is a zero the
    // compiler cannot see through: the sources come through the vector cache,
    // where loads return in order and a round can be on its way while the one
    // before it is summed. Read through the scalar cache, every round is a
    // miss (a leaf is a few lines that few waves share), waited for in full,
    // and pushes out the node records (16,384 particles, 16 targets a wave:
    // walk 0.488 -> 0.455 ms; 262,144 and 2,097,152 the same).
    std::uint32_t j = b;
    LeafRound v = load_round(leaf_rel, j + lane0);
    while (j + 4 <= e) {
        const LeafRound w = load_round(leaf_rel, j + 4 + lane0);
        pair(v.q[0]);
        pair(v.q[1]);
        pair(v.q[2]);
        pair(v.q[3]);
        v = w;
        j += 4;
    }
    if (j < e) {
        pair(v.q[0]);
        if (j + 1 < e) pair(v.q[1]);
        if (j + 2 < e) pair(v.q[2]);
    }
}

__device__ __forceinline__ void kahan(WalkTarget& t) {
    kahan(t.px, t.sx, t.kx);
    kahan(t.py, t.sy, t.ky);
    kahan(t.pz, t.sz, t.kz);
}

// A wave's stack of pending sibling lists, level d in lane d of a few vector
// registers. Writing is one v_writelane a word (no lane-compare, whatever the
// execution mask); the lane select goes through m0, since the instruction can
// read only one scalar register.
__device__ __forceinline__ void lane_write(std::uint32_t& reg, std::uint32_t value, std::uint32_t lane) {
    asm("s_mov_b32 m0, %2\n\ts_nop 0\n\tv_writelane_b32 %0, %1, m0"
        : "+v"(reg)
        : "s"(__builtin_amdgcn_readfirstlane(static_cast<int>(value))),
          "s"(__builtin_amdgcn_readfirstlane(static_cast<int>(lane)))
        : "m0");
}
__device__ __forceinline__ std::uint32_t lane_read(std::uint32_t reg, std::uint32_t lane) {
    return static_cast<std::uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(reg), static_cast<int>(lane)));
}

// The wave's counts (idle lanes count none): pairs and accepted nodes.
struct WalkCounts {
    unsigned long long pp, pc;
};
template<int kR> __device__ WalkCounts wave_counts(const WalkTarget (&t)[kR]) {
    unsigned long long v[2] = {0, 0};
#pragma unroll
    for (int r = 0; r < kR; ++r) {
        v[0] += t[r].pp;
        v[1] += t[r].pc;
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) v[k] += __shfl_xor(v[k], off, 64);
    }
    return {v[0], v[1]};
}

// One system's counts from a wave that walked several.
__device__ void add_counts(unsigned long long* __restrict__ stats, std::uint32_t seg,
                           unsigned long long pp, unsigned long long pc, unsigned long long visits,
                           unsigned long long slots) {
    unsigned long long* st = stats + 4 * static_cast<std::size_t>(seg);
    atomicAdd(&st[0], pp);
    atomicAdd(&st[1], pc);
    atomicAdd(&st[2], visits);
    atomicAdd(&st[3], slots);
}

// How much of a target's walk lies within d nodes of its own leaf, in the
// depth-first order: the cells a walk opens on each level lie around the
// target at the scale of that level, so the visits thin out as 1 / d beyond the
// nearest few hundred nodes, all of which it visits. Only the balance of a
// split walk rests on it. kNearNodes 256 to 2048 measured alike (16,384
// particles in four parts: walk 0.29 to 0.33 ms).
constexpr float kNearNodes = 512.f;
__device__ __forceinline__ float walk_weight(float d) {
    return d <= kNearNodes ? d : kNearNodes * (1.f + __logf(d / kNearNodes));
}
__device__ __forceinline__ float walk_reach(float weight) {
    return weight <= kNearNodes ? weight : kNearNodes * __expf(weight / kNearNodes - 1.f);
}

// Wave-coherent walk. Each of the first kLanes lanes owns kR targets (wave w
// owns the kLanes kR sorted particles from kLanes kR w, target r of lane l
// being kLanes r + l; with kLanes = 32 the other half of the wave holds none,
// which doubles the waves a small system gets). The wave goes through the nodes
// that any of its targets visits, in depth-first order, each loaded once; every
// target takes part in exactly the nodes of a walk of its own.
//
// The targets that reach a node are one lane mask per set r in scalar
// registers, not a next-node index per lane: all targets that opened a cell
// reach each of its children, and all that reached the cell go on after it. So
// opening a cell pushes the mask of its sibling list with the escape index that
// ends it, and reaching that index pops it. Which lanes accept is one compare
// and scalar logic, and the next node needs no reduction over the lanes.
//
// kMany: the targets may belong to several systems (a batch); the systems of
// a wave's targets are then walked one after another.
//
// kSplit > 1: a group of targets is walked by kSplit waves, the parts, each a
// range of the nodes. With one wave a group, a small launch leaves a SIMD a
// wave or two, which issue at half the rate a SIMD can and wait out every load,
// and the launch lasts as long as its slowest wave (16,384 particles, 1024 waves of 16
// targets: 0.30 ms on average, 0.51 the slowest, 183 running after three
// quarters of the time). A target's partial sum starts at zero after each leaf
// it visits, so its walk is a row of runs, leaf to leaf, that do not depend on
// one another: a part computes the runs that begin at a leaf among its nodes,
// each to its end, which may lie among the next part's (`tail`). Its own
// first nodes, up to the first leaf, are the part before's run; it walks them
// only to find that leaf. The runs of part 0 go into the Kahan sums as they
// end; those of the others wait in LDS until the sums of the part before are
// there, then go in in order: the sums see the same partials in the same
// order, and the results are the same bits. A part whose room in LDS is full
// waits for the part before it and then adds its runs directly; part 0 waits
// for nobody, so every wait ends. A visit is counted by the part that owns the node.
//
// The one-wave walk of one system is held to 64 vector registers, eight waves
// a SIMD (of 67 it would take; 2,097,152 particles: 8.6 -> 8.3 ms), that of
// several systems to 72, seven waves (of 75; 147 systems of 4096 to 16,384
// particles, a whole evaluation: 2.12 -> 2.01 ms; eight waves, with registers
// spilled, 1.99, but 0.77 instead of 0.76 ms for 40 systems).
template<int kR, bool kSafe, bool kQuad, int kLanes, bool kMany, int kSplit>
__global__ __launch_bounds__(kSplit == 1 ? kBlock : 64 * kSplit,
                             kSplit == 1 && kR == 1 ? (kMany ? 7 : 8) : 1) void tree_walk(
    const WalkNode* __restrict__ nodes, const QuadF* __restrict__ quads,
    const double4* __restrict__ node_geo,
    const float4* __restrict__ root_rel, const float4* __restrict__ leaf_rel,
    const std::uint32_t* __restrict__ leaf_of, const std::uint32_t* __restrict__ index,
    const std::uint32_t* __restrict__ counters, const std::uint32_t* __restrict__ seg_of,
    const std::uint32_t* __restrict__ seg_start, const std::uint32_t* __restrict__ first_node,
    std::uint32_t n, float eps2, double G, std::uint32_t runs,
    double* __restrict__ ax, double* __restrict__ ay, double* __restrict__ az,
    unsigned long long* __restrict__ stats, unsigned long long* __restrict__ wave_stats) {
    static_assert(kSplit == 1 || kR == 1);
    // The parts of a split walk have the same targets.
    constexpr int kSlots = kSplit == 1 ? kBlock : 64;
    const std::uint32_t wave = kSplit == 1
                                   ? xcd_block(blockIdx.x, gridDim.x) * (kBlock / 64) + threadIdx.x / 64
                                   : xcd_block(blockIdx.x, gridDim.x);
    const std::uint32_t part = kSplit == 1 ? 0u : __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const std::uint32_t lane = threadIdx.x & 63;
    const std::uint32_t M = counters[0];
    WalkTarget t[kR];
    std::uint32_t seg[kR];
    std::uint64_t todo[kR];  // targets whose system the wave has not walked yet
    // Each lane's targets' own leaf centres, read at every leaf visit: held in
    // LDS rather than registers (12 KB a block at two targets a lane) or
    // re-read from memory at each visit. A lane reads only its own slots.
    __shared__ double s_own[kR][3][kSlots];
    // What the parts of a split walk hand on: the chain of Kahan sums, the
    // counts, and who has finished.
    extern __shared__ float s_runs[];
    __shared__ float s_chain[6][kLanes];
    __shared__ unsigned long long s_count[kSplit][4];
    __shared__ std::uint32_t s_done[kSplit];
    const std::uint32_t slot = kSplit == 1 ? threadIdx.x : lane;
#pragma unroll
    for (int r = 0; r < kR; ++r) {
        const std::uint32_t i = wave * (kLanes * kR) + kLanes * r + lane;
        const bool valid = lane < kLanes && i < n;
        const std::uint32_t ic = valid ? i : n - 1;
        t[r].xi = root_rel[ic];
        t[r].oi = leaf_rel[ic];
        t[r].own = leaf_of[ic];
        const double4 ca = node_geo[t[r].own];
        if (part == 0) {
            s_own[r][0][slot] = ca.x;
            s_own[r][1][slot] = ca.y;
            s_own[r][2][slot] = ca.z;
        }
        seg[r] = kMany ? seg_of[ic] : 0u;
        todo[r] = __ballot(valid);
        t[r].sx = t[r].sy = t[r].sz = t[r].kx = t[r].ky = t[r].kz = 0.f;
        t[r].px = t[r].py = t[r].pz = 0.f;
        t[r].pc = t[r].pp = 0;
    }
    if constexpr (kSplit > 1) {
        if (threadIdx.x < kSplit) s_done[threadIdx.x] = 0;
        __syncthreads();
    }
    // An FP32 instruction with a scalar operand issues at half the rate of one
    // that reads only vector registers: eps^2 enters every term.
    asm volatile("" : "+v"(eps2));
    std::uint32_t lane0 = 0;  // leaf_pairs
    asm volatile("" : "+v"(lane0));
    std::uint32_t steps = 0;
    std::uint32_t systems = 0;   // systems walked by this wave
    std::uint32_t seg0 = 0;      // the first of them
    // Visits that accepted nothing (leaves and opened cells), one per target;
    // the other counts are kept per target.
    unsigned long long stopped = 0;
    // A split walk: the runs kept for the replay, whether the sums so far are
    // here yet (`direct`), and the targets whose last run ends with the walk.
    std::uint32_t kept = 0;
    bool direct = part == 0;
    std::uint64_t last_run = 0;
    float* const my_runs = s_runs + (part == 0 ? 0u : part - 1) * (runs * 3u * kLanes) + lane;
    auto keep_run = [&](WalkTarget& w) {
        float* const run = my_runs + kept * (3u * kLanes);
        run[0] = w.px;
        run[kLanes] = w.py;
        run[2 * kLanes] = w.pz;
        ++kept;
    };
    // The sums of the parts before this one, then this part's runs so far.
    auto join_chain = [&] {
        // Not an atomic load: one in the walk would keep the node records out of
        // the scalar cache.
        while (*static_cast<volatile std::uint32_t*>(&s_done[part - 1]) == 0) __builtin_amdgcn_s_sleep(1);
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        WalkTarget& w = t[0];
        if (lane < kLanes) {
            w.sx = s_chain[0][lane];
            w.sy = s_chain[1][lane];
            w.sz = s_chain[2][lane];
            w.kx = s_chain[3][lane];
            w.ky = s_chain[4][lane];
            w.kz = s_chain[5][lane];
        }
        for (std::uint32_t e = 0; e < kept; ++e) {
            const float* const run = my_runs + e * (3u * kLanes);
            kahan(run[0], w.sx, w.kx);
            kahan(run[kLanes], w.sy, w.ky);
            kahan(run[2 * kLanes], w.sz, w.kz);
        }
        direct = true;
    };
    while (true) {
        std::uint32_t own_seg = 0;
        std::uint64_t mask[kR];
        bool left = false;
#pragma unroll
        for (int r = kR - 1; r >= 0; --r) {
            if (todo[r] != 0) {
                left = true;
                if constexpr (kMany) {
                    own_seg = lane_read(seg[r], static_cast<std::uint32_t>(__builtin_ctzll(todo[r])));
                }
            }
        }
        if (!left) break;
#pragma unroll
        for (int r = 0; r < kR; ++r) {
            mask[r] = kMany ? __ballot(seg[r] == own_seg) & todo[r] : todo[r];
            todo[r] &= ~mask[r];
        }
        if (kMany && systems > 0) {
            // A second system: the counts so far belong to the one before it.
            const WalkCounts c = wave_counts(t);
            if (lane == 0) {
                add_counts(stats, seg0, c.pp, c.pc, c.pc + stopped,
                           static_cast<unsigned long long>(steps) * (kR * kLanes) / 64);
            }
#pragma unroll
            for (int r = 0; r < kR; ++r) t[r].pc = t[r].pp = 0;
            stopped = 0;
            steps = 0;
        }
        seg0 = own_seg;
        ++systems;
        // The stack: the escape index that ends a sibling list and its masks.
        std::uint32_t st_end = 0, st_lo[kR], st_hi[kR];
#pragma unroll
        for (int r = 0; r < kR; ++r) st_lo[r] = st_hi[r] = 0;
        std::uint32_t depth = 0, end = 0;  // the outermost list ends nowhere
        std::uint32_t cur = kMany ? __builtin_amdgcn_readfirstlane(first_node[seg_start[own_seg]]) : 0u;
        std::uint32_t stop = M;
        // A split walk: the targets whose current run is this part's, and
        // those still walking.
        std::uint64_t open = 0, alive = ~std::uint64_t{0};
        bool tail = false;
        std::uint32_t main_steps = 0, main_pc = 0, main_pp = 0;
        unsigned long long main_stopped = 0;
        auto up = [&] {
            // The end of one or more sibling lists: back to the masks of the
            // lists they lie in (cur > 0, so never past the outermost).
            while (cur == end) {
                --depth;
                end = lane_read(st_end, depth);
#pragma unroll
                for (int r = 0; r < kR; ++r) {
                    mask[r] = static_cast<std::uint64_t>(lane_read(st_lo[r], depth)) |
                              static_cast<std::uint64_t>(lane_read(st_hi[r], depth)) << 32;
                    if constexpr (kSplit > 1) mask[r] &= alive;
                }
            }
        };
        auto open_cell = [&](std::uint32_t next, const std::uint64_t (&rest)[kR]) {
            lane_write(st_end, end, depth);
#pragma unroll
            for (int r = 0; r < kR; ++r) {
                lane_write(st_lo[r], static_cast<std::uint32_t>(mask[r]), depth);
                lane_write(st_hi[r], static_cast<std::uint32_t>(mask[r] >> 32), depth);
                mask[r] = rest[r];
            }
            ++depth;  // at most 21 levels
            end = next;
        };
        if constexpr (kSplit > 1) {
            const std::uint32_t first = static_cast<std::uint32_t>(__builtin_ctzll(mask[0]));
            const std::uint32_t last = 63u - static_cast<std::uint32_t>(__builtin_clzll(mask[0]));
            const std::uint32_t at = wave * kLanes + (kSplit == 2 ? first : (first + last) / 2);
            const std::uint32_t home = __builtin_amdgcn_readfirstlane(leaf_of[at]);
            const std::uint32_t root = cur;
            const std::uint32_t system_end = kMany ? seg_start[own_seg + 1] : n;
            const std::uint32_t node_end =
                system_end < n ? __builtin_amdgcn_readfirstlane(first_node[system_end]) : M;
            const float left = walk_weight(static_cast<float>(home - root));
            const float right = walk_weight(static_cast<float>(node_end - home));
            // The node at which part k begins.
            auto cut = [&](std::uint32_t k) {
                if (kSplit == 2) return home;
                const float w = (left + right) * static_cast<float>(k) / kSplit - left;
                const float d = w < 0 ? -walk_reach(-w) : walk_reach(w);
                const float node = fminf(fmaxf(static_cast<float>(home) + d, static_cast<float>(root)),
                                         static_cast<float>(node_end));
                return static_cast<std::uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(node)));
            };
            if (part + 1 < kSplit) stop = cut(part + 1);
            open = part == 0 ? mask[0] : 0;
            const std::uint32_t begin = part > 0 ? cut(part) : 0u;
            if (part > 0) {
                // Down to this part's first node.
                while (cur < begin) {
                    const float4 na = nodes[cur].a;
                    const uint4 nb = nodes[cur].b;
                    const std::uint32_t next = max(nb.y, cur + 1);
                    if (next <= begin) {
                        cur = next;
                        continue;
                    }
                    float dx, dy, dz;
                    const float r2 = separation(t[0], na, dx, dy, dz);
                    const std::uint64_t rest[kR] = {mask[0] & ~__ballot(r2 >= __builtin_bit_cast(float, nb.x))};
                    if (rest[0] == 0) {
                        cur = next;
                        up();
                        break;
                    }
                    open_cell(next, rest);
                    ++cur;
                }
                depth = __builtin_amdgcn_readfirstlane(depth);
                end = __builtin_amdgcn_readfirstlane(end);
            }
        }
        while (true) {
            // cur only ever grows, so the loop ends whatever the records hold.
            while (cur < stop) {
                ++steps;
                const float4 na = nodes[cur].a;
                const uint4 nb = nodes[cur].b;
                float4 qa{}, qb{};
                if constexpr (kQuad) {
                    qa = quads[cur].a;
                    qb = quads[cur].b;
                }
                // Every scalar load of the iteration is issued here and waited for once;
                // left to itself the compiler sinks them into the branches below, one
                // dependent wait each.
                asm volatile("" ::"s"(na.x), "s"(na.y), "s"(na.z), "s"(na.w), "s"(nb.x), "s"(nb.y), "s"(nb.z),
                             "s"(nb.w));
                if constexpr (kQuad) {
                    asm volatile("" ::"s"(qa.x), "s"(qa.y), "s"(qa.z), "s"(qa.w), "s"(qb.x), "s"(qb.y),
                                 "s"(qb.z), "s"(qb.w));
                }
                const float acc = __builtin_bit_cast(float, nb.x);
                std::uint64_t rest[kR], any = 0;
#pragma unroll
                for (int r = 0; r < kR; ++r) {
                    rest[r] = 0;
                    if (kR > 1 && mask[r] == 0) continue;
                    float dx, dy, dz;
                    const float r2 = separation(t[r], na, dx, dy, dz);
                    const std::uint64_t far = __ballot(r2 >= acc) & mask[r];
                    rest[r] = mask[r] & ~far;
                    any |= rest[r];
                    if (__builtin_amdgcn_inverse_ballot_w64(far)) {
                        accept<kSafe, kQuad>(t[r], na.w, qa, qb, dx, dy, dz, r2, eps2);
                        ++t[r].pc;
                    }
                }
                // The successor when nothing opens: an escape index always lies past its
                // node; the maximum only keeps a corrupted record from looping.
                const std::uint32_t step = cur + 1;
                const std::uint32_t next = max(nb.y, step);
                std::uint32_t go = next;
                if (any != 0) {
#pragma unroll
                    for (int r = 0; r < kR; ++r) stopped += __popcll(rest[r]);
                    if (nb.w != 0) {
                        const double4 cb = node_geo[cur];
                        const std::uint32_t b = nb.z, e = nb.z + nb.w;
#pragma unroll
                        for (int r = 0; r < kR; ++r) {
                            if (rest[r] == 0) continue;
                            if (__builtin_amdgcn_inverse_ballot_w64(rest[r])) {
                                leaf_pairs<kSafe>(t[r], cb, s_own[r][0][slot], s_own[r][1][slot],
                                                  s_own[r][2][slot], leaf_rel, b, e, eps2, lane0);
                                if constexpr (kSplit == 1) {
                                    kahan(t[r]);
                                } else if (__builtin_amdgcn_inverse_ballot_w64(open)) {
                                    if (direct) {
                                        kahan(t[r]);
                                    } else {
                                        keep_run(t[r]);
                                    }
                                }
                                t[r].px = t[r].py = t[r].pz = 0.f;
                                t[r].pp += nb.w - (t[r].own == cur ? 1u : 0u);
                            }
                            if constexpr (kSplit > 1) {
                                if (tail) {
                                    open &= ~rest[r];
                                    alive = open;
                                    mask[r] &= open;
                                    if (open == 0) stop = 0;
                                } else {
                                    open |= rest[r];
                                }
                                if (!direct && __ballot(kept == runs) != 0) {
                                    join_chain();
                                }
                            }
                        }
                    } else {
                        // Open: the children for those that did, then everyone here
                        // goes on at `next`.
                        open_cell(next, rest);
                        go = step;
                    }
                }
                cur = go;
                up();
            }
            if constexpr (kSplit == 1) break;
            if (tail || part + 1 == kSplit || open == 0) break;
            // Past this part's nodes: only the runs already open go on, each to
            // its end. The part that owns these nodes counts them.
            tail = true;
            main_steps = steps;
            main_stopped = stopped;
            main_pc = t[0].pc;
            main_pp = t[0].pp;
            alive = open;
            mask[0] &= open;
            stop = M;
        }
        if constexpr (kSplit > 1) {
            if (tail) {
                steps = main_steps;
                stopped = main_stopped;
                t[0].pc = main_pc;
                t[0].pp = main_pp;
            }
            last_run |= open;
        }
    }
    if constexpr (kSplit > 1) {
        if (__builtin_amdgcn_inverse_ballot_w64(last_run)) {
            if (direct) {
                kahan(t[0]);
            } else {
                keep_run(t[0]);
            }
        }
        if (!direct) join_chain();
    } else {
#pragma unroll
        for (int r = 0; r < kR; ++r) kahan(t[r]);
    }
    // Counts: a wave inside one system writes its sums to its own slot, summed
    // per system by walk_counts (atomics on one address would serialise every
    // wave); a wave spanning systems adds them per system.
    const WalkCounts c = wave_counts(t);
    unsigned long long count[4] = {c.pp, c.pc, c.pc + stopped, steps};
    const bool mixed = kMany && systems > 1;
    if (mixed) {
        if (lane == 0) add_counts(stats, seg0, count[0], count[1], count[2], count[3] * (kR * kLanes) / 64);
        for (int k = 0; k < 4; ++k) count[k] = 0;
    }
    if constexpr (kSplit > 1) {
        if (part + 1 < kSplit) {
            if (lane < kLanes) {
                s_chain[0][lane] = t[0].sx;
                s_chain[1][lane] = t[0].sy;
                s_chain[2][lane] = t[0].sz;
                s_chain[3][lane] = t[0].kx;
                s_chain[4][lane] = t[0].ky;
                s_chain[5][lane] = t[0].kz;
            }
            if (lane == 0) {
                for (int k = 0; k < 4; ++k) s_count[part][k] = count[k];
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            if (lane == 0) *static_cast<volatile std::uint32_t*>(&s_done[part]) = 1;
            return;
        }
        for (int q = 0; q + 1 < kSplit; ++q) {
            for (int k = 0; k < 4; ++k) count[k] += s_count[q][k];
        }
    }
#pragma unroll
    for (int r = 0; r < kR; ++r) {
        const std::uint32_t i = wave * (kLanes * kR) + kLanes * r + lane;
        if (lane < kLanes && i < n) {
            const std::uint32_t dst = index[i];
            ax[dst] = G * (static_cast<double>(t[r].sx) - static_cast<double>(t[r].kx));
            ay[dst] = G * (static_cast<double>(t[r].sy) - static_cast<double>(t[r].ky));
            az[dst] = G * (static_cast<double>(t[r].sz) - static_cast<double>(t[r].kz));
        }
    }
    if (lane == 0) {
        unsigned long long* mine_slot = wave_stats + 4 * static_cast<std::size_t>(wave);
        mine_slot[0] = count[0];
        mine_slot[1] = count[1];
        mine_slot[2] = count[2];
        mine_slot[3] = count[3] * (kR * kLanes) / 64;  // lane-target slots, 64 per count
    }
}

// One block per system: the wave slots over its particle range, summed (a wave
// spanning two systems left zeros and added its counts directly).
__global__ __launch_bounds__(kBlock) void walk_counts(const unsigned long long* __restrict__ wave_stats,
                                                      std::uint32_t waves, std::uint32_t per_wave,
                                                      const std::uint32_t* __restrict__ seg_start,
                                                      unsigned long long* __restrict__ stats) {
    __shared__ unsigned long long s[4][kBlock];
    const std::uint32_t seg = blockIdx.x;
    std::uint32_t w0 = 0, w1 = waves;
    if (seg_start != nullptr) {
        w0 = seg_start[seg] / per_wave;
        w1 = min(waves, (seg_start[seg + 1] + per_wave - 1) / per_wave);
    }
    unsigned long long acc[4] = {0, 0, 0, 0};
    for (std::uint32_t w = w0 + threadIdx.x; w < w1; w += kBlock) {
        for (int c = 0; c < 4; ++c) acc[c] += wave_stats[4 * static_cast<std::size_t>(w) + c];
    }
    for (int c = 0; c < 4; ++c) s[c][threadIdx.x] = acc[c];
    __syncthreads();
    for (int h = kBlock / 2; h > 0; h >>= 1) {
        if (static_cast<int>(threadIdx.x) < h) {
            for (int c = 0; c < 4; ++c) s[c][threadIdx.x] += s[c][threadIdx.x + h];
        }
        __syncthreads();
    }
    if (threadIdx.x < 4) atomicAdd(&stats[4 * static_cast<std::size_t>(seg) + threadIdx.x], s[threadIdx.x][0]);
}

template<typename T> T* carve(char*& p, std::size_t count) {
    T* out = reinterpret_cast<T*>(p);
    p += (sizeof(T) * count + 255) & ~static_cast<std::size_t>(255);
    return out;
}

struct Layout {
    // Per particle.
    std::uint8_t* d;
    std::uint8_t* leaf_level;
    std::uint32_t* chain;
    std::uint32_t* first_node;
    std::uint32_t* leaf_of;
    double4* sorted;
    float4* root_rel;
    float4* leaf_rel;
    std::uint32_t* scan_scratch;
    // Per node.
    std::uint32_t* begin;
    std::uint32_t* count;
    std::uint32_t* next;
    std::uint8_t* level;
    std::uint32_t* children;  // 8 per node: an internal node's children in DFS order, then kNoChild
    double4* geo;
    double4* moment;
    WalkNode* walk;
    double* quad64;  // 6 per node, null without quadrupoles
    QuadF* quadf;
    // Counters.
    std::uint32_t* c32;
    unsigned long long* c64;
    uint2* block_counts;               // per block of tree_chains: {leaves, depth}
    unsigned long long* wave_stats;    // per walk wave: {pp, pc, visits, steps}
};

std::size_t node_bound(std::uint64_t n, std::uint64_t cap) {
    // Leaves partition the particles (<= n); internal nodes of one level are
    // disjoint cells of > cap particles (<= n / (cap + 1) per level, 21 levels).
    const std::uint64_t by_levels = n + 21 * (n / (cap + 1)) + 22;
    const std::uint64_t by_chains = 22 * n;
    return static_cast<std::size_t>(std::min(by_levels, by_chains));
}

// Bytes of one tree arena for n particles, `nodes` node slots and `segments` systems.
std::size_t layout_bytes(std::uint64_t n, std::size_t nodes, bool quadrupole, std::uint32_t segments) {
    // Every carved array is rounded up to 256 bytes: 22 arrays of padding.
    const std::size_t per_particle = 2 * n + 3 * 4 * n + 32 * n + 2 * 16 * n + 16 * kLeafPad +
                                     4 * scan_scratch_words(n);
    const std::size_t per_quad = quadrupole ? 6 * sizeof(double) + sizeof(QuadF) : 0;
    const std::size_t per_node = nodes * (4 * 3 + 1 + 4 * kMaxChildren + 32 + 32 + sizeof(WalkNode) + per_quad);
    const std::size_t counters = 16 + 8 * 4 * static_cast<std::size_t>(segments) +
                                 8 * ((n + kBlock - 1) / kBlock) + 512;
    return per_particle + per_node + counters + 22 * 256 + 64;
}

Layout layout(orr_ctx* ctx, std::uint64_t n, std::size_t nodes, bool quadrupole, std::uint32_t segments,
              bool allocate) {
    const std::size_t bytes = layout_bytes(n, nodes, quadrupole, segments);
    if (allocate) ctx->tree_work.reserve(bytes);
    char* p = static_cast<char*>(ctx->tree_work.ptr);
    Layout L{};
    L.d = carve<std::uint8_t>(p, n);
    L.leaf_level = carve<std::uint8_t>(p, n);
    L.chain = carve<std::uint32_t>(p, n);
    L.first_node = carve<std::uint32_t>(p, n);
    L.leaf_of = carve<std::uint32_t>(p, n);
    L.sorted = carve<double4>(p, n);
    L.root_rel = carve<float4>(p, n);
    L.leaf_rel = carve<float4>(p, n + kLeafPad);
    L.scan_scratch = carve<std::uint32_t>(p, scan_scratch_words(n));
    L.begin = carve<std::uint32_t>(p, nodes);
    L.count = carve<std::uint32_t>(p, nodes);
    L.next = carve<std::uint32_t>(p, nodes);
    L.level = carve<std::uint8_t>(p, nodes);
    L.children = carve<std::uint32_t>(p, kMaxChildren * nodes);
    L.geo = carve<double4>(p, nodes);
    L.moment = carve<double4>(p, nodes);
    L.walk = carve<WalkNode>(p, nodes);
    if (quadrupole) {
        L.quad64 = carve<double>(p, 6 * nodes);
        L.quadf = carve<QuadF>(p, nodes);
    }
    L.c32 = carve<std::uint32_t>(p, 4);
    L.c64 = carve<unsigned long long>(p, 4 * static_cast<std::size_t>(segments));
    L.block_counts = carve<uint2>(p, (n + kBlock - 1) / kBlock);
    // The walk's counts lie where the chain lengths were, which nothing reads once
    // the chains are placed: 32 bytes a wave of at least kMinLanes targets, or of a
    // block of four waves of twice that, in 4 bytes a particle (at least 256).
    static_assert(32 <= 4 * kMinLanes && 4 * 32 <= 256);
    L.wave_stats = reinterpret_cast<unsigned long long*>(L.chain);
    return L;
}

}  // namespace

std::size_t tree_bytes(std::uint64_t n, std::uint64_t leaf_capacity, bool quadrupole,
                       std::uint32_t segments) {
    if (n == 0) return 0;
    // As tree_evaluate_segments sizes its arena.
    const std::uint64_t cap = std::min<std::uint64_t>(std::max<std::uint64_t>(leaf_capacity, 1), n);
    const std::size_t bound = node_bound(n, cap) + 22 * static_cast<std::size_t>(segments);
    return layout_bytes(n, bound, quadrupole, segments);
}

namespace {

// Every launch of one evaluation on ctx->stream, no host synchronisation: the
// part a graph captures.
void tree_enqueue(orr_ctx* ctx, const orr_tree_args& a, const SegmentView& segs,
                  unsigned long long* seg_stats) {
    const std::uint64_t n = a.count;
    ctx->tree_last_n = n;
    ctx->tree_last_segments = segs.count;
    if (n == 0) return;
    if (n >= (std::uint64_t{1} << 31)) fail(ORR_ERR_LENGTH, "tree: 2^31 or more particles");
    // octree.cpp:189-194 parameter correction.
    const double theta = std::clamp(a.opening_angle, 0.0, 1.0);
    const std::uint64_t cap64 = std::max<std::uint64_t>(a.leaf_capacity, 1);
    const std::uint32_t cap = static_cast<std::uint32_t>(std::min<std::uint64_t>(cap64, n));
    const std::size_t bound = node_bound(n, cap) + 22 * static_cast<std::size_t>(segs.count);
    ctx->tree_last_bound = bound;
    ctx->tree_last_theta = theta;
    ctx->tree_last_quadrupole = a.quadrupole != 0;
    const Layout L = layout(ctx, n, bound, a.quadrupole != 0, segs.count, true);
    const std::uint32_t n32 = static_cast<std::uint32_t>(n);
    const std::uint32_t blocks = (n32 + kBlock - 1) / kBlock;
    const std::uint32_t node_blocks = static_cast<std::uint32_t>(std::min<std::size_t>(4096, (bound + kBlock - 1) / kBlock));
    const std::uint32_t* seg_of = segs.count > 1 ? segs.seg_of : nullptr;
    const std::uint32_t* seg_start = segs.count > 1 ? segs.start : nullptr;
    unsigned long long* counts64 = seg_stats != nullptr ? seg_stats : L.c64;

    morton_enqueue_segments(ctx, a.x, a.y, a.z, n, segs, a.m);
    const std::uint64_t* codes = ctx->order_codes.as<std::uint64_t>();
    const std::uint32_t* index = ctx->order_index.as<std::uint32_t>();
    const double* cube = ctx->order_bbox.as<double>();
    {
        PhaseTimer t(ctx, kBuild);
        hipLaunchKernelGGL(tree_levels, dim3(blocks), dim3(kBlock), 0, ctx->stream, codes, seg_of, n32,
                           L.d, L.c32, seg_stats != nullptr ? nullptr : L.c64, 4 * segs.count);
        ORR_LAUNCHED("tree_levels");
        hipLaunchKernelGGL(tree_chain, dim3(blocks), dim3(kBlock), 0, ctx->stream, L.d, n32, cap,
                           L.chain, L.leaf_level);
        ORR_LAUNCHED("tree_chain");
        exclusive_scan_u32(ctx, L.chain, L.first_node, n, L.scan_scratch, &L.c32[0]);
        hipLaunchKernelGGL(tree_chains, dim3(blocks), dim3(kBlock), 0, ctx->stream, L.d,
                           L.leaf_level, L.chain, L.first_node, n32, L.block_counts, L.begin,
                           L.level);
        ORR_LAUNCHED("tree_chains");
        hipLaunchKernelGGL(tree_node_fill, dim3(node_blocks), dim3(kBlock), 0, ctx->stream, codes,
                           L.leaf_level, L.first_node, n32, seg_of, seg_start, cube, L.c32,
                           L.begin, L.level, L.count, L.next, L.geo, L.leaf_of);
        ORR_LAUNCHED("tree_node_fill");
    }
    {
        PhaseTimer t(ctx, kGather);
        hipLaunchKernelGGL(tree_gather, dim3(blocks), dim3(kBlock), 0, ctx->stream,
                           ctx->order_aos.as<double4>(), index, n32, cube, seg_of, L.leaf_of, L.geo,
                           L.sorted, L.root_rel, L.leaf_rel);
        ORR_LAUNCHED("tree_gather");
    }
    {
        PhaseTimer t(ctx, kMoments);
        hipLaunchKernelGGL(tree_links, dim3(node_blocks + 1), dim3(kBlock), 0, ctx->stream, L.c32,
                           L.level, L.leaf_level, L.begin, L.next, L.block_counts, blocks, L.children,
                           L.moment);
        ORR_LAUNCHED("tree_links");
        hipLaunchKernelGGL(tree_moments, dim3(node_blocks), dim3(kBlock), 0, ctx->stream, L.c32,
                           L.level, L.leaf_level, L.begin, L.count, L.next, L.children, L.geo, L.sorted,
                           theta, cube, seg_of, seg_start, n32, L.moment, L.walk, L.quad64, L.quadf);
        ORR_LAUNCHED("tree_moments");
    }
    {
        PhaseTimer t(ctx, kWalk);
        const float eps2 = static_cast<float>(a.softening_squared);
        const bool safe = !(a.softening_squared > 0);
        const bool quad = a.quadrupole != 0;
        // One target a lane at every size (2^21 particles, quadrupoles: 8.3 ms
        // with one or two; below, one is faster); two only when configured.
        const int R = ctx->walk_targets_per_lane != 0 ? ctx->walk_targets_per_lane : 1;
        // Fewer targets a wave and several waves a group for a small launch;
        // zero in the context means choose by that rule. A target's walk and
        // sums do not depend on which targets share its wave nor on the parts,
        // so the results are the same bits either way.
        const std::uint64_t full_waves = (n + 64u * R - 1) / (64u * R);
        const WalkShape shape = ctx->walk_lanes != 0 || R != 1
                                    ? WalkShape{ctx->walk_lanes != 0 ? ctx->walk_lanes
                                                : full_waves <= kHalfLaneWaves ? 32 : 64, 1}
                                    : walk_shape(full_waves, segs.count > 1 ? segs.longest : n, theta);
        const int lanes = shape.lanes, split = shape.parts;
        using Walk = decltype(&tree_walk<1, true, true, 64, false, 1>);
        auto many = [&](auto r, auto l, auto p, auto sv, auto q) -> Walk {
            constexpr int kRr = decltype(r)::value, kLl = decltype(l)::value, kP = decltype(p)::value;
            constexpr bool kS = decltype(sv)::value, kQ = decltype(q)::value;
            return seg_of != nullptr ? tree_walk<kRr, kS, kQ, kLl, true, kP>
                                     : tree_walk<kRr, kS, kQ, kLl, false, kP>;
        };
        using Yes = std::true_type;
        using No = std::false_type;
        auto pick = [&](auto r, auto l, auto p) -> Walk {
            return safe ? (quad ? many(r, l, p, Yes{}, Yes{}) : many(r, l, p, Yes{}, No{}))
                        : (quad ? many(r, l, p, No{}, Yes{}) : many(r, l, p, No{}, No{}));
        };
        using One = std::integral_constant<int, 1>;
        using Two = std::integral_constant<int, 2>;
        using Four = std::integral_constant<int, 4>;
        using Eight = std::integral_constant<int, 8>;
        using Quarter = std::integral_constant<int, 16>;
        using Half = std::integral_constant<int, 32>;
        using Full = std::integral_constant<int, 64>;
        const Walk walk = R == 2         ? (lanes == 32 ? pick(Two{}, Half{}, One{}) : pick(Two{}, Full{}, One{}))
                          : split == 8   ? pick(One{}, Quarter{}, Eight{})
                          : split == 4   ? pick(One{}, Quarter{}, Four{})
                          : split == 2   ? pick(One{}, Half{}, Two{})
                          : lanes == 32  ? pick(One{}, Half{}, One{})
                                         : pick(One{}, Full{}, One{});
        const std::uint32_t per_wave = static_cast<std::uint32_t>(lanes * R);
        const std::uint32_t groups = split == 1 ? kBlock / 64 : 1;  // a block
        const std::uint32_t per_block = groups * per_wave;
        const std::uint32_t walk_blocks = (n32 + per_block - 1) / per_block;
        const std::uint32_t run_bytes = 12u * static_cast<std::uint32_t>(lanes * (split - 1));
        const std::uint32_t runs = split == 1 ? 0 : split_runs(walk_blocks, run_bytes);
        hipLaunchKernelGGL(walk, dim3(walk_blocks), dim3(split == 1 ? kBlock : 64 * split),
                           static_cast<std::size_t>(runs) * run_bytes, ctx->stream, L.walk, L.quadf, L.geo, L.root_rel, L.leaf_rel, L.leaf_of, index, L.c32, seg_of,
                           seg_start, L.first_node, n32, eps2, a.gravitational_constant, runs, a.ax,
                           a.ay, a.az, counts64, L.wave_stats);
        ORR_LAUNCHED("tree_walk");
        hipLaunchKernelGGL(walk_counts, dim3(segs.count), dim3(kBlock), 0, ctx->stream,
                           L.wave_stats, walk_blocks * groups, per_wave, seg_start, counts64);
        ORR_LAUNCHED("walk_counts");
    }
}

// The counts and tree summary of the evaluation last enqueued on ctx (syncs).
void tree_read_stats(orr_ctx* ctx, unsigned long long* seg_stats, orr_tree_stats* stats) {
    const std::uint64_t n = ctx->tree_last_n;
    const std::uint32_t segments = ctx->tree_last_segments;
    if (n == 0) return;
    const Layout L = layout(ctx, n, ctx->tree_last_bound, ctx->tree_last_quadrupole, segments, false);
    const unsigned long long* counts64 = seg_stats != nullptr ? seg_stats : L.c64;
    std::uint32_t c32[4];
    std::vector<unsigned long long> c64(4 * static_cast<std::size_t>(segments));
    ORR_HIP(hipMemcpyAsync(c32, L.c32, sizeof(c32), hipMemcpyDeviceToHost, ctx->stream));
    ORR_HIP(hipMemcpyAsync(c64.data(), counts64, c64.size() * sizeof(unsigned long long),
                           hipMemcpyDeviceToHost, ctx->stream));
    ctx->sync();
    stats->node_count = c32[0];
    stats->leaf_count = c32[1];
    stats->depth = c32[2];
    for (std::uint32_t sgm = 0; sgm < segments; ++sgm) {
        stats->particle_particle += c64[4 * sgm];
        stats->particle_cell += c64[4 * sgm + 1];
        stats->node_visits += c64[4 * sgm + 2];
        stats->wave_steps += c64[4 * sgm + 3];
    }
    ctx->last_tree = *stats;
}

}  // namespace

void tree_evaluate_segments(orr_ctx* ctx, const orr_tree_args& a, const SegmentView& segs,
                            unsigned long long* seg_stats, orr_tree_stats* stats) {
    if (stats != nullptr) std::memset(stats, 0, sizeof(*stats));
    ctx->last_tree = orr_tree_stats{};
    tree_enqueue(ctx, a, segs, seg_stats);
    if (stats != nullptr) tree_read_stats(ctx, seg_stats, stats);
}

// One system: replayed as a captured graph where run_captured allows (the
// key: every argument and the walk setting).
void tree_evaluate(orr_ctx* ctx, const orr_tree_args& a, orr_tree_stats* stats) {
    if (stats != nullptr) std::memset(stats, 0, sizeof(*stats));
    ctx->last_tree = orr_tree_stats{};
    if (a.count == 0) {
        tree_enqueue(ctx, a, SegmentView{}, nullptr);
        return;
    }
    std::vector<unsigned char> key;
    for (const void* p : {static_cast<const void*>(a.x), static_cast<const void*>(a.y),
                          static_cast<const void*>(a.z), static_cast<const void*>(a.m),
                          static_cast<const void*>(a.ax), static_cast<const void*>(a.ay),
                          static_cast<const void*>(a.az)}) {
        key_add(key, p);
    }
    key_add(key, a.count);
    key_add(key, a.softening_squared);
    key_add(key, a.gravitational_constant);
    key_add(key, a.opening_angle);
    key_add(key, a.leaf_capacity);
    key_add(key, a.quadrupole);
    key_add(key, ctx->walk_targets_per_lane);
    key_add(key, ctx->walk_lanes);
    run_captured(ctx, ctx->tree_graph, std::move(key),
                 [&] { tree_enqueue(ctx, a, SegmentView{}, nullptr); });
    if (stats != nullptr) tree_read_stats(ctx, nullptr, stats);
}

void tree_copy_segment_counts(orr_ctx* ctx, std::uint64_t* out) {
    const std::uint64_t n = ctx->tree_last_n;
    const std::size_t words = 4 * static_cast<std::size_t>(ctx->tree_last_segments);
    if (n == 0 || ctx->tree_work.ptr == nullptr) {
        for (std::size_t k = 0; k < words; ++k) out[k] = 0;
        return;
    }
    const Layout L = layout(ctx, n, ctx->tree_last_bound, ctx->tree_last_quadrupole,
                            ctx->tree_last_segments, false);
    static_assert(sizeof(unsigned long long) == sizeof(std::uint64_t));
    ORR_HIP(hipMemcpyAsync(out, L.c64, words * sizeof(std::uint64_t), hipMemcpyDeviceToHost,
                           ctx->stream));
    ctx->sync();
}

void tree_copy_quadrupoles(orr_ctx* ctx, double* out) {
    const std::uint64_t n = ctx->tree_last_n;
    if (n == 0 || ctx->tree_work.ptr == nullptr) return;
    if (!ctx->tree_last_quadrupole) fail(ORR_ERR_INVALID_ARGUMENT, "the last tree had no quadrupoles");
    const Layout L = layout(ctx, n, ctx->tree_last_bound, true, ctx->tree_last_segments, false);
    std::uint32_t M = 0;
    ORR_HIP(hipMemcpyAsync(&M, L.c32, sizeof(M), hipMemcpyDeviceToHost, ctx->stream));
    ctx->sync();
    if (M == 0) return;
    ORR_HIP(hipMemcpyAsync(out, L.quad64, 6 * sizeof(double) * M, hipMemcpyDeviceToHost, ctx->stream));
    ctx->sync();
}

void tree_copy_nodes(orr_ctx* ctx, double* mass, double* cx, double* cy, double* cz, double* acc,
                     std::uint64_t* next, std::uint64_t* first, std::uint64_t* count) {
    const std::uint64_t n = ctx->tree_last_n;
    if (n == 0 || ctx->tree_work.ptr == nullptr) return;
    const Layout L = layout(ctx, n, ctx->tree_last_bound, ctx->tree_last_quadrupole, ctx->tree_last_segments, false);
    std::uint32_t M = 0;
    ORR_HIP(hipMemcpyAsync(&M, L.c32, sizeof(M), hipMemcpyDeviceToHost, ctx->stream));
    ctx->sync();
    std::vector<double4> mom(M), geo(M);
    std::vector<WalkNode> walk(M);
    std::vector<std::uint32_t> nx(M), b(M), c(M);
    if (M > 0) {
        ORR_HIP(hipMemcpyAsync(mom.data(), L.moment, M * sizeof(double4), hipMemcpyDeviceToHost, ctx->stream));
        ORR_HIP(hipMemcpyAsync(geo.data(), L.geo, M * sizeof(double4), hipMemcpyDeviceToHost, ctx->stream));
        ORR_HIP(hipMemcpyAsync(walk.data(), L.walk, M * sizeof(WalkNode), hipMemcpyDeviceToHost, ctx->stream));
        ORR_HIP(hipMemcpyAsync(nx.data(), L.next, M * sizeof(std::uint32_t), hipMemcpyDeviceToHost, ctx->stream));
        ctx->sync();
    }
    const double theta = ctx->tree_last_theta;
    for (std::uint32_t k = 0; k < M; ++k) {
        if (mass) mass[k] = mom[k].w;
        if (cx) cx[k] = mom[k].x;
        if (cy) cy[k] = mom[k].y;
        if (cz) cz[k] = mom[k].z;
        if (acc) {
            // The FP64 radius of octree.cpp:374-387 (the walk holds it rounded to FP32).
            const double ox = mom[k].x - geo[k].x, oy = mom[k].y - geo[k].y, oz = mom[k].z - geo[k].z;
            const double offset = std::sqrt((ox * ox) + (oy * oy) + (oz * oz));
            if (!(theta > 0)) {
                acc[k] = std::numeric_limits<double>::infinity();
            } else {
                const double r = (geo[k].w / theta) + offset;
                acc[k] = r * r;
            }
        }
        if (next) next[k] = nx[k];
        if (first) first[k] = walk[k].b.z;
        if (count) count[k] = walk[k].b.w;
    }
}

}  // namespace orr
