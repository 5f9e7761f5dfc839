// Size limits of the library's 32-bit index spaces and of its launches (host-only, no HIP: the CPU tests compile it
// with g++).
//
// The EGG-kept adjacency is a CSR with int32 row offsets (Taubin, PCA and the normals' edge list index it
// with int32), and a mesh's corner lists (two entries per triangle corner) use uint32 offsets. A count past
// these limits would wrap and make the kernels index out of bounds, so the entry points refuse it with
// EGT_ERR_UNSUPPORTED instead.
//
// A launch's threads are a 32-bit count: HIP refuses 2^32 and more. Kernels with several threads per point reach that
// before the point count's own limit of 2^31 - 1: their work goes out in as many launches as it takes, or in another
// shape.
#pragma once
#include <cstdint>

namespace egt {

// Largest number of kept neighbour slots (CSR entries) of one handle, all clouds together.
constexpr int64_t CSR_MAX_ENTRIES = INT32_MAX;
// Largest triangle count of a mesh handle: 6 corner-list entries per triangle within int32.
constexpr int64_t MESH_MAX_TRIANGLES = INT32_MAX / 6;

// Null when a CSR of `total` entries fits, else the error message.
inline const char* csr_total_error(uint64_t total) {
    return total > (uint64_t)CSR_MAX_ENTRIES
               ? "the kept neighbour slots exceed 2^31 - 1 (int32 CSR offsets): split the point set or lower k"
               : nullptr;
}

// Null when a mesh of ntri triangles fits, else the error message.
inline const char* mesh_triangles_error(int64_t ntri) {
    return ntri > MESH_MAX_TRIANGLES ? "more than (2^31 - 1) / 6 triangles (int32 corner-list offsets)" : nullptr;
}

// Iterations that the Taubin passes of a small cloud run in one launch, at most: its pass counter is an int (two passes
// an iteration) and the launch has the GPU to itself for as long as it runs, up to about 10 s here. More iterations
// run a launch per pass.
constexpr int MAX_RESIDENT_ITERATIONS = 1 << 20;
inline bool resident_iterations(int iterations) { return iterations >= 1 && iterations <= MAX_RESIDENT_ITERATIONS; }

// Workgroups of 256 threads in one launch.
constexpr int64_t MAX_GROUPS = ((int64_t)1 << 32) / 256 - 1;

// launch(first, count) for consecutive ranges of at most `most` of `items` items.
template <class Launch>
void in_launches(int64_t items, int64_t most, Launch&& launch) {
    for (int64_t first = 0; first < items; first += most) launch(first, items - first < most ? items - first : most);
}

// Queries a wave of the wave-per-query search serves one after another. More of them reuse the ranges of the last
// box, fewer give more waves: a 10,000-point torus at k=40 0.105 ms with one query a wave against 0.117, 0.169 and
// 0.513 with 2, 4 and 16; 150,000 points 0.958, 0.939, 0.965 and 1.194; 1.5M points 6.93, 6.65, 6.57 and 6.78;
// 16M points (4 and 16) 52.1 and 53.3, a 16M-point cluster mixture 67.7 and 70.5. Where four would take more threads
// than a launch, 16 (as a chunk number for the launch in the kernel would: 46 spilled scalars against 42, a 4M-point
// mixture at k=64 16.35 -> 16.43 ms).
inline int queries_per_wave(int64_t queries) {
    return queries < 100000 ? 1 : queries < 300000 ? 2 : queries <= MAX_GROUPS / 4 * 64 ? 4 : 16;
}
// Its workgroups (four waves) per chunk of 64 queries, and the queries of one launch; a larger search runs a lane per
// query, whatever shape is named.
inline int wave_groups_per_chunk(int qpw) { return 16 / qpw; }
constexpr int64_t WAVE_MAX_QUERIES = MAX_GROUPS * 64;

}  // namespace egt
