/*
 * gz_results.hip -- results of a run formed on the device.
 *
 * Ranks, labels and BFS words leave the device arrays in original-id order
 * and in their final form, so that one copy into the caller's array ends a
 * getter (the reference formats them while it writes its output,
 * graphdata.c:1119-1138).  On the host the same work was a download of the
 * words, a gather through the id map and one through the out-degrees: 4.2 M
 * renumbered ranks took 23 ms, mostly cache misses and page faults of the
 * intermediate arrays; here it is one streaming kernel (16 or 24 bytes read
 * and 8 scattered per vertex) and the copy.
 */
#include "gz_host_internal.h"
#include "gz_internal.h"

namespace {

unsigned gz_result_blocks(uint64_t n)
{
    const uint64_t b = (n + GZ_BLOCK - 1) / GZ_BLOCK;
    return (unsigned)(b < 1 ? 1 : b > 65536 ? 65536 : b);
}

/* out[original id] = the vertex word, or (outdeg != nullptr) the rank:
 * props * outdeg', outdeg' = V for sinks. */
__global__ __launch_bounds__(GZ_BLOCK) void gz_k_result_words(const uint64_t* __restrict__ words,
                                                              const double* __restrict__ outdeg,
                                                              const uint64_t* __restrict__ original, uint64_t n,
                                                              uint64_t* __restrict__ out)
{
    const double nv = (double)n;
    for (uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n; v += (uint64_t)gridDim.x * blockDim.x) {
        uint64_t w = words[v];
        if (outdeg != nullptr) {
            const double od = outdeg[v];
            w = (uint64_t)__double_as_longlong(__longlong_as_double((long long)w) * (0.0 == od ? nv : od));
        }
        out[original != nullptr ? original[v] : v] = w;
    }
}

/* BFS words as parents (original ids, -1 for the root and unreached vertices)
 * and depths (UINT64_MAX unreached); either output may be null. */
__global__ __launch_bounds__(GZ_BLOCK) void gz_k_result_bfs(const uint64_t* __restrict__ words,
                                                            const uint64_t* __restrict__ original, uint64_t n,
                                                            int64_t* __restrict__ parents,
                                                            uint64_t* __restrict__ depths)
{
    for (uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n; v += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t w = words[v], at = original != nullptr ? original[v] : v;
        const uint64_t parent = w & GZ_BFS_PARENT_NONE; /* all ones in an unvisited word too */
        int64_t p = -1;
        if (parent != GZ_BFS_PARENT_NONE) p = (int64_t)(original != nullptr ? original[parent] : parent);
        if (parents != nullptr) parents[at] = p;
        if (depths != nullptr) depths[at] = w == GZ_BFS_UNVISITED ? ~0ull : w >> 48;
    }
}

struct gz_vertex_list {
    uint64_t v[64];
};

/* info[2 i], info[2 i + 1] = device vertex and out-degree of original vertex i
 * of the list. */
__global__ void gz_k_vertex_info(gz_vertex_list list, uint32_t count, const uint32_t* __restrict__ device_ids,
                                 const double* __restrict__ outdeg, uint64_t* __restrict__ info)
{
    const uint32_t i = threadIdx.x;
    if (i >= count) return;
    const uint64_t v = device_ids != nullptr ? (uint64_t)device_ids[list.v[i]] : list.v[i];
    info[2 * i] = v;
    info[2 * i + 1] = (uint64_t)outdeg[v];
}

}  // namespace

uint64_t* gz_result_buffer(int which)
{
    gz_scratch_reserve(0, gz_graph.num_vertices);
    return which ? gz_scratch.active_prefix : gz_scratch.active_vertices;
}

extern "C" void gz_dev_result_words(const uint64_t* words, const double* outdeg, const uint64_t* original, uint64_t n,
                                    uint64_t* out)
{
    if (n == 0) return;
    if (outdeg == nullptr && original == nullptr) {
        gz_copy_to_host(out, words, n * sizeof(uint64_t));
        return;
    }
    uint64_t* d = gz_result_buffer(0);
    hipLaunchKernelGGL(gz_k_result_words, dim3(gz_result_blocks(n)), dim3(GZ_BLOCK), 0, gz_stream, words, outdeg,
                       original, n, d);
    GZ_LAUNCH_CHECK();
    gz_copy_to_host(out, d, n * sizeof(uint64_t));
}

extern "C" void gz_dev_result_bfs(const uint64_t* words, const uint64_t* original, uint64_t n, int64_t* parents,
                                  uint64_t* depths)
{
    if (n == 0 || (parents == nullptr && depths == nullptr)) return;
    uint64_t* dd = depths ? gz_result_buffer(0) : nullptr;
    int64_t* dp = parents ? (int64_t*)gz_result_buffer(1) : nullptr;
    hipLaunchKernelGGL(gz_k_result_bfs, dim3(gz_result_blocks(n)), dim3(GZ_BLOCK), 0, gz_stream, words, original, n, dp,
                       dd);
    GZ_LAUNCH_CHECK();
    if (parents) gz_copy_to_host(parents, dp, n * sizeof(int64_t));
    if (depths) gz_copy_to_host(depths, dd, n * sizeof(uint64_t));
}

extern "C" void gz_dev_vertex_info(const uint64_t* vertices, uint32_t count, const uint32_t* device_ids,
                                   const double* outdeg, uint64_t* info)
{
    if (count == 0 || count > 64) return;
    gz_vertex_list list;
    for (uint32_t i = 0; i < count; ++i) list.v[i] = vertices[i];
    gz_scratch_reserve(0, gz_graph.num_vertices);
    uint64_t* d = gz_scratch.reduce_tmp + 1024; /* past the reduction slots, 128 words */
    hipLaunchKernelGGL(gz_k_vertex_info, dim3(1), dim3(64), 0, gz_stream, list, count, device_ids, outdeg, d);
    GZ_LAUNCH_CHECK();
    gz_copy_to_host(info, d, 2 * (size_t)count * sizeof(uint64_t));
}
