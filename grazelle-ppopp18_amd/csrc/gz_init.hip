/*
 * gz_init.hip -- device-side initialisation of vertex arrays and frontiers
 * (graph_helper_initialize_vertex_info, graphdata.c:279-287, and
 * graph_helper_create_and_initialize_frontiers, graphdata.c:290-319, with the
 * per-algorithm callbacks execution_pr.c:64-88, execution_cc.c:234-258,
 * execution_bfs.c:70-116).  Filling on the device keeps repeated runs (many
 * BFS roots) off PCIe.
 */
#include "gz_internal.h"
#include "gz_host_internal.h"

/* The start of a run in one launch each: the vertex arrays, the frontier
 * bitmaps (fwords words each; 0: left alone) and the reduce buffer's eight
 * words.  Separate fills were four to six launches of 2 us with gaps of 5 us,
 * 20 of the 370 us of a CC run on R-MAT s16. */
__device__ __forceinline__ void gz_reset_reduce(uint64_t* __restrict__ reduce)
{
    if (reduce != nullptr && blockIdx.x == 0 && threadIdx.x < 8) reduce[threadIdx.x] = 0;
}

/* PageRank: props = (1/V) / outdeg', accumulators 0, every frontier bit set. */
__global__ __launch_bounds__(GZ_BLOCK) void gz_k_pr_reset(double* __restrict__ props, double* __restrict__ acc,
                                                          const double* __restrict__ outdeg, uint64_t n,
                                                          uint64_t* __restrict__ has, uint64_t* __restrict__ wants,
                                                          uint64_t fwords, uint64_t* __restrict__ reduce)
{
    const uint64_t first = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (uint64_t)gridDim.x * blockDim.x;
    const double nv = (double)n;
    gz_reset_reduce(reduce);
    for (uint64_t v = first; v < n + 8; v += stride) {
        if (v < n) {
            const double od = outdeg[v];
            props[v] = (1.0 / nv) / (0.0 == od ? nv : od);
        } else {
            props[v] = 0.0;
        }
        acc[v] = 0.0;
    }
    for (uint64_t w = first; w < fwords; w += stride) {
        has[w] = ~0ull;
        wants[w] = ~0ull;
    }
}

/* CC: each vertex labelled with its original id, HasInfo* clear, every other
 * frontier bit set. */
__global__ __launch_bounds__(GZ_BLOCK) void gz_k_cc_reset(uint64_t* __restrict__ labels, uint64_t n,
                                                          const uint64_t* __restrict__ original,
                                                          uint64_t* __restrict__ next, uint64_t* __restrict__ has,
                                                          uint64_t* __restrict__ wants, uint64_t fwords,
                                                          uint64_t* __restrict__ reduce)
{
    const uint64_t first = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (uint64_t)gridDim.x * blockDim.x;
    gz_reset_reduce(reduce);
    for (uint64_t v = first; v < n; v += stride) labels[v] = original != nullptr ? original[v] : v;
    for (uint64_t w = first; w < fwords; w += stride) {
        next[w] = 0;
        has[w] = ~0ull;
        wants[w] = ~0ull;
    }
}

__global__ __launch_bounds__(GZ_BLOCK) void gz_k_fill(uint64_t* __restrict__ p, uint64_t value, uint64_t n)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = value;
}

/* The start of a BFS from `root` in one launch (execution_bfs.c:106-116 and
 * :70-102): every word unvisited but the root's (no parent), HasInfo* clear,
 * HasInfo = {root}, WantsInfo = every vertex but the root.  `original` is the
 * root's original id; its device vertex and out-degree go to info. */
__global__ __launch_bounds__(GZ_BLOCK) void gz_k_bfs_reset(uint64_t* __restrict__ words, uint64_t n,
                                                           uint64_t* __restrict__ acc, uint64_t* __restrict__ has,
                                                           uint64_t* __restrict__ wants, uint64_t fwords,
                                                           uint64_t original,
                                                           const uint32_t* __restrict__ device_ids,
                                                           const double* __restrict__ outdeg,
                                                           uint64_t* __restrict__ info,
                                                           uint64_t* __restrict__ reduce)
{
    gz_reset_reduce(reduce);
    const uint64_t root = device_ids != nullptr ? (uint64_t)device_ids[original] : original;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        __hip_atomic_store(&info[0], root, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
        __hip_atomic_store(&info[1], (uint64_t)outdeg[root], __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    const uint64_t first = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = first; i < n; i += stride) words[i] = (i == root) ? GZ_BFS_PARENT_NONE : GZ_BFS_UNVISITED;
    const uint64_t rw = root >> 6, rbit = 1ull << (root & 63);
    for (uint64_t w = first; w < fwords; w += stride) {
        acc[w] = 0;
        has[w] = (w == rw) ? rbit : 0ull;
        wants[w] = (w == rw) ? ~rbit : ~0ull;
    }
}

static unsigned gz_blocks_for(uint64_t n)
{
    uint64_t b = (n + GZ_BLOCK - 1) / GZ_BLOCK;
    if (b < 1) b = 1;
    if (b > 8192) b = 8192;
    return (unsigned)b;
}

/* Pinned, mapped: the device vertex and out-degree of the last start's root. */
static uint64_t* gz_bfs_info = nullptr;
static uint64_t* gz_bfs_info_dev = nullptr;
static uint64_t gz_bfs_info_root = ~0ull;

void gz_dev_bfs_reset(uint64_t* words, uint64_t n, uint64_t* acc, uint64_t* has, uint64_t* wants, uint64_t fwords,
                      uint64_t root, const uint32_t* device_ids, const double* outdeg, uint64_t* reduce)
{
    if (gz_bfs_info == nullptr) {
        GZ_CHECK(hipHostMalloc((void**)&gz_bfs_info, 2 * sizeof(uint64_t), hipHostMallocMapped | hipHostMallocCoherent));
        GZ_CHECK(hipHostGetDevicePointer((void**)&gz_bfs_info_dev, gz_bfs_info, 0));
    }
    gz_bfs_info_root = root;
    hipLaunchKernelGGL(gz_k_bfs_reset, dim3(gz_blocks_for(n > fwords ? n : fwords)), dim3(GZ_BLOCK), 0, gz_stream, words,
                       n, acc, has, wants, fwords, root, device_ids, outdeg, gz_bfs_info_dev,
                       reduce);
    GZ_LAUNCH_CHECK();
}

void gz_dev_bfs_start_forget(void) { gz_bfs_info_root = ~0ull; }

int gz_dev_bfs_start_info(uint64_t root, uint64_t* device_root, uint64_t* outdeg)
{
    if (gz_bfs_info == nullptr || root != gz_bfs_info_root) return 0;
    *device_root = gz_bfs_info[0];
    *outdeg = gz_bfs_info[1];
    return 1;
}

extern "C" void gz_dev_pr_reset(double* props, double* acc, const double* outdeg, uint64_t n, uint64_t* has,
                                uint64_t* wants, uint64_t fwords, uint64_t* reduce)
{
    hipLaunchKernelGGL(gz_k_pr_reset, dim3(gz_blocks_for(n + 8)), dim3(GZ_BLOCK), 0, gz_stream, props, acc, outdeg, n,
                       has, wants, fwords, reduce);
    GZ_LAUNCH_CHECK();
}

extern "C" void gz_dev_cc_reset(uint64_t* labels, uint64_t n, const uint64_t* original, uint64_t* next, uint64_t* has,
                                uint64_t* wants, uint64_t fwords, uint64_t* reduce)
{
    hipLaunchKernelGGL(gz_k_cc_reset, dim3(gz_blocks_for(n > fwords ? n : fwords)), dim3(GZ_BLOCK), 0, gz_stream, labels,
                       n, original, next, has, wants, fwords, reduce);
    GZ_LAUNCH_CHECK();
}

extern "C" void gz_dev_fill_u64(uint64_t* p, uint64_t value, uint64_t n)
{
    if (n == 0) return;
    hipLaunchKernelGGL(gz_k_fill, dim3(gz_blocks_for(n)), dim3(GZ_BLOCK), 0, gz_stream, p, value, n);
    GZ_LAUNCH_CHECK();
}

/* In-degrees from either layout: the pull list holds each destination's
 * in-edges as its vectors' valid lanes; in the push list every valid lane
 * names one destination. */
__global__ __launch_bounds__(GZ_BLOCK) void gz_k_indegrees(const gz_vec_t* __restrict__ vecs, uint64_t count,
                                                           int pull_layout, uint32_t* __restrict__ indeg)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (uint64_t)gridDim.x * blockDim.x) {
        const gz_lanes v = gz_load_vector(vecs, i);
        const uint64_t l[4] = {v.l0, v.l1, v.l2, v.l3};
        if (pull_layout) {
            uint32_t c = 0;
#pragma unroll
            for (int k = 0; k < 4; ++k) c += gz_lane_valid(l[k]) ? 1u : 0u;
            atomicAdd(&indeg[gz_shared_vertex(v)], c);
        } else {
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (gz_lane_valid(l[k])) atomicAdd(&indeg[gz_lane_id(l[k])], 1u);
        }
    }
}

extern "C" void gz_dev_indegrees(const gz_vec_t* vecs, uint64_t count, int pull_layout, uint32_t* indeg, uint64_t n)
{
    gz_device_zero(indeg, (n + 8) * sizeof(uint32_t));
    if (count == 0) return;
    hipLaunchKernelGGL(gz_k_indegrees, dim3(gz_blocks_for(count)), dim3(GZ_BLOCK), 0, gz_stream, vecs, count,
                       pull_layout, indeg);
    GZ_LAUNCH_CHECK();
}
