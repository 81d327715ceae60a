/*
 * gz_ingress.hip -- device Vector-Sparse ingress: the edge lists are built in
 * HBM instead of by the host packer.
 *
 * The reference loads -pull / -push files with a producer thread and one
 * packing consumer per layout (source/graphdata.c:595-951), which at a
 * billion edges is minutes of host time.  Here the same result is computed
 * as a device pipeline over 64-bit keys (group << b | neighbour), b = bits of
 * V-1:
 *   1. keys: drawn by the R-MAT kernel (the host generator's exact stream) or
 *      converted from uploaded (src, dst) pairs, optionally both directions; a
 *      self-loop becomes the all-ones key, itself a self-loop, which sorts last;
 *   2. LSD radix sort over the 2b key bits (pull: group = dst);
 *   3. drop the all-ones keys and duplicates (a key equal to its predecessor)
 *      and note each group's first and end position among the kept keys, in
 *      two passes over the keys (tile counts, then the write);
 *   4. vector counts ceil(deg / 4) and their exclusive scan = the CSR vector
 *      offsets;
 *   5. pack: edge i of group g at rank r goes to lane r % 4 of vector
 *      offsets[g] + r / 4, which is the flush rule of graphdata.c:679-686 on a
 *      group-sorted list (a vector closes when the shared vertex changes or it
 *      holds four edges);
 *   6. the push layout: the kept keys, in (dst, src) order, sorted again by
 *      their b source bits alone (the sort is stable); FP64 outdegrees are its
 *      group sizes (graphdata.c:814 counts sources of the pull file, which is
 *      the same number).
 * The result equals gz_edges_sort(..., dedupe) + gz_pack_vectors on the host
 * bit for bit, invalid lanes included (shared-vertex piece, neighbour 0).
 */
#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>
#include <rocprim/iterator/counting_iterator.hpp>
#include <rocprim/iterator/transform_iterator.hpp>

#include "grazelle_host.h"
#include "gz_host_internal.h"
#include "gz_internal.h"

namespace {

__device__ __forceinline__ uint64_t gz_splitmix64_dev(uint64_t x)
{
    x += 0x9e3779b97f4a7c15ull;
    x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ull;
    x = (x ^ (x >> 27)) * 0x94d049bb133111ebull;
    return x ^ (x >> 31);
}

/* The key (group << b | neighbour) of an edge, all ones for a self-loop when
 * `drop` (a renumbered graph counts self-loops first, gz_k_remap_keys then
 * drops them). */
__host__ __device__ __forceinline__ uint64_t gz_no_key(uint32_t b) { return b < 32 ? (1ull << (2 * b)) - 1ull : ~0ull; }

__device__ __forceinline__ uint64_t gz_edge_key(uint64_t g, uint64_t nbr, uint32_t b, int drop)
{
    return (drop && g == nbr) ? gz_no_key(b) : ((g << b) | nbr);
}

/* The R-MAT draw of rmat.c for edges [0, n): key (dst << b | src), and with
 * `both` also (src << b | dst) at the odd slot.  Ids are shifted by id_base
 * (one graph of a disjoint union). */
__global__ void gz_k_rmat_keys(uint64_t seed, uint64_t edge_offset, uint32_t scale, uint64_t nv, uint32_t ta,
                               uint32_t tb, uint32_t tc, uint64_t n, uint32_t b, int both, int drop,
                               uint64_t id_base, uint64_t* __restrict__ keys)
{
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += stride) {
        uint64_t x = gz_splitmix64_dev(seed ^ gz_splitmix64_dev(edge_offset + e));
        uint64_t s = 0, d = 0;
        for (uint32_t l = 0; l < scale; ++l) {
            if (l && (l & 3) == 0) x = gz_splitmix64_dev(x);
            const uint32_t u = (uint32_t)((x >> (16 * (l & 3))) & 0xffff);
            const uint32_t sb = (u >= tb) ? 1u : 0u;
            const uint32_t db = ((u >= ta && u < tb) || (u >= tc)) ? 1u : 0u;
            s = (s << 1) | sb;
            d = (d << 1) | db;
        }
        if (s >= nv) s %= nv;
        if (d >= nv) d %= nv;
        s += id_base;
        d += id_base;
        if (both) {
            keys[2 * e] = gz_edge_key(d, s, b, drop);
            keys[2 * e + 1] = gz_edge_key(s, d, b, drop);
        } else {
            keys[e] = gz_edge_key(d, s, b, drop);
        }
    }
}

/* The same for uploaded (src, dst) pairs; *bad becomes the smallest index of
 * an endpoint (word of `pairs`) that is not below nv. */
__global__ void gz_k_pairs_keys(const gz_u64x2* __restrict__ pairs, uint64_t n, uint32_t b, int both, int drop,
                                uint64_t nv, uint64_t* __restrict__ keys, unsigned long long* __restrict__ bad)
{
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += stride) {
        const gz_u64x2 sd = pairs[e];
        const uint64_t s = sd.x, d = sd.y;
        if (s >= nv || d >= nv) atomicMin(bad, (unsigned long long)(2 * e + (s >= nv ? 0 : 1)));
        if (both) {
            keys[2 * e] = gz_edge_key(d, s, b, drop);
            keys[2 * e + 1] = gz_edge_key(s, d, b, drop);
        } else {
            keys[e] = gz_edge_key(d, s, b, drop);
        }
    }
}

/* ---- sorted keys, tile by tile ------------------------------------------------
 * The passes below walk a sorted key array in tiles of GZ_TILE keys, a
 * wavefront taking GZ_TILE_ROWS rows of 64 consecutive keys with every row's
 * load in flight at once.  A key needs its neighbours: they come from the
 * next lanes, and from one extra load at each end of the wavefront's rows. */
#define GZ_TILE_ROWS 16
#define GZ_TILE_WAVE (GZ_TILE_ROWS * GZ_WAVE)
#define GZ_TILE (GZ_WAVES_PER_BLOCK * GZ_TILE_WAVE)

struct gz_tile_keys {
    uint64_t k[GZ_TILE_ROWS], before, after; /* before: the key ahead of the rows; after: the one behind */
};

/* The wavefront's keys of tile `tile`; positions past n read as `pad`. */
__device__ __forceinline__ uint64_t gz_tile_load(gz_tile_keys& t, const uint64_t* __restrict__ keys, uint64_t n,
                                                 uint64_t tile, uint64_t pad)
{
    const uint64_t base = tile * GZ_TILE + (uint64_t)(threadIdx.x / GZ_WAVE) * GZ_TILE_WAVE;
#pragma unroll
    for (int r = 0; r < GZ_TILE_ROWS; ++r) {
        const uint64_t i = base + (uint64_t)(r * GZ_WAVE + gz_lane());
        t.k[r] = i < n ? keys[i] : pad;
    }
    t.before = (base > 0 && base <= n) ? keys[base - 1] : pad;
    t.after = base + GZ_TILE_WAVE < n ? keys[base + GZ_TILE_WAVE] : pad;
    return base;
}

/* The keys ahead of and behind each lane's key of row r. */
__device__ __forceinline__ uint64_t gz_tile_prev(const gz_tile_keys& t, int r)
{
    const uint64_t x = (uint64_t)__shfl_up((unsigned long long)t.k[r], 1, GZ_WAVE);
    const uint64_t edge = r == 0 ? t.before : gz_shfl_u64(t.k[r > 0 ? r - 1 : 0], GZ_WAVE - 1);
    return gz_lane() == 0 ? edge : x;
}

__device__ __forceinline__ uint64_t gz_tile_next(const gz_tile_keys& t, int r)
{
    const uint64_t x = (uint64_t)__shfl_down((unsigned long long)t.k[r], 1, GZ_WAVE);
    const uint64_t edge = r == GZ_TILE_ROWS - 1 ? t.after : gz_shfl_u64(t.k[r < GZ_TILE_ROWS - 1 ? r + 1 : r], 0);
    return gz_lane() == GZ_WAVE - 1 ? edge : x;
}

/* Whether row r's keys count: kept (not all ones, not a duplicate), or, for
 * kHeads, the first of their (key >> b). */
template <bool kHeads>
__device__ __forceinline__ bool gz_tile_flag(const gz_tile_keys& t, int r, uint64_t i, uint64_t n, uint32_t b,
                                             uint64_t none)
{
    const uint64_t k = t.k[r], p = gz_tile_prev(t, r);
    if (kHeads) return i < n && (i == 0 || (k >> b) != (p >> b));
    return i < n && k != none && (i == 0 || k != p);
}

/* sums[tile] = keys of the tile that count. */
template <bool kHeads>
__global__ __launch_bounds__(GZ_BLOCK) void gz_k_tile_count(const uint64_t* __restrict__ keys, uint64_t n, uint32_t b,
                                                            uint64_t none, uint64_t tiles, uint64_t* __restrict__ sums)
{
    __shared__ uint32_t lds[GZ_WAVES_PER_BLOCK];
    for (uint64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        gz_tile_keys t;
        const uint64_t base = gz_tile_load(t, keys, n, tile, none);
        uint32_t c = 0;
#pragma unroll
        for (int r = 0; r < GZ_TILE_ROWS; ++r)
            c += (uint32_t)__popcll(
                __ballot(gz_tile_flag<kHeads>(t, r, base + (uint64_t)(r * GZ_WAVE + gz_lane()), n, b, none)));
        if (gz_lane() == 0) lds[threadIdx.x / GZ_WAVE] = c;
        __syncthreads();
        if (threadIdx.x == 0) {
            uint64_t x = 0;
            for (int w = 0; w < GZ_WAVES_PER_BLOCK; ++w) x += lds[w];
            sums[tile] = x;
        }
        __syncthreads();
    }
}

/* Counting keys of the tile ahead of this wavefront's rows, given its own
 * count (every thread of the workgroup calls it). */
__device__ __forceinline__ uint64_t gz_tile_wave_base(uint32_t mine, uint32_t* lds)
{
    if (gz_lane() == 0) lds[threadIdx.x / GZ_WAVE] = mine;
    __syncthreads();
    uint64_t x = 0;
    for (int w = 0; w < (int)(threadIdx.x / GZ_WAVE); ++w) x += lds[w];
    __syncthreads();
    return x;
}

/* Pass 2 of the dedupe: the kept keys to out, in order, and each group's
 * first and end positions there (groups without kept keys keep their zeros).
 * Equal keys are adjacent and self-loops are all ones, so a group's first raw
 * key is kept and its last raw key ends it.  Bound by memory: 8 bytes read
 * and 8 written per key (the flag array and the library's select it replaced
 * moved 18 and took 2.2 ms for the 67 M keys of R-MAT s22; this and its count
 * pass take 0.4). */
__global__ __launch_bounds__(GZ_BLOCK) void gz_k_kept_write(const uint64_t* __restrict__ keys, uint64_t n, uint32_t b,
                                                            uint64_t none, uint64_t tiles,
                                                            const uint64_t* __restrict__ tile_base,
                                                            uint64_t* __restrict__ out, uint64_t* __restrict__ first,
                                                            uint64_t* __restrict__ end)
{
    __shared__ uint32_t lds[GZ_WAVES_PER_BLOCK];
    const uint64_t below = (1ull << gz_lane()) - 1ull;
    for (uint64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        gz_tile_keys t;
        const uint64_t base = gz_tile_load(t, keys, n, tile, none);
        uint64_t kept[GZ_TILE_ROWS];
        uint32_t c = 0;
#pragma unroll
        for (int r = 0; r < GZ_TILE_ROWS; ++r) {
            kept[r] = __ballot(gz_tile_flag<false>(t, r, base + (uint64_t)(r * GZ_WAVE + gz_lane()), n, b, none));
            c += (uint32_t)__popcll(kept[r]);
        }
        uint64_t pos = tile_base[tile] + gz_tile_wave_base(c, lds);
#pragma unroll
        for (int r = 0; r < GZ_TILE_ROWS; ++r) {
            const uint64_t k = t.k[r], g = k >> b;
            const uint64_t at = pos + (uint64_t)__popcll(kept[r] & below);
            const bool keep = (kept[r] >> gz_lane()) & 1ull;
            const uint64_t p = gz_tile_prev(t, r), q = gz_tile_next(t, r);
            if (keep) out[at] = k;
            if (k != none) { /* padding reads as `none` */
                const bool head = base + (uint64_t)(r * GZ_WAVE + gz_lane()) == 0 || (p >> b) != g;
                if (head) first[g] = at;
                if (q == none || (q >> b) != g) end[g] = at + (keep ? 1 : 0);
            }
            pos += (uint64_t)__popcll(kept[r]);
        }
    }
}

/* Group bounds of sorted keys without duplicates, the group being the low b
 * bits (groups without keys keep their zeros). */
__global__ void gz_k_low_bounds(const uint64_t* __restrict__ keys, uint64_t m, uint32_t b, uint64_t* __restrict__ first,
                                uint64_t* __restrict__ end)
{
    const uint64_t mask = (1ull << b) - 1ull;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += stride) {
        const uint64_t g = keys[i] & mask;
        if (i == 0 || (keys[i - 1] & mask) != g) first[g] = i;
        if (i == m - 1 || (keys[i + 1] & mask) != g) end[g] = i + 1;
    }
}

/* Vectors of group v, 0 past the last group. */
struct gz_group_vectors {
    const uint64_t* first;
    const uint64_t* end;
    uint64_t nv;
    __device__ uint64_t operator()(uint64_t v) const { return v < nv ? (end[v] - first[v] + 3) / 4 : 0; }
};

__device__ __forceinline__ uint64_t gz_piece(uint64_t g, int l)
{
    const int shift = 15 * l;
    const uint64_t mask = (l == 3) ? 0x7ull : 0x7fffull;
    return ((g >> shift) & mask) << 48;
}

/* The group is the high bits of a key, or the low b bits when `low`. */
__global__ void gz_k_pack(const uint64_t* __restrict__ keys, uint64_t m, uint32_t b, int low,
                          const uint64_t* __restrict__ first, const uint64_t* __restrict__ end,
                          const uint64_t* __restrict__ voff, uint64_t* __restrict__ lanes)
{
    const uint64_t mask = (1ull << b) - 1ull;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += stride) {
        const uint64_t k = keys[i];
        const uint64_t g = low ? k & mask : k >> b, nbr = low ? k >> b : k & mask;
        const uint64_t r = i - first[g];
        const uint64_t j = voff[g] + r / 4;
        const int l = (int)(r & 3);
        lanes[4 * j + l] = GZ_LANE_VALID_BIT | gz_piece(g, l) | nbr;
        if (l == 0) {
            const uint64_t left = end[g] - i;
            for (int q = (left < 4 ? (int)left : 4); q < 4; ++q) lanes[4 * j + q] = gz_piece(g, q);
        }
    }
}

__global__ void gz_k_outdegrees(const uint64_t* __restrict__ first, const uint64_t* __restrict__ end, uint64_t nv,
                                double* __restrict__ outdeg)
{
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v < nv + 8; v += stride)
        outdeg[v] = (v < nv) ? (double)(end[v] - first[v]) : 0.0;
}

unsigned gz_grid_for(uint64_t n)
{
    const uint64_t blocks = (n + GZ_BLOCK - 1) / GZ_BLOCK;
    return (unsigned)(blocks < 65536 ? (blocks ? blocks : 1) : 65536);
}

/* Slice size actually used: at most V / (8 T), so the windows fit, and at
 * most 2^23, so that packed window offsets fit in 23 bits. */
uint64_t gz_slices_effective(uint64_t slice_vertices, uint32_t tiers, uint64_t nv)
{
    uint64_t cap = nv / ((uint64_t)GZ_XCDS * tiers);
    if (cap > (1ull << 23)) cap = 1ull << 23;
    return slice_vertices < cap ? slice_vertices : cap;
}

uint32_t gz_id_bits(uint64_t nv)
{
    uint32_t b = 1;
    while (b < 64 && (nv - 1) >> b) ++b;
    return b;
}

unsigned gz_tile_grid(uint64_t tiles) { return (unsigned)(tiles < 65536 ? tiles : 65536); }

/* Sort keys[0, n) over bits [begin, end), stably; the sorted keys end in
 * *sorted (one of a or b_buf). */
void gz_sort_keys(uint64_t* a, uint64_t* b_buf, uint64_t n, uint32_t begin, uint32_t end, uint64_t** sorted)
{
    rocprim::double_buffer<uint64_t> db(a, b_buf);
    size_t tmp_bytes = 0;
    GZ_CHECK(rocprim::radix_sort_keys(nullptr, tmp_bytes, db, (size_t)n, begin, end, gz_stream));
    void* tmp = gz_pool_malloc(tmp_bytes ? tmp_bytes : 1, 0);
    GZ_CHECK(rocprim::radix_sort_keys(tmp, tmp_bytes, db, (size_t)n, begin, end, gz_stream));
    gz_pool_free(tmp);
    *sorted = db.current();
}

/* out[0 .. n) = exclusive scan of in[0 .. n). */
template <typename It>
void gz_scan(It in, uint64_t* out, uint64_t n)
{
    size_t tmp_bytes = 0;
    GZ_CHECK(rocprim::exclusive_scan(nullptr, tmp_bytes, in, out, (uint64_t)0, (size_t)n, rocprim::plus<uint64_t>(),
                                     gz_stream));
    void* tmp = gz_pool_malloc(tmp_bytes ? tmp_bytes : 1, 0);
    GZ_CHECK(rocprim::exclusive_scan(tmp, tmp_bytes, in, out, (uint64_t)0, (size_t)n, rocprim::plus<uint64_t>(),
                                     gz_stream));
    gz_pool_free(tmp);
}

/* Build one layout from sorted, duplicate-free keys[0, m) and the bounds of
 * their groups (the low key bits when `low`). */
void gz_build_layout(const uint64_t* keys, uint64_t m, uint32_t b, int low, uint64_t nv, const uint64_t* first,
                     const uint64_t* end, gz_vec_t** d_vecs, uint64_t** d_offsets, uint64_t* vector_count)
{
    uint64_t* voff = (uint64_t*)gz_pool_malloc((nv + 1) * sizeof(uint64_t), 0);
    gz_scan(rocprim::make_transform_iterator(rocprim::make_counting_iterator<uint64_t>(0),
                                             gz_group_vectors{first, end, nv}),
            voff, nv + 1);
    uint64_t total = 0;
    gz_copy_to_host(&total, voff + nv, sizeof(uint64_t));
    gz_vec_t* vecs = (gz_vec_t*)gz_pool_malloc((total ? total : 1) * sizeof(gz_vec_t), 0);
    if (m) {
        hipLaunchKernelGGL(gz_k_pack, dim3(gz_grid_for(m)), dim3(GZ_BLOCK), 0, gz_stream, keys, m, b, low, first, end,
                           voff, (uint64_t*)vecs);
        GZ_LAUNCH_CHECK();
    }
    *d_vecs = vecs;
    *d_offsets = voff;
    *vector_count = total;
}

__global__ void gz_k_count_sources(const uint64_t* __restrict__ keys, uint64_t n, uint32_t b, uint32_t* __restrict__ cnt)
{
    const uint64_t mask = (1ull << b) - 1ull;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
        atomicAdd(&cnt[keys[i] & mask], 1u);
}

/* Fewest keys, and most id bits, of the bucketed count below.  A renumbering
 * load of R-MAT with edge factor 16, atomics / buckets: 2^18 keys 1022 / 1011
 * us, 2^20 1426 / 1210, 2^21 2122 / 1716, 2^24 12.2 / 10.2 ms; each id bit
 * above 24 doubles the times a bucket's ids are read back. */
#define GZ_COUNT_BUCKET_KEYS (1ull << 19)
#define GZ_COUNT_BUCKET_BITS 28

/* ---- counting sources by buckets -------------------------------------------
 * One atomic per key on a count per vertex runs at 7 G keys/s here (67 M keys
 * of R-MAT s22: 9.24 ms): atomics from different XCDs on one line take turns.
 * Instead the sources are partitioned by their high bits into at most 1024
 * buckets, staged through LDS so that a bucket's ids leave in runs, and each
 * bucket is then counted in LDS, 2^14 ids at a time.  Memory-bound: 8 bytes
 * per key read twice, 4 written, 4 read back per 2^14 ids of a bucket: 0.58 ms
 * for those 67 M keys (sizes 0.14, scatter 0.31, count 0.13), and 16.1 ms in
 * place of 128.8 for 1.49 G keys over 41.7 M ids. */
#define GZ_COUNT_BUCKETS 1024
#define GZ_COUNT_IDS_LOG2 14
#define GZ_COUNT_THREADS 1024
#define GZ_COUNT_TILE 16384                      /* keys a workgroup partitions at a time */
#define GZ_COUNT_SEGMENT 131072                  /* partitioned ids a workgroup counts */
#define GZ_COUNT_PAD 64                          /* words between bucket cursors: a line of their own each */

__global__ __launch_bounds__(GZ_COUNT_THREADS) void gz_k_bucket_sizes(const uint64_t* __restrict__ keys, uint64_t n,
                                                                      uint64_t mask, uint32_t shift,
                                                                      uint32_t buckets,
                                                                      unsigned long long* __restrict__ sizes)
{
    __shared__ uint32_t hist[GZ_COUNT_BUCKETS];
    hist[threadIdx.x] = 0;
    __syncthreads();
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
        atomicAdd(&hist[(keys[i] & mask) >> shift], 1u);
    __syncthreads();
    if (threadIdx.x < buckets && hist[threadIdx.x])
        atomicAdd(&sizes[(uint64_t)threadIdx.x * GZ_COUNT_PAD], (unsigned long long)hist[threadIdx.x]);
}

/* One workgroup: base[k] = ids of the buckets before k (base[buckets] = n),
 * and the cursors, which held the sizes, start there. */
__global__ __launch_bounds__(GZ_COUNT_THREADS) void gz_k_bucket_bases(unsigned long long* __restrict__ cursors,
                                                                      uint32_t buckets, uint64_t* __restrict__ base)
{
    __shared__ uint64_t waves[GZ_COUNT_THREADS / GZ_WAVE];
    const uint32_t k = threadIdx.x;
    const uint64_t size = k < buckets ? (uint64_t)cursors[(uint64_t)k * GZ_COUNT_PAD] : 0;
    uint64_t incl = size;
#pragma unroll
    for (int o = 1; o < GZ_WAVE; o <<= 1) {
        const uint64_t t = (uint64_t)__shfl_up((unsigned long long)incl, o, GZ_WAVE);
        if (gz_lane() >= o) incl += t;
    }
    if (gz_lane() == GZ_WAVE - 1) waves[k / GZ_WAVE] = incl;
    __syncthreads();
    for (uint32_t w = 0; w < k / GZ_WAVE; ++w) incl += waves[w];
    if (k < buckets) {
        base[k] = incl - size;
        cursors[(uint64_t)k * GZ_COUNT_PAD] = incl - size;
        if (k == buckets - 1) base[buckets] = incl;
    }
}

__global__ __launch_bounds__(GZ_COUNT_THREADS) void gz_k_bucket_scatter(const uint64_t* __restrict__ keys, uint64_t n,
                                                                        uint64_t mask, uint32_t shift,
                                                                        uint64_t tiles,
                                                                        unsigned long long* __restrict__ cursors,
                                                                        uint32_t* __restrict__ ids)
{
    constexpr int kPer = GZ_COUNT_TILE / GZ_COUNT_THREADS;
    __shared__ uint32_t stage[GZ_COUNT_TILE];  /* ids in bucket order */
    __shared__ uint16_t owner[GZ_COUNT_TILE];  /* their buckets */
    __shared__ uint32_t hist[GZ_COUNT_BUCKETS], start[GZ_COUNT_BUCKETS];
    __shared__ uint64_t out[GZ_COUNT_BUCKETS]; /* where the bucket's first staged id goes */
    __shared__ uint32_t waves[GZ_COUNT_THREADS / GZ_WAVE];
    const uint32_t t = threadIdx.x, low = (1u << shift) - 1u;
    for (uint64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const uint64_t first = tile * GZ_COUNT_TILE;
        const uint32_t count = (uint32_t)(n - first < GZ_COUNT_TILE ? n - first : GZ_COUNT_TILE);
        hist[t] = 0;
        __syncthreads();
        uint32_t id[kPer], rank[kPer];
#pragma unroll
        for (int r = 0; r < kPer; ++r) {
            const uint32_t i = (uint32_t)r * GZ_COUNT_THREADS + t;
            id[r] = i < count ? (uint32_t)(keys[first + i] & mask) : 0u;
        }
#pragma unroll
        for (int r = 0; r < kPer; ++r)
            rank[r] = (uint32_t)r * GZ_COUNT_THREADS + t < count ? atomicAdd(&hist[id[r] >> shift], 1u) : 0u;
        __syncthreads();
        const uint32_t size = hist[t];
        uint32_t incl = size;
#pragma unroll
        for (int o = 1; o < GZ_WAVE; o <<= 1) {
            const uint32_t x = __shfl_up(incl, o, GZ_WAVE);
            if (gz_lane() >= o) incl += x;
        }
        if (gz_lane() == GZ_WAVE - 1) waves[t / GZ_WAVE] = incl;
        __syncthreads();
        for (uint32_t w = 0; w < t / GZ_WAVE; ++w) incl += waves[w];
        start[t] = incl - size;
        if (size) out[t] = atomicAdd(&cursors[(uint64_t)t * GZ_COUNT_PAD], (unsigned long long)size);
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kPer; ++r) {
            if ((uint32_t)r * GZ_COUNT_THREADS + t >= count) continue;
            const uint32_t k = id[r] >> shift, at = start[k] + rank[r];
            stage[at] = id[r] & low;
            owner[at] = (uint16_t)k;
        }
        __syncthreads();
        for (uint32_t i = t; i < count; i += GZ_COUNT_THREADS) {
            const uint32_t k = owner[i];
            ids[out[k] + (i - start[k])] = stage[i];
        }
        __syncthreads();
    }
}

/* cnt[v] += the ids of v among a segment of the partitioned ids, bucket by
 * bucket (a segment holds a part of a large bucket or several small ones). */
__global__ __launch_bounds__(GZ_COUNT_THREADS) void gz_k_bucket_count(const uint32_t* __restrict__ ids, uint64_t n,
                                                                      uint32_t shift, uint32_t buckets,
                                                                      const uint64_t* __restrict__ base, uint64_t nv,
                                                                      uint32_t* __restrict__ cnt)
{
    __shared__ uint32_t hist[1 << GZ_COUNT_IDS_LOG2];
    const uint64_t lo = (uint64_t)blockIdx.x * GZ_COUNT_SEGMENT;
    const uint64_t hi = lo + GZ_COUNT_SEGMENT < n ? lo + GZ_COUNT_SEGMENT : n;
    uint32_t k = 0; /* the last bucket that starts at or before lo */
    for (uint32_t z = buckets; z - k > 1;) {
        const uint32_t mid = (k + z) / 2;
        if (base[mid] <= lo)
            k = mid;
        else
            z = mid;
    }
    for (; k < buckets && base[k] < hi; ++k) {
        const uint64_t b = base[k] > lo ? base[k] : lo, e = base[k + 1] < hi ? base[k + 1] : hi;
        if (b >= e) continue;
        for (uint32_t part = 0; part < 1u << (shift - GZ_COUNT_IDS_LOG2); ++part) {
            const uint64_t v0 = ((uint64_t)k << shift) + ((uint64_t)part << GZ_COUNT_IDS_LOG2);
            if (v0 >= nv) break;
            for (uint32_t i = threadIdx.x; i < 1u << GZ_COUNT_IDS_LOG2; i += GZ_COUNT_THREADS) hist[i] = 0;
            __syncthreads();
            for (uint64_t i = b + threadIdx.x; i < e; i += GZ_COUNT_THREADS) {
                const uint32_t id = ids[i];
                if (id >> GZ_COUNT_IDS_LOG2 == part) atomicAdd(&hist[id & ((1u << GZ_COUNT_IDS_LOG2) - 1u)], 1u);
            }
            __syncthreads();
            for (uint32_t i = threadIdx.x; i < 1u << GZ_COUNT_IDS_LOG2; i += GZ_COUNT_THREADS)
                if (hist[i]) atomicAdd(&cnt[v0 + i], hist[i]); /* an id counted is below nv */
            __syncthreads();
        }
    }
}

/* cnt[s] = keys whose source is s, cnt cleared beforehand; `ids` holds n words
 * of scratch. */
void gz_count_sources(const uint64_t* keys, uint64_t n, uint32_t b, uint64_t nv, uint32_t* ids, uint32_t* cnt)
{
    if (n == 0) return;
    if (n < GZ_COUNT_BUCKET_KEYS || b > GZ_COUNT_BUCKET_BITS) {
        hipLaunchKernelGGL(gz_k_count_sources, dim3(gz_grid_for(n)), dim3(GZ_BLOCK), 0, gz_stream, keys, n, b, cnt);
        GZ_LAUNCH_CHECK();
        return;
    }
    const uint32_t shift = b > GZ_COUNT_IDS_LOG2 + 10 ? b - 10 : GZ_COUNT_IDS_LOG2;
    const uint32_t buckets = (uint32_t)((nv - 1) >> shift) + 1;
    const uint64_t mask = (1ull << b) - 1ull;
    const uint64_t tiles = (n + GZ_COUNT_TILE - 1) / GZ_COUNT_TILE;
    const uint64_t segments = (n + GZ_COUNT_SEGMENT - 1) / GZ_COUNT_SEGMENT;
    const size_t cursor_words = (size_t)buckets * GZ_COUNT_PAD;
    unsigned long long* cursors =
        (unsigned long long*)gz_pool_malloc((cursor_words + buckets + 1) * sizeof(uint64_t), 1); /* zero-filled */
    uint64_t* base = (uint64_t*)cursors + cursor_words;
    hipLaunchKernelGGL(gz_k_bucket_sizes, dim3((unsigned)(tiles < 1024 ? tiles : 1024)), dim3(GZ_COUNT_THREADS), 0,
                       gz_stream, keys, n, mask, shift, buckets, cursors);
    GZ_LAUNCH_CHECK();
    hipLaunchKernelGGL(gz_k_bucket_bases, dim3(1), dim3(GZ_COUNT_THREADS), 0, gz_stream, cursors, buckets, base);
    GZ_LAUNCH_CHECK();
    hipLaunchKernelGGL(gz_k_bucket_scatter, dim3((unsigned)(tiles < 4096 ? tiles : 4096)), dim3(GZ_COUNT_THREADS), 0,
                       gz_stream, keys, n, mask, shift, tiles, cursors, ids);
    GZ_LAUNCH_CHECK();
    hipLaunchKernelGGL(gz_k_bucket_count, dim3((unsigned)segments), dim3(GZ_COUNT_THREADS), 0, gz_stream, ids, n, shift,
                       buckets, base, nv, cnt);
    GZ_LAUNCH_CHECK();
    gz_pool_free(cursors);
}

/* sort key: out-degree descending (as `most` less the degree), then id ascending */
__global__ void gz_k_degree_order(const uint32_t* __restrict__ cnt, uint64_t nv, uint32_t b, uint64_t most,
                                  uint64_t* __restrict__ order)
{
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v < nv; v += stride)
        order[v] = ((most - cnt[v]) << b) | v;
}

/* Rank i of the degree order becomes id i, except that each of the first
 * `tiers` runs of 8*S ranks is dealt round robin into eight S-id windows:
 * rank t*8S + q -> t*8S + (q % 8) * S + q / 8. */
__global__ void gz_k_permutation(const uint64_t* __restrict__ order, uint64_t nv, uint32_t b,
                                 uint64_t slice_vertices, uint32_t tiers, uint64_t* __restrict__ old_of_new, uint32_t* __restrict__ new_of_old)
{
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    const uint64_t tier = (uint64_t)GZ_XCDS * slice_vertices;
    const uint64_t hot = tier * tiers;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nv; i += stride) {
        const uint64_t old = order[i] & ((1ull << b) - 1ull);
        uint64_t id = i;
        if (i < hot) {
            const uint64_t t = i / tier, q = i - t * tier;
            id = t * tier + (q % GZ_XCDS) * slice_vertices + q / GZ_XCDS;
        }
        old_of_new[id] = old;
        new_of_old[old] = (uint32_t)id;
    }
}

__global__ void gz_k_remap_keys(uint64_t* __restrict__ keys, uint64_t n, uint32_t b,
                                const uint32_t* __restrict__ new_of_old)
{
    const uint64_t mask = (1ull << b) - 1ull;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        const uint64_t k = keys[i];
        keys[i] = gz_edge_key(new_of_old[k >> b], new_of_old[k & mask], b, 1);
    }
}

/* Renumber the vertices by raw out-degree, descending (ties by id), and
 * rewrite the keys in place (`scratch`: n words).  Returns the device array of
 * original ids, indexed by new id, and its inverse in *device_ids.  The hot
 * sources of a power-law graph then share cache lines, which is what the pull
 * gathers need once the vertex array no longer fits in the caches. */
uint64_t* gz_relabel_by_outdegree(uint64_t* keys, uint64_t* scratch, uint64_t n, uint32_t b, uint64_t nv,
                                  uint64_t slice_vertices, uint32_t tiers, uint32_t** device_ids)
{
    uint32_t* cnt = (uint32_t*)gz_pool_malloc(nv * sizeof(uint32_t), 1);
    gz_count_sources(keys, n, b, nv, (uint32_t*)scratch, cnt);
    const uint64_t most = n < 0xffffffffull ? n : 0xffffffffull; /* counts are 32-bit */
    uint64_t* order = (uint64_t*)gz_pool_malloc(nv * sizeof(uint64_t), 0);
    uint64_t* order_b = (uint64_t*)gz_pool_malloc(nv * sizeof(uint64_t), 0);
    hipLaunchKernelGGL(gz_k_degree_order, dim3(gz_grid_for(nv)), dim3(GZ_BLOCK), 0, gz_stream, cnt, nv, b,
                       most, order);
    GZ_LAUNCH_CHECK();
    uint64_t* sorted = order;
    if (nv > 1) gz_sort_keys(order, order_b, nv, 0, b + gz_id_bits(most + 1), &sorted);
    uint64_t* old_of_new = (uint64_t*)gz_pool_malloc((nv + 8) * sizeof(uint64_t), 0);
    uint32_t* new_of_old = cnt; /* counts are no longer needed */
    hipLaunchKernelGGL(gz_k_permutation, dim3(gz_grid_for(nv)), dim3(GZ_BLOCK), 0, gz_stream, sorted, nv, b,
                       slice_vertices, tiers, old_of_new, new_of_old);
    GZ_LAUNCH_CHECK();
    if (n) {
        hipLaunchKernelGGL(gz_k_remap_keys, dim3(gz_grid_for(n)), dim3(GZ_BLOCK), 0, gz_stream, keys, n, b, new_of_old);
        GZ_LAUNCH_CHECK();
    }
    gz_pool_free(order);
    gz_pool_free(order_b);
    *device_ids = new_of_old;
    return old_of_new;
}

/* Keys already in a[0, n): optionally renumber, sort, drop self-loops and
 * duplicates, build both layouts and hand them to the graph record. */
void gz_ingress_from_keys(uint64_t nv, uint64_t* a, uint64_t* b_buf, uint64_t n, uint32_t b, uint32_t flags)
{
    const uint32_t slice_log2 = (flags >> 8) & 0x3fu;
    uint32_t tiers = (flags >> 14) & 0x3u;
    if (tiers == 0) tiers = 1;
    const uint32_t blocks = (flags >> 16) & 0x7u;
    const uint64_t slice_vertices = slice_log2 ? gz_slices_effective(1ull << slice_log2, tiers, nv) : 0;
    uint64_t* old_of_new = nullptr;
    uint32_t* new_of_old = nullptr;
    if (flags & GZ_INGRESS_RELABEL_BY_OUTDEGREE)
        old_of_new = gz_relabel_by_outdegree(a, b_buf, n, b, nv, slice_vertices, tiers, &new_of_old);
    uint64_t* sorted = a;
    if (n > 1) gz_sort_keys(a, b_buf, n, 0, 2 * b, &sorted);
    uint64_t* other = (sorted == a) ? b_buf : a;
    uint64_t m = 0;
    uint64_t* first = (uint64_t*)gz_pool_malloc(nv * sizeof(uint64_t), 1);
    uint64_t* end = (uint64_t*)gz_pool_malloc(nv * sizeof(uint64_t), 1);
    if (n) {
        const uint64_t none = gz_no_key(b);
        const uint64_t tiles = (n + GZ_TILE - 1) / GZ_TILE;
        uint64_t* sums = (uint64_t*)gz_pool_malloc(2 * (tiles + 1) * sizeof(uint64_t), 1); /* sums[tiles] stays 0 */
        uint64_t* base = sums + tiles + 1;
        hipLaunchKernelGGL(gz_k_tile_count<false>, dim3(gz_tile_grid(tiles)), dim3(GZ_BLOCK), 0, gz_stream, sorted, n,
                           b, none, tiles, sums);
        GZ_LAUNCH_CHECK();
        gz_scan(sums, base, tiles + 1);
        hipLaunchKernelGGL(gz_k_kept_write, dim3(gz_tile_grid(tiles)), dim3(GZ_BLOCK), 0, gz_stream, sorted, n, b,
                           none, tiles, base, other, first, end);
        GZ_LAUNCH_CHECK();
        gz_copy_to_host(&m, base + tiles, sizeof(uint64_t));
        gz_pool_free(sums);
    }

    gz_device_layouts_t L;
    L.num_vertices = nv;
    L.num_edges = m;
    L.original_ids = old_of_new;
    L.device_ids = new_of_old;
    gz_build_layout(other, m, b, 0, nv, first, end, &L.pull, &L.pull_offsets, &L.pull_count);
    /* push layout: the kept keys by source (still unique) */
    uint64_t* push_sorted = other;
    if (m > 1) gz_sort_keys(other, sorted, m, 0, b, &push_sorted);
    gz_device_zero(first, nv * sizeof(uint64_t));
    gz_device_zero(end, nv * sizeof(uint64_t));
    if (m) {
        hipLaunchKernelGGL(gz_k_low_bounds, dim3(gz_grid_for(m)), dim3(GZ_BLOCK), 0, gz_stream, push_sorted, m, b, first,
                           end);
        GZ_LAUNCH_CHECK();
    }
    gz_build_layout(push_sorted, m, b, 1, nv, first, end, &L.push, &L.push_offsets, &L.push_count);
    L.outdeg = (double*)gz_pool_malloc((nv + 8) * sizeof(double), 0);
    hipLaunchKernelGGL(gz_k_outdegrees, dim3(gz_grid_for(nv + 8)), dim3(GZ_BLOCK), 0, gz_stream, first, end, nv,
                       L.outdeg);
    GZ_LAUNCH_CHECK();
    gz_pool_free(first);
    gz_pool_free(end);
    gz_graph_adopt_device(&L);
    if (slice_log2) gz_graph_build_source_slices(1ull << slice_log2, tiers, blocks, GZ_SLICE_BLOCK_VERTICES);
    gz_synchronize();
}

/* Whether the key kernels drop self-loops (a renumbering counts them first). */
int gz_drop_first(uint32_t flags) { return (flags & GZ_INGRESS_RELABEL_BY_OUTDEGREE) ? 0 : 1; }

void gz_check_vertex_count(uint64_t nv)
{
    if (nv == 0 || nv > 0xffffffffull) {
        fprintf(stderr, "grazelle: device ingress needs 1 <= V <= 2^32 (got %llu)\n", (unsigned long long)nv);
        exit(65);
    }
}

}  // namespace

/* Upload n host pairs and append their keys; dies with `what` and the first
 * endpoint that is not below nv.  The check rides on the key kernel's reads: a
 * host loop over the endpoints cost more than the upload (a load of 3 M pairs,
 * CC and its labels: 4.00 ms with the loop, 2.59 without). */
static void gz_upload_keys(const uint64_t* pairs, uint64_t n, uint32_t b, int both, int drop, uint64_t nv,
                           uint64_t* keys, const char* what)
{
    if (n == 0) return;
    uint64_t* d = (uint64_t*)gz_pool_malloc((2 * n + 2) * sizeof(uint64_t), 0);
    unsigned long long* bad = (unsigned long long*)(d + 2 * n);
    gz_dev_fill_u64((uint64_t*)bad, ~0ull, 1);
    gz_copy_to_device(d, pairs, 2 * n * sizeof(uint64_t));
    hipLaunchKernelGGL(gz_k_pairs_keys, dim3(gz_grid_for(n)), dim3(GZ_BLOCK), 0, gz_stream, (const gz_u64x2*)d, n, b,
                       both, drop, nv, keys, bad);
    GZ_LAUNCH_CHECK();
    uint64_t at = 0;
    gz_copy_to_host(&at, bad, sizeof(at));
    gz_pool_free(d);
    if (at != ~0ull) {
        fprintf(stderr, "grazelle: %s %llu is not below V = %llu\n", what, (unsigned long long)pairs[at],
                (unsigned long long)nv);
        exit(65);
    }
}

extern "C" int gz_graph_build_pairs_device(uint64_t num_vertices, uint64_t num_edges, const uint64_t* pairs,
                                           int symmetrize, uint32_t flags)
{
    gz_runtime_init(0);
    gz_graph_drop();
    gz_check_vertex_count(num_vertices);
    const uint32_t b = gz_id_bits(num_vertices);
    const uint64_t n = symmetrize ? 2 * num_edges : num_edges;
    uint64_t* a = (uint64_t*)gz_pool_malloc((n ? n : 1) * sizeof(uint64_t), 0);
    uint64_t* bb = (uint64_t*)gz_pool_malloc((n ? n : 1) * sizeof(uint64_t), 0);
    gz_upload_keys(pairs, num_edges, b, symmetrize, gz_drop_first(flags), num_vertices, a, "edge endpoint");
    gz_ingress_from_keys(num_vertices, a, bb, n, b, flags);
    gz_pool_free(a);
    gz_pool_free(bb);
    return 0;
}

extern "C" int gz_graph_build_rmat_device(const gz_rmat_params_t* p, uint64_t num_vertices, int symmetrize,
                                          uint64_t extra_edges, const uint64_t* extra_pairs, uint32_t flags)
{
    gz_runtime_init(0);
    gz_graph_drop();
    const uint64_t rmat_nv = p->num_vertices ? p->num_vertices : (1ull << p->scale);
    uint64_t nv = num_vertices > rmat_nv ? num_vertices : rmat_nv;
    gz_check_vertex_count(nv);
    const uint32_t b = gz_id_bits(nv);
    const uint64_t per = symmetrize ? 2 : 1;
    const uint64_t n = per * (p->num_edges + extra_edges);
    uint64_t* a = (uint64_t*)gz_pool_malloc((n ? n : 1) * sizeof(uint64_t), 0);
    uint64_t* bb = (uint64_t*)gz_pool_malloc((n ? n : 1) * sizeof(uint64_t), 0);
    if (p->num_edges) {
        const uint32_t ta = (uint32_t)(p->a * 65536.0);
        const uint32_t tb = (uint32_t)((p->a + p->b) * 65536.0);
        const uint32_t tc = (uint32_t)((p->a + p->b + p->c) * 65536.0);
        hipLaunchKernelGGL(gz_k_rmat_keys, dim3(gz_grid_for(p->num_edges)), dim3(GZ_BLOCK), 0, gz_stream, p->seed,
                           p->edge_offset, p->scale, rmat_nv, ta, tb, tc, p->num_edges, b, symmetrize, gz_drop_first(flags),
                           (uint64_t)0, a);
        GZ_LAUNCH_CHECK();
    }
    gz_upload_keys(extra_pairs, extra_edges, b, symmetrize, gz_drop_first(flags), nv, a + per * p->num_edges,
                   "extra edge endpoint");
    gz_ingress_from_keys(nv, a, bb, n, b, flags);
    gz_pool_free(a);
    gz_pool_free(bb);
    return 0;
}

extern "C" int gz_graph_build_rmat_union_device(const gz_rmat_params_t* params, uint32_t count, int symmetrize,
                                                uint64_t* vertex_bases)
{
    gz_runtime_init(0);
    gz_graph_drop();
    uint64_t nv = 0, n = 0;
    const uint64_t per = symmetrize ? 2 : 1;
    for (uint32_t g = 0; g < count; ++g) {
        vertex_bases[g] = nv;
        nv += params[g].num_vertices ? params[g].num_vertices : (1ull << params[g].scale);
        n += per * params[g].num_edges;
    }
    vertex_bases[count] = nv;
    gz_check_vertex_count(nv);
    const uint32_t b = gz_id_bits(nv);
    uint64_t* a = (uint64_t*)gz_pool_malloc((n ? n : 1) * sizeof(uint64_t), 0);
    uint64_t* bb = (uint64_t*)gz_pool_malloc((n ? n : 1) * sizeof(uint64_t), 0);
    uint64_t at = 0;
    for (uint32_t g = 0; g < count; ++g) {
        const gz_rmat_params_t* p = &params[g];
        if (p->num_edges == 0) continue;
        const uint32_t ta = (uint32_t)(p->a * 65536.0);
        const uint32_t tb = (uint32_t)((p->a + p->b) * 65536.0);
        const uint32_t tc = (uint32_t)((p->a + p->b + p->c) * 65536.0);
        const uint64_t gnv = vertex_bases[g + 1] - vertex_bases[g];
        hipLaunchKernelGGL(gz_k_rmat_keys, dim3(gz_grid_for(p->num_edges)), dim3(GZ_BLOCK), 0, gz_stream, p->seed,
                           p->edge_offset, p->scale, gnv, ta, tb, tc, p->num_edges, b, symmetrize, 1, vertex_bases[g],
                           a + at);
        GZ_LAUNCH_CHECK();
        at += per * p->num_edges;
    }
    gz_ingress_from_keys(nv, a, bb, n, b, 0);
    gz_pool_free(a);
    gz_pool_free(bb);
    return 0;
}

/* ---- source-sliced pull layout ---------------------------------------------
 * From the loaded pull vectors: every valid lane becomes the key
 * (slice << 2b | dst << b | src) (invalid lanes all ones), and a stable radix
 * pass over the 7 slice bits groups the keys by slice while keeping the
 * (dst, src) order.  A run is the keys of one (slice, dst) pair: numbered in
 * key order, run r is the slice accumulator r, and its number less its slice's
 * first one is the destination's local rank.  All slices are then built
 * together, in a number of launches that does not grow with theirs:
 *   runs    each run's first key and destination (tile counts, then a write)
 *   vectors the exclusive scan of the runs' ceil(length / 4)
 *   pack    each vector's packed neighbours and local rank, in place
 *   mask    per 64-vertex block, the slice bits of its vertices and the
 *           number of its first run in each slice */
namespace {

__global__ void gz_k_slice_keys(const gz_vec_t* __restrict__ vecs, uint64_t nvec, uint32_t b, uint64_t slice_vertices,
                                uint32_t tiers, uint32_t blocks, uint64_t block_vertices, uint64_t* __restrict__ keys)
{
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < 4 * nvec; i += stride) {
        const gz_vec_t* v = vecs + i / 4;
        const uint64_t l = v->lane[i % 4];
        if (!gz_lane_valid(l)) {
            keys[i] = ~0ull;
            continue;
        }
        gz_lanes w;
        w.l0 = v->lane[0];
        w.l1 = v->lane[1];
        w.l2 = v->lane[2];
        w.l3 = v->lane[3];
        const uint64_t d = gz_shared_vertex(w);
        const uint64_t s = gz_lane_id(l);
        const uint64_t x = gz_slice_of_source(s, slice_vertices, tiers, blocks, block_vertices);
        keys[i] = (x << (2 * b)) | (d << b) | s;
    }
}

/* first[x] = first key whose slice field is >= x, x in [0, nslices] */
__global__ void gz_k_slice_bounds(const uint64_t* __restrict__ keys, uint64_t n, uint32_t b, uint32_t nslices,
                                  uint64_t* __restrict__ first)
{
    const uint64_t x = threadIdx.x;
    if (x > nslices) return;
    uint64_t lo = 0, hi = n;
    while (lo < hi) {
        const uint64_t mid = lo + ((hi - lo) >> 1);
        if ((keys[mid] >> (2 * b)) < x)
            lo = mid + 1;
        else
            hi = mid;
    }
    first[x] = lo;
}

/* Run r's first key (run_first[r], with run_first[runs] = n) and its
 * destination; the runs ahead of each tile come from the tile counts. */
__global__ __launch_bounds__(GZ_BLOCK) void gz_k_slice_runs(const uint64_t* __restrict__ keys, uint64_t n, uint32_t b,
                                                            uint64_t tiles, const uint64_t* __restrict__ tile_base,
                                                            uint64_t* __restrict__ run_first, uint32_t* __restrict__ gid)
{
    __shared__ uint32_t lds[GZ_WAVES_PER_BLOCK];
    const uint64_t below = (1ull << gz_lane()) - 1ull, mask = (1ull << b) - 1ull;
    for (uint64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        gz_tile_keys t;
        const uint64_t base = gz_tile_load(t, keys, n, tile, ~0ull);
        uint64_t heads[GZ_TILE_ROWS];
        uint32_t c = 0;
#pragma unroll
        for (int r = 0; r < GZ_TILE_ROWS; ++r) {
            heads[r] = __ballot(gz_tile_flag<true>(t, r, base + (uint64_t)(r * GZ_WAVE + gz_lane()), n, b, ~0ull));
            c += (uint32_t)__popcll(heads[r]);
        }
        uint64_t at = tile_base[tile] + gz_tile_wave_base(c, lds);
#pragma unroll
        for (int r = 0; r < GZ_TILE_ROWS; ++r) {
            if ((heads[r] >> gz_lane()) & 1ull) {
                const uint64_t run = at + (uint64_t)__popcll(heads[r] & below);
                run_first[run] = base + (uint64_t)(r * GZ_WAVE + gz_lane());
                gid[run] = (uint32_t)((t.k[r] >> b) & mask);
            }
            at += (uint64_t)__popcll(heads[r]);
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) run_first[tile_base[tiles]] = n;
}

/* Vectors of run r, 0 past the last run. */
struct gz_run_vectors {
    const uint64_t* run_first;
    uint64_t runs;
    __device__ uint64_t operator()(uint64_t r) const { return r < runs ? (run_first[r + 1] - run_first[r] + 3) / 4 : 0; }
};

/* For slice x in [0, nslices]: its first run (first key lo[x] starts one) and
 * its first vector. */
__global__ void gz_k_slice_firsts(const uint64_t* __restrict__ lo, uint32_t nslices,
                                  const uint64_t* __restrict__ run_first, uint64_t runs,
                                  const uint64_t* __restrict__ run_vec, uint64_t* __restrict__ first_run,
                                  uint64_t* __restrict__ first_vec)
{
    const uint32_t x = threadIdx.x;
    if (x > nslices) return;
    uint64_t a = 0, z = runs;
    while (a < z) {
        const uint64_t mid = a + ((z - a) >> 1);
        if (run_first[mid] < lo[x])
            a = mid + 1;
        else
            z = mid;
    }
    first_run[x] = a;
    first_vec[x] = run_vec[a];
}

struct gz_slice_pack_t {
    uint64_t S, H;
    uint32_t blocks, nslices;
    uint64_t block_first, block_span, cold_first; /* first vector of the block slices, their count, and the cold slice's first */
    const uint64_t* first_run;                    /* [nslices + 1], device */
    uint32_t* nbr24;
    uint64_t* nbr16;
    gz_u32x4* nbr;
    uint32_t* shared;
};

/* The packed vectors (gz_walk.h) of every slice: the lane that holds a
 * vector's first key writes it.  Window slices: 12 bytes, four 24-bit offsets
 * from the window's first vertex (empty lanes all ones), bit 23 of the first
 * set on the first vector of each destination.  Block slices: 8 bytes, four
 * 16-bit offsets from the block's first vertex (GZ_PACKED16_NONE for an empty
 * lane), bit 15 of the first the flag.  The cold slice: 16 bytes, four 32-bit
 * ids (GZ_PACKED_NONE), flag in bit 31.  shared: the local rank. */
__global__ __launch_bounds__(GZ_BLOCK) void gz_k_slice_pack(const uint64_t* __restrict__ keys, uint64_t n, uint32_t b,
                                                            uint64_t tiles, const uint64_t* __restrict__ tile_base,
                                                            const uint64_t* __restrict__ run_first,
                                                            const uint64_t* __restrict__ run_vec, gz_slice_pack_t p)
{
    __shared__ uint32_t lds[GZ_WAVES_PER_BLOCK];
    const uint64_t upto = (2ull << gz_lane()) - 1ull, mask = (1ull << b) - 1ull;
    for (uint64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        gz_tile_keys t;
        const uint64_t base = gz_tile_load(t, keys, n, tile, ~0ull);
        uint64_t heads[GZ_TILE_ROWS];
        uint32_t c = 0;
#pragma unroll
        for (int r = 0; r < GZ_TILE_ROWS; ++r) {
            heads[r] = __ballot(gz_tile_flag<true>(t, r, base + (uint64_t)(r * GZ_WAVE + gz_lane()), n, b, ~0ull));
            c += (uint32_t)__popcll(heads[r]);
        }
        uint64_t at = tile_base[tile] + gz_tile_wave_base(c, lds);
#pragma unroll
        for (int r = 0; r < GZ_TILE_ROWS; ++r) {
            const uint64_t i = base + (uint64_t)(r * GZ_WAVE + gz_lane());
            /* the key's run: heads up to and including it, less one (a key
             * that is no head has one ahead of it) */
            const uint64_t run = at + (uint64_t)__popcll(heads[r] & upto) - 1;
            at += (uint64_t)__popcll(heads[r]);
            if (i >= n) continue;
            const uint64_t rf = run_first[run], rank = i - rf;
            if (rank & 3) continue;
            const uint64_t j = run_vec[run] + rank / 4;
            const uint64_t left = run_first[run + 1] - i;
            const uint64_t k0 = t.k[r];
            const uint32_t x = (uint32_t)(k0 >> (2 * b));
            const uint64_t s0 = k0 & mask;
            const uint64_t s1 = left > 1 ? keys[i + 1] & mask : 0, s2 = left > 2 ? keys[i + 2] & mask : 0,
                           s3 = left > 3 ? keys[i + 3] & mask : 0;
            const bool first = rank == 0;
            p.shared[j] = (uint32_t)(run - p.first_run[x]);
            if (x + 1 == p.nslices) {
                gz_u32x4 a;
                a.x = (uint32_t)s0 | (first ? 0x80000000u : 0u);
                a.y = left > 1 ? (uint32_t)s1 : GZ_PACKED_NONE;
                a.z = left > 2 ? (uint32_t)s2 : GZ_PACKED_NONE;
                a.w = left > 3 ? (uint32_t)s3 : GZ_PACKED_NONE;
                p.nbr[j - p.cold_first] = a;
                continue;
            }
            const uint32_t level = x / GZ_XCDS;
            const uint64_t window = gz_slice_window(x, p.S, p.blocks);
            if (level >= 1 && level <= p.blocks) {
                const uint64_t w = window + (uint64_t)level * p.H;
                const uint64_t f0 = (s0 - w) | (first ? GZ_PACKED16_FIRST : 0u);
                const uint64_t f1 = left > 1 ? s1 - w : GZ_PACKED16_NONE;
                const uint64_t f2 = left > 2 ? s2 - w : GZ_PACKED16_NONE;
                const uint64_t f3 = left > 3 ? s3 - w : GZ_PACKED16_NONE;
                p.nbr16[j - p.block_first] = f0 | (f1 << 16) | (f2 << 32) | (f3 << 48);
                continue;
            }
            const uint32_t f0 = (uint32_t)(s0 - window) | (first ? 0x800000u : 0u);
            const uint32_t f1 = left > 1 ? (uint32_t)(s1 - window) : 0xffffffu;
            const uint32_t f2 = left > 2 ? (uint32_t)(s2 - window) : 0xffffffu;
            const uint32_t f3 = left > 3 ? (uint32_t)(s3 - window) : 0xffffffu;
            uint32_t* w = p.nbr24 + 3 * (j - (level > p.blocks ? p.block_span : 0));
            w[0] = f0 | (f1 << 24);
            w[1] = (f1 >> 8) | (f2 << 16);
            w[2] = (f2 >> 16) | (f3 << 8);
        }
    }
}

/* mask[v] bit x: v has vectors in slice x; rank_base[k * nslices + x]: the
 * first run of slice x whose destination is not below 64 k.  A wavefront takes
 * `per` consecutive 64-vertex blocks: lane x finds slice x's run at the first
 * of them by binary search in the runs' destinations (ascending inside a
 * slice) and steps it from block to block by the runs the block held.  The
 * lanes meet in a row of LDS words of their wavefront's own. */
template <typename M>
__global__ __launch_bounds__(GZ_BLOCK) void gz_k_slice_mask(const uint32_t* __restrict__ gid, uint32_t nslices,
                                                            const uint64_t* __restrict__ first_run, uint64_t nv,
                                                            uint64_t nblocks, uint64_t per, M* __restrict__ mask,
                                                            uint32_t* __restrict__ rank_base)
{
    __shared__ unsigned long long bits[GZ_WAVES_PER_BLOCK][GZ_WAVE];
    const int lane = gz_lane();
    unsigned long long* mine = bits[threadIdx.x / GZ_WAVE];
    const uint64_t wave = (uint64_t)blockIdx.x * GZ_WAVES_PER_BLOCK + threadIdx.x / GZ_WAVE;
    const uint64_t k0 = wave * per;
    if (k0 >= nblocks) return;
    const uint64_t k1 = k0 + per < nblocks ? k0 + per : nblocks;
    uint32_t at = 0, end = 0;
    if ((uint32_t)lane < nslices) {
        at = (uint32_t)first_run[lane];
        end = (uint32_t)first_run[lane + 1];
        uint32_t z = end;
        while (at < z) {
            const uint32_t mid = at + ((z - at) >> 1);
            if ((uint64_t)gid[mid] < k0 * GZ_WAVE)
                at = mid + 1;
            else
                z = mid;
        }
    }
    for (uint64_t k = k0; k < k1; ++k) {
        if ((uint32_t)lane < nslices) rank_base[k * nslices + (uint32_t)lane] = at;
        mine[lane] = 0;
        gz_wave_lds_sync();
        const uint64_t stop = (k + 1) * GZ_WAVE;
        for (uint32_t x0 = 0; x0 < nslices; x0 += 8) {
            uint32_t g[8];
#pragma unroll
            for (uint32_t u = 0; u < 8; ++u) {
                const uint32_t x = x0 + u; /* lanes from nslices on hold empty ranges; x stays below 64 */
                const uint32_t i = (uint32_t)__builtin_amdgcn_readlane((int)at, (int)x) + (uint32_t)lane;
                g[u] = i < (uint32_t)__builtin_amdgcn_readlane((int)end, (int)x) ? gid[i] : 0xffffffffu;
            }
#pragma unroll
            for (uint32_t u = 0; u < 8; ++u) {
                const bool in = (uint64_t)g[u] < stop;
                if (in) atomicOr(&mine[g[u] & (GZ_WAVE - 1)], 1ull << (x0 + u));
                const uint32_t c = (uint32_t)__popcll(__ballot(in));
                if ((uint32_t)lane == x0 + u) at += c;
            }
        }
        gz_wave_lds_sync();
        const uint64_t v = k * GZ_WAVE + (uint64_t)lane;
        if (v < nv) mask[v] = (M)mine[lane];
    }
}

/* 32-bit copy of the FP64 out-degrees (integral, below 2^32: V <= 2^28 here). */
__global__ void gz_k_outdeg32(const double* __restrict__ outdeg, uint64_t n, uint32_t* __restrict__ out)
{
    /* grid-stride: gz_grid_for caps the grid at 65,536 workgroups */
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        out[i] = (uint32_t)outdeg[i];
}

/* A block that keeps the packed arrays away from the vertex arrays in device
 * memory while they are allocated (nullptr: none), given back afterwards.
 *
 * The pull's streams of packed vectors slow its gathers of the properties (and
 * the vertex phase's streams its stores of them) by their distance in physical
 * memory, with a period of 32 GiB: PageRank over the 41.7 M-vertex graph, 10
 * iterations, takes 52.4 to 52.5 ms where the packed arrays begin 8 to 23 GiB
 * past the properties (modulo 32), 53.4 to 53.6 from 25 to 38; pull 4358 and
 * vertex phase 937 us there, 4332 and 903 with the pages of an older build,
 * whose 57 temporary lists broke them up.  Pages lie as the device hands them
 * out: on one that nothing else has used in the order of the allocations, so
 * the distance is what lies between, this layout's two key buffers and the
 * runs' ids (25 GiB for that graph); on one with other tenants anywhere, and the
 * block neither helps nor harms (measured on such a one: 52.1 ms with and
 * without).  Smaller vertex arrays stay in the 256 MB last-level cache.
 *
 * The block is taken only where the device has the `need` bytes of the build's
 * remaining arrays beside it, and a GiB: no build fails for it. */
void* gz_slices_spacer(uint64_t nv, uint64_t between, uint64_t need)
{
    size_t idle = 0, whole = 0;
    void* p = nullptr;
    if (hipMemGetInfo(&idle, &whole) == hipSuccess) {
        const uint64_t bytes = gz_slices_spacer_bytes(nv, between, need, idle);
        if (bytes == 0 || hipMalloc(&p, bytes) == hipSuccess) return p;
    }
    (void)hipGetLastError(); /* as well without */
    return nullptr;
}

}  // namespace

/* Bytes of that block (0: none). */
extern "C" uint64_t gz_slices_spacer_bytes(uint64_t nv, uint64_t between, uint64_t need, uint64_t idle)
{
    const uint64_t gib = 1ull << 30, period = 32 * gib, aim = 15 * gib;
    const uint64_t at = between % period, bytes = (aim + period - at) % period;
    if (nv * sizeof(double) <= gib / 4 || (at >= 8 * gib && at <= 22 * gib)) return 0;
    return idle >= need && idle - need >= bytes + gib ? bytes : 0;
}

extern "C" int gz_graph_build_source_slices(uint64_t slice_vertices, uint32_t tiers, uint32_t blocks,
                                            uint64_t block_vertices)
{
    gz_runtime_init(0);
    if (gz_graph.pull_vectors == nullptr) {
        fprintf(stderr, "grazelle: the source-sliced layout needs a pull layout\n");
        exit(65);
    }
    const uint64_t nv = gz_graph.num_vertices, nvec = gz_graph.pull_vector_count;
    const uint32_t b = gz_id_bits(nv);
    if (2 * b + GZ_SLICE_KEY_BITS > 64) {
        fprintf(stderr, "grazelle: the source-sliced layout needs V <= 2^28 (V = %llu)\n", (unsigned long long)nv);
        exit(65);
    }
    if (tiers < 1 || tiers > GZ_MAX_TIERS || blocks + tiers > GZ_MAX_LEVELS) {
        fprintf(stderr, "grazelle: source-sliced tiers must be 1..%d and tiers + blocks at most %d (got %u, %u)\n",
                GZ_MAX_TIERS, GZ_MAX_LEVELS, tiers, blocks);
        exit(65);
    }
    gz_source_slices_release();
    const uint64_t S = gz_slices_effective(slice_vertices, tiers, nv);
    /* as many of the requested blocks as fit in a window after its block 0 */
    const uint64_t H = blocks ? block_vertices : 0;
    if (H > GZ_PACKED16_NONE) {
        fprintf(stderr, "grazelle: LDS blocks hold at most %u sources (got %llu)\n", GZ_PACKED16_NONE,
                (unsigned long long)H);
        exit(65);
    }
    if (blocks && (H == 0 || S / H < 1))
        blocks = 0;
    else if (blocks && S / H - 1 < blocks)
        blocks = (uint32_t)(S / H - 1);
    const uint32_t ns = GZ_XCDS * (tiers + blocks) + 1;
    const bool wide_mask = ns > 32;
    const uint64_t n = 4 * nvec;
    uint64_t* a = (uint64_t*)gz_pool_malloc((n ? n : 1) * sizeof(uint64_t), 0);
    uint64_t* bb = (uint64_t*)gz_pool_malloc((n ? n : 1) * sizeof(uint64_t), 0);
    /* per slice: first key, first run, first vector (zero without edges) */
    uint64_t* firsts = (uint64_t*)gz_pool_malloc(3 * (GZ_MAX_SLICES + 1) * sizeof(uint64_t), 1);
    uint64_t* first_run = firsts + GZ_MAX_SLICES + 1;
    uint64_t* first_vec = first_run + GZ_MAX_SLICES + 1;
    uint64_t* sorted = a;
    uint64_t m = 0, runs = 0, tiles = 0;
    uint64_t *tile_base = nullptr, *run_first = nullptr, *run_vec = nullptr;
    if (n) {
        hipLaunchKernelGGL(gz_k_slice_keys, dim3(gz_grid_for(n)), dim3(GZ_BLOCK), 0, gz_stream, gz_graph.pull_vectors,
                           nvec, b, S, tiers, blocks, H, a);
        GZ_LAUNCH_CHECK();
        gz_sort_keys(a, bb, n, 2 * b, 2 * b + GZ_SLICE_KEY_BITS, &sorted);
        hipLaunchKernelGGL(gz_k_slice_bounds, dim3(1), dim3(64), 0, gz_stream, sorted, n, b, ns, firsts);
        GZ_LAUNCH_CHECK();
        gz_copy_to_host(&m, firsts + ns, sizeof(uint64_t));
        tiles = (m + GZ_TILE - 1) / GZ_TILE;
    }
    if (m) {
        uint64_t* sums = (uint64_t*)gz_pool_malloc(2 * (tiles + 1) * sizeof(uint64_t), 1); /* sums[tiles] stays 0 */
        tile_base = sums + tiles + 1;
        hipLaunchKernelGGL(gz_k_tile_count<true>, dim3(gz_tile_grid(tiles)), dim3(GZ_BLOCK), 0, gz_stream, sorted, m, b,
                           ~0ull, tiles, sums);
        GZ_LAUNCH_CHECK();
        gz_scan(sums, tile_base, tiles + 1);
        gz_copy_to_host(&runs, tile_base + tiles, sizeof(uint64_t));
    }
    if (runs + 8 > 0xffffffffull) {
        fprintf(stderr, "grazelle: the sliced layout needs fewer than 2^32 slice accumulators\n");
        exit(65);
    }
    gz_slices.gid = (uint32_t*)gz_pool_malloc((runs + 8) * sizeof(uint32_t), 1);
    if (m) {
        run_first = (uint64_t*)gz_pool_malloc((runs + 1) * sizeof(uint64_t), 0);
        run_vec = (uint64_t*)gz_pool_malloc((runs + 1) * sizeof(uint64_t), 0);
        hipLaunchKernelGGL(gz_k_slice_runs, dim3(gz_tile_grid(tiles)), dim3(GZ_BLOCK), 0, gz_stream, sorted, m, b, tiles,
                           tile_base, run_first, gz_slices.gid);
        GZ_LAUNCH_CHECK();
        gz_scan(rocprim::make_transform_iterator(rocprim::make_counting_iterator<uint64_t>(0),
                                                 gz_run_vectors{run_first, runs}),
                run_vec, runs + 1);
        hipLaunchKernelGGL(gz_k_slice_firsts, dim3(1), dim3(64), 0, gz_stream, firsts, ns, run_first, runs, run_vec,
                           first_run, first_vec);
        GZ_LAUNCH_CHECK();
    }
    uint64_t host_firsts[3 * (GZ_MAX_SLICES + 1)];
    gz_copy_to_host(host_firsts, firsts, sizeof(host_firsts));
    memset(&gz_slices.part_base, 0, sizeof(gz_slices.part_base));
    for (uint32_t x = 0; x <= ns; ++x) {
        gz_slices.part_base.off[x] = host_firsts[GZ_MAX_SLICES + 1 + x];
        gz_slices.begin[x] = host_firsts[2 * (GZ_MAX_SLICES + 1) + x];
    }
    const uint64_t total = gz_slices.begin[ns];
    const uint64_t cold = total - gz_slices.begin[ns - 1];
    const uint64_t block_first = gz_slices.begin[GZ_XCDS];
    const uint64_t block_span = gz_slices.begin[GZ_XCDS * (blocks + 1)] - block_first;
    const uint64_t window_total = gz_slices.begin[ns - 1] - block_span;
    const uint64_t rank_blocks = (nv + GZ_WAVE - 1) / GZ_WAVE;
    const uint64_t need = 3 * window_total * sizeof(uint32_t) + block_span * sizeof(uint64_t) +
                          cold * sizeof(gz_u32x4) + total * sizeof(uint32_t) +
                          nv * ((wide_mask ? sizeof(uint64_t) : sizeof(uint32_t)) + sizeof(uint32_t)) +
                          ns * rank_blocks * sizeof(uint32_t) + runs * sizeof(double);
    void* spacer = gz_slices_spacer(nv, 2 * n * sizeof(uint64_t) + runs * sizeof(uint32_t), need);
    gz_slices.nbr24 = (uint32_t*)gz_pool_malloc((window_total ? 3 * window_total : 1) * sizeof(uint32_t), 0);
    gz_slices.nbr16 = (uint64_t*)gz_pool_malloc((block_span ? block_span : 1) * sizeof(uint64_t), 0);
    gz_slices.block_span = block_span;
    gz_slices.nbr = (gz_u32x4*)gz_pool_malloc((cold ? cold : 1) * sizeof(gz_u32x4), 0);
    gz_slices.shared = (uint32_t*)gz_pool_malloc((total ? total : 1) * sizeof(uint32_t), 0);
    if (m) {
        const gz_slice_pack_t pack{S,         H,          blocks,    ns, block_first, block_span, gz_slices.begin[ns - 1],
                                   first_run, gz_slices.nbr24, gz_slices.nbr16, gz_slices.nbr, gz_slices.shared};
        hipLaunchKernelGGL(gz_k_slice_pack, dim3(gz_tile_grid(tiles)), dim3(GZ_BLOCK), 0, gz_stream, sorted, m, b, tiles,
                           tile_base, run_first, run_vec, pack);
        GZ_LAUNCH_CHECK();
    }
    gz_slices.mask = gz_pool_malloc((nv + 8) * (wide_mask ? sizeof(uint64_t) : sizeof(uint32_t)), 1);
    gz_slices.rank_blocks = rank_blocks;
    gz_slices.rank_base = (uint32_t*)gz_pool_malloc(ns * gz_slices.rank_blocks * sizeof(uint32_t), 0);
    /* consecutive blocks per wavefront: few enough that the chip is full */
    uint64_t per = gz_slices.rank_blocks / ((uint64_t)gz_cu_count * 32);
    per = per < 1 ? 1 : per > 64 ? 64 : per;
    const uint64_t mask_waves = (gz_slices.rank_blocks + per - 1) / per;
    const unsigned mask_grid = (unsigned)((mask_waves + GZ_WAVES_PER_BLOCK - 1) / GZ_WAVES_PER_BLOCK);
    if (wide_mask)
        hipLaunchKernelGGL(gz_k_slice_mask<uint64_t>, dim3(mask_grid), dim3(GZ_BLOCK), 0, gz_stream, gz_slices.gid, ns,
                           first_run, nv, gz_slices.rank_blocks, per, (uint64_t*)gz_slices.mask, gz_slices.rank_base);
    else
        hipLaunchKernelGGL(gz_k_slice_mask<uint32_t>, dim3(mask_grid), dim3(GZ_BLOCK), 0, gz_stream, gz_slices.gid, ns,
                           first_run, nv, gz_slices.rank_blocks, per, (uint32_t*)gz_slices.mask, gz_slices.rank_base);
    GZ_LAUNCH_CHECK();
    gz_slices.parts = (double*)gz_pool_malloc((runs + 8) * sizeof(double), 1);
    gz_slices.outdeg32 = (uint32_t*)gz_pool_malloc((nv + 8) * sizeof(uint32_t), 1);
    hipLaunchKernelGGL(gz_k_outdeg32, dim3(gz_grid_for(nv)), dim3(GZ_BLOCK), 0, gz_stream, gz_graph.vertex_outdegrees,
                       nv, gz_slices.outdeg32);
    GZ_LAUNCH_CHECK();
    GZ_CHECK(hipStreamSynchronize(gz_stream));
    if (spacer) GZ_CHECK(hipFree(spacer));
    gz_pool_free(run_vec);
    gz_pool_free(run_first);
    if (tile_base) gz_pool_free(tile_base - (tiles + 1));
    gz_pool_free(firsts);
    gz_pool_free(a);
    gz_pool_free(bb);
    gz_slices.base_list = gz_graph.pull_vectors;
    gz_slices.base_count = nvec;
    gz_slices.slice_vertices = S;
    gz_slices.tiers = tiers;
    gz_slices.blocks = blocks;
    gz_slices.block_vertices = H;
    gz_slices.nslices = ns;
    return 0;
}
