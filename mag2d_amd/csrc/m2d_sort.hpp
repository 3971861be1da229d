// m2d_sort.hpp -- the sort of a particle store by tile, for the 2D and the 3D
// stores: keys, rocPRIM's radix sort of (key, slot), and the gather of the
// components into the new order.
//
// A random store's gather is bound by its reads: 4 bytes wanted of every
// cache line they touch, once per component (16.7M slots of 6 components
// 1955 us, 4.2M of 5 354 us).  Such a store is first packed into records of
// 32 bytes by the key kernel, which streams, and the gather then touches one
// line a particle (keys and gather 74 + 1955 -> 188 + 431 us, 15 + 354 -> 52 +
// 93 us).  A store that is nearly in tile order reads whole lines either way,
// and packing only adds to it; a sample of neighbouring slots tells the two
// apart on the device.
#pragma once
#include <rocprim/device/device_radix_sort.hpp>
#include "m2d_objects.hpp"

namespace m2d {

// component pointers of a store, x first
template <int NC>
struct Columns {
    float *c[NC];
};

// Clears the live count and samples 2016 pairs of neighbouring slots, 32
// evenly spread wavefronts of 64 slots: *scattered = more than 3/8 of the
// pairs of live slots lie in two tiles.  (A whole sort of 4.2M slots of which
// a share was moved at random, gather direct and packed: none 166 and 206 us,
// 0.15 206 and 219, 0.2 222 and 223, 0.3 253 and 227, 1.0 478 and 245; a share
// of 0.2 leaves 0.36 of the pairs in two tiles.)  Key: slot -> (tile << 6 |
// cell), dead_key for an empty slot.  One block.
constexpr int kSampleWaves = 32;
template <class Key>
__global__ void __launch_bounds__(1024) k_sort_sample(Key key, int64_t n, uint32_t dead_key,
                                                      unsigned long long *live, uint32_t *scattered)
{
    __shared__ int s_pairs, s_differ;
    if (threadIdx.x == 0) s_pairs = s_differ = 0;
    __syncthreads();
    const int lane = threadIdx.x & 63;
    int pairs = 0, differ = 0;
#pragma unroll
    for (int r = 0; r < kSampleWaves / 16; r++) {
        const int64_t p = (n / kSampleWaves) * (r * 16 + (threadIdx.x >> 6)) + lane;
        const uint32_t a = p < n ? key(p) : dead_key, b = __shfl_down(a, 1);
        const bool both = lane < 63 && a != dead_key && b != dead_key;
        pairs += __popcll(__ballot(both));
        differ += __popcll(__ballot(both && (a >> 6) != (b >> 6)));
    }
    if (lane == 0) {
        atomicAdd(&s_pairs, pairs);
        atomicAdd(&s_differ, differ);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        *live = 0ull;
        *scattered = 8 * s_differ > 3 * s_pairs ? 1u : 0u;
    }
}

// Every slot's key and index, a scattered store's records (rec may be null), and zeros
// in bounds[0, n_bounds), which the gather fills
template <class Key, int NC>
__global__ void __launch_bounds__(256) k_sort_keys(Key key, Columns<NC> src, int64_t n, uint32_t *keys, uint32_t *vals,
                                                   float4 *rec, const uint32_t *scattered, int *bounds,
                                                   int64_t n_bounds)
{
    const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
    for (int64_t q = p; q < n_bounds; q += (int64_t)gridDim.x * 256) bounds[q] = 0;
    if (p >= n) return;
    keys[p] = key(p);
    vals[p] = (uint32_t)p;
    if (rec && *scattered) {
        float v[8];
#pragma unroll
        for (int c = 0; c < 8; c++) v[c] = c < NC ? src.c[c < NC ? c : 0][p] : 0.f;
        rec[2 * p] = make_float4(v[0], v[1], v[2], v[3]);
        rec[2 * p + 1] = make_float4(v[4], v[5], v[6], v[7]);
    }
}

// The components in key order, the live count, and [start, end) of every
// non-empty tile (tstart and tend zero on entry)
template <int NC>
__global__ void __launch_bounds__(256) k_sort_gather(Columns<NC> src, Columns<NC> dst, int64_t n, const uint32_t *keys,
                                                     const uint32_t *vals, uint32_t dead_key,
                                                     unsigned long long *n_live, const float4 *rec,
                                                     const uint32_t *scattered, int *tstart, int *tend)
{
    // destination ranges in XCD-contiguous order: a nearly sorted store's
    // sources of neighbouring ranges share cache lines, and then one L2
    const unsigned nb = (unsigned)((n + 255) / 256);
    const unsigned b = xcd_block(blockIdx.x, nb);
    if (b >= nb) return;
    const int64_t i = (int64_t)b * 256 + threadIdx.x;
    if (i >= n) return;
    const uint32_t k = keys[i];
    if (k == dead_key) {
        dst.c[0][i] = dead_value();
        return;
    }
    const int64_t s = vals[i];
    float v[8];
    if (rec && *scattered) {
        const float4 a = rec[2 * s], e = rec[2 * s + 1];
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
        v[4] = e.x; v[5] = e.y; v[6] = e.z; v[7] = e.w;
    } else {
#pragma unroll
        for (int c = 0; c < NC; c++) v[c] = src.c[c][s];
    }
    const bool last = i == n - 1;
    const uint32_t before = i == 0 ? dead_key : keys[i - 1], after = last ? dead_key : keys[i + 1];
    const uint32_t t = k >> 6;
    if (i == 0 || (before >> 6) != t) tstart[t] = (int)i;
    if (after == dead_key || (after >> 6) != t) tend[t] = (int)(i + 1);
    if (after == dead_key) *n_live = (unsigned long long)(i + 1);
#pragma unroll
    for (int c = 0; c < NC; c++) dst.c[c][i] = v[c];
}

// The smallest key width whose largest value, the dead key, is above every
// live key of `tiles` tiles
inline int sort_key_bits(uint64_t tiles)
{
    int bits = 0;
    while ((1ull << bits) <= (tiles << 6)) bits++;
    return bits;
}
inline uint32_t sort_dead_key(int bits) { return bits == 32 ? 0xFFFFFFFFu : (uint32_t)((1ull << bits) - 1); }

// The sort's scratch: keys and slots, the sorted ones, the radix sort's
// temporaries and the sample's answer.  n > 0.
struct SortScratch {
    uint32_t *k0, *k1, *v0, *v1, *scattered;
    void *radix;
};
int sort_scratch(m2d_ctx *ctx, size_t n, size_t radix_bytes, SortScratch &s);
// The records' memory, 32 bytes a slot, where a quarter of what is free holds
// it; null otherwise, and in a call that is being captured in a graph (whose
// replays would keep the address).  After the call's other allocations, which
// may give it back (dev_malloc).
float4 *sort_records(m2d_ctx *ctx, size_t n);
// Queue the schedule of a tile-sorted store: tiling_begin before the gather,
// which fills T->tile_start and T->tile_end (adjacent, zeroed before it) and
// tiling_finish after it
int tiling_begin(m2d_ctx *ctx, const float *x, int64_t n, int ntx, int nty, int ntz, int cap, m2d_tiling *&T);
int tiling_finish(m2d_ctx *ctx, m2d_tiling *T, const float *x, int64_t n, int cap, int round);

// Up to this many slots by merge sort, whose launches grow with the count;
// above, by digits: a whole sort of 200k slots takes 83 and 90 us, of 300k 143
// and 96, of 1M 243 and 117.  (rocPRIM's own limit is 1M.)
constexpr size_t kMergeSortSlots = 1 << 18;
using SortConfig = rocprim::radix_sort_config<rocprim::default_config, rocprim::default_config,
                                              rocprim::default_config, kMergeSortSlots>;

// src in key order into dst, ranking key bits [lo, bits), and dst's schedule
// (tiles ntx * nty * ntz of 64 cells; cap and round as tiling_finish)
template <int NC, class Key>
int sort_store(m2d_ctx *ctx, const Key &key, const Columns<NC> &src, const Columns<NC> &dst, size_t n, int lo,
               int bits, int ntx, int nty, int ntz, int cap, int round, int64_t *n_live)
{
    const uint32_t dead_key = sort_dead_key(bits);
    size_t temp = 0;
    hipError_t e = rocprim::radix_sort_pairs<SortConfig>(nullptr, temp, (const uint32_t *)nullptr, (uint32_t *)nullptr,
                                                         (const uint32_t *)nullptr, (uint32_t *)nullptr, n, lo, bits,
                                                         ctx->stream);
    M2D_CHECK(e == hipSuccess, M2D_ERR_HIP, "radix_sort_pairs size query: %s", hipGetErrorString(e));
    SortScratch w;
    M2D_TRY(sort_scratch(ctx, n, temp, w));
    m2d_tiling *T;
    M2D_TRY(tiling_begin(ctx, dst.c[0], (int64_t)n, ntx, nty, ntz, cap, T));
    float4 *const rec = sort_records(ctx, n);
    unsigned long long *live = ctx->counters + CNT_LIVE;
    const unsigned blocks = (unsigned)((n + 255) / 256);
    k_sort_sample<<<1, 1024, 0, ctx->stream>>>(key, (int64_t)n, dead_key, live, w.scattered);
    k_sort_keys<<<blocks, 256, 0, ctx->stream>>>(key, src, (int64_t)n, w.k0, w.v0, rec, w.scattered, T->tile_start,
                                                 2 * (int64_t)ntx * nty * ntz);
    M2D_HIP(hipGetLastError());
    e = rocprim::radix_sort_pairs<SortConfig>(w.radix, temp, w.k0, w.k1, w.v0, w.v1, n, lo, bits, ctx->stream);
    M2D_CHECK(e == hipSuccess, M2D_ERR_HIP, "radix_sort_pairs: %s", hipGetErrorString(e));
    k_sort_gather<<<xcd_grid(blocks), 256, 0, ctx->stream>>>(src, dst, (int64_t)n, w.k1, w.v1, dead_key, live, rec,
                                                             w.scattered, T->tile_start, T->tile_end);
    M2D_HIP(hipGetLastError());
    M2D_TRY(tiling_finish(ctx, T, dst.c[0], (int64_t)n, cap, round));
    if (n_live) {
        M2D_TRY(read_counters(ctx));
        *n_live = (int64_t)ctx->h_counters[CNT_LIVE];
    }
    return M2D_OK;
}

}  // namespace m2d
