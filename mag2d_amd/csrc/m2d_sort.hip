// m2d_sort.hip -- stable reordering of a species' particles by tile, and the
// tile schedule of the sorted store.
//
// The reference keeps particles in insertion order with holes
// (particles.hpp:223-249).  Here the store is periodically rebuilt in tile
// order (8 x 8-cell tiles, row-major), dropping empty slots: each block of
// the particle pass then gathers from and deposits into one small window of
// the grid, held in LDS.  Inside a tile the particles keep their old slot
// order, so the result is deterministic.  They are deliberately not ordered
// by cell: the 64 lanes of a wave would then share one or two cells, and
// their LDS atomics on the same four nodes would serialise (a cell-ordered
// store runs the pass about 1.5x slower until the particles have mixed).
// The key holds the cell too (tile << 6 | cell) and the radix sort ranks the
// tile bits only (rocPRIM's LSD radix sort of the key/slot pairs).
#include <cstring>
#include <new>
#include "m2d_sort.hpp"

namespace m2d {

struct SortGeom {
    int nx, nz, ntz;
    double idx, idz, xmin, zmin;
};

__device__ __forceinline__ uint32_t cell_key(const SortGeom &g, double x, double z)
{
    double X = (x - g.xmin) * g.idx, Z = (z - g.zmin) * g.idz;
    int i = X >= 0.0 ? (int)fmin(X, (double)(g.nx - 2)) : 0;
    int j = Z >= 0.0 ? (int)fmin(Z, (double)(g.nz - 2)) : 0;
    uint32_t tile = (uint32_t)((i / kTile) * g.ntz + (j / kTile));
    return (tile << kTileShift) | ((uint32_t)(i % kTile) << 3) | (uint32_t)(j % kTile);
}

// a slot's key; that of a long-time position (xl, zl not null) is the FP64 sum's
struct Key2 {
    const float *x, *z, *xl, *zl;
    SortGeom g;
    uint32_t dead_key;
    __device__ __forceinline__ uint32_t operator()(int64_t p) const
    {
        const float v = x[p];
        return is_dead(v) ? dead_key : xl ? cell_key(g, pos64(v, xl[p]), pos64(z[p], zl[p])) : cell_key(g, v, z[p]);
    }
};

// The schedule's order class of a chunk [a, e): the rounds of `round`
// slots the pass takes over it (its rounds start at a rounded down to 64),
// less one, at most kSchedClasses - 1; round = 0: class 0 for all
constexpr int kSchedClasses = 8;
__device__ __forceinline__ int chunk_class(int a, int e, int round)
{
    if (round <= 0) return 0;
    const int r = (e - (a & ~63) + round - 1) / round - 1;
    return min(max(r, 0), kSchedClasses - 1);
}

// A tile's chunks [start, end), start + cap, ... by class: all but the last
// are cap slots long and of one class (cap is a multiple of 64)
struct TileChunks {
    int a, e, n, full, last;  // n chunks: n - 1 of class full, one of class last
    __device__ __forceinline__ TileChunks(const int *tstart, const int *tend, int t, int ntiles, int cap, int round)
    {
        a = t < ntiles ? tstart[t] : 0;
        e = t < ntiles ? tend[t] : 0;
        n = e > a ? (e - a + cap - 1) / cap : 0;
        full = chunk_class(a, a + cap, round);
        last = chunk_class(a + (n - 1) * cap, e, round);
    }
};

// The schedule: chunks in descending class (the longest first), each class
// in tile order.  Blocks start in index order as earlier ones retire, so the
// launch ends on short blocks.  At most kSchedBlocks blocks of kSchedThreads
// threads take `per` consecutive tiles a thread; k_tile_count sums each
// block's chunks by class, k_tile_schedule adds up the blocks before its own
// and places its chunks.  (One block for all tiles was a serial chain of
// uncoalesced reads: 143 us for 32768 tiles, 17 us for 256.)
constexpr int kSchedThreads = 256, kSchedBlocks = 256;
static inline int sched_per(int ntiles)
{
    return (ntiles + kSchedThreads * kSchedBlocks - 1) / (kSchedThreads * kSchedBlocks);
}

__global__ void __launch_bounds__(kSchedThreads) k_tile_count(const int *tstart, const int *tend, int ntiles, int per,
                                                              int cap, int round, int *totals)
{
    __shared__ int s[kSchedClasses];
    if (threadIdx.x < kSchedClasses) s[threadIdx.x] = 0;
    __syncthreads();
    const int lo = (blockIdx.x * kSchedThreads + threadIdx.x) * per;
    for (int q = 0; q < per; q++) {
        const TileChunks t(tstart, tend, lo + q, ntiles, cap, round);
        if (t.n > 1) atomicAdd(&s[t.full], t.n - 1);
        if (t.n > 0) atomicAdd(&s[t.last], 1);
    }
    __syncthreads();
    if (threadIdx.x < kSchedClasses) totals[blockIdx.x * kSchedClasses + threadIdx.x] = s[threadIdx.x];
}

__global__ void __launch_bounds__(kSchedThreads) k_tile_schedule(const int *tstart, const int *tend, int ntiles,
                                                                 int per, int cap, int round, const int *totals,
                                                                 int4 *sched, unsigned int *n_chunks)
{
    __shared__ int s[kSchedClasses][kSchedThreads];  // this thread's next chunk of each class
    __shared__ int s_all[kSchedClasses], s_before[kSchedClasses], s_wave[kSchedClasses][kSchedThreads / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (tid < kSchedClasses) s_all[tid] = s_before[tid] = 0;
    __syncthreads();
    for (int b = tid; b < (int)gridDim.x * kSchedClasses; b += kSchedThreads) {
        const int v = totals[b];
        if (v) {
            atomicAdd(&s_all[b % kSchedClasses], v);
            if (b < (int)blockIdx.x * kSchedClasses) atomicAdd(&s_before[b % kSchedClasses], v);
        }
    }
    const int lo = (blockIdx.x * kSchedThreads + tid) * per;
#pragma unroll
    for (int c = 0; c < kSchedClasses; c++) s[c][tid] = 0;
    for (int q = 0; q < per; q++) {
        const TileChunks t(tstart, tend, lo + q, ntiles, cap, round);
        if (t.n > 1) s[t.full][tid] += t.n - 1;
        if (t.n > 0) s[t.last][tid]++;
    }
    // exclusive scan over the block's threads
    int own[kSchedClasses], sum[kSchedClasses];
#pragma unroll
    for (int c = 0; c < kSchedClasses; c++) {
        sum[c] = own[c] = s[c][tid];
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int v = __shfl_up(sum[c], o);
            if (lane >= o) sum[c] += v;
        }
        if (lane == 63) s_wave[c][wave] = sum[c];
    }
    __syncthreads();
    // class c starts after every chunk of the classes above it
    int base = 0;
#pragma unroll
    for (int c = kSchedClasses - 1; c >= 0; c--) {
        int first = base + s_before[c] + sum[c] - own[c];
        for (int w = 0; w < wave; w++) first += s_wave[c][w];
        s[c][tid] = first;
        base += s_all[c];
    }
    for (int q = 0; q < per; q++) {
        const TileChunks t(tstart, tend, lo + q, ntiles, cap, round);
        for (int k = 0; k < t.n; k++) {
            const int a = t.a + k * cap;
            sched[s[k == t.n - 1 ? t.last : t.full][tid]++] = make_int4(lo + q, a, min(t.e, a + cap), 0);
        }
    }
    if (blockIdx.x == 0 && tid == 0) *n_chunks = (unsigned int)base;
}

m2d_tiling *find_tiling(m2d_ctx *ctx, const float *x, int64_t n)
{
    for (m2d_tiling *t : ctx->tilings)
        if (t->x == x && t->n == n) return t;
    return nullptr;
}

void forget_tiling(m2d_ctx *ctx, const float *x)
{
    for (m2d_tiling *t : ctx->tilings)
        if (t->x == x) t->x = nullptr;
}

void free_tilings(m2d_ctx *ctx)
{
    for (m2d_tiling *t : ctx->tilings) {
        if (t->buf.ptr) (void)hipFree(t->buf.ptr);
        delete t;
    }
    ctx->tilings.clear();
}

int sort_scratch(m2d_ctx *ctx, size_t n, size_t radix_bytes, SortScratch &s)
{
    auto up = [](size_t v) { return (v + 255) / 256 * 256; };
    const size_t arr = up(n * 4);
    M2D_TRY(ensure(ctx, ctx->sortbuf, 4 * arr + up(radix_bytes) + 256));
    uint8_t *b = (uint8_t *)ctx->sortbuf.ptr;
    s.k0 = (uint32_t *)b;
    s.k1 = (uint32_t *)(b + arr);
    s.v0 = (uint32_t *)(b + 2 * arr);
    s.v1 = (uint32_t *)(b + 3 * arr);
    s.scattered = (uint32_t *)(b + 4 * arr);
    s.radix = b + 4 * arr + 256;
    return M2D_OK;
}

float4 *sort_records(m2d_ctx *ctx, size_t n)
{
    const size_t need = n * 2 * sizeof(float4);
    if (capturing(ctx)) return nullptr;
    if (ctx->pack.bytes < need) {
        size_t avail = 0, total = 0;
        if (hipMemGetInfo(&avail, &total) != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
        if (need > avail / 4 || ensure(ctx, ctx->pack, need, true) != M2D_OK) return nullptr;
    }
    return (float4 *)ctx->pack.ptr;
}

// the schedule record of the store at x (n slots, tiles ntx * nty * ntz, nty
// = 1 in 2D, 64 cells each; a tile's slots are cut into chunks of at most cap)
int tiling_begin(m2d_ctx *ctx, const float *x, int64_t n, int ntx, int nty, int ntz, int cap, m2d_tiling *&T)
{
    forget_tiling(ctx, x);
    T = nullptr;
    for (m2d_tiling *t : ctx->tilings)
        if (t->x == nullptr) { T = t; break; }
    if (!T) {
        if (ctx->tilings.size() >= 8) {  // reuse the oldest record
            T = ctx->tilings.front();
            ctx->tilings.erase(ctx->tilings.begin());
        } else {
            T = new (std::nothrow) m2d_tiling();
            M2D_CHECK(T, M2D_ERR_NO_MEMORY, "tiling: host allocation");
        }
        ctx->tilings.push_back(T);
    }
    T->x = nullptr;
    const int ntiles = ntx * nty * ntz;
    const int max_chunks = ntiles + (int)(n / cap) + 1;
    const size_t words = 2 * (size_t)ntiles + 4 * (size_t)max_chunks + kSchedBlocks * kSchedClasses + 4;
    M2D_TRY(ensure(ctx, T->buf, words * sizeof(int)));
    int *b = (int *)T->buf.ptr;
    T->sched = (int4 *)b;  // first: 16-byte aligned
    T->tile_start = b + 4 * (size_t)max_chunks;
    T->tile_end = T->tile_start + ntiles;
    T->totals = T->tile_end + ntiles;
    T->n_chunks = (unsigned int *)(T->totals + kSchedBlocks * kSchedClasses);
    T->ntx = ntx;
    T->nty = nty;
    T->ntz = ntz;
    T->max_chunks = max_chunks;
    return M2D_OK;
}

// The schedule from the tiles' bounds: chunks ordered longest first by the
// rounds of `round` slots the pass takes over them (round = 0: tile order
// only).  From here on the pass finds it by the store's x and n.
static_assert(kChunkCap % 64 == 0 && kChunkCap3 % 64 == 0, "a tile's full chunks are of one class");
int tiling_finish(m2d_ctx *ctx, m2d_tiling *T, const float *x, int64_t n, int cap, int round)
{
    const int ntiles = T->ntx * T->nty * T->ntz, per = sched_per(ntiles);
    const unsigned blocks = (unsigned)((ntiles + kSchedThreads * per - 1) / (kSchedThreads * per));
    k_tile_count<<<blocks, kSchedThreads, 0, ctx->stream>>>(T->tile_start, T->tile_end, ntiles, per, cap, round,
                                                            T->totals);
    k_tile_schedule<<<blocks, kSchedThreads, 0, ctx->stream>>>(T->tile_start, T->tile_end, ntiles, per, cap, round,
                                                               T->totals, T->sched, T->n_chunks);
    M2D_HIP(hipGetLastError());
    T->n = n;
    T->x = x;
    return M2D_OK;
}

// Sort n 32-bit keys in ascending order from `in` into `out` (stream-ordered,
// temporaries in the context's sort buffer).
int sort_keys_u32(m2d_ctx *ctx, const uint32_t *in, uint32_t *out, size_t n)
{
    if (n == 0) return M2D_OK;
    size_t temp = 0;
    hipError_t e = rocprim::radix_sort_keys(nullptr, temp, in, out, n, 0, 32, ctx->stream);
    M2D_CHECK(e == hipSuccess, M2D_ERR_HIP, "radix_sort_keys size query: %s", hipGetErrorString(e));
    M2D_TRY(ensure(ctx, ctx->sortbuf, temp + 256));
    e = rocprim::radix_sort_keys(ctx->sortbuf.ptr, temp, in, out, n, 0, 32, ctx->stream);
    M2D_CHECK(e == hipSuccess, M2D_ERR_HIP, "radix_sort_keys: %s", hipGetErrorString(e));
    return M2D_OK;
}

}  // namespace m2d

using namespace m2d;

extern "C" {

int m2d_sort_2d(m2d_ctx *ctx, m2d_fields2d *f, const m2d_particles2d *src, const m2d_particles2d *dst,
                int64_t *n_live)
{
    M2D_CHECK(ctx && f && src && dst, M2D_ERR_BAD_ARG, "m2d_sort_2d: NULL argument");
    M2D_CHECK(src->n >= 0 && src->n < (1ll << 31), M2D_ERR_BAD_ARG, "m2d_sort_2d: %lld slots",
              (long long)src->n);
    M2D_CHECK(dst->n == src->n, M2D_ERR_BAD_ARG, "m2d_sort_2d: dst holds %lld slots, src %lld",
              (long long)dst->n, (long long)src->n);
    M2D_CHECK(src->n == 0 || (src->x && src->z && src->vx && src->vy && src->vz && dst->x && dst->z &&
                              dst->vx && dst->vy && dst->vz),
              M2D_ERR_BAD_ARG, "m2d_sort_2d: NULL particle array");
    M2D_CHECK(src->x != dst->x, M2D_ERR_BAD_ARG, "m2d_sort_2d: src and dst must differ");
    M2D_CHECK((src->xl == nullptr) == (src->zl == nullptr) && (dst->xl == nullptr) == (dst->zl == nullptr) &&
                  (src->xl == nullptr) == (dst->xl == nullptr),
              M2D_ERR_BAD_ARG, "m2d_sort_2d: src and dst must both hold position remainders or neither");
    const size_t n = (size_t)src->n;
    SortGeom g;
    g.nx = f->nx; g.nz = f->nz;
    const int ntx = (f->nx - 2) / kTile + 1;
    g.ntz = (f->nz - 2) / kTile + 1;
    g.idx = f->idx; g.idz = f->idz;
    g.xmin = f->p.grid.xmin; g.zmin = f->p.grid.zmin;
    const int bits = sort_key_bits((uint64_t)ntx * g.ntz);
    M2D_CHECK(bits <= 32, M2D_ERR_BAD_ARG, "m2d_sort_2d: grid too large for 32-bit keys");
    forget_tiling(ctx, src->x);
    if (n == 0) {
        forget_tiling(ctx, dst->x);
        if (n_live) *n_live = 0;
        return M2D_OK;
    }
    const Key2 key{src->x, src->z, src->xl, src->zl, g, sort_dead_key(bits)};
    if (src->xl) {
        const Columns<7> from{{src->x, src->z, src->vx, src->vy, src->vz, src->xl, src->zl}},
            to{{dst->x, dst->z, dst->vx, dst->vy, dst->vz, dst->xl, dst->zl}};
        return sort_store(ctx, key, from, to, n, kTileShift, bits, ntx, 1, g.ntz, kChunkCap, kRound2, n_live);
    }
    const Columns<5> from{{src->x, src->z, src->vx, src->vy, src->vz}},
        to{{dst->x, dst->z, dst->vx, dst->vy, dst->vz}};
    return sort_store(ctx, key, from, to, n, kTileShift, bits, ntx, 1, g.ntz, kChunkCap, kRound2, n_live);
}

int m2d_sort_forget_2d(m2d_ctx *ctx, const m2d_particles2d *p)
{
    M2D_CHECK(ctx && p, M2D_ERR_BAD_ARG, "m2d_sort_forget_2d: NULL argument");
    forget_tiling(ctx, p->x);
    return M2D_OK;
}

}  // extern "C"
