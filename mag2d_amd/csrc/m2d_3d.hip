// m2d_3d.hip -- the 3D path: Field3D gather/deposit (Field3D.hpp:40-163),
// the Species<CARTESIAN3D> step (species3d.cpp:3-94) as one pass, its cell
// sort, and the 7-point Poisson solve that replaces Solver (fields3d.cpp:35-101).
//
// Solver: FP64 iterative refinement around FP32 conjugate gradients on the
// Dirichlet-eliminated SPD system 6u - sum_free u_nb = ..., preconditioned by
// one symmetric geometric multigrid V-cycle: coarse node I sits on fine node
// 2I, every level carries a 7-point operator of its own (mg3_setup),
// restriction is P^T / 2 (full weighting with the h^2 of the coarser
// spacing), one red-black Gauss-Seidel sweep smooths on either side, and the
// coarsest level is solved by a dense inverse.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <new>
#include "m2d_objects.hpp"
#include "m2d_sort.hpp"
#include "m2d_scatter.hpp"

namespace m2d {

struct Mg3Level {
    int nx = 0, ny = 0, nz = 0;
    size_t n = 0;
    uint8_t *nbm = nullptr;   // per node: bits 0-5 set for links to free neighbours -x,-y,-z,+z,+y,+x;
                              // 0x40: colour (i+j+k) & 1; 0x80: pinned
    float *di = nullptr;      // inverse diagonal (level 0: 1/6, no array)
    float *x = nullptr, *b = nullptr;  // not on level 0
};

}  // namespace m2d

struct m2d_fields3d {
    m2d_ctx *ctx = nullptr;
    m2d_fields3d_params p{};
    int nx = 0, ny = 0, nz = 0;
    size_t n = 0;
    double idx = 0, idy = 0, idz = 0;
    uint8_t *mask = nullptr;
    uint8_t *cellfree = nullptr;   // cell (i,j,k) at its lower corner: any of 8 corners FREE
    double *voltage = nullptr, *u = nullptr, *rho = nullptr;
    float *tx = nullptr, *ty = nullptr, *tz = nullptr;  // (u_m - u_{m-e}) * 1/h per axis, FP32
    std::vector<m2d::Mg3Level> lv;
    float *coarse_inv = nullptr;   // inverse of the coarsest operator over all its nodes (symmetric)
    bool coarse_dense = true;
    unsigned int *ticket = nullptr;  // block counter of the fused reductions
    float *pr = nullptr, *pz = nullptr, *pp = nullptr, *pp2 = nullptr, *pq = nullptr, *pe = nullptr;
    double *dots = nullptr, *h_dots = nullptr, *partial = nullptr;
    int npartial = 0;
    m2d::SolveEst est;  // the last solve's passes and iterations: what the next queues
};

namespace m2d {

__device__ __forceinline__ bool dir3(uint8_t m) { return m == M2D_FIXED || m == M2D_FIXED_RF; }

// ------------------------------------------------------------------ tables and solve kernels
// Kernels of a thread a node run in blocks of 64 x 4 nodes (k, j) and a grid
// of (nz / 64, ny / 4, nx), which stops at the 65535 blocks that a launch takes
// along y and z: their threads step on to the nodes past it.
static dim3 planes3(int nx, int ny, int nz)
{
    return dim3((unsigned)((nz + 63) / 64), (unsigned)std::min((ny + 3) / 4, 65535), (unsigned)std::min(nx, 65535));
}

__global__ void __launch_bounds__(256) k3_tables(const double *u, int nx, int ny, int nz, double idx, double idy,
                                                 double idz, float *tx, float *ty, float *tz)
{
    const int k = blockIdx.x * 64 + threadIdx.x;
    if (k >= nz) return;
    for (int i = blockIdx.z; i < nx; i += gridDim.z)
        for (int j = blockIdx.y * 4 + threadIdx.y; j < ny; j += gridDim.y * 4) {
            const size_t m = ((size_t)i * ny + j) * nz + k, sx = (size_t)ny * nz;
            const double c = u[m], ux = u[i >= 1 ? m - sx : m], uy = u[j >= 1 ? m - nz : m], uz = u[k >= 1 ? m - 1 : m];
            tx[m] = (float)((c - ux) * idx);
            ty[m] = (float)((c - uy) * idy);
            tz[m] = (float)((c - uz) * idz);
        }
}

// u += e on free nodes
__global__ void k3_add_correction(const uint8_t *mask, double *u, const float *e, size_t n, const int *stop)
{
    if (stopped(stop)) return;
    size_t m = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (m < n && !dir3(mask[m])) u[m] += (double)e[m];
}

// ---- the finest level's stencils outside the V-cycle.  A block of 64 x 4
// threads (k, j) takes DI planes of i: a thread reads its column of nodes and
// the two columns beside it along j whole, before it stores anything (the
// arrays do not alias), and gets the neighbours along k from the lanes beside
// it.  A node then costs 3 reads and a bit instead of 7, all in flight
// together.  DI is 8 where that fills the GPU, 4 on smaller grids.
constexpr int kMarchK = 64, kMarchJ = 4;
struct Cols3 {
    int nx, ny, nz;
    int di() const { return (size_t)nx * ny * nz >= (1 << 20) ? 8 : 4; }
    dim3 grid() const
    {
        return dim3((unsigned)((nz + kMarchK - 1) / kMarchK), (unsigned)((ny + kMarchJ - 1) / kMarchJ),
                    (unsigned)((nx + di() - 1) / di()));
    }
    unsigned blocks() const
    {
        const dim3 g = grid();
        return g.x * g.y * g.z;
    }
};

// the thread's column: j, k (clamped onto the grid), whether it is inside
struct Column3 {
    bool in;
    int lane, k;
    size_t col, up, dn;  // offsets in a plane: its node, j - 1, j + 1 (clamped: never a free node's)
    __device__ explicit Column3(const Cols3 &g)
    {
        lane = threadIdx.x & 63;
        const int jj = blockIdx.y * kMarchJ + (threadIdx.x >> 6), kk = blockIdx.x * kMarchK + lane;
        in = jj < g.ny && kk < g.nz;
        const int j = min(jj, g.ny - 1);
        k = min(kk, g.nz - 1);
        col = (size_t)j * g.nz + k;
        up = col - (j > 0 ? g.nz : 0);
        dn = col + (j < g.ny - 1 ? g.nz : 0);
    }
};

// DI + 2 planes of the column from plane i0 - 1 on and DI of each column
// beside it (planes clamped onto the grid, as no free node lies on a face),
// and what the first and the last lane have beside them along k
template <class T, int DI>
struct Reach3 {
    T c[DI + 2], up[DI], dn[DI], edge[DI];
    template <class F>
    __device__ __forceinline__ void read(const Column3 &C, const Cols3 &g, int i0, F at)
    {
        const size_t sx = (size_t)g.ny * g.nz;
        const size_t e = C.lane == 0 ? (C.k > 0 ? C.col - 1 : C.col) : (C.k < g.nz - 1 ? C.col + 1 : C.col);
#pragma unroll
        for (int t = 0; t < DI + 2; t++) c[t] = at((size_t)min(max(i0 - 1 + t, 0), g.nx - 1) * sx + C.col);
#pragma unroll
        for (int t = 0; t < DI; t++) {
            const size_t base = (size_t)min(i0 + t, g.nx - 1) * sx;
            up[t] = at(base + C.up);
            dn[t] = at(base + C.dn);
            if (C.lane == 0 || C.lane == 63) edge[t] = at(base + e);
        }
    }
    __device__ __forceinline__ T left(const Column3 &C, int t) const
    {
        const T v = __shfl_up(c[t + 1], 1);
        return C.lane == 0 ? edge[t] : v;
    }
    __device__ __forceinline__ T right(const Column3 &C, int t) const
    {
        const T v = __shfl_down(c[t + 1], 1);
        return C.lane == 63 ? edge[t] : v;
    }
};

// The FP64 residual b - A u of the free rows (matrix_init, fields3d.cpp:35-76),
// its negative d in FP32 (0 on Dirichlet nodes), and its norms finished in the
// same launch: out[0] = |r|^2, out[1] = |b_eff|^2 (b with the Dirichlet
// neighbours moved to the right-hand side), out[2] = |d|^2.
template <int DI, class Post>
__global__ void __launch_bounds__(kRedBlock) k3_residual64_fin(Cols3 g, const uint8_t *__restrict__ mask,
                                                              const double *__restrict__ b,
                                                              const double *__restrict__ u, float *__restrict__ d,
                                                              double *partial, unsigned int *ticket, double *out,
                                                              int fin, const int *stop, Post post)
{
    const int stopped_ = stop ? *stop : 0;  // read beside the operands
    const Column3 C(g);
    const int i0 = blockIdx.z * DI;
    const size_t sx = (size_t)g.ny * g.nz;
    Reach3<double, DI> U;
    Reach3<int, DI> P;
    double bv[DI];
    P.read(C, g, i0, [&](size_t m) { return (int)dir3(mask[m]); });
    U.read(C, g, i0, [&](size_t m) { return u[m]; });
#pragma unroll
    for (int t = 0; t < DI; t++) bv[t] = b[(size_t)min(i0 + t, g.nx - 1) * sx + C.col];
    if (stopped_) return;
    double v[3] = {0, 0, 0};
#pragma unroll
    for (int t = 0; t < DI; t++) {
        const double ul = U.left(C, t), ur = U.right(C, t);
        const int pl = P.left(C, t), pr = P.right(C, t);
        if (!C.in || i0 + t >= g.nx) continue;
        float dm = 0.f;
        if (!P.c[t + 1]) {
            double au = -6.0 * U.c[t + 1];
            au += U.c[t]; au += U.up[t]; au += ul; au += ur; au += U.dn[t]; au += U.c[t + 2];
            double be = bv[t];
            if (P.c[t]) be -= U.c[t];
            if (P.up[t]) be -= U.up[t];
            if (pl) be -= ul;
            if (pr) be -= ur;
            if (P.dn[t]) be -= U.dn[t];
            if (P.c[t + 2]) be -= U.c[t + 2];
            const double r = bv[t] - au;
            dm = (float)(-r);
            v[0] += r * r;
            v[1] += be * be;
            v[2] += (double)dm * dm;
        }
        d[(size_t)(i0 + t) * sx + C.col] = dm;
    }
    finish_sums<3>(v, partial, ticket, out, fin, post);
}

// Solver::solve rows (fields3d.cpp:86-93); Dirichlet values into u
__global__ void k3_rhs(const uint8_t *__restrict__ mask, const double *__restrict__ voltage, double *rho, double *u,
                       size_t n, double scale)
{
    size_t m = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= n) return;
    const double r = rho[m];
    const bool d = dir3(mask[m]);
    const double b = d ? voltage[m] : r * -scale;
    rho[m] = b;
    if (d) u[m] = b;
}

// Neighbour masks of the 7-point levels: one byte per node replaces the
// seven Dirichlet flags a stencil update reads.  Bits 0-5: linked to the
// free neighbour -x, -y, -z, +z, +y, +x; kNbBlack: colour 1 of the
// red-black order; kNbSelf: the node itself is pinned.
constexpr uint8_t kNbSelf = 0x80, kNbBlack = 0x40;

// The CG direction and the operator in one launch: p' = z + beta p (first:
// p' = z), q = A' p' = 6 p' - sum over the neighbours (p' is 0 on Dirichlet
// nodes, as z is; q too) and out = p'.q.  Each node's p' is formed again at
// its neighbours from z and p (the same operations, so the same bits) and
// written to pn, not p, which other blocks are still reading.
template <int DI>
__global__ void __launch_bounds__(kRedBlock) k3_dir_apply_dot(Cols3 g, const uint8_t *__restrict__ nbm,
                                                             const float *__restrict__ z,
                                                             const float *__restrict__ p, float *__restrict__ pn,
                                                             float *__restrict__ q, const double *rz_new,
                                                             const double *rz_old, int first, double *partial,
                                                             unsigned int *ticket, double *out, int fin,
                                                             const int *stop)
{
    const int stopped_ = stop ? *stop : 0;  // read beside the operands
    const float beta = first ? 0.f : cg_beta(rz_new, rz_old);
    const Column3 C(g);
    const int i0 = blockIdx.z * DI;
    const size_t sx = (size_t)g.ny * g.nz;
    Reach3<float, DI> D;
    uint8_t nb[DI];
    if (first) D.read(C, g, i0, [&](size_t m) { return z[m]; });
    else D.read(C, g, i0, [&](size_t m) { return fmaf(beta, p[m], z[m]); });
#pragma unroll
    for (int t = 0; t < DI; t++) nb[t] = nbm[(size_t)min(i0 + t, g.nx - 1) * sx + C.col];
    if (stopped_) return;
    double v[1] = {0};
#pragma unroll
    for (int t = 0; t < DI; t++) {
        const float l = D.left(C, t), r = D.right(C, t), c = D.c[t + 1];
        if (!C.in || i0 + t >= g.nx) continue;
        const float y = nb[t] & kNbSelf ? 0.f : 6.f * c - D.c[t] - D.up[t] - l - r - D.dn[t] - D.c[t + 2];
        const size_t m = (size_t)(i0 + t) * sx + C.col;
        pn[m] = c;
        q[m] = y;
        v[0] += (double)c * y;
    }
    finish_sums<1>(v, partial, ticket, out, fin);
}

// ------------------------------------------------------------------ the V-cycle
// sum of the free neighbours' values at node m of an array with strides si,
// sj, 1 (in LDS tiles and in the coarse cycle's arrays)
template <class T>
__device__ __forceinline__ float links7(uint8_t nb, const T *x, int m, int si, int sj)
{
    float s = 0.f;
    if (nb & 1) s += x[m - si];
    if (nb & 2) s += x[m - sj];
    if (nb & 4) s += x[m - 1];
    if (nb & 8) s += x[m + 1];
    if (nb & 16) s += x[m + sj];
    if (nb & 32) s += x[m + si];
    return s;
}

// Smoothing is one red-black sweep down and one (in reverse) up, which lets
// each side of a level be one launch over LDS tiles:
//   down, from x = 0:  red x = b / d;  black x = (b + sum red) / d;
//     the residual is then 0 on the black nodes and sum of the black
//     neighbours on the red ones; restrict it
//   up:  red x = b / d + P x_c  (the descent's red values are formed again,
//     so the descent stores nothing but the coarse right-hand side, and its
//     black values are not needed);  black x = (b + sum red) / d;
//     red x = (b + sum black) / d
// Two sweeps a side converge in 0.7 times the iterations but take 11
// launches a level instead of 2; the half sweeps ran at about 7.7 us each on
// 128^3 (every one reads and writes the level) and at the 2.5 us of an empty
// launch on small grids.
//
// A block holds a tile of TI x TJ x TK fine nodes with its halo in LDS, red
// and black nodes in arrays of their own (a half sweep then reads
// consecutive words): 3 nodes below and 2 above going down (black needs red
// one ring out, the residual black, the restriction the residual), 2 on both
// sides going up.  A thread keeps its place (j, k) in the tile's plane and
// steps through the planes, so that the index arithmetic is done once (it
// bound a version that divided a linear index at every node: 38 us a side
// at 128^3).  Tiles of 8 x 8 x 64 with 512 threads reload 2.9 times their
// nodes through L2 and fill the GPU from 2^20 nodes on; smaller levels are
// bound by latency and take 4 x 8 x 32 with 256 threads, several times the
// blocks.
//
// FINEST: the links of the finest level are those to free neighbours, so
// its sums need no masks where pinned nodes hold 0; the diagonal is 6.
template <int TI, int TJ, int TK, int LO, int HI>
struct Tile3 {
    static constexpr int SI = TI + LO + HI, SJ = TJ + LO + HI, SK = TK + LO + HI;
    static constexpr int HK = (SK + 1) / 2;  // nodes of a colour in a row
    static constexpr int PH = SJ * HK;       // and in a plane
    static constexpr int N = SI * PH;
};

// the sum over the links of the node at half-row index h of the other
// colour's array x; s = e & 1 of its position e = 2 (h % HK) + s.  All six
// are read and the unlinked ones dropped: no branch waits for the mask.
template <int HK, int PH, bool FINEST>
__device__ __forceinline__ float links_half(const float *x, int h, int s, uint8_t nb)
{
    const float q[6] = {x[h - PH], x[h - HK], x[h - 1 + s], x[h + s], x[h + HK], x[h + PH]};
    if (FINEST) return ((q[0] + q[5]) + (q[1] + q[4])) + (q[2] + q[3]);
    float v = 0.f;
#pragma unroll
    for (int l = 0; l < 6; l++) v += nb >> l & 1 ? q[l] : 0.f;
    return v;
}

// The tile's masks and right-hand sides from memory: red nodes get b / d,
// black ones b, pinned ones and those outside the grid 0.  A thread's
// column of nodes is read whole before any is stored (clamped addresses,
// so that no load waits behind a branch).
template <class G, int THREADS, bool FINEST>
__device__ __forceinline__ void tile3_load(const uint8_t *nbm, const float *di, const float *b, int nx, int ny, int nz,
                                           int i0, int j0, int k0, float *sr, float *sk, float *sdr, float *sdk,
                                           uint8_t *nr, uint8_t *nk)
{
    const int par0 = (i0 + j0 + k0) & 1;  // colour of the held corner
#pragma unroll
    for (int r = 0; r < (G::SJ * G::SK + THREADS - 1) / THREADS; r++) {
        const int p = threadIdx.x + r * THREADS, c = p / G::SK, e = p % G::SK;
        if (p >= G::SJ * G::SK) break;
        const int j = j0 + c, k = k0 + e;
        const bool in = (unsigned)j < (unsigned)ny && (unsigned)k < (unsigned)nz;
        const int m0 = min(max(j, 0), ny - 1) * nz + min(max(k, 0), nz - 1), h0 = c * G::HK + (e >> 1);
        uint8_t nb[G::SI];
        float v[G::SI], d[FINEST ? 1 : G::SI];
#pragma unroll
        for (int a = 0; a < G::SI; a++) {
            const size_t m = (size_t)min(max(i0 + a, 0), nx - 1) * ny * nz + m0;
            nb[a] = nbm[m];
            v[a] = b[m];
            if (!FINEST) d[a] = di[m];
        }
#pragma unroll
        for (int a = 0; a < G::SI; a++) {
            const uint8_t q = in && (unsigned)(i0 + a) < (unsigned)nx ? nb[a] : kNbSelf;
            const int h = a * G::PH + h0;
            const bool black = (par0 + a + c + e) & 1;
            float w = v[a];
            if (!black) w *= FINEST ? 1.f / 6.f : d[a];
            if (q & kNbSelf) w = 0.f;
            (black ? sk : sr)[h] = w;
            (black ? nk : nr)[h] = q;
            if (!FINEST) (black ? sdk : sdr)[h] = d[a];
        }
    }
}

// black = (b + sum red) / d one ring inside the tile.  The rows' ends (e
// outside the ring) are computed from whatever lies beside them and not used.
template <class G, int THREADS, bool FINEST>
__device__ __forceinline__ void tile3_black(int par0, const float *sr, float *sk, const float *sdk, const uint8_t *nk)
{
#pragma unroll
    for (int r = 0; r < (G::PH + THREADS - 1) / THREADS; r++) {
        const int p = threadIdx.x + r * THREADS, c = p / G::HK;
        if (c < 1 || c > G::SJ - 2) continue;
#pragma unroll
        for (int a = 1; a < G::SI - 1; a++) {
            const int h = a * G::PH + p;
            const uint8_t nb = nk[h];
            const float v = sk[h] + links_half<G::HK, G::PH, FINEST>(sr, h, (par0 + a + c + 1) & 1, nb);
            sk[h] = nb & kNbSelf ? 0.f : v * (FINEST ? 1.f / 6.f : sdk[h]);
        }
    }
}

template <int TI, int TJ, int TK, int THREADS, bool FINEST>
__global__ void __launch_bounds__(THREADS) k3_down(const uint8_t *nbm, const float *di, const float *b, int nx, int ny,
                                                   int nz, float *bc, const uint8_t *nbmc, int cx, int cy, int cz,
                                                   const int *stop)
{
    using G = Tile3<TI, TJ, TK, 3, 2>;
    constexpr int HK = G::HK, PH = G::PH;
    __shared__ float sr[G::N], sk[G::N], sdr[FINEST ? 1 : G::N], sdk[FINEST ? 1 : G::N];
    __shared__ uint8_t nr[G::N], nk[G::N];
    const int stopped_ = stop ? *stop : 0;  // read beside the operands
    const int i0 = (int)blockIdx.z * TI - 3, j0 = (int)blockIdx.y * TJ - 3, k0 = (int)blockIdx.x * TK - 3;
    const int par0 = (i0 + j0 + k0) & 1;
    tile3_load<G, THREADS, FINEST>(nbm, di, b, nx, ny, nz, i0, j0, k0, sr, sk, sdr, sdk, nr, nk);
    if (stopped_) return;  // uniform
    __syncthreads();
    tile3_black<G, THREADS, FINEST>(par0, sr, sk, sdk, nk);
    __syncthreads();
    // the residual on the red nodes two rings inside, in their place
#pragma unroll
    for (int r = 0; r < (PH + THREADS - 1) / THREADS; r++) {
        const int p = threadIdx.x + r * THREADS, c = p / HK;
        if (c < 2 || c > G::SJ - 3) continue;
#pragma unroll
        for (int a = 2; a < G::SI - 2; a++) {
            const int h = a * PH + p;
            const uint8_t nb = nr[h];
            const float v = links_half<HK, PH, FINEST>(sk, h, (par0 + a + c) & 1, nb);
            sr[h] = nb & kNbSelf ? 0.f : v;
        }
    }
    __syncthreads();
    // P^T r / 2: of the 27 fine nodes around a coarse one 13 are red, the
    // node itself (weight 1) and the twelve two steps away (1/4 each);
    // pinned ones hold 0
    constexpr int CI = TI / 2, CJ = TJ / 2, CK = TK / 2;
#pragma unroll
    for (int t0 = 0; t0 < CI * CJ * CK; t0 += THREADS) {
        const int t = t0 + threadIdx.x, a = t / (CJ * CK), c = t / CK % CJ, e = t % CK;
        const int I = blockIdx.z * CI + a, J = blockIdx.y * CJ + c, K = blockIdx.x * CK + e;
        if (t >= CI * CJ * CK || I >= cx || J >= cy || K >= cz) continue;
        const size_t M = ((size_t)I * cy + J) * cz + K;
        const uint8_t nb = nbmc[M];
        // its fine node is at (3 + 2 a, 3 + 2 c, 3 + 2 e): half-row index
        // e + 1, odd; the red nodes beside it at +-1 are even: e + 1, e + 2
        const float *q = sr + ((3 + 2 * a) * G::SJ + 3 + 2 * c) * HK + 1 + e;
        const float v = (q[-PH - HK] + q[-PH + HK] + q[PH - HK] + q[PH + HK]) +
                        (q[-PH] + q[-PH + 1] + q[PH] + q[PH + 1]) + (q[-HK] + q[-HK + 1] + q[HK] + q[HK + 1]);
        bc[M] = nb & kNbSelf ? 0.f : 0.5f * fmaf(0.25f, v, q[0]);
    }
}

// DOT: out's product with b as well, dot = b.out (the CG's r.z)
template <int TI, int TJ, int TK, int THREADS, bool FINEST, bool DOT>
__global__ void __launch_bounds__(THREADS) k3_up(const uint8_t *nbm, const float *di, const float *b, int nx, int ny,
                                                 int nz, const float *xc, int cx, int cy, int cz, float *out,
                                                 double *partial, unsigned int *ticket, double *dot, int fin,
                                                 const int *stop)
{
    using G = Tile3<TI, TJ, TK, 2, 2>;
    constexpr int HK = G::HK, PH = G::PH;
    constexpr int QI = TI / 2 + 3, QJ = TJ / 2 + 3, QK = TK / 2 + 3;
    __shared__ float sr[G::N], sk[G::N], sdr[FINEST ? 1 : G::N], sdk[FINEST ? 1 : G::N], sc[QI * QJ * QK];
    __shared__ uint8_t nr[G::N], nk[G::N];
    const int stopped_ = stop ? *stop : 0;
    const int i0 = (int)blockIdx.z * TI - 2, j0 = (int)blockIdx.y * TJ - 2, k0 = (int)blockIdx.x * TK - 2;  // even
    // the coarse nodes the prolongation reads: from fine node i0 / 2 on
    constexpr int NQ = (QI * QJ * QK + THREADS - 1) / THREADS;
    float qv[NQ];
#pragma unroll
    for (int r = 0; r < NQ; r++) {
        const int t = threadIdx.x + r * THREADS;
        const int I = i0 / 2 + t / (QJ * QK), J = j0 / 2 + t / QK % QJ, K = k0 / 2 + t % QK;
        const bool in = (unsigned)I < (unsigned)cx && (unsigned)J < (unsigned)cy && (unsigned)K < (unsigned)cz;
        const float v = xc[((size_t)min(max(I, 0), cx - 1) * cy + min(max(J, 0), cy - 1)) * cz + min(max(K, 0), cz - 1)];
        qv[r] = in ? v : 0.f;
    }
    tile3_load<G, THREADS, FINEST>(nbm, di, b, nx, ny, nz, i0, j0, k0, sr, sk, sdr, sdk, nr, nk);
#pragma unroll
    for (int r = 0; r < NQ; r++)
        if (threadIdx.x + r * THREADS < QI * QJ * QK) sc[threadIdx.x + r * THREADS] = qv[r];
    if (stopped_) return;  // uniform
    __syncthreads();
    // red += P x_c: a red node has no odd coordinate or two, and takes one
    // coarse node or the mean of four
#pragma unroll
    for (int r = 0; r < (PH + THREADS - 1) / THREADS; r++) {
        const int p = threadIdx.x + r * THREADS, c = p / HK, kk = p % HK;
        if (p >= PH) break;
        const float *qc = sc + (c >> 1) * QK + kk;
        const int oj = c & 1;
#pragma unroll
        for (int a = 0; a < G::SI; a++) {
            const int h = a * PH + p, s = (a + c) & 1, oi = a & 1;
            const float *q = qc + (a >> 1) * (QJ * QK);
            const int s1 = oi ? QJ * QK : oj ? QK : 0, s2 = s ? 1 : oj ? QK : 0;  // 0, 0: the node itself four times
            const float v = 0.25f * ((q[0] + q[s1]) + (q[s2] + q[s1 + s2]));
            sr[h] = nr[h] & kNbSelf ? 0.f : sr[h] + v;
        }
    }
    __syncthreads();
    tile3_black<G, THREADS, FINEST>(0, sr, sk, sdk, nk);
    __syncthreads();
    double acc[1] = {0};
    static_assert(TJ * TK % THREADS == 0 || THREADS % (TJ * TK) == 0, "whole planes of threads");
    constexpr int ROWS = THREADS > TJ * TK ? THREADS / (TJ * TK) : 1;  // planes at once
    constexpr int REP = THREADS < TJ * TK ? TJ * TK / THREADS : 1;
#pragma unroll
    for (int r = 0; r < REP; r++) {
        const int p = (threadIdx.x + r * THREADS) % (TJ * TK), c = 2 + p / TK, e = 2 + p % TK;
        const int j = j0 + c, k = k0 + e;
        if (j >= ny || k >= nz) continue;
        const int m0 = j * nz + k, h0 = c * HK + (e >> 1), a0 = 2 + threadIdx.x / (TJ * TK);
        float bm[TI / ROWS];
#pragma unroll
        for (int t = 0; t < TI / ROWS; t++) bm[t] = b[(size_t)min(i0 + a0 + t * ROWS, nx - 1) * ny * nz + m0];
#pragma unroll
        for (int t = 0; t < TI / ROWS; t++) {
            const int a = a0 + t * ROWS, i = i0 + a, h = a * PH + h0;
            const bool black = (a + c + e) & 1;
            const uint8_t nb = (black ? nk : nr)[h];
            const float w = bm[t] + links_half<HK, PH, FINEST>(sk, h, e & 1, nb);
            float x = w * (FINEST ? 1.f / 6.f : sdr[h]);
            if (black) x = sk[h];
            if (nb & kNbSelf) x = 0.f;
            if (i < nx) {
                out[(size_t)i * ny * nz + m0] = x;
                if (DOT) acc[0] += (double)bm[t] * x;
            }
        }
    }
    if constexpr (DOT) finish_sums<1, THREADS>(acc, partial, ticket, dot, fin);
}

// x = A^-1 b on the coarsest level, with the inverse held for all its nodes
// (rows and columns of pinned ones 0): a wavefront a row.  On 9^3 nodes the
// 2 MB are read once from L2 by 183 blocks; one workgroup running the levels
// below 17^3 in its LDS took 15-17 us.
__global__ void __launch_bounds__(256) k3_dense(const float *inv, const float *b, float *x, int n, const int *stop)
{
    const int stopped_ = stop ? *stop : 0;
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= n) return;
    float s = 0.f;
#pragma unroll 4
    for (int c = lane; c < n; c += 64) s = fmaf(inv[(size_t)row * n + c], b[c], s);
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (lane == 0 && !stopped_) x[row] = s;
}

// Half sweep of colour on a coarsest level that is too large for a dense
// solve (a side below 5 nodes) and for k3_sweeps: the finest level of a thin
// grid (di null: its diagonal is 6) or a coarse one.  Threads cover only the
// nodes of the colour: thread (kk, j, i) updates k = 2 kk + parity, blocks of
// 64 x 4 (kk, j).
constexpr int kRbgsX = 64, kRbgsY = 4;
__global__ void __launch_bounds__(kRbgsX * kRbgsY) k3_rbgs(const uint8_t *nbm, const float *di, float *x,
                                                           const float *b, int nx, int ny, int nz, int colour,
                                                           const int *stop)
{
    if (stopped(stop)) return;
    const int i = blockIdx.z, j = blockIdx.y * kRbgsY + threadIdx.y;
    const int k = 2 * (blockIdx.x * kRbgsX + threadIdx.x) + ((i + j + colour) & 1);
    if (i >= nx || j >= ny || k >= nz) return;
    const int m = (i * ny + j) * nz + k;
    const uint8_t nb = nbm[m];
    if (!(nb & kNbSelf)) x[m] = (b[m] + links7(nb, x, m, ny * nz, nz)) * (di ? di[m] : 1.f / 6.f);
}

__global__ void k3_zero(float *x, size_t n, const int *stop)
{
    if (stopped(stop)) return;
    size_t m = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (m < n) x[m] = 0.f;
}

// A coarsest level too large for a dense solve (a thin grid's): kCoarseSweeps
// symmetric red-black sweeps from zero, half of them in reverse order, by one
// workgroup with barriers between the half sweeps.  A thread keeps its nodes'
// right-hand sides, diagonals and links in registers and x is in LDS: with
// all of them in memory a solve of 90 x 90 x 5 nodes took 6.0 ms, of 5 x 90 x
// 90 3.0 (now 2.0 and 1.1).  Larger levels take a launch a half sweep
// (k3_rbgs), 80 of about 2.5 us: a solve of 90 x 90 x 6 nodes, whose 8464
// coarse nodes one workgroup swept in memory, 8.5 ms, now 4.0; of 200 x 200 x
// 5 27.2 and 5.4.
constexpr int kMaxLevels3 = 16;
constexpr int kSweepsPer = 8;
constexpr size_t kSweepsNodes = (size_t)kSweepsPer * kCoarseThreads;
__global__ void __launch_bounds__(kCoarseThreads) k3_sweeps(const uint8_t *nbm, const float *di, const float *b,
                                                            float *x, int ny, int nz, int n, int sweeps,
                                                            const int *stop)
{
    if (stopped(stop)) return;
    __shared__ float sx[kSweepsNodes];
    uint8_t nb[kSweepsPer];
    float bv[kSweepsPer], d[kSweepsPer];
#pragma unroll
    for (int q = 0; q < kSweepsPer; q++) {
        const int m = threadIdx.x + q * kCoarseThreads, at = min(m, n - 1);
        nb[q] = m < n ? nbm[at] : kNbSelf;
        bv[q] = b[at];
        d[q] = di[at];
        sx[m] = 0.f;
    }
    __syncthreads();
    for (int h = 0; h < 2 * sweeps; h++) {
        const uint8_t colour = (h & 1) == (h < sweeps ? 0 : 1) ? 0 : kNbBlack;
#pragma unroll
        for (int q = 0; q < kSweepsPer; q++) {
            const int m = threadIdx.x + q * kCoarseThreads;
            if ((nb[q] & (kNbSelf | kNbBlack)) == colour) sx[m] = (bv[q] + links7(nb[q], sx, m, ny * nz, nz)) * d[q];
        }
        __syncthreads();
    }
#pragma unroll
    for (int q = 0; q < kSweepsPer; q++) {
        const int m = threadIdx.x + q * kCoarseThreads;
        if (m < n) x[m] = sx[m];
    }
}

// ------------------------------------------------------------------ point kernels (FP64)
struct Grid3 {
    int nx, ny, nz;
    double idx, idy, idz, hx, hy, hz;  // h = (n-1) d idx: the clamp limits of grad
};

__device__ __forceinline__ double d3at(const double *d, const Grid3 &g, int i, int j, int k)
{
    return d[((size_t)i * g.ny + j) * g.nz + k];
}

// Field3D::interpolate (Field3D.hpp:68-96); out of range gives NaN
__global__ void k_interp3d(const double *d, Grid3 g, const double *xs, const double *ys, const double *zs,
                           int64_t n, double *out)
{
    int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    double x = xs[p], y = ys[p], z = zs[p];
    const double X = x * g.idx, Y = y * g.idy, Z = z * g.idz;
    if (!(X >= 0 && X < g.nx - 1.0 && Y >= 0 && Y < g.ny - 1.0 && Z >= 0 && Z < g.nz - 1.0)) {
        out[p] = NAN;
        return;
    }
    const int i = (int)X, j = (int)Y, k = (int)Z;
    double u = x * g.idx - i, v = y * g.idy - j, w = z * g.idz - k;
    double r = 0;
    r += (1 - u) * (1 - v) * (1 - w) * d3at(d, g, i, j, k);
    r += u * (1 - v) * (1 - w) * d3at(d, g, i + 1, j, k);
    r += (1 - u) * v * (1 - w) * d3at(d, g, i, j + 1, k);
    r += u * v * (1 - w) * d3at(d, g, i + 1, j + 1, k);
    r += (1 - u) * (1 - v) * w * d3at(d, g, i, j, k + 1);
    r += u * (1 - v) * w * d3at(d, g, i + 1, j, k + 1);
    r += (1 - u) * v * w * d3at(d, g, i, j + 1, k + 1);
    r += u * v * w * d3at(d, g, i + 1, j + 1, k + 1);
    out[p] = r;
}

// Field3D::grad_component (Field3D.hpp:112-141), FP64: clamped half a cell
// inside along the differenced axis, staggered differences, trilinear weights
__device__ double grad3_component(const double *d, const Grid3 &g, double x, double y, double z, int ex, int ey,
                                  int ez)
{
    double X = fmin(fmax(x * g.idx, 0.5 * ex), g.hx - 0.5 * ex) + 0.5 * ex;
    double Y = fmin(fmax(y * g.idy, 0.5 * ey), g.hy - 0.5 * ey) + 0.5 * ey;
    double Z = fmin(fmax(z * g.idz, 0.5 * ez), g.hz - 0.5 * ez) + 0.5 * ez;
    int i = min((int)X, g.nx - 2), j = min((int)Y, g.ny - 2), k = min((int)Z, g.nz - 2);
    double u = X - i, v = Y - j, w = Z - k;
    double gg[8];
    for (int c = 0; c < 8; c++) {
        int a = i + (c & 1), b = j + ((c >> 1) & 1), e = k + ((c >> 2) & 1);
        gg[c] = d3at(d, g, a, b, e) - d3at(d, g, a - ex, b - ey, e - ez);
    }
    double r = (1 - u) * (1 - v) * (1 - w) * gg[0] + u * (1 - v) * (1 - w) * gg[1] +
               (1 - u) * v * (1 - w) * gg[2] + u * v * (1 - w) * gg[3] + (1 - u) * (1 - v) * w * gg[4] +
               u * (1 - v) * w * gg[5] + (1 - u) * v * w * gg[6] + u * v * w * gg[7];
    return r * (g.idx * ex + g.idy * ey + g.idz * ez);
}

__global__ void k_grad3d(const double *d, Grid3 g, const double *xs, const double *ys, const double *zs,
                         int64_t n, double *gx, double *gy, double *gz)
{
    int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    gx[p] = grad3_component(d, g, xs[p], ys[p], zs[p], 1, 0, 0);
    gy[p] = grad3_component(d, g, xs[p], ys[p], zs[p], 0, 1, 0);
    gz[p] = grad3_component(d, g, xs[p], ys[p], zs[p], 0, 0, 1);
}

// ------------------------------------------------------------------ the 3D pass
struct PushArgs3 {
    float *x, *y, *z, *vx, *vy, *vz;
    int64_t n;
    const float *tx, *ty, *tz;
    const uint8_t *cellfree;
    Grid3 g;
    float bx1, by1, bz1;           // largest floats <= x_max, y_max, z_max
    double xper, yper, zper;
    float qmdt2, tx_, ty_, tz_, sx, sy, sz, dt;
    int rotate, push, boundary, periodic;
    uint64_t trial_thr;
    uint64_t seed;
    uint32_t stream;
    uint64_t step;
    const McDev *mcc;
    uint32_t *cq;
    unsigned long long *cq_len;
    unsigned long long *acc;
    int rec;                       // acc holds cell records (untiled deposit, see deposit_buffer)
    unsigned long long *counters;
};

// one E component through the FP32 difference table: the clamp and the
// cell index in FP64 on the FP32 position, weights FP32
__device__ __forceinline__ float gather3_component(const float *t, const Grid3 &g, double x, double y, double z,
                                                   int ex, int ey, int ez)
{
    double X = fmin(fmax(x * g.idx, 0.5 * ex), g.hx - 0.5 * ex) + 0.5 * ex;
    double Y = fmin(fmax(y * g.idy, 0.5 * ey), g.hy - 0.5 * ey) + 0.5 * ey;
    double Z = fmin(fmax(z * g.idz, 0.5 * ez), g.hz - 0.5 * ez) + 0.5 * ez;
    int i = min(max((int)X, 0), g.nx - 2), j = min(max((int)Y, 0), g.ny - 2), k = min(max((int)Z, 0), g.nz - 2);
    const float u = (float)(X - i), v = (float)(Y - j), w = (float)(Z - k);
    const size_t sx = (size_t)g.ny * g.nz;
    const float *c = t + ((size_t)i * g.ny + j) * g.nz + k;
    float a0 = c[0], a1 = c[sx], a2 = c[g.nz], a3 = c[sx + g.nz];
    float a4 = c[1], a5 = c[sx + 1], a6 = c[g.nz + 1], a7 = c[sx + g.nz + 1];
    float lo = (1.f - v) * ((1.f - u) * a0 + u * a1) + v * ((1.f - u) * a2 + u * a3);
    float hi = (1.f - v) * ((1.f - u) * a4 + u * a5) + v * ((1.f - u) * a6 + u * a7);
    return (1.f - w) * lo + w * hi;
}

// eight CIC weights in 2^-31 fixed point, corrected on the largest so a
// particle deposits exactly 2^31 (order-independent integer sums)
__device__ __forceinline__ bool cic3(double X, double Y, double Z, const Grid3 &g, int &cell, uint32_t w[8])
{
    // range in FP64 before any conversion: cells [0, n-2] on every axis
    if (!(X >= 0.0 && X < g.nx - 1.0 && Y >= 0.0 && Y < g.ny - 1.0 && Z >= 0.0 && Z < g.nz - 1.0)) return false;
    const int i = (int)X, j = (int)Y, k = (int)Z;
    // offsets and their complements from FP64, each rounded once (see the
    // 2D cic_weights)
    const double du = X - i, dv = Y - j, dw = Z - k;
    const float S = 2147483648.0f;
    const float a[2] = {(float)(1.0 - du), (float)du}, b[2] = {(float)(1.0 - dv), (float)dv},
                c[2] = {(float)(1.0 - dw), (float)dw};
    uint32_t s = 0;
#pragma unroll
    for (int q = 0; q < 8; q++) {
        w[q] = __float2uint_rn(a[q & 1] * b[(q >> 1) & 1] * c[q >> 2] * S);
        s += w[q];
    }
    // the first largest weight takes the rounding's remainder (selects, not
    // an index: a computed index would put w in memory)
    int km = 0;
    uint32_t wm = w[0];
#pragma unroll
    for (int q = 1; q < 8; q++)
        if (w[q] > wm) { km = q; wm = w[q]; }
#pragma unroll
    for (int q = 0; q < 8; q++)
        if (q == km) w[q] += 0x80000000u - s;
    cell = (int)(((size_t)i * g.ny + j) * g.nz + k);
    return true;
}

// The deposits of a wavefront's lanes in memory: cell = its lower corner's
// node (-1: none), w8 its corners' weights.  They pass through LDS (stage:
// kStage3 words of the wavefront's own) so that round r serves lanes 8 r ..
// 8 r + 7, eight lanes adding the corners of one particle: an instruction's
// lanes then fall on 8 records of 64 bytes (or 8 x 4 node rows), not 64 x 8
// nodes.  In cell order (many lanes of equal cells) the lanes' weights are
// summed first.  All 64 lanes must call it together.
constexpr int kStage3 = 64 * 9;
__device__ __forceinline__ void wave_deposit3(int cell, const uint32_t w8[8], const Grid3 &g, unsigned long long *acc,
                                              int rec, uint32_t *stage)
{
    const int lane = __lane_id();
    const size_t sx = (size_t)g.ny * g.nz;
    auto corner = [&](int q) { return ((q & 1) ? sx : 0) + (((q >> 1) & 1) ? (size_t)g.nz : 0) + (q >> 2); };
    if (cells_repeat(cell)) {  // uniform
        unsigned long long s[8];
#pragma unroll
        for (int q = 0; q < 8; q++) s[q] = cell >= 0 ? w8[q] : 0ull;
        if (segment_sums<8>(cell, s)) {
#pragma unroll
            for (int q = 0; q < 8; q++)
                if (s[q]) atomicAdd(acc + (rec ? (size_t)cell * 8 + q : (size_t)cell + corner(q)), s[q]);
        }
        return;
    }
#pragma unroll
    for (int q = 0; q < 8; q++) stage[lane * 9 + q] = cell >= 0 ? w8[q] : 0u;
    stage[lane * 9 + 8] = (uint32_t)cell;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int q = lane & 7;
    const size_t off = rec ? (size_t)q : corner(q);
    const int mul = rec ? 8 : 1;
#pragma unroll
    for (int r = 0; r < 8; r++) {
        const int src = 8 * r + (lane >> 3);
        const int c = (int)stage[src * 9 + 8];
        const uint32_t v = stage[src * 9 + q];
        if (c >= 0 && v) atomicAdd(acc + ((size_t)c * mul + off), (unsigned long long)v);
    }
}

// rho += charge * (sum of the records of the 8 cells around the node) *
// 2^-31 (launched on planes3)
__global__ void __launch_bounds__(256) k3_flush_rec(const unsigned long long *rec, double *rho, double charge, int nx,
                                                    int ny, int nz)
{
    const int k = blockIdx.x * 64 + threadIdx.x;
    if (k >= nz) return;
    const size_t sx = (size_t)ny * nz;
    for (int i = blockIdx.z; i < nx; i += gridDim.z)
        for (int j = blockIdx.y * 4 + threadIdx.y; j < ny; j += gridDim.y * 4) {
            const size_t m = (size_t)i * sx + (size_t)j * nz + k;
            unsigned long long v = 0;
#pragma unroll
            for (int q = 0; q < 8; q++) {
                const int a = q & 1, b = (q >> 1) & 1, c = q >> 2;
                if (i >= a && j >= b && k >= c) v += rec[8 * (m - a * sx - (size_t)b * nz - c) + q];
            }
            if (v) rho[m] += charge * ((double)(long long)v * kInvFix);
        }
}

// mod (mymath.cpp:62-67)
__device__ __forceinline__ double mod3(double x, double y)
{
    if (x >= 0.0 && x <= y) return x;
    return x - y * (int)(x / y) + (x < 0 ? y : 0);
}

// 3D sort tiles: 4 x 4 x 4 cells, key = tile << 6 | cell in tile; the deposit
// window of a tile spans its cells plus a halo of 2 cells: 9 nodes per axis
constexpr int kTile3 = 4, kHalo3 = 2, kWin3 = kTile3 + 1 + 2 * kHalo3, kWinN3 = kWin3 * kWin3 * kWin3;

struct Step3 {
    bool removed = false, coll = false, nan_pos = false, bad = false;
    int cell = -1;        // deposit cell (lower corner node), -1: none
    int ci = 0, cj = 0, ck = 0;
    uint32_t w8[8];
};

// Species<CARTESIAN3D>::advance for the particle in slot p (species3d.cpp:10-92):
// gather, Boris, drift, MCC trial, box / mod, is_free, deposit weights
template <bool DEPOSIT, bool MCC>
__device__ __forceinline__ void step3(const PushArgs3 &a, int64_t p, Step3 &o)
{
    float x = a.x[p];
    if (is_dead(x)) return;
    float y = a.y[p], z = a.z[p];
    float vx = a.vx[p], vy = a.vy[p], vz = a.vz[p];
    if (a.push) {
        // E = -grad u (ElMag3D::E, fields3d.hpp:91-97)
        const double xd = x, yd = y, zd = z;
        const float ex = -gather3_component(a.tx, a.g, xd, yd, zd, 1, 0, 0);
        const float ey = -gather3_component(a.ty, a.g, xd, yd, zd, 0, 1, 0);
        const float ez = -gather3_component(a.tz, a.g, xd, yd, zd, 0, 0, 1);
        // species3d.cpp:24-61
        vx = fmaf(ex, a.qmdt2, vx);
        vy = fmaf(ey, a.qmdt2, vy);
        vz = fmaf(ez, a.qmdt2, vz);
        if (a.rotate) {
            float vpx = vx - vy * a.tz_ + vz * a.ty_;
            float vpy = vy - vz * a.tx_ + vx * a.tz_;
            float vpz = vz - vx * a.ty_ + vy * a.tx_;
            vx = vx - vpy * a.sz + vpz * a.sy;
            vy = vy - vpz * a.sx + vpx * a.sz;
            vz = vz - vpx * a.sy + vpy * a.sx;
        }
        vx = fmaf(ex, a.qmdt2, vx);
        vy = fmaf(ey, a.qmdt2, vy);
        vz = fmaf(ez, a.qmdt2, vz);
        x = fmaf(vx, a.dt, x);
        y = fmaf(vy, a.dt, y);
        z = fmaf(vz, a.dt, z);
        // MCC trial (species3d.cpp:64-67); the velocity change is applied after the pass
        if (MCC) {
            uint32_t c0 = (uint32_t)(p >> 2), c1 = (uint32_t)a.step, c2 = 0u;
            uint32_t c3 = (kPurposeTrial << 24) | ((uint32_t)(a.step >> 32) & 0xFFFFFFu);
            philox4x32_10(c0, c1, c2, c3, (uint32_t)a.seed, (uint32_t)(a.seed >> 32) ^ a.stream);
            const int q = (int)(p & 3);
            const uint32_t tw = q == 0 ? c0 : q == 1 ? c1 : q == 2 ? c2 : c3;
            if ((uint64_t)tw < a.trial_thr) {
                unsigned long long at = atomicAdd(a.cq_len, 1ull);
                a.cq[at] = (uint32_t)p;
                o.coll = true;
            }
        }
    }
    if (a.boundary) {
        // species3d.cpp:69-85
        if (x > a.bx1 || x < 0.f || y > a.by1 || y < 0.f || z > a.bz1 || z < 0.f || x != x || y != y || z != z) {
            if (x != x || y != y || z != z) { o.removed = true; o.nan_pos = true; }
            else if (!a.periodic) o.removed = true;
            else {
                x = (float)mod3(x, a.xper);
                y = (float)mod3(y, a.yper);
                z = (float)mod3(z, a.zper);
            }
        }
        if (!o.removed) {
            // Geometry::is_free (fields3d.hpp:48-55)
            const double X = (double)x * a.g.idx, Y = (double)y * a.g.idy, Z = (double)z * a.g.idz;
            bool fr = false;
            if (X >= 0.0 && X < a.g.nx - 1.0 && Y >= 0.0 && Y < a.g.ny - 1.0 && Z >= 0.0 && Z < a.g.nz - 1.0)
                fr = a.cellfree[((size_t)(int)X * a.g.ny + (int)Y) * a.g.nz + (int)Z] != 0;
            o.removed = !fr;
        }
    }
    if (DEPOSIT && !o.removed) {
        const double X = (double)x * a.g.idx, Y = (double)y * a.g.idy, Z = (double)z * a.g.idz;
        if (cic3(X, Y, Z, a.g, o.cell, o.w8)) {
            o.ci = (int)X; o.cj = (int)Y; o.ck = (int)Z;
        } else {
            o.cell = -1;
            o.bad = true;
        }
    }
    if (o.removed) {
        a.x[p] = dead_value();
    } else {
        a.x[p] = x; a.y[p] = y; a.z[p] = z;
        a.vx[p] = vx; a.vy[p] = vy; a.vz[p] = vz;
    }
}

__device__ __forceinline__ void deposit8_global(unsigned long long *acc, const Grid3 &g, int cell,
                                                const uint32_t w8[8])
{
    const size_t sx = (size_t)g.ny * g.nz;
#pragma unroll
    for (int q = 0; q < 8; q++) {
        const size_t m = (size_t)cell + ((q & 1) ? sx : 0) + (((q >> 1) & 1) ? (size_t)g.nz : 0) + (q >> 2);
        if (w8[q]) atomicAdd(acc + m, (unsigned long long)w8[q]);
    }
}

// untiled: one particle per thread, deposit summed across the wavefront
template <bool DEPOSIT, bool MCC>
__global__ void __launch_bounds__(256) k_advance3d(PushArgs3 a)
{
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    __shared__ uint32_t stage[DEPOSIT ? 4 * kStage3 : 1];
    Step3 o;
    if (p < a.n) step3<DEPOSIT, MCC>(a, p, o);
    if (DEPOSIT) wave_deposit3(o.cell, o.w8, a.g, a.acc, a.rec, stage + (threadIdx.x >> 6) * kStage3);
    wave_count(&a.counters[CNT_REMOVED], o.removed);
    if (MCC) wave_count(&a.counters[CNT_COLL], o.coll);
    if (__ballot(o.nan_pos) && __lane_id() == 0) raise_flag(a.counters, M2D_FLAG_NAN);
    if (__ballot(o.bad) && __lane_id() == 0) raise_flag(a.counters, M2D_FLAG_OUT_OF_RANGE);
}

// tiled (store sorted by m2d_sort_3d): block b runs chunk sched[b] of one
// sort tile and sums its deposits in an LDS window of the tile + halo, then
// adds the window's non-zero nodes to the 64-bit grid with atomics (integer
// sums: the grid does not depend on their order); deposits that leave the
// window go to the grid directly.  Six waves per SIMD (at most 80 VGPRs):
// the pass waits on its 24 gathers, and 4 waves (111 VGPRs unconstrained)
// ran it 12% slower.
template <bool MCC>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(6))) k_advance3d_tiled(PushArgs3 a, const int4 *sched,
                                                         const unsigned int *n_chunks, int nty3, int ntz3)
{
    __shared__ unsigned long long win[kWinN3];
    // plain block order: grouping chunks per XCD (contiguous ranges or runs
    // of 8 to 128 chunks) made this pass 3-27% slower
    const unsigned ch = blockIdx.x;
    if (ch >= *n_chunks) return;  // uniform, before any barrier
    const int4 s = sched[ch];
    const int t = s.x;
    const int wi0 = (t / (nty3 * ntz3)) * kTile3 - kHalo3, wj0 = ((t / ntz3) % nty3) * kTile3 - kHalo3,
              wk0 = (t % ntz3) * kTile3 - kHalo3;
    for (int k = threadIdx.x; k < kWinN3; k += 256) win[k] = 0ull;
    __syncthreads();
    bool nan_any = false, bad_any = false;
    int n_removed = 0, n_coll = 0, n_spill = 0;
    for (int64_t p = s.y + threadIdx.x; p < s.z; p += 256) {
        Step3 o;
        step3<true, MCC>(a, p, o);
        n_removed += o.removed;
        n_coll += o.coll;
        nan_any |= o.nan_pos;
        bad_any |= o.bad;
        if (o.cell >= 0) {
            const int da = o.ci - wi0, db = o.cj - wj0, dc = o.ck - wk0;
            if ((unsigned)da < (unsigned)(kWin3 - 1) && (unsigned)db < (unsigned)(kWin3 - 1) &&
                (unsigned)dc < (unsigned)(kWin3 - 1)) {
                unsigned long long *w = win + (da * kWin3 + db) * kWin3 + dc;
#pragma unroll
                for (int q = 0; q < 8; q++) {
                    const int off = ((q & 1) ? kWin3 * kWin3 : 0) + (((q >> 1) & 1) ? kWin3 : 0) + (q >> 2);
                    atomicAdd(w + off, (unsigned long long)o.w8[q]);  // a zero weight adds 0: no branch
                }
            } else {
                deposit8_global(a.acc, a.g, o.cell, o.w8);
                n_spill++;
            }
        }
    }
    __syncthreads();
    for (int k = threadIdx.x; k < kWinN3; k += 256) {
        const unsigned long long v = win[k];
        if (!v) continue;
        // window node (da, db, dc) of the tile's window: only nodes of the
        // grid receive deposits, so a non-zero entry lies on the grid
        const int i = wi0 + k / (kWin3 * kWin3), j = wj0 + (k / kWin3) % kWin3, l = wk0 + k % kWin3;
        if ((unsigned)i < (unsigned)a.g.nx && (unsigned)j < (unsigned)a.g.ny && (unsigned)l < (unsigned)a.g.nz)
            atomicAdd(a.acc + ((size_t)i * a.g.ny + j) * a.g.nz + l, v);
    }
    int sum = n_removed;
    for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
    if (__lane_id() == 0 && sum) atomicAdd(&a.counters[CNT_REMOVED], (unsigned long long)sum);
    int sp = n_spill;
    for (int off = 32; off > 0; off >>= 1) sp += __shfl_xor(sp, off);
    if (__lane_id() == 0 && sp) atomicAdd(&a.counters[CNT_SPILL], (unsigned long long)sp);
    if (MCC) {
        int c = n_coll;
        for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off);
        if (__lane_id() == 0 && c) atomicAdd(&a.counters[CNT_COLL], (unsigned long long)c);
    }
    if (__ballot(nan_any) && __lane_id() == 0) raise_flag(a.counters, M2D_FLAG_NAN);
    if (__ballot(bad_any) && __lane_id() == 0) raise_flag(a.counters, M2D_FLAG_OUT_OF_RANGE);
}

// BaseSpecies::scatter for the queued slots (velocity only, after the pass)
__global__ void __launch_bounds__(256) k_scatter3d(PushArgs3 a, unsigned long long *next_len)
{
    const unsigned long long len = *a.cq_len;
    const unsigned long long start = (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x;
    const unsigned long long stride = (unsigned long long)gridDim.x * blockDim.x;
    if (start == 0) *next_len = 0ull;
    for (unsigned long long k = start; k < len; k += stride) {
        const uint32_t p = a.cq[k];
        if (is_dead(a.x[p])) continue;
        float vx = a.vx[p], vy = a.vy[p], vz = a.vz[p];
        Rng rg;
        rg.begin(a.seed, a.stream, p, a.step, kPurposeMcc);
        scatter(*a.mcc, rg, vx, vy, vz, a.counters);
        a.vx[p] = vx; a.vy[p] = vy; a.vz[p] = vz;
    }
}

// leapfrog start: rotation by -dt/2, then a backward half kick
__global__ void __launch_bounds__(256) k_advance_init3d(PushArgs3 a)
{
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= a.n) return;
    const float x = a.x[p];
    if (is_dead(x)) return;
    const float y = a.y[p], z = a.z[p];
    float vx = a.vx[p], vy = a.vy[p], vz = a.vz[p];
    const double xd = x, yd = y, zd = z;
    const float ex = -gather3_component(a.tx, a.g, xd, yd, zd, 1, 0, 0);
    const float ey = -gather3_component(a.ty, a.g, xd, yd, zd, 0, 1, 0);
    const float ez = -gather3_component(a.tz, a.g, xd, yd, zd, 0, 0, 1);
    if (a.rotate) {
        float vpx = vx - vy * a.tz_ + vz * a.ty_;
        float vpy = vy - vz * a.tx_ + vx * a.tz_;
        float vpz = vz - vx * a.ty_ + vy * a.tx_;
        vx = vx - vpy * a.sz + vpz * a.sy;
        vy = vy - vpz * a.sx + vpx * a.sz;
        vz = vz - vpx * a.sy + vpy * a.sx;
    }
    a.vx[p] = fmaf(ex, a.qmdt2, vx);
    a.vy[p] = fmaf(ey, a.qmdt2, vy);
    a.vz[p] = fmaf(ez, a.qmdt2, vz);
}

// Field3D::accumulate for every live particle
__global__ void __launch_bounds__(256) k_accumulate3d(const float *xs, const float *ys, const float *zs,
                                                      int64_t n, Grid3 g, unsigned long long *acc, int rec,
                                                      unsigned long long *counters)
{
    __shared__ uint32_t stage[4 * kStage3];
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int cell = -1;
    uint32_t w8[8];
    bool bad = false;
    if (p < n) {
        const float x = xs[p];
        if (!is_dead(x) &&
            !cic3((double)x * g.idx, (double)ys[p] * g.idy, (double)zs[p] * g.idz, g, cell, w8)) {
            cell = -1;
            bad = true;
        }
    }
    wave_deposit3(cell, w8, g, acc, rec, stage + (threadIdx.x >> 6) * kStage3);
    if (__ballot(bad) && __lane_id() == 0) raise_flag(counters, M2D_FLAG_OUT_OF_RANGE);
}

// ------------------------------------------------------------------ sort
// tile-major cell key: (tile << 6) | cell in its 4 x 4 x 4 tile
struct Key3 {
    const float *x, *y, *z;
    Grid3 g;
    int nty3, ntz3;
    uint32_t dead_key;
    __device__ __forceinline__ uint32_t operator()(int64_t p) const
    {
        const float v = x[p];
        if (is_dead(v)) return dead_key;
        auto idx = [](double X, int nmax) { return X >= 0.0 ? (int)fmin(X, (double)nmax) : 0; };
        const int i = idx((double)v * g.idx, g.nx - 2), j = idx((double)y[p] * g.idy, g.ny - 2),
                  k = idx((double)z[p] * g.idz, g.nz - 2);
        const uint32_t tile = (uint32_t)(((i / kTile3) * nty3 + j / kTile3) * ntz3 + k / kTile3);
        return (tile << 6) | (uint32_t)((i % kTile3) * 16 + (j % kTile3) * 4 + k % kTile3);
    }
};

// ------------------------------------------------------------------ host helpers
static int dmalloc3(m2d_ctx *ctx, void **p, size_t bytes)
{
    hipError_t e = dev_malloc(ctx, p, bytes < 16 ? 16 : bytes);
    if (e != hipSuccess)
        return set_error(M2D_ERR_NO_MEMORY, "hipMalloc(%zu): %s", bytes, hipGetErrorString(e));
    return M2D_OK;
}

static Grid3 grid3_of(const m2d_grid3d &g)
{
    Grid3 r;
    r.nx = g.nx; r.ny = g.ny; r.nz = g.nz;
    r.idx = 1.0 / g.dx; r.idy = 1.0 / g.dy; r.idz = 1.0 / g.dz;
    r.hx = (g.nx - 1) * g.dx * r.idx;
    r.hy = (g.ny - 1) * g.dy * r.idy;
    r.hz = (g.nz - 1) * g.dz * r.idz;
    return r;
}

static int check_grid3(const m2d_grid3d *g)
{
    M2D_CHECK(g, M2D_ERR_BAD_ARG, "3D grid is NULL");
    M2D_CHECK(g->nx >= 3 && g->ny >= 3 && g->nz >= 3 && g->dx > 0 && g->dy > 0 && g->dz > 0, M2D_ERR_BAD_ARG,
              "3D grid %dx%dx%d spacing %g,%g,%g", g->nx, g->ny, g->nz, g->dx, g->dy, g->dz);
    M2D_CHECK((size_t)g->nx * g->ny * g->nz < (1ull << 31), M2D_ERR_BAD_ARG, "3D grid too large");
    return M2D_OK;
}

static int check_parts3(const m2d_particles3d *p)
{
    M2D_CHECK(p, M2D_ERR_BAD_ARG, "3D particle store is NULL");
    M2D_CHECK(p->n >= 0 && p->n < (1ll << 31), M2D_ERR_BAD_ARG, "3D store of %lld slots", (long long)p->n);
    M2D_CHECK(p->n == 0 || (p->x && p->y && p->z && p->vx && p->vy && p->vz), M2D_ERR_BAD_ARG,
              "3D particle arrays must be non-NULL");
    return M2D_OK;
}

// Blocks of the linear reductions over the finest level: a block per 256 nodes
// up to kRed3Blocks, then that many, whose threads stride over several nodes
// (four at a time).  kRed3Blocks = kFinBlocks, so that the sums are finished
// in the launch itself.  A solve of 128^3 nodes: 256, 512 and 1024 blocks
// 1.46, 1.45 and 1.46 ms, 2048 1.48, as many as 256 nodes each give 1.58
// (96 x 112 x 128: 1.34, 1.34, 1.34, 1.37 and 1.42).
constexpr size_t kRed3Blocks = 1024;
static unsigned red_blocks3(size_t n)
{
    return (unsigned)std::min<size_t>((n + kRedBlock - 1) / kRedBlock, kRed3Blocks);
}

static unsigned up_blocks3(const m2d_fields3d *f);

// a level on the host while the hierarchy is built
struct Host3 {
    int n[3];
    std::vector<uint8_t> nbm;      // as Mg3Level::nbm
    std::vector<float> cond[6];    // conductance of each link, to a free neighbour (1) or to a Dirichlet value
    size_t size() const { return (size_t)n[0] * n[1] * n[2]; }
    int stride(int q) const  // of link q: -x, -y, -z, +z, +y, +x
    {
        const int s[6] = {-n[1] * n[2], -n[2], -1, 1, n[2], n[1] * n[2]};
        return s[q];
    }
    float diag(size_t m) const
    {
        float d = 0.f;
        for (int q = 0; q < 6; q++) d += cond[q].empty() ? 1.f : cond[q][m];
        return d;
    }
};

// Inverse of the coarsest 7-point operator on its free nodes, as a matrix over
// all its nodes with zeros for the pinned ones.  The operator is symmetric and
// positive definite, so its nodes are swept one after the other on the lower
// triangle, without pivoting; sweeping all of them leaves minus the inverse.
// Rows the sweep has not reached yet are outside the band and cost nothing:
// q^3 / 6 operations (343 free nodes of 9^3: 2 ms, by whole rows 5.7).
static bool dense_inverse7(const Host3 &V, std::vector<float> &inv)
{
    const size_t n = V.size();
    std::vector<int> pos(n, -1), id;
    for (size_t m = 0; m < n; m++)
        if (!(V.nbm[m] & kNbSelf)) { pos[m] = (int)id.size(); id.push_back((int)m); }
    const int q = (int)id.size();
    std::vector<double> a((size_t)q * q, 0.0), v(q);
    for (int r = 0; r < q; r++) {
        const int m = id[r];
        a[(size_t)r * q + r] = V.diag(m);
        for (int l = 0; l < 3; l++)  // the links to earlier nodes
            if (V.nbm[m] >> l & 1) a[(size_t)r * q + pos[m + V.stride(l)]] = -1.0;
    }
    for (int c = 0; c < q; c++) {
        for (int t = 0; t < q; t++) v[t] = t < c ? a[(size_t)c * q + t] : a[(size_t)t * q + c];
        if (!(v[c] > 1e-300)) return false;
        const double d = 1.0 / v[c];
        for (int r = 0; r < q; r++) {
            if (r == c || v[r] == 0.0) continue;
            double *rr = &a[(size_t)r * q];
            const double f = v[r] * d;
            for (int t = 0; t <= r; t++) rr[t] -= f * v[t];
        }
        for (int t = 0; t < q; t++) (t < c ? a[(size_t)c * q + t] : a[(size_t)t * q + c]) = v[t] * d;
        a[(size_t)c * q + c] = -d;
    }
    inv.assign(n * n, 0.f);
    for (int r = 0; r < q; r++)
        for (int c = 0; c < q; c++)
            inv[(size_t)id[r] * n + id[c]] = (float)-a[(size_t)std::max(r, c) * q + std::min(r, c)];
    return true;
}

// Coarse level of F: node I is free where fine node 2I is, faces are pinned.
// An even side of f nodes gets f / 2 + 1 coarse ones, the last of them one
// fine node past the grid: its neighbours then lie one node too far from the
// wall on every level, where f / 2 nodes would bring the wall 2^l - 1 nodes
// closer on level l.  A link that meets a Dirichlet node halfway (the fine
// node between two coarse ones, or a shorter distance taken over from the
// finer level) ends there, with the conductance 1 / (distance in coarse
// spacings) to its value, so electrodes keep their size on coarse levels.
// On a quadrupole trap of 64^3 the two bring the CG's residual per iteration
// down by 9 instead of 4 (with the one sweep of this V-cycle), and by 20 with
// two sweeps.
static Host3 coarsen3(const Host3 &F)
{
    Host3 C;
    for (int d = 0; d < 3; d++) C.n[d] = F.n[d] / 2 + 1;
    C.nbm.assign(C.size(), kNbSelf);
    for (auto &c : C.cond) c.assign(C.size(), 1.f);
    for (int I = 0; I < C.n[0]; I++)
        for (int J = 0; J < C.n[1]; J++)
            for (int K = 0; K < C.n[2]; K++) {
                const size_t M = ((size_t)I * C.n[1] + J) * C.n[2] + K;
                uint8_t bits = (I + J + K) & 1 ? kNbBlack : 0;
                const bool face = I == 0 || J == 0 || K == 0 || I == C.n[0] - 1 || J == C.n[1] - 1 || K == C.n[2] - 1;
                const size_t m = ((size_t)(2 * I) * F.n[1] + 2 * J) * F.n[2] + 2 * K;
                if (face || (F.nbm[m] & kNbSelf)) {
                    C.nbm[M] = bits | kNbSelf;
                    continue;
                }
                for (int q = 0; q < 6; q++) {
                    auto cond = [&](size_t at) { return F.cond[q].empty() ? 1.f : F.cond[q][at]; };
                    if (!(F.nbm[m] >> q & 1)) {
                        C.cond[q][M] = 2.f * cond(m);
                    } else {
                        const size_t mid = m + F.stride(q);
                        if (F.nbm[mid] >> q & 1) bits |= (uint8_t)(1u << q);
                        else C.cond[q][M] = 2.f * cond(mid) / (1.f + cond(mid));
                    }
                }
                C.nbm[M] = bits;
            }
    return C;
}

constexpr size_t kCoarsest3 = 800;      // coarsening stops at this many nodes (9^3 = 729 and fewer)
// nodes for the dense coarsest solve: below kCoarsest3, or of a level with a
// side that cannot be halved, of whose nodes few are free then (10 MB to read
// at most: a solve of 36 x 36 x 6 nodes 455 us, by sweeps 2.0 ms)
constexpr int kCoarseDenseMax = 1600;
constexpr int kCoarseSweeps = 40;       // symmetric RB-GS sweeps otherwise

// tiles of the finest and of the other levels (see k3_down)
constexpr size_t kLargeTiles3 = 1 << 20;

static int mg3_setup(m2d_fields3d *f, const std::vector<uint8_t> &mask)
{
    std::vector<Host3> lv(1);
    {
        Host3 &V = lv[0];
        V.n[0] = f->nx; V.n[1] = f->ny; V.n[2] = f->nz;
        V.nbm.resize(f->n);
        auto pinned = [&](size_t m) { return mask[m] == M2D_FIXED || mask[m] == M2D_FIXED_RF; };
        size_t m = 0;
        for (int i = 0; i < f->nx; i++)
            for (int j = 0; j < f->ny; j++)
                for (int k = 0; k < f->nz; k++, m++) {
                    uint8_t bits = (i + j + k) & 1 ? kNbBlack : 0;
                    if (pinned(m)) bits |= kNbSelf;
                    else  // a free node never sits on a face (checked at creation)
                        for (int q = 0; q < 6; q++)
                            if (!pinned(m + V.stride(q))) bits |= (uint8_t)(1u << q);
                    V.nbm[m] = bits;
                }
    }
    // down to kCoarsest3 nodes, or to a side that cannot be halved
    while (lv.back().size() > kCoarsest3 && lv.back().n[0] >= 5 && lv.back().n[1] >= 5 && lv.back().n[2] >= 5)
        lv.push_back(coarsen3(lv.back()));
    const size_t L = lv.size();
    M2D_CHECK(L <= (size_t)kMaxLevels3, M2D_ERR_BAD_ARG, "Fields3D: %d multigrid levels", (int)L);
    f->lv.resize(L);
    std::vector<float> di;
    for (size_t l = 0; l < L; l++) {
        Mg3Level &V = f->lv[l];
        const Host3 &H = lv[l];
        V.nx = H.n[0]; V.ny = H.n[1]; V.nz = H.n[2];
        V.n = H.size();
        M2D_TRY(dmalloc3(f->ctx, (void **)&V.nbm, V.n));
        M2D_HIP(hipMemcpy(V.nbm, H.nbm.data(), V.n, hipMemcpyHostToDevice));
        if (l == 0) continue;
        di.resize(V.n);
        for (size_t m = 0; m < V.n; m++) di[m] = 1.f / H.diag(m);
        M2D_TRY(dmalloc3(f->ctx, (void **)&V.di, sizeof(float) * V.n));
        M2D_TRY(dmalloc3(f->ctx, (void **)&V.x, sizeof(float) * V.n));
        M2D_TRY(dmalloc3(f->ctx, (void **)&V.b, sizeof(float) * V.n));
        M2D_HIP(hipMemcpy(V.di, di.data(), sizeof(float) * V.n, hipMemcpyHostToDevice));
        // the descent's tiles need not cover the last, pinned nodes
        M2D_HIP(hipMemset(V.b, 0, sizeof(float) * V.n));
    }
    f->coarse_dense = lv.back().size() <= (size_t)kCoarseDenseMax;
    if (f->coarse_dense) {
        std::vector<float> inv;
        M2D_CHECK(dense_inverse7(lv.back(), inv), M2D_ERR_BAD_ARG, "Fields3D: coarsest multigrid operator is singular");
        M2D_TRY(dmalloc3(f->ctx, (void **)&f->coarse_inv, sizeof(float) * inv.size()));
        M2D_HIP(hipMemcpy(f->coarse_inv, inv.data(), sizeof(float) * inv.size(), hipMemcpyHostToDevice));
    }
    const size_t n = f->n;
    for (float **q : {&f->pr, &f->pz, &f->pp, &f->pp2, &f->pq, &f->pe}) M2D_TRY(dmalloc3(f->ctx, (void **)q, sizeof(float) * n));
    // 16 scalars, then the solve's control block
    M2D_TRY(dmalloc3(f->ctx, (void **)&f->dots, sizeof(double) * 32));
    M2D_HIP(hipHostMalloc((void **)&f->h_dots, sizeof(double) * 32));
    // up to three sums per block of the fused reductions, one per tile of the ascent
    f->npartial = (int)std::max({red_blocks3(n), up_blocks3(f), 3 * Cols3{f->nx, f->ny, f->nz}.blocks()});
    M2D_TRY(dmalloc3(f->ctx, (void **)&f->partial, sizeof(double) * f->npartial));
    M2D_TRY(dmalloc3(f->ctx, (void **)&f->ticket, sizeof(unsigned int) * kTicketWords));
    M2D_HIP(hipMemset(f->ticket, 0, sizeof(unsigned int) * kTicketWords));
    return M2D_OK;
}

static unsigned blocks_for(size_t n) { return (unsigned)((n + 255) / 256); }

static dim3 tiles3(const Mg3Level &V, int ti, int tj, int tk)
{
    return dim3((unsigned)((V.nz + tk - 1) / tk), (unsigned)((V.ny + tj - 1) / tj), (unsigned)((V.nx + ti - 1) / ti));
}

// (the levels below the finest always take the small tiles)
static dim3 tiles3(const Mg3Level &V)
{
    return !V.di && V.n >= kLargeTiles3 ? tiles3(V, 8, 8, 64) : tiles3(V, 4, 8, 32);
}

static unsigned up_blocks3(const m2d_fields3d *f)
{
    const dim3 g = tiles3(f->lv[0]);
    return g.x * g.y * g.z;
}

template <bool FINEST>
static void launch_down3(const Mg3Level &V, const Mg3Level &C, const float *b, hipStream_t s, const int *stop)
{
    auto go = [&](auto kern, int threads) {
        kern<<<tiles3(V), threads, 0, s>>>(V.nbm, V.di, b, V.nx, V.ny, V.nz, C.b, C.nbm, C.nx, C.ny, C.nz, stop);
    };
    if (FINEST && V.n >= kLargeTiles3) go(k3_down<8, 8, 64, 512, true>, 512);
    else go(k3_down<4, 8, 32, 256, FINEST>, 256);
}

template <bool FINEST>
static void launch_up3(const Mg3Level &V, const Mg3Level &C, const float *b, float *out, hipStream_t s,
                       const int *stop, double *partial = nullptr, unsigned int *ticket = nullptr,
                       double *dot = nullptr, int fin = 0)
{
    auto go = [&](auto kern, int threads) {
        kern<<<tiles3(V), threads, 0, s>>>(V.nbm, V.di, b, V.nx, V.ny, V.nz, C.x, C.nx, C.ny, C.nz, out, partial,
                                           ticket, dot, fin, stop);
    };
    if (FINEST && V.n >= kLargeTiles3) go(k3_up<8, 8, 64, 512, true, true>, 512);
    else go(k3_up<4, 8, 32, 256, FINEST, FINEST>, 256);
}

// out = V-cycle of rhs and dot = rhs.out
static int vcycle3(m2d_fields3d *f, const float *rhs, float *out, double *dot, const int *stop)
{
    hipStream_t s = f->ctx->stream;
    const int L = (int)f->lv.size();
    Mg3Level &Z = f->lv[L - 1];
    for (int l = 0; l < L - 1; l++) {
        if (l == 0) launch_down3<true>(f->lv[0], f->lv[1], rhs, s, stop);
        else launch_down3<false>(f->lv[l], f->lv[l + 1], f->lv[l].b, s, stop);
    }
    const float *zb = L == 1 ? rhs : Z.b;
    float *zx = L == 1 ? out : Z.x;
    if (f->coarse_dense) {
        k3_dense<<<(unsigned)((Z.n + 3) / 4), 256, 0, s>>>(f->coarse_inv, zb, zx, (int)Z.n, stop);
    } else if (L > 1 && Z.n <= kSweepsNodes) {
        k3_sweeps<<<1, kCoarseThreads, 0, s>>>(Z.nbm, Z.di, zb, zx, Z.ny, Z.nz, (int)Z.n, kCoarseSweeps, stop);
    } else {
        const dim3 g((unsigned)(((Z.nz + 1) / 2 + kRbgsX - 1) / kRbgsX), (unsigned)((Z.ny + kRbgsY - 1) / kRbgsY),
                     (unsigned)Z.nx);
        k3_zero<<<blocks_for(Z.n), 256, 0, s>>>(zx, Z.n, stop);
        for (int h = 0; h < 2 * kCoarseSweeps; h++)
            k3_rbgs<<<g, dim3(kRbgsX, kRbgsY), 0, s>>>(Z.nbm, Z.di, zx, zb, Z.nx, Z.ny, Z.nz,
                                                       h < kCoarseSweeps ? h & 1 : ~h & 1, stop);
    }
    for (int l = L - 2; l >= 1; l--) launch_up3<false>(f->lv[l], f->lv[l + 1], f->lv[l].b, f->lv[l].x, s, stop);
    if (L > 1) {
        reduce_launch<1>(up_blocks3(f), f->partial, dot, s, [&](int fin) {
            launch_up3<true>(f->lv[0], f->lv[1], rhs, out, s, stop, f->partial, f->ticket, dot, fin);
        }, stop);
    } else {
        const unsigned rb = red_blocks3(f->n);
        reduce_launch<1>(rb, f->partial, dot, s, [&](int fin) {
            k_dot_fin<<<rb, kRedBlock, 0, s>>>(rhs, out, f->n, f->partial, f->ticket, dot, fin, stop);
        }, stop);
    }
    M2D_HIP(hipGetLastError());
    return M2D_OK;
}

static SolveCtl *solve_ctl3(m2d_fields3d *f) { return (SolveCtl *)(f->dots + 16); }

// Iterations from + 1 .. to of the open FP32 PCG pass on A' e = d (d in pr,
// e in pe), from 0: the pass's start; every launch stops with the pass
// (SolveCtl::stop_pcg).  cur: which of dots[0], dots[4] holds the current
// r.z, (iterations run - 1) & 1.  dots: [1] p.q, [2] r.r
static int queue_pcg3(m2d_fields3d *f, int from, int to, int &cur)
{
    hipStream_t s = f->ctx->stream;
    const size_t n = f->n;
    const unsigned rb = red_blocks3(n);
    const Mg3Level &V = f->lv[0];
    const Cols3 g{V.nx, V.ny, V.nz};
    SolveCtl *ctl = solve_ctl3(f);
    const int *stop = &ctl->stop_pcg;
    // iteration it's direction goes to P[it & 1], the previous one's is read from the other
    float *const P[2] = {f->pp, f->pp2};
    if (from == 0) {
        M2D_TRY(vcycle3(f, f->pr, f->pz, f->dots, stop));
        cur = 0;
    }
    for (int it = from + 1; it <= to; it++) {
        if (it > 1) {
            M2D_TRY(vcycle3(f, f->pr, f->pz, f->dots + 4 * (cur ^ 1), stop));
            cur ^= 1;
        }
        const float *pold = P[(it - 1) & 1];
        float *pnew = P[it & 1];
        reduce_launch<1>(g.blocks(), f->partial, f->dots + 1, s, [&](int fin) {
            auto go = [&](auto kern) {
                kern<<<g.grid(), kRedBlock, 0, s>>>(g, V.nbm, f->pz, pold, pnew, f->pq, f->dots + 4 * cur,
                                                    f->dots + 4 * (cur ^ 1), it == 1, f->partial, f->ticket,
                                                    f->dots + 1, fin, stop);
            };
            if (g.di() == 8) go(k3_dir_apply_dot<8>);
            else go(k3_dir_apply_dot<4>);
        }, stop);
        reduce_launch<1>(rb, f->partial, f->dots + 2, s, [&](int fin) {
            k_cg_update_dot<<<rb, kRedBlock, 0, s>>>(f->pe, f->pr, pnew, f->pq, f->dots + 4 * cur, f->dots + 1, n,
                                                     it == 1, f->partial, f->ticket, f->dots + 2, fin, stop,
                                                     CtlCheck{ctl});
        }, stop, CtlCheck{ctl});
    }
    M2D_HIP(hipGetLastError());
    return M2D_OK;
}

// the FP64 residual of u, its norms, and the refinement's decision on them;
// first: the solve's first one, which starts a fresh control block
static void queue_residual3(m2d_fields3d *f, double tol, bool first)
{
    hipStream_t s = f->ctx->stream;
    const Cols3 g{f->nx, f->ny, f->nz};
    SolveCtl *ctl = solve_ctl3(f);
    const int *stop = first ? nullptr : &ctl->stop_outer;
    const CtlEval eval{ctl, tol, kMaxOuter};
    auto go = [&](auto kern, auto post) {
        reduce_launch<3>(g.blocks(), f->partial, f->dots + 8, s, [&](int fin) {
            kern<<<g.grid(), kRedBlock, 0, s>>>(g, f->mask, f->rho, f->u, f->pr, f->partial, f->ticket, f->dots + 8,
                                                fin, stop, post);
        }, stop, post);
    };
    if (g.di() == 8) {
        if (first) go(k3_residual64_fin<8, CtlFirst>, CtlFirst{eval});
        else go(k3_residual64_fin<8, CtlEval>, eval);
    } else {
        if (first) go(k3_residual64_fin<4, CtlFirst>, CtlFirst{eval});
        else go(k3_residual64_fin<4, CtlEval>, eval);
    }
}

static int build_tables3(m2d_fields3d *f)
{
    k3_tables<<<planes3(f->nx, f->ny, f->nz), dim3(64, 4), 0, f->ctx->stream>>>(
        f->u, f->nx, f->ny, f->nz, f->idx, f->idy, f->idz, f->tx, f->ty, f->tz);
    M2D_HIP(hipGetLastError());
    return M2D_OK;
}

static double *field3_ptr(m2d_fields3d *f, int which)
{
    switch (which) {
    case M2D_FIELD_U: return f->u;
    case M2D_FIELD_RHO: return f->rho;
    case M2D_FIELD_VOLTAGE: return f->voltage;
    default: return nullptr;
    }
}

static float f32_below(double v)  // largest float <= v
{
    float r = (float)v;
    if ((double)r > v) r = nextafterf(r, -INFINITY);
    return r;
}

static uint64_t trial_thr3(double prob)
{
    if (!(prob > 0.0)) return 0;
    if (prob >= 1.0) return 1ull << 32;
    return (uint64_t)ceil(prob * 4294967296.0 - 0.5);
}

static void fill_args3(PushArgs3 &a, m2d_fields3d *f, const m2d_species2d *s, const m2d_particles3d *p,
                       double rot_scale, double kick_scale)
{
    a.x = p->x; a.y = p->y; a.z = p->z; a.vx = p->vx; a.vy = p->vy; a.vz = p->vz; a.n = p->n;
    a.tx = f->tx; a.ty = f->ty; a.tz = f->tz;
    a.cellfree = f->cellfree;
    a.g = grid3_of(f->p.grid);
    a.bx1 = f32_below(f->p.x_max); a.by1 = f32_below(f->p.y_max); a.bz1 = f32_below(f->p.z_max);
    a.xper = f->p.x_max; a.yper = f->p.y_max; a.zper = f->p.z_max;
    const double tmp = rot_scale * s->charge * s->dt / (2.0 * s->mass);
    const double tx = f->p.Bx * tmp, ty = f->p.By * tmp, tz = f->p.Bz * tmp;
    const double sc = 2.0 / (1 + tx * tx + ty * ty + tz * tz);
    a.tx_ = (float)tx; a.ty_ = (float)ty; a.tz_ = (float)tz;
    a.sx = (float)(tx * sc); a.sy = (float)(ty * sc); a.sz = (float)(tz * sc);
    a.rotate = tx != 0.0 || ty != 0.0 || tz != 0.0;
    a.qmdt2 = (float)(kick_scale * s->charge / s->mass * s->dt / 2.0);
    a.dt = (float)s->dt;
    a.push = 1;
    a.boundary = 0;
    a.periodic = f->p.boundary == M2D_BC_PERIODIC;
    a.trial_thr = 0;
    a.seed = f->ctx->seed;
    a.stream = s->stream;
    a.step = s->niter;
    a.mcc = nullptr; a.cq = nullptr; a.cq_len = nullptr;
    a.acc = nullptr;
    a.rec = 0;
    a.counters = f->ctx->counters;
}

// Records pay from one particle per eight nodes on: 295k particles took 78 us
// of atomics at the nodes against 15 us on 128^3, and 172 against 16 us on
// 64^3; the records' flush and clearing, 64 bytes a node to read and to
// write, take 33 and about 25 us on 96 x 112 x 128 (1.4M nodes).  On grids whose records stay within
// 1 GiB.
static bool use_rec3(int64_t particles, size_t nodes)
{
    return (size_t)particles >= nodes / 8 && particles >= 16384 && nodes <= (1u << 24);
}

static int flush_rec3(m2d_ctx *ctx, double *rho, double charge, int nx, int ny, int nz)
{
    k3_flush_rec<<<planes3(nx, ny, nz), dim3(64, 4), 0, ctx->stream>>>((const unsigned long long *)ctx->rec.ptr, rho,
                                                                       charge, nx, ny, nz);
    M2D_HIP(hipGetLastError());
    return rec_done(ctx, (size_t)nx * ny * nz, 8);
}

static void free3(m2d_fields3d *f)
{
    for (void *q : {(void *)f->mask, (void *)f->cellfree, (void *)f->voltage, (void *)f->u, (void *)f->rho,
                    (void *)f->tx, (void *)f->ty, (void *)f->tz, (void *)f->coarse_inv, (void *)f->pr,
                    (void *)f->pz, (void *)f->pp, (void *)f->pp2, (void *)f->pq, (void *)f->pe,
                    (void *)f->dots, (void *)f->partial, (void *)f->ticket})
        if (q) (void)hipFree(q);
    for (Mg3Level &V : f->lv)
        for (void *q : {(void *)V.nbm, (void *)V.di, (void *)V.x, (void *)V.b})
            if (q) (void)hipFree(q);
    if (f->h_dots) (void)hipHostFree(f->h_dots);
}

}  // namespace m2d

using namespace m2d;

extern "C" {

int m2d_fields3d_create(m2d_ctx *ctx, const m2d_fields3d_params *p, const uint8_t *mask, const double *voltage,
                        m2d_fields3d **out)
{
    M2D_CHECK(ctx && p && mask && voltage && out, M2D_ERR_BAD_ARG, "m2d_fields3d_create: NULL argument");
    *out = nullptr;
    M2D_TRY(check_grid3(&p->grid));
    M2D_CHECK(p->x_max > 0 && p->y_max > 0 && p->z_max > 0, M2D_ERR_BAD_ARG, "m2d_fields3d_create: box");
    const m2d_grid3d &g = p->grid;
    const size_t n = (size_t)g.nx * g.ny * g.nz;
    for (int i = 0; i < g.nx; i++)
        for (int j = 0; j < g.ny; j++)
            for (int k = 0; k < g.nz; k++) {
                const uint8_t m = mask[((size_t)i * g.ny + j) * g.nz + k];
                M2D_CHECK(m <= M2D_BOUNDARY, M2D_ERR_BAD_ARG, "mask value %d at (%d,%d,%d)", (int)m, i, j, k);
                const bool face = i == 0 || j == 0 || k == 0 || i == g.nx - 1 || j == g.ny - 1 || k == g.nz - 1;
                M2D_CHECK(!face || m == M2D_FIXED || m == M2D_FIXED_RF, M2D_ERR_BAD_ARG,
                          "m2d_fields3d_create: node (%d,%d,%d) on a grid face is not Dirichlet", i, j, k);
            }
    M2D_HIP(hipSetDevice(ctx->device));
    m2d_fields3d *f = new (std::nothrow) m2d_fields3d();
    M2D_CHECK(f, M2D_ERR_NO_MEMORY, "m2d_fields3d_create: host allocation");
    f->ctx = ctx;
    ctx_retain(ctx);
    f->p = *p;
    f->nx = g.nx; f->ny = g.ny; f->nz = g.nz;
    f->n = n;
    f->idx = 1.0 / g.dx; f->idy = 1.0 / g.dy; f->idz = 1.0 / g.dz;
    int r = M2D_OK;
    auto fail = [&](int code) { m2d_fields3d_destroy(f); return code; };
    if ((r = dmalloc3(f->ctx, (void **)&f->mask, n)) || (r = dmalloc3(f->ctx, (void **)&f->cellfree, n)) ||
        (r = dmalloc3(f->ctx, (void **)&f->voltage, 8 * n)) || (r = dmalloc3(f->ctx, (void **)&f->u, 8 * n)) ||
        (r = dmalloc3(f->ctx, (void **)&f->rho, 8 * n)) || (r = dmalloc3(f->ctx, (void **)&f->tx, 4 * n)) ||
        (r = dmalloc3(f->ctx, (void **)&f->ty, 4 * n)) || (r = dmalloc3(f->ctx, (void **)&f->tz, 4 * n)))
        return fail(r);
    std::vector<uint8_t> hm(mask, mask + n), cf(n, 0);
    for (int i = 0; i + 1 < g.nx; i++)
        for (int j = 0; j + 1 < g.ny; j++)
            for (int k = 0; k + 1 < g.nz; k++) {
                bool any = false;
                for (int c = 0; c < 8; c++)
                    any = any || hm[((size_t)(i + (c & 1)) * g.ny + j + ((c >> 1) & 1)) * g.nz + k + (c >> 2)] ==
                                     M2D_FREE;
                cf[((size_t)i * g.ny + j) * g.nz + k] = any;
            }
    if (hipMemcpy(f->mask, mask, n, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(f->cellfree, cf.data(), n, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(f->voltage, voltage, 8 * n, hipMemcpyHostToDevice) != hipSuccess)
        return fail(set_error(M2D_ERR_HIP, "m2d_fields3d_create: upload failed"));
    if ((r = fill_bytes(ctx, f->u, 0, 8 * n)) || (r = fill_bytes(ctx, f->rho, 0, 8 * n))) return fail(r);
    if ((r = mg3_setup(f, hm))) return fail(r);
    if ((r = build_tables3(f))) return fail(r);
    if (hipStreamSynchronize(ctx->stream) != hipSuccess)
        return fail(set_error(M2D_ERR_HIP, "m2d_fields3d_create: synchronise failed"));
    *out = f;
    return M2D_OK;
}

int m2d_fields3d_destroy(m2d_fields3d *f)
{
    if (!f) return M2D_OK;
    if (f->ctx) (void)hipStreamSynchronize(f->ctx->stream);
    free3(f);
    if (f->ctx) ctx_release(f->ctx);
    delete f;
    return M2D_OK;
}

double *m2d_fields3d_data(m2d_fields3d *f, int which) { return f ? field3_ptr(f, which) : nullptr; }

int m2d_fields3d_upload(m2d_fields3d *f, int which, const double *host)
{
    M2D_CHECK(f && host, M2D_ERR_BAD_ARG, "m2d_fields3d_upload: NULL argument");
    double *d = field3_ptr(f, which);
    M2D_CHECK(d, M2D_ERR_BAD_ARG, "m2d_fields3d_upload: unknown field %d", which);
    M2D_HIP(hipMemcpyAsync(d, host, 8 * f->n, hipMemcpyHostToDevice, f->ctx->stream));
    if (which == M2D_FIELD_U) M2D_TRY(build_tables3(f));
    M2D_HIP(hipStreamSynchronize(f->ctx->stream));
    return M2D_OK;
}

int m2d_fields3d_download(m2d_fields3d *f, int which, double *host)
{
    M2D_CHECK(f && host, M2D_ERR_BAD_ARG, "m2d_fields3d_download: NULL argument");
    double *d = field3_ptr(f, which);
    M2D_CHECK(d, M2D_ERR_BAD_ARG, "m2d_fields3d_download: unknown field %d", which);
    M2D_HIP(hipMemcpyAsync(host, d, 8 * f->n, hipMemcpyDeviceToHost, f->ctx->stream));
    M2D_HIP(hipStreamSynchronize(f->ctx->stream));
    return M2D_OK;
}

int m2d_fields3d_reset(m2d_fields3d *f)
{
    M2D_CHECK(f, M2D_ERR_BAD_ARG, "m2d_fields3d_reset: NULL argument");
    return fill_bytes(f->ctx, f->rho, 0, 8 * f->n);
}

int m2d_fields3d_solve(m2d_fields3d *f, double tol, m2d_solve_info *info)
{
    M2D_CHECK(f, M2D_ERR_BAD_ARG, "m2d_fields3d_solve: NULL argument");
    hipStream_t s = f->ctx->stream;
    const size_t n = f->n;
    const unsigned gb = blocks_for(n);
    k3_rhs<<<gb, 256, 0, s>>>(f->mask, f->voltage, f->rho, f->u, n, f->p.rhs_scale);
    M2D_HIP(hipGetLastError());
    if (tol <= 0) tol = 1e-10;
    SolveCtl *ctl = solve_ctl3(f);
    SolveCtl *h = (SolveCtl *)(f->h_dots + 16);
    queue_residual3(f, tol, true);
    M2D_TRY(queue_refinement(
        s, ctl, h, f->dots, f->est, tol, 80,
        [&](int from, int to, int &cur) { return queue_pcg3(f, from, to, cur); },
        [&] { k3_add_correction<<<gb, 256, 0, s>>>(f->mask, f->u, f->pe, n, &ctl->no_add); },
        [&] { queue_residual3(f, tol, false); }));
    const int outer = h->outer;
    const double rel = h->rel;
    if (info) { info->outer_iters = outer; info->inner_iters = h->iters; info->rel_residual = rel; }
    if (h->nan) return set_error(M2D_ERR_NAN, "Fields3D solve: residual is not finite");
    M2D_TRY(build_tables3(f));
    if (rel > tol)
        return set_error(M2D_ERR_NOT_CONVERGED, "Fields3D solve: relative residual %.3e > %.3e after %d steps",
                         rel, tol, outer);
    return M2D_OK;
}

int m2d_accumulate_3d(m2d_ctx *ctx, const m2d_grid3d *g, const m2d_particles3d *p, double charge, double *rho)
{
    M2D_CHECK(ctx && rho, M2D_ERR_BAD_ARG, "m2d_accumulate_3d: NULL argument");
    M2D_TRY(check_grid3(g));
    M2D_TRY(check_parts3(p));
    const size_t n = (size_t)g->nx * g->ny * g->nz;
    int rec = use_rec3(p->n, n);
    unsigned long long *acc;
    M2D_TRY(deposit_buffer(ctx, n, 8, rec, acc));
    if (p->n > 0) {
        k_accumulate3d<<<blocks_for((size_t)p->n), 256, 0, ctx->stream>>>(
            p->x, p->y, p->z, p->n, grid3_of(*g), acc, rec, ctx->counters);
        M2D_HIP(hipGetLastError());
    }
    if (rec) return flush_rec3(ctx, rho, charge, g->nx, g->ny, g->nz);
    k_flush<<<blocks_for(n), 256, 0, ctx->stream>>>((unsigned long long *)ctx->acc.ptr, rho, charge, n);
    M2D_HIP(hipGetLastError());
    return M2D_OK;
}

int m2d_interpolate_3d(m2d_ctx *ctx, const m2d_grid3d *g, const double *data, const double *x, const double *y,
                       const double *z, int64_t n, double *out)
{
    M2D_CHECK(ctx && data && (n == 0 || (x && y && z && out)), M2D_ERR_BAD_ARG, "m2d_interpolate_3d: NULL argument");
    M2D_TRY(check_grid3(g));
    if (n > 0) {
        k_interp3d<<<blocks_for((size_t)n), 256, 0, ctx->stream>>>(data, grid3_of(*g), x, y, z, n, out);
        M2D_HIP(hipGetLastError());
    }
    return M2D_OK;
}

int m2d_grad_3d(m2d_ctx *ctx, const m2d_grid3d *g, const double *data, const double *x, const double *y,
                const double *z, int64_t n, double *gx, double *gy, double *gz)
{
    M2D_CHECK(ctx && data && (n == 0 || (x && y && z && gx && gy && gz)), M2D_ERR_BAD_ARG,
              "m2d_grad_3d: NULL argument");
    M2D_TRY(check_grid3(g));
    if (n > 0) {
        k_grad3d<<<blocks_for((size_t)n), 256, 0, ctx->stream>>>(data, grid3_of(*g), x, y, z, n, gx, gy, gz);
        M2D_HIP(hipGetLastError());
    }
    return M2D_OK;
}

int m2d_advance_3d(m2d_ctx *ctx, m2d_fields3d *f, const m2d_species2d *s, const m2d_particles3d *p,
                   const m2d_mcc *mcc, double *rho, uint32_t flags, m2d_step_stats *stats)
{
    M2D_CHECK(ctx && f && s, M2D_ERR_BAD_ARG, "m2d_advance_3d: NULL argument");
    M2D_CHECK(f->ctx == ctx, M2D_ERR_BAD_ARG, "m2d_advance_3d: fields belong to another context");
    M2D_TRY(check_parts3(p));
    M2D_CHECK(s->mass > 0 && s->dt > 0, M2D_ERR_BAD_ARG, "m2d_advance_3d: mass and dt must be > 0");
    M2D_CHECK((flags & ~(M2D_STEP_PUSH | M2D_STEP_BOUNDARY | M2D_STEP_DEPOSIT)) == 0, M2D_ERR_BAD_ARG,
              "m2d_advance_3d: unknown flags 0x%x", flags);
    const bool deposit = (flags & M2D_STEP_DEPOSIT) != 0;
    M2D_CHECK(!deposit || rho, M2D_ERR_BAD_ARG, "m2d_advance_3d: DEPOSIT needs rho");
    M2D_CHECK(!mcc || !mcc->h.partner_update, M2D_ERR_UNSUPPORTED,
              "m2d_advance_3d: COULOMB (partner update) runs in m2d_advance_2d only");
    M2D_CHECK(!mcc || !mcc_partners_alias(mcc, p->x), M2D_ERR_UNSUPPORTED,
              "m2d_advance_3d: partners from the colliding species' own store run in m2d_advance_2d only");
    if (stats) {
        M2D_TRY(zero_words(ctx, ctx->counters + CNT_REMOVED, 2));
        M2D_TRY(zero_words(ctx, ctx->counters + CNT_SPILL, 1));
    }
    PushArgs3 a;
    fill_args3(a, f, s, p, 1.0, 1.0);
    a.push = (flags & M2D_STEP_PUSH) != 0;
    a.boundary = (flags & M2D_STEP_BOUNDARY) != 0;
    // an empty store queues nothing (and leaves the alternating counters)
    const bool use_mcc = p->n > 0 && a.push && mcc && std::isfinite(s->lifetime) && s->lifetime > 0;
    unsigned long long *next_len = nullptr;
    if (use_mcc) {
        a.trial_thr = trial_thr3(1.0 - exp(-s->dt / s->lifetime));  // species3d.cpp:8
        a.mcc = mcc->d;
        M2D_TRY(ensure(ctx, ctx->cq, (size_t)p->n * sizeof(uint32_t)));
        a.cq = (uint32_t *)ctx->cq.ptr;
        // a call that failed between its pass and its scatter left the
        // alternating counters unknown: clear both first
        if (ctx->cq_dirty) M2D_TRY(zero_words(ctx, ctx->counters + CNT_QLEN, 2));
        ctx->cq_dirty = true;
        const int slot = (int)(ctx->launch_seq++ & 1);
        a.cq_len = ctx->counters + CNT_QLEN + slot;
        next_len = ctx->counters + CNT_QLEN + (slot ^ 1);
    }
    // a store sorted by m2d_sort_3d deposits through per-chunk LDS windows
    const int ntx3 = (f->nx - 2) / kTile3 + 1, nty3 = (f->ny - 2) / kTile3 + 1, ntz3 = (f->nz - 2) / kTile3 + 1;
    const m2d_tiling *T = deposit ? find_tiling(ctx, p->x, p->n) : nullptr;
    if (T && (T->ntx != ntx3 || T->nty != nty3 || T->ntz != ntz3)) T = nullptr;
    if (deposit) {
        a.rec = !T && use_rec3(p->n, f->n);
        M2D_TRY(deposit_buffer(ctx, f->n, 8, a.rec, a.acc));
    }
    if (p->n > 0) {
        if (T) {
            launch_timed(ctx, use_mcc ? k_advance3d_tiled<true> : k_advance3d_tiled<false>, dim3(T->max_chunks),
                         dim3(256), a, T->sched, T->n_chunks, nty3, ntz3);
        } else {
            void (*kern)(PushArgs3) = deposit ? (use_mcc ? k_advance3d<true, true> : k_advance3d<true, false>)
                                              : (use_mcc ? k_advance3d<false, true> : k_advance3d<false, false>);
            launch_timed(ctx, kern, dim3(blocks_for((size_t)p->n)), dim3(256), a);
        }
        M2D_HIP(hipGetLastError());
        if (use_mcc) {
            k_scatter3d<<<64, 256, 0, ctx->stream>>>(a, next_len);
            M2D_HIP(hipGetLastError());
            ctx->cq_dirty = false;
        }
    }
    if (a.rec) {
        M2D_TRY(flush_rec3(ctx, rho, s->charge, f->nx, f->ny, f->nz));
    } else if (deposit) {
        k_flush<<<blocks_for(f->n), 256, 0, ctx->stream>>>(a.acc, rho, s->charge, f->n);
        M2D_HIP(hipGetLastError());
    }
    if (stats) {
        M2D_TRY(read_counters(ctx));
        stats->removed = (int64_t)ctx->h_counters[CNT_REMOVED];
        stats->collisions = (int64_t)ctx->h_counters[CNT_COLL];
        stats->spilled = (int64_t)ctx->h_counters[CNT_SPILL];
    }
    return M2D_OK;
}

int m2d_advance_init_3d(m2d_ctx *ctx, m2d_fields3d *f, const m2d_species2d *s, const m2d_particles3d *p)
{
    M2D_CHECK(ctx && f && s, M2D_ERR_BAD_ARG, "m2d_advance_init_3d: NULL argument");
    M2D_TRY(check_parts3(p));
    M2D_CHECK(s->mass > 0 && s->dt > 0, M2D_ERR_BAD_ARG, "m2d_advance_init_3d: mass and dt must be > 0");
    PushArgs3 a;
    fill_args3(a, f, s, p, -0.5, -1.0);
    if (p->n > 0) {
        k_advance_init3d<<<blocks_for((size_t)p->n), 256, 0, ctx->stream>>>(a);
        M2D_HIP(hipGetLastError());
    }
    return M2D_OK;
}

int m2d_sort_3d(m2d_ctx *ctx, m2d_fields3d *f, const m2d_particles3d *src, const m2d_particles3d *dst,
                int64_t *n_live)
{
    M2D_CHECK(ctx && f && src && dst, M2D_ERR_BAD_ARG, "m2d_sort_3d: NULL argument");
    M2D_TRY(check_parts3(src));
    M2D_TRY(check_parts3(dst));
    M2D_CHECK(dst->n == src->n, M2D_ERR_BAD_ARG, "m2d_sort_3d: dst holds %lld slots, src %lld",
              (long long)dst->n, (long long)src->n);
    M2D_CHECK(src->n == 0 || src->x != dst->x, M2D_ERR_BAD_ARG, "m2d_sort_3d: src and dst must differ");
    const size_t n = (size_t)src->n;
    forget_tiling(ctx, src->x);
    forget_tiling(ctx, dst->x);
    if (n == 0) {
        if (n_live) *n_live = 0;
        return M2D_OK;
    }
    const Grid3 g = grid3_of(f->p.grid);
    const int ntx3 = (g.nx - 2) / kTile3 + 1, nty3 = (g.ny - 2) / kTile3 + 1, ntz3 = (g.nz - 2) / kTile3 + 1;
    const int bits = sort_key_bits((uint64_t)ntx3 * nty3 * ntz3);
    M2D_CHECK(bits <= 32, M2D_ERR_BAD_ARG, "m2d_sort_3d: grid too large for 32-bit keys");
    // tile-major cell order.  Unlike the 2D store (ordered by tile only), a
    // 3D cell holds few particles (8 on average at the 16M-ion, 128^3
    // workload), so the lanes of a wave spread over several cells anyway, and
    // the cell order's gather locality wins: the tiled pass runs 419 us on a
    // cell-ordered store against 505 us on a tile-ordered one
    const Key3 key{src->x, src->y, src->z, g, nty3, ntz3, sort_dead_key(bits)};
    const Columns<6> from{{src->x, src->y, src->z, src->vx, src->vy, src->vz}},
        to{{dst->x, dst->y, dst->z, dst->vx, dst->vy, dst->vz}};
    return sort_store(ctx, key, from, to, n, 0, bits, ntx3, nty3, ntz3, kChunkCap3, 256, n_live);
}

int m2d_sort_forget_3d(m2d_ctx *ctx, const m2d_particles3d *p)
{
    M2D_CHECK(ctx && p, M2D_ERR_BAD_ARG, "m2d_sort_forget_3d: NULL argument");
    forget_tiling(ctx, p->x);
    return M2D_OK;
}

int m2d_count_live_3d(m2d_ctx *ctx, const m2d_particles3d *p, int64_t *n_live)
{
    M2D_TRY(check_parts3(p));
    const m2d_particles2d v{p->x, p->z, p->vx, p->vy, p->vz, p->n};
    return m2d_count_live_2d(ctx, &v, n_live);
}

int m2d_mean_energy_3d(m2d_ctx *ctx, const m2d_particles3d *p, double mass, double *mean_eV, int64_t *n_live)
{
    M2D_TRY(check_parts3(p));
    const m2d_particles2d v{p->x, p->z, p->vx, p->vy, p->vz, p->n};
    return m2d_mean_energy_2d(ctx, &v, mass, mean_eV, n_live);
}

}  // extern "C"
