// m2d_direct2d.hip -- the direct form of the 2D Poisson solve, for fields
// whose free nodes fill a rectangle: EMPTY and any grid whose electrodes leave
// a box (a frame, thick walls, end caps along whole walls).  Electrodes with
// gaps between them or inside the box (the named traps, a probe) leave no
// rectangle.
//
// On a full m x n rectangle between Dirichlet nodes the 5-point operator
// A' = 4 - (sum of neighbours) is diagonal in the discrete sine basis:
//   A'^-1 D = S_m (Lambda^-1 o (S_m D S_n)) S_n,
//   S_m[i][p] = sqrt(2 / (m+1)) sin(pi (i+1)(p+1) / (m+1)),
//   Lambda[p][q] = 4 sin^2(pi (p+1) / (2(m+1))) + 4 sin^2(pi (q+1) / (2(n+1))),
// so a solve is four dense products, on the FP64 matrix cores.  A solve of a
// warm-started 128^2 trap is then 7 dependent launches instead of about 60
// (multigrid-PCG, m2d_fields2d.hip), which is what bounds both.
#include "m2d_objects.hpp"
#include <cmath>

namespace m2d {

typedef double f64x4 __attribute__((ext_vector_type(4)));

// ------------------------------------------------------------------ set-up
// S (P x P, the m x m sine matrix padded with zeros) and the eigenvalue
// terms lam[p] = 4 sin^2(pi (p+1) / (2(m+1))) (padding: 1, never used but
// divided by).  The sine's argument is reduced in integers.
__global__ void k_dst_matrix(int m, int P, double *S, double *lam)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x, i = blockIdx.y;
    if (p >= P) return;
    const int64_t period = 2 * (int64_t)(m + 1);
    double v = 0.0;
    if (i < m && p < m) v = sqrt(2.0 / (m + 1)) * sinpi((double)((int64_t)(i + 1) * (p + 1) % period) / (m + 1));
    S[(size_t)i * P + p] = v;
    if (i == 0) {
        const double s = sinpi((double)(p + 1) / (double)period);
        lam[p] = p < m ? 4.0 * s * s : 1.0;
    }
}

// ------------------------------------------------------------------ the products
// C = S B for a symmetric S (rows x rows) and a row-major B (rows x cols),
// both padded to multiples of kDstPad.  S being symmetric, both operands are
// read k-major: 16 lanes take 16 consecutive doubles of one row of S and of
// B, whole 128-byte lines.  The products that need the other side are formed
// transposed instead (stages 1 and 3 store C^T), so every stage reads alike.
//   stage 1: T1 = S_m D       D = the FP64 residual on the grid; stores T1^T
//   stage 2: T2^T = S_n T1^T, divided by Lambda
//   stage 3: T3^T = S_n T2^T, stores T3
//   stage 4: E = S_m T3 = A'^-1 D, subtracted from u on the rectangle (A u = -A' u
//            + Dirichlet terms, so A (u - E) = A u + D = b)
// A block of four wavefronts owns an output tile of 16 NT x 16 NT; each
// wavefront sums a quarter of k in v_mfma_f64_16x16x4 accumulators and the
// quarters meet in LDS in a fixed order (the same bits on every run).  The
// work is latency-bound up to 256^2 (64 tiles of 16 x 16 at 128^2, 8 matrix
// instructions a wavefront), hence the split of k and the smallest tile
// there; larger grids have tiles enough and take 32 x 32 (NT = 2), which
// halves the reads.
constexpr int kDstThreads = 256;

struct DstStage {
    const double *S;
    int ldS;
    const double *B;       // row-major; stage 1: the grid array at the rectangle's corner
    int ldB;
    int K, kvalid, cvalid; // rows of B, those inside the rectangle, columns inside it
    double *C;             // stages 1, 3: C^T (ldC = rows); stage 2: C
    int ldC;
    const double *lrow, *lcol;  // stage 2
    int rvalid;            // stage 4: rows inside the rectangle
    const int *ahead;      // a pass that may well be needless: its stop flag, waited for before any operand is read
    SolveCtl *ctl;
};

template <int STAGE, int NT>
__global__ void __launch_bounds__(kDstThreads) k_dst_stage(DstStage a)
{
    constexpr int T = 16 * NT;
    __shared__ double part[4][T][T + 1];
    const int stop = a.ctl->stop_outer;
    if (stopped(a.ahead)) return;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, c = lane & 15, kk = lane >> 4;
    const int row0 = blockIdx.y * T, col0 = blockIdx.x * T;
    const int len = a.K / 4, k0 = wave * len;
    f64x4 acc[NT][NT];
#pragma unroll
    for (int s = 0; s < NT; s++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[s][t] = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
    for (int k = k0 + kk; k < k0 + len; k += 4) {
        double A[NT], B[NT];
#pragma unroll
        for (int s = 0; s < NT; s++) A[s] = a.S[(size_t)k * a.ldS + row0 + 16 * s + c];
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const int col = col0 + 16 * t + c;
            if (STAGE == 1) B[t] = k < a.kvalid && col < a.cvalid ? a.B[(size_t)k * a.ldB + col] : 0.0;
            else B[t] = a.B[(size_t)k * a.ldB + col];
        }
#pragma unroll
        for (int s = 0; s < NT; s++)
#pragma unroll
            for (int t = 0; t < NT; t++) acc[s][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[s], B[t], acc[s][t], 0, 0, 0);
    }
    if (stop) return;  // uniform; a first pass reads it beside its operands, not before them
    // accumulator r of lane l: row l / 16 + 4 r, column l % 16 of its 16 x 16 tile
#pragma unroll
    for (int s = 0; s < NT; s++)
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) part[wave][16 * s + kk + 4 * r][16 * t + c] = acc[s][t][r];
    __syncthreads();
    for (int e = threadIdx.x; e < T * T; e += kDstThreads) {
        // consecutive threads along the stored array's rows
        const int i = STAGE == 1 || STAGE == 3 ? e % T : e / T, j = STAGE == 1 || STAGE == 3 ? e / T : e % T;
        double v = ((part[0][i][j] + part[1][i][j]) + part[2][i][j]) + part[3][i][j];
        const int row = row0 + i, col = col0 + j;
        if (STAGE == 1 || STAGE == 3) a.C[(size_t)col * a.ldC + row] = v;
        else if (STAGE == 2) a.C[(size_t)row * a.ldC + col] = v / (a.lrow[row] + a.lcol[col]);
        else if (row < a.rvalid && col < a.cvalid) a.C[(size_t)row * a.ldC + col] -= v;
    }
    if (STAGE == 4 && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) {
        // one pass done: nothing else in this launch reads these
        SolveCtl *ctl = a.ctl;
        if (ctl->outer < kMaxPasses) ctl->pass_count[ctl->outer] = 1;
        ctl->outer++;
        ctl->iters++;
        ctl->max_pass_iters = 1;
    }
}

template <int STAGE>
static void launch_stage(const DstStage &a, int rows, int cols, hipStream_t s)
{
    // 16 x 16 tiles while they number at most two a CU
    if ((rows / 16) * (cols / 16) <= 512)
        k_dst_stage<STAGE, 1><<<dim3(cols / 16, rows / 16), kDstThreads, 0, s>>>(a);
    else
        k_dst_stage<STAGE, 2><<<dim3(cols / 32, rows / 32), kDstThreads, 0, s>>>(a);
}

// u -= A'^-1 r on the rectangle (r: FP64 residual on the grid), unless the
// solve has stopped; counts one pass of one iteration.  surplus: the pass is
// one of several queued together, which the first may have made needless: its
// products then wait for the stop flag before they read their operands (at
// 1024^2 a needless pass took 226 us, now 8)
int direct2d_pass(m2d_fields2d *f, double *u, SolveCtl *ctl, bool surplus)
{
    const Direct2 &d = f->direct;
    hipStream_t s = f->ctx->stream;
    const size_t corner = (size_t)d.i0 * f->nz + d.j0;
    DstStage a{};
    a.ctl = ctl;
    a.ahead = surplus ? &ctl->stop_outer : nullptr;
    a.S = d.sm; a.ldS = d.M; a.B = f->mg.r64 + corner; a.ldB = f->nz;
    a.K = d.M; a.kvalid = d.m; a.cvalid = d.n; a.C = d.t0; a.ldC = d.M;
    launch_stage<1>(a, d.M, d.N, s);
    a.S = d.sn; a.ldS = d.N; a.B = d.t0; a.ldB = d.M;
    a.K = d.N; a.C = d.t1; a.ldC = d.M; a.lrow = d.ln; a.lcol = d.lm;
    launch_stage<2>(a, d.N, d.M, s);
    a.B = d.t1; a.C = d.t0; a.ldC = d.N;
    launch_stage<3>(a, d.N, d.M, s);
    a.S = d.sm; a.ldS = d.M; a.B = d.t0; a.ldB = d.N;
    a.K = d.M; a.C = u + corner; a.ldC = f->nz; a.rvalid = d.m; a.cvalid = d.n;
    launch_stage<4>(a, d.M, d.N, s);
    M2D_HIP(hipGetLastError());
    return M2D_OK;
}

// The rule: the free nodes are every node of one rectangle, of at most
// kDirectMax nodes a side.  Measured from u = 0 to 1e-10, host read
// included, multigrid-PCG against this: 32^2 354 -> 68 us, 128^2 626 -> 65,
// 256^2 924 -> 69, 512^2 1390 -> 125, 768^2 1975 -> 212, 1024^2 2725 -> 604
// (there FP64 rounding leaves 1e-10 after one pass and a second one runs).
// Past it the n^3 products grow faster than the multigrid's work per node
// and one pass no longer meets the default tolerance.  Creation is cheaper
// too (1024^2: 123 -> 10 ms): no hierarchy is built.
constexpr int kDirectMax = 1024;

bool direct2d_fits(const std::vector<uint8_t> &mask, int nx, int nz, Direct2 &d)
{
    int i0 = nx, i1 = -1, j0 = nz, j1 = -1;
    size_t free_nodes = 0;
    for (int i = 0; i < nx; i++)
        for (int j = 0; j < nz; j++) {
            const uint8_t m = mask[(size_t)i * nz + j];
            if (m == M2D_FIXED || m == M2D_FIXED_RF) continue;
            free_nodes++;
            i0 = std::min(i0, i); i1 = std::max(i1, i);
            j0 = std::min(j0, j); j1 = std::max(j1, j);
        }
    if (!free_nodes) return false;
    const int m = i1 - i0 + 1, n = j1 - j0 + 1;
    if (free_nodes != (size_t)m * n || m > kDirectMax || n > kDirectMax) return false;
    d.i0 = i0; d.j0 = j0; d.m = m; d.n = n;
    d.M = (m + kDstPad - 1) / kDstPad * kDstPad;
    d.N = (n + kDstPad - 1) / kDstPad * kDstPad;
    return true;
}

int direct2d_setup(m2d_fields2d *f)
{
    Direct2 &d = f->direct;
    const size_t M = d.M, N = d.N;
    const size_t words = M * M + M + N * N + N + 2 * M * N;
    hipError_t e = dev_malloc(f->ctx, (void **)&d.buf, words * sizeof(double));
    if (e != hipSuccess)
        return set_error(M2D_ERR_NO_MEMORY, "Fields: hipMalloc(%zu): %s", words * sizeof(double), hipGetErrorString(e));
    d.sm = d.buf;
    d.sn = d.sm + M * M;
    d.t0 = d.sn + N * N;
    d.t1 = d.t0 + M * N;
    d.lm = d.t1 + M * N;
    d.ln = d.lm + M;
    hipStream_t s = f->ctx->stream;
    k_dst_matrix<<<dim3((d.M + 255) / 256, d.M), 256, 0, s>>>(d.m, d.M, d.sm, d.lm);
    k_dst_matrix<<<dim3((d.N + 255) / 256, d.N), 256, 0, s>>>(d.n, d.N, d.sn, d.ln);
    M2D_HIP(hipGetLastError());
    return M2D_OK;
}

}  // namespace m2d
