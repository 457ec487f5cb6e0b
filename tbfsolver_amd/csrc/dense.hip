// dense.hip -- dense exact solve of one multigrid level (the bottom of the
// hierarchy, or the reference's coarsest level when it is solved directly).
//
// G = (M + c 1 1^T)^-1 (I - 1 1^T / n) (-V), with M = -V A the V-scaled symmetric
// matrix of poissMat.f90:746-763: x = G q is the Lagrange-constrained exact solve
// (poissMat.f90:246-259,467-503, sum x = 0).  G is formed once per solve by
// inverting the symmetric positive definite M + c 1 1^T without pivoting, in
// place (the Gauss-Jordan exchange step: a_pp <- 1/a_pp, the pivot row scaled, the
// pivot column scaled and negated, the rest updated by rank one).
//
// The inversion is a chain of n dependent pivots, so its latency per pivot is what
// bounds it, not its 2 n^3 operations:
//   n <= 64   one workgroup, the matrix in registers (4 rows of a column per
//             thread), pivot row and column exchanged through LDS, one barrier per
//             pivot
//   n > 64    32 x 32 tiles, one launch per block of 32 pivots: every workgroup
//             updates one tile from the previous matrix to the next one (two
//             buffers, so no workgroup waits for another) with FP64 MFMA, and the
//             one that owns the next diagonal tile inverts it before it ends
// Against one workgroup eliminating [A | I] in HBM with four barriers a pivot: a PCG
// solve with a 315-cell bottom (72x40x56) 26.9 -> 2.8 ms, one with a 64-cell bottom
// (128^3, FP64) 4.45 -> 4.19 ms.
#include "dense.hpp"
#include "mg_launch.hpp"
#include "reduce.hpp"

namespace tbfg {

namespace {

constexpr int kTile = 32;
constexpr int kTileLd = kTile + 1;  // padded LDS rows
constexpr int kSmall = 64;          // largest single-workgroup inversion

using d4 = __attribute__((ext_vector_type(4))) double;

// one row of the operator: the six face coefficients times the cell's volume and
// the cells behind the faces (x, z periodic; a wall face points at the cell itself)
struct OpRow {
    double va[6];
    int nb[6];
};

template <class T>
__device__ __forceinline__ OpRow op_row(const LevelDev<double>& L, const T* __restrict__ beta,
                                        const double* __restrict__ vol, int c)
{
    const int nx = L.nx, ny = L.ny, nz = L.nz;
    const int i = c % nx, r = c / nx, j = r % ny, k = r / ny;
    OpRow o;
    o.nb[0] = i + 1 < nx ? c + 1 : c + 1 - nx;
    o.nb[1] = i > 0 ? c - 1 : c - 1 + nx;
    o.nb[2] = j + 1 < ny ? c + nx : c;
    o.nb[3] = j > 0 ? c - nx : c;
    o.nb[4] = k + 1 < nz ? c + nx * ny : c - k * nx * ny;
    o.nb[5] = k > 0 ? c - nx * ny : c + (nz - 1) * nx * ny;
    const double bc = (double)beta[c], v = vol[c];
    const double f[6] = {L.a[0].ip[i], L.a[0].im[i], L.a[1].ip[j], L.a[1].im[j], L.a[2].ip[k], L.a[2].im[k]};
#pragma unroll
    for (int q = 0; q < 6; ++q)
        o.va[q] = o.nb[q] == c ? 0.0 : v * (0.5 * ((double)beta[o.nb[q]] + bc) * f[q]);
    return o;
}

__device__ __forceinline__ double op_diag(const OpRow& o)
{
    double d = 0.0;
#pragma unroll
    for (int q = 0; q < 6; ++q) d += o.va[q];
    return d;
}

// M[c][col] (several faces may lead to the same cell on axes of one or two cells)
__device__ __forceinline__ double op_entry(const OpRow& o, double diag, int c, int col)
{
    double x = col == c ? diag : 0.0;
#pragma unroll
    for (int q = 0; q < 6; ++q)
        if (o.nb[q] == col && col != c) x -= o.va[q];
    return x;
}

// c of the shift: the mean diagonal entry over n
__device__ __forceinline__ double shift_of(double trace, int n)
{
    return (trace > 0.0 ? trace : 1.0) / ((double)n * n);
}

// In-place inverse of an NB x NB matrix held by NB^2/4 threads, v[u] = element
// (4 (t / NB) + u, t % NB).  The pivot row and column of the next step are put
// into the other pair of LDS buffers as soon as they are updated: one barrier per
// pivot.  groups: 4 pivots each (rows beyond are those of an identity).
template <int NB>
__device__ __forceinline__ void invert_regs(double (&v)[4], double (*rowb)[NB], double (*colb)[NB], int groups)
{
    const int c = threadIdx.x % NB, rg = threadIdx.x / NB;
    if (rg == 0) rowb[0][c] = v[0];
    if (c == 0)
#pragma unroll
        for (int u = 0; u < 4; ++u) colb[0][4 * rg + u] = v[u];
    __syncthreads();
    for (int g = 0; g < groups; ++g) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int p = 4 * g + s, b = s & 1;
            const double d = 1.0 / rowb[b][p];
            const double pr = rowb[b][c] * d;
            double pc[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) pc[u] = colb[b][4 * rg + u];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                double x = c == p ? -pc[u] * d : fma(-pc[u], pr, v[u]);
                if (u == s && rg == g) x = c == p ? d : pr;
                v[u] = x;
            }
            if (rg == g + (s == 3 ? 1 : 0)) rowb[b ^ 1][c] = v[(s + 1) & 3];
            if (c == p + 1)
#pragma unroll
                for (int u = 0; u < 4; ++u) colb[b ^ 1][4 * rg + u] = v[u];
            __syncthreads();
        }
    }
}

template <class T>
__global__ void __launch_bounds__(kSmall * kSmall / 4)
    k_dense_small(LevelDev<double> L, const T* __restrict__ beta, const double* __restrict__ vol,
                  double* __restrict__ G)
{
    __shared__ double rowb[2][kSmall], colb[2][kSmall];
    __shared__ double sVa[6][kSmall], sDiag[kSmall];
    __shared__ int sNb[6][kSmall];
    const int n = L.nx * L.ny * L.nz;
    const int t = threadIdx.x;
    if (t < kSmall) {
        double dg = 0.0;
        if (t < n) {
            const OpRow o = op_row(L, beta, vol, t);
            dg = op_diag(o);
#pragma unroll
            for (int q = 0; q < 6; ++q) {
                sVa[q][t] = o.va[q];
                sNb[q][t] = o.nb[q];
            }
        }
        sDiag[t] = dg;
    }
    __syncthreads();
    const int c = t % kSmall, rg = t / kSmall;
    double trace = sDiag[c];  // lanes of a wavefront = the columns
    for (int off = 32; off > 0; off >>= 1) trace += __shfl_xor(trace, off, 64);
    const double shift = shift_of(trace, n);
    double v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int r = 4 * rg + u;
        if (r < n && c < n) {
            OpRow o;
#pragma unroll
            for (int q = 0; q < 6; ++q) {
                o.va[q] = sVa[q][r];
                o.nb[q] = sNb[q][r];
            }
            v[u] = op_entry(o, sDiag[r], r, c) + shift;
        } else {
            v[u] = r == c ? 1.0 : 0.0;
        }
    }
    invert_regs<kSmall>(v, rowb, colb, (n + 3) / 4);
    const double vc = c < n ? vol[c] : 0.0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int r = 4 * rg + u;
        double s = c < n ? v[u] : 0.0;
        for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
        if (r < n && c < n) G[r * n + c] = -vc * (v[u] - s / (double)n);
    }
}

// M + c 1 1^T padded to N x N by an identity, one wavefront per row; every
// workgroup forms the trace itself, in one fixed order
template <class T>
__global__ void __launch_bounds__(256)
    k_dense_build(LevelDev<double> L, const T* __restrict__ beta, const double* __restrict__ vol, int N,
                  double* __restrict__ W)
{
    __shared__ double lds[4];
    const int n = L.nx * L.ny * L.nz;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double tr = 0.0;
    for (int c = threadIdx.x; c < n; c += 256) tr += op_diag(op_row(L, beta, vol, c));
    for (int off = 32; off > 0; off >>= 1) tr += __shfl_xor(tr, off, 64);
    if (lane == 0) lds[wave] = tr;
    __syncthreads();
    const double shift = shift_of(((lds[0] + lds[1]) + lds[2]) + lds[3], n);
    const int r = blockIdx.x * 4 + wave;  // N is a multiple of 32
    double* row = W + (size_t)r * N;
    if (r >= n) {
        for (int c = lane; c < N; c += 64) row[c] = c == r ? 1.0 : 0.0;
        return;
    }
    const OpRow o = op_row(L, beta, vol, r);
    const double diag = op_diag(o);
    for (int c = lane; c < N; c += 64) row[c] = c < n ? op_entry(o, diag, r, c) + shift : 0.0;
}

// the inverse of a 32 x 32 tile in LDS, written to D (row-major)
__device__ __forceinline__ void invert_tile(const double* tile, double (*rowb)[kTile], double (*colb)[kTile],
                                            double* __restrict__ D)
{
    const int c = threadIdx.x % kTile, rg = threadIdx.x / kTile;
    double v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = tile[(4 * rg + u) * kTileLd + c];
    invert_regs<kTile>(v, rowb, colb, kTile / 4);
#pragma unroll
    for (int u = 0; u < 4; ++u) D[(4 * rg + u) * kTile + c] = v[u];
}

__device__ __forceinline__ void load_tile(const double* __restrict__ src, int ld, double* tile)
{
    const int c = threadIdx.x % kTile, rg = threadIdx.x / kTile;
    double v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = src[(size_t)(4 * rg + u) * ld + c];
#pragma unroll
    for (int u = 0; u < 4; ++u) tile[(4 * rg + u) * kTileLd + c] = v[u];
}

// c += s A B for this wavefront's 16 x 16 quarter (r0, c0) of a 32 x 32 product;
// MFMA 16x16x4 FP64: lane l holds A[l % 16][l / 16], B[l / 16][l % 16] and the
// results (l / 16 + 4 v, l % 16)
__device__ __forceinline__ d4 tile_mma(const double* A, const double* B, int r0, int c0, double s, d4 c)
{
    const int lr = threadIdx.x & 15, lk = (threadIdx.x & 63) >> 4;
#pragma unroll
    for (int k = 0; k < kTile; k += 4)
        c = __builtin_amdgcn_mfma_f64_16x16x4f64(s * A[(r0 + lr) * kTileLd + k + lk],
                                                 B[(k + lk) * kTileLd + c0 + lr], c, 0, 0, 0);
    return c;
}

__global__ void __launch_bounds__(256) k_dense_first(const double* __restrict__ W, int N, double* __restrict__ D)
{
    __shared__ double sA[kTile * kTileLd];
    __shared__ double rowb[2][kTile], colb[2][kTile];
    load_tile(W, N, sA);
    __syncthreads();
    invert_tile(sA, rowb, colb, D);
}

// One block step: the exchange of the 32 pivots of diagonal tile k, whose inverse
// P is in Dk, from W to Wn; the owner of tile (k+1, k+1) leaves its inverse in Dn.
__global__ void __launch_bounds__(256)
    k_dense_step(const double* __restrict__ W, double* __restrict__ Wn, int N, int k, const double* __restrict__ Dk,
                 double* __restrict__ Dn)
{
    __shared__ double sP[kTile * kTileLd], sA[kTile * kTileLd], sB[kTile * kTileLd], sT[kTile * kTileLd];
    __shared__ double rowb[2][kTile], colb[2][kTile];
    const int nt = N / kTile;
    const int i = blockIdx.x / nt, j = blockIdx.x % nt;
    const int wave = threadIdx.x >> 6, r0 = (wave >> 1) * 16, c0 = (wave & 1) * 16;
    const int lr = threadIdx.x & 15, lk = (threadIdx.x & 63) >> 4;
    auto at = [&](int a, int b) { return W + (size_t)a * kTile * N + (size_t)b * kTile; };
    load_tile(Dk, kTile, sP);
    if (j != k) load_tile(at(k, j), N, sB);
    if (i != k) load_tile(at(i, k), N, sA);
    __syncthreads();
    d4 out = {0.0, 0.0, 0.0, 0.0};
    if (i == k && j == k) {
#pragma unroll
        for (int v = 0; v < 4; ++v) out[v] = sP[(r0 + lk + 4 * v) * kTileLd + c0 + lr];
    } else if (i == k) {
        out = tile_mma(sP, sB, r0, c0, 1.0, out);
    } else if (j == k) {
        out = tile_mma(sA, sP, r0, c0, -1.0, out);
    } else {
        const double* a = at(i, j) + (size_t)(r0 + lk) * N + c0 + lr;
        d4 c;
#pragma unroll
        for (int v = 0; v < 4; ++v) c[v] = a[(size_t)4 * v * N];
        const d4 t = tile_mma(sP, sB, r0, c0, 1.0, out);
#pragma unroll
        for (int v = 0; v < 4; ++v) sT[(r0 + lk + 4 * v) * kTileLd + c0 + lr] = t[v];
        __syncthreads();
        out = tile_mma(sA, sT, r0, c0, -1.0, c);
    }
    double* w = Wn + (size_t)i * kTile * N + (size_t)j * kTile + (size_t)(r0 + lk) * N + c0 + lr;
#pragma unroll
    for (int v = 0; v < 4; ++v) w[(size_t)4 * v * N] = out[v];
    if (i == k + 1 && j == k + 1) {
        // (sP was last read before the barrier above)
#pragma unroll
        for (int v = 0; v < 4; ++v) sP[(r0 + lk + 4 * v) * kTileLd + c0 + lr] = out[v];
        __syncthreads();
        invert_tile(sP, rowb, colb, Dn);
    }
}

// G[r][c] = -V_c (B[r][c] - mean of row r), one wavefront per row
__global__ void __launch_bounds__(256)
    k_dense_fin(const double* __restrict__ B, int N, int n, const double* __restrict__ vol, double* __restrict__ G)
{
    const int lane = threadIdx.x & 63, r = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (r >= n) return;
    const double* row = B + (size_t)r * N;
    double s = 0.0;
    for (int c = lane; c < n; c += 64) s += row[c];
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    s /= (double)n;
    for (int c = lane; c < n; c += 64) G[(size_t)r * n + c] = -vol[c] * (row[c] - s);
}

// x = G q, one wavefront per row, q staged in LDS.  Bound by reading G once (from
// the MALL after the first application): 1152 cells, 10.6 MB.
__global__ void __launch_bounds__(256)
    k_dense_apply(int n, const double* __restrict__ G, const double* __restrict__ q, double* __restrict__ x,
                  PcgState* st, const int* done)
{
    __shared__ double sq[kDenseDirectCells];
    const bool run = !(done && *done);
    if (blockIdx.x == 0 && threadIdx.x == 0) st->coarse_due = run ? 1 : 0;
    if (!run) return;
    for (int c = threadIdx.x; c < n; c += 256) sq[c] = q[c];
    __syncthreads();
    const int lane = threadIdx.x & 63, r = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (r >= n) return;
    const double* row = G + (size_t)r * n;
    double acc = 0.0;
#pragma unroll 8
    for (int c = lane; c < n; c += 64) acc += row[c] * sq[c];
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if (lane == 0) x[r] = acc;
}

// The diagnostics of one such solve (tbfg_pcg_coarse_stats): the V-weighted norm of
// its residual over that of the right-hand side projected onto the range of A
// (q - (sum V q) / (n V)), counted as one inner iteration; a zero right-hand side
// counts no call.  One workgroup, at most two cells per thread.
__device__ __forceinline__ void dense_check(const DenseCheck& a, PcgState* st)
{
    __shared__ double lds[32 * 2];
    __shared__ double s_shift;
    const LevelDev<double>& L = a.L;
    const double *beta = a.beta, *vol = a.vol, *q = a.q, *x = a.x;
    const int n = L.nx * L.ny * L.nz;
    double v[2], qc[2], ax[2], sum[1] = {0.0};
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int c = (int)threadIdx.x + u * 1024;
        v[u] = qc[u] = ax[u] = 0.0;
        if (c < n) {
            const OpRow o = op_row(L, beta, vol, c);
            v[u] = vol[c];
            qc[u] = q[c];
            double a = 0.0;
#pragma unroll
            for (int f = 0; f < 6; ++f) a += o.va[f] * (x[o.nb[f]] - x[c]);
            ax[u] = a / v[u];
            sum[0] += v[u] * qc[u];
        }
    }
    block_sum<1>(sum, lds);
    if (threadIdx.x == 0) s_shift = sum[0] / (double)n;
    __syncthreads();
    double rr[2] = {0.0, 0.0};
#pragma unroll
    for (int u = 0; u < 2; ++u)
        if ((int)threadIdx.x + u * 1024 < n) {
            const double r0 = qc[u] - s_shift / v[u], r = r0 - ax[u];
            rr[0] += v[u] * r0 * r0;
            rr[1] += v[u] * r * r;
        }
    block_sum<2>(rr, lds);
    if (threadIdx.x == 0 && rr[0] > 0.0) {
        st->coarse_calls += 1;
        st->coarse_iters += 1;
        if (st->coarse_iters_max < 1) st->coarse_iters_max = 1;
        const double rel = sqrt(rr[1] / rr[0]);
        if (rel > st->coarse_res_max) st->coarse_res_max = rel;
    }
}
__global__ void __launch_bounds__(1024) k_dense_check(DenseCheck a, PcgState* st, const int* done)
{
    if (done && *done) return;
    dense_check(a, st);
}

// k_fin_dots with the check beside it, in a second workgroup: nothing reads the diagnostics
// before the solve ends, and as a launch of its own the check cost 7.3 us of the 186 that an
// iteration takes at 96x64x96.  The first workgroup may set done, so the second goes by
// whether the solve it checks ran.
__global__ void __launch_bounds__(1024)
    k_fin_dots_check(unsigned nblocks, size_t ncell, int init, PcgState* st, Reducer red, int32_t* host_done,
                     DenseCheck a)
{
    if (blockIdx.x == 0)
        fin_dots(nblocks, ncell, init, st, red, host_done);
    else if (st->coarse_due)
        dense_check(a, st);
}

int padded(int n) { return (n + kTile - 1) / kTile * kTile; }

}  // namespace

size_t dense_work_doubles(size_t n)
{
    if (n <= (size_t)kSmall) return 1;
    const size_t N = (size_t)padded((int)n);
    return 2 * N * N + 2 * kTile * kTile;
}

template <class T>
int launch_dense_setup(const LevelDev<double>& L, const T* beta, const double* vol, double* work, double* G,
                       void* stream)
{
    hipStream_t s = (hipStream_t)stream;
    const int n = L.nx * L.ny * L.nz;
    if (n <= kSmall) {
        hipLaunchKernelGGL(k_dense_small<T>, dim3(1), dim3(kSmall * kSmall / 4), 0, s, L, beta, vol, G);
        TBFG_HIP(hipGetLastError());
        return TBFG_OK;
    }
    const int N = padded(n), nt = N / kTile;
    double* W[2] = {work, work + (size_t)N * N};
    double* D[2] = {work + 2 * (size_t)N * N, work + 2 * (size_t)N * N + kTile * kTile};
    hipLaunchKernelGGL(k_dense_build<T>, dim3(N / 4), dim3(256), 0, s, L, beta, vol, N, W[0]);
    hipLaunchKernelGGL(k_dense_first, dim3(1), dim3(256), 0, s, W[0], N, D[0]);
    for (int k = 0; k < nt; ++k)
        hipLaunchKernelGGL(k_dense_step, dim3(nt * nt), dim3(256), 0, s, W[k & 1], W[(k + 1) & 1], N, k, D[k & 1],
                           D[(k + 1) & 1]);
    hipLaunchKernelGGL(k_dense_fin, dim3(ceil_div(n, 4)), dim3(256), 0, s, W[nt & 1], N, n, vol, G);
    TBFG_HIP(hipGetLastError());
    return TBFG_OK;
}
int launch_dense_solve(const DenseCheck& a, const double* G, double* x, bool check, PcgState* st, const int* done,
                       void* stream)
{
    hipStream_t s = (hipStream_t)stream;
    const int n = a.L.nx * a.L.ny * a.L.nz;
    if (n > kDenseDirectCells) {
        set_error("launch_dense_solve: %d cells (at most %d)", n, kDenseDirectCells);
        return TBFG_EINVAL;
    }
    hipLaunchKernelGGL(k_dense_apply, dim3(ceil_div(n, 4)), dim3(256), 0, s, n, G, a.q, x, st, done);
    if (check) hipLaunchKernelGGL(k_dense_check, dim3(1), dim3(1024), 0, s, a, st, done);
    TBFG_HIP(hipGetLastError());
    return TBFG_OK;
}
int launch_fin_dots_check(unsigned nblocks, size_t ncell, int init, PcgState* st, const Reducer& red,
                          int32_t* host_done, const DenseCheck& a, void* stream)
{
    hipLaunchKernelGGL(k_fin_dots_check, dim3(2), dim3(1024), 0, (hipStream_t)stream, nblocks, ncell, init, st, red,
                       host_done, a);
    TBFG_HIP(hipGetLastError());
    return TBFG_OK;
}

template int launch_dense_setup<double>(const LevelDev<double>&, const double*, const double*, double*, double*,
                                        void*);
template int launch_dense_setup<float>(const LevelDev<double>&, const float*, const double*, double*, double*,
                                       void*);

}  // namespace tbfg
