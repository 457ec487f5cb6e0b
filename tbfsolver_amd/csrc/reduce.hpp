// reduce.hpp -- deterministic block and grid reductions (device code).
#pragma once
#include "mg_kernels.hpp"

namespace tbfg {

// Sums over the workgroup (at most 16 wavefronts), valid in thread 0.
template <int NV>
__device__ __forceinline__ void block_sum(double (&v)[NV], double* lds /* >= 32*NV */)
{
    const int lane = threadIdx.x + blockDim.x * threadIdx.y;
    const int nthreads = blockDim.x * blockDim.y;
#pragma unroll
    for (int q = 0; q < NV; ++q)
        for (int off = 32; off > 0; off >>= 1) v[q] += __shfl_down(v[q], off, 64);
    const int wave = lane >> 6;
    const int nwaves = (nthreads + 63) >> 6;
    if ((lane & 63) == 0)
        for (int q = 0; q < NV; ++q) lds[wave * NV + q] = v[q];
    __syncthreads();
    if (lane < 64) {
        // sum q in lane q, its LDS reads issued together, in the order of the wavefronts
        // (one lane reading 80 values one by one took half of a finalize's 5 us)
        const int q = lane < NV ? lane : NV - 1;
        double s = 0.0;
        if (nwaves <= 4) {
#pragma unroll
            for (int w = 0; w < 4; ++w) s += w < nwaves ? lds[w * NV + q] : 0.0;
        } else {
#pragma unroll
            for (int w = 0; w < 16; ++w) s += w < nwaves ? lds[w * NV + q] : 0.0;
        }
        if (NV == 1)
            v[0] = s;
        else
#pragma unroll
            for (int u = 0; u < NV; ++u) v[u] = __shfl(s, u, 64);
    }
}

// Deterministic grid reduction in two launches: every block of the producing
// kernel writes its NV partial sums (block_partial); a one-block finalize
// kernel adds them in block order (final_sum).  No device-scope fence is
// needed, which matters on a multi-XCD part where such a fence writes back L2.
template <int NV>
__device__ __forceinline__ void block_partial(double (&v)[NV], const Reducer& red)
{
    __shared__ double lds[32 * 8];
    const int lane = threadIdx.x + blockDim.x * threadIdx.y;
    const unsigned bid = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
    block_sum<NV>(v, lds);
    if (lane == 0)
        for (int q = 0; q < NV; ++q) red.partials[(size_t)bid * NV + q] = v[q];
}

// one block; thread 0 receives the totals
template <int NV>
__device__ __forceinline__ void final_sum(const Reducer& red, unsigned nblocks, double (&tot)[NV])
{
    __shared__ double lds[32 * 8];
    double acc[NV];
#pragma unroll
    for (int q = 0; q < NV; ++q) acc[q] = 0.0;
    // several partials of a thread in flight: a loop of single loads waits for each
    constexpr int U = NV == 1 ? 8 : 2;
    for (unsigned b0 = threadIdx.x; b0 < nblocks; b0 += U * blockDim.x) {
        double x[U][NV];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const unsigned b = b0 + u * blockDim.x;
#pragma unroll
            for (int q = 0; q < NV; ++q) x[u][q] = red.partials[(size_t)(b < nblocks ? b : b0) * NV + q];
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int q = 0; q < NV; ++q) acc[q] += b0 + u * blockDim.x < nblocks ? x[u][q] : 0.0;
    }
    block_sum<NV>(acc, lds);
    if (threadIdx.x == 0)
        for (int q = 0; q < NV; ++q) tot[q] = acc[q];
}

// The sum of n partials in every thread of a 256-thread workgroup, in the order in which 1024
// threads and their 16 wavefronts add them.
__device__ __forceinline__ double sum_by_1024(const double* __restrict__ partials, unsigned n)
{
    __shared__ double lds[16];
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    for (unsigned b = 0; b < n; b += 1024) {
        double x[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const unsigned e = b + u * 256 + threadIdx.x;
            x[u] = partials[e < n ? e : 0];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) acc[u] += b + u * 256 + threadIdx.x < n ? x[u] : 0.0;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
#pragma unroll
        for (int u = 0; u < 4; ++u) acc[u] += __shfl_down(acc[u], off, 64);
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int u = 0; u < 4; ++u) lds[4 * u + (threadIdx.x >> 6)] = acc[u];
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < 16; ++w) s += lds[w];
    return s;
}

// ||r|| and the stop test (pcg.f90:331-355,359-429), by one workgroup of at least 256 threads
__device__ __forceinline__ void fin_update(const FinUpdate& f)
{
    __shared__ double lds[32];
    PcgState* st = f.st;
    const int done = st->done, iter = st->iter + 1, max_iter = st->max_iter;
    const double qq = st->qq, tol = st->tol;
    double tot[1] = {0.0};
    for (unsigned b0 = 0; b0 < f.n; b0 += 2048) {  // the order of 256 threads
        double x[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const unsigned e = b0 + u * 256 + threadIdx.x;
            x[u] = f.partials[e < f.n ? e : 0];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) tot[0] += threadIdx.x < 256 && b0 + u * 256 + threadIdx.x < f.n ? x[u] : 0.0;
    }
    block_sum<1>(tot, lds);
    if (threadIdx.x == 0 && !done) {
        st->rr = tot[0];
        st->iter = iter;
        const double res = sqrt(tot[0]) / sqrt(qq + 2.2250738585072014e-308);
        st->res = res;
        if (!isfinite(res)) {
            st->done = 1;
            st->status = TBFG_ENUMERIC;
        } else if (res <= tol) {
            st->done = 1;
            st->status = TBFG_OK;
        } else if (iter >= max_iter) {
            st->done = 1;
            st->status = TBFG_ENOTCONVERGED;
        }
    }
}

// The scalars of the next direction from the sums of the dot products (pcg.f90:294-327), by
// one workgroup.  host_done (pinned host memory, may be NULL) receives the stop flag: the
// host's stop test of the iteration that ends here, without a copy in the stream.
__device__ __forceinline__ void fin_dots(unsigned nblocks, size_t ncell, int init, PcgState* st, const Reducer& red,
                                         int32_t* host_done)
{
    int done = st->done;
    const int flexible = st->flexible;
    const double alpha = st->alpha, delta = st->delta;
    double tot[5];
    final_sum<5>(red, nblocks, tot);
    if (threadIdx.x == 0) {
        if (!done) {
            const double m = tot[2] / (double)ncell;
            const double rz = tot[0] - m * tot[3];
            st->zmean = m;
            if (init) {
                st->delta = rz;
                st->gamma = 0.0;
            } else {
                const double qz = tot[1] - m * tot[4];
                const double g = flexible ? (-alpha * qz / delta) : (rz / delta);
                st->gamma = g;
                st->delta = rz;
                if (!isfinite(g) || !isfinite(rz)) {
                    st->done = done = 1;
                    st->status = TBFG_ENUMERIC;
                }
            }
        }
        st->halted = done;
        if (host_done) __hip_atomic_store(host_done, done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

}  // namespace tbfg
