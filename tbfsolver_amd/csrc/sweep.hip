// sweep.hip -- one full red/black Gauss-Seidel sweep per launch (rbgs.f90:205-259:
// the red half-sweep, then the black one), out of place: pin holds the level's
// values before the sweep and is only read, pout receives the values after it.
// Three kernels, chosen per level (pcg_create, smooth):
//   k_row_sweep    marches along z with whole rows of up to 256 cells in a wavefront
//   k_sweep        marches along z with tiles staged in LDS: rows longer than that, the tile
//                  shapes a tuning table names, the dot products under bf16 storage
//   k_point_sweep  no march, a thread per pair of cells: small levels and odd row lengths
// The values a workgroup needs from beyond its cells are recomputed from pin, so
// no workgroup waits on another and the result equals the two half-sweep launches up to
// the rounding of fused multiply-adds.
//
// k_sweep: a workgroup owns a TX x TY tile of cells in the (x, y) plane and a chunk of
// planes in z, and marches through the chunk one plane at a time.  At plane
// step k it computes the red cells of plane k over the tile plus a one-cell
// ring and then the black cells of plane k-1 over the tile, which need the new
// red values of planes k-2, k-1, k.  Every input plane is staged once in LDS (p and
// beta with a two-cell ring, q with a one-cell ring), loaded into registers one step
// ahead so that the HBM latency of plane k+2 overlaps the arithmetic of plane k.  HBM
// traffic per cell: p in, beta, q, p out -- once per sweep, where two half-sweep
// launches stream every array twice.
#include "mg_kernels.hpp"
#include "mg_launch.hpp"
#include "reduce.hpp"
#include "smooth.hpp"
#include "tune.hpp"

#include <hip/hip_ext.h>

#include <algorithm>
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <type_traits>

namespace tbfg {

namespace {

constexpr int kSweepMaxChunk = 58;  // planes per workgroup (z face factors staged in LDS)
constexpr int kZT = kSweepMaxChunk + 6;

template <class T, int TX, int TY, int NT>
struct SweepShape {
    static constexpr int PX = TX + 4, PY = TY + 4, PS = PX * PY;  // p, beta planes: tile + 2-cell ring
    static constexpr int QX = TX + 2, QY = TY + 2, QS = QX * QY;  // q, new-red planes: tile + 1-cell ring
    static constexpr int NP = (PS + NT - 1) / NT;
    static constexpr int NQ = (QS + NT - 1) / NT;
    static constexpr int NBLACK = TY * (TX / 2);                    // black cells of a tile plane
    // ring depth 4 for every staged plane (the plane steps run in groups of 4,
    // so the slot of a plane is a constant of the unrolled step): a slot is
    // refilled at least one full step after its last reader, so two barriers
    // per plane step suffice
    static constexpr int RING = 4;
};

__device__ __forceinline__ int wrapi(int i, int n) { return i < 0 ? i + n : (i >= n ? i - n : i); }
__device__ __forceinline__ int clampi(int j, int n) { return j < 0 ? 0 : (j >= n ? n - 1 : j); }

template <int NT, class T, int N>
__device__ __forceinline__ void stash_plane(const T (&reg)[N], T* __restrict__ dst, int S)
{
#pragma unroll
    for (int m = 0; m < N; ++m) dst[min((int)threadIdx.x + m * NT, S - 1)] = reg[m];
}

// raw buffer loads: a plane's loads share one scalar byte offset (the plane
// base) and differ by a fixed per-thread 32-bit offset, so no 64-bit address
// arithmetic per load; a load outside the array's bytes returns 0
__device__ __forceinline__ __amdgpu_buffer_rsrc_t plane_rsrc(const void* base, size_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0,
                                             (int)(bytes < 0x7fffffffu ? bytes : 0x7fffffffu), 0x00020000);
}
template <class T>
__device__ __forceinline__ T buf_load(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff);
template <>
__device__ __forceinline__ float buf_load<float>(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}
template <>
__device__ __forceinline__ double buf_load<double>(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff)
{
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
}
template <>
__device__ __forceinline__ bf16s buf_load<bf16s>(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff)
{
    return bf16s{__builtin_amdgcn_raw_buffer_load_b16(r, voff, soff, 0)};
}

template <class T>
struct Vec2;
template <>
struct Vec2<float> {
    using type = float2;
};
template <>
struct Vec2<double> {
    using type = double2;
};

// Per-thread column history: the values a thread used at its tile cell two
// plane steps earlier (same colour parity, same column) that the next step of
// the same parity needs again.
template <class T>
struct ColHist {
    T bf;  // beta(k-1)
    T bc;  // beta(k-2)
    T pf;  // p_old(k-1)
    T r;   // new red value at k-2
};

// The tile height TY divides ny, so every thread stores on every step: no
// branch around the stores, which lets the compiler wait for the loads of a
// plane without waiting for the stores issued after them.
//
// Thread t owns the pair of columns (tx0 + 2h, tx0 + 2h + 1) of tile row
// t / (TX/2).  At plane step k its red cell of plane k and its black cell of
// plane k-1 share one column (both have gx + gy + k odd), which alternates
// between the two columns of the pair from step to step; the beta, p_old and
// red values of that column from two steps earlier stay in registers.  The
// red cells of the ring around the tile are a second, smaller round.
// DOTS (the finest level's last sweep of a preconditioner application): the
// sums of k_pcg_dots -- r.z, qv.z, sum z, sum r, sum qv of the new values z --
// accumulate while the plane is written, one partial per workgroup, instead of
// a separate pass over r, z and qv.  r and qv of a plane are loaded with the
// plane registers, two steps ahead.
// TQ, TB: the storage types of q and beta (bf16s on a bf16-stored finest
// level: the loads convert to T, LDS and arithmetic stay in T).
template <class T, class TQ, class TB, int TX, int TY, int NT, bool FIRST, bool DOTS, int PD>
__global__ void __launch_bounds__(NT)
    k_sweep(LevelDev<T> L, const TB* __restrict__ beta, const TQ* __restrict__ q, const T* __restrict__ pin,
            T* __restrict__ pout, int kc, int tiles_x, int ntiles, const int* done, SweepDots dots)
{
    using Sh = SweepShape<T, TX, TY, NT>;
    static_assert(Sh::NBLACK == NT, "one tile cell pair per thread");
    static_assert(PD % 2 == 0, "the register sets alternate with the colour parity of the steps");
    constexpr int PX = Sh::PX, PS = Sh::PS, QX = Sh::QX, QS = Sh::QS, QY = Sh::QY;
    constexpr int RING = Sh::RING;
    constexpr int NRING = QX + TY;  // red cells of the one-cell ring
    __shared__ T sP[(FIRST ? 1 : RING) * PS];
    __shared__ T sB[RING * PS];
    __shared__ T sQ[RING * QS];
    // new red values: two slots (the black cells of step k read those of step
    // k-1, and the slot is next written after the first barrier of step k+1)
    __shared__ T sR[2 * QS];
    // face factors times 1/2 (exact), so a face coefficient is (beta + beta') * f
    __shared__ T sTx[2 * QX];    // x, tile columns -1..TX
    __shared__ T sTy[2 * QY];    // y, tile rows -1..TY
    __shared__ T sTz[2 * kZT];  // z, planes k0-1.. of the chunk's plane steps

    if (done && *done) return;
    const int nx = L.nx, ny = L.ny, nz = L.nz;
    // consecutive tiles of a chunk on one XCD (blocks go round-robin to the 8 XCDs)
    unsigned id = blockIdx.x;
    if ((gridDim.x & 7u) == 0) id = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    const int tile = (int)(id % (unsigned)ntiles);
    const int chunk = (int)(id / (unsigned)ntiles);
    const int k0 = chunk * kc;
    double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};  // DOTS
    if (k0 >= nz) {  // (the launch covers nz exactly; an empty chunk adds nothing)
        if (DOTS) block_partial<5>(acc, dots.red);
        return;
    }
    const int k1 = min(nz, k0 + kc);
    const int tx0 = (tile % tiles_x) * TX;
    const int ty0 = (tile / tiles_x) * TY;

    // plane steps k0-1 .. k1 (and up to 3 more, which compute red cells only)
    const int nsteps = (k1 - k0 + 2 + 3) & ~3;
    auto slot = [&](int k) { return (k - k0 + RING) & (RING - 1); };
    // the planes touched lie in [k0 - 2, k1 + 9] and nz >= 16
    auto modz = [&](int k) { return k < 0 ? k + nz : (k >= nz ? k - nz : k); };

    const T half = (T)0.5;
    for (int t = threadIdx.x; t < QX; t += NT) {
        const int gx = wrapi(tx0 + t - 1, nx);
        sTx[t] = half * L.a[0].ip[gx];
        sTx[QX + t] = half * L.a[0].im[gx];
    }
    for (int t = threadIdx.x; t < QY; t += NT) {
        const int gy = clampi(ty0 + t - 1, ny);
        sTy[t] = half * L.a[1].ip[gy];
        sTy[QY + t] = half * L.a[1].im[gy];
    }
    // (vector loads of these inside the plane loop would wait behind the
    // prefetch of the next planes)
    for (int t = threadIdx.x; t < nsteps + 1; t += NT) {
        const int kw = modz(k0 - 1 + t);
        sTz[t] = half * L.a[2].ip[kw];
        sTz[kZT + t] = half * L.a[2].im[kw];
    }

    // in-plane byte offsets of the cells this thread loads (fixed for the
    // chunk; unsigned, so a load is a uniform plane base plus this offset)
    unsigned offp[Sh::NP], offq[Sh::NQ];
#pragma unroll
    for (int m = 0; m < Sh::NP; ++m) {
        const int t = min((int)threadIdx.x + m * NT, PS - 1);
        const int yy = t / PX, xx = t - yy * PX;
        offp[m] = (unsigned)(nx * clampi(ty0 + yy - 2, ny) + wrapi(tx0 + xx - 2, nx)) * (unsigned)sizeof(T);
    }
#pragma unroll
    for (int m = 0; m < Sh::NQ; ++m) {
        const int t = min((int)threadIdx.x + m * NT, QS - 1);
        const int yy = t / QX, xx = t - yy * QX;
        offq[m] = (unsigned)(nx * clampi(ty0 + yy - 1, ny) + wrapi(tx0 + xx - 1, nx)) * (unsigned)sizeof(TQ);
    }
    const size_t plane_sz = (size_t)nx * ny;
    const size_t level_sz = plane_sz * nz;
    const __amdgpu_buffer_rsrc_t rs_p = plane_rsrc(pin, level_sz * sizeof(T));
    const __amdgpu_buffer_rsrc_t rs_b = plane_rsrc(beta, level_sz * sizeof(TB));
    const __amdgpu_buffer_rsrc_t rs_q = plane_rsrc(q, level_sz * sizeof(TQ));
    // this thread's tile cell pair and the column used at steps of each parity
    const int row = threadIdx.x / (TX / 2), h = threadIdx.x - row * (TX / 2);
    const int gy = ty0 + row;
    const bool wall_s = gy == 0, wall_n = gy == ny - 1;
    const size_t pair_off = (size_t)nx * gy + tx0 + 2 * h;

    // planes of p and beta at kp, of q at kp - 1, into registers.  The last
    // planes a chunk needs are p and beta at k1 + 1 and q at k1; a fetch for a
    // later plane step (the prefetch of the last steps, the red-only steps
    // that round the march up to a group of 4) loads that plane again, a
    // cache hit, where a load of the next planes would cost HBM traffic for
    // values no cell uses.
    const int klast = k1 + 1;
    auto fetch_pb = [&](T(&rp)[Sh::NP], T(&rb)[Sh::NP], int kp) {
        kp = min(kp, klast);
        const unsigned so = (unsigned)(plane_sz * modz(kp) * sizeof(T));
        const unsigned sob = (unsigned)(plane_sz * modz(kp) * sizeof(TB));
#pragma unroll
        for (int m = 0; m < Sh::NP; ++m) {
            if (!FIRST) rp[m] = buf_load<T>(rs_p, offp[m], so);
            rb[m] = (T)buf_load<TB>(rs_b, offp[m] / (unsigned)sizeof(T) * (unsigned)sizeof(TB), sob);
        }
    };
    // ... and, for DOTS, r and qv of this thread's pair on plane kp - 2 (the
    // black plane of the step that stashes these registers)
    auto fetch = [&](T(&rp)[Sh::NP], T(&rb)[Sh::NP], T(&rq)[Sh::NQ], double2& dr, double2& dq, int kp) {
        fetch_pb(rp, rb, kp);
        kp = min(kp, klast);
        const unsigned so = (unsigned)(plane_sz * modz(kp - 1) * sizeof(TQ));
#pragma unroll
        for (int m = 0; m < Sh::NQ; ++m) rq[m] = (T)buf_load<TQ>(rs_q, offq[m], so);
        if (DOTS) {
            const size_t o = plane_sz * modz(kp - 2) + pair_off;
            dr = *reinterpret_cast<const double2*>(dots.r + o);
            if (!dots.init) dq = *reinterpret_cast<const double2*>(dots.qv + o);
        }
    };
    auto stash = [&](const T(&rp)[Sh::NP], const T(&rb)[Sh::NP], int sl) {
        if (!FIRST) stash_plane<NT, T, Sh::NP>(rp, sP + sl * PS, PS);
        stash_plane<NT, T, Sh::NP>(rb, sB + sl * PS, PS);
    };

    // prologue: planes k0-2 and k0-1 of p and beta into LDS; the next two
    // planes into the two register sets (loads run two plane steps ahead)
    {
        T rp[Sh::NP], rb[Sh::NP];
        fetch_pb(rp, rb, k0 - 2);
        stash(rp, rb, slot(k0 - 2));
        fetch_pb(rp, rb, k0 - 1);
        stash(rp, rb, slot(k0 - 1));
    }
    // PD register sets: the loads of a plane are issued PD steps before the
    // step that stashes them
    T rps[PD][Sh::NP], rbs[PD][Sh::NP], rqs[PD][Sh::NQ];
    double2 drs[PD], dqs[PD];
#pragma unroll
    for (int u = 0; u < PD; ++u) {
        drs[u] = double2{0.0, 0.0};
        dqs[u] = double2{0.0, 0.0};
        fetch(rps[u], rbs[u], rqs[u], drs[u], dqs[u], k0 + u);
        // keep each set's loads ahead of the next set's: the wait before a
        // plane step then covers only the loads of the set it stashes
        __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();  // tables and planes k0-2, k0-1 in LDS

    const T ipy = sTy[row + 1], imy = sTy[QY + row + 1];

    // column of the steps with the parity of k: red (gx + gy + k) odd (nz is
    // even, so the parity of a plane index is that of its periodic image)
    auto colx = [&](int k) { return 2 * h + ((tx0 + gy + k + 1) & 1); };
    ColHist<T> hA, hB;  // steps k0-1, k0+1, ... and k0, k0+2, ...
    {
        const int xa = colx(k0 - 1), xb = colx(k0);
        hA.bf = sB[slot(k0 - 2) * PS + (row + 2) * PX + xa + 2];
        hB.bf = sB[slot(k0 - 1) * PS + (row + 2) * PX + xb + 2];
        hA.pf = FIRST ? (T)0 : sP[(FIRST ? 0 : slot(k0 - 2)) * PS + (row + 2) * PX + xa + 2];
        hB.pf = FIRST ? (T)0 : sP[(FIRST ? 0 : slot(k0 - 1)) * PS + (row + 2) * PX + xb + 2];
        hA.bc = hB.bc = hA.r = hB.r = (T)0;  // first read two steps later
    }

    // S: the ring slot of plane k (a constant of the unrolled step)
    auto step = [&](int k, int S, T(&rp)[Sh::NP], T(&rb)[Sh::NP], T(&rq)[Sh::NQ], double2& dr, double2& dq,
                    ColHist<T>& H) {
        const int Sp = (S + 1) & (RING - 1), Sm = (S + RING - 1) & (RING - 1);
        const int SpP = FIRST ? 0 : Sp, SP0 = FIRST ? 0 : S, SmP = FIRST ? 0 : Sm;
        // planes k+1 (p, beta) and k (q) into LDS, then start loading planes
        // k+PD+1 and k+PD into the same registers (past the chunk end: unused)
        stash(rp, rb, Sp);
        stash_plane<NT, T, Sh::NQ>(rq, sQ + S * QS, QS);
        const double2 r_pair = dr, qv_pair = dq;  // plane k-1
        fetch(rp, rb, rq, dr, dq, k + PD + 1);
        __syncthreads();

        const T* B0 = sB + S * PS;
        const T* Bp = sB + Sp * PS;
        const T* Bm = sB + Sm * PS;
        const T* P0 = sP + SP0 * PS;
        const T* Pp = sP + SpP * PS;
        const T* Pm = sP + SmP * PS;
        const T* Q0 = sQ + S * QS;
        T* R0 = sR + (S & 1) * QS;

        // ---- red cell of plane k at this thread's column
        const int xr = colx(k);
        const int ipc = (row + 2) * PX + xr + 2;
        const int iqc = (row + 1) * QX + xr + 1;
        const T ipx = sTx[xr + 1], imx = sTx[QX + xr + 1];
        const T p_self = H.pf;  // p_old(k-1) at this column
        T red_c, b_c, b_f;
        {
            const T azp = sTz[k - k0 + 1], azm = sTz[kZT + k - k0 + 1];
            const T bc = B0[ipc];
            const T bf = Bp[ipc];
            const T aR = (B0[ipc + 1] + bc) * ipx;
            const T aL = (bc + B0[ipc - 1]) * imx;
            const T aT = (B0[ipc + PX] + bc) * ipy;
            const T aB = (bc + B0[ipc - PX]) * imy;
            const T aF = (bf + bc) * azp;
            const T aK = (bc + H.bf) * azm;
            const T den = aR + aL + aT + aB + aF + aK;
            const T qc = Q0[iqc];
            T num;
            T pf = (T)0;
            if (FIRST) {
                num = -qc;
            } else {
                // rows outside the walls hold the wall row itself: the
                // Neumann ghost of the reference equals the cell's own value
                pf = Pp[ipc];
                num = -qc + (aR * P0[ipc + 1] + aL * P0[ipc - 1]) + (aT * P0[ipc + PX] + aB * P0[ipc - PX]) +
                      (aF * pf + aK * H.pf);
            }
            red_c = smooth_div(num, den);
            R0[iqc] = red_c;
            b_c = bc;
            b_f = bf;
            H.pf = pf;
        }
        // ---- red cells of the ring around the tile
        for (int t = threadIdx.x; t < NRING; t += NT) {
            int qrow, xx;
            if (t < QX) {  // rows -1 and TY, every second cell
                qrow = t < QX / 2 ? 0 : QY - 1;
                const int hh = t < QX / 2 ? t : t - QX / 2;
                xx = 2 * hh + ((tx0 + ty0 + qrow - 1 + k) & 1);
            } else if (t < QX + TY / 2) {  // column -1, every second row
                xx = 0;
                qrow = 1 + 2 * (t - QX) + ((tx0 + ty0 + k) & 1);
            } else {  // column TX
                xx = QX - 1;
                qrow = 1 + 2 * (t - QX - TY / 2) + ((tx0 + TX + ty0 + k + 1) & 1);
            }
            const int gyr = ty0 + qrow - 1;
            if (gyr < 0 || gyr >= ny) continue;
            const int ip = (qrow + 1) * PX + xx + 1;
            const T bc = B0[ip];
            const T aR = (B0[ip + 1] + bc) * sTx[xx];
            const T aL = (bc + B0[ip - 1]) * sTx[QX + xx];
            const T aT = (B0[ip + PX] + bc) * sTy[qrow];
            const T aB = (bc + B0[ip - PX]) * sTy[QY + qrow];
            const T aF = (Bp[ip] + bc) * sTz[k - k0 + 1];
            const T aK = (bc + Bm[ip]) * sTz[kZT + k - k0 + 1];
            const T den = aR + aL + aT + aB + aF + aK;
            const T qc = Q0[qrow * QX + xx];
            T num;
            if (FIRST) {
                num = -qc;
            } else {
                num = -qc + (aR * P0[ip + 1] + aL * P0[ip - 1]) + (aT * P0[ip + PX] + aB * P0[ip - PX]) +
                      (aF * Pp[ip] + aK * Pm[ip]);
            }
            R0[qrow * QX + xx] = smooth_div(num, den);
        }
        __syncthreads();

        // ---- black cell of plane k-1 at the same column; write the pair
        if (k > k0 && k <= k1) {
            const int kb = k - 1;
            const T azp = sTz[kb - k0 + 1], azm = sTz[kZT + kb - k0 + 1];
            const T* B1 = sB + Sm * PS;
            const T* Q1 = sQ + Sm * QS;
            const T* R1 = sR + (Sm & 1) * QS;
            const T bc = H.bf;  // beta(k-1) at this column
            const T aR = (B1[ipc + 1] + bc) * ipx;
            const T aL = (bc + B1[ipc - 1]) * imx;
            const T aT = (B1[ipc + PX] + bc) * ipy;
            const T aB = (bc + B1[ipc - PX]) * imy;
            const T aF = (b_c + bc) * azp;  // beta(k)
            const T aK = (bc + H.bc) * azm; // beta(k-2)
            const T den = aR + aL + aT + aB + aF + aK;
            const T self = FIRST ? (T)0 : p_self;
            const T pn = wall_n ? self : R1[iqc + QX];
            const T ps = wall_s ? self : R1[iqc - QX];
            const T num = -Q1[iqc] + (aR * R1[iqc + 1] + aL * R1[iqc - 1]) + (aT * pn + aB * ps) +
                          (aF * red_c + aK * H.r);
            const T vb = smooth_div(num, den);
            const int par = xr - 2 * h;
            const T vr = R1[iqc + 1 - 2 * par];  // the red cell sharing the aligned pair
            typename Vec2<T>::type v;
            v.x = par ? vr : vb;
            v.y = par ? vb : vr;
            *reinterpret_cast<typename Vec2<T>::type*>(pout + plane_sz * modz(kb) + pair_off) = v;
            if (DOTS) {  // the order of k_pcg_dots, cell by cell
                const double z0 = (double)v.x, z1 = (double)v.y;
                acc[0] += r_pair.x * z0;
                acc[2] += z0;
                acc[3] += r_pair.x;
                if (!dots.init) {
                    acc[1] += qv_pair.x * z0;
                    acc[4] += qv_pair.x;
                }
                acc[0] += r_pair.y * z1;
                acc[2] += z1;
                acc[3] += r_pair.y;
                if (!dots.init) {
                    acc[1] += qv_pair.y * z1;
                    acc[4] += qv_pair.y;
                }
            }
        }
        H.bc = b_c;
        H.bf = b_f;
        H.r = red_c;
    };

    // steps k0-1 .. in groups of 4 (slot of step k0-1+4m+u: (u + 3) & 3)
    for (int k = k0 - 1; k < k0 - 1 + nsteps; k += 4) {
#pragma unroll
        for (int u = 0; u < 4; ++u)
            step(k + u, (u + 3) & 3, rps[u % PD], rbs[u % PD], rqs[u % PD], drs[u % PD], dqs[u % PD],
                 (u & 1) ? hB : hA);
    }
    if (DOTS) block_partial<5>(acc, dots.red);
}

// One full red/black sweep of a level per launch (rbgs.f90:205-259) without any
// exchange between threads, out of place like k_sweep: a thread owns the red and the
// black cell of an x pair and computes from pin, beside its own red cell, the five
// other red cells its black cell reads -- seven cell updates instead of two, from 25
// values of beta, 19 of p and 7 of q that all load at once (the neighbours' loads hit
// in L1).  On small levels the time is the chain of one round of loads, two dependent
// updates and the launch itself; staging a brick in LDS added its index arithmetic, two
// barriers and the serial rounds of its cells.  Any even nx, nz; any ny.  Per launch,
// bricks -> this: FP32 196 K cells 6.7 -> 5.9 us, 25 K 6.3 -> 4.6; FP64 262 K 8.4 -> 7.5,
// 74 K 6.6 -> 5.5; two half-sweeps at 20 K (72x40x56's level 1) 8.1 -> 4.6.
// DOTS: the sums of k_pcg_dots as in k_sweep, one partial per workgroup.
template <class T, class TQ, bool FIRST, bool DOTS>
__global__ void __launch_bounds__(256)
    k_point_sweep(LevelDev<T> L, const T* __restrict__ beta, const TQ* __restrict__ q, const T* __restrict__ pin,
                  T* __restrict__ pout, uint32_t m_hx, uint32_t m_ny, int npairs, const int* done, SweepDots dots)
{
    if (done && *done) return;
    unsigned id = blockIdx.x, nblk = gridDim.x;  // consecutive blocks on one XCD
    if (FIRST && dots.fin.n) {
        if (id == 0) {
            fin_update(dots.fin);
            return;
        }
        --id, --nblk;
    }
    if ((nblk & 7u) == 0) id = (id & 7u) * (nblk >> 3) + (id >> 3);
    const int tp = (int)(id * 256u + threadIdx.x);
    const bool own = tp < npairs;  // (the last block's idle threads follow the last pair)
    const int t = own ? tp : npairs - 1;
    const int nx = L.nx, ny = L.ny, nz = L.nz;
    const int hx = nx >> 1;
    const int row = hx == 1 ? t : (int)__umulhi((uint32_t)t, m_hx), h = t - row * hx;
    const int k = ny == 1 ? row : (int)__umulhi((uint32_t)row, m_ny), j = row - k * ny;
    const int par = (j + k) & 1;  // offset of the black cell in the pair ((i + j + k) even)
    const int xb = 2 * h + par;
    const int e1 = xb + 1 < nx ? xb + 1 : 0, w1 = xb > 0 ? xb - 1 : nx - 1;
    const int e2 = e1 + 1 < nx ? e1 + 1 : 0, w2 = w1 > 0 ? w1 - 1 : nx - 1;
    const int jn = min(j + 1, ny - 1), js = max(j - 1, 0), jn2 = min(j + 2, ny - 1), js2 = max(j - 2, 0);
    const int kf = k + 1 < nz ? k + 1 : 0, kb = k > 0 ? k - 1 : nz - 1;
    const int kf2 = kf + 1 < nz ? kf + 1 : 0, kb2 = kb > 0 ? kb - 1 : nz - 1;
    auto rw = [&](int jj, int kk) { return nx * (jj + ny * kk); };
    const int rc = rw(j, k), rn = rw(jn, k), rs = rw(js, k), rf = rw(j, kf), rb = rw(j, kb);
    const int o_n2 = rw(jn2, k) + xb, o_s2 = rw(js2, k) + xb, o_f2 = rw(j, kf2) + xb, o_b2 = rw(j, kb2) + xb;
    const int o_nf = rw(jn, kf) + xb, o_nb = rw(jn, kb) + xb, o_sf = rw(js, kf) + xb, o_sb = rw(js, kb) + xb;

    // beta: row of the cell, the four rows beside it, the diagonals and second neighbours
    const T bw2 = beta[rc + w2], bw = beta[rc + w1], bc = beta[rc + xb], be = beta[rc + e1], be2 = beta[rc + e2];
    const T bnw = beta[rn + w1], bn = beta[rn + xb], bne = beta[rn + e1];
    const T bsw = beta[rs + w1], bs = beta[rs + xb], bse = beta[rs + e1];
    const T bfw = beta[rf + w1], bf = beta[rf + xb], bfe = beta[rf + e1];
    const T bbw = beta[rb + w1], bb = beta[rb + xb], bbe = beta[rb + e1];
    const T bn2 = beta[o_n2], bs2 = beta[o_s2], bf2 = beta[o_f2], bb2 = beta[o_b2];
    const T bnf = beta[o_nf], bnb = beta[o_nb], bsf = beta[o_sf], bsb = beta[o_sb];
    double2 dr = {0.0, 0.0}, dq = {0.0, 0.0};
    if (DOTS) {
        dr = *reinterpret_cast<const double2*>(dots.r + rc + 2 * h);
        if (!dots.init) dq = *reinterpret_cast<const double2*>(dots.qv + rc + 2 * h);
    }
    const T qc = (T)q[rc + xb], qe = (T)q[rc + e1], qw = (T)q[rc + w1], qn = (T)q[rn + xb], qs = (T)q[rs + xb],
            qf = (T)q[rf + xb], qb = (T)q[rb + xb];
    auto ld = [&](int o) { return FIRST ? (T)0 : pin[o]; };
    const T pc = ld(rc + xb), pw2 = ld(rc + w2), pe2 = ld(rc + e2);
    const T pnw = ld(rn + w1), pne = ld(rn + e1), psw = ld(rs + w1), pse = ld(rs + e1);
    const T pfw = ld(rf + w1), pfe = ld(rf + e1), pbw = ld(rb + w1), pbe = ld(rb + e1);
    const T pn2 = ld(o_n2), ps2 = ld(o_s2), pf2 = ld(o_f2), pb2 = ld(o_b2);
    const T pnf = ld(o_nf), pnb = ld(o_nb), psf = ld(o_sf), psb = ld(o_sb);
    // face factors times 1/2 (exact) at the cell and the two neighbours of each axis
    const T half = (T)0.5;
    const T xp = half * L.a[0].ip[xb], xm = half * L.a[0].im[xb];
    const T xpe = half * L.a[0].ip[e1], xme = half * L.a[0].im[e1], xpw = half * L.a[0].ip[w1], xmw = half * L.a[0].im[w1];
    const T yp = half * L.a[1].ip[j], ym = half * L.a[1].im[j];
    const T ypn = half * L.a[1].ip[jn], ymn = half * L.a[1].im[jn], yps = half * L.a[1].ip[js], yms = half * L.a[1].im[js];
    const T zp = half * L.a[2].ip[k], zm = half * L.a[2].im[k];
    const T zpf = half * L.a[2].ip[kf], zmf = half * L.a[2].im[kf], zpb = half * L.a[2].ip[kb], zmb = half * L.a[2].im[kb];

    // every load above before the arithmetic: the compiler otherwise saves registers by
    // loading in rounds that each wait (FP64, 74 K cells: 5.4 -> 4.9 us)
    __builtin_amdgcn_sched_barrier(0);

    const std::true_type red;
    // one update: centre beta, the six neighbours' beta and p
    auto update = [&](T qq, T c, T bE, T bW, T bN, T bS, T bF, T bB, T fxp, T fxm, T fyp, T fym, T fzp, T fzm, T pE, T pW,
                      T pN, T pS, T pF, T pB, auto red) {
        return smooth_cell<T, FIRST && decltype(red)::value>(
            qq, c, {bE, bW, bN, bS, bF, bB}, fxp, fxm, fyp, fym, fzp, fzm, {pE, pW, pN, pS, pF, pB});
    };
    const T re = update(qe, be, be2, bc, bne, bse, bfe, bbe, xpe, xme, yp, ym, zp, zm, pe2, pc, pne, pse, pfe, pbe, red);
    const T rwv = update(qw, bw, bc, bw2, bnw, bsw, bfw, bbw, xpw, xmw, yp, ym, zp, zm, pc, pw2, pnw, psw, pfw, pbw, red);
    const T rnv = update(qn, bn, bne, bnw, bn2, bc, bnf, bnb, xp, xm, ypn, ymn, zp, zm, pne, pnw, pn2, pc, pnf, pnb, red);
    const T rsv = update(qs, bs, bse, bsw, bc, bs2, bsf, bsb, xp, xm, yps, yms, zp, zm, pse, psw, pc, ps2, psf, psb, red);
    const T rfv = update(qf, bf, bfe, bfw, bnf, bsf, bf2, bc, xp, xm, yp, ym, zpf, zmf, pfe, pfw, pnf, psf, pf2, pc, red);
    const T rbv = update(qb, bb, bbe, bbw, bnb, bsb, bc, bb2, xp, xm, yp, ym, zpb, zmb, pbe, pbw, pnb, psb, pc, pb2, red);
    // the black cell: a wall's ghost is its own value before the sweep
    const T vb = update(qc, bc, be, bw, bn, bs, bf, bb, xp, xm, yp, ym, zp, zm, re, rwv, j + 1 < ny ? rnv : pc,
                        j > 0 ? rsv : pc, rfv, rbv, std::false_type());
    typename Vec2<T>::type v;
    v.x = par ? rwv : vb;
    v.y = par ? vb : re;
    if (own) *reinterpret_cast<typename Vec2<T>::type*>(pout + rc + 2 * h) = v;
    if (DOTS) {  // the order of k_pcg_dots, cell by cell
        double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
        if (own) {
            const double z0 = (double)v.x, z1 = (double)v.y;
            acc[0] = dr.x * z0 + dr.y * z1;
            acc[2] = z0 + z1;
            acc[3] = dr.x + dr.y;
            if (!dots.init) {
                acc[1] = dq.x * z0 + dq.y * z1;
                acc[4] = dq.x + dq.y;
            }
        }
        block_partial<5>(acc, dots.red);
    }
}

// The same sweep as a march along z with whole rows in a wavefront: a lane holds four
// cells along x (two red, two black), lr = nx / 4 lanes a row, rw = 64 / lr rows a
// wavefront, NW wavefronts a workgroup.  At step m a lane updates its red cells of plane
// m and then its black cells of plane m - 1, whose red neighbours are its own of planes
// m - 2, m - 1, m (registers), those of the lanes beside it (shuffles: the row's ends
// meet, so the periodic image is in the wavefront too) and those of the rows beside it
// (LDS, two slots, one barrier per step).  Every array is read as 4-cell vectors straight
// into registers, each plane's loads issued a step before their use; the rows beside a
// lane's own come from L1.  The rows of a wavefront have one parity of j, so which of the
// four cells are red is uniform and known in each unrolled step: nothing is selected per
// lane.  The red cells of the rows before and after the tile are recomputed, each plane
// by two wavefronts that own none.  x and z are uniform axes (validate_grid): one face
// factor each.
//
// Against k_sweep: 150 instead of 210 vector instructions per 4 cells, a fifth of the LDS
// traffic, no staging.  Per launch, plain / with the dots / from zero: 128x96x128 FP32
// 14.8 / - / 14.7 -> 8.6 / - / 9.1; 128^3 FP64 28.8 / 36 / 20.7 -> 19 / 26 / 13.7; with bf16
// q and beta 256x192x256 46.2 / - / 44.6 -> 35 / - / 33 (30 / 20 at the copy rate).  A march
// of the same steps without LDS (the neighbours' red cells recomputed) took twice as long,
// one with a lane per pair of cells 1.7 times: their loads of single cells strided the
// L1.  More wavefronts per CU (a bound on registers) spilled and lost; FP64, twice the
// registers, runs best with two row wavefronts.
template <class TS>
struct Quad {
    TS v[4];
};
template <>
struct alignas(8) Quad<bf16s> {
    bf16s v[4];
};
template <>
struct alignas(16) Quad<float> {
    float v[4];
};
template <>
struct alignas(8) Quad<double> {  // (a caller's array need only be aligned to its elements)
    double v[4];
};

template <class TS>
__device__ __forceinline__ Quad<TS> load4(const TS* __restrict__ base, unsigned e)
{
    return *reinterpret_cast<const Quad<TS>*>(reinterpret_cast<const char*>(base) + e * (unsigned)sizeof(TS));
}
template <class T, class TS>
__device__ __forceinline__ void widen(T (&d)[4], const Quad<TS>& x)
{
#pragma unroll
    for (int i = 0; i < 4; ++i) d[i] = (T)x.v[i];
}

// a lane's cells, and the rows beside them with q of its own: as loaded (in flight), and
// in the arithmetic's type
template <class T, class TB>
struct RawCentre {
    Quad<TB> b;
    Quad<T> p;
};
template <class T, class TQ, class TB>
struct RawSides {
    Quad<TB> bn, bs;
    Quad<T> pn, ps;
    Quad<TQ> q;
};
template <class T>
struct RowCentre {
    T b[4], p[4];
};

// wavefronts of a workgroup that own rows; two more compute the red cells of the rows
// before and after the tile
template <class T>
constexpr int row_waves() { return sizeof(T) == 4 ? 6 : 2; }

// TILES: rounded as k_sweep rounds with tiles of tx x ty cells (powers of two, tx >= 4):
// black cells take red neighbours across a tile's edge in their other rounding.
template <class T, class TQ, class TB, bool FIRST, bool DOTS, bool TILES>
__global__ void __launch_bounds__(64 * (row_waves<T>() + 2))
    k_row_sweep(LevelDev<T> L, const TB* __restrict__ beta, const TQ* __restrict__ q, const T* __restrict__ pin,
                T* __restrict__ pout, int kc, int lr, int rw, int ntiles, int tx, int ty, const int* done, SweepDots dots)
{
    constexpr int NW = row_waves<T>();
    constexpr int kSlot = 2 * 64 * (NW + 2);
    __shared__ T sR[(TILES ? 4 : 2) * kSlot];  // red values, rows -1 .. NW rw of 2 lr; as seen across a tile's edge
    if (done && *done) return;
    unsigned id = blockIdx.x, nblk = gridDim.x;  // consecutive tiles of a chunk on one XCD
    if (FIRST && dots.fin.n) {
        if (id == 0) {
            fin_update(dots.fin);
            return;
        }
        --id, --nblk;
    }
    if ((nblk & 7u) == 0) id = (id & 7u) * (nblk >> 3) + (id >> 3);
    const int nx = L.nx, ny = L.ny, nz = L.nz;
    const int k0 = (int)(id / (unsigned)ntiles) * kc, k1 = min(nz, k0 + kc);
    const int ty0 = (int)(id % (unsigned)ntiles) * NW * rw;
    const int lane = (int)threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), cls = wave & 1;
    // wavefronts NW, NW + 1: the row after the tile and the one before it
    const bool ring = wave >= NW;
    const int rows = ring ? 1 : rw;
    const int li = min(lane / lr, rows - 1), xl = lane / lr < rows ? lane - li * lr : 0;
    // row in the tile, of parity cls (ty0 and NW are even)
    const int r = ring ? (cls ? -1 : NW * rw) : 2 * ((wave >> 1) * rw + li) + cls;
    const bool put = lane / lr < rows && ty0 + r >= 0 && ty0 + r < ny;
    const bool own = put && !ring;
    const int j = min(max(ty0 + r, 0), ny - 1), jn = min(j + 1, ny - 1), js = max(j - 1, 0);
    const bool wall_n = j == ny - 1, wall_s = j == 0;
    const int left = li * lr + (xl > 0 ? xl - 1 : lr - 1), right = li * lr + (xl + 1 < lr ? xl + 1 : 0);
    const unsigned oc = (unsigned)(nx * j + 4 * xl), on = (unsigned)(nx * jn + 4 * xl), os = (unsigned)(nx * js + 4 * xl);
    // TILES: the row's neighbours and the lane's ends across a tile's edge
    const bool edge_n = TILES && ((j + 1) & (ty - 1)) == 0, edge_s = TILES && (j & (ty - 1)) == 0;
    const bool edge_e = TILES && ((4 * xl + 4) & (tx - 1)) == 0, edge_w = TILES && ((4 * xl) & (tx - 1)) == 0;
    const T half = (T)0.5;
    const T fx = half * L.a[0].ip[0], fz = half * L.a[2].ip[0];
    const T yp = half * L.a[1].ip[j], ym = half * L.a[1].im[j];
    const size_t plane = (size_t)nx * ny;
    auto wrap = [&](int k) { return k < 0 ? k + nz : (k >= nz ? k - nz : k); };
    auto load_c = [&](RawCentre<T, TB>& v, int k) __attribute__((always_inline)) {
        const size_t o = plane * (size_t)wrap(min(k, k1 + 1));  // (the last planes' prefetch: a plane already read)
        v.b = load4(beta + o, oc);
        if (!FIRST) v.p = load4(pin + o, oc);
    };
    auto load_s = [&](RawSides<T, TQ, TB>& v, int k) __attribute__((always_inline)) {
        const size_t o = plane * (size_t)wrap(min(k, k1 + 1));
        v.bn = load4(beta + o, on);
        v.bs = load4(beta + o, os);
        v.q = load4(q + o, oc);
        if (!FIRST) {
            v.pn = load4(pin + o, on);
            v.ps = load4(pin + o, os);
        }
    };
    auto take_c = [&](RowCentre<T>& d, const RawCentre<T, TB>& v) __attribute__((always_inline)) {
        widen(d.b, v.b);
        if (!FIRST) widen(d.p, v.p);
    };
    auto update = [&](T qq, T c, T bE, T bW, T bN, T bS, T bF, T bB, T fyp, T fym, T pE, T pW, T pN, T pS, T pF, T pB,
                      auto red) __attribute__((always_inline)) {
        return smooth_cell<T, FIRST && decltype(red)::value>(
            qq, c, {bE, bW, bN, bS, bF, bB}, fx, fx, fyp, fym, fz, fz, {pE, pW, pN, pS, pF, pB});
    };
    // the red cells of four (P: the parity of row + plane; red are 0, 2 if odd, 1, 3 if
    // even) from the rows about them; be, pe: the cell next to the four on the red side
    auto red2 = [&](auto par, T (&out)[2], T (&alt)[2], const T (&qq)[4], const T (&b)[4], const T (&bn)[4], const T (&bs)[4],
                    const T (&bf)[4], const T (&bk)[4], const T (&p)[4], const T (&pn)[4], const T (&ps)[4],
                    const T (&pf)[4], const T (&pk)[4], T be, T pe, T fyp, T fym) __attribute__((always_inline)) {
        constexpr int P = decltype(par)::value;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            constexpr int odd = P ? 0 : 1;
            const int e = 2 * i + odd;
            const T bE = e < 3 ? b[e < 3 ? e + 1 : 3] : be, bW = e > 0 ? b[e > 0 ? e - 1 : 0] : be;
            const T pE = e < 3 ? p[e < 3 ? e + 1 : 3] : pe, pW = e > 0 ? p[e > 0 ? e - 1 : 0] : pe;
            if constexpr (TILES)
                out[i] = smooth_red(qq[e], b[e], {bE, bW, bn[e], bs[e], bf[e], bk[e]}, fx, fx, fyp, fym, fz, fz,
                                    {pE, pW, pn[e], ps[e], pf[e], pk[e]}, alt[i]);
            else
                out[i] = update(qq[e], b[e], bE, bW, bn[e], bs[e], bf[e], bk[e], fyp, fym, pE, pW, pn[e], ps[e], pf[e],
                                pk[e], std::true_type());
        }
    };

    double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};  // DOTS: the sums of k_pcg_dots, one partial per workgroup
    RawCentre<T, TB> rc;       // plane m + 1 (at a step's start), then m + 2
    RawSides<T, TQ, TB> rs;    // plane m, then m + 1
    RowCentre<T> C[3];         // planes m - 1, m, m + 1
    T R2[2] = {(T)0, (T)0}, R1[2] = {(T)0, (T)0};  // new red values of planes m - 2, m - 1
    T X1 = (T)0;                                   // of plane m - 1, what the lane beside takes
    T kb[2] = {(T)0, (T)0};                        // beta of plane m - 2 behind the black cells of m - 1
    T kn[2] = {(T)0, (T)0}, ks[2] = {(T)0, (T)0}, kq[2] = {(T)0, (T)0};  // of plane m - 1: beta n, s and q there
    load_c(rc, k0 - 2);
    take_c(C[1], rc);
    load_c(rc, k0 - 1);
    take_c(C[2], rc);
    load_c(rc, k0);
    load_s(rs, k0 - 1);
    T* const mine = sR + (r + 1) * 2 * lr + 2 * xl;
    const int o_n = 2 * lr + (edge_n ? 2 * kSlot : 0), o_s = -2 * lr + (edge_s ? 2 * kSlot : 0);
    constexpr int kUnroll = sizeof(T) == 4 ? 4 : 2;  // steps per turn of the loop (registers)

    auto step = [&](auto par, int m, int sl) __attribute__((always_inline)) {
        constexpr int P = decltype(par)::value;        // parity of row + m
        constexpr int o_red = P ? 0 : 1, o_blk = P ? 1 : 0;  // of plane m; of plane m - 1 the other way round
        C[0] = C[1];
        C[1] = C[2];
        take_c(C[2], rc);
        const RowCentre<T>&Cm = C[0], &C0 = C[1], &Cp = C[2];
        T s_bn[4], s_bs[4], s_q[4], s_pn[4], s_ps[4];
        widen(s_bn, rs.bn);
        widen(s_bs, rs.bs);
        widen(s_q, rs.q);
        if (!FIRST) {
            widen(s_pn, rs.pn);
            widen(s_ps, rs.ps);
        }
        __builtin_amdgcn_sched_barrier(0);
        load_c(rc, m + 2);
        load_s(rs, m + 1);
        const bool black = m > k0;
        const size_t ob = plane * (size_t)wrap(m - 1) + oc;
        double dr[4] = {0.0, 0.0, 0.0, 0.0}, dq[4] = {0.0, 0.0, 0.0, 0.0};
        if (DOTS && black && !ring) {
            widen(dr, load4(dots.r + ob, 0));
            if (!dots.init) widen(dq, load4(dots.qv + ob, 0));
        }
        __builtin_amdgcn_sched_barrier(0);
        T R0[2], A0[2];
        {
            const T be = __shfl(C0.b[P ? 3 : 0], P ? left : right, 64);
            const T pe = FIRST ? (T)0 : __shfl(C0.p[P ? 3 : 0], P ? left : right, 64);
            red2(par, R0, A0, s_q, C0.b, s_bn, s_bs, Cp.b, Cm.b, C0.p, s_pn, s_ps, Cp.p, Cm.p, be, pe, yp, ym);
        }
        __syncthreads();  // plane m - 1 is in LDS, and plane m - 2's readers are done
        if (put) {
            mine[sl * kSlot] = R0[0];
            mine[sl * kSlot + 1] = R0[1];
            if (edge_n || edge_s) {
                mine[(2 + sl) * kSlot] = A0[0];
                mine[(2 + sl) * kSlot + 1] = A0[1];
            }
        }
        if (black && !ring) {
            // black cells of plane m - 1 at o_red + {0, 2} (the red positions of plane m)
            const T* at = mine + (sl ^ 1) * kSlot;
            const T be = __shfl(Cm.b[P ? 3 : 0], P ? left : right, 64);
            const T re = __shfl(X1, P ? left : right, 64);
            T vb[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int e = 2 * i + o_red;
                const T bE = e < 3 ? Cm.b[e < 3 ? e + 1 : 3] : be, bW = e > 0 ? Cm.b[e > 0 ? e - 1 : 0] : be;
                // its red neighbours along x: R1 holds the cells at o_blk + {0, 2}
                const T rE = P ? R1[i] : (i == 0 ? R1[1] : re), rW = P ? (i == 0 ? re : R1[0]) : R1[i];
                const T self = FIRST ? (T)0 : Cm.p[e];  // a wall's ghost: the cell before the sweep
                const T rn = wall_n ? self : at[o_n + i], rs = wall_s ? self : at[o_s + i];
                vb[i] = update(kq[i], Cm.b[e], bE, bW, kn[i], ks[i], C0.b[e], kb[i], yp, ym, rE, rW, rn, rs, R0[i],
                               R2[i], std::false_type());
            }
            if (own) {
                Quad<T> v;
                v.v[o_red] = vb[0], v.v[o_red + 2] = vb[1];
                v.v[o_blk] = R1[0], v.v[o_blk + 2] = R1[1];
                *reinterpret_cast<Quad<T>*>(pout + ob) = v;
                if (DOTS) {  // the order of k_pcg_dots, cell by cell
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const double z = (double)v.v[e];
                        acc[0] += dr[e] * z;
                        acc[2] += z;
                        acc[3] += dr[e];
                        if (!dots.init) {
                            acc[1] += dq[e] * z;
                            acc[4] += dq[e];
                        }
                    }
                }
            }
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int e = 2 * i + o_blk;  // plane m's black cells, the next step's
            kb[i] = Cm.b[e], kn[i] = s_bn[e], ks[i] = s_bs[e], kq[i] = s_q[e];
            R2[i] = R1[i], R1[i] = R0[i];
        }
        X1 = R0[P ? 0 : 1];  // (the next step takes the other side)
        if (P ? edge_w : edge_e) X1 = A0[P ? 0 : 1];
    };
    auto march = [&](auto p0) {  // p0: the parity of row + (k0 - 1)
        constexpr int A = decltype(p0)::value;
        const std::integral_constant<int, A> pa;
        const std::integral_constant<int, 1 - A> pb;
        for (int m = k0 - 1; m <= k1; m += kUnroll) {
#pragma unroll
            for (int u = 0; u < kUnroll; u += 2) {
                if (u > 0 && m + u > k1) break;
                step(pa, m + u, 0);
                if (m + u + 1 > k1) break;
                step(pb, m + u + 1, 1);
            }
        }
    };
    if ((cls + k0 - 1) & 1)
        march(std::integral_constant<int, 1>{});
    else
        march(std::integral_constant<int, 0>{});
    if (DOTS) block_partial<5>(acc, dots.red);
}

}  // namespace

template <class T>
bool point_supported(const LevelDev<T>& L)
{
    // pairs along x, the colours of a periodic z, indices of the launch and of its
    // divisions in 32 bits
    const uint64_t pairs = (uint64_t)(L.nx / 2) * L.ny * L.nz;
    return L.nx % 2 == 0 && L.nz % 2 == 0 && pairs * (uint64_t)std::max(L.nx / 2, L.ny) < ((uint64_t)1 << 32) &&
           pairs < ((uint64_t)1 << 30);
}

template <class T, class TQ>
int launch_point_sweep(const LevelDev<T>& L, const T* beta, const TQ* q, const T* pin, T* pout, bool first,
                       const int* done, void* stream, const SweepDots* dots, unsigned* nblocks_out)
{
    const bool wd = dots && dots->r;
    if (!point_supported(L) || (wd && first)) {
        set_error("launch_point_sweep: level %dx%dx%d not supported", L.nx, L.ny, L.nz);
        return TBFG_EINVAL;
    }
    auto magic = [](int d) { return d <= 1 ? 0u : (uint32_t)((((uint64_t)1 << 32) + (uint64_t)d - 1) / (uint64_t)d); };
    const int pairs = (L.nx / 2) * L.ny * L.nz;
    const unsigned nblocks = ceil_div((size_t)pairs, 256);
    if (wd && (size_t)nblocks * 5 > dots->capacity) {
        set_error("launch_point_sweep: %u workgroups exceed the reduction scratch", nblocks);
        return TBFG_EINVAL;
    }
    auto k = wd      ? k_point_sweep<T, TQ, false, true>
             : first ? k_point_sweep<T, TQ, true, false>
                     : k_point_sweep<T, TQ, false, false>;
    const unsigned fin = first && dots && dots->fin.n ? 1 : 0;
    hipLaunchKernelGGL(k, dim3(nblocks + fin), dim3(256), 0, (hipStream_t)stream, L, beta, q, pin, pout, magic(L.nx / 2),
                       magic(L.ny), pairs, done, dots ? *dots : SweepDots{});
    TBFG_HIP(hipGetLastError());
    if (nblocks_out) *nblocks_out = nblocks;
    return TBFG_OK;
}

template <class T>
bool row_supported(const LevelDev<T>& L)
{
    // rows of 4-cell lanes that fit a wavefront, the colours of a periodic z, the plane's
    // element offsets in 32-bit bytes
    return L.nx % 4 == 0 && L.nx >= 16 && L.nx <= 256 && L.nz % 2 == 0 && L.nz >= 4 &&
           (uint64_t)L.nx * L.ny < ((uint64_t)1 << 28);
}

struct SweepCfg {
    int tx, ty, nt;
};

template <class T, class TQ, class TB, bool FIRST, bool DOTS, bool TILES>
static int launch_row_form(const LevelDev<T>& L, const TB* beta, const TQ* q, const T* pin, T* pout, const int* done,
                           const SweepDots& dots, unsigned* nblocks_out, void* stream, const KernelEvents* kev,
                           const SweepCfg& c)
{
    // resident workgroups per CU and CU count, queried once (threads may race
    // to fill it; they store the same value)
    static std::atomic<int> occ{-1};
    auto k = k_row_sweep<T, TQ, TB, FIRST, DOTS, TILES>;
    int o = occ.load(std::memory_order_acquire);
    if (o < 0) {
        int dev = 0, ncu = 0, nb = 0;
        TBFG_HIP(hipGetDevice(&dev));
        TBFG_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
        TBFG_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k, 64 * (row_waves<T>() + 2), 0));
        o = (nb < 1 ? 1 : nb) * (ncu > 0 ? ncu : 256);
        occ.store(o, std::memory_order_release);
    }
    // one resident round of workgroups (a second, partly filled one costs as much as a
    // full one), chunks of at least 4 planes
    const int lr = L.nx / 4, rw = 64 / lr;
    const int ntiles = (int)ceil_div(L.ny, row_waves<T>() * rw);
    const int chunks = std::max(1, std::min(L.nz / 4, o / ntiles));
    int kc = (L.nz + chunks - 1) / chunks;
    const unsigned nblocks = (unsigned)ntiles * ceil_div(L.nz, kc);
    if (DOTS && (size_t)nblocks * 5 > dots.capacity) {
        set_error("launch_row_sweep: %u workgroups exceed the reduction scratch", nblocks);
        return TBFG_EINVAL;
    }
    const dim3 blk(64 * (row_waves<T>() + 2)), grd(nblocks + (FIRST && dots.fin.n ? 1 : 0));
    if (kev)
        hipExtLaunchKernelGGL(k, grd, blk, 0, (hipStream_t)stream, kev->start, kev->stop, 0, L, beta, q, pin,
                              pout, kc, lr, rw, ntiles, c.tx, c.ty, done, dots);
    else
        hipLaunchKernelGGL(k, grd, blk, 0, (hipStream_t)stream, L, beta, q, pin, pout, kc, lr, rw, ntiles, c.tx,
                           c.ty, done, dots);
    TBFG_HIP(hipGetLastError());
    if (nblocks_out) *nblocks_out = nblocks;
    return TBFG_OK;
}

// tile shapes with an instantiated kernel, in order of preference: in FP32
// the plain sweep runs fastest on 32x16 tiles (a smaller ring per cell), the
// sweep from zero and the one with the dot products on 64x8 (measured)
constexpr SweepCfg kShapesF[] = {{64, 8, 256}, {32, 16, 256}, {64, 16, 512}, {32, 8, 128}};
constexpr SweepCfg kShapesFPlain[] = {{32, 16, 256}, {64, 8, 256}, {64, 16, 512}, {32, 8, 128}};
constexpr SweepCfg kShapesD[] = {{64, 4, 128}, {64, 8, 256}, {32, 8, 128}};

// tuned (optional): whether TBFG_SWEEP_SHAPE or the tuning table names the shape
template <class T>
static bool pick_shape(const LevelDev<T>& L, SweepCfg& out, bool plain = false, bool* tuned_out = nullptr)
{
    if (tuned_out) *tuned_out = false;
    // nz even (the colour of a plane is its index's parity), nz >= 16 (a
    // chunk's plane steps wrap around z at most once); the level's arrays
    // addressable by 32-bit buffer offsets (< 2 GiB)
    if (L.nz < 16 || L.nz % 2 != 0 || L.ny % 2 != 0) return false;
    if ((size_t)L.nx * L.ny * L.nz * sizeof(T) >= ((size_t)1 << 31)) return false;
    const SweepCfg* tab = sizeof(T) == 4 ? (plain ? kShapesFPlain : kShapesF) : kShapesD;
    const int n = sizeof(T) == 4 ? (int)(sizeof kShapesF / sizeof kShapesF[0]) : (int)(sizeof kShapesD / sizeof kShapesD[0]);
    int want_tx = 0, want_ty = 0, want_nt = 0;
    int tuned[3];
    if (const char* e = std::getenv("TBFG_SWEEP_SHAPE"))
        std::sscanf(e, "%dx%dx%d", &want_tx, &want_ty, &want_nt);
    else if (tune_lookup(plain ? TBFG_TUNE_SWEEP : TBFG_TUNE_SWEEP_EDGE, L.nx, L.ny, L.nz, (int)sizeof(T), tuned)) {
        want_tx = tuned[0];
        want_ty = tuned[1];
        want_nt = tuned[2];
    }
    for (int pass = 0; pass < 2; ++pass)
        for (int i = 0; i < n; ++i) {
            const SweepCfg c = tab[i];
            if (pass == 0 && !(c.tx == want_tx && c.ty == want_ty && c.nt == want_nt)) continue;
            if (L.nx % c.tx == 0 && L.ny % c.ty == 0) {
                out = c;
                if (tuned_out) *tuned_out = pass == 0;
                return true;
            }
        }
    return false;
}

template <class T>
bool sweep_supported(const LevelDev<T>& L)
{
    SweepCfg c;
    return pick_shape(L, c);
}
template <class T>
bool sweep_named(const LevelDev<T>& L, bool plain)
{
    SweepCfg c;
    bool tuned = false;
    return pick_shape(L, c, plain, &tuned) && tuned;
}

template <class T, class TQ, class TB>
int launch_row_sweep(const LevelDev<T>& L, const TB* beta, const TQ* q, const T* pin, T* pout, bool first, bool tiles,
                     const int* done, void* stream, const SweepDots* dots, unsigned* nblocks_out,
                     const KernelEvents* kev)
{
    SweepCfg c{0, 0, 0};
    if (!row_supported(L) || (dots && dots->r && first) || (tiles && ((dots && dots->r) || !pick_shape(L, c, !first)))) {
        set_error("launch_row_sweep: level %dx%dx%d not supported", L.nx, L.ny, L.nz);
        return TBFG_EINVAL;
    }
    const SweepDots none{};
    auto go = [&](auto f, auto d, auto t) {
        return launch_row_form<T, TQ, TB, decltype(f)::value, decltype(d)::value, decltype(t)::value>(
            L, beta, q, pin, pout, done, dots ? *dots : none, nblocks_out, stream, kev, c);
    };
    const std::true_type yes;
    const std::false_type no;
    if (first) return go(yes, no, no);  // (from zero: no z term, one rounding)
    if constexpr (sizeof(T) == 4)
        if (tiles) return go(no, no, yes);
    return dots ? go(no, yes, no) : go(no, no, no);
}

// prefetch distance in plane steps: 4 in FP32 on long chunks; 2 in FP64, with
// the dot products (registers) and on short chunks (whose steps would not
// fill a group of 4)
template <class T, bool DOTS>
constexpr int sweep_pd_max()
{
    return sizeof(T) == 4 && !DOTS ? 4 : 2;
}

template <class T, class TQ, class TB, int TX, int TY, int NT, bool FIRST, bool DOTS>
static int launch_sweep_shape(const LevelDev<T>& L, const TB* beta, const TQ* q, const T* pin, T* pout,
                              const int* done, const SweepDots& dots, unsigned* nblocks_out, void* stream,
                              const KernelEvents* kev)
{
    constexpr int pdm = sweep_pd_max<T, DOTS>();
    // resident workgroups per CU and CU count, queried once (threads may race
    // to fill it; they store the same value)
    static std::atomic<int64_t> occ{-1};
    int64_t o = occ.load(std::memory_order_acquire);
    if (o < 0) {
        int dev = 0, ncu_q = 0, nb = 0;
        TBFG_HIP(hipGetDevice(&dev));
        TBFG_HIP(hipDeviceGetAttribute(&ncu_q, hipDeviceAttributeMultiprocessorCount, dev));
        TBFG_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_sweep<T, TQ, TB, TX, TY, NT, FIRST, DOTS, pdm>, NT, 0));
        o = ((int64_t)(nb < 1 ? 1 : nb) << 32) | (uint32_t)ncu_q;
        occ.store(o, std::memory_order_release);
    }
    const int per_cu = (int)(o >> 32), ncu = (int)(o & 0xffffffff);
    const int tiles_x = L.nx / TX;
    const int tiles_y = L.ny / TY;
    const int ntiles = tiles_x * tiles_y;
    // one resident wave of workgroups, chunks of at least 4 planes
    const int target = per_cu * (ncu > 0 ? ncu : 256);
    int chunks = (target + ntiles - 1) / ntiles;
    int kc = (L.nz + chunks - 1) / chunks;
    // kc + 2 plane steps run in groups of 4: kc = 4m + 2, from 6 to kSweepMaxChunk
    if (const char* e = std::getenv("TBFG_SWEEP_KC")) kc = std::atoi(e);  // A/B switch (planes per chunk)
    kc = ((kc + 2 + 3) / 4) * 4 - 2;
    if (kc < 6) kc = 6;
    if (kc > kSweepMaxChunk) kc = kSweepMaxChunk;
    const int pd = (pdm == 4 && kc >= 16) ? 4 : 2;
    chunks = (L.nz + kc - 1) / kc;
    const unsigned nblocks = (unsigned)ntiles * (unsigned)chunks;
    if (DOTS && (size_t)nblocks * 5 > dots.capacity) {
        set_error("launch_sweep: %u workgroups exceed the reduction scratch", nblocks);
        return TBFG_EINVAL;
    }
    auto k = pd == 4 ? k_sweep<T, TQ, TB, TX, TY, NT, FIRST, DOTS, pdm> : k_sweep<T, TQ, TB, TX, TY, NT, FIRST, DOTS, 2>;
    if (kev)
        hipExtLaunchKernelGGL(k, dim3(nblocks), dim3(NT), 0, (hipStream_t)stream, kev->start, kev->stop, 0, L, beta,
                              q, pin, pout, kc, tiles_x, ntiles, done, dots);
    else
        hipLaunchKernelGGL(k, dim3(nblocks), dim3(NT), 0, (hipStream_t)stream, L, beta, q, pin, pout, kc, tiles_x,
                           ntiles, done, dots);
    TBFG_HIP(hipGetLastError());
    if (nblocks_out) *nblocks_out = nblocks;
    return TBFG_OK;
}

template <class T, class TQ, class TB, int TX, int TY, int NT>
static int launch_sweep_first(const LevelDev<T>& L, const TB* beta, const TQ* q, const T* pin, T* pout, bool first,
                              const int* done, const SweepDots* dots, unsigned* nblocks_out, void* stream,
                              const KernelEvents* kev)
{
    const SweepDots none{};
    if (dots)  // the dot products follow a post-smoothing sweep, never the first
        return launch_sweep_shape<T, TQ, TB, TX, TY, NT, false, true>(L, beta, q, pin, pout, done, *dots, nblocks_out,
                                                                  stream, kev);
    return first ? launch_sweep_shape<T, TQ, TB, TX, TY, NT, true, false>(L, beta, q, pin, pout, done, none,
                                                                      nblocks_out, stream, kev)
                 : launch_sweep_shape<T, TQ, TB, TX, TY, NT, false, false>(L, beta, q, pin, pout, done, none,
                                                                       nblocks_out, stream, kev);
}

template <class T, class TQ, class TB>
int launch_sweep(const LevelDev<T>& L, const TB* beta, const TQ* q, const T* pin, T* pout, bool first,
                 const int* done, void* stream, const SweepDots* dots, unsigned* nblocks_out,
                 const KernelEvents* kev)
{
    if (dots && first) {
        set_error("launch_sweep: the fused dot products need a sweep from a non-zero start");
        return TBFG_EINVAL;
    }
    SweepCfg c;
    if (!pick_shape(L, c, !first && !dots)) {
        set_error("launch_sweep: level %dx%dx%d not supported", L.nx, L.ny, L.nz);
        return TBFG_EINVAL;
    }
#define TBFG_SWEEP_CASE(X, Y, N)                                                             \
    if (c.tx == X && c.ty == Y && c.nt == N)                                                \
        return launch_sweep_first<T, TQ, TB, X, Y, N>(L, beta, q, pin, pout, first, done, dots, nblocks_out, stream, kev);
    if constexpr (sizeof(T) == 4) {
        TBFG_SWEEP_CASE(64, 8, 256)
        TBFG_SWEEP_CASE(64, 16, 512)
        TBFG_SWEEP_CASE(32, 16, 256)
        TBFG_SWEEP_CASE(32, 8, 128)
    } else {
        TBFG_SWEEP_CASE(64, 4, 128)
        TBFG_SWEEP_CASE(64, 8, 256)
        TBFG_SWEEP_CASE(32, 8, 128)
    }
#undef TBFG_SWEEP_CASE
    set_error("launch_sweep: no kernel for shape %dx%dx%d", c.tx, c.ty, c.nt);
    return TBFG_EINVAL;
}

template bool row_supported<float>(const LevelDev<float>&);
template bool row_supported<double>(const LevelDev<double>&);
template int launch_row_sweep<float, float, float>(const LevelDev<float>&, const float*, const float*, const float*, float*, bool, bool,
                                             const int*, void*, const SweepDots*, unsigned*, const KernelEvents*);
template int launch_row_sweep<float, bf16s, bf16s>(const LevelDev<float>&, const bf16s*, const bf16s*, const float*, float*,
                                                   bool, bool, const int*, void*, const SweepDots*, unsigned*,
                                                   const KernelEvents*);
template int launch_row_sweep<double, double, double>(const LevelDev<double>&, const double*, const double*, const double*, double*, bool, bool,
                                             const int*, void*, const SweepDots*, unsigned*, const KernelEvents*);
template bool point_supported<float>(const LevelDev<float>&);
template bool point_supported<double>(const LevelDev<double>&);
template int launch_point_sweep<float, float>(const LevelDev<float>&, const float*, const float*, const float*,
                                              float*, bool, const int*, void*, const SweepDots*, unsigned*);
template int launch_point_sweep<double, double>(const LevelDev<double>&, const double*, const double*, const double*,
                                                double*, bool, const int*, void*, const SweepDots*, unsigned*);
template bool sweep_supported<float>(const LevelDev<float>&);
template bool sweep_supported<double>(const LevelDev<double>&);
template bool sweep_named<float>(const LevelDev<float>&, bool);
template bool sweep_named<double>(const LevelDev<double>&, bool);
template int launch_sweep<float, float, float>(const LevelDev<float>&, const float*, const float*, const float*,
                                               float*, bool, const int*, void*, const SweepDots*, unsigned*,
                                               const KernelEvents*);
template int launch_sweep<float, bf16s, bf16s>(const LevelDev<float>&, const bf16s*, const bf16s*, const float*,
                                               float*, bool, const int*, void*, const SweepDots*, unsigned*,
                                               const KernelEvents*);
template int launch_sweep<double, double, double>(const LevelDev<double>&, const double*, const double*, const double*,
                                          double*, bool, const int*, void*, const SweepDots*, unsigned*,
                                          const KernelEvents*);

}  // namespace tbfg
