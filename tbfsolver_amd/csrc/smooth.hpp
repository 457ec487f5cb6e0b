// smooth.hpp -- device arithmetic shared by the Gauss-Seidel kernels.
#pragma once
#include <hip/hip_runtime.h>

namespace tbfg {

// the smoother's division p = num / den (rbgs.f90:223-228): correctly rounded
// in FP64; in FP32 (the multigrid of mixed precision, a preconditioner) the
// hardware reciprocal (1 ulp) times num
template <class T>
__device__ __forceinline__ T smooth_div(T num, T den)
{
    return num / den;
}
template <>
__device__ __forceinline__ float smooth_div<float>(float num, float den)
{
    return num * __builtin_amdgcn_rcpf(den);
}

// The update of one cell from beta and p there and at its six neighbours and half the face
// factors (fx: towards E; gx: towards W).  The fused multiply-adds are written out and no
// others are formed, so that every kernel of the sweep rounds alike: with the compiler's
// own choice per kernel, a level of a few cells along two axes drifted by 1.4e-6 in FP32
// between two of them.  ZERO: all p are zero.
template <class T>
struct Around {
    T E, W, N, S, F, B;
};
template <class T>
struct CellSums {
    T den, xy, aF, aK;  // the sum of the six coefficients; -q and the x and y terms; z coefficients
};
template <class T>
__device__ __forceinline__ CellSums<T> smooth_sums(T q, T c, const Around<T>& b, T fx, T gx, T fy, T gy, T fz, T gz,
                                                   const Around<T>& p)
{
#pragma clang fp contract(off)
    const T sE = b.E + c, sW = c + b.W, sN = b.N + c, sS = c + b.S, sF = b.F + c, sB = c + b.B;
    const T aL = sW * gx;
    CellSums<T> r;
    r.den = __builtin_elementwise_fma(sE, fx, aL);
    r.den = __builtin_elementwise_fma(sN, fy, r.den);
    r.den = __builtin_elementwise_fma(sS, gy, r.den);
    r.den = __builtin_elementwise_fma(sF, fz, r.den);
    r.den = __builtin_elementwise_fma(sB, gz, r.den);
    r.xy = __builtin_elementwise_fma(sE * fx, p.E, aL * p.W) - q;
    r.xy = r.xy + __builtin_elementwise_fma(sN * fy, p.N, (sS * gy) * p.S);
    r.aF = sF * fz, r.aK = sB * gz;
    return r;
}
template <class T, bool ZERO>
__device__ __forceinline__ T smooth_cell(T q, T c, const Around<T>& b, T fx, T gx, T fy, T gy, T fz, T gz,
                                         const Around<T>& p)
{
#pragma clang fp contract(off)
    const CellSums<T> s = smooth_sums(q, c, b, fx, gx, fy, gy, fz, gz, p);
    return smooth_div(ZERO ? -q : s.xy + __builtin_elementwise_fma(s.aF, p.F, s.aK * p.B), s.den);
}
// A red cell as k_sweep's workgroups round it: the z term's product towards F rounded
// before the sum in the tile that owns the cell, that towards B (smooth_cell's) where a
// neighbouring tile recomputes it.
template <class T>
__device__ __forceinline__ T smooth_red(T q, T c, const Around<T>& b, T fx, T gx, T fy, T gy, T fz, T gz,
                                        const Around<T>& p, T& beside)
{
#pragma clang fp contract(off)
    const CellSums<T> s = smooth_sums(q, c, b, fx, gx, fy, gy, fz, gz, p);
    beside = smooth_div(s.xy + __builtin_elementwise_fma(s.aF, p.F, s.aK * p.B), s.den);
    return smooth_div(s.xy + __builtin_elementwise_fma(s.aK, p.B, s.aF * p.F), s.den);
}

}  // namespace tbfg
