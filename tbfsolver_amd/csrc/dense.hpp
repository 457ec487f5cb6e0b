// dense.hpp -- dense exact solve of one multigrid level (dense.hip).
#pragma once
#include "mg_kernels.hpp"

namespace tbfg {

// most cells of a level solved by launch_dense_solve
constexpr int kDenseDirectCells = 2048;

// doubles of scratch launch_dense_setup needs for a level of n cells
size_t dense_work_doubles(size_t n);

// G (n x n, row-major) with x = G q the exact solve of a level, from its beta and
// cell volumes; work: dense_work_doubles(n) doubles
template <class T>
int launch_dense_setup(const LevelDev<double>& L, const T* beta, const double* vol, double* work, double* G,
                       void* stream);

// x = G q by grid-wide kernels, and the solve's diagnostics into st
int launch_dense_solve(const LevelDev<double>& L, const double* beta, const double* vol, const double* G,
                       const double* q, double* x, PcgState* st, const int* done, void* stream);

}  // namespace tbfg
