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

// one exact solve of a level, for its diagnostics
struct DenseCheck {
    LevelDev<double> L;
    const double *beta, *vol, *q, *x;
};

// x = G q by grid-wide kernels; check: its diagnostics into st too
int launch_dense_solve(const DenseCheck& a, const double* G, double* x, bool check, PcgState* st, const int* done,
                       void* stream);

// launch_fin_dots, and beside it the diagnostics of the solve that launch_dense_solve left out
int launch_fin_dots_check(unsigned nblocks, size_t ncell, int init, PcgState* st, const Reducer& red,
                          int32_t* host_done, const DenseCheck& a, void* stream);

}  // namespace tbfg
