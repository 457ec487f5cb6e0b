// dense.hpp -- dense exact solve of one multigrid level (dense.hip).
#pragma once
#include "mg_kernels.hpp"

namespace tbfg {

// doubles of scratch launch_dense_setup needs for a level of n cells
size_t dense_work_doubles(size_t n);

// G (n x n, row-major) with x = G q the exact solve of a level, from its beta and
// cell volumes; work: dense_work_doubles(n) doubles
template <class T>
int launch_dense_setup(const LevelDev<double>& L, const T* beta, const double* vol, double* work, double* G,
                       void* stream);

}  // namespace tbfg
