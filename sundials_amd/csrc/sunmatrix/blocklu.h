// -----------------------------------------------------------------------------
// Interface between the block LU solver and its per-size kernels
// (blocklu_device.h, instantiated in the blocklu_inst_*.hip units).
// -----------------------------------------------------------------------------
#ifndef SUNAMD_BLOCKLU_H
#define SUNAMD_BLOCKLU_H

#include <hip/hip_runtime.h>

// the launches of one block size (getrf_scaled: null for the sizes between)
template <typename T>
struct LuLaunch
{
  void (*getrf)(int m, const double* A, T* F, int* piv, long nblocks, unsigned long long* info,
                hipStream_t s);
  void (*getrf_scaled)(bool save_src, const double* src, double c, double* save, double* scaled,
                       T* F, int* piv, long nblocks, unsigned long long* info, hipStream_t s);
  void (*getrs)(int m, const T* F, const int* piv, const double* b, double* x, long nblocks,
                double scale, hipStream_t s);
};

// Sizes with launches of their own, and the register-row lengths that serve the
// sizes between them with m at run time (the smallest one >= m).  At m = 21
// (FP32 factors, 50000 blocks) the run-time form factors in 0.10 ms and solves
// in 0.037 ms, where the LDS kernels it replaces, one lane working through the
// block, took 2.08 and 0.44 ms.
#define LU_SIZES(X) X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(12) X(16) X(24) X(32) X(48) X(64)
#define LU_ROW_SIZES(X) X(12) X(16) X(20) X(24) X(28) X(32) X(40) X(48) X(56) X(64)

template <int M, typename T>
const LuLaunch<T>* lu_size();
template <int M, typename T>
const LuLaunch<T>* lu_row_size();

#endif
