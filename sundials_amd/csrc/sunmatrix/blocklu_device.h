// -----------------------------------------------------------------------------
// Batched LU kernels of the block-diagonal solver (device part), instantiated
// per block size in the blocklu_inst_*.hip units.
//
// Kernel design (one m x m block per group of G = pow2ceil(m) lanes, 64/G
// blocks per 64-wide wavefront, four wavefronts per workgroup):
//   * lane r holds row r of its block in registers; every column load/store
//     is one coalesced 8*m-byte segment per block;
//   * partial pivoting without moving data: each lane carries the physical
//     row position it currently occupies; the pivot search (g_pivot) finds
//     the reference's "first maximum, strict >" choice in the reference's row
//     order, and a "swap" just exchanges two position tags;
//   * the pivot row is broadcast through LDS (lane reads when one block fills
//     the wavefront); each remaining row scales its multiplier with the
//     reciprocal of the pivot and subtracts pivot_row[j] * multiplier column
//     by column, skipping zero pivot-row entries -- the reference's exact
//     per-element operation sequence, so in FP64 the factors are
//     bit-identical;
//   * rows are written back to their final physical position, so the stored
//     factors and the pivot vector are those of the reference;
//   * GETRS permutes b through the pivot sequence, then runs the unit-lower
//     and upper sweeps, the solved entry broadcast by a lane read (groups of
//     64), an LDS shuffle (32) or DPP (up to 16), and each quotient formed
//     from the diagonal's reciprocal with two exact remainder steps
//     (correctly rounded, like the division).
// The common sizes up to 32 are compiled with m constant (of 48 and 64 the
// solve is); every other m up to 64 runs the kernel of the next size in a short
// list with m at run time.
// -----------------------------------------------------------------------------
#ifndef SUNAMD_BLOCKLU_DEVICE_H
#define SUNAMD_BLOCKLU_DEVICE_H

#include <hip/hip_runtime.h>

#include <climits>
#include <cmath>
#include <type_traits>

#include "../core/lane_ops.h"
#include "blocklu.h"

__host__ __device__ constexpr int pow2ceil(int m)
{
  return m <= 1 ? 1 : m <= 2 ? 2 : m <= 4 ? 4 : m <= 8 ? 8 : m <= 16 ? 16 : m <= 32 ? 32 : 64;
}

template <typename T>
__device__ __forceinline__ T to_t(double v)
{
  return (T)v;
}

// How k_getrf forms the matrix it factors from its source blocks A:
//   SRC_PLAIN  the blocks themselves;
//   SRC_SCALED c*A + I (SUNMatScaleAddI's per-element a*c, then +1 on the
//              diagonal), A read-only -- the Newton matrix from a saved
//              Jacobian without the copy and the scaling pass;
//   SRC_SAVE   as SRC_SCALED, and A's blocks are also written to `save` first
//              (a fresh Jacobian kept for later setups).
// With SRC_SCALED / SRC_SAVE and FP32 factors, `scaled` receives c*A + I in
// FP64 -- the matrix the separate copy / scale / factor calls leave in the
// solver's matrix; with FP64 factors the factors themselves go there.
enum GetrfSource
{
  SRC_PLAIN  = 0,
  SRC_SCALED = 1,
  SRC_SAVE   = 2
};

// wavefronts per workgroup of the register-row factorisation (each wavefront
// factors its own blocks; workgroups of several wavefronts put more blocks in
// flight per CU than one-wavefront workgroups)
#define LU_WAVES 4

// Factor nblocks m x m blocks in place (T = double) or into an FP32 factor
// array (T = float).  info receives min over failing blocks of
// (block*m + k + 1) for the first zero pivot k.  Lane r of a block's group of
// G = pow2ceil(M) lanes holds row r; the row swaps exchange position tags
// only, and the rows are written to their final positions at the end.
// RT: m is m_rt <= M at run time (M = the registers of a row; m_rt = M in the
// scaled forms), otherwise M.
//
// What bounds it (m = 32 FP64, 2^18 blocks: 4.3 GB, 0.73 ms at the copy
// rate): first VALU issue -- 6533 instructions per wavefront, 1.68 ms, with a
// (value, position) pair search of ~75 instructions per column and a compare
// and two selects per updated entry for the zero test.  The one-word search
// (lane_ops.h) takes ~20, the pivot's reciprocal is formed beside it, and the
// zero test is made once per column: each lane looks at one entry of the pivot
// row, and a column whose pivot row has no zero right of the pivot (all but
// the first few of a filled Newton matrix) runs without tests.  With 3151
// instructions it takes 1.48 ms, and no unit is full: the LDS data path is busy
// 59 % of the time and the vector units 53 %; a wavefront (3.9 per SIMD) waits
// for an operand 30 % of its time -- the search, publish and read chain of a
// column -- and 41 % for its turn to issue, mostly for an LDS instruction.
// Rows of more than 32 entries (one block per wavefront) take the pivot row
// from its lane entry by entry, and always in the RT form: its tests between
// the columns keep the compiler from collecting the scalars of many columns,
// which cost registers.  With m constant and 16 entries of the pivot row in
// scalar registers at a time, 64 x 64 FP64 blocks needed up to 256 registers
// (one wavefront per SIMD); now 144 to 161 (three).  40000 such blocks: set-up
// after a copy 2.55 -> 2.18 ms, one-pass set-up 3.44 -> 1.68 ms, FP32 1.21 ->
// 1.02 ms; 48 x 48 FP64 1.47 -> 1.27 and 1.22 -> 0.93 ms.
template <int M, typename T, int SRC = SRC_PLAIN, bool RT = false>
__global__ void __launch_bounds__(64 * LU_WAVES) k_getrf(const double* A, T* F /* may alias A */,
                                                         int* __restrict__ piv, long nblocks,
                                                         unsigned long long* info, int m_rt = M,
                                                         double c = 0.0, double* save = nullptr,
                                                         double* scaled = nullptr)
{
  using namespace sunamd_lane;
  constexpr int G   = pow2ceil(M);
  constexpr int BPW = 64 / G;
  // row stride: 16-byte aligned rows whose entries j fall in different banks
  constexpr int E16 = 16 / (int)sizeof(T);
  constexpr int PS  = (M + E16 - 1) / E16 * E16 + E16;
  __shared__ __align__(16) T prow[(G == 64) ? 1 : LU_WAVES * BPW][PS];
  __shared__ T pinv[LU_WAVES * BPW];
  __shared__ int ppos[LU_WAVES * BPW];

  const int m      = RT ? m_rt : M;
  const int lane   = threadIdx.x & 63;
  const int base   = lane / G * G;
  const int slot   = (threadIdx.x >> 6) * BPW + lane / G;
  const int r      = lane % G;
  const long blk   = (long)blockIdx.x * (LU_WAVES * BPW) + slot;
  const bool valid = (blk < nblocks) && (r < m);

  // every lane loads from inside block 0 or its own block (rows and columns
  // past m read row or column m-1), so the loads are unconditional and in
  // flight together; idle lanes' values are replaced afterwards (a load under
  // the validity test compiles to a branch per element, which waits for its
  // load wherever a conversion or the scaling follows it).  FP32 factors, and
  // the scaled forms at m > 32, take the FP64 source in chunks of 16 columns
  // (a scheduling barrier between chunks), so the loads in flight do not cost
  // the kernel its occupancy.
  const long blk_s = (blk < nblocks) ? blk : 0;
  const int r_s    = (r < m) ? r : m - 1;
  const double* Ab = A + blk_s * (long)m * m;
  const long o0    = blk * (long)m * m + r;
  constexpr int CH = ((sizeof(T) == 4 && M > 16) || (SRC != SRC_PLAIN && M > 32)) ? 16 : M;
  T a[M];
#pragma unroll
  for (int j0 = 0; j0 < M; j0 += CH)
  {
    double raw[CH];
#pragma unroll
    for (int q = 0; q < CH; q++)
    {
      if (j0 + q < M) { raw[q] = Ab[((RT && j0 + q >= m) ? m - 1 : j0 + q) * m + r_s]; }
    }
#pragma unroll
    for (int q = 0; q < CH; q++)
    {
      const int j = j0 + q;
      if (j >= M) { break; }
      if (SRC == SRC_PLAIN) { a[j] = valid ? to_t<T>(raw[q]) : (T)0; }
      else
      {
        double v = valid ? raw[q] : 0.0;
        if (SRC == SRC_SAVE && valid) { save[o0 + (long)j * M] = v; }
        v = v * c;
        if (j == r) { v = v + 1.0; }
        if (!std::is_same<T, double>::value && valid) { scaled[o0 + (long)j * M] = v; }
        a[j] = valid ? to_t<T>(v) : (T)0;
      }
      // the single-precision value is formed here, not where it is first
      // used (the compiler would otherwise keep the double until then)
      if constexpr (sizeof(T) == 4) { asm volatile("" : "+v"(a[j])); }
    }
    if constexpr (CH < M) { __builtin_amdgcn_sched_barrier(0); }
  }

  int pos  = r; // physical row currently held by this lane
  int myp  = 0; // pivot row chosen at step k == r
  int fail = 0;

  static_for<0, M>([&](auto kc) {
    constexpr int k = decltype(kc)::value;
    if (RT && k >= m) { return; }
    // every lane's 1 / a[k] is formed beside the pivot search, so the pivot
    // row's is ready when the search ends
    const T rk     = (T)1 / a[k];
    const bool win = g_pivot<G>(a[k], valid && pos >= k, pos, k, base);
    if constexpr (G == 64)
    {
      // one block per wavefront: the pivot row's lane is wavefront-uniform,
      // its entries are read straight from that lane's registers
      const int pl = __builtin_amdgcn_readfirstlane(__ffsll((long long)ballot(win)) - 1) & 63;
      const int bp = __builtin_amdgcn_readlane(pos, pl);
      const T pk   = readlane_d(a[k], pl);
      const T mult = readlane_d(rk, pl);
      if (r == k) { myp = bp; }
      if (pk == (T)0 && fail == 0) { fail = k + 1; }
      if (win) { pos = k; }
      else if (pos == k) { pos = bp; }
      const bool up = valid && pos > k && fail == 0;
      T l           = (T)0;
      if (up)
      {
        l    = a[k] * mult;
        a[k] = l;
      }
      // (in chunks so that columns past a run-time m are skipped)
      constexpr int PC = 16;
#pragma unroll
      for (int j0 = k + 1; j0 < M; j0 += PC)
      {
        if (RT && j0 >= m) { continue; }
#pragma unroll
        for (int q = 0; q < PC; q++)
        {
          if (j0 + q < M)
          {
            const T pj = readlane_d(a[j0 + q], pl);
            if (up && pj != (T)0) { a[j0 + q] = a[j0 + q] - pj * l; }
          }
        }
      }
    }
    else
    {
      // the pivot row (whose lane now takes position k) publishes columns
      // k+1..M-1, its reciprocal and the position it came from (with a flag
      // for a zero pivot)
      wave_sync();
      if (win)
      {
#pragma unroll
        for (int j = k + 1; j < M; j++) { prow[slot][j] = a[j]; }
        pinv[slot] = rk;
        ppos[slot] = pos | (a[k] == (T)0 ? 64 : 0);
      }
      wave_sync();
      const int pp = ppos[slot];
      const int bp = pp & 63;
      const T mult = pinv[slot];
      const T mine = prow[slot][r_s];
      if (r == k) { myp = bp; }
      if (pp >= 64 && fail == 0) { fail = k + 1; }
      if (win) { pos = k; }
      else if (pos == k) { pos = bp; }
      const bool up = valid && pos > k && fail == 0;
      const unsigned long long zeros = ballot(valid && r > k && mine == (T)0);
      T l = (T)0;
      if (up)
      {
        l    = a[k] * mult;
        a[k] = l;
      }
      if (zeros == 0)
      {
        if (up)
        {
#pragma unroll
          for (int j = k + 1; j < M; j++) { a[j] = a[j] - prow[slot][j] * l; }
        }
      }
      // (two ifs, not if / else: the entries then stay in their registers)
      if (zeros != 0)
      {
        // with two blocks in the wavefront, a column where both pivot rows
        // are zero is skipped on the scalar unit
        const unsigned both = (G == 32) ? (unsigned)zeros & (unsigned)(zeros >> 32) : 0u;
        if (up)
        {
#pragma unroll
          for (int j = k + 1; j < M; j++)
          {
            if ((both >> (j & 31)) & 1u) { continue; }
            const T pj = prow[slot][j];
            if (pj != (T)0) { a[j] = a[j] - pj * l; }
          }
        }
      }
    }
  });

  if (valid)
  {
    T* Fb = F + blk * (long)m * m;
#pragma unroll
    for (int j = 0; j < M; j++)
    {
      if (!RT || j < m) { Fb[j * m + pos] = a[j]; }
    }
    piv[blk * m + r] = myp;
    if (r == 0 && fail != 0)
    {
      atomicMin(info, (unsigned long long)(blk * m + fail));
    }
  }
}

// x = LU^{-1} P b per block (x may alias b); RT as in k_getrf.
//
// What bounds it: HBM for FP64 factors of common sizes (2^18 blocks of 32:
// 0.41 ms, 5.6 TB/s), VALU issue for FP32 factors and small blocks.  So a
// quotient is six instructions from the diagonal's reciprocal instead of a
// division in one lane, and b is loaded with the factors and permuted between
// lanes instead of a second, dependent load.
template <int M, typename T, bool RT = false>
__global__ void __launch_bounds__(64 * LU_WAVES) k_getrs(const T* __restrict__ F,
                                                         const int* __restrict__ piv,
                                                         const double* b, double* x, long nblocks,
                                                         double scale = 1.0, int m_rt = M)
{
  using namespace sunamd_lane;
  constexpr int G   = pow2ceil(M);
  constexpr int BPW = 64 / G;
  const int m       = RT ? m_rt : M;
  const int lane    = threadIdx.x & 63;
  const int r       = lane % G;
  const int base    = lane - r;
  const long blk    = ((long)blockIdx.x * LU_WAVES + (threadIdx.x >> 6)) * BPW + lane / G;
  const bool valid  = (blk < nblocks) && (r < m);

  // every lane loads from inside block 0 or its own block (rows and columns
  // past m read row or column m-1), so the loads are unconditional and all in
  // flight at once (a load under the validity test would be a branch per
  // element, and for FP32 factors the conversion made each one wait for its
  // load); idle lanes' results are not stored
  const long blk_s = (blk < nblocks) ? blk : 0;
  const int r_s    = (r < m) ? r : m - 1;
  const T* Fb      = F + blk_s * (long)m * m;
  const int* p     = piv + blk_s * m;
  int pv[M];
#pragma unroll
  for (int k = 0; k < M; k++) { pv[k] = p[(RT && k >= m) ? m - 1 : k]; }
  const double b_own = b[blk_s * m + r_s];
  T lu[M];
#pragma unroll
  for (int j = 0; j < M; j++) { lu[j] = Fb[((RT && j >= m) ? m - 1 : j) * m + r_s]; }

  // source position of b after the sequential swaps b[k] <-> b[p[k]]
  int idx = r_s;
#pragma unroll
  for (int k = M - 1; k >= 0; k--)
  {
    if (RT && k >= m) { continue; }
    const int pk = pv[k];
    if (idx == k) { idx = pk; }
    else if (idx == pk) { idx = k; }
  }
  // (pivots of an unfactored block are not trusted to stay in range)
  double bi = __shfl(b_own, base + (((unsigned)idx < (unsigned)m) ? idx : 0), 64);

  // L y = P b (unit lower)
  static_for<0, M - 1>([&](auto kc) {
    constexpr int k = decltype(kc)::value;
    if (RT && k >= m - 1) { return; }
    const double bk = g_bcast<G, k>(bi);
    if (lane_above<G, k>()) { bi = bi - (double)lu[k] * bk; }
  });
  // U x = y.  A lane's own entry is its quotient bi / d, formed where it is
  // broadcast and once more at the end; bi stays the numerator.
  const double y = bi;
  T dt           = lu[0];
  static_for<1, M>([&](auto jc) {
    constexpr int j = decltype(jc)::value;
    dt              = lane_is<G, j>() ? lu[j] : dt;
  });
  const double d    = (double)dt;
  const double rinv = 1.0 / d;
  static_for<0, M - 1>([&](auto kc) {
    constexpr int k = M - 1 - decltype(kc)::value;
    if (RT && k >= m) { return; }
    const double xk = g_bcast<G, k>(quotient(bi, d, rinv));
    if (lane_below<G, k>()) { bi = bi - (double)lu[k] * xk; }
  });
  double xi = quotient(bi, d, rinv);
  if (ballot(valid && !(quotient_safe(d) && (bi == 0.0 || quotient_safe(bi)))) != 0)
  {
    // a numerator or diagonal outside the quotient's range (or a zero
    // diagonal, an infinity, a NaN): the sweep with divisions
    bi = y;
    static_for<0, M - 1>([&](auto kc) {
      constexpr int k = M - 1 - decltype(kc)::value;
      if (RT && k >= m) { return; }
      const double xk = g_bcast<G, k>(bi / d);
      if (r < k) { bi = bi - (double)lu[k] * xk; }
    });
    xi = bi / d;
  }
  // scale * x is N_VScale's per-element product (exact for scale = 1)
  if (valid) { x[blk * m + r] = scale * xi; }
}

// ----------------------------------------------------------------------------
// launches
// ----------------------------------------------------------------------------
static inline unsigned lu_grid(int row, long nblocks)
{
  const long per = (long)LU_WAVES * (64 / pow2ceil(row));
  return (unsigned)((nblocks + per - 1) / per);
}

template <int M, typename T, bool RT>
void lu_getrf(int m, const double* A, T* F, int* piv, long nblocks, unsigned long long* info,
              hipStream_t s)
{
  k_getrf<M, T, SRC_PLAIN, RT>
    <<<lu_grid(M, nblocks), 64 * LU_WAVES, 0, s>>>(A, F, piv, nblocks, info, m);
}

template <int M, typename T, bool RT>
void lu_getrf_scaled(bool save_src, const double* src, double c, double* save, double* scaled,
                     T* F, int* piv, long nblocks, unsigned long long* info, hipStream_t s)
{
  if (save_src)
  {
    k_getrf<M, T, SRC_SAVE, RT><<<lu_grid(M, nblocks), 64 * LU_WAVES, 0, s>>>(
      src, F, piv, nblocks, info, M, c, save, scaled);
  }
  else
  {
    k_getrf<M, T, SRC_SCALED, RT><<<lu_grid(M, nblocks), 64 * LU_WAVES, 0, s>>>(
      src, F, piv, nblocks, info, M, c, save, scaled);
  }
}

template <int M, typename T, bool RT>
void lu_getrs(int m, const T* F, const int* piv, const double* b, double* x, long nblocks,
              double scale, hipStream_t s)
{
  k_getrs<M, T, RT><<<lu_grid(M, nblocks), 64 * LU_WAVES, 0, s>>>(F, piv, b, x, nblocks, scale, m);
}

template <int M, typename T>
const LuLaunch<T>* lu_size()
{
  constexpr bool RT          = M > 32; // rows longer than 32: see k_getrf
  static const LuLaunch<T> L = {lu_getrf<M, T, RT>, lu_getrf_scaled<M, T, RT>,
                                lu_getrs<M, T, false>};
  return &L;
}

template <int M, typename T>
const LuLaunch<T>* lu_row_size()
{
  static const LuLaunch<T> L = {lu_getrf<M, T, true>, nullptr, lu_getrs<M, T, true>};
  return &L;
}

#define LU_INSTANTIATE_SIZE(MM, T) template const LuLaunch<T>* lu_size<MM, T>();
#define LU_INSTANTIATE_ROW(MM, T) template const LuLaunch<T>* lu_row_size<MM, T>();

#endif
