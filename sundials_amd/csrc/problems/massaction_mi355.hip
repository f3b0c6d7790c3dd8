// -----------------------------------------------------------------------------
// Mass-action right-hand side and block Jacobian on the MI355X, and the
// coupled-system driver (every cell in one N_Vector, block-diagonal Jacobian,
// BDF + modified Newton + batched block LU).
//
// RHS and Jacobian: one group of G = pow2ceil(m) lanes per cell (lane =
// species, or Jacobian row), 64 / G cells per wavefront, one-wavefront
// workgroups striding over the cells.  The RHS evaluates each reaction's net
// rate once (reactions spread over the group's lanes, into LDS) and each
// species then adds its terms in reaction / role order -- the order in which
// the serial evaluation updates f_i -- so f is bit-identical to it.  The
// Jacobian row of each lane is assembled in LDS from that lane's terms only,
// in the serial evaluation's reaction / target / column order, and the block
// is streamed out column by column.  Rate constants are stored cell-major
// (cell * R + r), so a cell's rates are one coalesced read by its group; the
// species, rates and results move as whole rows of the cell.
// -----------------------------------------------------------------------------
#include <hip/hip_runtime.h>

#include <chrono>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "../batched/coupled_device.h"
#include "../core/lane_ops.h"
#include "../core/profiler_internal.h"
#include "sunamd/cvode_sunamd.h"
#include "sunamd/sunamd_profiler.h"
#include "sunamd/massaction_mi355.h"
#include "sunamd/nvector_mi355.h"
#include "sunamd/sunmatrix_mi355block.h"

struct SUNAMD_MassActionDev_
{
  int m, R;
  long ncells;
  int* idx;   // 4R
  int* soff;  // m+1: species s's terms are sent[soff[s] .. soff[s+1])
  int* sent;  // 4R term codes 4r + role (role 0, 1: reactants; 2, 3: products)
  double* kf; // ncells*R, cell-major
  double* kb;
  hipStream_t stream;
  unsigned rhs_grid, jac_grid; // launch sizes, chosen at the first call
};

static int hipfail(hipError_t e, const char* what)
{
  fprintf(stderr, "[sundials_amd massaction] %s failed: %s\n", what, hipGetErrorString(e));
  fflush(stderr);
  return -1;
}

// LDS of one workgroup: per group its species (m doubles), then the
// reaction table, the term offsets and the term codes; doubles counted in
// pairs so the int4 reads of the table are 16-byte aligned
static inline size_t ma_table_ints(int m, int R) { return (size_t)(8 * R + ((m + 2) & ~1)); }

__device__ __forceinline__ void ma_stage_tables(const int* __restrict__ idx,
                                                const int* __restrict__ soff,
                                                const int* __restrict__ sent, int* s_idx,
                                                int* s_soff, int* s_sent, int m, int R)
{
  for (int t = threadIdx.x; t < 4 * R; t += blockDim.x)
  {
    s_idx[t]  = idx[t];
    s_sent[t] = sent[t];
  }
  for (int t = threadIdx.x; t <= m; t += blockDim.x) { s_soff[t] = soff[t]; }
}

// A cell's operands on their way from HBM while the cell before it is worked
// on: its species of this lane and the rates of this lane's first two
// reactions (R = 1.5 m needs no more; further ones are loaded where they are
// used).  Lanes without a cell or a reaction read inside the arrays and drop
// the value, so the loads are unconditional; a workgroup's last pass fetches
// nothing (every workgroup would read the last cell).
struct MaNext
{
  double y, kf[2], kb[2];
};

__device__ __forceinline__ MaNext ma_fetch(const double* __restrict__ y,
                                           const double* __restrict__ kf,
                                           const double* __restrict__ kb, long cell, long ncells,
                                           int i, int m, int G, int R)
{
  MaNext n;
  const long c = cell < ncells ? cell : ncells - 1;
  n.y          = y[c * m + (i < m ? i : m - 1)];
#pragma unroll
  for (int q = 0; q < 2; q++)
  {
    const int r = (i + q * G < R) ? i + q * G : R - 1;
    n.kf[q]     = kf[c * R + r];
    n.kb[q]     = kb[c * R + r];
  }
  return n;
}

// f = RHS(y): per group, y (m), the net rates w (R) and a zero in LDS.  One
// wavefront per workgroup: its LDS exchanges need a wavefront-level ordering
// point only (a workgroup barrier would also wait for the next cell's loads).
//
// What bounds it: LDS and VALU issue about as much as HBM (m = 32, R = 48:
// 1280 bytes per cell; 2^18 cells in 57 us at the copy rate).  A lane's terms
// are the same for every cell, so the first MA_TERMS of them (their rate's
// place and sign) stay in registers instead of being read from LDS per cell,
// which pays from the second pass of a workgroup on: 2^18 cells 75 -> 66 us,
// 30000 cells 12.4 -> 9.5 us with one round of workgroups (14.1 with four).
constexpr int MA_TERMS = 12;

__global__ void __launch_bounds__(64) k_ma_rhs(const double* __restrict__ y,
                                               double* __restrict__ f,
                                               const int* __restrict__ idx,
                                               const int* __restrict__ soff,
                                               const int* __restrict__ sent,
                                               const double* __restrict__ kf,
                                               const double* __restrict__ kb, int m, int G,
                                               int R, long ncells)
{
  using sunamd_lane::wave_sync;
  extern __shared__ __align__(16) double sm[];
  const int gpw   = 64 / G;
  const long per  = (long)((m + R + 2) & ~1);
  const int grp   = threadIdx.x / G;
  const int i     = threadIdx.x % G;
  double* ys      = sm + grp * per;
  double* ws      = ys + m;
  int* s_idx      = (int*)(sm + gpw * per);
  int* s_sent     = s_idx + 4 * R;
  int* s_soff     = s_sent + 4 * R;
  const long step = (long)gridDim.x * gpw;
  MaNext nx       = ma_fetch(y, kf, kb, (long)blockIdx.x * gpw + grp, ncells, i, m, G, R);
  ma_stage_tables(idx, soff, sent, s_idx, s_soff, s_sent, m, R);
  __syncthreads();
  const int e0    = (i < m) ? s_soff[i] : 0;
  const int e1    = (i < m) ? s_soff[i + 1] : 0;
  const int4* ix4 = (const int4*)s_idx;
  // place of the term's rate, sign in the top bit; absent terms add ws[R] = 0
  // (the sum starts from +0, which no sum of it with zeros leaves)
  unsigned term[MA_TERMS];
#pragma unroll
  for (int q = 0; q < MA_TERMS; q++)
  {
    const int code = (e0 + q < e1) ? s_sent[e0 + q] : 4 * R + 2;
    term[q]        = (unsigned)(code >> 2) | ((code & 3) < 2 ? 0x80000000u : 0u);
  }
  const int most = e1 - e0 < MA_TERMS ? e1 - e0 : MA_TERMS; // terms of this lane in registers
  if (i == 0) { ws[R] = 0.0; }
  for (long c0 = (long)blockIdx.x * gpw; c0 < ncells; c0 += step)
  {
    const long cell = c0 + grp;
    const bool live = cell < ncells;
    const MaNext nc = nx;
    if (live && i < m) { ys[i] = nc.y; }
    wave_sync();
    if (c0 + step < ncells) { nx = ma_fetch(y, kf, kb, cell + step, ncells, i, m, G, R); }
    if (live)
    {
#pragma unroll
      for (int q = 0; q < 2; q++)
      {
        const int r = i + q * G;
        if (r < R)
        {
          const int4 ix   = ix4[r];
          const double wf = (nc.kf[q] * ys[ix.x]) * ys[ix.y];
          const double wb = (nc.kb[q] * ys[ix.z]) * ys[ix.w];
          ws[r]           = wf - wb;
        }
      }
      for (int r = i + 2 * G; r < R; r += G)
      {
        const int4 ix   = ix4[r];
        const double wf = (kf[cell * R + r] * ys[ix.x]) * ys[ix.y];
        const double wb = (kb[cell * R + r] * ys[ix.z]) * ys[ix.w];
        ws[r]           = wf - wb;
      }
    }
    wave_sync();
    if (live && i < m)
    {
      double acc = 0.0;
#pragma unroll
      for (int q0 = 0; q0 < MA_TERMS; q0 += 4)
      {
        if (q0 < most)
        {
          double w[4];
#pragma unroll
          for (int q = 0; q < 4; q++) { w[q] = ws[term[q0 + q] & 0x7fffffffu]; }
#pragma unroll
          for (int q = 0; q < 4; q++)
          {
            // acc - w is acc + (-w)
            const long long v = __double_as_longlong(w[q]) ^
                                ((long long)(term[q0 + q] & 0x80000000u) << 32);
            acc               = acc + __longlong_as_double(v);
          }
        }
      }
      for (int e = e0 + MA_TERMS; e < e1; e++)
      {
        const int code = s_sent[e];
        const double w = ws[code >> 2];
        acc            = ((code & 3) < 2) ? acc - w : acc + w;
      }
      f[cell * m + i] = acc;
    }
    wave_sync();
  }
}

// one term of a Jacobian row: the reaction's species and the partial
// derivatives of its rate, and whether the row loses by it
struct MaTerm
{
  int4 ix;
  double dw[4];
  bool loss;
};

// J = df/dy, block column-major: per group, the block (m*m), y (m) and the
// cell's rates (2R) in LDS.
//
// What bounds it: 8 m^2 bytes per cell to HBM (m = 32: 9.2 KB, 2^18 cells in
// 0.41 ms at the copy rate) against the chain of LDS updates of a row.  So the
// next cell's operands are fetched meanwhile, a term's operands are read while
// the one before it updates the row, and the block is cleared as it is
// written out (in pairs of doubles where m*m is even): 2^18 cells 560 -> 450 us.
template <bool PAIRS>
__global__ void __launch_bounds__(64) k_ma_jac(const double* __restrict__ y,
                                               double* __restrict__ J,
                                               const int* __restrict__ idx,
                                               const int* __restrict__ soff,
                                               const int* __restrict__ sent,
                                               const double* __restrict__ kf,
                                               const double* __restrict__ kb, int m, int G,
                                               int R, long ncells)
{
  using sunamd_lane::wave_sync;
  extern __shared__ __align__(16) double sj[];
  const int gpw   = 64 / G;
  const int mm    = m * m;
  const long per  = (long)((mm + m + 2 * R + 1) & ~1);
  const int grp   = threadIdx.x / G;
  const int i     = threadIdx.x % G;
  double* Jl      = sj + grp * per;
  double* ys      = Jl + mm;
  double* rk      = ys + m;
  int* s_idx      = (int*)(sj + gpw * per);
  int* s_sent     = s_idx + 4 * R;
  int* s_soff     = s_sent + 4 * R;
  const long step = (long)gridDim.x * gpw;
  MaNext nx       = ma_fetch(y, kf, kb, (long)blockIdx.x * gpw + grp, ncells, i, m, G, R);
  ma_stage_tables(idx, soff, sent, s_idx, s_soff, s_sent, m, R);
  for (int e = i; e < mm; e += G) { Jl[e] = 0.0; }
  __syncthreads();
  const int e0    = (i < m) ? s_soff[i] : 0;
  const int e1    = (i < m) ? s_soff[i + 1] : 0;
  const int4* ix4 = (const int4*)s_idx;
  auto term       = [&](int e) {
    MaTerm u;
    const int code   = s_sent[e];
    const int r      = code >> 2;
    u.loss           = (code & 3) < 2;
    u.ix             = ix4[r];
    const double kfv = rk[r], kbv = rk[R + r];
    u.dw[0] = kfv * ys[u.ix.y];
    u.dw[1] = kfv * ys[u.ix.x];
    u.dw[2] = -(kbv * ys[u.ix.w]);
    u.dw[3] = -(kbv * ys[u.ix.z]);
    return u;
  };
  for (long c0 = (long)blockIdx.x * gpw; c0 < ncells; c0 += step)
  {
    const long cell = c0 + grp;
    const bool live = cell < ncells;
    if (live)
    {
      if (i < m) { ys[i] = nx.y; }
#pragma unroll
      for (int q = 0; q < 2; q++)
      {
        const int r = i + q * G;
        if (r < R)
        {
          rk[r]     = nx.kf[q];
          rk[R + r] = nx.kb[q];
        }
      }
      for (int r = i + 2 * G; r < R; r += G)
      {
        rk[r]     = kf[cell * R + r];
        rk[R + r] = kb[cell * R + r];
      }
    }
    wave_sync();
    if (c0 + step < ncells) { nx = ma_fetch(y, kf, kb, cell + step, ncells, i, m, G, R); }
    if (live && e0 < e1)
    {
      // row i: the terms in which species i is a target, each adding the
      // reaction's partial derivatives to the columns of its four species
      MaTerm u = term(e0);
      for (int e = e0; e < e1; e++)
      {
        const MaTerm v   = term(e + 1 < e1 ? e + 1 : e);
        const int col[4] = {u.ix.x, u.ix.y, u.ix.z, u.ix.w};
#pragma unroll
        for (int q = 0; q < 4; q++)
        {
          const int a = col[q] * m + i;
          Jl[a]       = u.loss ? (Jl[a] - u.dw[q]) : (Jl[a] + u.dw[q]);
        }
        u = v;
      }
    }
    wave_sync();
    if (live)
    {
      double* Jc = J + cell * (long)mm;
      if (PAIRS)
      {
        for (int e = i; e < mm / 2; e += G)
        {
          double2* d = reinterpret_cast<double2*>(Jl) + e;
          reinterpret_cast<double2*>(Jc)[e] = *d;
          *d                                = make_double2(0.0, 0.0);
        }
      }
      else
      {
        for (int e = i; e < mm; e += G)
        {
          Jc[e] = Jl[e];
          Jl[e] = 0.0;
        }
      }
    }
    wave_sync();
  }
}

// The same for small blocks (m < 16), cell after cell: their few terms and
// bytes leave nothing for the operands fetched ahead to hide, and the form
// above takes up to 8 % longer (500000 cells, four rounds: m = 5, R = 8 84
// against 81 us; m = 11, R = 16 212 against 208; but m = 16, R = 24 301 against
// 359).
__global__ void __launch_bounds__(64) k_ma_jac_small(const double* __restrict__ y,
                                               double* __restrict__ J,
                                               const int* __restrict__ idx,
                                               const int* __restrict__ soff,
                                               const int* __restrict__ sent,
                                               const double* __restrict__ kf,
                                               const double* __restrict__ kb, int m, int G,
                                               int R, long ncells)
{
  using sunamd_lane::wave_sync;
  extern __shared__ __align__(16) double sj[];
  const int gpw   = 64 / G;
  const int mm    = m * m;
  const long per  = (long)((mm + m + 2 * R + 1) & ~1);
  const int grp   = threadIdx.x / G;
  const int i     = threadIdx.x % G;
  double* Jl      = sj + grp * per;
  double* ys      = Jl + mm;
  double* rk      = ys + m;
  int* s_idx      = (int*)(sj + gpw * per);
  int* s_sent     = s_idx + 4 * R;
  int* s_soff     = s_sent + 4 * R;
  ma_stage_tables(idx, soff, sent, s_idx, s_soff, s_sent, m, R);
  __syncthreads();
  const int e0    = (i < m) ? s_soff[i] : 0;
  const int e1    = (i < m) ? s_soff[i + 1] : 0;
  const int4* ix4 = (const int4*)s_idx;
  for (long c0 = (long)blockIdx.x * gpw; c0 < ncells; c0 += (long)gridDim.x * gpw)
  {
    const long cell = c0 + grp;
    const bool live = cell < ncells;
    if (live)
    {
      for (int e = i; e < mm; e += G) { Jl[e] = 0.0; }
      if (i < m) { ys[i] = y[cell * m + i]; }
      for (int r = i; r < R; r += G)
      {
        rk[r]     = kf[cell * R + r];
        rk[R + r] = kb[cell * R + r];
      }
    }
    wave_sync();
    if (live && i < m)
    {
      // row i: the terms in which species i is a target, each adding the
      // reaction's partial derivatives to the columns of its four species
      for (int e = e0; e < e1; e++)
      {
        const int code  = s_sent[e];
        const int r     = code >> 2;
        const bool loss = (code & 3) < 2;
        const int4 ix   = ix4[r];
        const double kfv = rk[r], kbv = rk[R + r];
        const int col[4]   = {ix.x, ix.y, ix.z, ix.w};
        const double dw[4] = {kfv * ys[ix.y], kfv * ys[ix.x], -(kbv * ys[ix.w]),
                              -(kbv * ys[ix.z])};
#pragma unroll
        for (int q = 0; q < 4; q++)
        {
          const int a = col[q] * m + i;
          Jl[a]       = loss ? (Jl[a] - dw[q]) : (Jl[a] + dw[q]);
        }
      }
    }
    wave_sync();
    if (live)
    {
      double* Jc = J + cell * (long)mm;
      for (int e = i; e < mm; e += G) { Jc[e] = Jl[e]; }
    }
    wave_sync();
  }
}

static int pow2ceil_h(int m)
{
  int g = 1;
  while (g < m) { g <<= 1; }
  return g;
}

// dynamic LDS of the RHS and Jacobian workgroups
static size_t ma_rhs_lds(int m, int R)
{
  const int gpw = 64 / pow2ceil_h(m);
  return sizeof(double) * (size_t)gpw * (size_t)((m + R + 2) & ~1) +
         sizeof(int) * ma_table_ints(m, R);
}

static size_t ma_jac_lds(int m, int R)
{
  const int gpw = 64 / pow2ceil_h(m);
  return sizeof(double) * (size_t)gpw * (size_t)((m * m + m + 2 * R + 1) & ~1) +
         sizeof(int) * ma_table_ints(m, R);
}

extern "C" SUNAMD_MassActionDev* SUNAMD_MassActionToDevice(const SUNAMD_MassAction* p,
                                                           void* stream)
{
  if (!p || p->m < 1 || p->m > 64 || p->R < 1) { return NULL; }
  if (ma_jac_lds(p->m, p->R) > 65536 || ma_rhs_lds(p->m, p->R) > 65536) { return NULL; }
  for (int t = 0; t < 4 * p->R; t++)
  {
    if (p->idx[t] < 0 || p->idx[t] >= p->m) { return NULL; }
  }
  SUNAMD_MassActionDev* d = (SUNAMD_MassActionDev*)calloc(1, sizeof(SUNAMD_MassActionDev));
  if (!d) { return NULL; }
  d->m      = p->m;
  d->R      = p->R;
  d->ncells = (long)p->ncells;
  d->stream = (hipStream_t)stream;
  const size_t nr = (size_t)p->R * (size_t)p->ncells;
  // species s's terms in reaction order, roles a b c d within a reaction:
  // the order in which the serial RHS and Jacobian accumulate them
  int* off  = (int*)calloc((size_t)p->m + 1, sizeof(int));
  int* ent  = (int*)malloc(sizeof(int) * 4 * (size_t)p->R);
  int* fill = (int*)malloc(sizeof(int) * (size_t)p->m);
  hipError_t e = (off && ent && fill) ? hipSuccess : hipErrorOutOfMemory;
  if (e == hipSuccess)
  {
    for (int t = 0; t < 4 * p->R; t++) { off[p->idx[t] + 1]++; }
    for (int q = 0; q < p->m; q++) { off[q + 1] += off[q]; }
    memcpy(fill, off, sizeof(int) * (size_t)p->m);
    for (int t = 0; t < 4 * p->R; t++) { ent[fill[p->idx[t]]++] = t; }
  }
  if (e == hipSuccess) { e = hipMalloc((void**)&d->idx, sizeof(int) * 4 * (size_t)p->R); }
  if (e == hipSuccess) { e = hipMalloc((void**)&d->soff, sizeof(int) * ((size_t)p->m + 1)); }
  if (e == hipSuccess) { e = hipMalloc((void**)&d->sent, sizeof(int) * 4 * (size_t)p->R); }
  if (e == hipSuccess) { e = hipMalloc((void**)&d->kf, sizeof(double) * nr); }
  if (e == hipSuccess) { e = hipMalloc((void**)&d->kb, sizeof(double) * nr); }
  if (e == hipSuccess)
  {
    e = hipMemcpy(d->idx, p->idx, sizeof(int) * 4 * (size_t)p->R, hipMemcpyHostToDevice);
  }
  if (e == hipSuccess)
  {
    e = hipMemcpy(d->soff, off, sizeof(int) * ((size_t)p->m + 1), hipMemcpyHostToDevice);
  }
  if (e == hipSuccess)
  {
    e = hipMemcpy(d->sent, ent, sizeof(int) * 4 * (size_t)p->R, hipMemcpyHostToDevice);
  }
  // the host problem keeps its rates cell-major already
  if (e == hipSuccess) { e = hipMemcpy(d->kf, p->kf, sizeof(double) * nr, hipMemcpyHostToDevice); }
  if (e == hipSuccess) { e = hipMemcpy(d->kb, p->kb, sizeof(double) * nr, hipMemcpyHostToDevice); }
  free(off);
  free(ent);
  free(fill);
  if (e != hipSuccess)
  {
    hipfail(e, "problem upload");
    SUNAMD_MassActionDevFree(d);
    return NULL;
  }
  return d;
}

extern "C" void SUNAMD_MassActionDevFree(SUNAMD_MassActionDev* d)
{
  if (!d) { return; }
  void* ps[] = {d->idx, d->soff, d->sent, d->kf, d->kb};
  for (void* q : ps)
  {
    if (q) { (void)hipFree(q); }
  }
  free(d);
}

// workgroups for a grid-stride launch: enough to fill every CU `rounds` times
// at the kernel's occupancy, no more than the cells need
template <typename K>
static unsigned ma_grid(K kern, size_t shm, long ncells, int gpw, int rounds)
{
  static int cus = 0;
  if (cus == 0)
  {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        cus < 1)
    {
      cus = 256;
    }
  }
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, 64, shm) != hipSuccess ||
      per_cu < 1)
  {
    per_cu = 1;
  }
  const long need = (ncells + gpw - 1) / gpw;
  const long full = (long)rounds * per_cu * cus;
  return (unsigned)(need < full ? need : full);
}

extern "C" int SUNAMD_MassActionRhsDevArrays(SUNAMD_MassActionDev* d, const double* dy,
                                             double* df)
{
  const int G   = pow2ceil_h(d->m);
  const int gpw = 64 / G;
  const size_t shm = ma_rhs_lds(d->m, d->R);
  if (d->ncells < 1) { return 0; }
  // one round: fewer table stagings and term lists, a longer run of prefetched
  // cells each (with four, 120000 cells of m = 5, R = 8 took 11.5 us, with one
  // 8.0; cell after cell without either it was 9.3)
  if (d->rhs_grid == 0) { d->rhs_grid = ma_grid(k_ma_rhs, shm, d->ncells, gpw, 1); }
  const unsigned g = d->rhs_grid;
  sunamd_prof_begin(SUNAMD_K_RHS, d->stream);
  k_ma_rhs<<<g, 64, shm, d->stream>>>(dy, df, d->idx, d->soff, d->sent, d->kf, d->kb, d->m, G,
                                      d->R, d->ncells);
  sunamd_prof_end(SUNAMD_K_RHS, d->stream);
  hipError_t e = hipGetLastError();
  return (e == hipSuccess) ? 0 : hipfail(e, "rhs launch");
}

extern "C" int SUNAMD_MassActionJacDevArrays(SUNAMD_MassActionDev* d, const double* dy,
                                             double* dJ)
{
  const int G   = pow2ceil_h(d->m);
  const int gpw = 64 / G;
  const size_t shm = ma_jac_lds(d->m, d->R);
  if (d->ncells < 1) { return 0; }
  // blocks of an even number of entries start on 16 bytes if the array does
  const int mm     = d->m * d->m;
  const bool pairs = mm % 2 == 0 && ((uintptr_t)dJ & 15u) == 0;
  const bool small = d->m < 16;
  auto kern        = small ? k_ma_jac_small : pairs ? k_ma_jac<true> : k_ma_jac<false>;
  if (d->jac_grid == 0)
  {
    // one round where writing the block outweighs the 16R updates of its
    // entries, four where the updates do and the wavefronts end unevenly
    // (120000 cells, one against four: m = 32, R = 48 209 / 223 us, R = 96
    // 487 / 362; m = 24, R = 36 188 / 161; 30000 cells of 64, R = 96 208 / 221)
    const int rounds = (mm >= 1024 && mm >= 16 * d->R) ? 1 : 4;
    d->jac_grid      = small ? ma_grid(k_ma_jac_small, shm, d->ncells, gpw, rounds)
                             : ma_grid(k_ma_jac<true>, shm, d->ncells, gpw, rounds);
  }
  const unsigned g = d->jac_grid;
  kern<<<g, 64, shm, d->stream>>>(dy, dJ, d->idx, d->soff, d->sent, d->kf, d->kb, d->m, G, d->R,
                                  d->ncells);
  hipError_t e = hipGetLastError();
  return (e == hipSuccess) ? 0 : hipfail(e, "jac launch");
}

extern "C" int SUNAMD_MassActionRhsDev(sunrealtype t, N_Vector y, N_Vector ydot,
                                       void* user_data)
{
  (void)t;
  SUNAMD_MassActionDev* d = (SUNAMD_MassActionDev*)user_data;
  return SUNAMD_MassActionRhsDevArrays(d, N_VGetDeviceArrayPointer(y),
                                       N_VGetDeviceArrayPointer(ydot));
}

extern "C" int SUNAMD_MassActionJacDev(sunrealtype t, N_Vector y, N_Vector fy, SUNMatrix J,
                                       void* user_data, N_Vector tmp1, N_Vector tmp2,
                                       N_Vector tmp3)
{
  (void)t;
  (void)fy;
  (void)tmp1;
  (void)tmp2;
  (void)tmp3;
  SUNAMD_MassActionDev* d = (SUNAMD_MassActionDev*)user_data;
  return SUNAMD_MassActionJacDevArrays(d, N_VGetDeviceArrayPointer(y),
                                       SUNMatrix_Mi355BlockDense_DeviceData(J));
}

struct SUNAMD_CoupledRun_
{
  SUNContext ctx;
  sunindextype N;
  N_Vector y, y0;
  SUNAMD_MassActionDev* dev;
  SUNMatrix A;
  SUNLinearSolver LS;
  void* cv;
  // the device-stepped integrator (coupled_device.hip) and what it needs
  int devstep;
  void* dstate;
  double rtol, atol;
  int lu_precision, reduction_order;
};

extern "C" int SUNAMD_CoupledSetDeviceStepping_Mi355(SUNAMD_CoupledRun* r, int onoff)
{
  if (!r) { return -1; }
  r->devstep = onoff ? 1 : 0;
  return 0;
}

extern "C" int SUNAMD_CoupledSetFusedKernels_Mi355(SUNAMD_CoupledRun* r, int onoff)
{
  if (!r || !r->cv) { return -1; }
  return CVodeSetUseIntegratorFusedKernels(r->cv, onoff ? SUNTRUE : SUNFALSE);
}

extern "C" void SUNAMD_CoupledFree_Mi355(SUNAMD_CoupledRun* r)
{
  if (!r) { return; }
  if (r->dstate) { sunamd_coupled_device_free(r->dstate); }
  if (r->cv) { CVodeFree(&r->cv); }
  if (r->LS) { SUNLinSolFree(r->LS); }
  if (r->A) { SUNMatDestroy(r->A); }
  if (r->dev) { SUNAMD_MassActionDevFree(r->dev); }
  if (r->y0) { N_VDestroy(r->y0); }
  if (r->y) { N_VDestroy(r->y); }
  if (r->ctx) { SUNContext_Free(&r->ctx); }
  free(r);
}

extern "C" SUNAMD_CoupledRun* SUNAMD_CoupledCreate_Mi355(const SUNAMD_MassAction* p,
                                                         double rtol, double atol,
                                                         int lu_precision,
                                                         int reduction_order)
{
  SUNAMD_CoupledRun* r = (SUNAMD_CoupledRun*)calloc(1, sizeof(SUNAMD_CoupledRun));
  if (!r) { return NULL; }
  bool ok = SUNContext_Create(SUN_COMM_NULL, &r->ctx) == 0;
  r->N    = (sunindextype)p->ncells * p->m;
  r->rtol = rtol;
  r->atol = atol;
  r->lu_precision    = lu_precision;
  r->reduction_order = reduction_order;
  if (ok) { ok = (r->y = N_VNew_Mi355(r->N, r->ctx)) != NULL; }
  if (ok) { ok = N_VSetReductionOrder_Mi355(r->y, reduction_order) == 0; }
  if (ok) { ok = (r->y0 = N_VClone(r->y)) != NULL; }
  if (ok) { ok = N_VCopyFromHostArray_Mi355(r->y0, p->y0) == 0; }
  if (ok) { N_VScale(1.0, r->y0, r->y); }
  if (ok) { ok = (r->dev = SUNAMD_MassActionToDevice(p, N_VGetStream_Mi355(r->y))) != NULL; }
  if (ok)
  {
    ok = (r->A = SUNMatrix_Mi355BlockDense(p->ncells, p->m, N_VGetStream_Mi355(r->y),
                                           r->ctx)) != NULL;
  }
  if (ok) { ok = (r->LS = SUNLinSol_Mi355BlockLU(r->y, r->A, lu_precision, r->ctx)) != NULL; }
  if (ok) { ok = (r->cv = CVodeCreate(CV_BDF, r->ctx)) != NULL; }
  if (ok) { ok = CVodeInit(r->cv, SUNAMD_MassActionRhsDev, 0.0, r->y) == 0; }
  if (ok) { ok = CVodeSStolerances(r->cv, rtol, atol) == 0; }
  if (ok) { ok = CVodeSetUserData(r->cv, r->dev) == 0; }
  if (ok) { ok = CVodeSetLinearSolver(r->cv, r->LS, r->A) == 0; }
  if (ok) { ok = CVodeSetJacFn(r->cv, SUNAMD_MassActionJacDev) == 0; }
  if (ok) { ok = CVodeSetMaxNumSteps(r->cv, 1000000) == 0; }
  if (ok) { ok = hipDeviceSynchronize() == hipSuccess; }
  if (!ok)
  {
    SUNAMD_CoupledFree_Mi355(r);
    return NULL;
  }
  return r;
}

static int coupled_run_device(SUNAMD_CoupledRun* r, double tout, SUNAMD_SolveStats* st)
{
  if (hipDeviceSynchronize() != hipSuccess) { return -1; }
  CoupledDeviceJob job;
  job.m            = r->dev->m;
  job.R            = r->dev->R;
  job.ncells       = r->dev->ncells;
  job.idx          = r->dev->idx;
  job.kf           = r->dev->kf;
  job.kb           = r->dev->kb;
  job.y0           = N_VGetDeviceArrayPointer(r->y0);
  job.yout         = N_VGetDeviceArrayPointer(r->y);
  job.lu           = SUNMatrix_Mi355BlockDense_DeviceData(r->A);
  job.piv          = SUNLinSol_Mi355BlockLU_DevicePivots(r->LS);
  job.rtol         = r->rtol;
  job.atol         = r->atol;
  job.tout         = tout;
  job.mxstep       = 1000000;
  job.lu_precision = r->lu_precision;
  job.sequential   = r->reduction_order == SUNAMD_REDUCE_SEQUENTIAL;
  job.stream       = (hipStream_t)N_VGetStream_Mi355(r->y);
  SUNAMD_SolveStats s;
  memset(&s, 0, sizeof(s));
  auto t0  = std::chrono::steady_clock::now();
  int flag = sunamd_coupled_device_run(job, &r->dstate, &s);
  if (hipDeviceSynchronize() != hipSuccess) { return -1; }
  auto t1 = std::chrono::steady_clock::now();
  s.wall_s = std::chrono::duration<double>(t1 - t0).count();
  s.flag   = flag;
  if (st) { *st = s; }
  return (flag < 0) ? flag : 0;
}

extern "C" int SUNAMD_CoupledRun_Mi355(SUNAMD_CoupledRun* r, double tout, SUNAMD_SolveStats* st)
{
  sunrealtype t = 0.0;
  if (r->devstep) { return coupled_run_device(r, tout, st); }
  if (hipDeviceSynchronize() != hipSuccess) { return -1; }
  long l0 = N_VGetNumLaunches_Mi355(r->y);
  auto t0 = std::chrono::steady_clock::now();
  N_VScale(1.0, r->y0, r->y);
  int flag = CVodeReInit(r->cv, 0.0, r->y);
  if (flag == 0) { flag = CVode(r->cv, tout, r->y, &t, CV_NORMAL); }
  if (hipDeviceSynchronize() != hipSuccess) { return -1; }
  auto t1 = std::chrono::steady_clock::now();
  if (st)
  {
    long counts[8];
    int orders[2];
    double steps[4];
    CVodeGetAllStats(r->cv, counts, orders, steps);
    st->nst      = counts[0];
    st->nfe      = counts[1];
    st->nsetups  = counts[2];
    st->netf     = counts[3];
    st->nni      = counts[4];
    st->nnf      = counts[5];
    st->ncfn     = counts[6];
    st->nje      = counts[7];
    st->qlast    = orders[0];
    st->qcur     = orders[1];
    st->hinused  = steps[0];
    st->hlast    = steps[1];
    st->hcur     = steps[2];
    st->tcur     = steps[3];
    st->wall_s   = std::chrono::duration<double>(t1 - t0).count();
    st->launches = N_VGetNumLaunches_Mi355(r->y) - l0;
    st->flag     = flag;
  }
  return (flag < 0) ? flag : 0;
}

extern "C" int SUNAMD_CoupledGetState_Mi355(SUNAMD_CoupledRun* r, double* yout)
{
  return N_VCopyToHostArray_Mi355(r->y, yout) == 0 ? 0 : -1;
}

extern "C" int SUNAMD_MassActionSolveCoupled_Mi355(const SUNAMD_MassAction* p, double rtol,
                                                   double atol, double tout,
                                                   int lu_precision, int reduction_order,
                                                   double* yout,
                                                   SUNAMD_SolveStats* st)
{
  SUNAMD_CoupledRun* r =
    SUNAMD_CoupledCreate_Mi355(p, rtol, atol, lu_precision, reduction_order);
  if (!r) { return -1; }
  int rc = SUNAMD_CoupledRun_Mi355(r, tout, st);
  if (rc == 0 && yout) { rc = SUNAMD_CoupledGetState_Mi355(r, yout); }
  SUNAMD_CoupledFree_Mi355(r);
  return rc;
}
