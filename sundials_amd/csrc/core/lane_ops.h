// -----------------------------------------------------------------------------
// lane_ops.h -- cross-lane primitives of the register-row LU kernels (the
// block solver's and the batched integrator's): DPP row permutations, lane
// reads and broadcasts, constant lane masks, the pivot search of a group of G
// lanes on one word per exchange, and quotients from an early reciprocal.
// -----------------------------------------------------------------------------
#ifndef SUNAMD_LANE_OPS_H
#define SUNAMD_LANE_OPS_H

#include <hip/hip_runtime.h>

#include <type_traits>

namespace sunamd_lane
{

// DPP row permutations used by the group reductions.  Every source lane is in
// the reading lane's own group, so no lane is invalid and the old value is
// never used: with bound_ctrl the compiler folds the permutation into the
// instruction that uses it (v_max_u32_dpp) instead of copying x first.
template <int CTRL>
__device__ __forceinline__ int dpp_i(int x)
{
  return __builtin_amdgcn_update_dpp(0, x, CTRL, 0xF, 0xF, true);
}

template <int CTRL>
__device__ __forceinline__ double dpp_v(double x)
{
  const long long u = __double_as_longlong(x);
  const int lo      = dpp_i<CTRL>((int)(u & 0xffffffffLL));
  const int hi      = dpp_i<CTRL>((int)(u >> 32));
  return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned int)lo);
}

template <int CTRL>
__device__ __forceinline__ float dpp_v(float x)
{
  return __int_as_float(dpp_i<CTRL>(__float_as_int(x)));
}

// lane l's value of x, for a lane index that is the same in the whole wavefront
__device__ __forceinline__ double readlane_d(double x, int l)
{
  const long long v = __double_as_longlong(x);
  const int lo      = __builtin_amdgcn_readlane((int)(v & 0xffffffffLL), l);
  const int hi      = __builtin_amdgcn_readlane((int)(v >> 32), l);
  return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned int)lo);
}

__device__ __forceinline__ float readlane_d(float x, int l)
{
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
}

// ---- pivot search of the double- and single-precision factorisations -------
// The dense GETRF's choice (sundials_dense.c:94-100): the largest |a_ik| over
// the rows at positions >= k, the first one on ties.  A (value, position) pair
// carried through every exchange takes about 75 VALU instructions per column
// in FP64; here the exchanges carry one 32-bit word, the value's
// high half, as an unsigned maximum (a DPP v_max_u32 per level), and the
// lanes that hold that maximum are counted with a ballot.  One holder is the
// pivot.  Several holders (a tie in the high half, all zero) are told apart by
// the low half and then by position; a value that is not finite starts the
// search again with a NaN counted as the reference's comparisons count it:
// chosen in the first row, never in a later one.

__device__ __forceinline__ unsigned high_word(double v)
{
  return (unsigned)((unsigned long long)__double_as_longlong(v) >> 32);
}
__device__ __forceinline__ unsigned abs_high(double v) { return high_word(v) & 0x7fffffffu; }
__device__ __forceinline__ unsigned abs_high(float v) { return __float_as_uint(v) & 0x7fffffffu; }
__device__ __forceinline__ unsigned low_word(double v)
{
  return (unsigned)(unsigned long long)__double_as_longlong(v);
}
__device__ __forceinline__ unsigned low_word(float) { return 0u; }
template <typename T>
inline constexpr unsigned kInfHigh = (sizeof(T) == 8) ? 0x7ff00000u : 0x7f800000u;

// lanes where x holds (the builtin takes the lane mask as it is; __ballot first
// makes integers of it)
__device__ __forceinline__ unsigned long long ballot(bool x) { return __builtin_amdgcn_ballot_w64(x); }

// unsigned maximum over a G-lane group (every lane ends with it)
template <int G>
__device__ __forceinline__ unsigned g_umax(unsigned v)
{
  auto mx = [](unsigned a, unsigned b) { return a > b ? a : b; };
  if constexpr (G >= 2) { v = mx(v, (unsigned)dpp_i<0xB1>((int)v)); }
  if constexpr (G >= 4) { v = mx(v, (unsigned)dpp_i<0x4E>((int)v)); }
  if constexpr (G >= 8) { v = mx(v, (unsigned)dpp_i<0x141>((int)v)); }
  if constexpr (G >= 16) { v = mx(v, (unsigned)dpp_i<0x140>((int)v)); }
  if constexpr (G >= 32)
  {
    // rows 2k and 2k+1 of 16 lanes change places in one of two copies, so the
    // copies hold the two rows' maxima side by side
    const auto w = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    v            = mx(w[0], w[1]);
  }
  if constexpr (G == 64)
  {
    const auto w = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    v            = mx(w[0], w[1]);
  }
  return v;
}

// True in the one lane of each group that holds column k's pivot.  ak: this
// lane's entry; cand: its row is valid and at a position >= k; base: the
// group's first lane.
template <int G, typename T>
__device__ __forceinline__ bool g_pivot(T ak, bool cand, int pos, int k, int base)
{
  unsigned hi = cand ? abs_high(ak) : 0u;
  unsigned mx = g_umax<G>(hi);
  bool win    = cand && hi == mx;
  const unsigned long long holders = ballot(win);
  // more than one holder in some group: on the scalar unit for groups of 32
  // and 64 lanes
  bool several;
  if constexpr (G == 64) { several = (holders & (holders - 1)) != 0; }
  else if constexpr (G == 32)
  {
    const unsigned h0 = (unsigned)holders, h1 = (unsigned)(holders >> 32);
    several = ((h0 & (h0 - 1u)) | (h1 & (h1 - 1u))) != 0;
  }
  else
  {
    const unsigned f = (unsigned)(holders >> base) & ((1u << G) - 1u);
    several          = ballot((f & (f - 1u)) != 0) != 0;
  }
  if (several || ballot(mx >= kInfHigh<T>) != 0)
  {
    const bool nan = ak != ak;
    if (nan) { hi = (cand && pos == k) ? 0x7fffffffu : 0u; }
    // (each maximum is taken by all lanes, outside the conditions)
    mx                 = g_umax<G>(hi);
    win                = cand && hi == mx;
    const unsigned lo  = (win && !nan) ? low_word(ak) : 0u;
    const unsigned mlo = g_umax<G>(lo);
    win                = win && lo == mlo;
    const unsigned at  = win ? 64u - (unsigned)pos : 0u;
    const unsigned mat = g_umax<G>(at);
    win                = win && at == mat;
  }
  return win;
}

// ---- constant sets of lanes ---------------------------------------------------
// Lanes whose index in their G-lane group is above / below / equal to k, as a
// condition: a constant mask moved into scalar registers where it is used (the
// moves are volatile: as plain constants the masks of a whole sweep are
// hoisted out of the integrators' step loop and spilled to vector lanes),
// instead of a vector compare.
template <int G>
constexpr unsigned long long lanes_mask(int lo, int hi)
{
  unsigned long long m = 0;
  for (int l = 0; l < 64; l++)
  {
    if (l % G >= lo && l % G < hi) { m |= 1ULL << l; }
  }
  return m;
}
template <unsigned long long MASK>
__device__ __forceinline__ bool in_lanes()
{
  unsigned lo, hi;
  asm volatile("s_mov_b32 %0, %1" : "=s"(lo) : "i"((int)(MASK & 0xffffffffULL)));
  asm volatile("s_mov_b32 %0, %1" : "=s"(hi) : "i"((int)(MASK >> 32)));
  return __builtin_amdgcn_inverse_ballot_w64(((unsigned long long)hi << 32) | lo);
}
template <int G, int K>
__device__ __forceinline__ bool lane_above()
{
  return in_lanes<lanes_mask<G>(K + 1, G)>();
}
template <int G, int K>
__device__ __forceinline__ bool lane_below()
{
  return in_lanes<lanes_mask<G>(0, K)>();
}
template <int G, int K>
__device__ __forceinline__ bool lane_is()
{
  return in_lanes<lanes_mask<G>(K, K + 1)>();
}

// ---- lane k of each G-lane group to all of its lanes, k a constant ----------
// A lane read for groups of 64; an LDS shuffle for 32 (one instruction beside
// the VALU, where two lane reads and a select are three in it); DPP for
// smaller groups: a row broadcast (row_newbcast) inside 16 lanes, restricted
// to banks of four lanes for two groups of 8, a quad permutation for 4 and 2.
template <int G, int K>
__device__ __forceinline__ int g_bcast(int x)
{
  if constexpr (G == 1) { return x; }
  else if constexpr (G == 2) { return dpp_i<(K == 0) ? 0xA0 : 0xF5>(x); }
  else if constexpr (G == 4) { return dpp_i<K * 0x55>(x); }
  else if constexpr (G == 8)
  {
    const int lo = __builtin_amdgcn_update_dpp(x, x, 0x150 + K, 0xF, 0x3, false);
    return __builtin_amdgcn_update_dpp(lo, x, 0x150 + K + 8, 0xF, 0xC, false);
  }
  else if constexpr (G == 16) { return dpp_i<0x150 + K>(x); }
  else if constexpr (G == 32) { return __shfl(x, K, 32); }
  else { return __builtin_amdgcn_readlane(x, K); }
}

template <int G, int K>
__device__ __forceinline__ double g_bcast(double x)
{
  const long long v = __double_as_longlong(x);
  const int lo      = g_bcast<G, K>((int)(v & 0xffffffffLL));
  const int hi      = g_bcast<G, K>((int)(v >> 32));
  return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned int)lo);
}

// f(integral constant) for each index of [B, E), in order; the index can be a
// template argument in f
template <int B, int E, typename F>
__device__ __forceinline__ void static_for(F&& f)
{
  if constexpr (B < E)
  {
    f(std::integral_constant<int, B>{});
    static_for<B + 1, E>(f);
  }
}

// ---- quotients by a divisor that is known early ------------------------------
// n / d as the division instruction sequence rounds it, from r = 1 / d
// (correctly rounded, taken off the chain): q0 = n r is within 1.5 ulp, one
// exact remainder step makes it faithful, a second one correctly rounded
// (Markstein, IBM J. Res. Dev. 34(1), 1990, theorem 8.2: r correctly rounded,
// q faithful).  Five dependent operations instead of about eleven.  Valid
// while neither remainder can underflow nor anything overflow, which
// quotient_safe tests; q0 has the sign, also of a zero quotient.
__device__ __forceinline__ double quotient(double n, double d, double r)
{
  const double q0 = n * r;
  const double q1 = __builtin_fma(__builtin_fma(-d, q0, n), r, q0);
  const double q2 = __builtin_fma(__builtin_fma(-d, q1, n), r, q1);
  return __builtin_copysign(q2, q0);
}

// |x| in [2^-400, 2^400)
__device__ __forceinline__ bool quotient_safe(double x)
{
  return (abs_high(x) >> 20) - (1023u - 400u) < 800u;
}

// wavefront-level ordering point for a group's LDS exchange
__device__ __forceinline__ void wave_sync()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

} // namespace sunamd_lane

#endif
