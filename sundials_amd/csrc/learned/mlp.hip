// -----------------------------------------------------------------------------
// MLP for the learned Newton initial iterate: forward, backward and Adam on
// the MI355X.  A training step is two launches:
//   k_rows   one workgroup per 16 rows of the batch runs the whole forward
//            and backward pass of its rows (activations in registers and LDS)
//            and leaves, transposed, the bf16 operands of the weight gradients;
//   k_update one workgroup per 16 x 16 tile of a weight matrix sums that
//            tile's gradient over the batch and applies Adam to it, writing
//            the FP32 master, the moments and the BF16 copies.
// Every product is v_mfma_f32_16x16x32_bf16 with FP32 accumulation; all sums
// have a fixed order.  Weights are kept in FP32 (master copy and Adam moments)
// and re-rounded to BF16 after every update.
//
// What bounds a step of 1024 rows (0.26 GFLOP, 1.1 MB of rows, 1.2 MB of
// parameters and moments) is latency: launches and the chain of dependent
// loads, not bandwidth or the matrix cores.  As separate GEMM, bias,
// activation, column-sum and Adam kernels it was 25 launches and a host
// synchronisation for the mask sum, 296 us; it takes 21 us (k_rows 12, k_update 4.5).
// -----------------------------------------------------------------------------
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <type_traits>
#include <vector>

#include "sunamd/learned_predictor.h"

namespace
{

constexpr int IN  = SUNAMD_MLP_IN_PAD;
constexpr int HID = SUNAMD_MLP_HID;
constexpr int OUT = SUNAMD_MLP_OUT;
// parameter offsets (floats)
constexpr long OW1 = 0;
constexpr long OB1 = OW1 + (long)HID * IN;
constexpr long OW2 = OB1 + HID;
constexpr long OB2 = OW2 + (long)HID * HID;
constexpr long OW3 = OB2 + HID;
constexpr long OB3 = OW3 + (long)OUT * HID;
constexpr long NP  = OB3 + OUT;
static_assert(NP == SUNAMD_MLP_NPARAM, "parameter layout");
// device weight block used by the integrator: bf16 W1 W2 W3, then FP32 biases
constexpr long NW_BF16 = (long)HID * IN + (long)HID * HID + (long)OUT * HID;

typedef float f32x4 __attribute__((ext_vector_type(4)));

__host__ __device__ inline uint16_t to_bf16(float f)
{
  uint32_t u;
  memcpy(&u, &f, 4);
  if ((u & 0x7f800000u) == 0x7f800000u && (u & 0x007fffffu)) { return (uint16_t)((u >> 16) | 0x40); }
  u += 0x7fffu + ((u >> 16) & 1u); // round to nearest even
  return (uint16_t)(u >> 16);
}

__host__ __device__ inline float from_bf16(uint16_t h)
{
  uint32_t u = (uint32_t)h << 16;
  float f;
  memcpy(&f, &u, 4);
  return f;
}

__device__ inline float silu(float z) { return z / (1.0f + expf(-z)); }

__device__ inline float dsilu(float z)
{
  float s = 1.0f / (1.0f + expf(-z));
  return s * (1.0f + z * (1.0f - s));
}

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

// device arrays one training step reads and writes
struct Net
{
  float* p;                        // FP32 master parameters
  float *m, *v;                    // Adam moments
  float* g;                        // gradient (where it is asked for)
  uint16_t *w1, *w2, *w3;          // bf16 weights, row-major [out][in]
  uint16_t *w2t, *w3t;             // their transposes [in][out], for the backward products
  float* bias;                     // b1 b2 b3
  uint16_t *xt, *a1t, *a2t;        // bf16 activations, transposed: [feature][row], row stride ldt
  uint16_t *dyt, *dz2t, *dz1t;     // bf16 output / hidden gradients, transposed likewise
  float* y;                        // [row][OUT] outputs (forward only)
  float* bpart;                    // per workgroup of k_rows: its rows' sums of dz1, dz2, dy
  float* lpart;                    // per workgroup of k_rows: its rows' squared error
  long ldt;
};

constexpr int RT     = 16;   // rows per workgroup of k_rows
constexpr int NB     = 2 * HID + OUT;
constexpr int XS     = 168;  // LDS row strides (bf16): 16-byte aligned rows, the 16 rows' operand
constexpr int HS     = 136;  // reads in different banks
constexpr int YS     = 72;
constexpr int MPARTS = 16;   // partial mask sums per step

// NS operands of row `row` (K contiguous bf16 at w + row * ld) for the lane's
// quarter of each 32-deep slice; k >= kmax reads as zero
template <int NS>
__device__ __forceinline__ void load_operands(const uint16_t* __restrict__ w, int row, int ld,
                                              int q, int kmax, bf16x8_t (&o)[NS])
{
#pragma unroll
  for (int t = 0; t < NS; t++)
  {
    const int k = 32 * t + 8 * q;
    o[t]        = *reinterpret_cast<const bf16x8_t*>(w + (long)row * ld + (k < kmax ? k : 0));
    if (k >= kmax) { o[t] = bf16x8_t{}; }
  }
}

// the 16 x 16 tile of in[16 x 32 NS] (LDS, row stride ls) times the operands:
// lane l holds rows 4(l/16) .. 4(l/16)+3 of column l%16
template <int NS>
__device__ __forceinline__ f32x4 tile_product(const uint16_t* in, int ls, int r, int q,
                                              const bf16x8_t (&o)[NS])
{
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int t = 0; t < NS; t++)
  {
    const bf16x8_t a = *reinterpret_cast<const bf16x8_t*>(in + r * ls + 32 * t + 8 * q);
    acc              = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, o[t], acc, 0, 0, 0);
  }
  return acc;
}

// a lane's four rows of one column into row-major LDS and, as 8 bytes, into
// the transposed array
__device__ __forceinline__ void put_column(const float (&v)[4], uint16_t* lds, int ls, int q,
                                           int col, uint16_t* __restrict__ t, long ldt, long row0)
{
  uint16_t h[4];
#pragma unroll
  for (int i = 0; i < 4; i++)
  {
    h[i] = to_bf16(v[i]);
    if (lds) { lds[(4 * q + i) * ls + col] = h[i]; }
  }
  if (t)
  {
    uint2 u;
    u.x = (uint32_t)h[0] | ((uint32_t)h[1] << 16);
    u.y = (uint32_t)h[2] | ((uint32_t)h[3] << 16);
    *reinterpret_cast<uint2*>(t + (long)col * ldt + row0 + 4 * q) = u;
  }
}

// sum of a column over the workgroup's 16 rows (every lane of the column)
__device__ __forceinline__ float column_sum(const float (&v)[4])
{
  float s = (v[0] + v[1]) + (v[2] + v[3]);
  s += __shfl_xor(s, 16, 64);
  s += __shfl_xor(s, 32, 64);
  return s;
}

// Forward (TRAIN = false: outputs to N.y) or forward and backward pass of 16
// rows, eight wavefronts, wavefront w owning columns 16 w .. 16 w + 15 of the
// hidden layers.  A lane keeps the pre-activations of its tile in registers
// from the forward to the backward pass.  All weight operands of the pass are
// requested before its first product, so their latency is paid once.
// The loss is divided by the mask's sum: inv_host is its reciprocal, or, where
// msum is given, msum[MPARTS] are partial sums of the mask on the device.
template <bool TRAIN>
__global__ void __launch_bounds__(512) k_rows(Net N, const float* __restrict__ x,
                                              const float* __restrict__ t,
                                              const float* __restrict__ mk, int B, float inv_host,
                                              const float* __restrict__ msum)
{
  __shared__ __align__(16) uint16_t sx[RT * XS];
  __shared__ __align__(16) uint16_t h1[RT * HS];
  __shared__ __align__(16) uint16_t h2[RT * HS];
  __shared__ __align__(16) uint16_t sdy[RT * YS];
  __shared__ __align__(16) uint16_t sdz[RT * HS];
  __shared__ float sl[4];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int r = lane & 15, q = lane >> 4;
  const long row0 = (long)blockIdx.x * RT;
  const int col   = 16 * wave + r;
  const bool last = wave < OUT / 16; // this wavefront owns output columns too

  bf16x8_t o1[5], o2[4], o3[4], o3t[2], o2t[4];
  load_operands<5>(N.w1, col, IN, q, IN, o1);
  load_operands<4>(N.w2, col, HID, q, HID, o2);
  if (last) { load_operands<4>(N.w3, col, HID, q, HID, o3); }
  if (TRAIN)
  {
    load_operands<2>(N.w3t, col, OUT, q, OUT, o3t);
    load_operands<4>(N.w2t, col, HID, q, HID, o2t);
  }
  const float b1 = N.bias[col], b2 = N.bias[HID + col];
  const float b3 = last ? N.bias[2 * HID + col] : 0.0f;
  float tv[4] = {0, 0, 0, 0}, mv[4] = {0, 0, 0, 0};
  if (TRAIN && last)
  {
#pragma unroll
    for (int i = 0; i < 4; i++)
    {
      tv[i] = t[(row0 + 4 * q + i) * OUT + col];
      mv[i] = mk[(row0 + 4 * q + i) * OUT + col];
    }
  }
  for (int e = tid; e < RT * 160; e += 512)
  {
    const int row = e / 160, k = e % 160;
    sx[row * XS + k] = (k < IN) ? to_bf16(x[(row0 + row) * IN + k]) : (uint16_t)0;
  }
  float inv = inv_host;
  if (TRAIN && msum)
  {
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < MPARTS; i++) { s += msum[i]; }
    inv = s > 0.0f ? 1.0f / s : 0.0f;
  }
  __syncthreads();

  float z1[4], z2[4], v[4];
  const f32x4 c1 = tile_product<5>(sx, XS, r, q, o1);
#pragma unroll
  for (int i = 0; i < 4; i++)
  {
    z1[i] = c1[i] + b1;
    v[i]  = silu(z1[i]);
  }
  put_column(v, h1, HS, q, col, TRAIN ? N.a1t : nullptr, N.ldt, row0);
  if (TRAIN)
  {
    // the inputs, transposed: thread j < IN writes feature j's 16 rows
    if (tid < IN)
    {
      uint32_t u[RT / 2];
#pragma unroll
      for (int i = 0; i < RT / 2; i++)
      {
        u[i] = (uint32_t)sx[2 * i * XS + tid] | ((uint32_t)sx[(2 * i + 1) * XS + tid] << 16);
      }
      uint4* d = reinterpret_cast<uint4*>(N.xt + (long)tid * N.ldt + row0);
      d[0]     = make_uint4(u[0], u[1], u[2], u[3]);
      d[1]     = make_uint4(u[4], u[5], u[6], u[7]);
    }
  }
  __syncthreads();
  const f32x4 c2 = tile_product<4>(h1, HS, r, q, o2);
#pragma unroll
  for (int i = 0; i < 4; i++)
  {
    z2[i] = c2[i] + b2;
    v[i]  = silu(z2[i]);
  }
  put_column(v, h2, HS, q, col, TRAIN ? N.a2t : nullptr, N.ldt, row0);
  __syncthreads();
  if (last)
  {
    const f32x4 c3 = tile_product<4>(h2, HS, r, q, o3);
    if (!TRAIN)
    {
#pragma unroll
      for (int i = 0; i < 4; i++) { N.y[(row0 + 4 * q + i) * OUT + col] = c3[i] + b3; }
    }
    else
    {
      // masked squared error and dY = 2 mask (Y - T) / (mask sum)
      float se = 0.0f;
#pragma unroll
      for (int i = 0; i < 4; i++)
      {
        const float d = (c3[i] + b3 - tv[i]) * mv[i];
        se += d * d;
        v[i] = 2.0f * d * inv;
      }
      put_column(v, sdy, YS, q, col, N.dyt, N.ldt, row0);
      const float cs = column_sum(v);
      if (q == 0) { N.bpart[(long)blockIdx.x * NB + 2 * HID + col] = cs; }
      for (int off = 32; off >= 1; off >>= 1) { se += __shfl_xor(se, off, 64); }
      if (lane == 0) { sl[wave] = se; }
    }
  }
  if (!TRAIN) { return; }
  __syncthreads();
  if (tid == 0) { N.lpart[blockIdx.x] = (((sl[0] + sl[1]) + sl[2]) + sl[3]) * inv; }
  const f32x4 e2 = tile_product<2>(sdy, YS, r, q, o3t);
#pragma unroll
  for (int i = 0; i < 4; i++) { v[i] = e2[i] * dsilu(z2[i]); }
  put_column(v, sdz, HS, q, col, N.dz2t, N.ldt, row0);
  const float s2 = column_sum(v);
  if (q == 0) { N.bpart[(long)blockIdx.x * NB + HID + col] = s2; }
  __syncthreads();
  const f32x4 e1 = tile_product<4>(sdz, HS, r, q, o2t);
#pragma unroll
  for (int i = 0; i < 4; i++) { v[i] = e1[i] * dsilu(z1[i]); }
  put_column(v, nullptr, 0, q, col, N.dz1t, N.ldt, row0);
  const float s1 = column_sum(v);
  if (q == 0) { N.bpart[(long)blockIdx.x * NB + col] = s1; }
  // an odd number of row blocks: the 32-deep slices of k_update read 16 rows
  // more, which are zero
  if ((B & 31) != 0 && row0 + RT == B)
  {
    for (int e = tid; e < IN + 4 * HID + OUT; e += 512)
    {
      uint16_t* d = (e < IN)                   ? N.xt + (long)e * N.ldt
                    : (e < IN + HID)           ? N.a1t + (long)(e - IN) * N.ldt
                    : (e < IN + 2 * HID)       ? N.a2t + (long)(e - IN - HID) * N.ldt
                    : (e < IN + 3 * HID)       ? N.dz2t + (long)(e - IN - 2 * HID) * N.ldt
                    : (e < IN + 4 * HID)       ? N.dz1t + (long)(e - IN - 3 * HID) * N.ldt
                                               : N.dyt + (long)(e - IN - 4 * HID) * N.ldt;
      uint4* z = reinterpret_cast<uint4*>(d + B);
      z[0]     = make_uint4(0, 0, 0, 0);
      z[1]     = make_uint4(0, 0, 0, 0);
    }
  }
}

struct AdamStep
{
  float lr, b1, b2, c1, c2, eps;
  int gradient_only; // no update, the gradient goes to Net::g
};

// one parameter's update from its value p0 and moments m0, v0; returns its
// new value
__device__ __forceinline__ float adam(const Net& N, const AdamStep& S, long i, float gi, float p0,
                                      float m0, float v0)
{
  const float mi = S.b1 * m0 + (1.0f - S.b1) * gi;
  const float vi = S.b2 * v0 + (1.0f - S.b2) * gi * gi;
  N.m[i]         = mi;
  N.v[i]         = vi;
  const float p  = p0 - S.lr * (mi / S.c1) / (sqrtf(vi / S.c2) + S.eps);
  N.p[i]         = p;
  return p;
}

constexpr int T1 = (HID / 16) * (IN / 16), T2 = (HID / 16) * (HID / 16), T3 = (OUT / 16) * (HID / 16);

// Gradient and update of one 16 x 16 tile of W1, W2 or W3 (workgroups
// 0 .. T1+T2+T3-1): dW[o][i] = sum over the batch of dz[b][o] act[b][i], the
// batch in 32-deep slices dealt to the four wavefronts in turn, their sums
// added in wavefront order.  The NB / 64 workgroups after those do the biases
// from the row blocks' column sums, the first of them also the loss.
__global__ void __launch_bounds__(256) k_update(Net N, AdamStep S, int B, float* __restrict__ loss)
{
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  int b = blockIdx.x;
  if (b >= T1 + T2 + T3)
  {
    // 64 bias entries: the row blocks dealt to the four wavefronts in turn
    __shared__ float sum[4][64];
    const int j  = (b - T1 - T2 - T3) * 64 + lane;
    const int nw = B / RT;
    float s      = 0.0f;
    int k        = wave;
    for (; k + 28 < nw; k += 32)
    {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; u++) { v[u] = N.bpart[(long)(k + 4 * u) * NB + j]; }
#pragma unroll
      for (int u = 0; u < 8; u++) { s += v[u]; }
    }
    for (; k < nw; k += 4) { s += N.bpart[(long)k * NB + j]; }
    sum[wave][lane] = s;
    __syncthreads();
    if (wave == 0)
    {
      s = ((sum[0][lane] + sum[1][lane]) + sum[2][lane]) + sum[3][lane];
      const long i = (j < HID) ? OB1 + j : (j < 2 * HID) ? OB2 + (j - HID) : OB3 + (j - 2 * HID);
      if (S.gradient_only) { N.g[i] = s; }
      else { N.bias[j] = adam(N, S, i, s, N.p[i], N.m[i], N.v[i]); }
    }
    else if (wave == 1 && b == T1 + T2 + T3)
    {
      float e = 0.0f;
      for (int w = lane; w < nw; w += 64) { e += N.lpart[w]; }
      for (int off = 32; off >= 1; off >>= 1) { e += __shfl_xor(e, off, 64); }
      if (lane == 0) { *loss = e; }
    }
    return;
  }
  const uint16_t *dz, *act;
  uint16_t *w, *wt;
  long off;
  int tiles, ld, ldw;
  if (b < T1) { dz = N.dz1t; act = N.xt; w = N.w1; wt = nullptr; off = OW1; tiles = IN / 16; ld = IN; ldw = 0; }
  else if (b < T1 + T2)
  {
    b -= T1;
    dz = N.dz2t; act = N.a1t; w = N.w2; wt = N.w2t; off = OW2; tiles = HID / 16; ld = HID; ldw = HID;
  }
  else
  {
    b -= T1 + T2;
    dz = N.dyt; act = N.a2t; w = N.w3; wt = N.w3t; off = OW3; tiles = HID / 16; ld = HID; ldw = OUT;
  }
  const int o0 = 16 * (b / tiles), i0 = 16 * (b % tiles);
  const int r = lane & 15, q = lane >> 4;
  const uint16_t* pa = dz + (long)(o0 + r) * N.ldt + 8 * q;
  const uint16_t* pb = act + (long)(i0 + r) * N.ldt + 8 * q;
  // the parameter of this thread and its moments, on their way meanwhile
  const int o = tid >> 4, c = tid & 15;
  const long wi  = (long)(o0 + o) * ld + i0 + c;
  const float p0 = N.p[off + wi], m0 = N.m[off + wi], v0 = N.v[off + wi];
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  const int slices = (B + 31) / 32;
  int s = wave;
  // eight slices' operands in flight before the first product
  for (; s + 28 < slices; s += 32)
  {
    bf16x8_t x[8], y[8];
#pragma unroll
    for (int u = 0; u < 8; u++)
    {
      x[u] = *reinterpret_cast<const bf16x8_t*>(pa + 32L * (s + 4 * u));
      y[u] = *reinterpret_cast<const bf16x8_t*>(pb + 32L * (s + 4 * u));
    }
#pragma unroll
    for (int u = 0; u < 8; u++) { acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[u], y[u], acc, 0, 0, 0); }
  }
  for (; s < slices; s += 4)
  {
    const bf16x8_t x = *reinterpret_cast<const bf16x8_t*>(pa + 32L * s);
    const bf16x8_t y = *reinterpret_cast<const bf16x8_t*>(pb + 32L * s);
    acc              = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, y, acc, 0, 0, 0);
  }
  __shared__ float part[4][16][17];
#pragma unroll
  for (int i = 0; i < 4; i++) { part[wave][4 * q + i][r] = acc[i]; }
  __syncthreads();
  const float gi = ((part[0][o][c] + part[1][o][c]) + part[2][o][c]) + part[3][o][c];
  if (S.gradient_only)
  {
    N.g[off + wi] = gi;
    return;
  }
  const uint16_t h = to_bf16(adam(N, S, off + wi, gi, p0, m0, v0));
  w[wi]            = h;
  if (wt) { wt[(long)(i0 + c) * ldw + o0 + o] = h; }
}

// partial sums of the mask of steps k0 .. k0 + gridDim.y - 1 (each step's batch
// as in SUNAMD_MLPTrain), MPARTS per step, in a fixed order
__global__ void __launch_bounds__(256) k_masksum(const float* __restrict__ mask, long n, int batch,
                                                 long k0, float* __restrict__ out)
{
  __shared__ float part[4];
  long start = ((k0 + blockIdx.y) * batch) % n;
  if (start + batch > n) { start = n - batch; }
  const float* mk  = mask + start * OUT;
  const long total = (long)batch * OUT, per = total / MPARTS; // batch % 16 == 0
  float s          = 0.0f;
  for (long i = threadIdx.x; i < per; i += 256) { s += mk[blockIdx.x * per + i]; }
  for (int off = 32; off >= 1; off >>= 1) { s += __shfl_xor(s, off, 64); }
  if ((threadIdx.x & 63) == 0) { part[threadIdx.x >> 6] = s; }
  __syncthreads();
  if (threadIdx.x == 0) { out[blockIdx.y * MPARTS + blockIdx.x] = ((part[0] + part[1]) + part[2]) + part[3]; }
}

__global__ void k_fill(float* __restrict__ x, long n, float val)
{
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
  {
    x[i] = val;
  }
}

// FP32 master -> device weight block (bf16 weights, FP32 biases) and the
// transposed bf16 copies
__global__ void k_pack(Net N)
{
  const long nw1 = (long)HID * IN, nw2 = (long)HID * HID;
  const float* p = N.p;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < NW_BF16 + NB;
       i += (long)gridDim.x * blockDim.x)
  {
    if (i < nw1) { N.w1[i] = to_bf16(p[OW1 + i]); }
    else if (i < nw1 + nw2)
    {
      const long j         = i - nw1;
      const uint16_t h     = to_bf16(p[OW2 + j]);
      N.w2[j]              = h;
      N.w2t[(j % HID) * HID + j / HID] = h;
    }
    else if (i < NW_BF16)
    {
      const long j         = i - nw1 - nw2;
      const uint16_t h     = to_bf16(p[OW3 + j]);
      N.w3[j]              = h;
      N.w3t[(j % HID) * OUT + j / HID] = h;
    }
    else
    {
      const long j = i - NW_BF16; // b1 b2 b3
      N.bias[j] = (j < HID) ? p[OB1 + j] : (j < 2 * HID) ? p[OB2 + (j - HID)] : p[OB3 + (j - 2 * HID)];
    }
  }
}

unsigned blocks_for(long n) { return (unsigned)((n + 255) / 256 < 2048 ? (n + 255) / 256 : 2048); }

} // namespace

// steps whose mask sums are taken in one launch
static constexpr int MCHUNK = 256;

struct SUNAMD_MLP_
{
  hipStream_t stream;
  int max_batch;
  long t;       // Adam step count
  void* wblock; // bf16 weights + FP32 biases
  void* work;   // everything k_rows and k_update exchange
  Net net;
  float* msum;  // MCHUNK x MPARTS partial mask sums
  float* loss;  // losses of the last ten steps, and of any other in the last entry
  float *hx, *ht, *hm; // staging for the host-array entry points (device)
};

static constexpr int LOSS_TAIL = 10;

static int mfail(hipError_t e, const char* what)
{
  fprintf(stderr, "[sundials_amd mlp] %s: %s\n", what, hipGetErrorString(e));
  return -1;
}

#define MCHK(call, what)                                 \
  do {                                                   \
    hipError_t e_ = (call);                              \
    if (e_ != hipSuccess) { return mfail(e_, what); }    \
  } while (0)

static int repack(SUNAMD_MLP* M)
{
  k_pack<<<blocks_for(NW_BF16 + NB), 256, 0, M->stream>>>(M->net);
  MCHK(hipGetLastError(), "pack");
  return 0;
}

extern "C" SUNAMD_MLP* SUNAMD_MLPCreate(uint64_t seed, int max_batch)
{
  if (max_batch < 16 || max_batch % 16) { return NULL; }
  SUNAMD_MLP* M = (SUNAMD_MLP*)calloc(1, sizeof(SUNAMD_MLP));
  if (!M) { return NULL; }
  M->max_batch = max_batch;
  const long B = max_batch;
  Net& N       = M->net;
  // transposed rows: a whole number of 32-row slices, and 8 entries more so
  // that consecutive features do not start in the same memory channel
  N.ldt        = (B + 31) / 32 * 32 + 8;
  bool ok      = hipStreamCreateWithFlags(&M->stream, hipStreamNonBlocking) == hipSuccess;
  ok = ok && hipMalloc(&M->wblock, sizeof(uint16_t) * NW_BF16 + sizeof(float) * NB) == hipSuccess;
  // one allocation for the rest, each array 256-byte aligned: sizes first,
  // then the pointers
  char* at     = nullptr;
  auto carve   = [&](auto** ptr, long elems) {
    *ptr = reinterpret_cast<std::remove_reference_t<decltype(*ptr)>>(at);
    at += (sizeof(**ptr) * (size_t)elems + 255) / 256 * 256;
  };
  auto layout = [&]() {
    carve(&N.p, NP);
    carve(&N.g, NP);
    carve(&N.m, NP);
    carve(&N.v, NP);
    carve(&N.w2t, (long)HID * HID);
    carve(&N.w3t, (long)HID * OUT);
    carve(&N.xt, (long)IN * N.ldt);
    carve(&N.a1t, (long)HID * N.ldt);
    carve(&N.a2t, (long)HID * N.ldt);
    carve(&N.dz1t, (long)HID * N.ldt);
    carve(&N.dz2t, (long)HID * N.ldt);
    carve(&N.dyt, (long)OUT * N.ldt);
    carve(&N.y, B * OUT);
    carve(&N.bpart, B / RT * NB);
    carve(&N.lpart, B / RT);
    carve(&M->msum, (long)MCHUNK * MPARTS);
    carve(&M->loss, LOSS_TAIL + 1);
    carve(&M->hx, B * IN);
    carve(&M->ht, B * OUT);
    carve(&M->hm, B * OUT);
  };
  layout();
  const size_t bytes = (size_t)(at - (char*)nullptr);
  ok                 = ok && hipMalloc(&M->work, bytes) == hipSuccess;
  if (!ok)
  {
    SUNAMD_MLPFree(M);
    return NULL;
  }
  at = (char*)M->work;
  layout();
  N.w1   = (uint16_t*)M->wblock;
  N.w2   = N.w1 + (long)HID * IN;
  N.w3   = N.w2 + (long)HID * HID;
  N.bias = (float*)(N.w1 + NW_BF16);
  // seeded init on the host (SplitMix64 -> uniform)
  std::vector<float> h(NP, 0.0f);
  uint64_t st = seed * 0x9E3779B97F4A7C15ull + 0x632BE59BD9B4E5Full;
  auto uni    = [&]() {
    st += 0x9E3779B97F4A7C15ull;
    uint64_t z = st;
    z          = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z          = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return (double)(z >> 11) * (1.0 / 9007199254740992.0);
  };
  auto init = [&](long off, int nout, int nin, int nin_used, double scale) {
    double a = scale * std::sqrt(6.0 / nin_used);
    for (int o = 0; o < nout; o++)
    {
      for (int i = 0; i < nin; i++)
      {
        h[off + (long)o * nin + i] = (i < nin_used) ? (float)((2.0 * uni() - 1.0) * a) : 0.0f;
      }
    }
  };
  init(OW1, HID, IN, SUNAMD_MLP_IN, 1.0);
  init(OW2, HID, HID, HID, 1.0);
  init(OW3, OUT, HID, HID, 0.1);
  if (SUNAMD_MLPSetParams(M, h.data()) != 0)
  {
    SUNAMD_MLPFree(M);
    return NULL;
  }
  return M;
}

extern "C" void SUNAMD_MLPFree(SUNAMD_MLP* M)
{
  if (!M) { return; }
  if (M->stream) { (void)hipStreamSynchronize(M->stream); }
  if (M->wblock) { (void)hipFree(M->wblock); }
  if (M->work) { (void)hipFree(M->work); }
  if (M->stream) { (void)hipStreamDestroy(M->stream); }
  free(M);
}

extern "C" int SUNAMD_MLPGetParams(SUNAMD_MLP* M, float* params)
{
  MCHK(hipStreamSynchronize(M->stream), "sync");
  MCHK(hipMemcpy(params, M->net.p, sizeof(float) * NP, hipMemcpyDeviceToHost), "get params");
  return 0;
}

extern "C" int SUNAMD_MLPSetParams(SUNAMD_MLP* M, const float* params)
{
  MCHK(hipStreamSynchronize(M->stream), "sync");
  MCHK(hipMemcpy(M->net.p, params, sizeof(float) * NP, hipMemcpyHostToDevice), "set params");
  k_fill<<<blocks_for(NP), 256, 0, M->stream>>>(M->net.m, NP, 0.0f);
  k_fill<<<blocks_for(NP), 256, 0, M->stream>>>(M->net.v, NP, 0.0f);
  M->t = 0;
  if (repack(M) != 0) { return -1; }
  MCHK(hipStreamSynchronize(M->stream), "set params sync");
  return 0;
}

extern "C" const void* SUNAMD_MLPDeviceWeights(SUNAMD_MLP* M) { return M->wblock; }

// forward pass of device rows x[B x IN] into net.y
static void forward_dev(SUNAMD_MLP* M, const float* x, int B)
{
  k_rows<false><<<B / RT, 512, 0, M->stream>>>(M->net, x, nullptr, nullptr, B, 0.0f, nullptr);
}

// loss and gradient of device rows (x, t, mask), then the update or (S's
// gradient_only) the gradient in net.g; the mask's sum as in k_rows
static void step_dev(SUNAMD_MLP* M, const float* x, const float* t, const float* mk, int B,
                     float inv, const float* msum, const AdamStep& S, float* loss)
{
  k_rows<true><<<B / RT, 512, 0, M->stream>>>(M->net, x, t, mk, B, inv, msum);
  k_update<<<T1 + T2 + T3 + NB / 64, 256, 0, M->stream>>>(M->net, S, B, loss);
}

extern "C" int SUNAMD_MLPForward(SUNAMD_MLP* M, const float* x, int B, float* y)
{
  if (B <= 0 || B > M->max_batch || B % 16) { return -1; }
  MCHK(hipMemcpyAsync(M->hx, x, sizeof(float) * B * IN, hipMemcpyHostToDevice, M->stream), "x");
  forward_dev(M, M->hx, B);
  MCHK(hipGetLastError(), "forward");
  MCHK(hipMemcpyAsync(y, M->net.y, sizeof(float) * B * OUT, hipMemcpyDeviceToHost, M->stream), "y");
  MCHK(hipStreamSynchronize(M->stream), "forward sync");
  return 0;
}

extern "C" int SUNAMD_MLPLossGrad(SUNAMD_MLP* M, const float* x, const float* t, const float* mask,
                                  int B, float* loss, float* grad)
{
  if (B <= 0 || B > M->max_batch || B % 16) { return -1; }
  float msum = 0.0f;
  for (long i = 0; i < (long)B * OUT; i++) { msum += mask[i]; }
  MCHK(hipMemcpyAsync(M->hx, x, sizeof(float) * B * IN, hipMemcpyHostToDevice, M->stream), "x");
  MCHK(hipMemcpyAsync(M->ht, t, sizeof(float) * B * OUT, hipMemcpyHostToDevice, M->stream), "t");
  MCHK(hipMemcpyAsync(M->hm, mask, sizeof(float) * B * OUT, hipMemcpyHostToDevice, M->stream),
       "mask");
  const AdamStep none = {0.0f, 0.0f, 0.0f, 1.0f, 1.0f, 0.0f, 1};
  step_dev(M, M->hx, M->ht, M->hm, B, msum > 0.0f ? 1.0f / msum : 0.0f, nullptr, none, M->loss);
  MCHK(hipGetLastError(), "backward");
  MCHK(hipMemcpyAsync(loss, M->loss, sizeof(float), hipMemcpyDeviceToHost, M->stream), "loss");
  MCHK(hipMemcpyAsync(grad, M->net.g, sizeof(float) * NP, hipMemcpyDeviceToHost, M->stream),
       "grad");
  MCHK(hipStreamSynchronize(M->stream), "grad sync");
  return 0;
}

extern "C" int SUNAMD_MLPTrain(SUNAMD_MLP* M, const float* x_dev, const float* t_dev,
                               const float* mask_dev, long n, int batch, int steps, float lr,
                               float* loss)
{
  if (batch <= 0 || batch > M->max_batch || batch % 16 || n < batch) { return -1; }
  hipStream_t s = M->stream;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const int first_tail = steps > LOSS_TAIL ? steps - LOSS_TAIL : 0;
  for (int k = 0; k < steps; k++)
  {
    if (k % MCHUNK == 0)
    {
      const int cnt = steps - k < MCHUNK ? steps - k : MCHUNK;
      k_masksum<<<dim3(MPARTS, (unsigned)cnt), 256, 0, s>>>(mask_dev, n, batch, k, M->msum);
    }
    long start = ((long)k * batch) % n;
    if (start + batch > n) { start = n - batch; }
    M->t++;
    const AdamStep S = {lr, b1, b2, 1.0f - powf(b1, (float)M->t), 1.0f - powf(b2, (float)M->t),
                        eps, 0};
    step_dev(M, x_dev + start * IN, t_dev + start * OUT, mask_dev + start * OUT, batch, 0.0f,
             M->msum + (k % MCHUNK) * MPARTS, S,
             M->loss + (k >= first_tail ? k - first_tail : LOSS_TAIL));
    MCHK(hipGetLastError(), "train step");
  }
  const int ntail = steps > 0 ? steps - first_tail : 0;
  float tail[LOSS_TAIL];
  if (ntail)
  {
    MCHK(hipMemcpyAsync(tail, M->loss, sizeof(float) * ntail, hipMemcpyDeviceToHost, s), "loss");
  }
  MCHK(hipStreamSynchronize(s), "train sync");
  double sum = 0.0;
  for (int k = 0; k < ntail; k++) { sum += tail[k]; }
  if (loss) { *loss = ntail ? (float)(sum / ntail) : 0.0f; }
  return 0;
}
