// vision_split.hip -- the vision tower's products and attention on the fp16 matrix units without
// giving up fp32: an fp32 operand X is held as two fp16 parts, hi = fp16(s X) and
// lo = fp16(s X - hi), with s a power of two that keeps |s X| at or below 2^15.  hi + lo carries
// 23 to 24 significant bits of every value down to 2^-16 of the bound s was made for, and an
// absolute error of 2^-40 of the bound below that, so a product over the two parts rounds like
// the fp32 one (the sums stay in fp32 inside the MFMA) as long as the bound is not far above what
// most values have, which the weights tell (k_vis_rows; api_vision.hip's kVisSpread): where it is, the
// product runs in fp32.  The weights of an mmproj-f16 file are fp16 values, and bf16 ones are fp16
// values times a power of two where a matrix's smallest are within about 2^-31 of its largest (one
// below leaves the product in fp32): exact in one part, so
// Y = X W^T takes two fp16 MFMAs (hi, lo) where v_mfma_f32_16x16x4_f32 needed eight of twice the
// length: 16 times the rate over 2.  The bounds come from the weights alone (api_vision.hip):
// LayerNorm's output is at most sqrt(D) max|g| + max|b| whatever its input.
//
//   k_vis_stats   max |x| and the largest row norm of a tensor, for the bounds;
//   k_vis_pack    a matrix as fp16 rows, a flag when a value is not exact;
//   k_vis_square, k_vis_rows  the sizes that inputs and outputs have, from the weights;
//   k_vis_gemm_s  Y = X W^T + b (+ R) (then GELU), X split, W fp16;
//   k_vis_ln_s    LayerNorm into split rows, over the sum of a split product's parts;
//   k_vis_heads_s QKV rows into split heads, the rotary applied;
//   k_vis_attend_s softmax attention over split q, k, v and probabilities.
//
// Split rows: a row of K values is Kp/32 blocks of 128 bytes (Kp = K rounded up to 64, zeros past
// K), each 32 hi halves then their 32 lo halves: 4 bytes a value, as fp32.
#include "exn_common.h"

#include <algorithm>
#include <type_traits>

namespace exn {

typedef __attribute__((address_space(3))) void lds_void;

#define VS_VOFF_NONE 0x80000000u   // past any extent: the DMA reads zeros

static inline unsigned sgrid(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

__device__ __forceinline__ void sdma16(const void* base, uint32_t extent, lds_void* dst, uint32_t voff, int soff) {
  __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)extent, 0x00020000);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, dst, 16, voff, soff, 0, 0);
}

// vmcnt(VM), lgkmcnt(0), then the workgroup's barrier
template <int VM>
__device__ __forceinline__ void wait_dma_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((VM & 15) | (0x7 << 4) | (0x0 << 8) | ((VM >> 4) << 14));
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// four values, already scaled, into their hi and lo halves.  The packed hi passes through an empty
// asm, so that lo is taken from the very bits stored: the compiler would otherwise convert twice,
// and where V is a product round once in one step (v_fma_mixlo_f16) and once in two, which differ on
// a tie.  The difference is one v_fma_mix_f32 a value.
__device__ __forceinline__ void split4(const f32x4 v, u32x2& hi, u32x2& lo) {
  uint32_t h0 = pack_f16x2(v[0], v[1]), h1 = pack_f16x2(v[2], v[3]);
  asm("" : "+v"(h0), "+v"(h1));
  hi = u32x2{h0, h1};
  lo = u32x2{pack_f16x2(__builtin_fmaf(f16_lo(h0), -1.f, v[0]), __builtin_fmaf(f16_hi(h0), -1.f, v[1])),
             pack_f16x2(__builtin_fmaf(f16_lo(h1), -1.f, v[2]), __builtin_fmaf(f16_hi(h1), -1.f, v[3]))};
}

// where column K (a multiple of 4) of a split row lies, in halves; its lo part is 32 further
__device__ __forceinline__ int split_at(int k) { return (k >> 5) * 64 + (k & 31); }

// --- the weights -----------------------------------------------------------------------------

// N fp16 (or bf16) values as fp32, subnormals, infinities and NaNs kept
__global__ void k_vis_widen(int64_t n, const uint16_t* __restrict__ x, int bf16, float* __restrict__ y) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) y[i] = bf16 ? bf16_to_f32(x[i]) : f16_to_f32(x[i]);
}

hipError_t vis_widen(hipStream_t s, int64_t n, const uint16_t* x, int bf16, float* y) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_vis_widen, dim3(sgrid(n, 256)), dim3(256), 0, s, n, x, bf16, y);
  return hipGetLastError();
}

// rec[0] = the bits of the largest |x|, rec[2] and rec[3] those of the largest row's sum of squares in
// double, which no fp32 row makes 0 or infinite (NaNs compare above every number, so a bound made
// from a tensor that holds one is not finite)
__global__ void __launch_bounds__(256)
k_vis_stats(int64_t rows, int64_t cols, const float* __restrict__ x, uint32_t* __restrict__ rec) {
  // a wave a row; one pair of atomics a workgroup (one a row took 100 us for 4304 rows)
  typedef unsigned long long u64;
  __shared__ uint32_t rm[4];
  __shared__ u64 rs[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t mb = 0u;
  u64 sb = 0u;
  for (int64_t row = (int64_t)blockIdx.x * 4 + wave; row < rows; row += (int64_t)gridDim.x * 4) {
    const float* r = x + row * cols;
    double s = 0.0;
    for (int64_t i = lane; i < cols; i += 64) {
      const float v = r[i];
      mb = max(mb, __float_as_uint(fabsf(v)));
      s += (double)v * (double)v;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    sb = max(sb, (u64)__double_as_longlong(fabs(s)));
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mb = max(mb, (uint32_t)__shfl_xor((int)mb, o, 64));
  if (lane == 0) {
    rm[wave] = mb;
    rs[wave] = sb;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    atomicMax(rec, max(max(rm[0], rm[1]), max(rm[2], rm[3])));
    atomicMax((u64*)(rec + 2), max(max(rs[0], rs[1]), max(rs[2], rs[3])));
  }
}

hipError_t vis_stats(hipStream_t s, int64_t rows, int64_t cols, const float* x, uint32_t* rec) {
  if (rows <= 0 || cols <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_vis_stats, dim3((unsigned)std::min<int64_t>((rows + 3) / 4, 512)), dim3(256), 0, s, rows, cols, x,
                     rec);
  return hipGetLastError();
}

// rows of K floats, times SCALE, as fp16 in the product's order: for each 32 columns of KP, the NP
// rows' 64 bytes (rows past ROWS and columns past K zero), so that a tile's k-step is one run of
// whole cache lines; *INEXACT set when a value changes
__global__ void __launch_bounds__(256)
k_vis_pack(int rows, int K, int KP, float scale, const float* __restrict__ x, uint16_t* __restrict__ y,
           uint32_t* inexact) {
  const int row = blockIdx.x, NP = gridDim.x;
  const float* r = x + (int64_t)row * K;
  bool bad = false;
  for (int i = threadIdx.x; i < KP; i += 256) {
    const float v = i < K && row < rows ? r[i] * scale : 0.f;
    const _Float16 h = (_Float16)v;
    bad |= (float)h != v;
    y[((int64_t)(i >> 5) * NP + row) * 32 + (i & 31)] = __builtin_bit_cast(uint16_t, h);
  }
  if (bad) atomicOr(inexact, 1u);
}

hipError_t vis_pack(hipStream_t s, int64_t rows, int K, int KP, float scale, const float* x, uint16_t* y,
                    uint32_t* inexact) {
  if (rows <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_vis_pack, dim3((unsigned)((rows + 63) / 64 * 64)), dim3(256), 0, s, (int)rows, K, KP, scale, x, y,
                     inexact);
  return hipGetLastError();
}

// a2[i] = g[i]^2 + b[i]^2: the mean square of a LayerNorm's output i over rows of no structure
__global__ void k_vis_square(int n, const float* __restrict__ g, const float* __restrict__ b, double* __restrict__ a2) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) a2[i] = (double)g[i] * g[i] + (double)b[i] * b[i];
}

hipError_t vis_square(hipStream_t s, int n, const float* g, const float* b, double* a2) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_vis_square, dim3(sgrid(n, 256)), dim3(256), 0, s, n, g, b, a2);
  return hipGetLastError();
}

__device__ __forceinline__ double gelu_d(double x) { return 0.5 * x * (1.0 + erf(x * 0.70710678118654752)); }

// For inputs of mean squares a2 (PERIOD of them, over and over along a row) without structure: t2[j],
// the mean square of W's output j (its deviation T_j about the bias), or of its GELU (three points
// of the normal distribution, exact for polynomials of degree 5), and *SPREAD, the bits of the
// largest |w_j|^2 / T_j^2: how much larger than an output's own size the error of a step of 1 in
// every input is.  A wave a row, sums in double.
__global__ void __launch_bounds__(256)
k_vis_rows(int rows, int cols, const float* __restrict__ w, const double* __restrict__ a2, int period,
           const float* __restrict__ bias, int gelu, double* __restrict__ t2, unsigned long long* spread) {
  const int lane = threadIdx.x & 63, row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const float* r = w + (int64_t)row * cols;
  double q = 0.0, t = 0.0;
  // COLS and PERIOD are multiples of 4: a lane's four columns never cross a period's end
  for (int i = 4 * lane, p = i; i < cols; i += 256, p += 256) {
    while (p >= period) p -= period;
    const f32x4 x = *(const f32x4*)(r + i);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const double v = (double)x[e] * x[e];
      q += v;
      t += v * a2[p + e];
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    q += __shfl_xor(q, o, 64);
    t += __shfl_xor(t, o, 64);
  }
  if (lane) return;
  const double b = bias[row], d = 1.7320508075688772 * sqrt(t);
  const double lo = gelu_d(b - d), md = gelu_d(b), hi = gelu_d(b + d);
  t2[row] = gelu ? (lo * lo + 4.0 * md * md + hi * hi) / 6.0 : t + b * b;
  if (q != 0.0) atomicMax(spread, (unsigned long long)__double_as_longlong(fabs(q / t)));   // a row of zeros has no error
}

hipError_t vis_rows(hipStream_t s, int rows, int cols, const float* w, const double* a2, int period, const float* bias,
                    int gelu, double* t2, double* spread) {
  if (rows <= 0 || cols <= 0) return hipSuccess;
  if (cols % 4 || period % 4 || period <= 0 || ((uintptr_t)w & 15)) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_vis_rows, dim3(sgrid(rows, 4)), dim3(256), 0, s, rows, cols, w, a2, period, bias, gelu, t2,
                     (unsigned long long*)spread);
  return hipGetLastError();
}

// --- LayerNorm -------------------------------------------------------------------------------

// One workgroup a row of WIDTH (a multiple of 4, at most 5120) of X, or, when S > 0, of
// bias + R + the S parts of a split product (each MN floats after the last, summed in order),
// written back to X; then LayerNorm (the mean, the mean square about it, (x - mean) /
// sqrt(var + 1e-6) w + b, as inspect/ref_vision.py:35-38 orders it), times SCALE, into split rows of
// KP, or, when YF is given, as fp32 rows.
__global__ void __launch_bounds__(256)
k_vis_ln_s(int width, int kp, float* __restrict__ x, int S, int64_t mn, const float* __restrict__ part,
           const float* __restrict__ bias, const float* __restrict__ w, const float* __restrict__ b, float scale,
           uint16_t* __restrict__ ys, float* __restrict__ yf) {
#pragma clang fp contract(off)
  __shared__ float red[2][4];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, w4 = width >> 2;
  f32x4* r = (f32x4*)(x + (int64_t)blockIdx.x * width);
  f32x4 v[5];
  float s = 0.f;
#pragma unroll
  for (int e = 0; e < 5; ++e) {
    const int i = t + 256 * e;
    v[e] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (i < w4) {
      v[e] = r[i];
      if (S > 0) {
        f32x4 a = ((const f32x4*)bias)[i];
        for (int p = 0; p < S; ++p) a = a + ((const f32x4*)(part + p * mn + (int64_t)blockIdx.x * width))[i];
        v[e] = a + v[e];
        r[i] = v[e];
      }
    }
    s += (v[e][0] + v[e][1]) + (v[e][2] + v[e][3]);
  }
  s = wave_sum(s);
  if (lane == 0) red[0][wave] = s;
  __syncthreads();
  const float mean = ((red[0][0] + red[0][1]) + (red[0][2] + red[0][3])) / (float)width;
  float q = 0.f;
#pragma unroll
  for (int e = 0; e < 5; ++e)
    if (t + 256 * e < w4)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float d = v[e][j] - mean;
        q += d * d;
      }
  q = wave_sum(q);
  if (lane == 0) red[1][wave] = q;
  __syncthreads();
  const float var = ((red[1][0] + red[1][1]) + (red[1][2] + red[1][3])) / (float)width;
  const float sd = __fsqrt_rn(var + 1e-6f);
#pragma unroll
  for (int e = 0; e < 5; ++e) {
    const int i = t + 256 * e;
    if (i < w4) {
      const f32x4 g = ((const f32x4*)w)[i], bb = ((const f32x4*)b)[i];
      f32x4 z;
#pragma unroll
      for (int j = 0; j < 4; ++j) z[j] = __fdiv_rn(v[e][j] - mean, sd) * g[j] + bb[j];
      if (yf) {
        ((f32x4*)(yf + (int64_t)blockIdx.x * width))[i] = z;
      } else {
        u32x2 hi, lo;
        split4(z * scale, hi, lo);
        uint16_t* o = ys + (int64_t)blockIdx.x * 2 * kp + split_at(4 * i);
        *(u32x2*)o = hi;
        *(u32x2*)(o + 32) = lo;
      }
    }
  }
}

hipError_t vis_ln_s(hipStream_t s, int64_t rows, int width, int kp, float* x, int S, const float* part,
                    const float* bias, const float* w, const float* b, float scale, uint16_t* ys, float* yf) {
  if (rows <= 0) return hipSuccess;
  if (width % 4 || width > 5120 || S < 0 || !ys == !yf) return hipErrorInvalidValue;
  if (ys && (width % 64 || kp != width)) return hipErrorInvalidValue;   // no columns past the width to clear
  hipLaunchKernelGGL(k_vis_ln_s, dim3((unsigned)rows), dim3(256), 0, s, width, kp, x, S, rows * width, part, bias, w, b,
                     scale, ys, yf);
  return hipGetLastError();
}

// --- the product -----------------------------------------------------------------------------

// x sigmoid(2u), u = sqrt(2/pi)(x + 0.044715 x^3): the tanh form of GELU with one exp2 and one
// reciprocal (about 1 ulp each) and no cancellation where tanh nears -1
__device__ __forceinline__ float gelu_sig(float v) {
  const float u2 = 2.3022082f * (v + 0.044715f * v * v * v);   // 2 sqrt(2/pi) log2(e)
  return __fdividef(v, 1.f + __builtin_amdgcn_exp2f(-u2));
}

// Y^T tiles: the W rows are the MFMAs' A operand and the X rows their B, so that a lane ends with
// 4 consecutive output columns of one row (v_mfma_f32_16x16x32_f16, D: lane l holds X row l % 16,
// W rows 4 (l / 16) + e).  Workgroup tiles of BM x BN, WMW x WNW waves of (16 MI) x (16 NI); a
// k-step of 32 moves the tile's X rows (128 bytes, hi and lo) and W rows (64 bytes) to LDS by DMA,
// NS stages.  A row's 16-byte chunk c is stored at c ^ (row / (256 / row bytes)), so that the 16
// rows a fragment read touches at one chunk fall in distinct banks.  Every W fragment meets two X
// fragments.  A step is two halves over the wave's W fragments, so that reads, DMA and MFMAs
// overlap with one barrier a step and no second set of fragments:
//   half 1: the X fragments against W's first NA, while W's others are read;
//   barrier: every read of the step's stage is done, and the next step's DMA has landed;
//   the DMA of step + NS into the stage just freed;
//   half 2: the X fragments against W's others, while the next step's first NA W fragments and,
//   each once its last MFMA is out, its X fragments are read.
// At 4096 rows QKV (3456 x 1152) takes 59 us (fp32 MFMAs: 295), ffn_up with GELU 78 (390), ffn_down
// 91 (352); at 320 rows QKV 15.
// OUT 0: fp32 + bias (+ R); 1: GELU (ACT 1 tanh, 2 erf), times OSCALE, into split rows of LDY; 2:
// fp32 sums of workgroup z's k-steps (split K) at z M N.
enum { VS_F32 = 0, VS_SPLIT = 1, VS_PART = 2 };
template <int WMW, int WNW, int MI, int NI, int NS, int OUT, int ACT>
__global__ void __launch_bounds__(WMW * WNW * 64)
k_vis_gemm_s(const uint16_t* __restrict__ X, const uint16_t* __restrict__ W, const float* __restrict__ bias,
             const float* R, void* Y, int M, int N, int KP, float descale, float oscale, int ldy) {
  constexpr int NW = WMW * WNW, BM = WMW * MI * 16, BN = WNW * NI * 16, NA = (NI + 1) / 2, NB = NI - NA;
  constexpr int XS = BM * 128, STAGE = XS + BN * 64, XI = XS / 1024, TI = STAGE / 1024;   // DMA instructions a stage
  constexpr int PER = (TI + NW - 1) / NW, REM = TI % NW;   // a wave's: PER, waves REM and up one less (REM > 0)
  static_assert(TI * 1024 == STAGE && NB > 0 && XI % NW == 0, "whole DMA instructions, two halves");
  extern __shared__ __align__(1024) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c16 = lane & 15, g = lane >> 4;
  const int wm = (wave / WNW) * 16 * MI, wn = (wave % WNW) * 16 * NI;
  // tile order: XCD x takes the x-th eighth of an order that walks 4 row tiles at a time, so that
  // the tiles an L2 serves at once share W and X
  int bm = blockIdx.y, bn = blockIdx.x;
  {
    const int gx = gridDim.x, gy = gridDim.y, G = gx * gy, b = blockIdx.y * gx + blockIdx.x;
    const int L = G % 8 == 0 ? (b % 8) * (G / 8) + b / 8 : b;
    constexpr int GM = 4;
    const int grp = L / (GM * gx), first = grp * GM, sz = min(gy - first, GM), in = L % (GM * gx);
    bm = first + in % sz;
    bn = in / sz;
  }
  const int tm = bm * BM, tn = bn * BN;
  const int nk = KP / 32, kt0 = (int)((int64_t)nk * blockIdx.z / gridDim.z),
            kt1 = (int)((int64_t)nk * (blockIdx.z + 1) / gridDim.z);
  const uint16_t* xb = X + (int64_t)tm * 2 * KP;
  const int NP = (N + 63) / 64 * 64;
  const uint16_t* wb = W + (int64_t)tn * 32;
  const uint32_t xext = (uint32_t)((int64_t)min(BM, M - tm) * KP * 4),
                 wext = (uint32_t)(max(0, min(BN, NP - tn)) * 64);
  // DMA: a stage is TI runs of 1 KB, wave w takes runs w, w + NW, ..: the first XI are X's (8 rows
  // each), the others W's (16 rows each)
  uint32_t off[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int p = wave + NW * i;
    const int rx = 8 * p + (lane >> 3), cx = (lane & 7) ^ ((rx >> 1) & 7);
    const int rw = 16 * (p - XI) + (lane >> 2), cw = (lane & 3) ^ ((rw >> 2) & 3);
    off[i] = i < XI / NW ? (uint32_t)(rx * KP * 4 + cx * 16) : (uint32_t)(rw * 64 + cw * 16);
  }
  auto issue1 = [&](int kt, int st, int i) {
    const int p = wave + NW * i;
    uint8_t* dst = smem + st * STAGE + p * 1024;
    if (REM && i == PER - 1 && wave >= REM) return;
    if (i < XI / NW) sdma16(xb, xext, (lds_void*)dst, off[i], kt * 128);
    else sdma16(wb + (int64_t)kt * NP * 32, wext, (lds_void*)dst, off[i], 0);
  };
  // all but the newest KEEP stages' DMA has landed, every LDS read is done, for every wave
  auto landed = [&](auto keep) {
    constexpr int KEEP = decltype(keep)::value;
    if (REM && wave >= REM) wait_dma_barrier<KEEP * (PER - 1)>();
    else wait_dma_barrier<KEEP * PER>();
  };
  const int xs = (c16 >> 1) & 7, ws = (c16 >> 2) & 3;   // a 16-row block's rows: the swizzle is c16's
  const uint8_t* xrd = smem + (wm + c16) * 128;
  const uint8_t* wrd = smem + XS + (wn + c16) * 64 + 16 * (g ^ ws);
  const int xh = 16 * (g ^ xs), xl = 16 * ((4 + g) ^ xs);
  f32x4 acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  f16x8 x[MI][2], a[NA], b[NB];
  // past the end the DMA re-reads the last step, and nothing reads it: every wait counts the same
#pragma unroll
  for (int p = 0; p < NS; ++p)
#pragma unroll
    for (int i = 0; i < PER; ++i) issue1(min(kt0 + p, kt1 - 1), p, i);
  landed(std::integral_constant<int, NS - 1>());
#pragma unroll
  for (int j = 0; j < NA; ++j) a[j] = *(const f16x8*)(wrd + j * 1024);
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    x[i][0] = *(const f16x8*)(xrd + i * 2048 + xh);
    x[i][1] = *(const f16x8*)(xrd + i * 2048 + xl);
  }
  int st = 0;
  for (int kt = kt0; kt < kt1; ++kt) {
    const int nx = st + 1 == NS ? 0 : st + 1, kn = min(kt + NS, kt1 - 1);
#pragma unroll
    for (int j = 0; j < NB; ++j) b[j] = *(const f16x8*)(wrd + st * STAGE + (NA + j) * 1024);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int j = 0; j < NA; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[j], x[i][u], acc[i][j], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    landed(std::integral_constant<int, NS - 2>());
#pragma unroll
    for (int j = 0; j < NA; ++j) a[j] = *(const f16x8*)(wrd + nx * STAGE + j * 1024);
#pragma unroll
    for (int i = 0; i < MI; ++i) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
#pragma unroll
        for (int j = 0; j < NB; ++j)
          acc[i][NA + j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b[j], x[i][u], acc[i][NA + j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int d = 0; d < PER; ++d)
          if (d * 2 * MI / PER == 2 * i + u) issue1(kn, st, d);
        __builtin_amdgcn_sched_barrier(0);
      }
      x[i][0] = *(const f16x8*)(xrd + nx * STAGE + i * 2048 + xh);
      x[i][1] = *(const f16x8*)(xrd + nx * STAGE + i * 2048 + xl);
      __builtin_amdgcn_sched_barrier(0);
    }
    st = nx;
  }
  wait_dma_barrier<0>();   // the last DMA has landed before the workgroup's LDS is another's
  {
#pragma clang fp contract(off)
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const int col = tn + wn + 16 * j + 4 * g;
      if (OUT == VS_SPLIT ? col >= ldy : col >= N) continue;
      f32x4 bj = {0.f, 0.f, 0.f, 0.f};
      if (OUT != VS_PART && col < N) bj = *(const f32x4*)(bias + col);
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        const int row = tm + wm + 16 * i + c16;
        if (row >= M) continue;
        f32x4 v = acc[i][j] * descale;
        if (OUT == VS_PART) {
          *(f32x4*)((float*)Y + ((int64_t)blockIdx.z * M + row) * N + col) = v;
          continue;
        }
        v = v + bj;
        if (OUT == VS_F32) {
          const int64_t o = (int64_t)row * N + col;
          if (R) v = v + *(const f32x4*)(R + o);
          *(f32x4*)((float*)Y + o) = v;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if (ACT == 1) v[e] = gelu_sig(v[e]);
            if (ACT == 2) v[e] = 0.5f * v[e] * (1.f + erff(v[e] * 0.70710678118654752f));
          }
          u32x2 hi, lo;
          split4(v * oscale, hi, lo);
          uint16_t* o = (uint16_t*)Y + (int64_t)row * 2 * ldy + split_at(col);
          *(u32x2*)o = hi;
          *(u32x2*)(o + 32) = lo;
        }
      }
    }
  }
}

template <int WMW, int WNW, int MI, int NI, int NS, int OUT, int ACT>
static hipError_t gemm_s_t(hipStream_t s, const uint16_t* x, const uint16_t* w, const float* bias, const float* r,
                           void* y, int M, int N, int KP, float descale, float oscale, int ldy, int S) {
  constexpr int BM = WMW * MI * 16, BN = WNW * NI * 16, lds = NS * (BM * 128 + BN * 64);
  const void* kern = (const void*)k_vis_gemm_s<WMW, WNW, MI, NI, NS, OUT, ACT>;
  const hipError_t e = ensure_lds(kern, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_vis_gemm_s<WMW, WNW, MI, NI, NS, OUT, ACT>),
                     dim3(sgrid(OUT == VS_SPLIT ? ldy : N, BN), sgrid(M, BM), S), dim3(WMW * WNW * 64), lds, s, x, w, bias,
                     r, y, M, N, KP, descale, oscale, ldy);
  return hipGetLastError();
}

// The tiles, and what a k-step of one costs (us) for a workgroup alone on its CU and for each of
// several that share one: fitted to K 1152 and 4304 at 80 to 4096 rows.  The 8-wave tiles fill a
// CU's LDS and run at 82% of the MFMA rate; the small ones, bound by the CU's LDS DMA (about
// 60 bytes a ns), are for grids that would leave CUs idle.
struct VisTile {
  int bm, bn;
  float alone, shared;
};
static const VisTile kVisTiles[] = {{256, 256, 1.06f, 1.06f}, {256, 288, 1.23f, 1.23f}, {128, 144, 0.56f, 0.56f},
                                    {128, 128, 0.46f, 0.38f}, {64, 128, 0.33f, 0.26f},  {64, 64, 0.20f, 0.18f},
                                    {32, 64, 0.165f, 0.11f}};
constexpr int kVisTileCount = sizeof(kVisTiles) / sizeof(kVisTiles[0]);

// the tile of the least cost for S parts of M x N x KP, and that cost
static int best_tile(int64_t M, int64_t N, int64_t KP, int S, float* cost) {
  int best = 0;
  *cost = 1e30f;
  for (int t = 0; t < kVisTileCount; ++t) {
    const VisTile& v = kVisTiles[t];
    const int64_t per_cu = ((int64_t)sgrid(M, v.bm) * sgrid(N, v.bn) * S + 255) / 256;
    const float c = (float)(KP / 32 / S) * (per_cu == 1 ? v.alone : v.shared * (float)per_cu);
    if (c < *cost) {
      *cost = c;
      best = t;
    }
  }
  return best;
}

template <int OUT, int ACT>
static hipError_t gemm_s_tile(hipStream_t s, const uint16_t* x, const uint16_t* w, const float* bias, const float* r,
                              void* y, int M, int N, int KP, float descale, float oscale, int ldy, int S) {
  float cost;
  switch (best_tile(M, N, KP, S, &cost)) {
    case 0: return gemm_s_t<4, 2, 4, 8, 3, OUT, ACT>(s, x, w, bias, r, y, M, N, KP, descale, oscale, ldy, S);
    case 1: return gemm_s_t<4, 2, 4, 9, 3, OUT, ACT>(s, x, w, bias, r, y, M, N, KP, descale, oscale, ldy, S);
    case 2: return gemm_s_t<4, 1, 2, 9, 5, OUT, ACT>(s, x, w, bias, r, y, M, N, KP, descale, oscale, ldy, S);
    case 3: return gemm_s_t<2, 2, 4, 4, 3, OUT, ACT>(s, x, w, bias, r, y, M, N, KP, descale, oscale, ldy, S);
    case 4: return gemm_s_t<2, 2, 2, 4, 4, OUT, ACT>(s, x, w, bias, r, y, M, N, KP, descale, oscale, ldy, S);
    case 5: return gemm_s_t<2, 2, 2, 2, 4, OUT, ACT>(s, x, w, bias, r, y, M, N, KP, descale, oscale, ldy, S);
  }
  return gemm_s_t<2, 2, 1, 2, 6, OUT, ACT>(s, x, w, bias, r, y, M, N, KP, descale, oscale, ldy, S);
}

static bool gemm_s_ok(const void* x, const void* w, int64_t M, int64_t N, int64_t KP) {
  return KP > 0 && KP % 64 == 0 && N % 4 == 0 && !((uintptr_t)x & 15) && !((uintptr_t)w & 15) &&
         M * KP * 4 < ((int64_t)1 << 31) && N * KP * 2 < ((int64_t)1 << 31);
}

hipError_t vis_gemm_s(hipStream_t s, const uint16_t* x, const uint16_t* w, const float* bias, const float* r, float* y,
                      uint16_t* ys, int64_t M, int64_t N, int64_t KP, float descale, float oscale, int64_t ldy, int act) {
  if (M <= 0 || N <= 0) return hipSuccess;
  if (!gemm_s_ok(x, w, M, N, KP) || !bias || (ys && (ldy < N || ldy % 64 || act < 1 || act > 2)) || (!ys && act))
    return hipErrorInvalidValue;
  if (!ys) return gemm_s_tile<VS_F32, 0>(s, x, w, bias, r, y, (int)M, (int)N, (int)KP, descale, 0.f, 0, 1);
  if (act == 1)
    return gemm_s_tile<VS_SPLIT, 1>(s, x, w, bias, nullptr, ys, (int)M, (int)N, (int)KP, descale, oscale, (int)ldy, 1);
  return gemm_s_tile<VS_SPLIT, 2>(s, x, w, bias, nullptr, ys, (int)M, (int)N, (int)KP, descale, oscale, (int)ldy, 1);
}

int vis_tile(int64_t M, int64_t N, int64_t KP, int S) {
  float cost;
  return best_tile(M, N, KP, S, &cost);
}

// S parts cost a k-step's share each, the parts' store and the LayerNorm's reads (8 bytes a value
// at about 4 TB/s); whole products read and write the residual in the epilogue instead
int vis_split(int64_t M, int64_t N, int64_t KP) {
  int best = 1;
  float least = 1e30f;
  for (int S = 1; S <= 8 && S <= KP / 192; ++S) {
    float c;
    best_tile(M, N, KP, S, &c);
    c += (float)(M * N) * 2e-6f * (float)S;
    if (c < least) {
      least = c;
      best = S;
    }
  }
  return best;
}

hipError_t vis_gemm_part(hipStream_t s, const uint16_t* x, const uint16_t* w, float* part, int64_t M, int64_t N,
                         int64_t KP, float descale, int S) {
  if (M <= 0 || N <= 0) return hipSuccess;
  if (!gemm_s_ok(x, w, M, N, KP) || S < 1 || S > KP / 64) return hipErrorInvalidValue;
  return gemm_s_tile<VS_PART, 0>(s, x, w, nullptr, nullptr, part, (int)M, (int)N, (int)KP, descale, 0.f, 0, S);
}

// --- heads, rotary ---------------------------------------------------------------------------

// A key's (or query's) row: 72 hi halves, 72 lo halves, 8 unused: 304 bytes, 3 banks' worth off a
// power of two, so that 16 rows at one 16-byte chunk lie in 16 distinct places of the 256 bytes
// the LDS serves at once.
#define VS_KR 152

// tokens t0 .. t0 + 63 of head h from the QKV rows, as k_vis_heads, into split q and k rows and
// V^T's two planes [head][72][np] (np: n rounded up to 64, zeros past n).  Within each aligned
// group of 32 keys V^T's column 8 g + j holds key 4 g + j (j < 4) or 16 + 4 g + j - 4: the order
// in which the score blocks leave a lane's 8 probabilities.
__global__ void __launch_bounds__(256)
k_vis_heads_s(int n, int np, int D, const float* __restrict__ qkv, const float* __restrict__ cs, float qs, float ks,
              float vs, uint16_t* __restrict__ q, uint16_t* __restrict__ k, uint16_t* __restrict__ vt, int64_t vplane) {
#pragma clang fp contract(off)
  __shared__ float vl[72][68];
  const int h = blockIdx.y, t0 = blockIdx.x * 64;
  // 18 groups of 4 dims a token
  for (int idx = threadIdx.x; idx < 64 * 18; idx += 256) {
    const int tl = idx / 18, d = 4 * (idx - 18 * tl), t = t0 + tl;
    f32x4 v4 = {0.f, 0.f, 0.f, 0.f};
    if (t < n) {
      const float* row = qkv + (int64_t)t * 3 * D + h * 72;
      const f32x4 c = *(const f32x4*)(cs + (int64_t)t * 144 + d), sn = *(const f32x4*)(cs + (int64_t)t * 144 + 72 + d);
      const int dr = d < 36 ? d + 36 : d - 36;
      const float sg = d < 36 ? -1.f : 1.f;
      const f32x4 rq = *(const f32x4*)(row + dr) * sg, rk = *(const f32x4*)(row + D + dr) * sg;
      const f32x4 qv = *(const f32x4*)(row + d) * c + rq * sn, kv = *(const f32x4*)(row + D + d) * c + rk * sn;
      v4 = *(const f32x4*)(row + 2 * D + d) * vs;
      u32x2 hi, lo;
      uint16_t* o = q + ((int64_t)h * n + t) * VS_KR + d;
      split4(qv * qs, hi, lo);
      *(u32x2*)o = hi;
      *(u32x2*)(o + 72) = lo;
      o = k + ((int64_t)h * n + t) * VS_KR + d;
      split4(kv * ks, hi, lo);
      *(u32x2*)o = hi;
      *(u32x2*)(o + 72) = lo;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) vl[d + e][tl] = v4[e];
  }
  __syncthreads();
  // 4 consecutive columns of V^T are 4 consecutive keys
  for (int idx = threadIdx.x; idx < 72 * 16; idx += 256) {
    const int d = idx >> 4, c4 = (idx & 15) * 4;
    const int key = (c4 & 32) + ((c4 & 4) << 2) + ((c4 & 24) >> 1);
    u32x2 hi, lo;
    split4(*(const f32x4*)&vl[d][key], hi, lo);
    uint16_t* o = vt + ((int64_t)h * 72 + d) * np + t0 + c4;
    *(u32x2*)o = hi;
    *(u32x2*)(o + vplane) = lo;
  }
}

hipError_t vis_heads_s(hipStream_t s, int n, int np, int heads, const float* qkv, const float* cs, float qs, float ks,
                       float vs, uint16_t* q, uint16_t* k, uint16_t* vt) {
  if (n <= 0) return hipSuccess;
  if (np % 64 || np < n || np >= n + 64) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_vis_heads_s, dim3(np / 64, heads), dim3(256), 0, s, n, np, heads * 72, qkv, cs, qs, ks, vs, q, k, vt,
                     (int64_t)heads * 72 * np);
  return hipGetLastError();
}

// --- attention -------------------------------------------------------------------------------

// Softmax attention of every patch over every patch: grid (ceil(n / (64 QB)), heads), four waves
// of QB blocks of 16 queries, taken transposed as k_vis_attend: S^T = K Q^T, O^T += V^T P^T on
// v_mfma_f32_16x16x32_f16, each product as hi hi + hi lo + lo hi (the lo lo term is at most 2^-24
// of |q||k| and 2^-24 of p|v|, below the sums' own rounding).  A head's 72 dims are 9 chunks of
// 8: 27 chunk pairs in 7 MFMAs of 4 chunks,
//   kh0-3 qh0-3, kh4-7 qh4-7, kh0-3 ql0-3, kh4-7 ql4-7, kl0-3 qh0-3, kl4-7 qh4-7,
//   (kh8 qh8, kh8 ql8, kl8 qh8, kl8 0),
// so that a K tile's rows are read as 5 fragments.  SC takes the scores' scale off (a power of
// two; q also carries log2(e)/sqrt(72), so they come in log2 units); the probabilities are
// exp2(s - max + 15), whose hi and lo parts keep 2^-40 of the largest.  64-key tiles of K (19 KB)
// and V^T's planes (9 KB each; row d's chunk c at c ^ (d / 2 % 8)) move to LDS by DMA, two stages.
// Keys past n score -inf; every tile holds a key below n, so the running max is finite.  The
// output is in v's scale: split rows of KP for attn_out, or (YF) times VDE as fp32 rows.  Bound by
// the MFMAs under the chip's power limit: 4096 patches 228 us (fp32 MFMAs 642), 1.09 PFLOP/s
// executed at 1.8 GHz; 320 patches 10 us.
#define VS_KT 19456
#define VS_VT 20480   // V^T's hi plane (72 rows of 128 bytes), 1 KB that starts with ones, the lo plane, 1 KB of zeros
#define VS_LDS (2 * VS_KT + 2 * VS_VT)
template <int QB>
__global__ void __launch_bounds__(256, 2)
k_vis_attend_s(int n, int np, int D, const uint16_t* __restrict__ q, const uint16_t* __restrict__ k,
               const uint16_t* __restrict__ vt, int64_t vplane, float sc, float vde, int kp, uint16_t* __restrict__ ys,
               float* __restrict__ yf) {
  extern __shared__ __align__(1024) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c16 = lane & 15, g = lane >> 4, h = blockIdx.y;
  const int q0 = blockIdx.x * 64 * QB + wave * 16 * QB;
  const uint16_t* kh = k + (int64_t)h * n * VS_KR;
  const uint16_t* vh = vt + (int64_t)h * 72 * np;
  f16x8 qf[QB][5];   // qh0-3, qh4-7, ql0-3, ql4-7, the mixed one
#pragma unroll
  for (int b = 0; b < QB; ++b) {
    const uint16_t* qr = q + ((int64_t)h * n + min(q0 + 16 * b + c16, n - 1)) * VS_KR;
#pragma unroll
    for (int c = 0; c < 4; ++c) qf[b][c] = *(const f16x8*)(qr + (c >> 1) * 72 + (c & 1) * 32 + 8 * g);
    qf[b][4] = *(const f16x8*)(qr + (g == 1 ? 136 : 64));
    if (g == 3) qf[b][4] = f16x8{0, 0, 0, 0, 0, 0, 0, 0};
  }
  // the rows of ones and zeros behind each plane (72 .. 79 of the fifth block: their sums are the
  // probabilities' own)
  if (tid < 128) {
    const int st = tid >> 6, i = tid & 63;
    *(uint32_t*)(smem + 2 * VS_KT + st * VS_VT + 9216 + 4 * i) = 0x3C003C00u;
    *(uint32_t*)(smem + 2 * VS_KT + st * VS_VT + 10240 + 9216 + 4 * i) = 0u;
  }
  const int nt = (n + 63) / 64;
  auto issue_k = [&](int t) {
    const int key0 = t * 64;
    uint8_t* base = smem + (t & 1) * VS_KT;
    const uint32_t kext = (uint32_t)(min(64, n - key0) * (VS_KR * 2));
#pragma unroll
    for (int i = 0; i < 5; ++i)
      if (wave + 4 * i < 19)
        sdma16(kh + (int64_t)key0 * VS_KR, kext, (lds_void*)(base + (wave + 4 * i) * 1024),
               (uint32_t)(1024 * (wave + 4 * i) + 16 * lane), 0);
  };
  auto issue_v = [&](int t) {
    const int key0 = t * 64;
    uint8_t* base = smem + 2 * VS_KT + (t & 1) * VS_VT;
    const uint32_t vext = (uint32_t)((72 * np - key0) * 2);
#pragma unroll
    for (int i = 0; i < 3; ++i)
      if (wave + 4 * i < 9) {
        const int P = 64 * (wave + 4 * i) + lane, d = P >> 3, c = (P & 7) ^ ((d >> 1) & 7);
        const uint32_t off = (uint32_t)(d * np * 2 + c * 16);
        sdma16(vh + key0, vext, (lds_void*)(base + (wave + 4 * i) * 1024), off, 0);
        sdma16(vh + vplane + key0, vext, (lds_void*)(base + 10240 + (wave + 4 * i) * 1024), off, 0);
      }
  };
  float m[QB];
  f32x4 o[5][QB], s[4][QB];
#pragma unroll
  for (int b = 0; b < QB; ++b) {
    m[b] = -INFINITY;
#pragma unroll
    for (int db = 0; db < 5; ++db) o[db][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const int e0 = 16 * (g ^ ((c16 >> 1) & 7)), e1 = 16 * ((4 + g) ^ ((c16 >> 1) & 7));
  const int vr0 = c16 * 128 + e0, vr1 = c16 * 128 + e1;
  const int vt0 = c16 < 8 ? 8192 + vr0 : 9216, vt1 = c16 < 8 ? 8192 + vr1 : 9216;
  const int krow = c16 * (VS_KR * 2), km = g < 2 ? 128 : 272;
  auto read_k = [&](f16x8 (&kf)[5], const uint8_t* kb_, int kb) {
    const uint8_t* kr = kb_ + krow + kb * (16 * VS_KR * 2);
#pragma unroll
    for (int c = 0; c < 4; ++c) kf[c] = *(const f16x8*)(kr + (c >> 1) * 144 + (c & 1) * 64 + 16 * g);
    kf[4] = *(const f16x8*)(kr + km);
  };
  auto scores = [&](const f16x8 (&kf)[5], int b) {
    f32x4 a = {0.f, 0.f, 0.f, 0.f};
    a = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[2], qf[b][0], a, 0, 0, 0);
    a = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[3], qf[b][1], a, 0, 0, 0);
    a = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[0], qf[b][2], a, 0, 0, 0);
    a = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[1], qf[b][3], a, 0, 0, 0);
    a = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[4], qf[b][4], a, 0, 0, 0);
    a = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[0], qf[b][0], a, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[1], qf[b][1], a, 0, 0, 0);
  };
  issue_k(0);
  issue_v(0);
  if (nt > 1) issue_k(1);
  wait_dma_barrier<0>();
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    f16x8 kf[5];
    read_k(kf, smem, kb);
#pragma unroll
    for (int b = 0; b < QB; ++b) s[kb][b] = scores(kf, b);
  }
  for (int t = 0; t < nt; ++t) {
    // tile t + 1's K and tile t's V are in; every wave is done with tile t's K and tile t - 1's V
    if (t > 0) wait_dma_barrier<0>();
    else __syncthreads();
    if (t + 2 < nt) issue_k(t + 2);
    if (t + 1 < nt) issue_v(t + 1);
    if (t * 64 + 64 > n) {
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (t * 64 + 16 * kb + 4 * g + e >= n)
#pragma unroll
            for (int b = 0; b < QB; ++b) s[kb][b][e] = -INFINITY;
    }
    const uint8_t* kn = smem + ((t + 1) & 1) * VS_KT;
    f16x8 ph[2][QB], pl[2][QB], kf[2][5];
    float alpha[QB], off[QB];
    f32x4 sn[4][QB];
    read_k(kf[0], kn, 0);
    bool moved = false;
#pragma unroll
    for (int b = 0; b < QB; ++b) {
      float mx = -INFINITY;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int e = 0; e < 4; ++e) mx = fmaxf(mx, s[kb][b][e]);
      float ma = mx, mb = mx;
      xswap16(ma, mb);
      mx = fmaxf(ma, mb);
      ma = mx;
      mb = mx;
      xswap32(ma, mb);
      // the running max rounded up to a whole number: the exponents' offset and the rescale are
      // then exact, whatever tile a key is in
      const float mn = fmaxf(m[b], ceilf(fmaxf(ma, mb) * sc));
      alpha[b] = __builtin_amdgcn_exp2f(m[b] - mn);
      moved |= mn != m[b];
      m[b] = mn;
      off[b] = 15.f - mn;
    }
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      if (kb < 3) read_k(kf[(kb + 1) & 1], kn, kb + 1);
#pragma unroll
      for (int b = 0; b < QB; ++b) {
        sn[kb][b] = scores(kf[kb & 1], b);
        f32x4 p;
#pragma unroll
        for (int e = 0; e < 4; ++e) p[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kb][b][e], sc, off[b]));
        u32x2 hi, lo;
        split4(p, hi, lo);
        ((u32x2*)&ph[kb >> 1][b])[kb & 1] = hi;
        ((u32x2*)&pl[kb >> 1][b])[kb & 1] = lo;
      }
    }
    // where no query's max moved (most tiles after the first few) there is nothing to rescale
    if (__any(moved)) {
#pragma unroll
      for (int b = 0; b < QB; ++b)
#pragma unroll
        for (int db = 0; db < 5; ++db) o[db][b] = o[db][b] * alpha[b];
    }
    const uint8_t* vb_ = smem + 2 * VS_KT + (t & 1) * VS_VT;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int db = 0; db < 5; ++db) {
        const uint8_t* vr = vb_ + (db < 4 ? db * 2048 + (u ? vr1 : vr0) : (u ? vt1 : vt0));
        const f16x8 va = *(const f16x8*)vr, vb = *(const f16x8*)(vr + 10240);
#pragma unroll
        for (int b = 0; b < QB; ++b) o[db][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vb, ph[u][b], o[db][b], 0, 0, 0);
#pragma unroll
        for (int b = 0; b < QB; ++b) o[db][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va, pl[u][b], o[db][b], 0, 0, 0);
#pragma unroll
        for (int b = 0; b < QB; ++b) o[db][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va, ph[u][b], o[db][b], 0, 0, 0);
      }
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int b = 0; b < QB; ++b) s[kb][b] = sn[kb][b];
  }
#pragma unroll
  for (int b = 0; b < QB; ++b) {
    const float lt = __shfl(o[4][b][0], 32 + c16, 64);   // row 72
    const int qi = q0 + 16 * b + c16;
    if (qi >= n) continue;
#pragma unroll
    for (int db = 0; db < 5; ++db) {
      const int d0 = 16 * db + 4 * g;
      if (d0 >= 72) continue;
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = __fdiv_rn(o[db][b][e], lt);
      if (yf) {
        *(f32x4*)(yf + (int64_t)qi * D + h * 72 + d0) = v * vde;
      } else {
        u32x2 hi, lo;
        split4(v, hi, lo);
        uint16_t* y = ys + (int64_t)qi * 2 * kp + split_at(h * 72 + d0);
        *(u32x2*)y = hi;
        *(u32x2*)(y + 32) = lo;
      }
    }
  }
}

hipError_t vis_attend_s(hipStream_t s, int n, int np, int heads, const uint16_t* q, const uint16_t* k, const uint16_t* vt,
                        float sc, float vde, int kp, uint16_t* ys, float* yf) {
  if (n <= 0) return hipSuccess;
  if (np % 64 || np < n || np >= n + 64 || (int64_t)np * 144 >= ((int64_t)1 << 31) || (ys && kp != heads * 72))
    return hipErrorInvalidValue;
  const int64_t vplane = (int64_t)heads * 72 * np;
  // 128 queries a workgroup (half the reads of K and V) once the CUs hold more than two of 64 each:
  // 4096 patches 228 against 269 us, 3072 the same, 2048 70 against 64, 1024 33 against 24
  const bool two = (int64_t)sgrid(n, 128) * heads > 384;
  const void* kern = two ? (const void*)k_vis_attend_s<2> : (const void*)k_vis_attend_s<1>;
  const hipError_t e = ensure_lds(kern, VS_LDS);
  if (e != hipSuccess) return e;
  if (two)
    hipLaunchKernelGGL(k_vis_attend_s<2>, dim3(sgrid(n, 128), heads), dim3(256), VS_LDS, s, n, np, heads * 72, q, k,
                       vt, vplane, sc, vde, kp, ys, yf);
  else
    hipLaunchKernelGGL(k_vis_attend_s<1>, dim3(sgrid(n, 64), heads), dim3(256), VS_LDS, s, n, np, heads * 72, q, k,
                       vt, vplane, sc, vde, kp, ys, yf);
  return hipGetLastError();
}

}  // namespace exn
