// vision_split.hip -- the vision tower's products and attention on the fp16 matrix units without
// giving up fp32: an fp32 operand X is held as two fp16 parts, hi = fp16(s X) and
// lo = fp16(s X - hi), with s a power of two that keeps |s X| at or below 2^15.  hi + lo carries
// 23 to 24 significant bits of every value down to 2^-16 of the bound s was made for, and an
// absolute error of 2^-40 of the bound below that, so a product over the two parts rounds like
// the fp32 one (the sums stay in fp32 inside the MFMA).  The weights of an mmproj-f16 file are
// fp16 values, and bf16 ones become fp16 values times a power of two: exact in one part, so
// Y = X W^T takes two fp16 MFMAs (hi, lo) where v_mfma_f32_16x16x4_f32 needed eight of twice the
// length: 16 times the rate over 2.  The bounds come from the weights alone (api_vision.hip):
// LayerNorm's output is at most sqrt(D) max|g| + max|b| whatever its input.
//
//   k_vis_stats   max |x| and the largest row norm of a tensor, for the bounds;
//   k_vis_pack    a matrix as fp16 rows, a flag when a value is not exact;
//   k_vis_gemm_s  Y = X W^T + b (+ R) (then GELU), X split, W fp16;
//   k_vis_ln_s    LayerNorm into split rows, over the sum of a split product's parts;
//   k_vis_heads_s QKV rows into split heads, the rotary applied;
//   k_vis_attend_s softmax attention over split q, k, v and probabilities.
//
// Split rows: a row of K values is Kp/32 blocks of 128 bytes (Kp = K rounded up to 64, zeros past
// K), each 32 hi halves then their 32 lo halves: 4 bytes a value, as fp32.
#include "exn_common.h"

#include <algorithm>

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

// four values, already scaled, into their hi and lo halves.  The values pass through an empty asm:
// where V is a product, the compiler would otherwise round it to fp16 in one step for the stored
// hi (v_fma_mixlo_f16) and in two for the one that lo is taken from, and on a tie they differ.
__device__ __forceinline__ void split4(const f32x4 x, u32x2& hi, u32x2& lo) {
  float v[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    v[e] = x[e];
    asm("" : "+v"(v[e]));
  }
  hi = u32x2{pack_f16x2(v[0], v[1]), pack_f16x2(v[2], v[3])};
  lo = u32x2{pack_f16x2(v[0] - f16_lo(hi[0]), v[1] - f16_hi(hi[0])), pack_f16x2(v[2] - f16_lo(hi[1]), v[3] - f16_hi(hi[1]))};
}

// where column K (a multiple of 4) of a split row lies, in halves; its lo part is 32 further
__device__ __forceinline__ int split_at(int k) { return (k >> 5) * 64 + (k & 31); }

// --- the weights -----------------------------------------------------------------------------

// rec[0] = the bits of the largest |x|, rec[1] those of the largest row's sum of squares (NaNs
// compare above every number, so a bound made from a tensor that holds one is not finite)
__global__ void __launch_bounds__(256)
k_vis_stats(int64_t cols, const float* __restrict__ x, uint32_t* __restrict__ rec) {
  __shared__ float rm[4], rs[4];
  const float* r = x + (int64_t)blockIdx.x * cols;
  uint32_t mb = 0u;
  float s = 0.f;
  for (int64_t i = threadIdx.x; i < cols; i += 256) {
    const float v = r[i];
    mb = max(mb, __float_as_uint(fabsf(v)));
    s += v * v;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mb = max(mb, (uint32_t)__shfl_xor((int)mb, o, 64));
  s = wave_sum(s);
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    rm[wave] = __uint_as_float(mb);
    rs[wave] = s;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < 4; ++w) {
      mb = max(mb, __float_as_uint(rm[w]));
      s += rs[w];
    }
    atomicMax(rec, mb);
    atomicMax(rec + 1, __float_as_uint(fabsf(s)));
  }
}

hipError_t vis_stats(hipStream_t s, int64_t rows, int64_t cols, const float* x, uint32_t* rec) {
  if (rows <= 0 || cols <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_vis_stats, dim3((unsigned)rows), dim3(256), 0, s, cols, x, rec);
  return hipGetLastError();
}

// rows of K floats, times SCALE, as fp16 rows of KP (zeros past K); *INEXACT set when one changes
__global__ void __launch_bounds__(256)
k_vis_pack(int K, int KP, float scale, const float* __restrict__ x, uint16_t* __restrict__ y, uint32_t* inexact) {
  const float* r = x + (int64_t)blockIdx.x * K;
  bool bad = false;
  for (int i = threadIdx.x; i < KP; i += 256) {
    const float v = i < K ? r[i] * scale : 0.f;
    const _Float16 h = (_Float16)v;
    bad |= (float)h != v;
    y[(int64_t)blockIdx.x * KP + i] = __builtin_bit_cast(uint16_t, h);
  }
  if (bad) atomicOr(inexact, 1u);
}

hipError_t vis_pack(hipStream_t s, int64_t rows, int K, int KP, float scale, const float* x, uint16_t* y,
                    uint32_t* inexact) {
  if (rows <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_vis_pack, dim3((unsigned)rows), dim3(256), 0, s, K, KP, scale, x, y, inexact);
  return hipGetLastError();
}

// --- LayerNorm -------------------------------------------------------------------------------

// One workgroup a row of WIDTH (a multiple of 4, at most 5120) of X, or, when S > 0, of
// bias + R + the S parts of a split product (each MN floats after the last, summed in order),
// written back to X; then k_vis_ln's LayerNorm, times SCALE, into split rows of KP, or, when YF
// is given, as fp32 rows.
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
  if (width % 64 || width > 5120 || kp != width) return hipErrorInvalidValue;   // no columns past the width to clear
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
// k-step of BK moves the tile's X rows (4 BK bytes, hi and lo) and W rows (2 BK bytes) to LDS by
// DMA, NS stages, the step's DMA going out NS - 1 steps ahead.  A row's 16-byte chunk c is stored
// at c ^ (row / (256 / row bytes)), so that the 16 rows a fragment read touches at one chunk fall
// in distinct banks.  Every W fragment meets two X fragments.  OUT 0: fp32 + bias (+ R); 1: GELU
// (ACT 1 tanh, 2 erf), times OSCALE, into split rows of LDY; 2: fp32 sums of workgroup z's k-steps
// (split K) at z M N.
enum { VS_F32 = 0, VS_SPLIT = 1, VS_PART = 2 };
template <int WMW, int WNW, int MI, int NI, int BK, int NS, int OUT, int ACT>
__global__ void __launch_bounds__(WMW * WNW * 64)
k_vis_gemm_s(const uint16_t* __restrict__ X, const uint16_t* __restrict__ W, const float* __restrict__ bias,
             const float* R, void* Y, int M, int N, int KP, float descale, float oscale, int ldy) {
  constexpr int NW = WMW * WNW, BM = WMW * MI * 16, BN = WNW * NI * 16;
  constexpr int XR = 4 * BK, WR = 2 * BK, XC = XR / 16, WC = WR / 16;   // row bytes, chunks a row
  constexpr int XS = BM * XR, STAGE = XS + BN * WR, XI = XS / 1024 / NW, WI = BN * WR / 1024 / NW;
  static_assert(XI * 1024 * NW == XS && WI * 1024 * NW == BN * WR, "whole DMA instructions a wave");
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
  const int nk = KP / BK, kt0 = (int)((int64_t)nk * blockIdx.z / gridDim.z),
            kt1 = (int)((int64_t)nk * (blockIdx.z + 1) / gridDim.z);
  const uint16_t* xb = X + (int64_t)tm * 2 * KP;
  const uint16_t* wb = W + (int64_t)tn * KP;
  const uint32_t xext = (uint32_t)((int64_t)min(BM, M - tm) * KP * 4), 
                 wext = (uint32_t)((int64_t)max(0, min(BN, N - tn)) * KP * 2);
  auto xswz = [](int r) { return (r / (256 / XR)) % XC; };
  auto wswz = [](int r) { return (r / (256 / WR)) % WC; };
  uint32_t xoff[XI], woff[WI];
#pragma unroll
  for (int i = 0; i < XI; ++i) {
    const int P = 64 * (wave * XI + i) + lane, r = P / XC, c = (P % XC) ^ xswz(r);
    xoff[i] = (uint32_t)(r * KP * 4 + c * 16);
  }
#pragma unroll
  for (int i = 0; i < WI; ++i) {
    const int P = 64 * (wave * WI + i) + lane, r = P / WC, c = (P % WC) ^ wswz(r);
    woff[i] = (uint32_t)(r * KP * 2 + c * 16);
  }
  auto issue = [&](int kt, int st) {
    uint8_t* base = smem + st * STAGE;
#pragma unroll
    for (int i = 0; i < XI; ++i) sdma16(xb, xext, (lds_void*)(base + (wave * XI + i) * 1024), xoff[i], kt * XR);
#pragma unroll
    for (int i = 0; i < WI; ++i) sdma16(wb, wext, (lds_void*)(base + XS + (wave * WI + i) * 1024), woff[i], kt * WR);
  };
  // a fragment's row c16 of a 16-row block: its chunk c is at 16 (c ^ swz); the swizzle of row
  // 16 i + c16 is c16's, since 16 rows are whole periods of it
  const int xs = xswz(c16), ws = wswz(c16);
  const uint8_t* xrd = smem + (wm + c16) * XR;
  const uint8_t* wrd = smem + XS + (wn + c16) * WR;
  f32x4 acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int p = 0; p < NS - 1; ++p)
    if (kt0 + p < kt1) issue(kt0 + p, p);
  int st = 0;
  for (int kt = kt0; kt < kt1; ++kt) {
    // step kt's rows are in for every wave, and every wave is done with step kt - 1's stage
    if (kt + NS - 2 < kt1) wait_dma_barrier<(NS - 2) * (XI + WI)>();
    else wait_dma_barrier<0>();
    if (kt + NS - 1 < kt1) issue(kt + NS - 1, st == 0 ? NS - 1 : st - 1);
    const uint8_t* xr = xrd + st * STAGE;
    const uint8_t* wr = wrd + st * STAGE;
    st = st + 1 == NS ? 0 : st + 1;
#pragma unroll
    for (int h = 0; h < BK / 32; ++h) {
      f16x8 a[NI];
#pragma unroll
      for (int j = 0; j < NI; ++j) a[j] = *(const f16x8*)(wr + j * 16 * WR + 16 * ((4 * h + g) ^ ws));
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        const f16x8 xh = *(const f16x8*)(xr + i * 16 * XR + 16 * ((8 * h + g) ^ xs));
        const f16x8 xl = *(const f16x8*)(xr + i * 16 * XR + 16 * ((8 * h + 4 + g) ^ xs));
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[j], xh, acc[i][j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[j], xl, acc[i][j], 0, 0, 0);
      }
    }
  }
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

template <int WMW, int WNW, int MI, int NI, int BK, int NS, int OUT, int ACT>
static hipError_t gemm_s_t(hipStream_t s, const uint16_t* x, const uint16_t* w, const float* bias, const float* r,
                           void* y, int M, int N, int KP, float descale, float oscale, int ldy, int S) {
  constexpr int BM = WMW * MI * 16, BN = WNW * NI * 16, lds = NS * (BM * 4 + BN * 2) * BK;
  const void* kern = (const void*)k_vis_gemm_s<WMW, WNW, MI, NI, BK, NS, OUT, ACT>;
  const hipError_t e = ensure_lds(kern, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_vis_gemm_s<WMW, WNW, MI, NI, BK, NS, OUT, ACT>),
                     dim3(sgrid(OUT == VS_SPLIT ? ldy : N, BN), sgrid(M, BM), S), dim3(WMW * WNW * 64), lds, s, x, w, bias,
                     r, y, M, N, KP, descale, oscale, ldy);
  return hipGetLastError();
}

template <int OUT, int ACT>
static hipError_t gemm_s_tile(hipStream_t s, const uint16_t* x, const uint16_t* w, const float* bias, const float* r,
                              void* y, int M, int N, int KP, float descale, float oscale, int ldy, int S) {
  if ((int64_t)sgrid(M, 128) * sgrid(N, 128) >= 192)
    return gemm_s_t<2, 2, 4, 4, 32, 3, OUT, ACT>(s, x, w, bias, r, y, M, N, KP, descale, oscale, ldy, S);
  return gemm_s_t<2, 2, 2, 2, 64, 3, OUT, ACT>(s, x, w, bias, r, y, M, N, KP, descale, oscale, ldy, S);
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

int vis_split(int64_t M, int64_t N, int64_t KP) {
  // 64 x 64 tiles and about 256 workgroups, a part of at least 6 k-steps of 64
  const int64_t tiles = (int64_t)sgrid(M, 64) * sgrid(N, 64);
  const int64_t S = std::min<int64_t>(std::min<int64_t>(256 / tiles, KP / 384), 8);
  return S < 2 ? 1 : (int)S;
}

hipError_t vis_gemm_part(hipStream_t s, const uint16_t* x, const uint16_t* w, float* part, int64_t M, int64_t N,
                         int64_t KP, float descale, int S) {
  if (M <= 0 || N <= 0) return hipSuccess;
  if (!gemm_s_ok(x, w, M, N, KP) || S < 1 || S > KP / 64) return hipErrorInvalidValue;
  return gemm_s_t<2, 2, 2, 2, 64, 3, VS_PART, 0>(s, x, w, nullptr, nullptr, part, (int)M, (int)N, (int)KP, descale, 0.f, 0,
                                                S);
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
// output is in v's scale: split rows of KP for attn_out, or (YF) times VDE as fp32 rows.
#define VS_KT 19456
#define VS_STAGE (VS_KT + 2 * 9216)
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
  auto issue = [&](int t, int st) {
    const int key0 = t * 64;
    uint8_t* base = smem + st * VS_STAGE;
    const uint32_t kext = (uint32_t)(min(64, n - key0) * (VS_KR * 2)), vext = (uint32_t)((72 * np - key0) * 2);
    for (int i = wave; i < 37; i += 4) {
      if (i < 19) {
        sdma16(kh + (int64_t)key0 * VS_KR, kext, (lds_void*)(base + i * 1024), (uint32_t)(1024 * i + 16 * lane), 0);
      } else {
        const int P = 64 * ((i - 19) % 9) + lane, d = P >> 3, c = (P & 7) ^ ((d >> 1) & 7);
        sdma16(vh + (i < 28 ? 0 : vplane) + key0, vext, (lds_void*)(base + i * 1024), (uint32_t)(d * np * 2 + c * 16), 0);
      }
    }
  };
  float m[QB], l[QB];
  f32x4 o[5][QB];
#pragma unroll
  for (int b = 0; b < QB; ++b) {
    m[b] = -INFINITY;
    l[b] = 0.f;
#pragma unroll
    for (int db = 0; db < 5; ++db) o[db][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // V^T rows 72 .. 79 of the fifth block repeat row 71: their sums are not stored
  int voff[5];
#pragma unroll
  for (int db = 0; db < 5; ++db) voff[db] = min(16 * db + c16, 71);
  const int nt = (n + 63) / 64;
  issue(0, 0);
  for (int t = 0; t < nt; ++t) {
    wait_dma_barrier<0>();
    if (t + 1 < nt) issue(t + 1, (t + 1) & 1);
    const uint8_t* kb_ = smem + (t & 1) * VS_STAGE;
    const uint8_t* vb_ = kb_ + VS_KT;
    f32x4 s[4][QB];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      const uint8_t* kr = kb_ + (16 * kb + c16) * (VS_KR * 2);
      f16x8 kf[5];
#pragma unroll
      for (int c = 0; c < 4; ++c) kf[c] = *(const f16x8*)(kr + (c >> 1) * 144 + (c & 1) * 64 + 16 * g);
      kf[4] = *(const f16x8*)(kr + (g < 2 ? 128 : 272));
#pragma unroll
      for (int b = 0; b < QB; ++b) {
        f32x4 a = {0.f, 0.f, 0.f, 0.f};
        a = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[2], qf[b][0], a, 0, 0, 0);
        a = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[3], qf[b][1], a, 0, 0, 0);
        a = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[0], qf[b][2], a, 0, 0, 0);
        a = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[1], qf[b][3], a, 0, 0, 0);
        a = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[4], qf[b][4], a, 0, 0, 0);
        a = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[0], qf[b][0], a, 0, 0, 0);
        s[kb][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[1], qf[b][1], a, 0, 0, 0);
      }
    }
    if (t * 64 + 64 > n) {
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (t * 64 + 16 * kb + 4 * g + e >= n)
#pragma unroll
            for (int b = 0; b < QB; ++b) s[kb][b][e] = -INFINITY;
    }
    f16x8 ph[2][QB], pl[2][QB];
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
      // where no query's max moved (most tiles after the first few) there is nothing to rescale
      if (__any(mn != m[b])) {
        const float alpha = __builtin_amdgcn_exp2f(m[b] - mn);
        l[b] *= alpha;
#pragma unroll
        for (int db = 0; db < 5; ++db) o[db][b] = o[db][b] * alpha;
        m[b] = mn;
      }
      const float off = 15.f - mn;
      float ls = 0.f;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        f32x4 p;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          p[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kb][b][e], sc, off));
          ls += p[e];
        }
        u32x2 hi, lo;
        split4(p, hi, lo);
        ((u32x2*)&ph[kb >> 1][b])[kb & 1] = hi;
        ((u32x2*)&pl[kb >> 1][b])[kb & 1] = lo;
      }
      l[b] += ls;
    }
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int db = 0; db < 5; ++db) {
        const uint8_t* vr = vb_ + voff[db] * 128 + 16 * ((4 * u + g) ^ ((voff[db] >> 1) & 7));
        const f16x8 va = *(const f16x8*)vr, vb = *(const f16x8*)(vr + 9216);
#pragma unroll
        for (int b = 0; b < QB; ++b) {
          o[db][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vb, ph[u][b], o[db][b], 0, 0, 0);
          o[db][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va, pl[u][b], o[db][b], 0, 0, 0);
          o[db][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va, ph[u][b], o[db][b], 0, 0, 0);
        }
      }
  }
#pragma unroll
  for (int b = 0; b < QB; ++b) {
    float lt = l[b];
    lt += __shfl_xor(lt, 16, 64);
    lt += __shfl_xor(lt, 32, 64);
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
  // 128 queries a workgroup where that still gives every CU one, else 64
  const bool two = (int64_t)sgrid(n, 128) * heads >= 256;
  const void* kern = two ? (const void*)k_vis_attend_s<2> : (const void*)k_vis_attend_s<1>;
  const hipError_t e = ensure_lds(kern, 2 * VS_STAGE);
  if (e != hipSuccess) return e;
  if (two)
    hipLaunchKernelGGL(k_vis_attend_s<2>, dim3(sgrid(n, 128), heads), dim3(256), 2 * VS_STAGE, s, n, np, heads * 72, q, k,
                       vt, vplane, sc, vde, kp, ys, yf);
  else
    hipLaunchKernelGGL(k_vis_attend_s<1>, dim3(sgrid(n, 64), heads), dim3(256), 2 * VS_STAGE, s, n, np, heads * 72, q, k,
                       vt, vplane, sc, vde, kp, ys, yf);
  return hipGetLastError();
}

}  // namespace exn
