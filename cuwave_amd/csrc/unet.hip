// The U-Net preconditioner's training and inference kernels for gfx950:
// 3x3 convolutions (stride 1, zero padding 1) as implicit GEMMs on the
// bfloat16 matrix cores with float32 accumulation, and the AdamW step. No
// reference counterpart: the reference has no learned preconditioner.
//
// Activations are NHWC bfloat16 (channels innermost, so the reduction axis
// of a GEMM tile is contiguous); a convolution's weights are (cout, 9 cin),
// row k = tap cin + ci with tap = 3 (dh + 1) + (dw + 1), in float32 for the
// optimiser and in bfloat16 for the kernels.
//
// - forward: y[p][co] = act(bias[co] + sum_{tap, ci} x[p + off(tap)][ci] w[co][tap][ci]),
//   a GEMM of M = pixels, N = cout, K = 9 cin; the x tile is gathered per
//   tap (zero off the image) and staged in LDS with the weight tile.
// - backward data: the same kernel on dy with the weights flipped in space
//   and transposed in channels (wd[ci][tap][co] = w[co][8 - tap][ci]).
// - backward weight: dw[co][tap][ci] = sum_p dy[p][co] x[p + off(tap)][ci],
//   a GEMM of M = 9 cin, N = cout reduced over the pixels: each block sums a
//   contiguous run of pixels into a float32 partial, and a second kernel
//   adds the partials in a fixed order (deterministic, no atomics).
//
// MFMA v_mfma_f32_32x32x16_bf16: lane l holds A[l % 32][8 (l / 32) + i] and
// B[8 (l / 32) + i][l % 32], i = 0 .. 7, and D[8 (r / 4) + 4 (l / 32) + r % 4][l % 32]
// in accumulator register r.
#include <hip/hip_runtime.h>

#include <stdint.h>

#include <string>

#include "../../include/cuwave_amd.h"
#include "common.hpp"

namespace cwh {
int fail(const std::string &what);
} // namespace cwh

namespace {

using cwh::fail;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kThreads = 256;

__device__ __forceinline__ uint16_t to_bf16(float v) {
  const uint32_t bits = __float_as_uint(v);
  if ((bits & 0x7f800000u) == 0x7f800000u) // inf and nan keep their class
    return (uint16_t)((bits >> 16) | ((bits & 0xffffu) ? 0x40u : 0u));
  return (uint16_t)((bits + 0x7fffu + ((bits >> 16) & 1u)) >> 16);
}

__device__ __forceinline__ float from_bf16(uint16_t b) {
  return __uint_as_float((uint32_t)b << 16);
}

struct Image {
  int n, h, w; // batch, height, width
  int64_t pixels;
};

// the pixel p + off(tap) of pixel p, -1 off the image
__device__ __forceinline__ int64_t shifted(const Image &im, int64_t p, int tap) {
  const int64_t hw = (int64_t)im.h * im.w;
  const int b = (int)(p / hw);
  const int rest = (int)(p - (int64_t)b * hw);
  const int y = rest / im.w + tap / 3 - 1;
  const int x = rest % im.w + tap % 3 - 1;
  if (y < 0 || y >= im.h || x < 0 || x >= im.w)
    return -1;
  return (int64_t)b * hw + (int64_t)y * im.w + x;
}

// ------------------------------------------------------------ forward
// One block: a tile of kTH x kTW pixels of one image and every output channel
// (BN = cout, 32 / 64 / 128). What bounds it is the LDS, then HBM: a 32 -> 32
// layer has 36 flops a byte of activations, so the input has to reach the
// block once. The tile's input with its one-pixel halo is staged KC channels
// at a time and read nine times from LDS, with the KC channels' weights beside
// it; the nine taps need no further load and no barrier between them. A wave
// holds RW rows of 32 pixels by NT tiles of 32 channels and keeps the RW + 2
// input rows of a column shift in registers for the three taps that share
// them, so a tap costs a wave NT weight reads and a third of RW + 2 input
// reads for RW NT matrix instructions.
//
// The matrix instruction's rows are channels and its columns pixels, so a lane
// ends with runs of four channels of one pixel; the two halves of the wave
// trade runs and store 16 bytes each. Blocks go to the XCDs in contiguous runs
// of tiles: the halo a tile shares with its neighbours is in the same L2.
constexpr int kTH = 8, kTW = 32;
constexpr int kHaloW = kTW + 2, kHaloPixels = (kTH + 2) * kHaloW;

__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  const bf16x2 v = {(__bf16)lo, (__bf16)hi};
  return __builtin_bit_cast(uint32_t, v);
}

// the 16-byte slot of chunk c of staged pixel p: the chunks of a pixel are
// permuted by its place among 16, so 16 neighbouring pixels' same chunk sits
// in 16 different slots of the 64 banks
template <int S> __device__ __forceinline__ int staged(int p, int c) {
  return p * S + (c ^ (S == 4 ? (p >> 2) & 3 : (p >> 3) & 1));
}

template <int BN, int KC>
__global__ void __launch_bounds__(kThreads)
conv3x3_fwd(Image im, int tiles_x, int tiles_y, int cin, const uint4 *__restrict__ x,
            const uint4 *__restrict__ wt, const float *__restrict__ bias, int relu,
            uint16_t *__restrict__ y) {
  constexpr int S = KC / 8;                     // 16-byte chunks a pixel a stage
  constexpr int WN = BN == 128 ? 2 : 1;         // waves along the channels
  constexpr int RW = kTH * WN / 4;              // pixel rows a wave
  constexpr int NT = BN / WN / 32;              // channel tiles a wave
  __shared__ uint4 sx[kHaloPixels * S];
  __shared__ uint4 sw[9 * S * BN];              // [tap][chunk][channel]
  const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64;
  const int tile = cw::xcd_tile(blockIdx.x, gridDim.x);
  const int x0 = tile % tiles_x * kTW, y0 = tile / tiles_x % tiles_y * kTH;
  const int base = tile / (tiles_x * tiles_y) * im.h * im.w;  // the image's first pixel
  const int cin8 = cin / 8, krow8 = 9 * cin8;
  const int row0 = wave / WN * RW, n0 = wave % WN * (32 * NT);
  f32x16 acc[RW][NT];
#pragma unroll
  for (int i = 0; i < RW; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        acc[i][j][r] = 0.0f;
  for (int c0 = 0; c0 < cin8; c0 += S) {
    if (c0)
      __syncthreads();
#pragma unroll
    for (int k = 0; k < (kHaloPixels * S + kThreads - 1) / kThreads; ++k) {
      const int t = tid + k * kThreads;
      const int c = t % S, p = t / S;
      const int py = y0 + p / kHaloW - 1, px = x0 + p % kHaloW - 1;
      if (p < kHaloPixels) {
        uint4 v = {0, 0, 0, 0};
        if (py >= 0 && py < im.h && px >= 0 && px < im.w)
          v = x[(int64_t)(base + py * im.w + px) * cin8 + c0 + c];
        sx[staged<S>(p, c)] = v;
      }
    }
#pragma unroll
    for (int k = 0; k < (9 * S * BN + kThreads - 1) / kThreads; ++k) {
      const int t = tid + k * kThreads;
      const int c = t % S, n = t / S % BN, tap = t / (S * BN);
      if (tap < 9)
        sw[(tap * S + c) * BN + n] = wt[n * krow8 + tap * cin8 + c0 + c];
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < KC / 16; ++kk) {
      const int c = 2 * kk + lane / 32;
#pragma unroll
      for (int dw = 0; dw < 3; ++dw) {
        bf16x8 in[RW + 2];
#pragma unroll
        for (int i = 0; i < RW + 2; ++i)
          in[i] = __builtin_bit_cast(
              bf16x8, sx[staged<S>((row0 + i) * kHaloW + lane % 32 + dw, c)]);
#pragma unroll
        for (int dh = 0; dh < 3; ++dh)
#pragma unroll
          for (int j = 0; j < NT; ++j) {
            const bf16x8 w = __builtin_bit_cast(
                bf16x8, sw[((3 * dh + dw) * S + c) * BN + n0 + 32 * j + lane % 32]);
#pragma unroll
            for (int i = 0; i < RW; ++i)
              acc[i][j] =
                  __builtin_amdgcn_mfma_f32_32x32x16_bf16(w, in[i + dh], acc[i][j], 0, 0, 0);
          }
      }
    }
  }
  // epilogue: bias, activation, bfloat16; accumulator register r of a lane is
  // channel 8 (r / 4) + 4 (lane / 32) + r % 4 of pixel lane % 32
  const int px = x0 + lane % 32, half = lane / 32;
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int n = n0 + 32 * j;
    float4 b[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
      b[q] = bias ? *reinterpret_cast<const float4 *>(bias + n + 8 * q + 4 * half)
                  : float4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < RW; ++i) {
      const int py = y0 + row0 + i;
      uint2 v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float f[4] = {acc[i][j][4 * q] + b[q].x, acc[i][j][4 * q + 1] + b[q].y,
                      acc[i][j][4 * q + 2] + b[q].z, acc[i][j][4 * q + 3] + b[q].w};
        if (relu)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            f[e] = f[e] > 0.0f ? f[e] : 0.0f;
        v[q] = uint2{pack_bf16(f[0], f[1]), pack_bf16(f[2], f[3])};
      }
#pragma unroll
      for (int q = 0; q < 4; q += 2) {
        // the low half keeps run q and takes the high half's, the high half
        // run q + 1: eight channels in order each
        const uint2 give = half ? v[q] : v[q + 1];
        const uint2 got = {__shfl_xor(give.x, 32), __shfl_xor(give.y, 32)};
        const uint4 out = half ? uint4{got.x, got.y, v[q + 1].x, v[q + 1].y}
                               : uint4{v[q].x, v[q].y, got.x, got.y};
        if (px < im.w && py < im.h)
          *reinterpret_cast<uint4 *>(y + (int64_t)(base + py * im.w + px) * BN + n + 8 * q +
                                     8 * half) = out;
      }
    }
  }
}

template <int BN, int KC>
void launch_fwd(const cw_conv3x3_args &a, const Image &im, hipStream_t s) {
  const int tx = (a.w + kTW - 1) / kTW, ty = (a.h + kTH - 1) / kTH;
  hipLaunchKernelGGL((conv3x3_fwd<BN, KC>), dim3(tx * ty * a.n), dim3(kThreads), 0, s, im, tx, ty,
                     a.cin, (const uint4 *)a.x, (const uint4 *)a.weight, (const float *)a.bias,
                     a.relu, (uint16_t *)a.y);
}

// ------------------------------------------------------- backward weight
// one block: 128 rows of the (tap, ci) axis x BN output channels, summed
// over its run of pixels 32 at a time; the partial goes to part[split]
template <int BN>
__global__ void __launch_bounds__(kThreads)
conv3x3_wgrad(Image im, int cin, const uint4 *__restrict__ x, const uint4 *__restrict__ dy,
              int64_t run, float *__restrict__ part) {
  constexpr int P = 32; // pixels a step
  __shared__ __attribute__((aligned(16))) uint16_t sx[2][128][P + 8];
  __shared__ __attribute__((aligned(16))) uint16_t sd[2][BN][P + 8];
  const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64;
  const int krows = 9 * cin;
  const int r0 = blockIdx.x * 128;
  const int split = blockIdx.y;
  const int64_t p_begin = (int64_t)split * run;
  const int64_t p_end = p_begin + run < im.pixels ? p_begin + run : im.pixels;
  const int cin8 = cin / 8;
  constexpr int cout8 = BN / 8;
  constexpr int DPT = (P * cout8 + kThreads - 1) / kThreads; // dy chunks a thread
  // staging: x chunk (pixel xp, rows xr .. xr + 7) twice; dy chunks (pixel dp,
  // channels dc .. dc + 7)
  uint4 rx[2], rd[DPT];
  auto load = [&](int64_t q0) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int t = tid + h * kThreads;       // 512 chunks: 32 pixels x 16
      const int xp = t / 16, xr = r0 + (t % 16) * 8;
      rx[h] = uint4{0, 0, 0, 0};
      const int64_t p = q0 + xp;
      if (p < p_end && xr < krows) {
        const int tap = xr / cin, ci = xr % cin;
        const int64_t q = shifted(im, p, tap);
        if (q >= 0)
          rx[h] = x[q * cin8 + ci / 8];
      }
    }
#pragma unroll
    for (int h = 0; h < DPT; ++h) {
      const int t = tid + h * kThreads;
      const int dp = t / cout8, dc = (t % cout8) * 8;
      rd[h] = uint4{0, 0, 0, 0};
      const int64_t p = q0 + dp;
      if (dp < P && p < p_end)
        rd[h] = dy[p * cout8 + dc / 8];
    }
  };
  f32x16 acc[BN / 32];
#pragma unroll
  for (int j = 0; j < BN / 32; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      acc[j][r] = 0.0f;
  const int64_t steps = (p_end - p_begin + P - 1) / P;
  if (steps > 0)
    load(p_begin);
  for (int64_t s = 0; s < steps; ++s) {
    const int buf = (int)(s & 1);
    // transposed into LDS: [row][pixel], [channel][pixel]
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int t = tid + h * kThreads;
      const int xp = t / 16, xr = (t % 16) * 8;
      const uint16_t *v = reinterpret_cast<const uint16_t *>(&rx[h]);
#pragma unroll
      for (int i = 0; i < 8; ++i)
        sx[buf][xr + i][xp] = v[i];
    }
#pragma unroll
    for (int h = 0; h < DPT; ++h) {
      const int t = tid + h * kThreads;
      const int dp = t / cout8, dc = (t % cout8) * 8;
      if (dp < P) {
        const uint16_t *v = reinterpret_cast<const uint16_t *>(&rd[h]);
#pragma unroll
        for (int i = 0; i < 8; ++i)
          sd[buf][dc + i][dp] = v[i];
      }
    }
    __syncthreads();
    if (s + 1 < steps)
      load(p_begin + (s + 1) * P);
    // rows of P + 8 bfloat16 (80 bytes), so a lane's eight pixels are one
    // aligned 16-byte LDS read
#pragma unroll
    for (int k = 0; k < P; k += 16) {
      const bf16x8 av = __builtin_bit_cast(
          bf16x8, *reinterpret_cast<const uint4 *>(&sx[buf][wave * 32 + lane % 32][k + 8 * (lane / 32)]));
#pragma unroll
      for (int j = 0; j < BN / 32; ++j) {
        const bf16x8 bv = __builtin_bit_cast(
            bf16x8, *reinterpret_cast<const uint4 *>(&sd[buf][j * 32 + lane % 32][k + 8 * (lane / 32)]));
        acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, bv, acc[j], 0, 0, 0);
      }
    }
  }
  // the partial: part[split][row][co]
  float *out = part + (int64_t)split * krows * BN;
#pragma unroll
  for (int j = 0; j < BN / 32; ++j) {
    const int n = j * 32 + lane % 32;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = r0 + wave * 32 + 8 * (r / 4) + 4 * (lane / 32) + r % 4;
      if (row < krows)
        out[(int64_t)row * BN + n] = acc[j][r];
    }
  }
}

// dw[co][row] = sum over the splits in order of part[split][row][co]
__global__ void __launch_bounds__(kThreads)
conv3x3_wgrad_sum(int krows, int cout, int splits, const float *__restrict__ part,
                  float *__restrict__ dw) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (int64_t)krows * cout)
    return;
  const int row = (int)(t / cout), co = (int)(t % cout);
  float s = 0.0f;
  for (int k = 0; k < splits; ++k)
    s += part[((int64_t)k * krows + row) * cout + co];
  dw[(int64_t)co * krows + row] = s;
}

// the kernels' weights from the float32 master: wt (cout, 9 cin) as is and
// wd (cin, 9 cout) flipped in space and transposed in channels
__global__ void __launch_bounds__(kThreads)
conv3x3_weights(int cout, int cin, const float *__restrict__ w, uint16_t *__restrict__ wt,
                uint16_t *__restrict__ wd) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (int64_t)cout * 9 * cin)
    return;
  const int co = (int)(t / (9 * cin)), k = (int)(t % (9 * cin));
  const int tap = k / cin, ci = k % cin;
  const uint16_t b = to_bf16(w[t]);
  wt[t] = b;
  if (wd)
    wd[(int64_t)ci * 9 * cout + (8 - tap) * cout + co] = b;
}

// AdamW (decoupled weight decay, bias-corrected moments)
__global__ void __launch_bounds__(kThreads)
adamw(int64_t count, float *__restrict__ p, const float *__restrict__ g, float *__restrict__ m,
      float *__restrict__ v, float lr, float beta1, float beta2, float eps, float decay,
      float c1, float c2) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count)
    return;
  const float gi = g[i];
  float pi = p[i] * (1.0f - lr * decay);
  const float mi = beta1 * m[i] + (1.0f - beta1) * gi;
  const float vi = beta2 * v[i] + (1.0f - beta2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float mhat = mi / c1, vhat = vi / c2;
  pi -= lr * mhat / (sqrtf(vhat) + eps);
  p[i] = pi;
}

int check_conv(const cw_conv3x3_args *a) {
  if (!a)
    return fail("args is NULL");
  if (a->n < 1 || a->h < 1 || a->w < 1)
    return fail("the image needs a positive batch, height and width");
  if (a->cin < 16 || a->cin % 16)
    return fail("cin must be a positive multiple of 16");
  if (a->cout != 32 && a->cout != 64 && a->cout != 128)
    return fail("cout must be 32, 64 or 128");
  if ((int64_t)a->n * a->h * a->w * (a->cin > a->cout ? a->cin : a->cout) >= (int64_t)1 << 31)
    return fail("the image overflows the int32 element index of a row");
  return 0;
}

int hip_status(const char *where) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    fail(std::string(where) + ": " + hipGetErrorString(e));
    return 2;
  }
  return 0;
}

} // namespace

extern "C" {

int cw_conv3x3_bf16_fwd(const cw_conv3x3_args *a, void *stream) {
  if (int e = check_conv(a))
    return e;
  if (!a->x || !a->weight || !a->y)
    return fail("the forward needs x, weight and y");
  const Image im{a->n, a->h, a->w, (int64_t)a->n * a->h * a->w};
  const auto s = (hipStream_t)stream;
  const bool wide = a->cin % 32 == 0;
  switch (a->cout) {
  case 32:
    wide ? launch_fwd<32, 32>(*a, im, s) : launch_fwd<32, 16>(*a, im, s);
    break;
  case 64:
    launch_fwd<64, 16>(*a, im, s);
    break;
  default:
    launch_fwd<128, 16>(*a, im, s);
  }
  return hip_status("conv3x3_fwd");
}

int cw_conv3x3_bf16_bwd_data(const cw_conv3x3_args *a, void *stream) {
  // dy (cout channels) through the flipped, transposed weights into dx (cin)
  if (int e = check_conv(a))
    return e;
  if (!a->dy || !a->weight_flipped || !a->dx)
    return fail("the backward data pass needs dy, the flipped weights and dx");
  if (a->cin != 32 && a->cin != 64 && a->cin != 128)
    return fail("the backward data pass writes 32, 64 or 128 channels");
  cw_conv3x3_args b = *a;
  b.cin = a->cout;
  b.cout = a->cin;
  b.x = a->dy;
  b.weight = a->weight_flipped;
  b.bias = nullptr;
  b.relu = 0;
  b.y = a->dx;
  return cw_conv3x3_bf16_fwd(&b, stream);
}

int cw_conv3x3_bf16_bwd_weight(const cw_conv3x3_args *a, void *stream) {
  if (int e = check_conv(a))
    return e;
  if (!a->x || !a->dy || !a->dweight || !a->workspace || a->splits < 1)
    return fail("the backward weight pass needs x, dy, dweight, a workspace and splits");
  const Image im{a->n, a->h, a->w, (int64_t)a->n * a->h * a->w};
  const int krows = 9 * a->cin;
  const int64_t run = (im.pixels + a->splits - 1) / a->splits;
  const dim3 grid((krows + 127) / 128, a->splits);
  const auto s = (hipStream_t)stream;
  const uint4 *x = (const uint4 *)a->x, *dy = (const uint4 *)a->dy;
  float *part = (float *)a->workspace;
  switch (a->cout) {
  case 32: hipLaunchKernelGGL(conv3x3_wgrad<32>, grid, dim3(kThreads), 0, s, im, a->cin, x, dy, run, part); break;
  case 64: hipLaunchKernelGGL(conv3x3_wgrad<64>, grid, dim3(kThreads), 0, s, im, a->cin, x, dy, run, part); break;
  default: hipLaunchKernelGGL(conv3x3_wgrad<128>, grid, dim3(kThreads), 0, s, im, a->cin, x, dy, run, part); break;
  }
  if (int e = hip_status("conv3x3_wgrad"))
    return e;
  const int64_t total = (int64_t)krows * a->cout;
  hipLaunchKernelGGL(conv3x3_wgrad_sum, dim3((int)((total + kThreads - 1) / kThreads)),
                     dim3(kThreads), 0, s, krows, a->cout, a->splits, (const float *)part,
                     (float *)a->dweight);
  return hip_status("conv3x3_wgrad_sum");
}

int cw_conv3x3_weights(int32_t cout, int32_t cin, const void *w, void *wt, void *wd,
                       void *stream) {
  if (cout < 1 || cin < 1 || !w || !wt)
    return fail("the weight transform needs cout, cin, w and wt");
  const int64_t total = (int64_t)cout * 9 * cin;
  hipLaunchKernelGGL(conv3x3_weights, dim3((int)((total + kThreads - 1) / kThreads)),
                     dim3(kThreads), 0, (hipStream_t)stream, cout, cin, (const float *)w,
                     (uint16_t *)wt, (uint16_t *)wd);
  return hip_status("conv3x3_weights");
}

int cw_adamw(const cw_adamw_args *a, void *stream) {
  if (!a || a->count < 0 || (a->count && (!a->param || !a->grad || !a->m || !a->v)))
    return fail("AdamW needs param, grad, m and v");
  if (a->step < 1)
    return fail("AdamW steps count from 1");
  if (!a->count)
    return 0;
  const float c1 = 1.0f - powf(a->beta1, (float)a->step);
  const float c2 = 1.0f - powf(a->beta2, (float)a->step);
  hipLaunchKernelGGL(adamw, dim3((int)((a->count + kThreads - 1) / kThreads)), dim3(kThreads),
                     0, (hipStream_t)stream, a->count, (float *)a->param, (const float *)a->grad,
                     (float *)a->m, (float *)a->v, a->lr, a->beta1, a->beta2, a->eps,
                     a->weight_decay, c1, c2);
  return hip_status("adamw");
}

} // extern "C"
