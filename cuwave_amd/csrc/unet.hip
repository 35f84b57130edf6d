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
//   added tap by tap. A block takes a tile of 8 x 32 pixels, whose input with
//   its halo is in LDS once for all nine taps (conv3x3_fwd); images of a few
//   pixels a side and more than 128 channels take runs of 128 pixels, gathered
//   a tap at a time (conv3x3_fwd_flat): the same sums in the same order.
// - backward data: the same kernels on dy with the weights flipped in space
//   and transposed in channels (wd[ci][tap][co] = w[co][8 - tap][ci]).
// - backward weight: dw[co][tap][ci] = sum_p dy[p][co] x[p + off(tap)][ci].
//   A block marches down the rows of a strip of 64 columns with every tap's
//   sums in registers (conv3x3_wgrad); small images and layers take runs of
//   pixels a block (conv3x3_wgrad_flat). Either writes its float32 partial to a
//   slice, and slices_sum adds the slices in a fixed order (deterministic, no
//   atomics).
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
// (BN = cout, 32 / 64 / 128). A 32 -> 32 layer has 144 flops a byte of
// activations read and written, so the input has to reach the block once; what
// bounds it then is the LDS, its bandwidth and, from 64 channels up, its size:
// two blocks a CU at 64, one at 128 (which has eight waves for it: with four
// 128 -> 64 at 16 x 290 x 304 took 526 us). The sums run tap by tap, 16 channels an
// instruction within a tap: a pre-activation within rounding of zero takes the
// sign this order gives it, the ReLU's gradient follows that sign, and another
// order turns some of them (a few in 1e8), each worth up to |dy w| in the
// gradient at the input.
//
// So the tile's input with its one-pixel halo is staged once for all nine taps,
// every channel of it (KC >= cin), and the weights T taps at a time in two LDS
// buffers in turn: the next taps' are in registers while these are multiplied,
// one barrier a turn. KC is the least of 16, 32, 64 and 128 that holds cin
// (channels past cin are zeros), T is 3 where that is 32 or less and a tap's
// products are too few to cover a barrier. A wave holds RW rows of 32 pixels
// by NT tiles of 32 channels: RW + NT 16-byte LDS reads a lane for RW NT matrix
// instructions, which at two by two is the LDS's rate at the instructions' own.
//
// At 16 x 580 x 608: 32 -> 32 220 us (279 with the taps innermost and the
// channels staged in turn, 611 by the flat kernel), 64 -> 32 405 (417, 1240);
// at half that 64 -> 64 199 (183, 424), 128 -> 64 363 (319, 841); 128 -> 128 at
// a quarter 133 (180, 306).
//
// A plane of LDS holds eight channels of every staged pixel, so a wave's reads
// are runs of 32 pixels; kPlane keeps the writes (a pixel's planes one after
// the other) off each other's banks. The weights' channels are permuted by
// their chunk for the same reason.
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

// the 16-byte slots of an LDS plane: 16 / S modulo the 16 slots of the 64 banks
template <int S> constexpr int plane_slots() {
  return (kHaloPixels - 16 / S + 15) / 16 * 16 + 16 / S;
}

template <int BN, int KC, int T, int THREADS>
__global__ void __launch_bounds__(THREADS, 2)
conv3x3_fwd(Image im, int tiles_x, int tiles_y, int cin, const uint4 *__restrict__ x,
            const uint4 *__restrict__ wt, const float *__restrict__ bias, int relu,
            uint16_t *__restrict__ y) {
  constexpr int S = KC / 8;                     // 16-byte chunks a pixel a stage
  constexpr int WAVES = THREADS / 64;
  constexpr int WN = BN == 128 ? 2 : 1;         // waves along the channels
  constexpr int RW = kTH * WN / WAVES;          // pixel rows a wave
  constexpr int NT = BN / WN / 32;              // channel tiles a wave
  constexpr int kPlane = plane_slots<S>();
  constexpr int kWeights = T * S * BN;          // chunks of weights a stage
  constexpr int kMine = (kWeights + THREADS - 1) / THREADS;
  __shared__ uint4 sx[S * kPlane];              // [chunk][pixel]
  __shared__ uint4 sw[2][kWeights];             // [tap][chunk][channel ^ chunk]
  const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64, half = lane / 32;
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
  uint4 ahead[kMine];
  auto fetch_weights = [&](int stage) {
#pragma unroll
    for (int k = 0; k < kMine; ++k) {
      const int t = tid + k * THREADS;
      const int c = t % S, n = t / S % BN, tap = t / (S * BN);
      ahead[k] = uint4{0, 0, 0, 0};
      if (tap < T && c < cin8)
        ahead[k] = wt[n * krow8 + (stage * T + tap) * cin8 + c];
    }
  };
  auto stage_weights = [&](int stage) {
#pragma unroll
    for (int k = 0; k < kMine; ++k) {
      const int t = tid + k * THREADS;
      const int c = t % S, n = t / S % BN, tap = t / (S * BN);
      if (tap < T)
        sw[stage & 1][(tap * S + c) * BN + (n ^ (c & 15))] = ahead[k];
    }
  };
  fetch_weights(0);
#pragma unroll
  for (int k = 0; k < (kHaloPixels * S + THREADS - 1) / THREADS; ++k) {
    const int t = tid + k * THREADS;
    const int c = t % S, p = t / S;
    const int py = y0 + p / kHaloW - 1, px = x0 + p % kHaloW - 1;
    if (p < kHaloPixels) {
      uint4 v = {0, 0, 0, 0};
      if (py >= 0 && py < im.h && px >= 0 && px < im.w && c < cin8)
        v = x[(int64_t)(base + py * im.w + px) * cin8 + c];
      sx[c * kPlane + p] = v;
    }
  }
  stage_weights(0);
  for (int stage = 0; stage < 9 / T; ++stage) {
    __syncthreads();
    if (stage + 1 < 9 / T)
      fetch_weights(stage + 1);
    const uint4 *weights = sw[stage & 1];
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const uint4 *from = sx + (row0 + (stage * T + t) / 3) * kHaloW + lane % 32 +
                          (stage * T + t) % 3;
#pragma unroll
      for (int kk = 0; kk < KC / 16; ++kk) {
        const int c = 2 * kk + half;
        bf16x8 in[RW], w[NT];
#pragma unroll
        for (int i = 0; i < RW; ++i)
          in[i] = __builtin_bit_cast(bf16x8, from[c * kPlane + i * kHaloW]);
#pragma unroll
        for (int j = 0; j < NT; ++j)
          w[j] = __builtin_bit_cast(
              bf16x8, weights[(t * S + c) * BN + ((n0 + 32 * j + lane % 32) ^ (c & 15))]);
#pragma unroll
        for (int i = 0; i < RW; ++i)
#pragma unroll
          for (int j = 0; j < NT; ++j)
            acc[i][j] =
                __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[j], in[i], acc[i][j], 0, 0, 0);
      }
    }
    if (stage + 1 < 9 / T)
      stage_weights(stage + 1);
  }
  // epilogue: bias, activation, bfloat16; accumulator register r of a lane is
  // channel 8 (r / 4) + 4 (lane / 32) + r % 4 of pixel lane % 32
  const int px = x0 + lane % 32;
  const bool wide = (reinterpret_cast<uintptr_t>(y) & 15) == 0; // else two bytes a store
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int n = n0 + 32 * j;
    float b[16];
#pragma unroll
    for (int r = 0; r < 16; ++r)
      b[r] = bias ? bias[n + 8 * (r / 4) + 4 * half + r % 4] : 0.0f;
#pragma unroll
    for (int i = 0; i < RW; ++i) {
      const int py = y0 + row0 + i;
      uint2 v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float f[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          f[e] = acc[i][j][4 * q + e] + b[4 * q + e];
          if (relu)
            f[e] = f[e] > 0.0f ? f[e] : 0.0f;
        }
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
        if (px >= im.w || py >= im.h)
          continue;
        uint16_t *to = y + (int64_t)(base + py * im.w + px) * BN + n + 8 * q + 8 * half;
        if (wide) {
          *reinterpret_cast<uint4 *>(to) = out;
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            to[e] = (uint16_t)((&out.x)[e / 2] >> (16 * (e & 1)));
        }
      }
    }
  }
}

// What the tiles waste or don't hold: images of a few pixels a side, and more
// channels than 128. One block: 128 pixels of the whole batch in memory order x
// BN output channels, wave w the pixels 32 w .. 32 w + 31 and every channel, its
// input gathered from memory once a tap, 16 channels a barrier: the same sums
// in the same order.
constexpr int kBM = 128; // pixels a flat block takes (4 waves x 32)
constexpr int kBK = 16;  // reduction step: 16 channels of one tap

template <int BN>
__global__ void __launch_bounds__(kThreads)
conv3x3_fwd_flat(Image im, int cin, const uint4 *__restrict__ x, const uint4 *__restrict__ wt,
            const float *__restrict__ bias, int relu, uint16_t *__restrict__ y) {
  __shared__ uint4 sa[2][kBM * 2];  // [m][k]: 16 bf16 a row, two uint4
  __shared__ uint4 sb[2][BN * 2];   // [n][k]
  const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64;
  const int64_t m0 = (int64_t)blockIdx.x * kBM;
  const int steps = 9 * (cin / kBK);
  const int cin8 = cin / 8;      // uint4 chunks a pixel
  const int krow8 = 9 * cin8;    // uint4 chunks a weight row
  // the chunk this thread stages: pixel am, half ah; weight row bn, half bh
  const int am = tid / 2, ah = tid % 2;
  const int bn = tid / 2, bh = tid % 2;
  uint4 ra = {0, 0, 0, 0}, rb = {0, 0, 0, 0};
  auto load = [&](int s) {
    const int tap = s / (cin / kBK), c0 = (s % (cin / kBK)) * kBK;
    const int64_t p = m0 + am;
    ra = uint4{0, 0, 0, 0};
    if (p < im.pixels) {
      const int64_t q = shifted(im, p, tap);
      if (q >= 0)
        ra = x[q * cin8 + c0 / 8 + ah];
    }
    if (bn < BN)
      rb = wt[(int64_t)bn * krow8 + tap * cin8 + c0 / 8 + bh];
  };
  f32x16 acc[BN / 32];
#pragma unroll
  for (int j = 0; j < BN / 32; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      acc[j][r] = 0.0f;
  load(0);
  for (int s = 0; s < steps; ++s) {
    const int buf = s & 1;
    sa[buf][am * 2 + ah] = ra;
    if (bn < BN)
      sb[buf][bn * 2 + bh] = rb;
    __syncthreads();
    if (s + 1 < steps)
      load(s + 1);
    const uint4 a = sa[buf][(wave * 32 + lane % 32) * 2 + lane / 32];
    const bf16x8 av = __builtin_bit_cast(bf16x8, a);
#pragma unroll
    for (int j = 0; j < BN / 32; ++j) {
      const uint4 b = sb[buf][(j * 32 + lane % 32) * 2 + lane / 32];
      acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, __builtin_bit_cast(bf16x8, b),
                                                      acc[j], 0, 0, 0);
    }
  }
  // epilogue: bias, activation, bfloat16
#pragma unroll
  for (int j = 0; j < BN / 32; ++j) {
    const int n = j * 32 + lane % 32;
    const float b = bias ? bias[n] : 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int m = wave * 32 + 8 * (r / 4) + 4 * (lane / 32) + r % 4;
      const int64_t p = m0 + m;
      if (p >= im.pixels)
        continue;
      float v = acc[j][r] + b;
      if (relu)
        v = v > 0.0f ? v : 0.0f;
      y[p * BN + n] = to_bf16(v);
    }
  }
}

template <int BN, int KC>
void launch_fwd(const cw_conv3x3_args &a, const Image &im, hipStream_t s) {
  const int tx = (a.w + kTW - 1) / kTW, ty = (a.h + kTH - 1) / kTH;
  constexpr int threads = KC == 128 ? 512 : 256;
  hipLaunchKernelGGL((conv3x3_fwd<BN, KC, KC <= 32 ? 3 : 1, threads>), dim3(tx * ty * a.n),
                     dim3(threads), 0, s, im, tx, ty, a.cin, (const uint4 *)a.x, (const uint4 *)a.weight,
                     (const float *)a.bias, a.relu, (uint16_t *)a.y);
}

// Whether the flat kernel takes the layer. It costs a pixel of an image what it
// costs any other, the tiles a pixel of the padded image a third to a fifth of
// that: tiles, where they fill the card, from the share of true pixels up at
// which both took the same time (at 16 channels to 32 in 0.19, 40000 x 6: 31
// and 32 us; at 64 to 64 0.30, 2048 images of 12 x 12 (0.28): 82 and 92, of 4 x
// 40 (0.31): 88 and 83; at 128 to 128 0.33, the same two: 235 and 289, 266 and
// 280, 25000 x 12 (0.38): 266 and 239), and tiles always where the card holds
// all of them at once (4096 images of 8 x 8 at 128 channels 214 and 280 us, one
// of 8 x 8 51 and 16). Past 128 channels the tile would be staged again for
// each tap (6 x 200 x 225, 256 to 128: 446 us flat, 697 so).
bool flat_fwd(const cw_conv3x3_args &a) {
  if (a.cin > 128)
    return true;
  const int64_t tiles = (int64_t)a.n * ((a.h + kTH - 1) / kTH) * ((a.w + kTW - 1) / kTW);
  const int at_once = a.cin <= 32 ? 1024 : a.cin <= 64 ? 512 : 256;
  const double least = a.cin <= 32 ? 0.2 : a.cin <= 64 ? 0.3 : 0.33;
  return tiles > at_once && (double)a.n * a.h * a.w < least * (double)(tiles * (kTH * kTW));
}

template <int BN>
void launch_fwd(const cw_conv3x3_args &a, const Image &im, hipStream_t s) {
  if (flat_fwd(a))
    hipLaunchKernelGGL(conv3x3_fwd_flat<BN>, dim3((int)((im.pixels + kBM - 1) / kBM)),
                       dim3(kThreads), 0, s, im, a.cin, (const uint4 *)a.x,
                       (const uint4 *)a.weight, (const float *)a.bias, a.relu, (uint16_t *)a.y);
  else if (a.cin <= 16)
    launch_fwd<BN, 16>(a, im, s);
  else if (a.cin <= 32)
    launch_fwd<BN, 32>(a, im, s);
  else if (a.cin <= 64)
    launch_fwd<BN, 64>(a, im, s);
  else
    launch_fwd<BN, 128>(a, im, s);
}

// ------------------------------------------------------- backward weight
// dw[co][tap][ci] = sum over pixels of dy[co] x shifted by the tap: a product
// whose reduction runs along the pixels, so both operands are wanted with
// eight neighbouring pixels of one channel a lane where memory has eight
// channels of one pixel. A thread takes four pixels by eight channels and
// writes them to LDS transposed (two packed pixels an instruction).
//
// A block marches down the rows of a strip of kWStrip columns, CI input and CO
// output channels wide, two input rows in LDS (one being filled) and a ring of
// four gradient rows. An input row meets the gradient rows below, at and above
// it, and its eight-pixel runs shifted by -1, 0 and +1 pixel come from one
// 16-byte read and the words either side: nine matrix instructions for four
// and a half LDS reads, every tap of a (CI, CO) tile accumulated in one pass
// over the data. What bounds it is HBM: x and dy are read once for every 64
// channels of the other. The nine tiles of sums are 144 registers, so two
// blocks a CU; the host asks for splits that give each CU its two.
//
// The waves take the (32, 32) channel tiles, and where there are fewer than
// four the strip's 16-column steps between them, summed through LDS at the
// end. Each split's sums go to its own workspace slice and a second kernel
// adds the slices in a fixed order (deterministic, no atomics).
constexpr int kWStrip = 64;

// the 16-byte slot of eight-pixel run k of channel c, a row of eight runs: 16
// neighbouring channels' same run, and the same run of channels eight apart,
// fall in different slots of the 64 banks
__device__ __forceinline__ int run_slot(int c, int k) {
  return c * 8 + (k ^ ((c >> 1 ^ c >> 3) & 7));
}

// four pixels of eight channels (one uint4 a pixel) into a transposed row:
// pixels 4 q .. 4 q + 3 of channels 8 cg .. 8 cg + 7
__device__ __forceinline__ void put_transposed(uint4 *row, int cg, int q, const uint4 *v) {
  const uint32_t *w[4] = {&v[0].x, &v[1].x, &v[2].x, &v[3].x};
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    // the low or the high halves of two pixels' word i / 2
    const uint32_t pick = i & 1 ? 0x07060302u : 0x05040100u;
    const uint2 two = {__builtin_amdgcn_perm(w[1][i / 2], w[0][i / 2], pick),
                       __builtin_amdgcn_perm(w[3][i / 2], w[2][i / 2], pick)};
    reinterpret_cast<uint2 *>(&row[run_slot(8 * cg + i, q / 2)])[q & 1] = two;
  }
}

template <int CI, int CO>
__global__ void __launch_bounds__(kThreads, 2)
conv3x3_wgrad(Image im, int strips, int cin, int cout, const uint4 *__restrict__ x,
              const uint4 *__restrict__ dy, int run, float *__restrict__ part) {
  constexpr int TI = CI / 32, TO = CO / 32;
  constexpr int KW = 4 / (TI * TO);       // waves that share a tile
  constexpr int KS = kWStrip / 16 / KW;   // 16-column steps a wave takes
  __shared__ uint4 sx[2][CI * 8];
  __shared__ uint32_t halo[2][2][CI];     // the pixel left (high half) and right (low half)
  __shared__ uint4 sd[4][CO * 8];
  const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64, half = lane / 32;
  const int kw = wave % KW, ti = wave / KW % TI, to = wave / (KW * TI);
  const int ciblocks = (cin + CI - 1) / CI;
  const int ci0 = blockIdx.x % ciblocks * CI, co0 = blockIdx.x / ciblocks * CO;
  const int split = blockIdx.y;
  const int cin8 = cin / 8, cout8 = cout / 8;
  // staging: threads 0 .. 127 four pixels of x each, the rest of dy (CI = 32
  // or CO = 32 fill half of theirs), 2 CI / 8 threads a halo pixel too
  const bool on_x = tid < 128;
  const int task = on_x ? tid : tid - 128;
  const int groups = on_x ? CI / 8 : CO / 8;
  const int cg = task % groups, q = task / groups;
  const bool mine = q < kWStrip / 4 && (!on_x || ci0 + 8 * cg < cin);
  const bool zeroed = on_x && q < kWStrip / 4 && ci0 + 8 * cg >= cin; // channels past the last
  const bool edge = tid < 2 * (CI / 8);
  const int ecg = tid % (CI / 8), eside = tid / (CI / 8);
  f32x16 acc[9];
#pragma unroll
  for (int j = 0; j < 9; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      acc[j][r] = 0.0f;
  // the split's run of gradient rows, strip after strip of each image
  const int64_t total = (int64_t)im.n * strips * im.h;
  int64_t at = (int64_t)split * run;
  const int64_t end = at + run < total ? at + run : total;
  while (at < end) {
    const int s = (int)(at / im.h);
    const int a = (int)(at - (int64_t)s * im.h);
    const int b = (int)(end - (int64_t)s * im.h < im.h ? end - (int64_t)s * im.h : im.h);
    at += b - a;
    const int c0 = s % strips * kWStrip;                 // the strip's first column
    const int base = s / strips * im.h * im.w;           // the image's first pixel
    const bool ragged = im.w - c0 < kWStrip;             // the image ends in the strip
    uint4 v[4], ev;
    // input row r into the x registers, gradient row r + 1 into the dy ones
    auto fetch = [&](int r) {
      const int row = on_x ? r : r + 1;
      const bool there = on_x ? r >= 0 && r < im.h : row >= a && row < b;
      const uint4 *src = on_x ? x + ci0 / 8 + cg : dy + co0 / 8 + cg;
      const int step = on_x ? cin8 : cout8;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int col = c0 + 4 * q + i;
        v[i] = uint4{0, 0, 0, 0};
        if (mine && there && col < im.w)
          v[i] = src[(int64_t)(base + row * im.w + col) * step];
      }
      const int col = eside ? c0 + kWStrip : c0 - 1;
      ev = uint4{0, 0, 0, 0};
      if (edge && r >= 0 && r < im.h && col >= 0 && col < im.w && ci0 + 8 * ecg < cin)
        ev = x[(int64_t)(base + r * im.w + col) * cin8 + ci0 / 8 + ecg];
    };
    auto stage = [&](int r) {
      if (mine || zeroed)
        put_transposed(on_x ? sx[r & 1] : sd[(r + 1) & 3], cg, q, v);
      if (edge) {
        const uint32_t *w = &ev.x;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const uint32_t px = i & 1 ? w[i / 2] >> 16 : w[i / 2] & 0xffffu;
          halo[r & 1][eside][8 * ecg + i] = eside ? px : px << 16;
        }
      }
    };
    __syncthreads(); // the rows of the segment before have been read
    fetch(a - 1);
    stage(a - 1);
    for (int r = a - 1; r <= b; ++r) {
      __syncthreads();
      if (r < b)
        fetch(r + 1);
      const uint4 *xr = sx[r & 1];
      const int ci = 32 * ti + lane % 32, co = 32 * to + lane % 32;
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        const int g = 2 * (kw + KW * k) + half; // this lane's run of eight pixels
        const uint4 m = xr[run_slot(ci, g)];
        const uint32_t left =
            g ? xr[run_slot(ci, g ? g - 1 : 0)].w : halo[r & 1][0][ci];
        const uint32_t right =
            g < 7 ? xr[run_slot(ci, g < 7 ? g + 1 : 7)].x : halo[r & 1][1][ci];
        const uint32_t a0 = __builtin_amdgcn_alignbit(m.x, left, 16);
        const uint32_t a1 = __builtin_amdgcn_alignbit(m.y, m.x, 16);
        const uint32_t a2 = __builtin_amdgcn_alignbit(m.z, m.y, 16);
        const uint32_t a3 = __builtin_amdgcn_alignbit(m.w, m.z, 16);
        const uint32_t a4 = __builtin_amdgcn_alignbit(right, m.w, 16);
        uint4 before = {a0, a1, a2, a3};
        if (ragged) { // the column past the last meets the last one's value: no pixel
          const int d = im.w - c0 - 8 * g;
          const uint32_t keep = d & 1 ? 0x0000ffffu : 0xffff0000u;
          before.x &= d >> 1 == 0 ? keep : ~0u;
          before.y &= d >> 1 == 1 ? keep : ~0u;
          before.z &= d >> 1 == 2 ? keep : ~0u;
          before.w &= d >> 1 == 3 ? keep : ~0u;
        }
        const bf16x8 in[3] = {__builtin_bit_cast(bf16x8, before),
                              __builtin_bit_cast(bf16x8, m),
                              __builtin_bit_cast(bf16x8, uint4{a1, a2, a3, a4})};
#pragma unroll
        for (int dh = 0; dh < 3; ++dh) {
          const int row = r + 1 - dh; // the gradient row whose tap dh is input row r
          if (row < a || row >= b)
            continue;
          const bf16x8 d = __builtin_bit_cast(bf16x8, sd[row & 3][run_slot(co, g)]);
#pragma unroll
          for (int dw = 0; dw < 3; ++dw)
            acc[3 * dh + dw] =
                __builtin_amdgcn_mfma_f32_32x32x16_bf16(d, in[dw], acc[3 * dh + dw], 0, 0, 0);
        }
      }
      if (r < b)
        stage(r + 1);
    }
  }
  // the waves of a tile summed into its first, a tap at a time
  if constexpr (KW > 1) {
    float *sums = reinterpret_cast<float *>(sd); // (KW - 1) tiles' 4 KB fit the ring
    static_assert(sizeof(sd) >= (size_t)TI * TO * (KW - 1) * 4096, "the sums need room");
#pragma unroll
    for (int j = 0; j < 9; ++j) {
      __syncthreads();
      if (kw)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          sums[(((ti + TI * to) * (KW - 1) + kw - 1) * 16 + r) * 64 + lane] = acc[j][r];
      __syncthreads();
      if (!kw)
        for (int o = 0; o < KW - 1; ++o)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            acc[j][r] += sums[(((ti + TI * to) * (KW - 1) + o) * 16 + r) * 64 + lane];
    }
    if (kw)
      return;
  }
  // the partial: part[split][co][tap][ci], dw's own order
  const int ci = ci0 + 32 * ti + lane % 32;
  if (ci >= cin)
    return;
  float *out = part + (int64_t)split * cout * 9 * cin;
#pragma unroll
  for (int j = 0; j < 9; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int co = co0 + 32 * to + 8 * (r / 4) + 4 * half + r % 4;
      out[(co * 9 + j) * cin + ci] = acc[j][r];
    }
}

// What the strips waste: images of a few pixels a side, and layers of so few
// pixels that a strip's march is one or two blocks long. One block: 128 rows of
// the (tap, ci) axis x BN output channels, summed over its run of pixels of the
// whole batch 32 at a time, x gathered from memory once a tap.
template <int BN>
__global__ void __launch_bounds__(kThreads)
conv3x3_wgrad_flat(Image im, int cin, const uint4 *__restrict__ x, const uint4 *__restrict__ dy,
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
        acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bv, av, acc[j], 0, 0, 0);
      }
    }
  }
  // the partial: part[split][co][row], dw's own order
  const int row = r0 + wave * 32 + lane % 32;
  if (row >= krows)
    return;
  float *out = part + (int64_t)split * krows * BN;
#pragma unroll
  for (int j = 0; j < BN / 32; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      out[(j * 32 + 8 * (r / 4) + 4 * (lane / 32) + r % 4) * krows + row] = acc[j][r];
}

// out = the sum over the slices: a thread one value of every fourth slice, eight
// loads in flight, the four threads' sums then added in order
__global__ void __launch_bounds__(kThreads)
slices_sum(int total, int splits, const float *__restrict__ part, float *__restrict__ out) {
  __shared__ float sums[4][64];
  const int lane = threadIdx.x % 64, group = threadIdx.x / 64;
  const int t = blockIdx.x * 64 + lane;
  float s = 0.0f;
  if (t < total) {
#pragma unroll 8
    for (int k = group; k < splits; k += 4)
      s += part[(int64_t)k * total + t];
  }
  sums[group][lane] = s;
  __syncthreads();
  if (group || t >= total)
    return;
  out[t] = s + sums[1][lane] + sums[2][lane] + sums[3][lane];
}

void launch_slices_sum(int total, int slices, const void *part, void *out, hipStream_t s) {
  hipLaunchKernelGGL(slices_sum, dim3((total + 63) / 64), dim3(kThreads), 0, s, total, slices,
                     (const float *)part, (float *)out);
}

// ------------------------------------------------- passes over activations
// Both run at HBM's rate with 16 bytes (eight channels of a pixel) a thread:
// what they save is passes. Per-channel sums stay in registers over a block's
// pixels, are added over the block's threads of a channel in a fixed order,
// and leave as one slice a block for slices_sum.
__device__ __forceinline__ void unpack8(const uint4 &v, float *f) {
  const uint32_t *w = &v.x;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = __uint_as_float(w[i] << 16);
    f[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
  }
}

// the N values a thread holds summed over the block's threads t % G equal,
// thread t < G ending with its sums
template <int N, int G>
__device__ __forceinline__ void block_sums(float *s, float *lds) {
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
#pragma unroll
  for (int i = 0; i < N; ++i) {
#pragma unroll
    for (int m = G; m < 64; m <<= 1)
      s[i] += __shfl_xor(s[i], m);
    if (lane < G)
      lds[(wave * N + i) * G + lane] = s[i];
  }
  __syncthreads();
  if (threadIdx.x < G)
#pragma unroll
    for (int i = 0; i < N; ++i) {
      s[i] = lds[i * G + threadIdx.x];
      for (int o = 1; o < kThreads / 64; ++o)
        s[i] += lds[(o * N + i) * G + threadIdx.x];
    }
}

// the gradient before the activation, dy where y > 0, and its sums over the
// pixels (the bias' gradient) in the same pass: 6 bytes a value instead of the
// 16 of a comparison, a select, a conversion and a sum. y NULL (no
// activation): the sums alone
template <int C>
__global__ void __launch_bounds__(kThreads)
relu_bias_grad(int64_t chunks, const uint4 *__restrict__ dy, const uint4 *__restrict__ y,
               uint4 *__restrict__ dpre, float *__restrict__ part) {
  constexpr int G = C / 8;
  __shared__ float lds[kThreads / 64 * 8 * G];
  float s[8] = {};
  const int64_t step = (int64_t)gridDim.x * kThreads; // a multiple of G
  for (int64_t t = (int64_t)blockIdx.x * kThreads + threadIdx.x; t < chunks; t += step) {
    uint4 d = dy[t];
    if (y) {
      float f[8];
      const uint4 yy = y[t];
      unpack8(yy, f);
      uint32_t *w = &d.x;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        w[i] &= (f[2 * i] > 0.0f ? 0xffffu : 0u) | (f[2 * i + 1] > 0.0f ? 0xffff0000u : 0u);
      dpre[t] = d;
    }
    float f[8];
    unpack8(d, f);
#pragma unroll
    for (int i = 0; i < 8; ++i)
      s[i] += f[i];
  }
  block_sums<8, G>(s, lds);
  if (threadIdx.x < G)
#pragma unroll
    for (int i = 0; i < 8; ++i)
      part[(int64_t)blockIdx.x * C + threadIdx.x * 8 + i] = s[i];
}

// the 1x1 output layer on kHeadC channels: y[p][o] = b[o] + sum_c x[p][c] w[c][o],
// float32 from bfloat16 activations, four threads a pixel
constexpr int kHeadC = 32, kHeadG = kHeadC / 8;

template <int O>
__global__ void __launch_bounds__(kThreads)
head_fwd(int64_t pixels, const uint4 *__restrict__ x, const float *__restrict__ w,
         const float *__restrict__ b, float *__restrict__ y) {
  const int64_t t = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  const int c = 8 * (threadIdx.x % kHeadG);
  const int64_t p = t / kHeadG;
  float f[8] = {};
  if (p < pixels)
    unpack8(x[t], f);
#pragma unroll
  for (int o = 0; o < O; ++o) {
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      s += f[i] * w[(c + i) * O + o];
#pragma unroll
    for (int m = 1; m < kHeadG; m <<= 1)
      s += __shfl_xor(s, m);
    if (p < pixels && c == 0)
      y[p * O + o] = s + b[o];
  }
}

// its gradients in one pass: dx = dy w^T in bfloat16, and the sums x^T dy and
// dy over the pixels as slices (kHeadC O values of dw, then O of db)
template <int O>
__global__ void __launch_bounds__(kThreads)
head_bwd(int64_t pixels, const uint4 *__restrict__ x, const float *__restrict__ w,
         const float *__restrict__ dy, uint4 *__restrict__ dx, float *__restrict__ part) {
  __shared__ float lds[kThreads / 64 * 9 * O * kHeadG];
  const int c = 8 * (threadIdx.x % kHeadG);
  float ws[8 * O], s[9 * O] = {};
#pragma unroll
  for (int i = 0; i < 8 * O; ++i)
    ws[i] = w[c * O + i];
  const int64_t step = (int64_t)gridDim.x * kThreads;
  for (int64_t t = (int64_t)blockIdx.x * kThreads + threadIdx.x; t / kHeadG < pixels; t += step) {
    float f[8], d[O];
#pragma unroll
    for (int o = 0; o < O; ++o)
      d[o] = dy[t / kHeadG * O + o];
    unpack8(x[t], f);
    float g[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      g[i] = 0.0f;
#pragma unroll
      for (int o = 0; o < O; ++o) {
        g[i] += d[o] * ws[i * O + o];
        s[i * O + o] += f[i] * d[o];
      }
    }
#pragma unroll
    for (int o = 0; o < O; ++o)
      s[8 * O + o] += d[o];
    if (dx)
      dx[t] = uint4{pack_bf16(g[0], g[1]), pack_bf16(g[2], g[3]), pack_bf16(g[4], g[5]),
                    pack_bf16(g[6], g[7])};
  }
  block_sums<9 * O, kHeadG>(s, lds);
  if (threadIdx.x >= kHeadG)
    return;
  float *out = part + (int64_t)blockIdx.x * (kHeadC + 1) * O;
#pragma unroll
  for (int i = 0; i < 8 * O; ++i)
    out[c * O + i] = s[i];
  if (c == 0)
#pragma unroll
    for (int o = 0; o < O; ++o)
      out[kHeadC * O + o] = s[8 * O + o];
}

template <int CI, int CO>
void launch_wgrad(const cw_conv3x3_args &a, const Image &im, int slices, hipStream_t s) {
  const int strips = (a.w + kWStrip - 1) / kWStrip;
  const int64_t rows = (int64_t)a.n * strips * a.h;
  const int run = (int)((rows + slices - 1) / slices);
  hipLaunchKernelGGL((conv3x3_wgrad<CI, CO>), dim3((a.cin + CI - 1) / CI * (a.cout / CO), slices),
                     dim3(kThreads), 0, s, im, strips, a.cin, a.cout, (const uint4 *)a.x,
                     (const uint4 *)a.dy, run, (float *)a.workspace);
}

template <int BN>
void launch_wgrad_flat(const cw_conv3x3_args &a, const Image &im, int slices, hipStream_t s) {
  const int64_t run = (im.pixels + slices - 1) / slices;
  hipLaunchKernelGGL(conv3x3_wgrad_flat<BN>, dim3((9 * a.cin + 127) / 128, slices), dim3(kThreads),
                     0, s, im, a.cin, (const uint4 *)a.x, (const uint4 *)a.dy, run,
                     (float *)a.workspace);
}

// Whether the flat kernel takes the weight gradient: where the strips' columns
// and each march's two rows more than it sums leave fewer than a few true
// pixels in a hundred (both took the same time at 32 channels at 0.016, 20000
// images of 2 x 2: 157 and 152 us; at 64 at 0.05, 16384 of 4 x 4: 297 and 336;
// at 128 at 0.08, 60000 x 4: 681 and 880, 40000 x 6: 677 and 612), and where
// the layer has so few pixels that the strips' blocks are too few and their
// marches too short (one image of 16 x 16 at 64 channels 10.5 and 22 us; at 64
// channels both took 21 us at about 1500 pixels, at 128 at 800).
bool flat_wgrad(const cw_conv3x3_args &a) {
  const int most = a.cin > a.cout ? a.cin : a.cout;
  const double pixels = (double)a.n * a.h * a.w;
  const double least = most <= 32 ? 0.016 : most <= 64 ? 0.05 : 0.08;
  const double marched = (double)a.n * (a.h + 2) * ((a.w + kWStrip - 1) / kWStrip * kWStrip);
  return pixels * most < 1e5 || pixels < least * marched;
}

// a pass sums fewer slices than it was given room for where a slice would be
// shorter than six rows of a strip, or 2048 pixels (sixteen always: a small
// layer's blocks)
int launch_wgrad(const cw_conv3x3_args &a, const Image &im, hipStream_t s) {
  if (flat_wgrad(a)) {
    int64_t slices = im.pixels / 2048;
    slices = slices < 16 ? 16 : slices > 256 ? 256 : slices;
    slices = slices < a.splits ? slices : a.splits;
    switch (a.cout) {
    case 32: launch_wgrad_flat<32>(a, im, (int)slices, s); break;
    case 64: launch_wgrad_flat<64>(a, im, (int)slices, s); break;
    default: launch_wgrad_flat<128>(a, im, (int)slices, s); break;
    }
    return (int)slices;
  }
  int64_t slices = (int64_t)a.n * a.h * ((a.w + kWStrip - 1) / kWStrip) / 6;
  slices = slices < 1 ? 1 : slices < a.splits ? slices : a.splits;
  if (a.cin <= 32)
    a.cout == 32 ? launch_wgrad<32, 32>(a, im, (int)slices, s)
                 : launch_wgrad<32, 64>(a, im, (int)slices, s);
  else
    a.cout == 32 ? launch_wgrad<64, 32>(a, im, (int)slices, s)
                 : launch_wgrad<64, 64>(a, im, (int)slices, s);
  return (int)slices;
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

// the activations are read and written 16 bytes a thread
bool aligned(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

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
  switch (a->cout) {
  case 32: launch_fwd<32>(*a, im, s); break;
  case 64: launch_fwd<64>(*a, im, s); break;
  default: launch_fwd<128>(*a, im, s); break;
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
  const auto s = (hipStream_t)stream;
  const int slices = launch_wgrad(*a, im, s);
  if (int e = hip_status("conv3x3_wgrad"))
    return e;
  const int total = 9 * a->cin * a->cout;
  launch_slices_sum(total, slices, a->workspace, a->dweight, s);
  return hip_status("slices_sum");
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

int cw_relu_bias_grad(int64_t pixels, int32_t channels, const void *dy, const void *y, void *dpre,
                      void *workspace, int32_t slices, void *dbias, void *stream) {
  if (pixels < 1 || !dy || !workspace || !dbias || slices < 1)
    return fail("the bias gradient needs pixels, dy, a workspace, slices and dbias");
  if (channels != 32 && channels != 64 && channels != 128)
    return fail("channels must be 32, 64 or 128");
  if (y && !dpre)
    return fail("a masked gradient needs dpre");
  if (!aligned(dy) || !aligned(y) || (y && !aligned(dpre)))
    return fail("dy, y and dpre must be 16-byte aligned");
  const int64_t chunks = pixels * (channels / 8);
  const auto s = (hipStream_t)stream;
  const uint4 *d = (const uint4 *)dy, *yy = (const uint4 *)y;
  uint4 *out = (uint4 *)dpre;
  float *part = (float *)workspace;
  const dim3 grid(slices), block(kThreads);
  switch (channels) {
  case 32: hipLaunchKernelGGL(relu_bias_grad<32>, grid, block, 0, s, chunks, d, yy, out, part); break;
  case 64: hipLaunchKernelGGL(relu_bias_grad<64>, grid, block, 0, s, chunks, d, yy, out, part); break;
  default: hipLaunchKernelGGL(relu_bias_grad<128>, grid, block, 0, s, chunks, d, yy, out, part); break;
  }
  launch_slices_sum(channels, slices, workspace, dbias, s);
  return hip_status("relu_bias_grad");
}

int cw_head_fwd(int64_t pixels, int32_t outputs, const void *x, const void *w, const void *b, void *y,
                void *stream) {
  if (pixels < 1 || !x || !w || !b || !y)
    return fail("the output layer needs pixels, x, w, b and y");
  if (!aligned(x))
    return fail("x must be 16-byte aligned");
  const int64_t threads = pixels * kHeadG;
  const dim3 grid((int)((threads + kThreads - 1) / kThreads)), block(kThreads);
  const auto s = (hipStream_t)stream;
  const uint4 *xx = (const uint4 *)x;
  const float *ww = (const float *)w, *bb = (const float *)b;
  float *yy = (float *)y;
  switch (outputs) {
  case 1: hipLaunchKernelGGL(head_fwd<1>, grid, block, 0, s, pixels, xx, ww, bb, yy); break;
  case 2: hipLaunchKernelGGL(head_fwd<2>, grid, block, 0, s, pixels, xx, ww, bb, yy); break;
  case 3: hipLaunchKernelGGL(head_fwd<3>, grid, block, 0, s, pixels, xx, ww, bb, yy); break;
  case 4: hipLaunchKernelGGL(head_fwd<4>, grid, block, 0, s, pixels, xx, ww, bb, yy); break;
  default: return fail("the output layer is built for 1 to 4 outputs");
  }
  return hip_status("head_fwd");
}

int cw_head_bwd(int64_t pixels, int32_t outputs, const void *x, const void *w, const void *dy, void *dx,
                void *workspace, int32_t slices, void *dwb, void *stream) {
  if (pixels < 1 || !x || !w || !dy || !workspace || !dwb || slices < 1)
    return fail("the output layer's backward needs pixels, x, w, dy, a workspace, slices and dwb");
  if (!aligned(x) || !aligned(dx))
    return fail("x and dx must be 16-byte aligned");
  const dim3 grid(slices), block(kThreads);
  const auto s = (hipStream_t)stream;
  const uint4 *xx = (const uint4 *)x;
  const float *ww = (const float *)w, *dd = (const float *)dy;
  uint4 *out = (uint4 *)dx;
  float *part = (float *)workspace;
  switch (outputs) {
  case 1: hipLaunchKernelGGL(head_bwd<1>, grid, block, 0, s, pixels, xx, ww, dd, out, part); break;
  case 2: hipLaunchKernelGGL(head_bwd<2>, grid, block, 0, s, pixels, xx, ww, dd, out, part); break;
  case 3: hipLaunchKernelGGL(head_bwd<3>, grid, block, 0, s, pixels, xx, ww, dd, out, part); break;
  case 4: hipLaunchKernelGGL(head_bwd<4>, grid, block, 0, s, pixels, xx, ww, dd, out, part); break;
  default: return fail("the output layer is built for 1 to 4 outputs");
  }
  launch_slices_sum((kHeadC + 1) * outputs, slices, workspace, dwb, s);
  return hip_status("head_bwd");
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
