// Learned warm start: a small BF16 U-Net that maps a (template, reference) pair to a displacement
// field, with its forward pass, backward pass and Adam update written for gfx950 (no counterpart in
// the reference; the gradient flow then refines its prediction).
//
// Network (S scales, base width C): per scale two 3x3 convolutions with ReLU (C, 2C, 4C, ... channels),
// 2x2 average pooling between encoder scales, nearest-neighbour upsampling whose output is
// concatenated with the encoder's skip tensor before the decoder's two convolutions, and a 1x1 head to
// 2 channels (the displacement in pixels). The input's 2 channels are padded to 16.
//
// Layout: activations NHWC in BF16 (channels innermost, so a convolution's reduction dimension is
// contiguous); gradients of activations NHWC in FP32; weights FP32 masters [9][Cout][Cin] with BF16
// copies packed in MFMA operand order for the forward and for the data gradient.
// A 3x3 convolution is an implicit GEMM on MFMA (v_mfma_f32_32x32x16_bf16): rows = output channels
// (weights), columns = 32 consecutive pixels, reduction = 9 taps x input channels in steps of 16;
// FP32 accumulation, bias and ReLU fused into the epilogue. The upsampling and the concatenation are
// not materialised: the convolution reads channel c < C1 from the coarse tensor at (y/2, x/2) and the
// rest from the skip tensor. The data gradient is the same kernel over the pre-activation gradient with
// flipped taps and transposed weights; its output stays where it is written, and the next layer's ReLU
// gradient gathers it from there (summing over upsampled pixels, adding the pooled tensor's share). The
// weight gradient reduces over ranges of pixels on MFMA and sums the ranges in a fixed order
// (deterministic).
#include "ms_gpu.h"

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <random>
#include <string>
#include <type_traits>
#include <vector>

namespace msg {
int set_error(int code, const std::string &m);  // the calling thread's msg_last_error() (ms_gpu.hip)
}

namespace {

int ufail(int code, const std::string &m) { return msg::set_error(code, "msg_unet: " + m); }
#define UHIP(x)                                                                                    \
  do {                                                                                             \
    hipError_t e_ = (x);                                                                           \
    if (e_ != hipSuccess) return ufail(MSG_ERR_HIP, std::string(#x) + ": " + hipGetErrorString(e_)); \
  } while (0)
#define UCHK(x)                  \
  do {                           \
    int r_ = (x);                \
    if (r_ != MSG_OK) return r_; \
  } while (0)

typedef unsigned short bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// FP32 -> BF16, round to nearest even (NaN stays NaN)
__host__ __device__ inline bf16 f2bf(float f) {
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_bit_cast(bf16, (__bf16)f);  // one conversion instruction
#endif
  uint32_t u;
  memcpy(&u, &f, 4);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (bf16)((u >> 16) | 0x40);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (bf16)(u >> 16);
}
__host__ __device__ inline float bf2f(bf16 h) {
  const uint32_t u = (uint32_t)h << 16;
  float f;
  memcpy(&f, &u, 4);
  return f;
}
__device__ inline bf16x8 as_bf16x8(u16x8 v) { return __builtin_bit_cast(bf16x8, v); }

inline int cdivu(long a, long b) { return (int)((a + b - 1) / b); }

// Workgroup ids in an order that gives each of the 8 XCDs a contiguous range (ids are dispatched
// round-robin over them): neighbouring tiles and the channel blocks of one tile share an L2.
__device__ inline int xcd_order(int wg, int total) {
  const int xcd = wg % 8, base = total / 8, extra = total % 8;
  return xcd * base + (xcd < extra ? xcd : extra) + wg / 8;
}

// The input of a convolution at H x W: channels [0, c1) from x1 (H/2 x W/2 and upsampled when up1),
// channels [c1, c1 + c2) from x2 (H x W). c1 and c2 are multiples of 16 (c2 may be 0).
struct ConvIn {
  const bf16 *x1;
  const bf16 *x2;
  int c1, c2, up1;
};

// 16 bytes per lane from global memory straight to LDS, no registers in between: lane l's to dst + 16 l, dst aligned
// (dst is the same for the whole wave; inactive lanes write nothing). Complete after lds_loads_done.
__device__ __forceinline__ void load_to_lds(const bf16 *src, bf16 *dst) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)src,
                                   (__attribute__((address_space(3))) void *)dst, 16, 0, 0);
}
__device__ __forceinline__ void lds_loads_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// what pixels outside the image read
__device__ __align__(16) const bf16 conv_zeros[8] = {0, 0, 0, 0, 0, 0, 0, 0};

// Permutation of a staged pixel's 16-byte slots (8 channels each) by its column, so that 8 or 16 lanes
// reading the same channels of consecutive columns hit distinct banks.
template <int SEG>
__device__ __forceinline__ int conv_perm(int col) {
  if constexpr (SEG % 16 == 0)
    return col & 15;
  else if constexpr (SEG % 8 == 0)
    return ((col >> 1) & 3) | (((col ^ (col >> 3)) & 1) << 2);
  else if constexpr (SEG % 4 == 0)
    return ((col >> 2) & 1) | ((((col >> 1) ^ (col >> 3)) & 1) << 1);
  else
    return ((col >> 2) ^ (col >> 3)) & 1;
}

// Stages rows of 34 pixels (32 with a 1-pixel halo) of a convolution's input in LDS, NB blocks of SEG
// slots per pixel ([block][pixel][slot]), by TH threads. What a thread loads differs between rows only by the
// row's start, so the divisions, bounds and channel arithmetic are done once per tile, not per load (they
// were most of a tile's instructions).
template <int SEG, int NB, int TH, bool PERMUTE>
struct RowStager {
  static constexpr int HC = 34, PIECES = NB * HC * SEG, PER = (PIECES + TH - 1) / TH;
  int off[PER];          // offset within the row of the source
  unsigned second = 0, ok = 0;  // bit per load: from x2; inside the image's columns and the channels
  __device__ __forceinline__ RowStager(const ConvIn &in, int c0, int x0, int W) {
    const int cin = in.c1 + in.c2;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int i = (int)threadIdx.x + TH * j, blk = i / (HC * SEG), r = i - blk * (HC * SEG);
      const int col = r / SEG, slot = r % SEG, seg = PERMUTE ? slot ^ conv_perm<SEG>(col) : slot;
      const int c = c0 + (blk * SEG + seg) * 8, gx = x0 + col - 1;
      const bool s2 = c >= in.c1;
      off[j] = s2 ? gx * in.c2 + c - in.c1 : (in.up1 ? gx >> 1 : gx) * in.c1 + c;
      second |= (unsigned)s2 << j;
      ok |= (unsigned)(i < PIECES && gx >= 0 && gx < W && c < cin) << j;
    }
  }
  // row gy of image b to dst (wave0: this wave's first thread)
  __device__ __forceinline__ void row(const ConvIn &in, int b, int gy, int H, int W, bf16 *dst, int wave0) const {
    const bool inside = gy >= 0 && gy < H;
    const bf16 *r1 = in.x1 + (long)(in.up1 ? (b * (H >> 1) + (gy >> 1)) * (W >> 1) : (b * H + gy) * W) * in.c1;
    const bf16 *r2 = in.x2 + (long)(b * H + gy) * W * in.c2;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const bf16 *src = ((second >> j) & 1 ? r2 : r1) + off[j];
      if (!(inside && ((ok >> j) & 1))) src = conv_zeros;
      if ((int)threadIdx.x + TH * j < PIECES) load_to_lds(src, dst + (wave0 + TH * j) * 8);
    }
  }
};

// ------------------------------------------------------------------------------------------------
// 3x3 convolution, forward (or data gradient, with its own packed weights):
// y[p][co] = act(bias[co] + sum_tap sum_ci w[tap][co][ci] in[p + off(tap)][ci]),
// every sum over the taps in order and, within a tap, over 16 input channels per instruction in order:
// both kernels below and any tile give the same bits. (Activations are rounded to BF16 after every layer,
// so another order of these FP32 sums would differ in the network's output as much as its rounding does.)
//
// Weights are packed in operand order, [block of 32 output channels][tap][16 input channels][lane][8]:
// a fragment is one contiguous kilobyte, read by a wave in one instruction.
// ------------------------------------------------------------------------------------------------
__host__ __device__ inline long packed_weight(int row, int k, int tap, int ktotal) {
  return ((((long)(row >> 5) * 9 + tap) * (ktotal / 16) + k / 16) * 64 + (row & 31) + 32 * ((k >> 3) & 1)) * 8 + (k & 7);
}

// acc + bias, ReLU, stored: lane (pixel column, half kh); a tile's rows are the output channels
// (r/4)*8 + kh*4 + r%4 from co0
template <typename OutT>
__device__ __forceinline__ void conv_store(const f32x16 &acc, const float *__restrict__ bias, int relu, int kh, int co0,
                                           OutT *__restrict__ dst) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int co = j * 8 + kh * 4;
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[e] = acc[j * 4 + e] + (bias ? bias[co0 + co + e] : 0.f);
      if (relu) v[e] = v[e] > 0.f ? v[e] : 0.f;
    }
    if constexpr (sizeof(OutT) == 2)
      *(u16x4 *)(dst + co) = u16x4{f2bf(v[0]), f2bf(v[1]), f2bf(v[2]), f2bf(v[3])};
    else
      *(f32x4 *)(dst + co) = f32x4{v[0], v[1], v[2], v[3]};
  }
}

// Input tile in LDS. A workgroup of WM x WR waves computes 32 columns x WR NP rows of one image and
// 32 NT WM output channels; a wave NT x NP MFMA tiles (rows: channels, columns: the 32 pixels of one row).
// The tile's pixels with a 1-pixel halo and all CIN input channels are staged once; the weights too where
// they are small (CIN <= 32), else a wave streams its fragments from L2, a group of steps ahead. One step (16
// channels of one tap) is NT weight and NP pixel fragments of 1 KB for NT NP instructions of 32 cycles: with
// the pixels from LDS (128 B per cycle) and the weights from L1 (64 B per cycle), four waves keep both
// below the matrix cores' rate from NT = NP = 2 on. The 14 convolutions of a forward pass of 8 pairs of
// 256^2 (4 scales, 32 channels), operands through the caches as in k_conv3x3: 1049 us, 150 TFLOP/s; so:
// 390 us, 430 TFLOP/s. What is left is a workgroup's staging, which only other workgroups overlap (one or
// two more fit a compute unit's LDS), and at 32 output channels, NT = 1, 0.8 to 1 instruction per LDS read (2 beyond):
// the matrix cores are busy 7 to 23 % of a launch, no bank conflicts.
template <int CIN, int WM, int WR, int NT, int NP, typename OutT>
__global__ void __launch_bounds__(64 * WM * WR)
k_conv3x3_tile(ConvIn in, const bf16 *__restrict__ w, const float *__restrict__ bias, OutT *__restrict__ y, int H,
               int W, int cout, int relu) {
  constexpr int TH = 64 * WM * WR, SEG = CIN / 8, NKS = CIN / 16, ROWS = WR * NP, HC = 34;
  constexpr int NLD = (ROWS + 2) * HC * SEG, WF = 9 * NKS * 512;  // pieces of the tile; values of a weight block
  constexpr bool ALDS = CIN <= 32;
  constexpr int PERM = SEG % 16 == 0 ? 15 : SEG % 8 == 0 ? 7 : SEG % 4 == 0 ? 3 : 1;  // slot bits permuted
  constexpr int G = NKS <= 4 || NKS == 6 ? NKS : 4, NG = 9 * NKS / G;  // steps per group, groups
  __shared__ alignas(16) bf16 sx[NLD * 8 + (ALDS ? WM * NT * WF : 2 * TH)];  // pixels; weights or what touching them returns
  bf16 *sw = sx + NLD * 8;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wm = wave % WM, wr = wave / WM;
  const int wave0 = __builtin_amdgcn_readfirstlane(wave * 64);
  const int tilesx = W / 32, tilesy = H / ROWS, ncb = cout / (32 * NT * WM);
  int id = xcd_order(blockIdx.x, gridDim.x);
  const int cb = (id % ncb) * (WM * NT);
  id /= ncb;
  const int x0 = (id % tilesx) * 32;
  id /= tilesx;
  const int y0 = (id % tilesy) * ROWS, b = id / tilesy;
  const int px = lane & 31, kh = lane >> 5;

  {
    const RowStager<SEG, 1, TH, true> st(in, 0, x0, W);
#pragma unroll 2
    for (int r = 0; r < ROWS + 2; ++r) st.row(in, b, y0 + r - 1, H, W, sx + r * HC * CIN, wave0);
  }
  if constexpr (ALDS) {
    constexpr int NW = WM * NT * WF / 8;
#pragma unroll
    for (int k = 0; k < (NW + TH - 1) / TH; ++k) {
      const int i = tid + TH * k;
      if (i < NW) load_to_lds(w + (long)cb * WF + i * 8, sw + (wave0 + TH * k) * 8);
    }
  }
  if constexpr (!ALDS) {
    // every line of the weights this workgroup will stream, touched now: the caches start a kernel cold, and
    // a miss per group of steps, one after another in every workgroup, costs more than the arithmetic
    constexpr int NLINE = WM * NT * WF * 2 / 128;
    const bf16 *wb = w + (long)cb * WF;
#pragma unroll 4
    for (int k = 0; k < (NLINE + TH - 1) / TH; ++k) {
      const int i = tid + TH * k;
      if (i < NLINE)
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(wb + i * 64),
                                         (__attribute__((address_space(3))) void *)(sw + wave0 * 2), 4, 0, 0);
    }
  }
  const bf16 *ap = (ALDS ? sw + wm * NT * WF : w + ((long)cb + wm * NT) * WF) + lane * 8;
  // weight fragments of group g (the last group's next is itself: loaded, not used)
  auto load_a = [&](int g, u16x8(&v)[G][NT]) {
#pragma unroll
    for (int j = 0; j < G; ++j)
#pragma unroll
      for (int t = 0; t < NT; ++t) v[j][t] = *(const u16x8 *)(ap + t * WF + (g * G + j) * 512);
  };
  u16x8 a[2][G][NT], bv[3][NP];
  if constexpr (!ALDS) load_a(0, a[0]);
  lds_loads_done();
  __syncthreads();
  if constexpr (ALDS) load_a(0, a[0]);

  // this lane's pixel of the wave's first halo row for the tap of group g, with its slot permutation and the
  // group's first channels
  auto group_at = [&](int g) {
    const int tap = g / (NKS / G), seg = 2 * G * (g % (NKS / G)), dy = tap / 3, col = px + tap % 3;
    const int o = ((wr * NP + dy) * HC + col) * CIN + (kh ^ conv_perm<SEG>(col)) * 8;
    return (o ^ ((seg & PERM) * 8)) + (seg & ~PERM) * 8;
  };
  // pixel fragments of step j of the group at o (a group's slots differ from its first's by 2 j in bits
  // below the next group's)
  auto load_b = [&](int o, int j, u16x8(&v)[NP]) {
    const bf16 *p = sx + (o ^ ((2 * j & PERM) * 8)) + (2 * j & ~PERM) * 8;
#pragma unroll
    for (int q = 0; q < NP; ++q) v[q] = *(const u16x8 *)(p + q * HC * CIN);
  };
  f32x16 acc[NT][NP];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int q = 0; q < NP; ++q)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[t][q][r] = 0.f;
  // pixel fragments two steps ahead
  int o = group_at(0), on = group_at(NG > 1 ? 1 : 0);
  load_b(o, 0, bv[0]);
  load_b(G > 1 ? o : on, G > 1 ? 1 : 0, bv[1]);
  for (int g = 0; g < NG; ++g) {
    const int gn = g + 1 < NG ? g + 1 : g, o2 = group_at(g + 2 < NG ? g + 2 : NG - 1);
    load_a(gn, a[1]);
#pragma unroll
    for (int j = 0; j < G; ++j) {
      constexpr int P = G > 1 ? 2 : 1;
      if constexpr (G > 1)
        load_b(j + P < G ? o : on, j + P < G ? j + P : j + P - G, bv[2]);
      else
        load_b(o2, 0, bv[2]);
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int q = 0; q < NP; ++q)
          acc[t][q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(a[0][j][t]), as_bf16x8(bv[0][q]), acc[t][q], 0, 0, 0);
#pragma unroll
      for (int q = 0; q < NP; ++q) {
        bv[0][q] = bv[1][q];
        bv[1][q] = bv[2][q];
      }
    }
#pragma unroll
    for (int j = 0; j < G; ++j)
#pragma unroll
      for (int t = 0; t < NT; ++t) a[0][j][t] = a[1][j][t];
    o = on;
    on = o2;
  }
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      const int co0 = (cb + wm * NT + t) * 32;
      conv_store(acc[t][q], bias, relu, kh, co0, y + ((long)(b * H + y0 + wr * NP + q) * W + x0 + px) * cout + co0);
    }
}

// Any multiples of 64 input and output channels, the input read through the caches: for the networks
// whose input tile does not fit LDS. One wave: 64 output channels and 32 NP consecutive pixels of one
// image row (W % (32 NP) == 0); four waves per workgroup along the pixels. Wide layers are small images with few
// waves, so what bounds it is the way to L2: the operands of 4 steps (of 16 channels) are in flight while the 4
// steps before them multiply. A forward of 4 scales from 256 channels at 256^2 (512 to 2048 channels here): 6.4 ms
// with a step's loads waited for by the step, 6.8 ms so from packed weights (a new line each step), 3.1 ms now (4
// images: 23.9, 15.9, 10.7 ms; 13.5 ms at one wave per SIMD, which the registers of four tiles would take unbounded).
template <int NP, typename OutT>
__global__ void __launch_bounds__(256, 2)
k_conv3x3(ConvIn in, const bf16 *__restrict__ w, const float *__restrict__ bias, OutT *__restrict__ y, int B, int H,
          int W, int cout, int relu) {
  constexpr int NT = 2;  // tiles of 32 output channels
  const int cin = in.c1 + in.c2;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long M = (long)B * H * W;
  const long m0 = ((long)blockIdx.x * 4 + wave) * 32 * NP;
  if (m0 >= M) return;  // whole waves only (M % (32 NP) == 0)
  const int n0 = blockIdx.y * 32 * NT;
  const int px = lane & 31, kh = lane >> 5;
  // the NP tiles lie in one image row: same row and batch, x advancing by 32
  const int x0 = (int)((m0 + px) % W);
  const long t0 = (m0 + px) / W;
  const int yy = (int)(t0 % H), b = (int)(t0 / H);
  f32x16 acc[NT][NP];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int q = 0; q < NP; ++q)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[t][q][r] = 0.f;
  const int Hh = H >> 1, Wh = W >> 1;
  constexpr int U = 4;                          // steps per group
  const int ng = cin / (16 * U), total = 9 * ng;  // groups of a tap, of all
  const bf16 *wp = w + packed_weight(n0, 0, 0, cin) + lane * 8;
  const long wblk = 9L * cin * 32;  // values of 32 output channels
  auto load = [&](int i, u16x8(&a)[U][NT], u16x8(&v)[U][NP]) {
    const int tap = i / ng, c0 = (i - tap * ng) * 16 * U, sy = yy + tap / 3 - 1;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int j = 0; j < U; ++j) a[j][t] = *(const u16x8 *)(wp + t * wblk + ((long)i * U + j) * 512);
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      const int sx = x0 + 32 * q + tap % 3 - 1;
      const bool inb = sy >= 0 && sy < H && sx >= 0 && sx < W;
      const long o1 = (in.up1 ? ((long)b * Hh + (sy >> 1)) * Wh + (sx >> 1) : ((long)b * H + sy) * W + sx) * in.c1;
      const long o2 = (((long)b * H + sy) * W + sx) * in.c2 - in.c1;
#pragma unroll
      for (int j = 0; j < U; ++j) {
        const int c = c0 + 16 * j + 8 * kh;
        const bf16 *p = c < in.c1 ? in.x1 + o1 + c : in.x2 + o2 + c;
        v[j][q] = *(const u16x8 *)(inb ? p : conv_zeros);
      }
    }
  };
  auto multiply = [&](const u16x8(&a)[U][NT], const u16x8(&v)[U][NP]) {
#pragma unroll
    for (int j = 0; j < U; ++j)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int q = 0; q < NP; ++q)
          acc[t][q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(a[j][t]), as_bf16x8(v[j][q]), acc[t][q], 0, 0, 0);
  };
  u16x8 a0[U][NT], v0[U][NP], a1[U][NT], v1[U][NP];
  load(0, a0, v0);
  for (int i = 0; i < total; i += 2) {  // (past the last group: that one again, unused)
    load(i + 1 < total ? i + 1 : total - 1, a1, v1);
    multiply(a0, v0);
    load(i + 2 < total ? i + 2 : total - 1, a0, v0);
    if (i + 1 < total) multiply(a1, v1);
  }
#pragma unroll
  for (int q = 0; q < NP; ++q)
#pragma unroll
    for (int t = 0; t < NT; ++t)
      conv_store(acc[t][q], bias, relu, kh, n0 + 32 * t, y + (m0 + 32 * q + px) * cout + n0 + 32 * t);
}

// ------------------------------------------------------------------------------------------------
// Weight gradient of a 3x3 convolution: part[split][tap][co][ci] = sum over the split's pixels of
// dz[p][co] in[p + off(tap)][ci].
//
// A workgroup takes 32 WM output x 32 WN input channels, all 9 taps, and a range of spatial tiles of R rows
// x 32 columns; its four waves are WM x WN channel blocks times KS = 4 / (WM WN) shares of a tile's rows,
// summed at the end in a fixed order. Per tile, dz and the input with a 1-pixel halo go to LDS as
// [row][channel block][pixel][32]. The reduction runs over pixels while both operands are channel-innermost:
// the transposing LDS read (ds_read_b64_tr_b16) gives a lane 4 consecutive pixels of its channel. A wave
// walks the input's rows: the three fragments of a row (one per column offset) meet the dz fragments of
// the three rows around it, which stay in registers, so 9 instructions take 4 KB from LDS (44 % of its
// bandwidth at full MFMA rate). The 14 layers of a training step of 8 pairs of 256^2: 1.22 ms (with each
// wave staging and gathering 16-bit operands by itself, 143 TFLOP/s) -> 0.41 ms.
// ------------------------------------------------------------------------------------------------
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));

// 8 pixels (from p, 32 values apart) of one channel per lane: the MFMA operand of 16 pixels x 32 channels
// whose lane addresses p holds (rows 4 apart for the second half)
__device__ __forceinline__ bf16x8 read_transposed(const bf16 *p) {
  typedef __attribute__((address_space(3))) s16x4 lds4;
  const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4 *)p);
  const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4 *)(p + 4 * 32));
  return __builtin_bit_cast(bf16x8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

template <int WM, int WN, int R>
__global__ void __launch_bounds__(256, 2)
k_conv3x3_wgrad(ConvIn in, const bf16 *__restrict__ dz, float *__restrict__ part, int B, int H, int W, int cout,
                int nsplit) {
  constexpr int KS = 4 / (WM * WN), RW = R / KS, HC = 34;
  constexpr int ZPIX = R * 32, XPIX = (R + 2) * HC;
  __shared__ alignas(16) bf16 lds[(ZPIX * WM + XPIX * WN) * 32];
  static_assert(sizeof(lds) >= 3 * 16 * 64 * sizeof(float), "the final sum over the row shares reuses the tile");
  bf16 *sz = lds, *sx = lds + ZPIX * WM * 32;
  const int cin = in.c1 + in.c2;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wave0 = wave * 64;  // this wave's first piece
  const int wm = wave % WM, wn = (wave / WM) % WN, ks = wave / (WM * WN);
  const int ncob = cout / (32 * WM), ncib = (cin + 32 * WN - 1) / (32 * WN);
  int id = xcd_order(blockIdx.x, gridDim.x);
  const int co0 = (id % ncob) * 32 * WM;
  id /= ncob;
  const int ci0 = (id % ncib) * 32 * WN, split = id / ncib;
  const int tilesx = W / 32, tilesy = H / R, ntile = B * tilesy * tilesx;
  const int tbeg = (int)((long)ntile * split / nsplit), tend = (int)((long)ntile * (split + 1) / nsplit);
  // a sweep of the 256 threads stages 2 / WM rows of dz, WM x 32 pixels x 4 slots each
  const int zrow = tid / (WM * 128), zblk = tid / 128 % WM, zoff = (tid % 128 / 4) * cout + co0 + 32 * zblk + 8 * (tid & 3);
  // transposing reads: 16 lanes take 4 pixels x 16 channels; the wave's four groups two channel halves and
  // pixels 0..3 and 8..11 (read_transposed adds 4..7 and 12..15)
  const int g = lane >> 4, sl = lane & 15;
  const int loff = (8 * (g >> 1) + (sl >> 2)) * 32 + 16 * (g & 1) + 4 * (sl & 3);
  const bf16 *az = sz + (ks * RW * WM + wm) * 32 * 32 + loff, *bx = sx + (ks * RW * WN + wn) * HC * 32 + loff;

  f32x16 acc[9];
#pragma unroll
  for (int t = 0; t < 9; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[t][r] = 0.f;

  for (int tile = tbeg; tile < tend; ++tile) {
    const int x0 = (tile % tilesx) * 32, y0 = (tile / tilesx % tilesy) * R, b = tile / tilesx / tilesy;
    if (tile > tbeg) __syncthreads();  // the previous tile's reads are done
    {
      const RowStager<4, WN, 256, false> st(in, ci0, x0, W);
#pragma unroll 1
      for (int r = 0; r < R + 2; ++r) st.row(in, b, y0 + r - 1, H, W, sx + r * WN * HC * 32, wave0);
    }
    const bf16 *zp = dz + ((long)(b * H + y0 + zrow) * W + x0) * cout + zoff;
#pragma unroll
    for (int k = 0; k < R * WM / 2; ++k) load_to_lds(zp + (long)k * (2 / WM) * W * cout, sz + (wave0 + 256 * k) * 8);
    lds_loads_done();
    __syncthreads();
#pragma unroll 1
    for (int xs = 0; xs < 2; ++xs) {  // 16 columns at a time
      bf16x8 a[3];
#pragma unroll
      for (int r = 0; r < RW + 2; ++r) {  // the input's row r - 1 relative to this wave's rows of dz
        if (r < RW) a[r % 3] = read_transposed(az + (r * WM * 32 + 16 * xs) * 32);
#pragma unroll
        for (int dx = 0; dx < 3; ++dx) {
          const bf16x8 bv = read_transposed(bx + (r * WN * HC + 16 * xs + dx) * 32);
#pragma unroll
          for (int dy = 0; dy < 3; ++dy)
            if (r - dy >= 0 && r - dy < RW)
              acc[dy * 3 + dx] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[(r - dy) % 3], bv, acc[dy * 3 + dx], 0, 0, 0);
        }
      }
    }
  }

  // lane: input channel ci, rows (r/4)*8 + kh*4 + r%4 of the output channels; addresses as the wave's base
  // plus one offset per lane
  const int ci = ci0 + wn * 32 + (lane & 31);
  const unsigned lo = (unsigned)(lane >> 5) * 4u * (unsigned)cin + (unsigned)(lane & 31);
  float *red = (float *)lds;
  float *out = part + ((long)split * 9 * cout + co0 + wm * 32) * cin + ci0 + wn * 32;
#pragma unroll
  for (int t = 0; t < 9; ++t) {
    if constexpr (KS > 1) {
      __syncthreads();
      if (ks > 0) {
#pragma unroll
        for (int r = 0; r < 16; ++r) red[((wave - WM * WN) * 16 + r) * 64 + lane] = acc[t][r];
      }
      __syncthreads();
    }
    if (ks == 0) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float v = acc[t][r];
#pragma unroll
        for (int k = 1; k < KS; ++k) v += red[((wave + (k - 1) * WM * WN) * 16 + r) * 64 + lane];
        if (ci < cin) out[(long)((r >> 2) * 8 + (r & 3)) * cin + lo] = v;
      }
    }
    out += (long)cout * cin;
  }
}

// out[c] = sum over rows r of part[r * stride + off(c)], one workgroup per column c: each thread sums
// the rows r = t, t + 256, ... in order, then a fixed tree over the 256 threads (deterministic).
// Bias gradients (rows: the blocks of k_relu_grad; beyond 1024 channels a pixel's channels span several
// rows) and the head's partials use it.
__device__ __forceinline__ void col_sum(const float *__restrict__ part, int c, int nrows, long stride, int C,
                                        float *__restrict__ out, float (&s)[256]) {
  float a = 0.f;
  const int per = (int)((C + stride - 1) / stride);  // rows per pixel
#pragma unroll 4
  for (int r = (int)(c / stride) + per * (int)threadIdx.x; r < nrows; r += per * 256) a += part[(long)r * stride + c % stride];
  s[threadIdx.x] = a;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if ((int)threadIdx.x < k) s[threadIdx.x] += s[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[c] = s[0];
}
__global__ void __launch_bounds__(256)
k_col_sum(const float *__restrict__ part, int nrows, long stride, int C, float *__restrict__ out) {
  __shared__ float s[256];
  col_sum(part, blockIdx.x, nrows, stride, C, out, s);
}

// The sums of a layer's gradients. Weights, dw[i] = sum over chunks of part[chunk][i]: a workgroup takes 64
// elements, its 4 waves every fourth chunk in order (8 loads in flight each), their sums added in order. (One
// thread per element over all chunks: 188 us per training step of 8 pairs of 256^2; so: 111 us, of more partial
// sums.) The last C workgroups form the bias gradients (col_sum) in the shade of the others: as a launch per layer
// of their own they took 72 us of a step (gradient with its copy to the host: 2.29 -> 2.24 ms).
__global__ void __launch_bounds__(256)
k_layer_sums(const float *__restrict__ part, int nchunks, long n, float *__restrict__ dw,
             const float *__restrict__ bpart, int nrows, long stride, int C, float *__restrict__ db) {
  __shared__ float s[256];
  const int nwg = (int)((n + 63) / 64);
  if ((int)blockIdx.x >= nwg) {  // uniform
    col_sum(bpart, (int)blockIdx.x - nwg, nrows, stride, C, db, s);
    return;
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long i = (long)blockIdx.x * 64 + lane, j = i < n ? i : n - 1;
  float a = 0.f;
  for (int c0 = wave; c0 < nchunks; c0 += 32) {
    float v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int c = c0 + 4 * k;
      v[k] = part[(long)(c < nchunks ? c : nchunks - 1) * n + j];
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) a += c0 + 4 * k < nchunks ? v[k] : 0.f;
  }
  s[threadIdx.x] = a;
  __syncthreads();
  if (wave == 0 && i < n) dw[i] = ((s[lane] + s[64 + lane]) + s[128 + lane]) + s[192 + lane];
}

// Where the gradient of an activation comes from: its own buffer; or, for the upsampled source of a
// decoder convolution, the sums over 2 x 2 pixels of that convolution's input gradient; or, for a skip
// tensor, its share of that gradient plus a quarter of the pooled tensor's.
enum GradMode { GRAD_OWN = 0, GRAD_UP = 1, GRAD_SKIP = 2 };
struct GradSrc {
  const float *g;     // own buffer, or the decoder convolution's input gradient
  const float *pool;  // GRAD_SKIP: the pooled tensor's gradient
  int stride, off;    // values per pixel of g, first channel
};

// dz = bf16(gradient * [y > 0]) and per-block partial sums of it (in FP32) per channel for the bias
// gradient, the gradient gathered from where the convolutions above left it (no copies, sums or clears of
// it in memory). A thread takes 4 consecutive channels; a block covers RELU_CHUNKS x 1024 consecutive
// values with each thread keeping its channels (C divides 1024), or with C a multiple of 1024 one pixel's
// 1024 channels. Bound by HBM: 8 pairs of 256^2, 14 layers, with the copies and clears that this replaces:
// 0.95 ms -> 0.24 ms.
constexpr int RELU_CHUNKS = 8, RELU_BLOCK = 1024;
template <int MODE>
__global__ void __launch_bounds__(256)
k_relu_grad(GradSrc s, const bf16 *__restrict__ y, bf16 *__restrict__ dz, long n, int logc, int H, int W,
            float *__restrict__ bpart) {
  const int C = 1 << logc, chunks = C <= RELU_BLOCK ? RELU_CHUNKS : 1;
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int k = 0; k < chunks; ++k) {
    const long i = ((long)blockIdx.x * chunks + k) * RELU_BLOCK + 4 * threadIdx.x;
    if (i < n) {
      const int c = (int)(i & (C - 1));
      const long p = i >> logc;
      f32x4 d;
      if constexpr (MODE == GRAD_OWN) {
        d = *(const f32x4 *)(s.g + i);
      } else {
        const int x = (int)(p % W), yy = (int)(p / W % H), b = (int)(p / W / H);
        if constexpr (MODE == GRAD_UP) {
          const float *r0 = s.g + (((long)b * 2 * H + 2 * yy) * 2 * W + 2 * x) * s.stride + s.off + c;
          const float *r1 = r0 + (long)2 * W * s.stride;
          d = (*(const f32x4 *)r0 + *(const f32x4 *)(r0 + s.stride)) + (*(const f32x4 *)r1 + *(const f32x4 *)(r1 + s.stride));
        } else {
          const f32x4 q = *(const f32x4 *)(s.pool + (((long)b * (H / 2) + yy / 2) * (W / 2) + x / 2) * C + c);
          d = *(const f32x4 *)(s.g + p * s.stride + s.off + c) + 0.25f * q;
        }
      }
      const u16x4 a = *(const u16x4 *)(y + i);
      u16x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float u = bf2f(a[e]) > 0.f ? d[e] : 0.f;
        o[e] = f2bf(u);
        v[e] += u;
      }
      *(u16x4 *)(dz + i) = o;
    }
  }
  __shared__ float sum[RELU_BLOCK];
#pragma unroll
  for (int e = 0; e < 4; ++e) sum[4 * threadIdx.x + e] = v[e];
  __syncthreads();
  const int win = C < RELU_BLOCK ? C : RELU_BLOCK;
  for (int c = threadIdx.x; c < win; c += 256) {
    float a = 0.f;
    for (int k = c; k < RELU_BLOCK; k += win) a += sum[k];
    bpart[(long)blockIdx.x * win + c] = a;
  }
}

// 2x2 average pooling, NHWC bf16: y[b][yy][x][c] = mean of x[b][2yy..][2x..][c]; 8 channels per thread
__global__ void __launch_bounds__(256)
k_pool(const bf16 *__restrict__ x, bf16 *__restrict__ y, int B, int H, int W, int C) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int Ho = H / 2, Wo = W / 2, C8 = C / 8;
  if (i >= (long)B * Ho * Wo * C8) return;
  const int c = (int)(i % C8) * 8;
  long t = i / C8;
  const int xo = (int)(t % Wo);
  t /= Wo;
  const int yo = (int)(t % Ho), b = (int)(t / Ho);
  const bf16 *r0 = x + (((long)b * H + 2 * yo) * W + 2 * xo) * C + c, *r1 = r0 + (long)W * C;
  const u16x8 v00 = *(const u16x8 *)r0, v01 = *(const u16x8 *)(r0 + C), v10 = *(const u16x8 *)r1,
              v11 = *(const u16x8 *)(r1 + C);
  u16x8 o;
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = f2bf(0.25f * ((bf2f(v00[e]) + bf2f(v01[e])) + (bf2f(v10[e]) + bf2f(v11[e]))));
  *(u16x8 *)(y + i * 8) = o;
}

// Input pairs [B][2][H][W] FP32 (template, reference) -> NHWC bf16 with 16 channels (14 zero).
__global__ void __launch_bounds__(256)
k_pack_input(const float *__restrict__ in, bf16 *__restrict__ x, int B, int H, int W) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long hw = (long)H * W, n = (long)B * hw;
  if (i >= n) return;
  const long b = i / hw, q = i % hw;
  const u16x8 v = {f2bf(in[(b * 2) * hw + q]), f2bf(in[(b * 2 + 1) * hw + q]), 0, 0, 0, 0, 0, 0};
  *(u16x8 *)(x + i * 16) = v;
  *(u16x8 *)(x + i * 16 + 8) = (u16x8)0;
}

// 1x1 head to 2 channels: out[b][o][y][x] = bh[o] + sum_c wh[o][c] x[p][c] (FP32, planar); 8 channels a load
__global__ void __launch_bounds__(256)
k_head(const bf16 *__restrict__ x, const float *__restrict__ wh, const float *__restrict__ bh,
       float *__restrict__ out, int B, int H, int W, int C) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long hw = (long)H * W, n = (long)B * hw;
  if (p >= n) return;
  float a0 = bh[0], a1 = bh[1];
  const bf16 *src = x + p * C;
  for (int c0 = 0; c0 < C; c0 += 32) {  // C is a multiple of 32
    u16x8 u[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) u[k] = *(const u16x8 *)(src + c0 + 8 * k);
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float v = bf2f(u[k][e]);
        a0 += wh[c0 + 8 * k + e] * v;
        a1 += wh[C + c0 + 8 * k + e] * v;
      }
  }
  const long b = p / hw, q = p % hw;
  out[(b * 2) * hw + q] = a0;
  out[(b * 2 + 1) * hw + q] = a1;
}

// Loss 1/(2 n) sum (out - target)^2 (n = all output values) and its gradient d = (out - target) / n;
// per-block partial sums of the loss in FP64.
__global__ void k_mse(const float *__restrict__ out, const float *__restrict__ tgt, float *__restrict__ d, long n,
                      double *__restrict__ lpart) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  double l = 0;
  if (i < n) {
    const float e = out[i] - tgt[i];
    d[i] = e / (float)n;
    l = 0.5 * (double)e * (double)e / (double)n;
  }
  __shared__ double s[256];
  s[threadIdx.x] = l;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if ((int)threadIdx.x < k) s[threadIdx.x] += s[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) lpart[blockIdx.x] = s[0];
}

// Head backward over 256 pixels per workgroup: dx[p][c] = sum_o wh[o][c] dout[o][p], and per-block
// partials of dwh[o][c] = sum_p dout[o][p] x[p][c] (2C) and dbh[o] = sum_p dout[o][p] (2). Thread t
// takes channel t % C of the pixels t / C, t / C + 256 / C, ... (C divides 256), so the loads and
// stores of a wave are consecutive channels; the 256 / C partial sums of a channel are added in a
// fixed order.
constexpr int HEAD_CMAX = 256;
__global__ void __launch_bounds__(256)
k_head_grad(const bf16 *__restrict__ x, const float *__restrict__ wh, const float *__restrict__ dout,
            float *__restrict__ dx, int B, int H, int W, int C, float *__restrict__ part) {
  const long hw = (long)H * W, n = (long)B * hw;
  const long p0 = (long)blockIdx.x * 256;
  const int t = threadIdx.x, c = t % C, G = 256 / C, g = t / C;
  const float w0 = wh[c], w1 = wh[C + c];
  float a0 = 0.f, a1 = 0.f, s0 = 0.f, s1 = 0.f;
  for (int q = g; q < 256; q += G) {
    const long p = p0 + q;
    if (p >= n) break;
    const long b = p / hw, r = p % hw;
    const float d0 = dout[(b * 2) * hw + r], d1 = dout[(b * 2 + 1) * hw + r];
    const float v = bf2f(x[p * C + c]);
    dx[p * C + c] = w0 * d0 + w1 * d1;
    a0 += d0 * v;
    a1 += d1 * v;
    s0 += d0;
    s1 += d1;
  }
  __shared__ float r0[256], r1[256], q0[256], q1[256];
  r0[t] = a0;
  r1[t] = a1;
  q0[t] = s0;
  q1[t] = s1;
  __syncthreads();
  float *dst = part + (long)blockIdx.x * (2 * C + 2);
  if (t < C) {
    float u0 = 0.f, u1 = 0.f;
    for (int k = 0; k < G; ++k) {
      u0 += r0[k * C + t];
      u1 += r1[k * C + t];
    }
    dst[t] = u0;
    dst[C + t] = u1;
  }
  if (t == 0) {  // every pixel once: the threads of channel 0
    float u0 = 0.f, u1 = 0.f;
    for (int k = 0; k < G; ++k) {
      u0 += q0[k * C];
      u1 += q1[k * C];
    }
    dst[2 * C] = u0;
    dst[2 * C + 1] = u1;
  }
}

// Adam (Kingma & Ba 2015, Algorithm 1) on FP32 masters.
__global__ void k_adam(float *__restrict__ w, const float *__restrict__ g, float *__restrict__ m1,
                       float *__restrict__ m2, long n, float lr, float b1, float b2, float eps, float c1, float c2) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float a = b1 * m1[i] + (1.f - b1) * gi, v = b2 * m2[i] + (1.f - b2) * gi * gi;
  m1[i] = a;
  m2[i] = v;
  w[i] -= lr * (a / c1) / (sqrtf(v / c2) + eps);
}

// BF16 copies of a layer's weights packed for the convolutions: wf (rows: output channels) for the
// forward, wd (rows: input channels, taps flipped) for the data gradient.
__global__ void k_weights_bf16(const float *__restrict__ w, bf16 *__restrict__ wf, bf16 *__restrict__ wd, int cout,
                               int cin) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long n = 9L * cout * cin;
  if (i >= n) return;
  const int ci = (int)(i % cin);
  const long t = i / cin;
  const int co = (int)(t % cout), tap = (int)(t / cout);
  const bf16 v = f2bf(w[i]);
  wf[packed_weight(co, ci, tap, cin)] = v;
  if (wd) wd[packed_weight(ci, co, 8 - tap, cout)] = v;
}

// ------------------------------------------------------------------------------------------------
// Host side
// ------------------------------------------------------------------------------------------------
struct Dev {
  void *p = nullptr;
  size_t n = 0;
  int ensure(size_t bytes) {
    if (n >= bytes) return MSG_OK;
    if (p) UHIP(hipFree(p));
    p = nullptr;
    n = 0;
    UHIP(hipMalloc(&p, bytes ? bytes : 16));
    n = bytes;
    return MSG_OK;
  }
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
  }
  template <typename T>
  T *as() const {
    return static_cast<T *>(p);
  }
};

// A tensor of the network: NHWC at scale s (H >> s, W >> s) with C channels.
struct Act {
  int scale, C;
  Dev y;   // bf16 values
  Dev dy;  // fp32 gradient (activations with mode GRAD_OWN, and the pooled ones)
  int mode = GRAD_OWN;
  int up_of = -1, skip_of = -1, pooled = -1;  // the decoder convolution that reads it, the pooled activation
};

struct Conv {
  int in1, in2;   // source activations (in2 < 0: none)
  int up1;        // in1 is upsampled
  int out;        // destination activation
  int cin1, cin2, cout, cin_real;
  long woff, boff;  // offsets in the flat parameter vector
  Dev dv;           // decoder convolutions with a skip tensor: fp32 gradient of their two inputs
};

}  // namespace

struct msg_unet {
  int scales = 4, base = 32;
  std::vector<Act> acts;
  std::vector<Conv> convs;
  std::vector<std::pair<int, int>> pools;  // (from, to)
  int head_in = -1;
  long whoff = 0, bhoff = 0, nparams = 0;
  Dev w, g, m1, m2;          // FP32 masters, gradient, Adam moments (flat)
  std::vector<Dev> wf, wd;   // per conv: bf16 forward / data-gradient weights
  Dev in_packed, out, dout, dz, part, bpart, hpart, lpart;
  int B = 0, H = 0, Wd = 0;
  long step = 0;
  hipStream_t s = nullptr;
};

namespace {

int build_graph(msg_unet *u) {
  const int S = u->scales, C = u->base;
  auto act = [&](int scale, int c) {
    u->acts.push_back(Act{scale, c});
    return (int)u->acts.size() - 1;
  };
  const int input = act(0, 16);
  std::vector<int> skip(S);
  int cur = input, ch = 16;
  for (int s = 0; s < S; ++s) {
    const int co = C << s;
    if (s > 0) {
      const int p = act(s, ch);
      u->pools.push_back({cur, p});
      cur = p;
    }
    const int a = act(s, co);
    u->convs.push_back(Conv{cur, -1, 0, a, ch, 0, co, s == 0 ? 2 : ch, 0, 0, Dev()});
    const int b = act(s, co);
    u->convs.push_back(Conv{a, -1, 0, b, co, 0, co, co, 0, 0, Dev()});
    skip[s] = b;
    cur = b;
    ch = co;
  }
  for (int s = S - 2; s >= 0; --s) {
    const int co = C << s;
    const int a = act(s, co);
    u->convs.push_back(Conv{cur, skip[s], 1, a, ch, co, co, ch + co, 0, 0, Dev()});
    const int b = act(s, co);
    u->convs.push_back(Conv{a, -1, 0, b, co, 0, co, co, 0, 0, Dev()});
    cur = b;
    ch = co;
  }
  u->head_in = cur;
  for (size_t k = 0; k < u->convs.size(); ++k)
    if (u->convs[k].in2 >= 0) {
      u->acts[u->convs[k].in1].mode = GRAD_UP;
      u->acts[u->convs[k].in1].up_of = (int)k;
      u->acts[u->convs[k].in2].mode = GRAD_SKIP;
      u->acts[u->convs[k].in2].skip_of = (int)k;
    }
  for (auto &q : u->pools) u->acts[q.first].pooled = q.second;
  long off = 0;
  for (auto &c : u->convs) {
    c.woff = off;
    off += 9L * c.cout * (c.cin1 + c.cin2);
    c.boff = off;
    off += c.cout;
  }
  u->whoff = off;
  off += 2L * C;
  u->bhoff = off;
  off += 2;
  u->nparams = off;
  return MSG_OK;
}

int refresh_bf16(msg_unet *u) {
  for (size_t k = 0; k < u->convs.size(); ++k) {
    const Conv &c = u->convs[k];
    const int cin = c.cin1 + c.cin2;
    const long n = 9L * c.cout * cin;
    hipLaunchKernelGGL(k_weights_bf16, dim3(cdivu(n, 256)), dim3(256), 0, u->s, u->w.as<float>() + c.woff,
                       u->wf[k].as<bf16>(), k == 0 ? nullptr : u->wd[k].as<bf16>(), c.cout, cin);
    UHIP(hipGetLastError());
  }
  return MSG_OK;
}

// Launch shape of the weight gradient: channel blocks per workgroup (wm x wn), rows per spatial tile, and
// the number of pixel ranges, each a partial sum. 64 x 64 channels where both are multiples (a staged
// pixel then meets most operands), the rows shared among waves otherwise. About two workgroups per compute
// unit, fewer where a range would fall below two tiles: every range costs a write and a read of its
// partial sums.
struct WgradGeom {
  int wm, wn, rows, nblocks, nsplit;
};
WgradGeom wgrad_geom(int B, int H, int W, int cin, int cout) {
  WgradGeom g;
  g.wm = cout % 64 == 0 ? 2 : 1;
  g.wn = g.wm == 2 && cin % 64 == 0 ? 2 : 1;
  g.rows = g.wm * g.wn == 1 ? 16 : 8;
  g.nblocks = (cout / (32 * g.wm)) * cdivu(cin, 32 * g.wn);
  const int ntile = B * (H / g.rows) * (W / 32);
  g.nsplit = std::max(1, std::min(cdivu(512, g.nblocks), cdivu(ntile, 2)));
  return g;
}

int ensure_acts(msg_unet *u, int B, int H, int W, bool grads) {
  if (H % (32 << (u->scales - 1)) != 0 || W % (32 << (u->scales - 1)) != 0)
    return ufail(MSG_ERR_ARG, "msg_unet: H and W must be multiples of 32 * 2^(scales-1)");
  if ((long)B * H * W * 16 >= (1L << 31)) return ufail(MSG_ERR_ARG, "batch x H x W too large");
  for (size_t k = 1; k < u->acts.size(); ++k) {  // activation 0 is the packed input
    Act &a = u->acts[k];
    const size_t px = (size_t)B * (H >> a.scale) * (W >> a.scale);
    UCHK(a.y.ensure(px * a.C * 2));
    if (grads && a.mode == GRAD_OWN) UCHK(a.dy.ensure(px * a.C * 4));
  }
  const size_t px0 = (size_t)B * H * W;
  UCHK(u->in_packed.ensure(px0 * 16 * 2));
  u->acts[0].y.p = u->in_packed.p;  // not owned (freed through in_packed)
  u->acts[0].y.n = 0;
  if (grads) {
    UCHK(u->out.ensure(px0 * 2 * 4));
    UCHK(u->dout.ensure(px0 * 2 * 4));
    size_t dzmax = 0, partmax = 0, bpmax = 0;
    for (auto &c : u->convs) {
      const int s = u->acts[c.out].scale;
      const size_t px = (size_t)B * (H >> s) * (W >> s);
      const int cin = c.cin1 + c.cin2;
      if (c.in2 >= 0) UCHK(c.dv.ensure(px * cin * 4));
      dzmax = std::max(dzmax, px * c.cout * 2);
      partmax = std::max(partmax, (size_t)wgrad_geom(B, H >> s, W >> s, cin, c.cout).nsplit * 9 * c.cout * cin * 4);
      bpmax = std::max(bpmax, (px * c.cout + RELU_BLOCK - 1) / RELU_BLOCK * RELU_BLOCK * 4);
    }
    UCHK(u->dz.ensure(dzmax));
    UCHK(u->part.ensure(partmax));
    UCHK(u->bpart.ensure(bpmax));
    UCHK(u->hpart.ensure((px0 + 255) / 256 * (2 * u->base + 2) * 4));
    UCHK(u->lpart.ensure((px0 * 2 + 255) / 256 * 8));
  }
  u->B = B;
  u->H = H;
  u->Wd = W;
  return MSG_OK;
}

template <int CIN, int WM, int WR, int NT, int NP, typename OutT>
void conv_tile(msg_unet *u, ConvIn in, const bf16 *w, const float *bias, OutT *y, int cout, int relu, int H, int W) {
  const dim3 grid((unsigned)((long)u->B * (W / 32) * (H / (WR * NP)) * (cout / (32 * NT * WM))));
  hipLaunchKernelGGL((k_conv3x3_tile<CIN, WM, WR, NT, NP, OutT>), grid, dim3(64 * WM * WR), 0, u->s, in, w, bias, y, H,
                     W, cout, relu);
}

// H and W are multiples of 32, cout of 32. Tiles by what LDS holds (16 rows of up to 64 input channels, 8
// of 96, 4 beyond) and by the work there is: the largest NT x NP that still gives every SIMD two waves, or
// one with 2 x 2. Only the channel counts that occur have kernels (base a power of two from 32 on): BF16 results
// from 16, 32, 64, 96, 128, 192, 256, 384 and more channels, FP32 results (data gradients) from powers of two, 32
// results or 96 from up to 96 channels only, other counts are multiples of 64.
template <typename OutT>
int launch_conv(msg_unet *u, ConvIn in, const bf16 *w, const float *bias, OutT *y, int cout, int relu, int H, int W) {
  constexpr bool FWD = sizeof(OutT) == 2;
  const int cin = in.c1 + in.c2;
  const long rows = (long)u->B * H * (W / 32);  // tiles of 32 pixels
  auto waves = [&](int nt, int np) { return rows / np * (cout / (32 * nt)); };
  const bool two = cout % 64 == 0, four = cout % 128 == 0;
  bool done = two || cin < 128;
#define CONV(CIN, WM, WR, NT, NP) conv_tile<CIN, WM, WR, NT, NP>(u, in, w, bias, y, cout, relu, H, W)
#define CONV_LARGE(CIN)                             \
  do {                                              \
    if (four && waves(2, 2) >= 1024)                \
      CONV(CIN, 2, 2, 2, 2);                        \
    else                                            \
      CONV(CIN, 2, 2, 1, 2);                        \
  } while (0)
  // 32 and 64 channels; the wide single-row tile where the results are not a multiple of 64
  auto small = [&](auto c) {
    constexpr int CIN = decltype(c)::value;
    if (two && waves(2, 4) >= 2048) {
      CONV(CIN, 1, 4, 2, 4);
      return;
    }
    if constexpr (CIN == 32 || !FWD)
      if (!two && waves(1, 4) >= 2048) {
        CONV(CIN, 1, 4, 1, 4);
        return;
      }
    if (two && waves(2, 2) >= 1024)
      CONV(CIN, 1, 4, 2, 2);
    else
      CONV(CIN, 1, 4, 1, 2);
  };
  if (done) {
    if (cin == 32)
      small(std::integral_constant<int, 32>());
    else if (cin == 64)
      small(std::integral_constant<int, 64>());
    else if (cin == 128)
      CONV_LARGE(128);
    else if (cin == 256)
      CONV_LARGE(256);
    else
      done = false;
    if constexpr (FWD) {
      if (!done) {
        done = true;
        if (cin == 16 && waves(1, 4) >= 1024)
          CONV(16, 1, 4, 1, 4);
        else if (cin == 16)
          CONV(16, 1, 4, 1, 2);
        else if (cin == 96 && waves(1, 4) >= 1024)
          CONV(96, 1, 2, 1, 4);
        else if (cin == 96)
          CONV(96, 1, 4, 1, 2);
        else if (cin == 192 && waves(2, 2) >= 1024)
          CONV(192, 1, 2, 2, 2);
        else if (cin == 192)
          CONV(192, 2, 2, 1, 2);
        else if (cin == 384)
          CONV_LARGE(384);
        else
          done = false;
      }
    }
  }
#undef CONV
#undef CONV_LARGE
  if (!done) {  // the input tile does not fit LDS
    if (!two || cin % 64 != 0) return ufail(MSG_ERR_ARG, "a convolution between channel counts that no network has");
    const int np = (W % 64 == 0) ? 2 : 1;
    const dim3 grid(cdivu((long)u->B * H * W, 128 * np), cout / 64);
    if (np == 2)
      hipLaunchKernelGGL((k_conv3x3<2, OutT>), grid, dim3(256), 0, u->s, in, w, bias, y, u->B, H, W, cout, relu);
    else
      hipLaunchKernelGGL((k_conv3x3<1, OutT>), grid, dim3(256), 0, u->s, in, w, bias, y, u->B, H, W, cout, relu);
  }
  UHIP(hipGetLastError());
  return MSG_OK;
}

ConvIn conv_input(msg_unet *u, const Conv &c) {
  ConvIn in;
  in.x1 = u->acts[c.in1].y.as<bf16>();
  in.x2 = c.in2 >= 0 ? u->acts[c.in2].y.as<bf16>() : nullptr;
  in.c1 = c.cin1;
  in.c2 = c.cin2;
  in.up1 = c.up1;
  return in;
}

int forward(msg_unet *u, const float *input, float *out) {
  const int B = u->B, H = u->H, W = u->Wd;
  const long px0 = (long)B * H * W;
  hipLaunchKernelGGL(k_pack_input, dim3(cdivu(px0, 256)), dim3(256), 0, u->s, input, u->in_packed.as<bf16>(), B, H, W);
  UHIP(hipGetLastError());
  size_t pi = 0;
  for (size_t k = 0; k < u->convs.size(); ++k) {
    const Conv &c = u->convs[k];
    // the pool feeding this convolution runs first
    while (pi < u->pools.size() && u->pools[pi].second == c.in1) {
      const Act &a = u->acts[u->pools[pi].first];
      const int Hs = H >> a.scale, Ws = W >> a.scale;
      const long n = (long)B * (Hs / 2) * (Ws / 2) * (a.C / 8);
      hipLaunchKernelGGL(k_pool, dim3(cdivu(n, 256)), dim3(256), 0, u->s, a.y.as<bf16>(),
                         u->acts[u->pools[pi].second].y.as<bf16>(), B, Hs, Ws, a.C);
      UHIP(hipGetLastError());
      ++pi;
    }
    const int s = u->acts[c.out].scale;
    UCHK(launch_conv(u, conv_input(u, c), u->wf[k].as<bf16>(), u->w.as<float>() + c.boff, u->acts[c.out].y.as<bf16>(),
                     c.cout, 1, H >> s, W >> s));
  }
  hipLaunchKernelGGL(k_head, dim3(cdivu(px0, 256)), dim3(256), 0, u->s, u->acts[u->head_in].y.as<bf16>(),
                     u->w.as<float>() + u->whoff, u->w.as<float>() + u->bhoff, out, B, H, W,
                     u->acts[u->head_in].C);
  UHIP(hipGetLastError());
  return MSG_OK;
}

int backward(msg_unet *u, const float *target, double *loss) {
  const int B = u->B, H = u->H, W = u->Wd;
  const long px0 = (long)B * H * W;
  float *g = u->g.as<float>();
  const long nout = px0 * 2;
  const int nlb = cdivu(nout, 256);
  hipLaunchKernelGGL(k_mse, dim3(nlb), dim3(256), 0, u->s, u->out.as<float>(), target, u->dout.as<float>(), nout,
                     u->lpart.as<double>());
  UHIP(hipGetLastError());
  // head
  const int C0 = u->acts[u->head_in].C;
  const int nhb = cdivu(px0, 256);
  hipLaunchKernelGGL(k_head_grad, dim3(nhb), dim3(256), 0, u->s, u->acts[u->head_in].y.as<bf16>(),
                     u->w.as<float>() + u->whoff, u->dout.as<float>(), u->acts[u->head_in].dy.as<float>(), B, H, W,
                     C0, u->hpart.as<float>());
  UHIP(hipGetLastError());
  hipLaunchKernelGGL(k_col_sum, dim3(2 * C0 + 2), dim3(256), 0, u->s, u->hpart.as<float>(), nhb,
                     (long)(2 * C0 + 2), 2 * C0 + 2, g + u->whoff);  // dwh then dbh are contiguous in the flat vector
  UHIP(hipGetLastError());
  for (int k = (int)u->convs.size() - 1; k >= 0; --k) {
    const Conv &c = u->convs[k];
    const Act &o = u->acts[c.out];
    const int Hs = H >> o.scale, Ws = W >> o.scale;
    const long px = (long)B * Hs * Ws;
    const long n = px * c.cout;
    const int win = std::min(c.cout, RELU_BLOCK);
    const int nb = cdivu(n, (long)RELU_BLOCK * (c.cout <= RELU_BLOCK ? RELU_CHUNKS : 1));
    int logc = 0;
    while ((1 << logc) < c.cout) ++logc;
    GradSrc gs{o.dy.as<float>(), nullptr, c.cout, 0};
    if (o.mode == GRAD_UP) {
      const Conv &q = u->convs[o.up_of];
      gs = {q.dv.as<float>(), nullptr, q.cin1 + q.cin2, 0};
      hipLaunchKernelGGL(k_relu_grad<GRAD_UP>, dim3(nb), dim3(256), 0, u->s, gs, o.y.as<bf16>(), u->dz.as<bf16>(), n,
                         logc, Hs, Ws, u->bpart.as<float>());
    } else if (o.mode == GRAD_SKIP) {
      const Conv &q = u->convs[o.skip_of];
      gs = {q.dv.as<float>(), u->acts[o.pooled].dy.as<float>(), q.cin1 + q.cin2, q.cin1};
      hipLaunchKernelGGL(k_relu_grad<GRAD_SKIP>, dim3(nb), dim3(256), 0, u->s, gs, o.y.as<bf16>(), u->dz.as<bf16>(), n,
                         logc, Hs, Ws, u->bpart.as<float>());
    } else {
      hipLaunchKernelGGL(k_relu_grad<GRAD_OWN>, dim3(nb), dim3(256), 0, u->s, gs, o.y.as<bf16>(), u->dz.as<bf16>(), n,
                         logc, Hs, Ws, u->bpart.as<float>());
    }
    UHIP(hipGetLastError());
    const ConvIn in = conv_input(u, c);
    const int cin = c.cin1 + c.cin2;
    const WgradGeom wg = wgrad_geom(B, Hs, Ws, cin, c.cout);
    const dim3 gw((unsigned)(wg.nblocks * wg.nsplit));
    float *pt = u->part.as<float>();
    const bf16 *zp = u->dz.as<bf16>();
    if (wg.wm == 2 && wg.wn == 2)
      hipLaunchKernelGGL((k_conv3x3_wgrad<2, 2, 8>), gw, dim3(256), 0, u->s, in, zp, pt, B, Hs, Ws, c.cout, wg.nsplit);
    else if (wg.wm == 2)
      hipLaunchKernelGGL((k_conv3x3_wgrad<2, 1, 8>), gw, dim3(256), 0, u->s, in, zp, pt, B, Hs, Ws, c.cout, wg.nsplit);
    else
      hipLaunchKernelGGL((k_conv3x3_wgrad<1, 1, 16>), gw, dim3(256), 0, u->s, in, zp, pt, B, Hs, Ws, c.cout, wg.nsplit);
    UHIP(hipGetLastError());
    const long nw = 9L * c.cout * cin;
    hipLaunchKernelGGL(k_layer_sums, dim3(cdivu(nw, 64) + c.cout), dim3(256), 0, u->s, pt, wg.nsplit, nw, g + c.woff,
                       u->bpart.as<float>(), nb, (long)win, c.cout, g + c.boff);
    UHIP(hipGetLastError());
    if (k == 0) continue;  // no gradient for the input
    // gradient of the input (FP32): of both sources for a decoder convolution, which the two activations'
    // k_relu_grad read; else the source's own
    ConvIn din;
    din.x1 = u->dz.as<bf16>();
    din.x2 = nullptr;
    din.c1 = c.cout;
    din.c2 = 0;
    din.up1 = 0;
    UCHK(launch_conv(u, din, u->wd[k].as<bf16>(), (const float *)nullptr,
                     (c.in2 >= 0 ? c.dv : u->acts[c.in1].dy).as<float>(), cin, 0, Hs, Ws));
  }
  if (loss) {
    std::vector<double> lp(nlb);
    UHIP(hipMemcpyAsync(lp.data(), u->lpart.p, sizeof(double) * nlb, hipMemcpyDeviceToHost, u->s));
    UHIP(hipStreamSynchronize(u->s));
    double a = 0;
    for (double v : lp) a += v;
    *loss = a;
  }
  return MSG_OK;
}

// He initialisation from the seed (the padded input channels stay zero), zero biases. flatten: the generator
// inlined into the loops, whatever else the file holds (a call per number doubles the two million draws' time).
__attribute__((flatten)) void he_init(const msg_unet *u, unsigned long long seed, std::vector<float> &h) {
  std::mt19937_64 rng(seed);
  std::normal_distribution<double> nd(0.0, 1.0);
  for (auto &c : u->convs) {
    const int cin = c.cin1 + c.cin2;
    const double sd = std::sqrt(2.0 / (9.0 * c.cin_real));
    for (int t = 0; t < 9; ++t)
      for (int o = 0; o < c.cout; ++o)
        for (int i = 0; i < cin; ++i)
          h[c.woff + ((long)t * c.cout + o) * cin + i] = (c.in1 != 0 || i < c.cin_real) ? (float)(sd * nd(rng)) : 0.f;
  }
  const double sdh = std::sqrt(1.0 / u->base);
  for (int k = 0; k < 2 * u->base; ++k) h[u->whoff + k] = (float)(sdh * nd(rng));
}

}  // namespace

extern "C" {

int msg_unet_create(msg_unet **net, int scales, int base_channels, unsigned long long seed) {
  // powers of two: every layer's channel count then divides 256 or is a multiple of it, which the
  // per-channel reductions assume
  if (!net || scales < 1 || scales > 6 || base_channels < 32 || base_channels > HEAD_CMAX ||
      (base_channels & (base_channels - 1)) != 0)
    return ufail(MSG_ERR_ARG, "msg_unet_create: scales in 1..6, base_channels 32, 64, 128 or 256");
  msg_unet *u = new msg_unet();
  u->scales = scales;
  u->base = base_channels;
  build_graph(u);
  int rc = MSG_OK;
  auto bail = [&](int r) {
    rc = r;
    return r;
  };
  if (bail(u->w.ensure(u->nparams * 4)) || bail(u->g.ensure(u->nparams * 4)) || bail(u->m1.ensure(u->nparams * 4)) ||
      bail(u->m2.ensure(u->nparams * 4))) {
    delete u;
    return rc;
  }
  u->wf.resize(u->convs.size());
  u->wd.resize(u->convs.size());
  for (size_t k = 0; k < u->convs.size(); ++k) {
    const Conv &c = u->convs[k];
    const size_t n = 9L * c.cout * (c.cin1 + c.cin2) * 2;
    if (u->wf[k].ensure(n) || u->wd[k].ensure(n)) {
      delete u;
      return MSG_ERR_HIP;
    }
  }
  if (hipStreamCreateWithFlags(&u->s, hipStreamNonBlocking) != hipSuccess) {
    delete u;
    return ufail(MSG_ERR_HIP, "msg_unet_create: stream");
  }
  std::vector<float> h(u->nparams, 0.f);
  he_init(u, seed, h);
  *net = u;
  return msg_unet_set_params(u, h.data());
}

int msg_unet_destroy(msg_unet *u) {
  if (!u) return MSG_OK;
  if (u->s) (void)hipStreamSynchronize(u->s);
  for (size_t k = 0; k < u->acts.size(); ++k) {
    if (k == 0) u->acts[0].y.p = nullptr;  // the packed input buffer, owned by in_packed
    u->acts[k].y.release();
    u->acts[k].dy.release();
  }
  for (Dev *d : {&u->w, &u->g, &u->m1, &u->m2, &u->in_packed, &u->out, &u->dout, &u->dz, &u->part,
                 &u->bpart, &u->hpart, &u->lpart})
    d->release();
  for (auto &c : u->convs) c.dv.release();
  for (auto &d : u->wf) d.release();
  for (auto &d : u->wd) d.release();
  if (u->s) (void)hipStreamDestroy(u->s);
  delete u;
  return MSG_OK;
}

int msg_unet_param_count(msg_unet *u, long long *count) {
  if (!u || !count) return ufail(MSG_ERR_ARG, "invalid argument");
  *count = u->nparams;
  return MSG_OK;
}

int msg_unet_get_params(msg_unet *u, float *host) {
  if (!u || !host) return ufail(MSG_ERR_ARG, "invalid argument");
  UHIP(hipMemcpyAsync(host, u->w.p, u->nparams * 4, hipMemcpyDeviceToHost, u->s));
  UHIP(hipStreamSynchronize(u->s));
  return MSG_OK;
}

int msg_unet_set_params(msg_unet *u, const float *host) {
  if (!u || !host) return ufail(MSG_ERR_ARG, "invalid argument");
  UHIP(hipMemcpyAsync(u->w.p, host, u->nparams * 4, hipMemcpyHostToDevice, u->s));
  UHIP(hipMemsetAsync(u->m1.p, 0, u->nparams * 4, u->s));
  UHIP(hipMemsetAsync(u->m2.p, 0, u->nparams * 4, u->s));
  u->step = 0;
  UCHK(refresh_bf16(u));
  UHIP(hipStreamSynchronize(u->s));
  return MSG_OK;
}

int msg_unet_forward(msg_unet *u, const float *in, float *out, int batch, int H, int W, void *stream) {
  if (!u || !in || !out || batch < 1) return ufail(MSG_ERR_ARG, "invalid argument");
  if (stream) UHIP(hipStreamSynchronize((hipStream_t)stream));
  UCHK(ensure_acts(u, batch, H, W, false));
  UCHK(forward(u, in, out));
  UHIP(hipStreamSynchronize(u->s));
  return MSG_OK;
}

int msg_unet_gradient(msg_unet *u, const float *in, const float *target, int batch, int H, int W, double *loss,
                      float *grad_host, void *stream) {
  if (!u || !in || !target || batch < 1) return ufail(MSG_ERR_ARG, "invalid argument");
  if (stream) UHIP(hipStreamSynchronize((hipStream_t)stream));
  UCHK(ensure_acts(u, batch, H, W, true));
  UCHK(forward(u, in, u->out.as<float>()));
  UCHK(backward(u, target, loss));
  if (grad_host) UHIP(hipMemcpyAsync(grad_host, u->g.p, u->nparams * 4, hipMemcpyDeviceToHost, u->s));
  UHIP(hipStreamSynchronize(u->s));
  return MSG_OK;
}

int msg_unet_adam_step(msg_unet *u, float lr) {
  if (!u || !(lr > 0)) return ufail(MSG_ERR_ARG, "invalid argument");
  ++u->step;
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = 1.f - std::pow(b1, (float)u->step), c2 = 1.f - std::pow(b2, (float)u->step);
  hipLaunchKernelGGL(k_adam, dim3(cdivu(u->nparams, 256)), dim3(256), 0, u->s, u->w.as<float>(), u->g.as<float>(),
                     u->m1.as<float>(), u->m2.as<float>(), u->nparams, lr, b1, b2, 1e-8f, c1, c2);
  UHIP(hipGetLastError());
  UCHK(refresh_bf16(u));
  UHIP(hipStreamSynchronize(u->s));
  return MSG_OK;
}

}  // extern "C"
