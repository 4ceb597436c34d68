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
// copies packed for the forward and for the data gradient (k_weights_bf16).
// A 3x3 convolution is an implicit GEMM on MFMA (v_mfma_f32_32x32x16_bf16): rows = output channels
// (weights), columns = 32 consecutive pixels, reduction = 9 taps x input channels in steps of 16;
// FP32 accumulation, bias and ReLU fused into the epilogue. The upsampling and the concatenation are
// not materialised: the convolution reads channel c < C1 from the coarse tensor at (y/2, x/2) and the
// rest from the skip tensor. The data gradient is the same kernel over the pre-activation gradient with
// flipped taps and transposed weights; the weight gradient reduces over pixels per chunk on MFMA and
// sums the chunks in a fixed order (deterministic).
#include "ms_gpu.h"

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <random>
#include <string>
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

// ------------------------------------------------------------------------------------------------
// 3x3 convolution, forward (or data gradient, with its own packed weights):
// y[p][co] = act(bias[co] + sum_tap sum_ci w[tap][co][ci] in[p + off(tap)][ci]).
//
// A workgroup of four waves computes 32 columns x 4 NP rows of one image and 32 NT output channels; a wave
// NP rows of them, NT x NP MFMA tiles (rows: channels, columns: the 32 pixels of one row). Per chunk of KC
// input channels the tile's pixels with a 1-pixel halo and the chunk's weights of all 9 taps go to LDS
// once; the input fragment of a row then serves the three taps of its column offset and every channel
// tile, a weight fragment all NP rows: (NP + 2) + 3 NT KB from LDS per 3 NT NP instructions, 12 KB per 24
// at NT = 2, NP = 4 (half of the LDS bandwidth at full MFMA rate). Operands read from the caches
// instead, 4 KB per 4 instructions, bound the kernel at 150 TFLOP/s. The 14 convolutions of a forward pass
// of 8 pairs of 256^2 (4 scales, 32 channels): 1049 -> 321 us, 530 TFLOP/s; the small batches and 32
// channels at full size are bound by the staging's latency and by HBM.
//
// LDS slots of 16 bytes (8 channels) are permuted within a pixel (or weight row) by bits of its column, so
// that 8 or 16 lanes reading the same channels of consecutive columns hit distinct banks.
// ------------------------------------------------------------------------------------------------
template <int KC>
__device__ __forceinline__ int conv_slot(int col, int seg) {
  if constexpr (KC == 32)
    return seg ^ (((col >> 2) & 1) | ((((col >> 1) ^ (col >> 3)) & 1) << 1));
  else
    return seg ^ (((col >> 2) ^ (col >> 3)) & 1);
}

// Packed weights: per block of 32 output channels and chunk of KC input channels, [tap][channel row][KC]
// with the rows' slots permuted, in the order the kernel copies them to LDS.
__host__ __device__ inline int conv_kc(int cin) { return cin % 32 == 0 ? 32 : 16; }

template <int NT, int NP, int KC, typename OutT>
__global__ void __launch_bounds__(256, 2)
k_conv3x3(ConvIn in, const bf16 *__restrict__ w, const float *__restrict__ bias, OutT *__restrict__ y, int B, int H,
          int W, int cout, int relu) {
  constexpr int SEG = KC / 8, HR = 4 * NP + 2, HC = 34, NLD = HR * HC * SEG, NIN = (NLD + 255) / 256;
  constexpr int WB = 9 * 32 * KC;  // values of one packed weight block
  __shared__ bf16 sx[HR * HC * KC];
  __shared__ bf16 sw[NT * WB];
  const int cin = in.c1 + in.c2;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int tilesx = W / 32, tilesy = H / (4 * NP), ncb = cout / (32 * NT);
  int t0 = xcd_order(blockIdx.x, gridDim.x);
  const int cb = t0 % ncb;
  t0 /= ncb;
  const int x0 = (t0 % tilesx) * 32;
  t0 /= tilesx;
  const int y0 = (t0 % tilesy) * (4 * NP), b = t0 / tilesy;
  const int px = lane & 31, kh = lane >> 5;
  const int nchunk = cin / KC;
  const int Hh = H >> 1, Wh = W >> 1;

  // the pixels this thread stages: index in the first source (at half size when upsampled) and in the
  // second; -1 outside the image (zeros)
  int p1[NIN], p2[NIN];
  unsigned slots = 0;  // the LDS slots within the pixels, 2 bits each
#pragma unroll
  for (int k = 0; k < NIN; ++k) {
    const int i = tid + 256 * k, pix = i / SEG, seg = i % SEG;
    const int row = pix / HC, col = pix % HC;
    const int gy = y0 + row - 1, gx = x0 + col - 1;
    const bool ok = i < NLD && gy >= 0 && gy < H && gx >= 0 && gx < W;
    p2[k] = ok ? (b * H + gy) * W + gx : -1;
    p1[k] = ok ? (in.up1 ? (b * Hh + (gy >> 1)) * Wh + (gx >> 1) : p2[k]) : -1;
    slots |= (unsigned)conv_slot<KC>(col, seg) << (2 * k);
  }

  f32x16 acc[NT][NP];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int q = 0; q < NP; ++q)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[t][q][r] = 0.f;

  for (int ch = 0; ch < nchunk; ++ch) {
    const int c0 = ch * KC;
    const bool first = c0 < in.c1;  // a chunk lies in one source
    const bf16 *src = first ? in.x1 + c0 : in.x2 + (c0 - in.c1);
    const int cs = first ? in.c1 : in.c2;
    u16x8 v[NIN];
#pragma unroll
    for (int k = 0; k < NIN; ++k) {
      const int p = first ? p1[k] : p2[k];
      v[k] = (u16x8)0;
      if (p >= 0) v[k] = *(const u16x8 *)(src + (long)p * cs + (tid % SEG) * 8);
    }
    constexpr int NW = WB / 8;  // 16-byte pieces of a weight block
    u16x8 wv[NT][(NW + 255) / 256];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const bf16 *wb = w + ((long)(cb * NT + t) * nchunk + ch) * WB;
#pragma unroll
      for (int k = 0; k < (NW + 255) / 256; ++k) {
        const int i = tid + 256 * k;
        if (i < NW) wv[t][k] = *(const u16x8 *)(wb + i * 8);
      }
    }
    if (ch) __syncthreads();  // the previous chunk's reads are done
#pragma unroll
    for (int k = 0; k < NIN; ++k)
      if (tid + 256 * k < NLD)
        *(u16x8 *)(sx + (tid / SEG + 256 / SEG * k) * KC + ((slots >> (2 * k)) & 3) * 8) = v[k];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int k = 0; k < (NW + 255) / 256; ++k) {
        const int i = tid + 256 * k;
        if (i < NW) *(u16x8 *)(sw + t * WB + i * 8) = wv[t][k];
      }
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < KC / 16; ++ks) {
      const bf16 *wr = sw + (px * SEG + conv_slot<KC>(px, 2 * ks + kh)) * 8;
#pragma unroll
      for (int dx = 0; dx < 3; ++dx) {
        const bf16 *xr = sx + ((wave * NP * HC + px + dx) * SEG + conv_slot<KC>(px + dx, 2 * ks + kh)) * 8;
        u16x8 bv[NP + 2];
#pragma unroll
        for (int r = 0; r < NP + 2; ++r) bv[r] = *(const u16x8 *)(xr + r * HC * KC);
#pragma unroll
        for (int dy = 0; dy < 3; ++dy)
#pragma unroll
          for (int t = 0; t < NT; ++t) {
            const u16x8 av = *(const u16x8 *)(wr + t * WB + (dy * 3 + dx) * 32 * KC);
#pragma unroll
            for (int q = 0; q < NP; ++q)
              acc[t][q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(av), as_bf16x8(bv[q + dy]), acc[t][q], 0, 0, 0);
          }
      }
    }
  }
  // lane: pixel px of row q; rows of the tile = output channels (r/4)*8 + kh*4 + r%4
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int co = (cb * NT + t) * 32 + j * 8 + kh * 4;
      float bs[4] = {0.f, 0.f, 0.f, 0.f};
      if (bias) {
#pragma unroll
        for (int e = 0; e < 4; ++e) bs[e] = bias[co + e];
      }
#pragma unroll
      for (int q = 0; q < NP; ++q) {
        OutT *dst = y + ((long)(b * H + y0 + wave * NP + q) * W + x0 + px) * cout + co;
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[e] = acc[t][q][j * 4 + e] + bs[e];
          if (relu) v[e] = v[e] > 0.f ? v[e] : 0.f;
        }
        if constexpr (sizeof(OutT) == 2)
          *(u16x4 *)dst = u16x4{f2bf(v[0]), f2bf(v[1]), f2bf(v[2]), f2bf(v[3])};
        else
          *(f32x4 *)dst = f32x4{v[0], v[1], v[2], v[3]};
      }
    }
}

// ------------------------------------------------------------------------------------------------
// Weight gradient of a 3x3 convolution: part[split][tap][co][ci] = sum over the split's pixels of
// dz[p][co] in[p + off(tap)][ci].
//
// A workgroup takes 32 WM output x 32 WN input channels, all 9 taps, and a range of spatial tiles of R rows
// x 32 columns; its four waves are WM x WN channel blocks times KS = 4 / (WM WN) shares of a tile's rows,
// summed at the end in a fixed order. Per tile, dz and the input with a 1-pixel halo go to LDS as
// [channel block][pixel][32]. The reduction runs over pixels while both operands are channel-innermost:
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

// 16 bytes per lane from global memory straight to LDS, no registers in between: lane l's to dst + 16 l
// (dst is the same for the whole wave; inactive lanes write nothing). Complete after lds_loads_done.
__device__ __forceinline__ void load_to_lds(const bf16 *src, bf16 *dst) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)src,
                                   (__attribute__((address_space(3))) void *)dst, 16, 0, 0);
}
__device__ __forceinline__ void lds_loads_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// what pixels outside the image read
__device__ __align__(16) const bf16 conv_zeros[8] = {0, 0, 0, 0, 0, 0, 0, 0};

template <int WM, int WN, int R>
__global__ void __launch_bounds__(256, 2)
k_conv3x3_wgrad(ConvIn in, const bf16 *__restrict__ dz, float *__restrict__ part, int B, int H, int W, int cout,
                int nsplit) {
  constexpr int KS = 4 / (WM * WN), RW = R / KS, HC = 34;
  constexpr int ZPIX = R * 32, XPIX = (R + 2) * HC;
  constexpr int NZ = ZPIX * WM * 4, NX = XPIX * WN * 4;  // 16-byte pieces
  __shared__ bf16 lds[(ZPIX * WM + XPIX * WN) * 32];
  static_assert(sizeof(lds) >= 3 * 16 * 64 * sizeof(float), "the final sum over the row shares reuses the tile");
  bf16 *sz = lds, *sx = lds + ZPIX * WM * 32;
  const int cin = in.c1 + in.c2;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wave0 = __builtin_amdgcn_readfirstlane(wave * 64);  // this wave's first piece
  const int wm = wave % WM, wn = (wave / WM) % WN, ks = wave / (WM * WN);
  const int ncob = cout / (32 * WM), ncib = (cin + 32 * WN - 1) / (32 * WN);
  int id = xcd_order(blockIdx.x, gridDim.x);
  const int co0 = (id % ncob) * 32 * WM;
  id /= ncob;
  const int ci0 = (id % ncib) * 32 * WN, split = id / ncib;
  const int tilesx = W / 32, tilesy = H / R, ntile = B * tilesy * tilesx;
  const int tbeg = (int)((long)ntile * split / nsplit), tend = (int)((long)ntile * (split + 1) / nsplit);
  const int Hh = H >> 1, Wh = W >> 1;
  // transposing reads: 16 lanes take 4 pixels x 16 channels; the wave's four groups two channel halves and
  // pixels 0..3 and 8..11 (read_transposed adds 4..7 and 12..15)
  const int g = lane >> 4, sl = lane & 15;
  const int loff = (8 * (g >> 1) + (sl >> 2)) * 32 + 16 * (g & 1) + 4 * (sl & 3);
  const bf16 *az = sz + (wm * ZPIX + ks * RW * 32) * 32 + loff, *bx = sx + (wn * XPIX + ks * RW * HC) * 32 + loff;

  f32x16 acc[9];
#pragma unroll
  for (int t = 0; t < 9; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[t][r] = 0.f;

  for (int tile = tbeg; tile < tend; ++tile) {
    const int x0 = (tile % tilesx) * 32, y0 = (tile / tilesx % tilesy) * R, b = tile / tilesx / tilesy;
    if (tile > tbeg) __syncthreads();  // the previous tile's reads are done
#pragma unroll
    for (int k = 0; k < (NZ + 255) / 256; ++k) {
      const int i = tid + 256 * k, seg = i & 3, pix = (i >> 2) % ZPIX, cb = (i >> 2) / ZPIX;
      const bf16 *src = dz + ((long)(b * H + y0 + pix / 32) * W + x0 + pix % 32) * cout + co0 + 32 * cb + 8 * seg;
      if (i < NZ) load_to_lds(src, sz + (wave0 + 256 * k) * 8);
    }
#pragma unroll
    for (int k = 0; k < (NX + 255) / 256; ++k) {
      const int i = tid + 256 * k, seg = i & 3, pix = (i >> 2) % XPIX, cb = (i >> 2) / XPIX;
      const int gy = y0 + pix / HC - 1, gx = x0 + pix % HC - 1, c = ci0 + 32 * cb + 8 * seg;
      const bf16 *src = conv_zeros;
      if (gy >= 0 && gy < H && gx >= 0 && gx < W && c < cin) {
        if (c < in.c1)
          src = in.x1 + (long)(in.up1 ? (b * Hh + (gy >> 1)) * Wh + (gx >> 1) : (b * H + gy) * W + gx) * in.c1 + c;
        else
          src = in.x2 + (long)((b * H + gy) * W + gx) * in.c2 + (c - in.c1);
      }
      if (i < NX) load_to_lds(src, sx + (wave0 + 256 * k) * 8);
    }
    lds_loads_done();
    __syncthreads();
#pragma unroll
    for (int xs = 0; xs < 2; ++xs) {  // 16 columns at a time
      bf16x8 a[3];
#pragma unroll
      for (int r = 0; r < RW + 2; ++r) {  // the input's row r - 1 relative to this wave's rows of dz
        if (r < RW) a[r % 3] = read_transposed(az + (r * 32 + 16 * xs) * 32);
#pragma unroll
        for (int dx = 0; dx < 3; ++dx) {
          const bf16x8 bv = read_transposed(bx + (r * HC + 16 * xs + dx) * 32);
#pragma unroll
          for (int dy = 0; dy < 3; ++dy)
            if (r - dy >= 0 && r - dy < RW)
              acc[dy * 3 + dx] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[(r - dy) % 3], bv, acc[dy * 3 + dx], 0, 0, 0);
        }
      }
    }
  }

  const int px = lane & 31, kh = lane >> 5, ci = ci0 + wn * 32 + px;
  float *red = (float *)lds;
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
      float *dst = part + (((long)split * 9 + t) * cout + co0 + wm * 32) * cin;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float v = acc[t][r];
#pragma unroll
        for (int k = 1; k < KS; ++k) v += red[((wave + (k - 1) * WM * WN) * 16 + r) * 64 + lane];
        const int orow = (r >> 2) * 8 + kh * 4 + (r & 3);
        if (ci < cin) dst[(long)orow * cin + ci] = v;
      }
    }
  }
}

// dw[i] = sum over chunks of part[chunk][i]: a workgroup takes 64 elements, its 4 waves every fourth chunk
// in order (8 loads in flight each), their sums added in order. (One thread per element over all chunks:
// 188 us per training step of 8 pairs of 256^2; so: 111 us, of more partial sums.)
__global__ void __launch_bounds__(256)
k_sum_chunks(const float *__restrict__ part, int nchunks, long n, float *__restrict__ dw) {
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
  __shared__ float s[4][64];
  s[wave][lane] = a;
  __syncthreads();
  if (wave == 0 && i < n) dw[i] = ((s[0][lane] + s[1][lane]) + s[2][lane]) + s[3][lane];
}

// dz = bf16(dy * [y > 0]) and per-block partial sums of dz (in FP32) per channel for the bias gradient.
// With C dividing 256 a block of 256 threads covers RELU_CHUNKS x 256 consecutive values and every
// thread keeps its channel; with C a multiple of 256 a block covers 256 channels of one pixel.
constexpr int RELU_CHUNKS = 16;
__global__ void k_relu_grad(const float *__restrict__ dy, const bf16 *__restrict__ y, bf16 *__restrict__ dz, long n,
                            int C, float *__restrict__ bpart) {
  const int chunks = C <= 256 ? RELU_CHUNKS : 1;
  float v = 0.f;
  for (int k = 0; k < chunks; ++k) {
    const long i = ((long)blockIdx.x * chunks + k) * 256 + threadIdx.x;
    if (i < n) {
      const float u = bf2f(y[i]) > 0.f ? dy[i] : 0.f;
      dz[i] = f2bf(u);
      v += u;
    }
  }
  __shared__ float s[256];
  s[threadIdx.x] = v;
  __syncthreads();
  // channels repeat every C threads (C divides 256 or 256 divides C)
  if (C <= 256) {
    if ((int)threadIdx.x < C) {
      float a = 0.f;
      for (int k = threadIdx.x; k < 256; k += C) a += s[k];
      bpart[(long)blockIdx.x * C + threadIdx.x] = a;
    }
  } else {
    bpart[(long)blockIdx.x * 256 + threadIdx.x] = v;  // C > 256: block covers part of one pixel
  }
}

// out[c] = sum over rows r of part[r * stride + off(c)], one workgroup per column c: each thread sums
// the rows r = t, t + 256, ... in order, then a fixed tree over the 256 threads (deterministic).
// Bias gradients (rows: the blocks of k_relu_grad; C > 256: a pixel's channels span C / 256 blocks)
// and the head's partials use it.
__global__ void __launch_bounds__(256)
k_col_sum(const float *__restrict__ part, int nrows, long stride, int C, float *__restrict__ out) {
  const int c = blockIdx.x;
  float a = 0.f;
  if (C <= 256 || stride != 256) {
    for (int r = threadIdx.x; r < nrows; r += 256) a += part[(long)r * stride + c];
  } else {
    const int per = C / 256;  // blocks per pixel
    for (int r = c / 256 + per * (int)threadIdx.x; r < nrows; r += per * 256) a += part[(long)r * 256 + (c % 256)];
  }
  __shared__ float s[256];
  s[threadIdx.x] = a;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if ((int)threadIdx.x < k) s[threadIdx.x] += s[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[c] = s[0];
}

// 2x2 average pooling, NHWC bf16: y[b][yy][x][c] = mean of x[b][2yy..][2x..][c]
__global__ void k_pool(const bf16 *__restrict__ x, bf16 *__restrict__ y, int B, int H, int W, int C) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int Ho = H / 2, Wo = W / 2;
  const long n = (long)B * Ho * Wo * C;
  if (i >= n) return;
  const int c = (int)(i % C);
  long t = i / C;
  const int xo = (int)(t % Wo);
  t /= Wo;
  const int yo = (int)(t % Ho), b = (int)(t / Ho);
  const long r0 = (((long)b * H + 2 * yo) * W + 2 * xo) * C + c, r1 = r0 + (long)W * C;
  const float s = (bf2f(x[r0]) + bf2f(x[r0 + C])) + (bf2f(x[r1]) + bf2f(x[r1 + C]));
  y[i] = f2bf(0.25f * s);
}
// dx[b][y][x][c] += 0.25 dy[b][y/2][x/2][c]
__global__ void k_pool_grad(const float *__restrict__ dy, float *__restrict__ dx, int B, int H, int W, int C) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long n = (long)B * H * W * C;
  if (i >= n) return;
  const int c = (int)(i % C);
  long t = i / C;
  const int x = (int)(t % W);
  t /= W;
  const int yy = (int)(t % H), b = (int)(t / H);
  dx[i] += 0.25f * dy[(((long)b * (H / 2) + yy / 2) * (W / 2) + x / 2) * C + c];
}

// The data gradient of the virtual input (FP32, H x W x (c1 + c2)) to its two sources: the coarse
// tensor (summed over each 2x2 block when upsampled) and the skip tensor, accumulated.
__global__ void k_split_grad1(const float *__restrict__ dv, float *__restrict__ d1, int B, int H, int W, int c1,
                              int c2, int up1) {
  const int cin = c1 + c2;
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int Hs = up1 ? H / 2 : H, Ws = up1 ? W / 2 : W;
  const long n = (long)B * Hs * Ws * c1;
  if (i >= n) return;
  const int c = (int)(i % c1);
  long t = i / c1;
  const int x = (int)(t % Ws);
  t /= Ws;
  const int yy = (int)(t % Hs), b = (int)(t / Hs);
  float a;
  if (up1) {
    const long r0 = (((long)b * H + 2 * yy) * W + 2 * x) * cin + c, r1 = r0 + (long)W * cin;
    a = (dv[r0] + dv[r0 + cin]) + (dv[r1] + dv[r1 + cin]);
  } else {
    a = dv[(((long)b * H + yy) * W + x) * cin + c];
  }
  d1[i] += a;
}
__global__ void k_split_grad2(const float *__restrict__ dv, float *__restrict__ d2, long npix, int c1, int c2) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= npix * c2) return;
  const long p = i / c2;
  const int c = (int)(i % c2);
  d2[i] += dv[p * (c1 + c2) + c1 + c];
}

// Input pairs [B][2][H][W] FP32 (template, reference) -> NHWC bf16 with 16 channels (14 zero).
__global__ void k_pack_input(const float *__restrict__ in, bf16 *__restrict__ x, int B, int H, int W) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long hw = (long)H * W, n = (long)B * hw;
  if (i >= n) return;
  const long b = i / hw, q = i % hw;
  bf16 *dst = x + i * 16;
  dst[0] = f2bf(in[(b * 2) * hw + q]);
  dst[1] = f2bf(in[(b * 2 + 1) * hw + q]);
#pragma unroll
  for (int c = 2; c < 16; ++c) dst[c] = 0;
}

// 1x1 head to 2 channels: out[b][o][y][x] = bh[o] + sum_c wh[o][c] x[p][c] (FP32, planar)
__global__ void k_head(const bf16 *__restrict__ x, const float *__restrict__ wh, const float *__restrict__ bh,
                       float *__restrict__ out, int B, int H, int W, int C) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long hw = (long)H * W, n = (long)B * hw;
  if (p >= n) return;
  float a0 = bh[0], a1 = bh[1];
  const bf16 *src = x + p * C;
  for (int c = 0; c < C; ++c) {
    const float v = bf2f(src[c]);
    a0 += wh[c] * v;
    a1 += wh[C + c] * v;
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

// Head backward over 256 pixels per workgroup: dx[p][c] += sum_o wh[o][c] dout[o][p], and per-block
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
    dx[p * C + c] += w0 * d0 + w1 * d1;
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

// BF16 copies of a layer's weights packed for k_conv3x3: wf (rows: output channels) for the forward, wd
// (rows: input channels, taps flipped) for the data gradient.
__global__ void k_weights_bf16(const float *__restrict__ w, bf16 *__restrict__ wf, bf16 *__restrict__ wd, int cout,
                               int cin) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long n = 9L * cout * cin;
  if (i >= n) return;
  const int ci = (int)(i % cin);
  const long t = i / cin;
  const int co = (int)(t % cout), tap = (int)(t / cout);
  const bf16 v = f2bf(w[i]);
  auto at = [](int row, int k, int tap, int ktotal) {
    const int kc = conv_kc(ktotal), r = row & 31, seg = (k % kc) >> 3;
    const int slot = kc == 32 ? conv_slot<32>(r, seg) : conv_slot<16>(r, seg);
    return ((((long)(row >> 5) * (ktotal / kc) + k / kc) * 9 + tap) * 32 + r) * kc + slot * 8 + (k & 7);
  };
  wf[at(co, ci, tap, cin)] = v;
  if (wd) wd[at(ci, co, 8 - tap, cout)] = v;
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
  Dev dy;  // fp32 gradient
};

struct Conv {
  int in1, in2;   // source activations (in2 < 0: none)
  int up1;        // in1 is upsampled
  int out;        // destination activation
  int cin1, cin2, cout, cin_real;
  long woff, boff;  // offsets in the flat parameter vector
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
  Dev in_packed, out, dout, dv, dz, part, bpart, hpart, lpart;
  int B = 0, H = 0, Wd = 0;
  long step = 0;
  hipStream_t s = nullptr;
};

namespace {

int build_graph(msg_unet *u) {
  const int S = u->scales, C = u->base;
  auto act = [&](int scale, int c) {
    u->acts.push_back(Act{scale, c, Dev(), Dev()});
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
    u->convs.push_back(Conv{cur, -1, 0, a, ch, 0, co, s == 0 ? 2 : ch, 0, 0});
    const int b = act(s, co);
    u->convs.push_back(Conv{a, -1, 0, b, co, 0, co, co, 0, 0});
    skip[s] = b;
    cur = b;
    ch = co;
  }
  for (int s = S - 2; s >= 0; --s) {
    const int co = C << s;
    const int a = act(s, co);
    u->convs.push_back(Conv{cur, skip[s], 1, a, ch, co, co, ch + co, 0, 0});
    const int b = act(s, co);
    u->convs.push_back(Conv{a, -1, 0, b, co, 0, co, co, 0, 0});
    cur = b;
    ch = co;
  }
  u->head_in = cur;
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
  g.wn = cin % 64 == 0 ? 2 : 1;
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
    if (grads) UCHK(a.dy.ensure(px * a.C * 4));
  }
  const size_t px0 = (size_t)B * H * W;
  UCHK(u->in_packed.ensure(px0 * 16 * 2));
  u->acts[0].y.p = u->in_packed.p;  // not owned (freed through in_packed)
  u->acts[0].y.n = 0;
  UCHK(u->out.ensure(px0 * 2 * 4));
  if (grads) {
    UCHK(u->dout.ensure(px0 * 2 * 4));
    size_t dvmax = 0, dzmax = 0, partmax = 0, bpmax = 0;
    for (auto &c : u->convs) {
      const int s = u->acts[c.out].scale;
      const size_t px = (size_t)B * (H >> s) * (W >> s);
      const int cin = c.cin1 + c.cin2;
      dvmax = std::max(dvmax, px * cin * 4);
      dzmax = std::max(dzmax, px * c.cout * 2);
      partmax = std::max(partmax, (size_t)wgrad_geom(B, H >> s, W >> s, cin, c.cout).nsplit * 9 * c.cout * cin * 4);
      bpmax = std::max(bpmax, (px * c.cout + 255) / 256 * 256 * 4);
    }
    UCHK(u->dv.ensure(dvmax));
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

template <int NT, int NP, typename OutT>
void launch_conv_tile(msg_unet *u, ConvIn in, const bf16 *w, const float *bias, OutT *y, int H, int W, int cout,
                      int relu) {
  const dim3 grid((unsigned)((long)u->B * (W / 32) * (H / (4 * NP)) * (cout / (32 * NT))));
  if (conv_kc(in.c1 + in.c2) == 32)
    hipLaunchKernelGGL((k_conv3x3<NT, NP, 32, OutT>), grid, dim3(256), 0, u->s, in, w, bias, y, u->B, H, W, cout, relu);
  else
    hipLaunchKernelGGL((k_conv3x3<NT, NP, 16, OutT>), grid, dim3(256), 0, u->s, in, w, bias, y, u->B, H, W, cout, relu);
}

// H and W are multiples of 32, cout of 32. The largest tile that still gives every compute unit two
// workgroups (one waits at its staging while the other computes); failing that, one; else the smallest.
template <typename OutT>
int launch_conv(msg_unet *u, ConvIn in, const bf16 *w, const float *bias, OutT *y, int cout, int relu, int H, int W) {
  const long rows = (long)u->B * (W / 32) * (H / 4) * (cout / 32);  // workgroups at NT = NP = 1
  const bool two = cout % 64 == 0;
  if (two && rows / 8 >= 512)
    launch_conv_tile<2, 4>(u, in, w, bias, y, H, W, cout, relu);
  else if (rows / 4 >= 512) {
    if (two)
      launch_conv_tile<2, 2>(u, in, w, bias, y, H, W, cout, relu);
    else
      launch_conv_tile<1, 4>(u, in, w, bias, y, H, W, cout, relu);
  } else if (rows / 2 >= 256)
    launch_conv_tile<1, 2>(u, in, w, bias, y, H, W, cout, relu);
  else
    launch_conv_tile<1, 1>(u, in, w, bias, y, H, W, cout, relu);
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

int forward(msg_unet *u, const float *input) {
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
      const long n = (long)B * (Hs / 2) * (Ws / 2) * a.C;
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
                     u->w.as<float>() + u->whoff, u->w.as<float>() + u->bhoff, u->out.as<float>(), B, H, W,
                     u->acts[u->head_in].C);
  UHIP(hipGetLastError());
  return MSG_OK;
}

int backward(msg_unet *u, const float *target, double *loss) {
  const int B = u->B, H = u->H, W = u->Wd;
  const long px0 = (long)B * H * W;
  float *g = u->g.as<float>();
  for (auto &a : u->acts)
    if (a.dy.p) UHIP(hipMemsetAsync(a.dy.p, 0, a.dy.n, u->s));
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
  size_t pi = u->pools.size();
  for (int k = (int)u->convs.size() - 1; k >= 0; --k) {
    const Conv &c = u->convs[k];
    const Act &o = u->acts[c.out];
    const int Hs = H >> o.scale, Ws = W >> o.scale;
    const long px = (long)B * Hs * Ws;
    const long n = px * c.cout;
    const int nb = cdivu(n, 256L * (c.cout <= 256 ? RELU_CHUNKS : 1));
    hipLaunchKernelGGL(k_relu_grad, dim3(nb), dim3(256), 0, u->s, o.dy.as<float>(), o.y.as<bf16>(), u->dz.as<bf16>(),
                       n, c.cout, u->bpart.as<float>());
    UHIP(hipGetLastError());
    hipLaunchKernelGGL(k_col_sum, dim3(c.cout), dim3(256), 0, u->s, u->bpart.as<float>(), nb,
                       (long)(c.cout <= 256 ? c.cout : 256), c.cout, g + c.boff);
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
    else if (wg.wn == 2)
      hipLaunchKernelGGL((k_conv3x3_wgrad<1, 2, 8>), gw, dim3(256), 0, u->s, in, zp, pt, B, Hs, Ws, c.cout, wg.nsplit);
    else
      hipLaunchKernelGGL((k_conv3x3_wgrad<1, 1, 16>), gw, dim3(256), 0, u->s, in, zp, pt, B, Hs, Ws, c.cout, wg.nsplit);
    UHIP(hipGetLastError());
    const long nw = 9L * c.cout * cin;
    hipLaunchKernelGGL(k_sum_chunks, dim3(cdivu(nw, 64)), dim3(256), 0, u->s, pt, wg.nsplit, nw, g + c.woff);
    UHIP(hipGetLastError());
    if (k == 0) continue;  // no gradient for the input
    // data gradient of the virtual input (FP32), then to its sources
    ConvIn din;
    din.x1 = u->dz.as<bf16>();
    din.x2 = nullptr;
    din.c1 = c.cout;
    din.c2 = 0;
    din.up1 = 0;
    UCHK(launch_conv(u, din, u->wd[k].as<bf16>(), (const float *)nullptr, u->dv.as<float>(), cin, 0, Hs, Ws));
    const Act &a1 = u->acts[c.in1];
    const long n1 = (long)B * (H >> a1.scale) * (W >> a1.scale) * c.cin1;
    hipLaunchKernelGGL(k_split_grad1, dim3(cdivu(n1, 256)), dim3(256), 0, u->s, u->dv.as<float>(), a1.dy.as<float>(),
                       B, Hs, Ws, c.cin1, c.cin2, c.up1);
    UHIP(hipGetLastError());
    if (c.in2 >= 0) {
      hipLaunchKernelGGL(k_split_grad2, dim3(cdivu(px * c.cin2, 256)), dim3(256), 0, u->s, u->dv.as<float>(),
                         u->acts[c.in2].dy.as<float>(), px, c.cin1, c.cin2);
      UHIP(hipGetLastError());
    }
    // a pooled activation passes its gradient on to the pool's source
    while (pi > 0 && u->pools[pi - 1].second == c.in1) {
      --pi;
      const Act &src = u->acts[u->pools[pi].first];
      const int Hp = H >> src.scale, Wp = W >> src.scale;
      const long np = (long)B * Hp * Wp * src.C;
      hipLaunchKernelGGL(k_pool_grad, dim3(cdivu(np, 256)), dim3(256), 0, u->s, a1.dy.as<float>(),
                         src.dy.as<float>(), B, Hp, Wp, src.C);
      UHIP(hipGetLastError());
    }
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
  // He initialisation from the seed (the padded input channels stay zero), zero biases
  std::vector<float> h(u->nparams, 0.f);
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
  for (Dev *d : {&u->w, &u->g, &u->m1, &u->m2, &u->in_packed, &u->out, &u->dout, &u->dv, &u->dz, &u->part,
                 &u->bpart, &u->hpart, &u->lpart})
    d->release();
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
  UCHK(forward(u, in));
  UHIP(hipMemcpyAsync(out, u->out.p, (size_t)batch * 2 * H * W * 4, hipMemcpyDeviceToDevice, u->s));
  UHIP(hipStreamSynchronize(u->s));
  return MSG_OK;
}

int msg_unet_gradient(msg_unet *u, const float *in, const float *target, int batch, int H, int W, double *loss,
                      float *grad_host, void *stream) {
  if (!u || !in || !target || batch < 1) return ufail(MSG_ERR_ARG, "invalid argument");
  if (stream) UHIP(hipStreamSynchronize((hipStream_t)stream));
  UCHK(ensure_acts(u, batch, H, W, true));
  UCHK(forward(u, in));
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
