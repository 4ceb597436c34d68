// Reconstruction statistics and input normalisation kernels.
#pragma once

#include "ms_device.h"

namespace msg {

// Per pixel over nimg warped frames (+Inf = no sample): mean of the finite samples in frame order,
// sample count, and median (SeriesMatching::averageSeries, matchSeries.h:404-444;
// MultiVector::getMedianVecOverComponents, aol/multiVector.cpp:99-117; Vector::getMedianValue,
// aol/vec.cpp:933-949: odd count -> middle element, even -> mean of the two middle elements).
// One wave64 per P pixels, 64/P lanes per pixel; the samples of the P pixels live in LDS (P * nimg
// doubles, at most 64 KiB) and the order statistics are found by counting, which needs no sort and
// no per-lane arrays: lane l of a pixel tests the candidates i = l, l + 64/P, ... and the lanes agree
// by shuffles (the k-th smallest value is unique, whichever candidate carries it).
constexpr int ST_LDS_DOUBLES = 8192;           // 64 KiB of samples per wave
constexpr int ST_MAXF = ST_LDS_DOUBLES;         // P = 1: one pixel per wave

// Pixels per wave for a series of nimg frames (64, 16, 4 or 1), or 0 beyond ST_MAXF.
inline int stats_pixels_per_wave(int nimg) {
  for (int p = 64; p >= 1; p /= 4)
    if ((long long)p * nimg <= ST_LDS_DOUBLES) return p;
  return 0;
}

template <typename S, int P>
__global__ void __launch_bounds__(64)
k_series_stats(const S *__restrict__ stack, int nimg, int nn, double fill, S *__restrict__ mean,
               S *__restrict__ count, S *__restrict__ median) {
  constexpr int L = 64 / P;  // lanes per pixel
  extern __shared__ double sv[];  // [nimg][P]
  const int q = threadIdx.x / L, l = threadIdx.x % L;
  const int j = blockIdx.x * P + q;
  const bool valid = j < nn;
  for (int f = l; f < nimg; f += L)
    sv[f * P + q] = valid ? ld(stack + (size_t)f * nn, j) : __builtin_inf();
  __syncthreads();
  if (!valid) return;
  double m = 0;
  int c = 0;
  for (int f = 0; f < nimg; ++f) {  // every lane of the pixel sums in frame order
    const double v = sv[f * P + q];
    if (v != __builtin_inf()) {
      m += v;
      ++c;
    }
  }
  m = (c > 0) ? m / c : fill;
  double med = fill;
  if (c > 0) {
    // k-th smallest finite sample: the value v_i with #(v < v_i) <= k < #(v <= v_i)
    const int k2 = c / 2, k1 = (c % 2 == 1) ? k2 : k2 - 1;
    double a = 0, b = 0;
    bool fa = false, fb = false;
    for (int i = l; i < nimg && !(fa && fb); i += L) {
      const double vi = sv[i * P + q];
      if (vi == __builtin_inf()) continue;
      int lt = 0, le = 0;
      for (int f = 0; f < nimg; ++f) {
        const double v = sv[f * P + q];
        if (v == __builtin_inf()) continue;
        lt += (v < vi);
        le += (v <= vi);
      }
      if (!fa && lt <= k1 && k1 < le) {
        a = vi;
        fa = true;
      }
      if (!fb && lt <= k2 && k2 < le) {
        b = vi;
        fb = true;
      }
    }
    // the lanes of one pixel are L consecutive lanes: butterfly over them
    for (int o = L / 2; o > 0; o /= 2) {
      const double oa = __shfl_xor(a, o), ob = __shfl_xor(b, o);
      const int ofa = __shfl_xor((int)fa, o), ofb = __shfl_xor((int)fb, o);
      if (!fa && ofa) {
        a = oa;
        fa = true;
      }
      if (!fb && ofb) {
        b = ob;
        fb = true;
      }
    }
    med = (c % 2 == 1) ? b : (a + b) / 2;
  }
  if (l == 0) {
    mean[j] = static_cast<S>(m);
    count[j] = static_cast<S>((double)c);
    median[j] = static_cast<S>(med);
  }
}

// The same statistics for series of at most 64 frames, one pixel per thread: the samples in registers,
// padded with +Inf to NP values and sorted by Batcher's odd-even merge network (191 compare-exchanges at
// NP = 32). Loads of consecutive pixels are coalesced and all of a pixel's are issued before the first is
// used: bound by the read of the stack. 31 frames of 1024^2 in FP32, with their warp: 252 us, with the
// counting above (nimg^2 comparisons per pixel) 625 us; it stays for longer series, whose samples do not
// fit the registers. NaN samples count (and make the mean NaN) but never match a rank: they sort
// behind the finite ones, and a median that falls on them is 0, as above.
__device__ __forceinline__ void cmp_swap(float &a, float &b) {  // no NaN
  const float lo = fminf(a, b), hi = fmaxf(a, b);
  a = lo;
  b = hi;
}
__device__ __forceinline__ void cmp_swap(double &a, double &b) {
  const double lo = fmin(a, b), hi = fmax(a, b);
  a = lo;
  b = hi;
}
template <typename S, int NP, int LO, int N, int R>
__device__ __forceinline__ void oe_merge(S (&v)[NP]) {
  if constexpr (2 * R < N) {
    oe_merge<S, NP, LO, N, 2 * R>(v);
    oe_merge<S, NP, LO + R, N, 2 * R>(v);
#pragma unroll
    for (int i = LO + R; i + R < LO + N; i += 2 * R) cmp_swap(v[i], v[i + R]);
  } else {
    cmp_swap(v[LO], v[LO + R]);
  }
}
template <typename S, int NP, int LO, int N>
__device__ __forceinline__ void oe_sort(S (&v)[NP]) {
  if constexpr (N > 1) {
    oe_sort<S, NP, LO, N / 2>(v);
    oe_sort<S, NP, LO + N / 2, N / 2>(v);
    oe_merge<S, NP, LO, N, 1>(v);
  }
}

constexpr int ST_SORT_MAX = 64;  // longest series the sorting network takes

template <typename S, int NP>
__global__ void __launch_bounds__(256)
k_series_stats_sort(const S *__restrict__ stack, int nimg, int nn, double fill, S *__restrict__ mean,
                    S *__restrict__ count, S *__restrict__ median) {
  const int j = blockIdx.x * 256 + threadIdx.x;
  if (j >= nn) return;
  const S inf = (S)__builtin_inf();
  S v[NP];
#pragma unroll
  for (int f = 0; f < NP; ++f) v[f] = f < nimg ? stack[(size_t)f * nn + j] : inf;
  double m = 0;
  int c = 0, real = 0;
#pragma unroll
  for (int f = 0; f < NP; ++f) {  // in frame order
    const bool have = v[f] != inf, num = v[f] == v[f];
    m += have ? (double)v[f] : 0.;
    c += have ? 1 : 0;
    real += have && num ? 1 : 0;
    v[f] = num ? v[f] : inf;
  }
  m = (c > 0) ? m / c : fill;
  oe_sort<S, NP, 0, NP>(v);
  const int k2 = c / 2, k1 = (c % 2 == 1) ? k2 : k2 - 1;
  double a = 0, b = 0;
#pragma unroll
  for (int f = 0; f < NP; ++f) {
    a = f == k1 && f < real ? (double)v[f] : a;
    b = f == k2 && f < real ? (double)v[f] : b;
  }
  mean[j] = static_cast<S>(m);
  count[j] = static_cast<S>((double)c);
  median[j] = static_cast<S>(c > 0 ? ((c % 2 == 1) ? b : (a + b) / 2) : fill);
}

// ------------------------------------------------------------------------------------------------
// Order statistics of images by radix selection: the two ranks prepareMultilevelArray needs of every
// image (its percentile bounds, or its minimum and maximum), found digit by digit from histograms
// instead of sorting the image. Keys are the values' bit patterns in increasing order (negative values
// complemented, positive ones with the sign bit set), so the result is the element a sort would put
// there. Pass p counts digit p of the elements that share the digits found so far, once per rank (one
// histogram serves both ranks while their prefixes agree); the next pass, and the normalisation after the
// last, find their rank's digit from those counts, every workgroup for itself (2048 counts from L2).
// Bound by one read of the images per digit (3 for FP32, 6 for FP64) and, for one image, by its 5 or 8 small
// launches (small images: k_normalize_one). 24 frames of 1024^2 in FP32: 160 us with the copy of the frames, where one library sort
// after another took 3.71 ms (21 launches and about 150 us per frame).
// ------------------------------------------------------------------------------------------------
constexpr int SEL_BITS = 11, SEL_BINS = 1 << SEL_BITS;
constexpr int SEL_THREADS = 256;

template <typename S>
struct SelKey;
template <>
struct SelKey<float> {
  typedef unsigned type;
  static constexpr int PASSES = 3;
  __device__ static type key(float v) {
    const unsigned u = __float_as_uint(v);
    return u & 0x80000000u ? ~u : u | 0x80000000u;
  }
  __device__ static float value(type k) { return __uint_as_float(k & 0x80000000u ? k & 0x7fffffffu : ~k); }
};
template <>
struct SelKey<double> {
  typedef unsigned long long type;
  static constexpr int PASSES = 6;
  __device__ static type key(double v) {
    const unsigned long long u = (unsigned long long)__double_as_longlong(v);
    return u >> 63 ? ~u : u | (1ull << 63);
  }
  __device__ static double value(type k) {
    return __longlong_as_double((long long)(k >> 63 ? k & ~(1ull << 63) : ~k));
  }
};
// right shift of digit p (the last digit holds the bits left over)
template <typename S>
__device__ __forceinline__ int sel_shift(int p) {
  const int s = (int)sizeof(S) * 8 - SEL_BITS * (p + 1);
  return s > 0 ? s : 0;
}

// What is known of a rank before a pass: the digits found so far and the rank among the elements that
// share them.
struct SelState {
  unsigned long long prefix;
  unsigned rank, pad;
};

// The digit that holds `rank` in counts h[SEL_BINS] and the rank within it, found by TH threads (t: the thread among
// them) and left in tmp[TH / 64], tmp[TH / 64 + 1]. tmp: TH / 64 + 2 words of LDS. Barriers of the whole workgroup.
template <int TH>
__device__ __forceinline__ void sel_find(const unsigned *__restrict__ h, unsigned rank, unsigned *tmp, int t) {
  constexpr int PER = SEL_BINS / TH, NW = TH / 64;
  unsigned c[PER], mine = 0;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    c[k] = h[t * PER + k];
    mine += c[k];
  }
  const int lane = t & 63, wid = t >> 6;
  unsigned inc = mine;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned v = __shfl_up(inc, o, 64);
    if (lane >= o) inc += v;
  }
  __syncthreads();  // earlier reads of tmp are done
  if (lane == 63) tmp[wid] = inc;
  __syncthreads();
  unsigned below = inc - mine;
  for (int w = 0; w < wid; ++w) below += tmp[w];
  if (rank >= below && rank - below < mine) {  // exactly one thread: the counts add up to more than rank
    unsigned r = rank - below;
    int k = 0;
#pragma unroll
    for (int j = 0; j < PER - 1; ++j)
      if (k == j && r >= c[j]) {
        r -= c[j];
        ++k;
      }
    tmp[NW] = t * PER + k;
    tmp[NW + 1] = r;
  }
  __syncthreads();
}
// The same for every thread of a workgroup of SEL_THREADS.
__device__ __forceinline__ void sel_digit(const unsigned *__restrict__ h, unsigned rank, unsigned *tmp,
                                          unsigned &digit, unsigned &rest) {
  sel_find<SEL_THREADS>(h, rank, tmp, threadIdx.x);
  digit = tmp[SEL_THREADS / 64];
  rest = tmp[SEL_THREADS / 64 + 1];
}

// State of both ranks of image `img` before digit p, from the state before digit p - 1 and that digit's
// counts (layout [pass][image][rank][SEL_BINS], rank 1's unused where the prefixes agreed).
template <typename S>
__device__ __forceinline__ void sel_advance(const unsigned *__restrict__ hist, const SelState *__restrict__ st, int img,
                                            int nimg, int p, unsigned rank0, unsigned rank1, unsigned *tmp,
                                            SelState (&s)[2]) {
  if (p == 0) {
    s[0] = {0, rank0, 0};
    s[1] = {0, rank1, 0};
    return;
  }
  SelState q[2];
  if (p == 1) {
    q[0] = {0, rank0, 0};
    q[1] = {0, rank1, 0};
  } else {
    q[0] = st[((size_t)(p - 1) * nimg + img) * 2];
    q[1] = st[((size_t)(p - 1) * nimg + img) * 2 + 1];
  }
  const int bits = sel_shift<S>(p - 2) - sel_shift<S>(p - 1);  // width of digit p - 1 (p == 1: see below)
  const int w = p == 1 ? SEL_BITS : bits;
  const bool same = q[0].prefix == q[1].prefix;
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const unsigned *h = hist + (((size_t)(p - 1) * nimg + img) * 2 + (same ? 0 : r)) * SEL_BINS;
    unsigned d, rest;
    sel_digit(h, q[r].rank, tmp, d, rest);
    s[r] = {(q[r].prefix << w) | d, rest, 0};
  }
}

// Counts of digit p. Grid (chunks of PT elements per thread, images).
template <typename S, int PT>
__global__ void __launch_bounds__(SEL_THREADS)
k_sel_count(const S *__restrict__ imgs, int nn, int nimg, int p, unsigned rank0, unsigned rank1,
            unsigned *__restrict__ hist, SelState *__restrict__ st) {
  typedef typename SelKey<S>::type K;
  __shared__ unsigned h[2][SEL_BINS];
  __shared__ unsigned tmp[6];
  const int img = blockIdx.y;
  const S *im = imgs + (size_t)img * nn;
  SelState s[2];
  sel_advance<S>(hist, st, img, nimg, p, rank0, rank1, tmp, s);
  if (p > 0 && blockIdx.x == 0 && threadIdx.x == 0) {
    st[((size_t)p * nimg + img) * 2] = s[0];
    st[((size_t)p * nimg + img) * 2 + 1] = s[1];
  }
  const bool two = s[0].prefix != s[1].prefix;
  for (int i = threadIdx.x; i < SEL_BINS; i += SEL_THREADS) h[0][i] = h[1][i] = 0;
  __syncthreads();
  const int shift = sel_shift<S>(p);
  const int top = p == 0 ? 0 : sel_shift<S>(p - 1);  // bits below the prefix
  const unsigned mask = p == 0 ? SEL_BINS - 1 : (unsigned)((1u << (top - shift)) - 1u);
  const K p0 = (K)s[0].prefix, p1 = (K)s[1].prefix;
  const int i0 = blockIdx.x * (PT * SEL_THREADS) + threadIdx.x;
  constexpr int RUN = 8;  // loads in flight per thread
  for (int k = 0; k < PT; k += RUN) {
    S v[RUN];
#pragma unroll
    for (int r = 0; r < RUN; ++r) {
      const int i = i0 + (k + r) * SEL_THREADS;
      v[r] = im[i < nn ? i : nn - 1];
    }
#pragma unroll
    for (int r = 0; r < RUN; ++r) {
      if (i0 + (k + r) * SEL_THREADS < nn) {
        const K key = SelKey<S>::key(v[r]);
        const unsigned d = (unsigned)(key >> shift) & mask;
        if (p == 0 || (key >> top) == p0) atomicAdd(&h[0][d], 1u);
        if (two && (key >> top) == p1) atomicAdd(&h[1][d], 1u);
      }
    }
  }
  __syncthreads();
  unsigned *g = hist + ((size_t)p * nimg + img) * 2 * SEL_BINS;
  for (int i = threadIdx.x; i < SEL_BINS; i += SEL_THREADS) {
    if (h[0][i]) atomicAdd(g + i, h[0][i]);
    if (two && h[1][i]) atomicAdd(g + SEL_BINS + i, h[1][i]);
  }
}

// prepareMultilevelArray (registration.h:331-347) with the image's elements of rank0 and rank1, lo and hi:
// saturate: clamp to [lo, hi], subtract the minimum (lo) and divide by the maximum (hi - lo);
// otherwise lo, hi are the extrema: subtract the minimum if negative or min_to_zero, divide by the
// (shifted) maximum.
struct NormScale {
  double lo, hi, mx;
  bool saturate, shifted;
  __device__ __forceinline__ NormScale(double l, double h, int sat, int min_to_zero)
      : lo(l), hi(h), saturate(sat), shifted(sat || l < 0. || min_to_zero) {
    mx = shifted ? hi + -1 * lo : hi;  // getMaxValue() of the shifted image
  }
  __device__ __forceinline__ double operator()(double v) const {
    if (saturate) v = v < lo ? lo : (v > hi ? hi : v);
    if (shifted) v += -1 * lo;  // addToAll(-1 * getMinValue())
    if (mx != 0) v /= mx;
    return v;
  }
};

// Grid as k_sel_count.
template <typename S, int PT>
__global__ void __launch_bounds__(SEL_THREADS)
k_normalize(S *__restrict__ imgs, int nn, int nimg, unsigned rank0, unsigned rank1, const unsigned *__restrict__ hist,
            const SelState *__restrict__ st, int saturate, int min_to_zero) {
  typedef typename SelKey<S>::type K;
  __shared__ unsigned tmp[6];
  const int img = blockIdx.y;
  SelState s[2];
  sel_advance<S>(hist, st, img, nimg, SelKey<S>::PASSES, rank0, rank1, tmp, s);
  const NormScale sc((double)SelKey<S>::value((K)s[0].prefix), (double)SelKey<S>::value((K)s[1].prefix), saturate,
                     min_to_zero);
  S *im = imgs + (size_t)img * nn;
  const int i0 = blockIdx.x * (PT * SEL_THREADS) + threadIdx.x;
  constexpr int RUN = 8;
  for (int k = 0; k < PT; k += RUN) {
    S in[RUN];
#pragma unroll
    for (int r = 0; r < RUN; ++r) {
      const int i = i0 + (k + r) * SEL_THREADS;
      in[r] = im[i < nn ? i : nn - 1];
    }
#pragma unroll
    for (int r = 0; r < RUN; ++r) {
      const int i = i0 + (k + r) * SEL_THREADS;
      const double v = sc((double)in[r]);
      if (i < nn) im[i] = static_cast<S>(v);
    }
  }
}

// The same for small images in one launch: a workgroup takes an image through all digits, its counts in LDS. Bound by
// the chain of its barriers and LDS round trips, about 1.5 us a digit. One image of 64^2, whole call: FP32 40 us in 5
// launches, 26 us so, FP64 61 us in 8 launches and 33 us (a library's sort of it: 34 and 41 us).
constexpr int SEL1_THREADS = 1024;

// Counts digit d of the lanes with `take` set; those that share the first one's digit in one addition, so that
// an image of one value (all lanes on one word of LDS) takes no longer than another (FP64 64^2: 16 us less).
// (The sweeps of larger images do without: it costs others 2 us of a workgroup's pass.)
__device__ __forceinline__ void sel_add(unsigned *h, unsigned d, bool take) {
  const unsigned long long act = __ballot(take);
  if (!act) return;
  const int first = __ffsll((long long)act) - 1;
  const unsigned d0 = __builtin_amdgcn_readlane(d, first);
  const unsigned long long same = __ballot(take && d == d0);
  if ((int)(threadIdx.x & 63) == first)
    atomicAdd(&h[d0], (unsigned)__popcll(same));
  else if (take && d != d0)
    atomicAdd(&h[d], 1u);
}

template <typename S>
__global__ void __launch_bounds__(SEL1_THREADS)
k_normalize_one(S *__restrict__ imgs, int nn, unsigned rank0, unsigned rank1, int saturate, int min_to_zero) {
  typedef typename SelKey<S>::type K;
  __shared__ unsigned h[2][SEL_BINS];
  constexpr int HALF = SEL1_THREADS / 2;  // threads that look for a rank's digit
  __shared__ unsigned tmp[2][HALF / 64 + 2];
  S *im = imgs + (size_t)blockIdx.x * nn;
  K prefix[2] = {0, 0};
  unsigned rank[2] = {rank0, rank1};
  constexpr int RUN = 4;  // loads in flight per thread
  const int wave0 = __builtin_amdgcn_readfirstlane(threadIdx.x & ~63), lane = threadIdx.x & 63;
  auto sweep = [&](const auto &f) {  // f(index, value, inside the image), by whole waves
    for (int w = wave0; w < nn; w += RUN * SEL1_THREADS) {
      S v[RUN];
#pragma unroll
      for (int r = 0; r < RUN; ++r) v[r] = im[min(w + r * SEL1_THREADS + lane, nn - 1)];
#pragma unroll
      for (int r = 0; r < RUN; ++r) {
        const int i = w + r * SEL1_THREADS + lane;
        if (w + r * SEL1_THREADS < nn) f(i, v[r], i < nn);
      }
    }
  };
  for (int p = 0; p < SelKey<S>::PASSES; ++p) {
    const int shift = sel_shift<S>(p), top = p == 0 ? 0 : sel_shift<S>(p - 1);
    const int w = p == 0 ? SEL_BITS : top - shift;
    const unsigned mask = (1u << w) - 1u;
    const bool two = prefix[0] != prefix[1];
    for (int i = threadIdx.x; i < SEL_BINS; i += SEL1_THREADS) h[0][i] = h[1][i] = 0;
    __syncthreads();
    sweep([&](int, S v, bool in) {
      const K key = SelKey<S>::key(v);
      const unsigned d = (unsigned)(key >> shift) & mask;
      sel_add(h[0], d, in && (p == 0 || (key >> top) == prefix[0]));
      if (two) sel_add(h[1], d, in && (key >> top) == prefix[1]);
    });
    __syncthreads();
    const int half = wave0 / HALF;
    sel_find<HALF>(h[two ? half : 0], rank[half], tmp[half], threadIdx.x % HALF);
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      prefix[r] = (prefix[r] << w) | tmp[r][HALF / 64];
      rank[r] = tmp[r][HALF / 64 + 1];
    }
  }
  const NormScale sc((double)SelKey<S>::value(prefix[0]), (double)SelKey<S>::value(prefix[1]), saturate, min_to_zero);
  sweep([&](int i, S v, bool in) {
    if (in) im[i] = static_cast<S>(sc((double)v));
  });
}

}  // namespace msg
