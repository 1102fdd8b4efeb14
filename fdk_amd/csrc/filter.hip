// Cosine pre-weighting and ramp/apodised row filtering on gfx950.
//
// Reference behaviour (peng-ac/fdk):
//   FilterCosCorrect / kernelCorrect    Filterlib/FilterLib.h:8-13,
//                                       FilterlibCufft/cudaFftFilter.cu:270-296
//   FilterImageRow (mean4 pad, IPP FFT) Filterlib/FilterLib.h:15-58
//   kernelPad/DotScale/Unpad + cuFFT    FilterlibCufft/cudaFftFilter.cu:14-61, 298-370
//   FilterProjImage                     FilterlibCufft/cudaFftFilter.cu:394-452
//
// Each detector row of nu samples is centred in N = 2^m samples at offset
// (N - nu) / 2, the pad takes the mean of the first / last 3 or 4 samples (or
// zero), the row is multiplied in the frequency domain by the real, even
// filter H and the centre nu samples of the inverse transform (1/N) are kept.
//
// MI355X design: one workgroup filters two rows at once as one complex
// transform (row a in the real part, row b in the imaginary part).  Because H
// is real and even, H * DFT(a + i b) inverts to filt(a) + i filt(b) exactly, so
// no real-to-complex unpacking is needed.  filter_wide_kernel (N = 2^7 .. 2^14) holds 16
// points a thread and runs radix-16 passes (the last ones of radix 2 to 16), the inverse
// as the forward passes' adjoint; other lengths run an in-place radix-2^2 FFT entered in
// bit-reversed order, the filter multiply doubling as the inverse's bit-reversal.  Loads
// apply the cos table, stores crop, optionally transpose (v fastest, what the
// backprojector reads) and convert to the stored dtype.  Twiddles are an FP64-built table.
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

#include "common.hpp"
#include "launch_rules.hpp"

namespace {

struct FilterArgs {
  const float* src;       // rows of nu samples
  long long src_view;     // elements between views
  int src_pitch;          // elements between rows
  float* dst;             // FP32 output (dtype handled by a second pass)
  long long dst_view;
  int dst_pitch;          // row pitch when not transposed
  int transpose;          // 1: dst[view][u][row] with row fastest, pitch = nrows
  const float* cos_table; // nrows x nu (pitch nu) or null
  const float* H;         // N
  const float2* tw;       // N twiddles e^{-2 pi i k / N}
  int nu, nrows, N, logN, pad;
  unsigned* minmax;       // per view {min, max} as ordered uints, or null
  // Output mode: kStoreF32 writes dst as floats; kStoreNone writes nothing
  // (the min/max pass of a two-pass 16-bit filter); kStoreF16 / kStoreBF16
  // write (p - min) / (max - min) of view {min, max} words qmm as 16-bit.
  int qmode;
  const unsigned* qmm;
  int far;                // kFilterWideFar: transposed FP32 stores check their points
};

constexpr int kStoreF32 = 0, kStoreNone = 1, kStoreF16 = 2, kStoreBF16 = 3;

__device__ inline unsigned brev_n(unsigned k, int logN) { return __brev(k) >> (32 - logN); }

__device__ inline float2 cmul(float2 a, float2 b) {
  return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// In-place FFT over buf (bit-reversed input -> natural output); sign = -1
// forward, +1 inverse (conjugate twiddles).  Radix-2 first stage when log2 N is
// odd, then fused radix-2^2 stages.
__device__ void fft_lds(float2* buf, const float2* __restrict__ tw, int N, int logN, float sign) {
  const int tid = threadIdx.x, nt = blockDim.x;
  int L = 1;
  if (logN & 1) {
    for (int q = tid; q < N / 2; q += nt) {
      const float2 x0 = buf[2 * q], x1 = buf[2 * q + 1];
      buf[2 * q] = make_float2(x0.x + x1.x, x0.y + x1.y);
      buf[2 * q + 1] = make_float2(x0.x - x1.x, x0.y - x1.y);
    }
    L = 2;
    __syncthreads();
  }
  for (; L < N; L *= 4) {
    const int s1 = N / (2 * L), s2 = N / (4 * L);
    for (int q = tid; q < N / 4; q += nt) {
      const int j = q % L;
      const int g = (q / L) * 4 * L + j;
      float2 w1 = tw[j * s1], w2 = tw[j * s2];
      w1.y *= -sign;  // table holds e^{-i...}; inverse conjugates
      w2.y *= -sign;
      const float2 x0 = buf[g], x1 = cmul(buf[g + L], w1);
      const float2 x2 = buf[g + 2 * L], x3 = cmul(buf[g + 3 * L], w1);
      const float2 y0 = make_float2(x0.x + x1.x, x0.y + x1.y);
      const float2 y1 = make_float2(x0.x - x1.x, x0.y - x1.y);
      const float2 y2 = make_float2(x2.x + x3.x, x2.y + x3.y);
      const float2 y3 = make_float2(x2.x - x3.x, x2.y - x3.y);
      const float2 t2 = cmul(y2, w2);
      float2 t3 = cmul(y3, w2);
      // forward: multiply by -i; inverse: by +i
      t3 = sign < 0 ? make_float2(t3.y, -t3.x) : make_float2(-t3.y, t3.x);
      buf[g] = make_float2(y0.x + t2.x, y0.y + t2.y);
      buf[g + 2 * L] = make_float2(y0.x - t2.x, y0.y - t2.y);
      buf[g + L] = make_float2(y1.x + t3.x, y1.y + t3.y);
      buf[g + 3 * L] = make_float2(y1.x - t3.x, y1.y - t3.y);
    }
    __syncthreads();
  }
}

// ------------------------------------------------ register DFTs of filter_wide_kernel
// v * (sign * i): sign -1 multiplies by -i, +1 by +i.
__device__ __forceinline__ float2 mul_si(float2 v, float sign) {
  return sign < 0 ? make_float2(v.y, -v.x) : make_float2(-v.y, v.x);
}
__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }

// X[k] = sum_n v[n] e^{sign 2 pi i n k / R}
__device__ __forceinline__ void dft2(float2& a, float2& b) {
  const float2 t = a;
  a = cadd(t, b);
  b = csub(t, b);
}

__device__ __forceinline__ void dft4(float2& v0, float2& v1, float2& v2, float2& v3, float sign) {
  const float2 a0 = cadd(v0, v2), a1 = csub(v0, v2), a2 = cadd(v1, v3);
  const float2 a3 = mul_si(csub(v1, v3), sign);
  v0 = cadd(a0, a2);
  v2 = csub(a0, a2);
  v1 = cadd(a1, a3);
  v3 = csub(a1, a3);
}

// e^{sign 2 pi i p / 16}, p = 0..9
__device__ __forceinline__ float2 w16(int p, float sign) {
  constexpr float c1 = 0.92387953251128674f, s1 = 0.38268343236508977f, c2 = 0.70710678118654752f;
  float2 w;
  switch (p) {
    case 0: w = make_float2(1.f, 0.f); break;
    case 1: w = make_float2(c1, s1); break;
    case 2: w = make_float2(c2, c2); break;
    case 3: w = make_float2(s1, c1); break;
    case 4: w = make_float2(0.f, 1.f); break;
    case 5: w = make_float2(-s1, c1); break;
    case 6: w = make_float2(-c2, c2); break;
    case 7: w = make_float2(-c1, s1); break;
    case 8: w = make_float2(-1.f, 0.f); break;
    default: w = make_float2(-c1, -s1); break;  // 9
  }
  w.y *= sign;
  return w;
}

template <int R>
__device__ __forceinline__ void dft(float2 (&v)[R], float sign);

template <>
__device__ __forceinline__ void dft<2>(float2 (&v)[2], float) {
  dft2(v[0], v[1]);
}

template <>
__device__ __forceinline__ void dft<4>(float2 (&v)[4], float sign) {
  dft4(v[0], v[1], v[2], v[3], sign);
}

template <>
__device__ __forceinline__ void dft<8>(float2 (&v)[8], float sign) {
  // even / odd halves, then X[k] = E[k] + W8^k O[k], X[k+4] = E[k] - W8^k O[k]
  dft4(v[0], v[2], v[4], v[6], sign);
  dft4(v[1], v[3], v[5], v[7], sign);
  float2 o[4] = {v[1], cmul(v[3], w16(2, sign)), mul_si(v[5], sign), cmul(v[7], w16(6, sign))};
  const float2 e[4] = {v[0], v[2], v[4], v[6]};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    v[k] = cadd(e[k], o[k]);
    v[k + 4] = csub(e[k], o[k]);
  }
}

template <>
__device__ __forceinline__ void dft<16>(float2 (&v)[16], float sign) {
  // F_e = DFT4(v[e], v[e+4], v[e+8], v[e+12]); X[k'+4q] = DFT4_e(W16^{e k'} F_e[k'])[q]
#pragma unroll
  for (int e = 0; e < 4; ++e) dft4(v[e], v[e + 4], v[e + 8], v[e + 12], sign);
  // v[e + 4k'] now holds F_e[k']
#pragma unroll
  for (int e = 1; e < 4; ++e)
#pragma unroll
    for (int k = 1; k < 4; ++k) v[e + 4 * k] = cmul(v[e + 4 * k], w16(e * k, sign));
  float2 x[16];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    float2 g0 = v[4 * k], g1 = v[1 + 4 * k], g2 = v[2 + 4 * k], g3 = v[3 + 4 * k];
    dft4(g0, g1, g2, g3, sign);
    x[k] = g0;
    x[k + 4] = g1;
    x[k + 8] = g2;
    x[k + 12] = g3;
  }
#pragma unroll
  for (int k = 0; k < 16; ++k) v[k] = x[k];
}

__device__ inline unsigned f2ord(float f) {
  const unsigned u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ inline float ord2f(unsigned o) {
  return __uint_as_float((o & 0x80000000u) ? (o & 0x7fffffffu) : ~o);
}

// q = (p - min) * (1 / (max - min)) as FP16 / BF16 bits (round to nearest even).
template <int Q>
__device__ inline unsigned short quantize16(float p, float lo, float inv) {
  const float q = (p - lo) * inv;
  if (Q == kStoreF16) return __half_as_ushort(__float2half_rn(q));
  const unsigned b = __float_as_uint(q);
  return (unsigned short)((b + 0x7fffu + ((b >> 16) & 1u)) >> 16);
}

// Crop, scale by 1/N and store one output sample pair (rows ra, ra+1 of the
// view) of the 16-bit modes.
template <int Q>
__device__ inline void store16(const FilterArgs& a, int view, int u, int ra, bool has_b, float fa,
                               float fb, float lo, float inv) {
  unsigned short* d = static_cast<unsigned short*>(static_cast<void*>(a.dst)) + view * a.dst_view;
  const unsigned short qa = quantize16<Q>(fa, lo, inv);
  const unsigned short qb = has_b ? quantize16<Q>(fb, lo, inv) : 0;
  if (a.transpose) {
    unsigned short* o = d + (long long)u * a.nrows + ra;
    if (has_b && (a.nrows & 1) == 0) {
      *reinterpret_cast<unsigned*>(o) = (unsigned)qa | ((unsigned)qb << 16);  // 4-byte aligned
    } else {
      o[0] = qa;
      if (has_b) o[1] = qb;
    }
  } else {
    d[(long long)ra * a.dst_pitch + u] = qa;
    if (has_b) d[(long long)(ra + 1) * a.dst_pitch + u] = qb;
  }
}

// Output side of the filter kernel: the 16-bit quantisation constants of the
// view and the running min/max of the values stored.
struct StoreCtx {
  float qlo, qinv, lo, hi;
};

__device__ __forceinline__ StoreCtx store_ctx(const FilterArgs& a, int view) {
  StoreCtx c{0.f, 0.f, INFINITY, -INFINITY};
  if (a.qmode == kStoreF16 || a.qmode == kStoreBF16) {
    c.qlo = ord2f(a.qmm[2 * view]);
    const float range = ord2f(a.qmm[2 * view + 1]) - c.qlo;
    c.qinv = range > 0.f ? 1.0f / range : 0.f;
  }
  return c;
}

// Widens a view's {min, max} words.  A look at the words first spares most of the
// atomics, which all waves of a view would queue up for (16 views of 2048^2 into FP16:
// 1.44 ms with an atomic a wave in the kernel this one replaced); a stale word only
// costs an atomic that changes nothing.
__device__ __forceinline__ void minmax_update(unsigned* mm, float lo, float hi) {
  const unsigned l = f2ord(lo), h = f2ord(hi);
  if (l < __hip_atomic_load(mm, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMin(mm, l);
  if (h > __hip_atomic_load(mm + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(mm + 1, h);
}

// Per-view min/max: a wave-level reduction, then one atomic per wave.
__device__ __forceinline__ void store_minmax(const FilterArgs& a, StoreCtx& c, int view) {
  if (!a.minmax) return;
  float lo = c.lo, hi = c.hi;
  for (int o = 32; o > 0; o >>= 1) {
    lo = fminf(lo, __shfl_xor(lo, o));
    hi = fmaxf(hi, __shfl_xor(hi, o));
  }
  if ((threadIdx.x & 63) == 0) minmax_update(a.minmax + 2 * view, lo, hi);
}

// Stores output sample u of rows ra (fa) and ra+1 (fb) in store mode Q's form
// and layout, and with MM tracks their min/max.
template <int Q, bool MM>
__device__ __forceinline__ void store_pair_q(const FilterArgs& a, StoreCtx& c, int view, int u, int ra,
                                             bool has_b, float fa, float fb) {
  if constexpr (Q == kStoreF16 || Q == kStoreBF16) {
    store16<Q>(a, view, u, ra, has_b, fa, fb, c.qlo, c.qinv);
  } else if constexpr (Q == kStoreF32) {
    float* d = a.dst + view * a.dst_view;
    if (a.transpose) {
      float* o = d + (long long)u * a.nrows + ra;
      if (has_b && (a.nrows & 1) == 0) {
        *reinterpret_cast<float2*>(o) = make_float2(fa, fb);  // 8-byte aligned: u*nrows + ra even
      } else {
        o[0] = fa;
        if (has_b) o[1] = fb;
      }
    } else {
      d[(long long)ra * a.dst_pitch + u] = fa;
      if (has_b) d[(long long)(ra + 1) * a.dst_pitch + u] = fb;
    }
  }
  if constexpr (MM) {
    c.lo = fminf(c.lo, has_b ? fminf(fa, fb) : fa);
    c.hi = fmaxf(c.hi, has_b ? fmaxf(fa, fb) : fa);
  }
}

// The same with the mode and min/max tracking chosen at run time.
__device__ __forceinline__ void store_pair(const FilterArgs& a, StoreCtx& c, int view, int u, int ra,
                                           bool has_b, float fa, float fb) {
  if (a.qmode == kStoreNone)
    store_pair_q<kStoreNone, true>(a, c, view, u, ra, has_b, fa, fb);
  else if (a.qmode == kStoreF16)
    store_pair_q<kStoreF16, true>(a, c, view, u, ra, has_b, fa, fb);
  else if (a.qmode == kStoreBF16)
    store_pair_q<kStoreBF16, true>(a, c, view, u, ra, has_b, fa, fb);
  else
    store_pair_q<kStoreF32, true>(a, c, view, u, ra, has_b, fa, fb);
}

// The other lengths (N < 128), 2^29 rows and more, and FDK_FILTER_FFT=inplace: the
// in-place bit-reversed radix-2^2 FFT, a block per row pair.
__global__ __launch_bounds__(256) void filter_rows_kernel(FilterArgs a) {
  extern __shared__ float2 buf[];
  const int view = blockIdx.y;
  // Row pairs remapped so that each XCD (hardware block b -> XCD b % 8) filters
  // a contiguous run of rows: the 8-byte transposed stores of neighbouring
  // pairs then meet in one L2 and leave it as whole lines.
  const unsigned gx = gridDim.x;
  const unsigned bx = (gx % 8u == 0u) ? (blockIdx.x % 8u) * (gx / 8u) + blockIdx.x / 8u : blockIdx.x;
  const int ra = 2 * (int)bx, rb = ra + 1;
  const bool has_b = rb < a.nrows;
  const float* sa = a.src + view * a.src_view + (long long)ra * a.src_pitch;
  const float* sb = sa + a.src_pitch;
  const float* ca = a.cos_table ? a.cos_table + (long long)ra * a.nu : nullptr;
  const float* cb = ca ? ca + a.nu : nullptr;
  const int off = (a.N - a.nu) >> 1;
  const int nu = a.nu;

  // Edge means of the cos-weighted rows (FilterLib.h:37-46 forms mean4 in
  // float; the mean3 variants of type.h:4202-4205 in double).
  float la = 0.f, lb = 0.f, rra = 0.f, rrb = 0.f;
  if (a.pad == FDK_PAD_MEAN4 || a.pad == FDK_PAD_MEAN3) {
    const int k = a.pad;
    float xa[8], xb[8];
    for (int q = 0; q < k; ++q) {
      const int il = q, ir = nu - 1 - q;
      xa[q] = sa[il] * (ca ? ca[il] : 1.f);
      xa[4 + q] = sa[ir] * (ca ? ca[ir] : 1.f);
      xb[q] = has_b ? sb[il] * (cb ? cb[il] : 1.f) : 0.f;
      xb[4 + q] = has_b ? sb[ir] * (cb ? cb[ir] : 1.f) : 0.f;
    }
    if (k == 4) {
      la = (xa[0] + xa[1] + xa[2] + xa[3]) / 4;
      rra = (xa[4] + xa[5] + xa[6] + xa[7]) / 4;
      lb = (xb[0] + xb[1] + xb[2] + xb[3]) / 4;
      rrb = (xb[4] + xb[5] + xb[6] + xb[7]) / 4;
    } else {
      la = (float)(((double)xa[0] + xa[1] + xa[2]) / 3);
      rra = (float)(((double)xa[4] + xa[5] + xa[6]) / 3);
      lb = (float)(((double)xb[0] + xb[1] + xb[2]) / 3);
      rrb = (float)(((double)xb[4] + xb[5] + xb[6]) / 3);
    }
  }
  for (int n = threadIdx.x; n < a.N; n += blockDim.x) {
    const int p = n - off;
    float va, vb;
    if (p < 0) { va = la; vb = lb; }
    else if (p >= nu) { va = rra; vb = rrb; }
    else {
      va = sa[p] * (ca ? ca[p] : 1.f);
      vb = has_b ? sb[p] * (cb ? cb[p] : 1.f) : 0.f;
    }
    buf[brev_n(n, a.logN)] = make_float2(va, vb);
  }
  __syncthreads();
  {
    fft_lds(buf, a.tw, a.N, a.logN, -1.f);
    // Filter multiply fused with the bit-reversal permutation of the inverse pass.
    for (int k = threadIdx.x; k < a.N; k += blockDim.x) {
      const unsigned r = brev_n(k, a.logN);
      if ((unsigned)k < r) {
        const float2 xk = buf[k], xr = buf[r];
        const float hk = a.H[k], hr = a.H[r];
        buf[k] = make_float2(xr.x * hr, xr.y * hr);
        buf[r] = make_float2(xk.x * hk, xk.y * hk);
      } else if ((unsigned)k == r) {
        const float hk = a.H[k];
        buf[k] = make_float2(buf[k].x * hk, buf[k].y * hk);
      }
    }
    __syncthreads();
    fft_lds(buf, a.tw, a.N, a.logN, 1.f);
  }
  const float inv = 1.0f / (float)a.N;
  StoreCtx sc = store_ctx(a, view);
  for (int u = threadIdx.x; u < nu; u += blockDim.x) {
    const float2 c = buf[off + u];
    store_pair(a, sc, view, u, ra, has_b, c.x * inv, c.y * inv);
  }
  store_minmax(a, sc, view);
}

// ------------------------------------------------------------ row filter, 16 points a thread
// filter_wide_kernel: T = N / 16 threads hold a row pair, 16 points each: point
// t + T i of thread t, i < 16.  Radices 16, 16, then N / 256 as one or two passes (16
// and 8 at N = 128).  In every pass a thread's inputs are its points t + T i, so
//  * forward, a pass reads them, twiddles, transforms and writes the self-sorted order;
//  * the inverse is the forward passes' adjoint in reverse order: read what the pass
//    wrote, conjugate transform, conjugate twiddles, write to t + T i.  It needs the
//    same twiddles in the same threads, and the last pass's outputs, the filter
//    multiply and the first adjoint's inputs are the same registers, as are the points
//    loaded and the points stored.
// A block keeps to its rows' place and walks over many pairs, so what depends on the
// thread alone is loaded once: H / N and the third and fourth pass's twiddles in
// registers, the second pass's 16 x 15 in LDS.  QUAD: two pairs in lockstep (half the
// barriers, twice the independent work), their transposed outputs one 16-byte store a
// point.  An XCD takes an eighth of the rows (32 at least) of one view, then of the next:
// the cos-table rows stay in its L2, and the stores of neighbouring rows meet there as
// lines.
//
// What bounds it: at 200 registers and 2 waves per SIMD vector issue is half the time
// (330 us of 600 at the size below), the rest LDS exchanges, barriers and the transposed
// stores (60 us; 220 us as 8-byte stores of a pair).  The form it replaces (256 threads a
// pair whatever N, twiddles and H loaded for every pair) kept the texture-address unit
// busy 90 % of the time: 60 strided twiddle loads, 64 row and cos loads of which half are
// pads, 32 loads of edge samples and 8 scattered stores a thread.  Measured, 32 views of
// 2048^2 transposed: 916 -> 598 us (row-major 765 -> 540); 32 of 1000^2 241 -> 90; 8 of
// 4096^2 into FP16 1900 -> 1025; 32 of 500 x 300 row-major 26 -> 19; one of 9000^2 (was in
// place) 2425 -> 782, although the 1024 threads of N = 16384 have 128 registers each and
// spill 114 (460 bytes a thread).
// Small calls: a launch costs 10.5 us whatever it does, and a wave's chain of loads and
// passes has to fit in that.  So rows that lie side by side in a wave (N < 1024) are
// loaded without branches, all 8 slices in flight (4 views of 500 x 300, N = 512, 14.3 us
// with a branch a point, 10.9), and few pairs get blocks of one or two (one view of 2000
// x 128 12.3 -> 10.5, two of 768^2 13.8 -> 12.1).
typedef unsigned u32x2_t __attribute__((ext_vector_type(2)));
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));

template <int M>
struct Wide {
  static constexpr int N = 1 << M, T = N / 16;
  static constexpr int THREADS = T > 256 ? T : 256, SMALL = T > 64 ? T : 64;  // of a block
  static constexpr int R2 = M == 7 ? 8 : 16;
  static constexpr int R3 = M <= 8 ? 1 : M >= 12 ? 16 : N / 256;
  static constexpr int R4 = M >= 13 ? N / 4096 : 1;
  static constexpr int SLOTS = N + N / 16;  // LDS points of a pair, one spare per 16
  static constexpr int TW2 = (R2 - 1) * 16;
  static constexpr size_t lds(bool quad, int pairs) {
    return sizeof(float2) * ((quad ? 2 : 1) * pairs * SLOTS + TW2);
  }
};

// Twiddles e^{-2 pi i k r / (NS R)} of a thread's 16 / R butterflies, r = 1 .. R-1.
template <int M, int R, int NS>
struct WideTw {
  static constexpr int B = 16 / R;
  float2 w[R > 1 ? B * (R - 1) : 1];
  __device__ __forceinline__ void load(const float2* __restrict__ tw, int t) {
    if constexpr (R > 1) {
#pragma unroll
      for (int q = 0; q < B; ++q) {
        const int k = (t + q * Wide<M>::T) & (NS - 1);
#pragma unroll
        for (int r = 1; r < R; ++r) w[q * (R - 1) + r - 1] = tw[k * r * (Wide<M>::N / (NS * R))];
      }
    }
  }
};

__device__ __forceinline__ float2 cmul_conj(float2 a, float2 w) {  // a * conj(w)
  return make_float2(a.x * w.x + a.y * w.y, a.y * w.x - a.x * w.y);
}

// The radix-R DFTs of a thread's points x[q + B r].
template <int R, bool INV>
__device__ __forceinline__ void wide_dft(float2 (&x)[16]) {
  constexpr int B = 16 / R;
#pragma unroll
  for (int q = 0; q < B; ++q) {
    float2 v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = x[q + B * r];
    dft<R>(v, INV ? 1.f : -1.f);
#pragma unroll
    for (int r = 0; r < R; ++r) x[q + B * r] = v[r];
  }
}

// LDS slot of point t + T i, and of output r of butterfly j = t + T q of a pass.
template <int M>
__device__ __forceinline__ int wide_own(int t, int i) {
  constexpr int T = Wide<M>::T;
  return T % 16 == 0 ? t + (t >> 4) + i * (T + T / 16) : (t + T * i) + ((t + T * i) >> 4);
}
template <int M, int R, int NS>
__device__ __forceinline__ int wide_out(int t, int q, int r) {
  const int j = t + Wide<M>::T * q, k = j & (NS - 1), o = (j - k) * R + k;
  if constexpr (NS == 1) return o + (o >> 4) + r;  // R = 16: one 16-point run
  else if constexpr (NS % 16 == 0) return o + (o >> 4) + r * (NS + NS / 16);
  else return (o + r * NS) + ((o + r * NS) >> 4);
}

template <int M, int R, int NS>
__device__ __forceinline__ void wide_put(float2* buf, const float2 (&x)[16], int t) {
  constexpr int B = 16 / R;
#pragma unroll
  for (int q = 0; q < B; ++q)
#pragma unroll
    for (int r = 0; r < R; ++r) buf[wide_out<M, R, NS>(t, q, r)] = x[q + B * r];
}
template <int M, int R, int NS>
__device__ __forceinline__ void wide_get(const float2* buf, float2 (&x)[16], int t) {
  constexpr int B = 16 / R;
#pragma unroll
  for (int q = 0; q < B; ++q)
#pragma unroll
    for (int r = 0; r < R; ++r) x[q + B * r] = buf[wide_out<M, R, NS>(t, q, r)];
}
template <int M>
__device__ __forceinline__ void wide_put_own(float2* buf, const float2 (&x)[16], int t) {
#pragma unroll
  for (int i = 0; i < 16; ++i) buf[wide_own<M>(t, i)] = x[i];
}
template <int M>
__device__ __forceinline__ void wide_get_own(const float2* buf, float2 (&x)[16], int t) {
#pragma unroll
  for (int i = 0; i < 16; ++i) x[i] = buf[wide_own<M>(t, i)];
}

template <int R, bool INV>
__device__ __forceinline__ void wide_twiddle(float2 (&x)[16], const float2* w) {
  constexpr int B = 16 / R;
#pragma unroll
  for (int q = 0; q < B; ++q)
#pragma unroll
    for (int r = 1; r < R; ++r) {
      const float2 f = w[q * (R - 1) + r - 1];
      x[q + B * r] = INV ? cmul_conj(x[q + B * r], f) : cmul(x[q + B * r], f);
    }
}

// The second pass's twiddles from LDS: tw2[(r - 1) 16 + k].
template <int M, bool INV>
__device__ __forceinline__ void wide_twiddle2(float2 (&x)[16], const float2* tw2, int t) {
  constexpr int R = Wide<M>::R2, B = 16 / R;
#pragma unroll
  for (int q = 0; q < B; ++q) {
    const int k = (t + q * Wide<M>::T) & 15;
#pragma unroll
    for (int r = 1; r < R; ++r) {
      const float2 f = tw2[(r - 1) * 16 + k];
      x[q + B * r] = INV ? cmul_conj(x[q + B * r], f) : cmul(x[q + B * r], f);
    }
  }
}

// Lane k of the thread's group of min(T, 64) lanes.
template <int T>
__device__ __forceinline__ float wide_lane(float v, int k) {
  if constexpr (T >= 64) return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), k));
  else return __shfl(v, k, T);
}

// The 16 points of a pair's rows (t + T i: sample t + T i - off), cos-weighted, the
// points left and right of the row set to the pads.  Loads past a resource's end read
// 0, so no address is clamped; slices that hold no sample are not loaded.
template <int M>
__device__ __forceinline__ void wide_load(const FilterArgs& a, const float* sa, const float* sb,
                                          const float* ca, const float* cb, bool live, bool has_b,
                                          int t, int off, float2 (&x)[16]) {
  constexpr int T = Wide<M>::T;
  const int nu = a.nu, row_bytes = nu * 4, kpad = a.pad;
  // Row a and b and their cos rows: resources of the rows where a wave has one pair,
  // clamped addresses where it has several (the rows differ between lanes; sa and sb are
  // rows of the view also where there is no pair, and what is read there is not used).
  const int na = live ? row_bytes : 0, nb = has_b ? row_bytes : 0;
  const __amdgpu_buffer_rsrc_t rxa = __builtin_amdgcn_make_buffer_rsrc((void*)sa, 0, na, fdk::kRawRsrcWord3);
  const __amdgpu_buffer_rsrc_t rxb = __builtin_amdgcn_make_buffer_rsrc((void*)sb, 0, nb, fdk::kRawRsrcWord3);
  const __amdgpu_buffer_rsrc_t rca = __builtin_amdgcn_make_buffer_rsrc((void*)ca, 0, ca ? na : 0, fdk::kRawRsrcWord3);
  const __amdgpu_buffer_rsrc_t rcb = __builtin_amdgcn_make_buffer_rsrc((void*)cb, 0, cb ? nb : 0, fdk::kRawRsrcWord3);
  const auto ld = [&](__amdgpu_buffer_rsrc_t r, const float* row, int p) {
    if constexpr (T >= 64) return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, p * 4, 0, 0));
    else return row[p];
  };
  float ea = 0.f, eb = 0.f;  // lanes 0..3: samples 0..3, lanes 4..7: nu-1 .. nu-4
  if (kpad) {
    const int l = threadIdx.x & 7, e = l < 4 ? l : nu + 3 - l;
    ea = ld(rxa, sa, e);
    eb = ld(rxb, sb, e);
    if (ca) {
      ea *= ld(rca, ca, e);
      eb *= ld(rcb, cb, e);
    }
  }
#pragma unroll
  for (int c = 0; c < 16; c += 8) {  // 8 slices in flight
    float xa[8], xb[8], wa[8], wb[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int lo = T * (c + i) - off;
      xa[i] = xb[i] = 0.f;
      wa[i] = wb[i] = 1.f;
      if (lo + T > 0 && lo < nu) {
        const int p = T >= 64 ? t + lo : min(max(t + lo, 0), nu - 1);
        xa[i] = ld(rxa, sa, p);
        xb[i] = ld(rxb, sb, p);
        if (ca) {
          wa[i] = ld(rca, ca, p);
          wb[i] = ld(rcb, cb, p);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      x[c + i] = make_float2(xa[i] * wa[i], xb[i] * wb[i]);
      if constexpr (T < 64) {  // nothing outside the row or in a row that does not exist
        const int p = t + T * (c + i) - off;
        const bool in = p >= 0 && p < nu;
        x[c + i].x = live && in ? x[c + i].x : 0.f;
        x[c + i].y = has_b && in ? x[c + i].y : 0.f;
      }
    }
  }
  if (kpad == 0) return;
  if constexpr (T < 64) {
    ea = live ? ea : 0.f;
    eb = has_b ? eb : 0.f;
  }
  const auto at = [&](float v, int k) { return wide_lane<T>(v, k); };
  float la, lb, ra, rb;
  if (kpad == 4) {
    la = (at(ea, 0) + at(ea, 1) + at(ea, 2) + at(ea, 3)) / 4;
    ra = (at(ea, 4) + at(ea, 5) + at(ea, 6) + at(ea, 7)) / 4;
    lb = (at(eb, 0) + at(eb, 1) + at(eb, 2) + at(eb, 3)) / 4;
    rb = (at(eb, 4) + at(eb, 5) + at(eb, 6) + at(eb, 7)) / 4;
  } else {
    la = (float)(((double)at(ea, 0) + at(ea, 1) + at(ea, 2)) / 3);
    ra = (float)(((double)at(ea, 4) + at(ea, 5) + at(ea, 6)) / 3);
    lb = (float)(((double)at(eb, 0) + at(eb, 1) + at(eb, 2)) / 3);
    rb = (float)(((double)at(eb, 4) + at(eb, 5) + at(eb, 6)) / 3);
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int lo = T * i - off;
    if (lo < 0 || lo + T > nu) {
      if (t + lo < 0) x[i] = make_float2(la, lb);
      else if (t + lo >= nu) x[i] = make_float2(ra, rb);
    }
  }
}

// Min/max of the lanes of one pair (all of a wave, or groups of T lanes).
template <int T>
__device__ __forceinline__ void wide_minmax(const FilterArgs& a, StoreCtx& c, int view, int t) {
  constexpr int L = T < 64 ? T : 64;
  float lo = c.lo, hi = c.hi;
#pragma unroll
  for (int o = L / 2; o > 0; o >>= 1) {
    lo = fminf(lo, __shfl_xor(lo, o, L));
    hi = fmaxf(hi, __shfl_xor(hi, o, L));
  }
  if ((t & (L - 1)) == 0) minmax_update(a.minmax + 2 * view, lo, hi);
}

// Stores the 16 points, cropped.  FP32 goes through a resource of the view (transposed)
// or the row: points outside the row fall outside it and are dropped.  Where their
// offsets could wrap into the view (a.far) each point is checked instead.
template <int M, int Q, bool MM, bool FAR = false>
__device__ __forceinline__ void wide_store(const FilterArgs& a, int view, int ra, bool live, bool has_b,
                                           int t, int off, const float2 (&x)[16]) {
  constexpr int T = Wide<M>::T;
  StoreCtx c = store_ctx(a, view);
  if constexpr (Q == kStoreF32 && T >= 64 && !FAR) {
    float* d = a.dst + view * a.dst_view;
    if (a.transpose) {
      const __amdgpu_buffer_rsrc_t rd = __builtin_amdgcn_make_buffer_rsrc(
          (void*)d, 0, live ? a.nu * a.nrows * 4 : 0, fdk::kRawRsrcWord3);
      const int o0 = (int)(((unsigned)(t - off) * a.nrows + ra) * 4u);  // wraps outside the row
      const bool both = has_b && (a.nrows & 1) == 0;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int lo = T * i - off;
        if (lo + T <= 0 || lo >= a.nu) continue;
        const int o = (int)((unsigned)o0 + (unsigned)(i * T * 4) * a.nrows);
        if (both) {
          __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2_t, x[i]), rd, o, 0, 0);
        } else {
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x[i].x), rd, o, 0, 0);
          // (t + lo >= 0: the row above must not take a value for the one below)
          if (has_b && t + lo >= 0 && t + lo < a.nu)
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x[i].y), rd, o + 4, 0, 0);
        }
      }
    } else {
      float* row = d + (long long)ra * a.dst_pitch;
      const __amdgpu_buffer_rsrc_t rda =
          __builtin_amdgcn_make_buffer_rsrc((void*)row, 0, live ? a.nu * 4 : 0, fdk::kRawRsrcWord3);
      const __amdgpu_buffer_rsrc_t rdb = __builtin_amdgcn_make_buffer_rsrc(
          (void*)(row + a.dst_pitch), 0, has_b ? a.nu * 4 : 0, fdk::kRawRsrcWord3);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int lo = T * i - off;
        if (lo + T <= 0 || lo >= a.nu) continue;
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x[i].x), rda, (t + lo) * 4, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x[i].y), rdb, (t + lo) * 4, 0, 0);
      }
    }
    if constexpr (MM) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int u = t + T * i - off;
        if (live && u >= 0 && u < a.nu) {
          c.lo = fminf(c.lo, has_b ? fminf(x[i].x, x[i].y) : x[i].x);
          c.hi = fmaxf(c.hi, has_b ? fmaxf(x[i].x, x[i].y) : x[i].x);
        }
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int u = t + T * i - off;
      if (live && u >= 0 && u < a.nu) store_pair_q<Q, MM>(a, c, view, u, ra, has_b, x[i].x, x[i].y);
    }
  }
  if constexpr (MM)
    if (live) wide_minmax<T>(a, c, view, t);
}

// The outputs of rows ra, ra+1 (w) and ra+2, ra+3 (x), transposed: one 16-byte store a
// point.
template <int M, bool MM>
__device__ __forceinline__ void wide_store4(const FilterArgs& a, int view, int ra, bool live, int t, int off,
                                            const float2 (&w)[16], const float2 (&x)[16]) {
  constexpr int T = Wide<M>::T;
  const int left = live ? a.nrows - ra : 0;  // rows of the four that exist
  if (left <= 0) return;
  float* d = a.dst + view * a.dst_view + ra;
  const int bytes = a.nu * a.nrows * 4 - ra * 4;
  StoreCtx c = store_ctx(a, view);
  const unsigned o0 = (unsigned)(t - off) * a.nrows * 4u;  // wraps outside the row
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int lo = T * i - off;
    if (lo + T <= 0 || lo >= a.nu) continue;
    const float2 y = w[i];
    const int o = (int)(o0 + (unsigned)(i * T * 4) * a.nrows);
    const bool in = t + lo >= 0 && t + lo < a.nu;
    if constexpr (T >= 64) {
      const __amdgpu_buffer_rsrc_t rd = __builtin_amdgcn_make_buffer_rsrc((void*)d, 0, bytes, fdk::kRawRsrcWord3);
      if (left >= 4) {  // outside the row the offset is negative or past the view: dropped
        const u32x4_t v = {__float_as_uint(y.x), __float_as_uint(y.y), __float_as_uint(x[i].x),
                           __float_as_uint(x[i].y)};
        __builtin_amdgcn_raw_buffer_store_b128(v, rd, o, 0, 0);
      } else if (in) {
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y.x), rd, o, 0, 0);
        if (left > 1) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y.y), rd, o + 4, 0, 0);
        if (left > 2) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x[i].x), rd, o + 8, 0, 0);
      }
    } else if (in) {
      float* q = d + (long long)(t + lo) * a.nrows;
      if (left >= 4) {
        typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
        *reinterpret_cast<f32x4_a4*>(q) = f32x4_a4{y.x, y.y, x[i].x, x[i].y};
      } else {
        q[0] = y.x;
        if (left > 1) q[1] = y.y;
        if (left > 2) q[2] = x[i].x;
      }
    }
    if (MM && in) {
      c.lo = fminf(c.lo, y.x);
      c.hi = fmaxf(c.hi, y.x);
      if (left > 1) c.lo = fminf(c.lo, y.y), c.hi = fmaxf(c.hi, y.y);
      if (left > 2) c.lo = fminf(c.lo, x[i].x), c.hi = fmaxf(c.hi, x[i].x);
      if (left > 3) c.lo = fminf(c.lo, x[i].y), c.hi = fmaxf(c.hi, x[i].y);
    }
  }
  if constexpr (MM) wide_minmax<T>(a, c, view, t);
}

struct WideGrid {
  int items, chunk;  // row quads in all (the last group padded), quads of one XCD
  int nviews, group;
};

template <int M, bool QUAD, int THREADS>
__global__ __launch_bounds__(THREADS, (M == 14 ? 4 : 2)) void filter_wide_kernel(FilterArgs a, WideGrid g) {
  using W = Wide<M>;
  constexpr int PB = THREADS / W::T;  // row pairs (or quads) per block
  constexpr int N = W::N, T = W::T, R2 = W::R2, R3 = W::R3, R4 = W::R4;
  constexpr int P = QUAD ? 2 : 1, ROWS = 2 * P;  // row pairs and rows of an item
  extern __shared__ float2 wide_lds[];
  const int t = threadIdx.x & (T - 1);
  const int sub = T >= 64 ? __builtin_amdgcn_readfirstlane(threadIdx.x / T) : (int)threadIdx.x / T;
  float2* tw2 = wide_lds;
  float2* buf[P];
#pragma unroll
  for (int p = 0; p < P; ++p) buf[p] = wide_lds + W::TW2 + (sub * P + p) * W::SLOTS;
  for (int k = threadIdx.x; k < W::TW2; k += THREADS)
    tw2[k] = a.tw[(k & 15) * (k / 16 + 1) * (N / (16 * R2))];
  WideTw<M, R3, 256> tw3;
  tw3.load(a.tw, t);
  WideTw<M, R4, 4096> tw4;
  tw4.load(a.tw, t);
  float h[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) h[i] = a.H[t + T * i] * (1.0f / N);  // exact: N is a power of two
  const int off = (N - a.nu) >> 1;
  const int nsets = (a.nrows + ROWS - 1) / ROWS, per_group = g.nviews * g.group;
  // (the first barrier below also covers tw2)

  // XCD x (block % 8) walks items [x chunk, (x + 1) chunk)
  const int xcd = blockIdx.x % 8u, stride = (int)(gridDim.x / 8u) * PB;
  const int end = min(g.items, (xcd + 1) * g.chunk);
  for (int it0 = xcd * g.chunk + (int)(blockIdx.x / 8u) * PB; it0 < end; it0 += stride) {
    const int it = it0 + sub;
    const int grp = it / per_group, in = it - grp * per_group;
    const int set = grp * g.group + in % g.group;
    const bool live = it < end && set < nsets;  // others only take part in the barriers
    const int view = live ? in / g.group : 0, ra = live ? ROWS * set : 0;
    float2 x[P][16];
#define WIDE_EACH _Pragma("unroll") for (int p = 0; p < P; ++p)
    WIDE_EACH {
      const int r = ra + 2 * p;
      const bool has_a = live && r < a.nrows, has_b = live && r + 1 < a.nrows;
      const float* sa = a.src + view * a.src_view + (long long)(has_a ? r : 0) * a.src_pitch;
      const float* ca = a.cos_table ? a.cos_table + (long long)(has_a ? r : 0) * a.nu : nullptr;
      wide_load<M>(a, sa, has_b ? sa + a.src_pitch : sa, ca, ca && has_b ? ca + a.nu : ca, has_a, has_b, t, off,
                   x[p]);
    }
    WIDE_EACH {
      wide_dft<16, false>(x[p]);
      wide_put<M, 16, 1>(buf[p], x[p], t);
    }
    __syncthreads();
    WIDE_EACH {
      wide_get_own<M>(buf[p], x[p], t);
      wide_twiddle2<M, false>(x[p], tw2, t);
      wide_dft<R2, false>(x[p]);
    }
    if constexpr (R3 > 1) {
      __syncthreads();
      WIDE_EACH wide_put<M, R2, 16>(buf[p], x[p], t);
      __syncthreads();
      WIDE_EACH {
        wide_get_own<M>(buf[p], x[p], t);
        wide_twiddle<R3, false>(x[p], tw3.w);
        wide_dft<R3, false>(x[p]);
        }
    }
    if constexpr (R4 > 1) {
      __syncthreads();
      WIDE_EACH wide_put<M, R3, 256>(buf[p], x[p], t);
      __syncthreads();
      WIDE_EACH {
        wide_get_own<M>(buf[p], x[p], t);
        wide_twiddle<R4, false>(x[p], tw4.w);
        wide_dft<R4, false>(x[p]);
      }
    }
    // The filter, then the adjoints; a thread writes only the points it alone has read
    // last, so the first needs no barrier before its writes.
    WIDE_EACH {
#pragma unroll
      for (int i = 0; i < 16; ++i) x[p][i] = make_float2(x[p][i].x * h[i], x[p][i].y * h[i]);
    }
    if constexpr (R4 > 1) {
      WIDE_EACH {
        wide_dft<R4, true>(x[p]);
        wide_twiddle<R4, true>(x[p], tw4.w);
        wide_put_own<M>(buf[p], x[p], t);
      }
      __syncthreads();
      WIDE_EACH wide_get<M, R3, 256>(buf[p], x[p], t);
      __syncthreads();
    }
    if constexpr (R3 > 1) {
      WIDE_EACH {
        wide_dft<R3, true>(x[p]);
        wide_twiddle<R3, true>(x[p], tw3.w);
        wide_put_own<M>(buf[p], x[p], t);
        }
      __syncthreads();
      WIDE_EACH wide_get<M, R2, 16>(buf[p], x[p], t);
      __syncthreads();
    }
    WIDE_EACH {
      wide_dft<R2, true>(x[p]);
      wide_twiddle2<M, true>(x[p], tw2, t);
      wide_put_own<M>(buf[p], x[p], t);
    }
    __syncthreads();
    WIDE_EACH {
      wide_get<M, 16, 1>(buf[p], x[p], t);
      wide_dft<16, true>(x[p]);
    }
#undef WIDE_EACH
    const bool has_b = live && ra + 1 < a.nrows;
    if constexpr (QUAD) {
      if (a.minmax) wide_store4<M, true>(a, view, ra, live, t, off, x[0], x[1]);
      else wide_store4<M, false>(a, view, ra, live, t, off, x[0], x[1]);
    } else if (a.qmode == kStoreNone) {
      wide_store<M, kStoreNone, true>(a, view, ra, live, has_b, t, off, x[0]);
    } else if (a.qmode == kStoreF16) {
      wide_store<M, kStoreF16, false>(a, view, ra, live, has_b, t, off, x[0]);
    } else if (a.qmode == kStoreBF16) {
      wide_store<M, kStoreBF16, false>(a, view, ra, live, has_b, t, off, x[0]);
    } else if (a.far) {
      if (a.minmax) wide_store<M, kStoreF32, true, true>(a, view, ra, live, has_b, t, off, x[0]);
      else wide_store<M, kStoreF32, false, true>(a, view, ra, live, has_b, t, off, x[0]);
    } else if (a.minmax) {
      wide_store<M, kStoreF32, true>(a, view, ra, live, has_b, t, off, x[0]);
    } else {
      wide_store<M, kStoreF32, false>(a, view, ra, live, has_b, t, off, x[0]);
    }
    __syncthreads();  // the last reads are done
  }
}

// FP32 staging -> FP16/BF16 with q = (p - min) / (max - min) per view, four
// samples per thread per step (16-byte loads, 8-byte stores) when the view
// size and both view strides are multiples of 4 (VEC), else one.
template <int DT, bool VEC>
__global__ __launch_bounds__(256) void quantize_kernel(const float* __restrict__ src, long long sview,
                                                       void* dst, long long dview, long long n,
                                                       const unsigned* minmax) {
  constexpr int Q = DT == FDK_F16 ? kStoreF16 : kStoreBF16;
  const int view = blockIdx.y;
  const float lo = ord2f(minmax[2 * view]), hi = ord2f(minmax[2 * view + 1]);
  const float range = hi - lo;
  const float inv = range > 0.f ? 1.0f / range : 0.f;
  const float* s = src + view * sview;
  unsigned short* d = static_cast<unsigned short*>(dst) + view * dview;
  const long long stride = (long long)gridDim.x * 256;
  if (VEC) {
    for (long long i = blockIdx.x * 256LL + threadIdx.x; 4 * i < n; i += stride) {
      const float4 p = reinterpret_cast<const float4*>(s)[i];
      const unsigned w0 = (unsigned)quantize16<Q>(p.x, lo, inv) | ((unsigned)quantize16<Q>(p.y, lo, inv) << 16);
      const unsigned w1 = (unsigned)quantize16<Q>(p.z, lo, inv) | ((unsigned)quantize16<Q>(p.w, lo, inv) << 16);
      reinterpret_cast<uint2*>(d)[i] = make_uint2(w0, w1);
    }
  } else {
    for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += stride)
      d[i] = quantize16<Q>(s[i], lo, inv);
  }
}

__global__ void minmax_init_kernel(unsigned* mm, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    mm[2 * i] = 0xffffffffu;
    mm[2 * i + 1] = 0u;
  }
}

__global__ void correct_kernel(const float* __restrict__ src, const float* __restrict__ table,
                               float* dst, int width, int height, int pitch, int tpitch) {
  const int x = blockIdx.x * 64 + threadIdx.x;
  const int y = blockIdx.y * 4 + threadIdx.y;
  const int z = blockIdx.z;
  if (x >= width || y >= height) return;
  const long long o = ((long long)z * height + y) * pitch + x;
  dst[o] = src[o] * table[(long long)y * tpitch + x];
}

// Twiddles e^{-2 pi i k / N}, k < N, evaluated in FP64 and rounded to float.
__global__ void twiddle_kernel(float2* tw, int N) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < N) {
    const double a = -2.0 * 3.141592653589793238462 * k / N;
    tw[k] = make_float2((float)cos(a), (float)sin(a));
  }
}

void launch_twiddles(float2* tw, int N, hipStream_t st) {
  hipLaunchKernelGGL(twiddle_kernel, dim3((N + 255) / 256), dim3(256), 0, st, tw, N);
}

// Device twiddle tables, one per (device, N), built on the first use and kept
// for the life of the process.
std::mutex g_tw_mutex;
std::map<std::pair<int, int>, float2*> g_tw;

int twiddles(int N, const float2** out) {
  int dev = 0;
  FDK_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(g_tw_mutex);
  auto it = g_tw.find({dev, N});
  if (it != g_tw.end()) {
    *out = it->second;
    return FDK_OK;
  }
  float2* d = nullptr;
  FDK_HIP(fdk::dev_malloc((void**)&d, sizeof(float2) * N));
  hipStream_t st = nullptr;
  FDK_HIP(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
  launch_twiddles(d, N, st);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  (void)hipStreamDestroy(st);
  if (e != hipSuccess) {
    (void)hipFree(d);
    return fdk::fail(FDK_ERR_HIP, "twiddle table: %s", hipGetErrorString(e));
  }
  g_tw[{dev, N}] = d;
  *out = d;
  return FDK_OK;
}

float host_ord2f(unsigned o) {
  const unsigned u = (o & 0x80000000u) ? (o & 0x7fffffffu) : ~o;
  float f;
  std::memcpy(&f, &u, sizeof(f));
  return f;
}

int log2_exact(int N) {
  int m = 0;
  while ((1 << m) < N) ++m;
  return (1 << m) == N ? m : -1;
}

// 1: filter_wide_kernel where it applies (default); FDK_FILTER_FFT=inplace keeps the
// in-place radix-2^2 FFT for every length.
int fft_choice() {
  static const int k = [] {
    const char* e = std::getenv("FDK_FILTER_FFT");
    return (e && std::strcmp(e, "inplace") == 0) ? 0 : 1;
  }();
  return k;
}

// Blocks per CU that the LDS and the registers (2 waves per SIMD; 4 at M = 14, whose
// block has 16 waves) allow.
template <int M, int THREADS>
constexpr int wide_resident() { return M <= 12 ? 512 / THREADS : 1; }

template <int M, bool QUAD, int THREADS>
int launch_wide_sets(const FilterArgs& a, int nviews, hipStream_t st) {
  using W = Wide<M>;
  constexpr int ROWS = QUAD ? 4 : 2, PB = THREADS / W::T;
  const int nsets = (a.nrows + ROWS - 1) / ROWS;
  const int group = std::max(32 / ROWS, (nsets + 7) / 8);  // 32 rows fill a 128-byte line
  const long long items = (long long)((nsets + group - 1) / group) * group * nviews;
  const long long chunk = ((items + 7) / 8 + PB - 1) / PB * PB;
  const long long per_xcd = std::min<long long>(chunk / PB, 32 * wide_resident<M, THREADS>());
  const WideGrid g{(int)items, (int)chunk, nviews, group};
  const void* fn = reinterpret_cast<const void*>(&filter_wide_kernel<M, QUAD, THREADS>);
  const size_t lds = W::lds(QUAD, PB);
  if (lds > 64 * 1024) FDK_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  hipLaunchKernelGGL((filter_wide_kernel<M, QUAD, THREADS>), dim3((unsigned)(8 * per_xcd)), dim3(THREADS), lds, st, a, g);
  FDK_HIP(hipGetLastError());
  return FDK_OK;
}

template <int M>
int launch_wide(const FilterArgs& a, int nviews, hipStream_t st) {
  using W = Wide<M>;
  const long long pairs = (long long)((a.nrows + 1) / 2) * nviews, waves = pairs * W::T / 64;
  if constexpr (M <= 13)
    if (a.transpose && a.qmode == kStoreF32 && !a.far && waves >= 4096)
      return launch_wide_sets<M, true, W::THREADS>(a, nviews, st);
  // Below two blocks a CU the pairs of a block of 256 threads would share a CU and leave
  // others idle.
  if constexpr (W::SMALL < W::THREADS)
    if (pairs * W::T / W::THREADS < 512) return launch_wide_sets<M, false, W::SMALL>(a, nviews, st);
  return launch_wide_sets<M, false, W::THREADS>(a, nviews, st);
}

int launch_filter(FilterArgs& a, int nviews, hipStream_t st) {
  FDK_REQUIRE(a.N >= 16 && a.N <= 16384 && log2_exact(a.N) > 0, "filter length %d must be a power of two in 16..16384", a.N);
  FDK_REQUIRE(a.nu >= 4 && a.nu <= a.N, "row length %d must be in 4..N (%d)", a.nu, a.N);
  FDK_REQUIRE(a.pad == FDK_PAD_ZERO || a.pad == FDK_PAD_MEAN3 || a.pad == FDK_PAD_MEAN4,
              "pad_mode %d not in {0, 3, 4}", a.pad);
  FDK_REQUIRE(a.nrows >= 1 && nviews >= 0, "bad row / view count");
  if (nviews == 0) return FDK_OK;
  a.logN = log2_exact(a.N);
  if (!a.tw)
    if (int r = twiddles(a.N, &a.tw)) return r;
  const auto form = fdk::rules::filter_form(a.nu, a.nrows, nviews, a.logN, a.transpose && a.qmode == kStoreF32);
  a.far = form == fdk::rules::kFilterWideFar;
  if (fft_choice() && form != fdk::rules::kFilterInPlace) {
    switch (a.logN) {
      case 7: return launch_wide<7>(a, nviews, st);
      case 8: return launch_wide<8>(a, nviews, st);
      case 9: return launch_wide<9>(a, nviews, st);
      case 10: return launch_wide<10>(a, nviews, st);
      case 11: return launch_wide<11>(a, nviews, st);
      case 12: return launch_wide<12>(a, nviews, st);
      case 13: return launch_wide<13>(a, nviews, st);
      case 14: return launch_wide<14>(a, nviews, st);
    }
  }
  const dim3 grid((a.nrows + 1) / 2, nviews);
  hipLaunchKernelGGL(filter_rows_kernel, grid, dim3(256), sizeof(float2) * a.N, st, a);
  FDK_HIP(hipGetLastError());
  return FDK_OK;
}

}  // namespace

extern "C" int fdk_correct_image(const float* dev_src, const float* dev_table, float* dev_dst,
                                 int width, int height, int depth, int pitch, int table_pitch,
                                 void* stream) {
  FDK_REQUIRE(dev_src && dev_table && dev_dst, "NULL pointer");
  FDK_REQUIRE(width > 0 && height > 0 && depth >= 0 && pitch >= width && table_pitch >= width,
              "bad image size");
  if (depth == 0) return FDK_OK;
  dim3 grid((width + 63) / 64, (height + 3) / 4, depth);
  hipLaunchKernelGGL(correct_kernel, grid, dim3(64, 4), 0, static_cast<hipStream_t>(stream),
                     dev_src, dev_table, dev_dst, width, height, pitch, table_pitch);
  FDK_HIP(hipGetLastError());
  return FDK_OK;
}

extern "C" int fdk_filter_rows(const float* dev_src, float* dev_dst, int width, int height,
                               int depth, int src_pitch, int dst_pitch, const float* dev_filter,
                               int N, int pad_mode, void* stream) {
  FDK_REQUIRE(dev_src && dev_dst && dev_filter, "NULL pointer");
  FDK_REQUIRE(src_pitch >= width && dst_pitch >= width, "pitch smaller than width");
  FilterArgs a{};
  a.src = dev_src;
  a.src_pitch = src_pitch;
  a.src_view = (long long)src_pitch * height;
  a.dst = dev_dst;
  a.dst_pitch = dst_pitch;
  a.dst_view = (long long)dst_pitch * height;
  a.transpose = 0;
  a.cos_table = nullptr;
  a.H = dev_filter;
  a.nu = width;
  a.nrows = height;
  a.N = N;
  a.pad = pad_mode;
  a.minmax = nullptr;
  // In place is safe: every row pair is read into LDS before it is written.
  return launch_filter(a, depth, static_cast<hipStream_t>(stream));
}

namespace {

FilterArgs view_args(const float* dev_src, int64_t view_stride_in, int nu, int nv,
                     const float* dev_cos, const float* dev_filter, int N, int pad_mode,
                     int transpose) {
  FilterArgs a{};
  a.src = dev_src;
  a.src_view = view_stride_in;
  a.src_pitch = nu;
  a.transpose = transpose;
  a.dst_pitch = nu;
  a.cos_table = dev_cos;
  a.H = dev_filter;
  a.nu = nu;
  a.nrows = nv;
  a.N = N;
  a.pad = pad_mode;
  return a;
}

// 16-bit output: FP32 filtered batch into `stage`, per-view {min, max} into
// `mm`, then (p - min) / (max - min) quantized into dst.  All on `st`.
int filter_views_q(FilterArgs a, int nviews, void* dev_dst, int64_t view_stride_out, int dtype,
                   float* stage, unsigned* mm, hipStream_t st) {
  const size_t view = (size_t)a.nu * a.nrows;
  hipLaunchKernelGGL(minmax_init_kernel, dim3((nviews + 255) / 256), dim3(256), 0, st, mm, nviews);
  a.dst = stage;
  a.dst_view = (long long)view;
  a.minmax = mm;
  if (int r = launch_filter(a, nviews, st)) return r;
  // 16-byte aligned FP32 rows and 8-byte aligned 16-bit rows: the staging
  // batch is a pool allocation, dev_dst's alignment is checked
  const bool vec = view % 4 == 0 && view_stride_out % 4 == 0 &&
                   reinterpret_cast<uintptr_t>(dev_dst) % 8 == 0;
  const size_t items = vec ? view / 4 : view;
  const int blocks = (int)std::min<size_t>(1024, (items + 255) / 256);
  const dim3 g(blocks, nviews);
  const long long n = (long long)view, sv = (long long)view, dv = (long long)view_stride_out;
  if (dtype == FDK_F16) {
    if (vec) hipLaunchKernelGGL((quantize_kernel<FDK_F16, true>), g, dim3(256), 0, st, stage, sv, dev_dst, dv, n, mm);
    else hipLaunchKernelGGL((quantize_kernel<FDK_F16, false>), g, dim3(256), 0, st, stage, sv, dev_dst, dv, n, mm);
  } else {
    if (vec) hipLaunchKernelGGL((quantize_kernel<FDK_BF16, true>), g, dim3(256), 0, st, stage, sv, dev_dst, dv, n, mm);
    else hipLaunchKernelGGL((quantize_kernel<FDK_BF16, false>), g, dim3(256), 0, st, stage, sv, dev_dst, dv, n, mm);
  }
  FDK_HIP(hipGetLastError());
  return FDK_OK;
}

int check_views(const float* dev_src, void* dev_dst, const float* dev_filter, int transpose,
                int dtype, int nu, int nv, int64_t view_stride_in, int64_t view_stride_out) {
  FDK_REQUIRE(dev_src && dev_dst && dev_filter, "NULL pointer");
  FDK_REQUIRE(transpose == 0 || transpose == 1, "transpose must be 0 or 1");
  FDK_REQUIRE(dtype == FDK_F32 || dtype == FDK_F16 || dtype == FDK_BF16, "unknown dtype %d", dtype);
  FDK_REQUIRE(nu > 0 && nv > 0, "bad view size %d x %d", nu, nv);
  FDK_REQUIRE(view_stride_in >= (int64_t)nu * nv && view_stride_out >= (int64_t)nu * nv,
              "view strides smaller than a view");
  return FDK_OK;
}

}  // namespace

extern "C" int fdk_filter_views(const float* dev_src, int64_t view_stride_in, void* dev_dst,
                                int64_t view_stride_out, int dtype, int nu, int nv, int nviews,
                                const float* dev_cos, const float* dev_filter, int N, int pad_mode,
                                int transpose, float* host_scale_offset, void* stream) {
  if (int r = check_views(dev_src, dev_dst, dev_filter, transpose, dtype, nu, nv, view_stride_in,
                          view_stride_out))
    return r;
  hipStream_t st = static_cast<hipStream_t>(stream);
  FilterArgs a = view_args(dev_src, view_stride_in, nu, nv, dev_cos, dev_filter, N, pad_mode,
                           transpose);
  if (dtype == FDK_F32) {
    a.dst = static_cast<float*>(dev_dst);
    a.dst_view = view_stride_out;
    a.minmax = nullptr;
    return launch_filter(a, nviews, st);
  }
  FDK_REQUIRE(host_scale_offset != nullptr, "FP16/BF16 output needs host_scale_offset");
  if (nviews <= 0) return FDK_OK;
  // FP32 staging of the filtered batch, per-view min/max, then quantize.
  const size_t view = (size_t)nu * nv;
  float* tmp = nullptr;
  unsigned* mm = nullptr;
  if (int r = fdk::stage_alloc((void**)&tmp, view * nviews * sizeof(float), st)) return r;
  if (int r = fdk::stage_alloc((void**)&mm, 2 * sizeof(unsigned) * nviews, st)) {
    (void)hipFreeAsync(tmp, st);
    return r;
  }
  int r = filter_views_q(a, nviews, dev_dst, view_stride_out, dtype, tmp, mm, st);
  std::vector<unsigned> hmm(2 * nviews);
  if (r == FDK_OK) {
    hipError_t e = hipMemcpyAsync(hmm.data(), mm, hmm.size() * sizeof(unsigned), hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e != hipSuccess) r = fdk::fail(FDK_ERR_HIP, "min/max readback: %s", hipGetErrorString(e));
  }
  (void)hipFreeAsync(tmp, st);
  (void)hipFreeAsync(mm, st);
  if (r != FDK_OK) return r;
  for (int v = 0; v < nviews; ++v) {
    const unsigned lo_o = hmm[2 * v], hi_o = hmm[2 * v + 1];
    const float lo = host_ord2f(lo_o), hi = host_ord2f(hi_o);
    host_scale_offset[2 * v] = hi - lo;
    host_scale_offset[2 * v + 1] = lo;
  }
  return FDK_OK;
}

extern "C" int fdk_filter_views_async(const float* dev_src, int64_t view_stride_in, void* dev_dst,
                                      int64_t view_stride_out, int dtype, int nu, int nv,
                                      int nviews, const float* dev_cos, const float* dev_filter,
                                      int N, int pad_mode, int transpose, float* dev_workspace,
                                      unsigned* dev_minmax, void* stream) {
  if (int r = check_views(dev_src, dev_dst, dev_filter, transpose, dtype, nu, nv, view_stride_in,
                          view_stride_out))
    return r;
  FDK_REQUIRE(dtype == FDK_F16 || dtype == FDK_BF16, "dtype %d is not a 16-bit storage type", dtype);
  FDK_REQUIRE(dev_workspace && dev_minmax, "workspace or min/max buffer is NULL");
  if (nviews <= 0) return FDK_OK;
  FilterArgs a = view_args(dev_src, view_stride_in, nu, nv, dev_cos, dev_filter, N, pad_mode,
                           transpose);
  return filter_views_q(a, nviews, dev_dst, view_stride_out, dtype, dev_workspace, dev_minmax,
                        static_cast<hipStream_t>(stream));
}

extern "C" int fdk_filter_proj_image(float* host_proj, int nu, int nv, int nviews,
                                     const float* host_cos, const float* host_filter, int N,
                                     int pad_mode, int depth, float* elapsed_ms) {
  FDK_REQUIRE(host_proj && host_filter, "NULL pointer");
  FDK_REQUIRE(nu > 0 && nv > 0 && nviews >= 0, "bad size");
  if (elapsed_ms) *elapsed_ms = 0.f;
  if (depth <= 0) depth = 32;
  const size_t view = (size_t)nu * nv;
  hipStream_t st = nullptr;
  FDK_HIP(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  float *d = nullptr, *dcos = nullptr, *dH = nullptr;
  int r = FDK_OK;
  hipError_t e = hipEventCreate(&ev0);
  if (e == hipSuccess) e = hipEventCreate(&ev1);
  if (e == hipSuccess) e = fdk::dev_malloc((void**)&d, view * depth * sizeof(float));
  if (e == hipSuccess) e = fdk::dev_malloc((void**)&dH, sizeof(float) * N);
  if (e == hipSuccess) e = hipMemcpy(dH, host_filter, sizeof(float) * N, hipMemcpyHostToDevice);
  if (e == hipSuccess && host_cos) e = fdk::dev_malloc((void**)&dcos, view * sizeof(float));
  if (e == hipSuccess && host_cos) e = hipMemcpy(dcos, host_cos, view * sizeof(float), hipMemcpyHostToDevice);
  if (e != hipSuccess) r = fdk::fail(e == hipErrorOutOfMemory ? FDK_ERR_OOM : FDK_ERR_HIP, "FilterProjImage setup: %s", hipGetErrorString(e));
  // Each batch -- upload, cos weighting + filter, download -- is timed between
  // two events and the batch times are summed (the reference's per-batch
  // timeGetTime sum, without the set-up).
  for (int v0 = 0; v0 < nviews && r == FDK_OK; v0 += depth) {
    const int cnt = std::min(depth, nviews - v0);
    e = hipEventRecord(ev0, st);
    if (e == hipSuccess)
      e = hipMemcpyAsync(d, host_proj + view * v0, view * cnt * sizeof(float), hipMemcpyHostToDevice, st);
    if (e != hipSuccess) { r = fdk::fail(FDK_ERR_HIP, "upload: %s", hipGetErrorString(e)); break; }
    r = fdk_filter_views(d, (int64_t)view, d, (int64_t)view, FDK_F32, nu, nv, cnt, dcos, dH, N,
                         pad_mode, 0, nullptr, st);
    if (r != FDK_OK) break;
    e = hipMemcpyAsync(host_proj + view * v0, d, view * cnt * sizeof(float), hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipEventRecord(ev1, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    float ms = 0.f;
    if (e == hipSuccess) e = hipEventElapsedTime(&ms, ev0, ev1);
    if (e != hipSuccess) r = fdk::fail(FDK_ERR_HIP, "download: %s", hipGetErrorString(e));
    else if (elapsed_ms) *elapsed_ms += ms;
  }
  (void)hipStreamSynchronize(st);
  if (d) (void)hipFree(d);
  if (dH) (void)hipFree(dH);
  if (dcos) (void)hipFree(dcos);
  if (ev0) (void)hipEventDestroy(ev0);
  if (ev1) (void)hipEventDestroy(ev1);
  (void)hipStreamDestroy(st);
  return r;
}

extern "C" int fdk_filter_frame_host(float* host_src, float* host_dst, int nu, int nv,
                                     const float* host_cos, const float* host_filter, int N,
                                     int pad_mode, int transpose) {
  FDK_REQUIRE(host_src && host_dst && host_cos && host_filter, "NULL pointer");
  FDK_REQUIRE(nu > 0 && nv > 0, "bad image size");
  const size_t view = (size_t)nu * nv;
  float *s = nullptr, *d = nullptr, *c = nullptr, *h = nullptr;
  hipError_t e = fdk::dev_malloc((void**)&s, view * 4);
  if (e == hipSuccess) e = fdk::dev_malloc((void**)&d, view * 4);
  if (e == hipSuccess) e = fdk::dev_malloc((void**)&c, view * 4);
  if (e == hipSuccess) e = fdk::dev_malloc((void**)&h, sizeof(float) * std::max(N, 1));
  if (e == hipSuccess) e = hipMemcpy(s, host_src, view * 4, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(c, host_cos, view * 4, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(h, host_filter, sizeof(float) * N, hipMemcpyHostToDevice);
  int r = e == hipSuccess ? FDK_OK : fdk::fail(FDK_ERR_HIP, "FilterEngine upload: %s", hipGetErrorString(e));
  if (r == FDK_OK)
    r = fdk_filter_views(s, (int64_t)view, d, (int64_t)view, FDK_F32, nu, nv, 1, c, h, N, pad_mode,
                         transpose, nullptr, nullptr);
  if (r == FDK_OK) r = fdk_correct_image(s, c, s, nu, nv, 1, nu, nu, nullptr);
  if (r == FDK_OK) {
    e = hipMemcpy(host_dst, d, view * 4, hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(host_src, s, view * 4, hipMemcpyDeviceToHost);
    if (e != hipSuccess) r = fdk::fail(FDK_ERR_HIP, "FilterEngine download: %s", hipGetErrorString(e));
  }
  if (s) (void)hipFree(s);
  if (d) (void)hipFree(d);
  if (c) (void)hipFree(c);
  if (h) (void)hipFree(h);
  return r;
}

// ------------------------------------------------------------ no-allocation filter
// fdk_filter_views without any allocation: the 16-bit forms run the filter
// twice (the first pass only forms each view's min/max, the second quantizes
// as it stores) instead of staging the FP32 batch, and the min/max words and
// the twiddle table live in `scratch`, a fixed device array of
// kScratchBytes per device.
namespace {
constexpr int kNoAllocViews = 1024;  // views per call
constexpr int kNoAllocN = 16384;     // FFT length
constexpr size_t kScratchMinmax = 2 * kNoAllocViews * sizeof(unsigned);
constexpr size_t kScratchBytes = kScratchMinmax + kNoAllocN * sizeof(float2);  // 136 KiB
constexpr int kMaxDevices = 64;
}  // namespace

// Per-view {min, max} words, then the twiddle table of the call's N.  Each
// device holds its own copy for the life of the process, shared by every call
// on that device.
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {
std::mutex g_scratch_mutex;
unsigned char* g_scratch[kMaxDevices] = {};

// The device address of the current device's `scratch`, looked up on the
// first call on that device (the array's name is not a device address in host
// code).
int scratch_ptr(unsigned char** out) {
  int dev = 0;
  FDK_HIP(hipGetDevice(&dev));
  FDK_REQUIRE(dev >= 0 && dev < kMaxDevices, "device %d beyond the %d supported", dev, kMaxDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr)
      return fdk::fail(FDK_ERR_HIP, "address of the filter scratch: %s", hipGetErrorString(e));
    g_scratch[dev] = static_cast<unsigned char*>(p);
  }
  *out = g_scratch[dev];
  return FDK_OK;
}
}  // namespace

extern "C" int fdk_filter_views_noalloc(const float* dev_src, int64_t view_stride_in,
                                        void* dev_dst, int64_t view_stride_out, int dtype, int nu,
                                        int nv, int nviews, const float* dev_cos,
                                        const float* dev_filter, int N, int pad_mode,
                                        int transpose, float* host_scale_offset, void* stream) {
  if (int r = check_views(dev_src, dev_dst, dev_filter, transpose, dtype, nu, nv, view_stride_in,
                          view_stride_out))
    return r;
  FDK_REQUIRE(nviews >= 0 && nviews <= kNoAllocViews,
              "%d views outside the no-allocation filter's 0..%d per call", nviews, kNoAllocViews);
  FDK_REQUIRE(N >= 16 && N <= kNoAllocN, "filter length %d outside the no-allocation filter's "
              "16..%d", N, kNoAllocN);
  FDK_REQUIRE(dtype == FDK_F32 || host_scale_offset != nullptr,
              "FP16/BF16 output needs host_scale_offset");
  if (dtype != FDK_F32 && nviews > 0) {
    // the second pass reads the source again: the 16-bit output must not overlap it
    const char* s0 = reinterpret_cast<const char*>(dev_src);
    const char* s1 = s0 + ((size_t)(nviews - 1) * view_stride_in + (size_t)nu * nv) * 4;
    const char* d0 = static_cast<const char*>(dev_dst);
    const char* d1 = d0 + ((size_t)(nviews - 1) * view_stride_out + (size_t)nu * nv) * 2;
    FDK_REQUIRE(d1 <= s0 || d0 >= s1, "16-bit output overlaps the source views");
  }
  if (nviews == 0) return FDK_OK;
  unsigned char* base = nullptr;
  if (int r = scratch_ptr(&base)) return r;
  unsigned* mm = reinterpret_cast<unsigned*>(base);
  float2* tw = reinterpret_cast<float2*>(base + kScratchMinmax);
  hipStream_t st = static_cast<hipStream_t>(stream);
  launch_twiddles(tw, N, st);  // the last call's table may be of another N
  FilterArgs a = view_args(dev_src, view_stride_in, nu, nv, dev_cos, dev_filter, N, pad_mode,
                           transpose);
  a.tw = tw;
  a.dst = static_cast<float*>(dev_dst);
  a.dst_view = view_stride_out;
  if (dtype == FDK_F32) return launch_filter(a, nviews, st);
  hipLaunchKernelGGL(minmax_init_kernel, dim3((nviews + 255) / 256), dim3(256), 0, st, mm, nviews);
  a.qmode = kStoreNone;
  a.minmax = mm;
  if (int r = launch_filter(a, nviews, st)) return r;
  a.qmode = dtype == FDK_F16 ? kStoreF16 : kStoreBF16;
  a.qmm = mm;
  a.minmax = nullptr;
  if (int r = launch_filter(a, nviews, st)) return r;
  // the words land in the caller's array and are turned into {scale, offset} there
  hipError_t e = hipMemcpyAsync(host_scale_offset, mm, 2 * sizeof(unsigned) * nviews,
                                hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  if (e != hipSuccess) return fdk::fail(FDK_ERR_HIP, "min/max readback: %s", hipGetErrorString(e));
  for (int v = 0; v < nviews; ++v) {
    unsigned w[2];
    std::memcpy(w, host_scale_offset + 2 * v, sizeof(w));
    const float lo = host_ord2f(w[0]), hi = host_ord2f(w[1]);
    host_scale_offset[2 * v] = hi - lo;
    host_scale_offset[2 * v + 1] = lo;
  }
  return FDK_OK;
}
