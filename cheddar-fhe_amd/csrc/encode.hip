// CKKS encoding and decoding on the device (src/core/Encode.cpp): the special
// (I)FFT over the slots in IEEE double, the truncation of scaled coefficients
// to residues, and the exact CRT back from residues to doubles. The operation
// order is the reference's, and this file, like every other, is compiled with
// -ffp-contract=off, so each result is the host encoder's bit for bit: a
// complex product is (ac - bd, ad + bc) with every product and sum rounded,
// and the twiddles are the host's own values.
//
// Non-finite values are not treated here (the host's complex product has a
// recovery path for them): callers keep them out (encode) or, where a result
// is not finite, take it from the host encoder (decode).
//
// The transform of 2^15 slots is 512 KiB: two passes of up to 8 and 7 radix-2
// stages through LDS. Stages of strides below 256 stay inside a block of 256
// slots, the others inside a column (slots 256 apart), so each pass reads and
// writes every slot once. A pass takes 4-5 us, its launch and the latency of
// its stages, or, where it reads or writes the message in pinned host memory,
// what the bus takes for 512 KiB (29.6 us reading, 15.8 us writing; a copy
// from and to pageable memory took 30 us beside the 7 us pass). The CRT of 2^16
// coefficients takes 6.4 us at 6 limbs. All of an encode at 24 limbs and 2^15
// slots: 110 us against 11-14 ms on the host, a decode at 6 limbs 118 us
// against 10.7 ms.
#include <algorithm>

#include "chd_device.h"
#include "cheddar_kernels.h"
#include "kernel_common.h"

namespace chd {
namespace {

constexpr int kBlockLog = 8;                // slots of a block pass
constexpr int kBlock = 1 << kBlockLog;
constexpr int kBlockThreads = kBlock / 2;   // one butterfly per thread
// columns per workgroup: the message is read from (and written to) pinned
// host memory in place, in pieces of 64 bytes per row and component
constexpr int kColTile = 8;
constexpr int kMaxRows = 128;               // 2^15 slots / 256
constexpr int kColThreads = kMaxRows / 2 * kColTile;
constexpr int kThreads = 256;

struct C64 {
  double re, im;
};
__device__ __forceinline__ C64 operator+(C64 a, C64 b) {
  return {a.re + b.re, a.im + b.im};
}
__device__ __forceinline__ C64 operator-(C64 a, C64 b) {
  return {a.re - b.re, a.im - b.im};
}
__device__ __forceinline__ C64 operator*(C64 a, C64 b) {
  return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}

// SpecialIFFT butterfly (Encode.cpp:84-109): x = a + b, y = (a - b) w
__device__ __forceinline__ void ifft_bfly(C64 &a, C64 &b, C64 w) {
  const C64 x = a + b;
  b = (a - b) * w;
  a = x;
}
// SpecialFFT butterfly (Encode.cpp:111-133)
__device__ __forceinline__ void fft_bfly(C64 &a, C64 &b, C64 w) {
  const C64 y = b * w;
  b = a - y;
  a = a + y;
}

__device__ __forceinline__ uint32_t brev(uint32_t x, int bits) {
  return bits == 0 ? 0 : __brev(x) >> (32 - bits);
}

// message value i: zero beyond its length
struct Msg {
  const double *re, *im;
  int stride, len;
  __device__ C64 at(int i) const {
    const size_t o = static_cast<size_t>(i) * stride;
    return i < len ? C64{re[o], im[o]} : C64{0.0, 0.0};
  }
};

// stages of stride >= 256 over the column tile blockIdx.x: rows
// 2^(log_slots - 8) rows of 256 slots; tw[s + j] is stage s's twiddle j
template <bool kInverse>
__device__ __forceinline__ void column_stages(C64 *x, int rows,
                                              const C64 *tw) {
  const int n = rows / 2 * kColTile;
  const int c = threadIdx.x % kColTile;
  const int k = threadIdx.x / kColTile;
  const int col = blockIdx.x * kColTile + c;
  for (int t = 1; t < rows; t *= 2) {
    const int sr = kInverse ? rows / 2 / t : t;  // stride in rows
    if (static_cast<int>(threadIdx.x) < n) {
      const int i = (k / sr) * 2 * sr + k % sr;
      const C64 w = tw[sr * kBlock + (k % sr) * kBlock + col];
      C64 &a = x[i * kColTile + c], &b = x[(i + sr) * kColTile + c];
      if constexpr (kInverse)
        ifft_bfly(a, b, w);
      else
        fft_bfly(a, b, w);
    }
    __syncthreads();
  }
}
// stages of stride < 2^bits over the 2^bits slots x
template <bool kInverse>
__device__ __forceinline__ void block_stages(C64 *x, int bits, const C64 *tw) {
  const int n = (1 << bits) / 2;
  const int k = threadIdx.x;
  for (int t = 0; t < bits; t++) {
    const int s = kInverse ? n >> t : 1 << t;
    if (k < n) {
      const int i = (k / s) * 2 * s + k % s;
      const C64 w = tw[s + k % s];
      if constexpr (kInverse)
        ifft_bfly(x[i], x[i + s], w);
      else
        fft_bfly(x[i], x[i + s], w);
    }
    __syncthreads();
  }
}

// encode, strides >= 256: message -> work
__global__ __launch_bounds__(kColThreads) void ifft_columns(Msg msg, C64 *work,
                                                            const C64 *tw,
                                                            int rows) {
  __shared__ C64 x[kMaxRows * kColTile];
  const int n = rows * kColTile;
  for (int e = threadIdx.x; e < n; e += kColThreads)
    x[e] = msg.at(e / kColTile * kBlock + blockIdx.x * kColTile +
                  e % kColTile);
  __syncthreads();
  column_stages<true>(x, rows, tw);
  for (int e = threadIdx.x; e < n; e += kColThreads)
    work[e / kColTile * kBlock + blockIdx.x * kColTile + e % kColTile] = x[e];
}

// encode, strides < 256: src -> coef[i] = (value i of the transform in
// natural order / slots) * scale
__global__ __launch_bounds__(kBlockThreads) void ifft_blocks(
    Msg src, C64 *coef, const C64 *tw, int log_slots, double scale) {
  __shared__ C64 x[kBlock];
  const int bits = min(log_slots, kBlockLog);
  const int base = blockIdx.x << bits;
  for (int e = threadIdx.x; e < (1 << bits); e += kBlockThreads)
    x[e] = src.at(base + e);
  __syncthreads();
  block_stages<true>(x, bits, tw);
  const double slots = static_cast<double>(1 << log_slots);
  for (int e = threadIdx.x; e < (1 << bits); e += kBlockThreads) {
    const C64 v = {x[e].re / slots, x[e].im / slots};
    coef[brev(base + e, log_slots)] = {v.re * scale, v.im * scale};
  }
}

// x (finite) truncated toward zero, modulo p in [0, p) (BigInt(double) and
// BigInt::Mod, BigInt_tommath.cpp:22-26); r2 = 2^64 mod p, pn = -p^-1
__device__ __forceinline__ uint32_t trunc_mod(double x, uint32_t p,
                                              uint32_t pn, uint32_t r2) {
  const double mag = trunc(fabs(x));
  uint32_t r;
  if (mag < static_cast<double>(p)) {
    r = static_cast<uint32_t>(mag);
  } else {
    // mag = u 2^sh with u < 2^63; u mod p as two Montgomery reductions:
    // u 2^-32, below 2^31 + p < 2^32, times 2^64 2^-32
    int sh = 0;
    double m = mag;
    if (mag >= 0x1p63) {
      sh = static_cast<int>((__double_as_longlong(mag) >> 52) & 0x7ff) - 1075;
      m = ldexp(mag, -sh);  // the 53-bit mantissa, exact
    }
    const uint64_t u = static_cast<uint64_t>(m);
    const uint32_t a = static_cast<uint32_t>(u) * pn;
    const uint64_t h = (static_cast<uint64_t>(a) * p + static_cast<uint32_t>(u));
    const uint32_t b = static_cast<uint32_t>((h >> 32) + (u >> 32));
    const uint64_t t = static_cast<uint64_t>(b) * r2;
    const uint32_t c = static_cast<uint32_t>(t) * pn;
    r = static_cast<uint32_t>((static_cast<uint64_t>(c) * p + t) >> 32);
    r = r >= p ? r - p : r;
    for (int i = 0; i < sh; i++) r = r + r >= p ? r + r - p : r + r;
  }
  return x < 0 && r != 0 ? p - r : r;
}

// ComplexVectorToPlaintext's residues (Encode.cpp:135-190): coefficient
// i gap of limb l holds re of coef[i], coefficient i gap + N/2 im, the rest
// zero. grid (N / 1024, limbs)
__global__ __launch_bounds__(kThreads) void encode_residues(
    chd_tables t, chd_limb_map m, const uint32_t *r2s, uint32_t *dst,
    const C64 *coef, int log_slots) {
  const int l = blockIdx.y;
  const int ti = m.tab_off + l + (l >= m.num_q ? m.tab_gap : 0);
  const uint32_t p = t.q[ti], pn = 0u - static_cast<uint32_t>(t.qinv[ti]);
  const uint32_t r2 = r2s[ti];
  const int k0 = (blockIdx.x * kThreads + threadIdx.x) * 4;
  const int log_gap = kLogN - 1 - log_slots;
  const bool imag = k0 >= kN / 2;
  uint32_t o[4];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int k = (k0 + j) & (kN / 2 - 1);
    const int i = k >> log_gap;
    o[j] = 0;
    if ((i << log_gap) == k)
      o[j] = trunc_mod(imag ? coef[i].im : coef[i].re, p, pn, r2);
  }
  *reinterpret_cast<uint4 *>(dst + (static_cast<size_t>(l) << kLogN) + k0) =
      make_uint4(o[0], o[1], o[2], o[3]);
}

// decode, strides < 256: in place on work (already in bit-reversed order)
__global__ __launch_bounds__(kBlockThreads) void fft_blocks(
    const C64 *work, double *out_re, double *out_im, int out_stride,
    const C64 *tw, int log_slots) {
  __shared__ C64 x[kBlock];
  const int bits = min(log_slots, kBlockLog);
  const int base = blockIdx.x << bits;
  for (int e = threadIdx.x; e < (1 << bits); e += kBlockThreads)
    x[e] = work[base + e];
  __syncthreads();
  block_stages<false>(x, bits, tw);
  for (int e = threadIdx.x; e < (1 << bits); e += kBlockThreads) {
    const size_t o = static_cast<size_t>(base + e) * out_stride;
    out_re[o] = x[e].re;
    out_im[o] = x[e].im;
  }
}

// decode, strides >= 256: work -> the message values
__global__ __launch_bounds__(kColThreads) void fft_columns(
    const C64 *work, double *out_re, double *out_im, int out_stride,
    const C64 *tw, int rows) {
  __shared__ C64 x[kMaxRows * kColTile];
  const int n = rows * kColTile;
  for (int e = threadIdx.x; e < n; e += kColThreads)
    x[e] = work[e / kColTile * kBlock + blockIdx.x * kColTile + e % kColTile];
  __syncthreads();
  column_stages<false>(x, rows, tw);
  for (int e = threadIdx.x; e < n; e += kColThreads) {
    const size_t o = static_cast<size_t>(e / kColTile * kBlock +
                                         blockIdx.x * kColTile + e % kColTile) *
                     out_stride;
    out_re[o] = x[e].re;
    out_im[o] = x[e].im;
  }
}

typedef const __attribute__((address_space(4))) uint32_t cu32;

// PlaintextToComplexVector's integer part (Encode.cpp:192-246): the value
// sum_j r_j (Q / q_j) mod Q of one coefficient, centred into (-Q/2, Q/2],
// as mp_get_double converts it (60-bit digits from the top, each step
// rounded), divided by the scale. A thread keeps its W-word integers in
// registers; the table [limbs + 2][W] (Q / q_j, then Q, then floor(Q / 2)) is
// read through scalar loads. grid over 2 slots values, real parts first.
template <int W>
__global__ __launch_bounds__(kThreads) void decode_crt(
    const uint32_t *res, int limbs, const uint32_t *table, C64 *work,
    int log_slots, double scale) {
  const int v = blockIdx.x * kThreads + threadIdx.x;
  const int slots = 1 << log_slots;
  if (v >= 2 * slots) return;
  const bool imag = v >= slots;
  const int i = v & (slots - 1);
  const uint32_t *r = res + (static_cast<size_t>(i) << (kLogN - 1 - log_slots)) +
                      (imag ? kN / 2 : 0);
  cu32 *tab = (cu32 *)table;
  uint32_t acc[W], sub[W];
#pragma unroll
  for (int w = 0; w < W; w++) acc[w] = 0;
  for (int j = 0; j < limbs; j++) {
    const uint64_t rj = r[static_cast<size_t>(j) << kLogN];
    uint64_t carry = 0;
#pragma unroll
    for (int w = 0; w < W; w++) {
      const uint64_t t = rj * tab[j * W + w] + acc[w] + carry;
      acc[w] = static_cast<uint32_t>(t);
      carry = t >> 32;
    }
  }
  // x - y into sub; true when x >= y
  auto minus = [&](auto x, auto y) {
    uint32_t borrow = 0;
#pragma unroll
    for (int w = 0; w < W; w++) {
      const uint64_t t = static_cast<uint64_t>(x(w)) - y(w) - borrow;
      sub[w] = static_cast<uint32_t>(t);
      borrow = static_cast<uint32_t>(t >> 63);
    }
    return borrow == 0;
  };
  auto a = [&](int w) { return acc[w]; };
  auto q = [&](int w) -> uint32_t { return tab[limbs * W + w]; };
  auto half = [&](int w) -> uint32_t { return tab[(limbs + 1) * W + w]; };
  // the sum is below limbs Q
  while (minus(a, q)) {
#pragma unroll
    for (int w = 0; w < W; w++) acc[w] = sub[w];
  }
  const bool neg = !minus(half, a);
  if (neg) {
    (void)minus(q, a);
#pragma unroll
    for (int w = 0; w < W; w++) acc[w] = sub[w];
  }
  // leading zero digits leave d at zero
  double d = 0.0;
#pragma unroll
  for (int k = (32 * W + 59) / 60 - 1; k >= 0; k--) {
    const int lo = 60 * k / 32, sh = 60 * k % 32;
    uint64_t digit = acc[lo] >> sh;
    if (lo + 1 < W) digit |= static_cast<uint64_t>(acc[lo + 1]) << (32 - sh);
    if (sh > 4 && lo + 2 < W)
      digit |= static_cast<uint64_t>(acc[lo + 2]) << (64 - sh);
    digit &= (1ull << 60) - 1;
    d = d * 0x1p60 + static_cast<double>(digit);
  }
  d = (neg ? -d : d) / scale;
  C64 &o = work[brev(i, log_slots)];
  if (imag)
    o.im = d;
  else
    o.re = d;
}

}  // namespace
}  // namespace chd

using namespace chd;

extern "C" int chd_k_encode_coefficients(double *coef, double *work,
                                         const double *msg_re,
                                         const double *msg_im, int msg_stride,
                                         int msg_len, int log_slots,
                                         double scale, const double *twiddles,
                                         void *stream) {
  if (!coef || !work || !msg_re || !msg_im || msg_stride < 1 || msg_len < 1 ||
      log_slots < 0 || log_slots > kLogN - 1 || msg_len > (1 << log_slots) ||
      !twiddles)
    return set_error(CHD_ERR_ARG,
                     "chd_k_encode_coefficients: invalid argument");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const C64 *tw = reinterpret_cast<const C64 *>(twiddles);
  Msg src{msg_re, msg_im, msg_stride, msg_len};
  if (log_slots > kBlockLog) {
    hipLaunchKernelGGL(ifft_columns, dim3(kBlock / kColTile),
                       dim3(kColThreads), 0, s, src,
                       reinterpret_cast<C64 *>(work), tw,
                       1 << (log_slots - kBlockLog));
    src = Msg{work, work + 1, 2, 1 << log_slots};
  }
  hipLaunchKernelGGL(ifft_blocks, dim3(1 << std::max(0, log_slots - kBlockLog)),
                     dim3(kBlockThreads), 0, s, src,
                     reinterpret_cast<C64 *>(coef), tw, log_slots, scale);
  return check_launch("chd_k_encode_coefficients");
}

extern "C" int chd_k_encode_residues(const chd_tables *t,
                                     const chd_limb_map *m,
                                     const uint32_t *mont_converter,
                                     uint32_t *dst, int num_limbs,
                                     const double *coef, int log_slots,
                                     void *stream) {
  if (!t || !m || !mont_converter || !dst || num_limbs < 1 || !coef ||
      log_slots < 0 || log_slots > kLogN - 1 || m->skip_len != 0)
    return set_error(CHD_ERR_ARG, "chd_k_encode_residues: invalid argument");
  hipLaunchKernelGGL(encode_residues, dim3(kN / (4 * kThreads), num_limbs),
                     dim3(kThreads), 0, static_cast<hipStream_t>(stream), *t,
                     *m, mont_converter, dst,
                     reinterpret_cast<const C64 *>(coef), log_slots);
  return check_launch("chd_k_encode_residues");
}

extern "C" int chd_k_decode_width(int words) {
  for (int w : {4, 8, 16, 24, 32, 48, 64})
    if (words <= w) return w;
  return 0;
}

extern "C" int chd_k_decode(double *out_re, double *out_im, int out_stride,
                            double *work, const uint32_t *residues, int limbs,
                            const uint32_t *table, int width, int log_slots,
                            double scale, const double *twiddles,
                            void *stream) {
  if (!out_re || !out_im || out_stride < 1 || !work || !residues ||
      limbs < 1 || !table || width < 1 || chd_k_decode_width(width) != width ||
      log_slots < 0 || log_slots > kLogN - 1 || !twiddles)
    return set_error(CHD_ERR_ARG, "chd_k_decode: invalid argument");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const C64 *tw = reinterpret_cast<const C64 *>(twiddles);
  C64 *x = reinterpret_cast<C64 *>(work);
  const dim3 g((2 << log_slots) / kThreads + ((2 << log_slots) % kThreads != 0));
#define CHD_DECODE_CRT(W)                                                  \
  case W:                                                                  \
    hipLaunchKernelGGL(decode_crt<W>, g, dim3(kThreads), 0, s, residues,   \
                       limbs, table, x, log_slots, scale);                 \
    break
  switch (width) {
    CHD_DECODE_CRT(4);
    CHD_DECODE_CRT(8);
    CHD_DECODE_CRT(16);
    CHD_DECODE_CRT(24);
    CHD_DECODE_CRT(32);
    CHD_DECODE_CRT(48);
    CHD_DECODE_CRT(64);
  }
#undef CHD_DECODE_CRT
  const bool cols = log_slots > kBlockLog;
  // with column stages to come, the block pass works in place
  hipLaunchKernelGGL(fft_blocks, dim3(1 << std::max(0, log_slots - kBlockLog)),
                     dim3(kBlockThreads), 0, s, x, cols ? work : out_re,
                     cols ? work + 1 : out_im, cols ? 2 : out_stride, tw,
                     log_slots);
  if (cols)
    hipLaunchKernelGGL(fft_columns, dim3(kBlock / kColTile), dim3(kColThreads),
                       0, s, x, out_re, out_im, out_stride, tw,
                       1 << (log_slots - kBlockLog));
  return check_launch("chd_k_decode");
}
