// The column stage of a base switch (ModUp, ModDown, Rescale) in one launch:
// for a tile of columns, GS stages 7..0 of every source limb's inverse NTT
// with its constant and centring, the BConv to every destination prime, and
// CT stages 0..7 of every destination limb's forward NTT
// (INTTAndMultConst / INTTForModDown, ModSwitchMatrixMult and the first half
// of NTTForModUp / NTTForModDown: src/core/NTT.cu:743-1128,
// src/core/ModSwitch.cu:23-171). None of the three needs data of another
// column (index = row * 256 + column), so the switched limbs go from the
// inverse row pass to the forward row pass through LDS instead of two passes
// over memory between three launches.
//
// Data between the row passes and this kernel is column-blocked: index
// row * 256 + col of a limb is word
//   ((col >> 2) * 256 + 16 * (row % 16) + row / 16) * 4 + (col & 3).
// A row pass's tile t, rows 16 r + t, is then 64 pieces of 256 contiguous bytes,
// and four columns are 4 KiB contiguous, whatever the tile width here.
//
// Work split. A workgroup (8 waves) owns kW = 2 columns of one job and all (or a
// 16-aligned part of) its destinations. A wave works on 4 / kW limbs at a
// time, 16 lanes per column of a limb and 16 rows per lane, so its exchanges
// between the two radix-16 halves are its own (wave-level fences; the
// workgroup meets only around the BConv). Limbs of one wave have different
// primes: primes and twiddles are per lane.
//
// Why this shape. The launch it replaces three of moved 56 MiB (ModUp) and 35
// MiB (merged ModDown) of a 24 + 8 limb, dnum 3 key switch between memory and
// the CUs; this one moves 24 and 16 MiB and is bound by the latency of its
// three phases at two to three waves per SIMD (26-28 % VALU-busy; its 4.6 and
// 3.4 M wave instructions are 7.4 and 5.6 us spread evenly; the 24 jobs of a
// hoisted batch keep the VALU 63 % busy): 20.0 and 15.2 us
// against 29.4 us (inverse columns + BConv + forward columns) and, with the
// row pass that follows, 25 against 31.7 us (inverse columns + BConv +
// single-pass NTT). One 24-limb product with merged rescale went from 89.3 to
// 80.4 us, a 5-limb one (5 launches instead of 8) from 54.0 to 45.0 us.
// Two columns per workgroup: one column (twice the workgroups, half the
// useful bytes per cache line and instruction) took 83.4 us per product, four
// (64 workgroups per job, whole limbs per wave) 85.0; 256 threads 86.7, 768
// threads 84.4.
//
// Arithmetic is unsigned: primes below 2^30 use the lazy butterflies of
// ntt.hip ([0, 4q) forward, [0, 2q) inverse). A wave that holds a larger prime
// (below 2^31, where 4q does not fit 32 bits) reduces both butterfly inputs
// instead: two more instructions, same residues. The BConv is bconv.hip's
// (int8 digit planes on the matrix cores, the same packed tables).
#include <algorithm>

#include "chd_device.h"
#include "cheddar_kernels.h"
#include "kernel_common.h"

namespace chd {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));

constexpr int kThreads = 512;
constexpr int kWaves = kThreads / 64;
constexpr int kW = 2;                // columns per workgroup
constexpr int kSub = 4 / kW;         // limbs per wave, workgroups per block
constexpr int kTiles = 256 / kW;
constexpr int kChunkSrc = 16;
constexpr int kMaxSrc = 32;
// LDS words of one column of one limb: 256 rows, one pad word per 16 (row r
// at r + r / 16), and 4 more so that the columns the matrix operands read
// together start 16 banks apart
constexpr int kColWords = 276;

struct SwitchBatch {
  chd_switch_job job[CHD_MAX_BCONV_JOBS];
};

__device__ __forceinline__ uint32_t umin(uint32_t a, uint32_t b) {
  return a < b ? a : b;
}
// |x - y| + z in one instruction (x >= y here: x - y + z)
__device__ __forceinline__ uint32_t sad(uint32_t x, uint32_t y, uint32_t z) {
  uint32_t r;
  asm("v_sad_u32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "v"(y), "v"(z));
  return r;
}
// b w 2^-32 mod q in [0, 2q) for b < 2^32, w < q < 2^31; qn = -q^-1 mod 2^32
__device__ __forceinline__ uint32_t mont_lo(uint32_t b, uint32_t w,
                                            uint32_t qn, uint32_t q) {
  const uint64_t t = static_cast<uint64_t>(b) * w;
  const uint32_t m = static_cast<uint32_t>(t) * qn;
  return static_cast<uint32_t>((static_cast<uint64_t>(m) * q + t) >> 32);
}
// a wave's LDS accesses execute in order; only the compiler must not move
// them across an exchange between its lanes
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// CT butterfly. kSmall (q < 2^30): a, b in [0, 4q), kRed false for a < 2q.
// Otherwise a in [0, 2q), any b, both results in [0, 2q).
template <bool kSmall, bool kRed>
__device__ __forceinline__ void ct(uint32_t &a, uint32_t &b, uint32_t w,
                                   uint32_t q, uint32_t qn) {
  const uint32_t d = mont_lo(b, w, qn, q);
  if constexpr (kSmall) {
    const uint32_t ar = kRed ? umin(a, a - 2 * q) : a;
    b = sad(2 * q, d, ar);
    a = ar + d;
  } else {
    const uint32_t ar = umin(a, a - q), dr = umin(d, d - q);
    b = sad(q, dr, ar);
    a = ar + dr;
  }
}
// GS butterfly. kSmall: a, b in [0, 2q); otherwise both in [0, q).
template <bool kSmall>
__device__ __forceinline__ void gs(uint32_t &a, uint32_t &b, uint32_t w,
                                   uint32_t q, uint32_t qn) {
  const uint32_t r = kSmall ? 2 * q : q;
  const uint32_t s = a + b;
  const uint32_t d = mont_lo(sad(r, b, a), w, qn, q);
  a = umin(s, s - r);
  b = kSmall ? d : umin(d, d - q);
}

// the 15 twiddles of stages 0..3 (words 1..15 of the limb's table)
__device__ __forceinline__ void load_top(const uint32_t *tw,
                                         uint32_t (&w)[16]) {
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const v4u v = *reinterpret_cast<const v4u *>(tw + 4 * i);
#pragma unroll
    for (int j = 0; j < 4; j++) w[4 * i + j] = v[j];
  }
}
// the 15 twiddles of stages 4..7 for rows 16 rg .. 16 rg + 15: stage s's are
// words (16 + rg) 2^(s - 4) + g; w[2^(s - 4) + g], w[0] unused
__device__ __forceinline__ void load_low(const uint32_t *tw, int rg,
                                         uint32_t (&w)[16]) {
  const uint32_t *p = tw + 16 + rg;
  w[0] = 0;
  w[1] = *p;
  const v2u a = *reinterpret_cast<const v2u *>(tw + 2 * (16 + rg));
  const v4u b = *reinterpret_cast<const v4u *>(tw + 4 * (16 + rg));
  const v4u c = *reinterpret_cast<const v4u *>(tw + 8 * (16 + rg));
  const v4u d = *reinterpret_cast<const v4u *>(tw + 8 * (16 + rg) + 4);
  w[2] = a[0];
  w[3] = a[1];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    w[4 + j] = b[j];
    w[8 + j] = c[j];
    w[12 + j] = d[j];
  }
}

// radix-16 over the registers; group g of stage t uses w[2^t + g]
template <bool kSmall, bool kFirst>
__device__ __forceinline__ void ct16(uint32_t (&x)[16],
                                     const uint32_t (&w)[16], uint32_t q,
                                     uint32_t qn) {
#pragma unroll
  for (int t = 0; t < 4; t++) {
    const int h = 8 >> t;
#pragma unroll
    for (int g = 0; g < (1 << t); g++)
#pragma unroll
      for (int k = g * 2 * h; k < g * 2 * h + h; k++) {
        if (kFirst && t == 0)
          ct<kSmall, false>(x[k], x[k + h], w[1 << t], q, qn);
        else
          ct<kSmall, true>(x[k], x[k + h], w[(1 << t) + g], q, qn);
      }
  }
}
template <bool kSmall>
__device__ __forceinline__ void gs16(uint32_t (&x)[16],
                                     const uint32_t (&w)[16], uint32_t q,
                                     uint32_t qn) {
#pragma unroll
  for (int t = 3; t >= 0; t--) {
    const int h = 8 >> t;
#pragma unroll
    for (int g = 0; g < (1 << t); g++)
#pragma unroll
      for (int k = g * 2 * h; k < g * 2 * h + h; k++)
        gs<kSmall>(x[k], x[k + h], w[(1 << t) + g], q, qn);
  }
}

// Inverse column stages of one column: x holds rows 16 rg + k as the inverse
// row pass left them (below 2q; below q for q >= 2^30); the centred
// MontMul(x, ce), split into signed byte digits, goes to xt.
template <bool kSmall>
__device__ __forceinline__ void inv_column(uint32_t (&x)[16],
                                           const uint32_t (&wl)[16],
                                           const uint32_t (&wt)[16], int rg,
                                           uint32_t q, uint32_t qn,
                                           uint32_t ce, uint32_t *xt) {
  if constexpr (!kSmall) {
#pragma unroll
    for (int k = 0; k < 16; k++) x[k] = umin(x[k], x[k] - q);
  }
  gs16<kSmall>(x, wl, q, qn);
#pragma unroll
  for (int k = 0; k < 16; k++) xt[17 * rg + k] = x[k];
  wave_lds_sync();
#pragma unroll
  for (int k = 0; k < 16; k++) x[k] = xt[17 * k + rg];
  gs16<kSmall>(x, wt, q, qn);
  wave_lds_sync();
#pragma unroll
  for (int k = 0; k < 16; k++) {
    uint32_t v = mont_lo(x[k], ce, qn, q);
    v = umin(v, v - q);
    v = v > (q >> 1) ? v - q : v;
    xt[17 * k + rg] = (v + 0x808080u) ^ 0x808080u;
  }
}

// Forward column stages of one column in xt (values in [0, 2q)); x gets rows
// 16 rg + k in the row pass's range.
template <bool kSmall>
__device__ __forceinline__ void fwd_column(uint32_t (&x)[16],
                                           const uint32_t (&wt)[16],
                                           const uint32_t (&wl)[16], int rg,
                                           uint32_t q, uint32_t qn,
                                           uint32_t *xt) {
#pragma unroll
  for (int k = 0; k < 16; k++) x[k] = xt[17 * k + rg];
  ct16<kSmall, true>(x, wt, q, qn);
#pragma unroll
  for (int k = 0; k < 16; k++) xt[17 * k + rg] = x[k];
  wave_lds_sync();
#pragma unroll
  for (int k = 0; k < 16; k++) x[k] = xt[17 * rg + k];
  ct16<kSmall, false>(x, wl, q, qn);
}

// what a lane needs of its destination limb
struct Dest {
  uint32_t q, qn;
  uint32_t wt[16], wl[16];
  uint32_t *dst;
};

template <int kChunks>
__global__ __launch_bounds__(kThreads) void switch_cols(chd_tables t,
                                                        chd_limb_map m,
                                                        SwitchBatch b,
                                                        int dst_per_part) {
  extern __shared__ __align__(16) uint32_t lds[];
  const chd_switch_job jb = b.job[blockIdx.y];
  const int k_lo = blockIdx.z * dst_per_part;
  if (k_lo >= jb.dst_len) return;
  const int nd = min(dst_per_part, jb.dst_len - k_lo);
  const int ns = jb.src_len;
  // column block and first column inside it; the 4 / kW workgroups of a
  // block get ids 8 apart (one XCD, whose L2 joins their pieces of a line)
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int cb = (slot / kSub) * 8 + xcd;
  const int sub = (slot % kSub) * kW;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & (kW - 1);
  const int rg = (lane / kW) & 15;
  const int lj = lane / (16 * kW);  // limb of the wave's 4 / kW
  // word of row rg of this lane's column; row rg + 16 k is 64 k words on
  const uint32_t gword = static_cast<uint32_t>((cb * 256 + rg) * 4 + sub + c);
  uint32_t *const dst_lds = lds + ns * kW * kColWords;

  // BConv steps of this wave: 32 coefficients x 16 destinations each,
  // consecutive, so that a tile's digit planes are loaded once. The first
  // tile's are requested here, behind the source columns.
  constexpr int kPairs = 8 * kW;
  const int nk = kChunks == 1 ? 1 : (ns + kChunkSrc - 1) / kChunkSrc;
  const int tile0 = k_lo >> 4;
  const int all_tiles = (jb.dst_len + 15) >> 4;
  const int rem = jb.dst_len & 15;
  const bool narrow = ns <= 8;
  const bool packed = narrow && rem != 0 && rem <= 8;
  const int units = ((nd + 15) >> 4) * kPairs;
  const int u_lo = wave * units / kWaves, u_hi = (wave + 1) * units / kWaves;
  const int r = lane & 15, g = lane >> 4;
  v4i bp[kChunks][4];
  uint32_t p = 0;
  int32_t pinv = 0;
  auto load_tile = [&](int tt) {
    const v4i *tab = static_cast<const v4i *>(jb.table) +
                     static_cast<size_t>(tt) * nk * 256 + lane;
#pragma unroll
    for (int ch = 0; ch < kChunks; ch++) {
      const v4i z = {0, 0, 0, 0};
#pragma unroll
      for (int pl = 0; pl < 4; pl++)
        bp[ch][pl] = ch < nk ? tab[256 * ch + 64 * pl] : z;
    }
    // dead columns beyond the last destination take its prime; the packed
    // tile's column c stands for destination 16 tt + (c & 7)
    const int col = packed && tt == all_tiles - 1 ? (r & 7) : r;
    const int kc = min(tt * 16 + col, jb.dst_len - 1);
    const int pos = kc + (kc >= jb.skip_lo ? jb.skip_len : 0);
    const int ti = m.tab_off + pos + (pos >= m.num_q ? m.tab_gap : 0);
    p = t.q[ti];
    pinv = t.qinv[ti];
  };
  int tile = tile0 + u_lo / kPairs;
  load_tile(tile);

  // 1. the source columns, as byte digits, into LDS
  for (int s0 = wave * kSub; s0 < ns; s0 += kWaves * kSub) {
    const int i = min(s0 + lj, ns - 1);
    const int ti = jb.src_tab + i + (i >= jb.src_num_q ? jb.src_tab_gap : 0);
    const uint32_t *src = jb.src + (static_cast<size_t>(i) << kLogN) + gword;
    uint32_t x[16];
#pragma unroll
    for (int k = 0; k < 16; k++) x[k] = src[64 * k];
    const uint32_t q = t.q[ti];
    const uint32_t qn = 0u - static_cast<uint32_t>(t.qinv[ti]);
    const uint32_t ce = jb.src_cst[i];
    const uint32_t *itw = t.itw + (static_cast<size_t>(ti) << kLogN);
    uint32_t wl[16], wt[16];
    load_low(itw, rg, wl);
    load_top(itw, wt);
    uint32_t *xt = lds + (i * kW + c) * kColWords;
    if (__all(q < (1u << 30)))
      inv_column<true>(x, wl, wt, rg, q, qn, ce, xt);
    else
      inv_column<false>(x, wl, wt, rg, q, qn, ce, xt);
  }
  __syncthreads();

  // prime, twiddles and output column of this lane's destination in the
  // wave's slot d0 (a lane beyond the last destination repeats it)
  auto load_dest = [&](Dest &d, int d0) {
    const int kk = k_lo + min(d0 + lj, nd - 1);
    const int pos = kk + (kk >= jb.skip_lo ? jb.skip_len : 0);
    const int ti = m.tab_off + pos + (pos >= m.num_q ? m.tab_gap : 0);
    const uint32_t *tw = t.tw + (static_cast<size_t>(ti) << kLogN);
    load_top(tw, d.wt);
    load_low(tw, rg, d.wl);
    d.q = t.q[ti];
    d.qn = 0u - static_cast<uint32_t>(t.qinv[ti]);
    d.dst = jb.dst + (static_cast<size_t>(pos) << kLogN) + gword;
  };

  // 2. BConv (bconv.hip's operand layout). Operand rows beyond the sources
  // meet zero digits of the table, so they may hold anything: they re-read
  // the last source.
  Dest de;
  {
    // this lane's operand words of a step's two coefficient tiles, step
    // offset apart (of narrow jobs, lanes 32..63 read the second tile's)
    const uint32_t *src_a[kChunks][4], *src_b[kChunks][4];
#pragma unroll
    for (int ch = 0; ch < kChunks; ch++)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int i = ch == 0 && narrow ? 4 * (g & 1) + j
                                        : kChunkSrc * ch + 4 * g + j;
        src_b[ch][j] = lds + min(i, ns - 1) * (kW * kColWords) + r + 17;
        src_a[ch][j] = src_b[ch][j] - (ch == 0 && narrow && g >= 2 ? 0 : 17);
      }
    for (int u = u_lo; u < u_hi; u++) {
      const int tl = u / kPairs, pr = u % kPairs;
      if (tile0 + tl != tile) {
        tile = tile0 + tl;
        load_tile(tile);
      }
      const bool pk = packed && tile == all_tiles - 1;
      // column pr / 8, 16-row groups 2 (pr % 8) and the next
      const int step = (pr >> 3) * kColWords + 34 * (pr & 7);
      v4i a[kChunks][2];
#pragma unroll
      for (int ch = 0; ch < kChunks; ch++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
          a[ch][0][j] = static_cast<int>(src_a[ch][j][step]);
          a[ch][1][j] = static_cast<int>(src_b[ch][j][step]);
        }
      if (u == u_hi - 1) load_dest(de, wave * kSub);
      // planes of one output joined and reduced (bconv.hip), in (0, 2p)
      auto finish = [&](const v4i(&d)[4], uint32_t *o) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const int32_t lo = d[0][i] + d[1][i] * 256;
          const int32_t hi = d[2][i] + d[3][i] * 256;
          const int64_t y = static_cast<int64_t>(hi) * 65536 + lo;
          o[i] = static_cast<uint32_t>(mont_reduce_lazy(y, p, pinv)) + p;
        }
      };
      const v4i z = {0, 0, 0, 0};
      if (!pk) {
        uint32_t *o =
            dst_lds + (tl * 16 + r) * (kW * kColWords) + 4 * g + step;
        v4i d[2][4];
#pragma unroll
        for (int mt = 0; mt < 2; mt++)
#pragma unroll
          for (int pl = 0; pl < 4; pl++) {
            d[mt][pl] = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                a[0][mt], bp[0][pl], z, 0, 0, 0);
#pragma unroll
            for (int ch = 1; ch < kChunks; ch++)
              d[mt][pl] = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                  a[ch][mt], bp[ch][pl], d[mt][pl], 0, 0, 0);
          }
        if (tl * 16 + r < nd) {
          finish(d[0], o);
          finish(d[1], o + 17);
        }
      } else {
        v4i d[4];
#pragma unroll
        for (int pl = 0; pl < 4; pl++)
          d[pl] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[0][0], bp[0][pl], z,
                                                        0, 0, 0);
        const int k = tl * 16 + (r & 7);
        if (k < nd)
          finish(d, dst_lds + k * (kW * kColWords) + 17 * (r >> 3) + 4 * g +
                        step);
      }
    }
  }
  __syncthreads();

  // 3. the destination columns
  for (int d0 = wave * kSub; d0 < nd; d0 += kWaves * kSub) {
    if (d0 != wave * kSub) load_dest(de, d0);
    uint32_t *xt = dst_lds + (min(d0 + lj, nd - 1) * kW + c) * kColWords;
    uint32_t x[16];
    if (__all(de.q < (1u << 30)))
      fwd_column<true>(x, de.wt, de.wl, rg, de.q, de.qn, xt);
    else
      fwd_column<false>(x, de.wt, de.wl, rg, de.q, de.qn, xt);
    if (d0 + lj < nd) {
#pragma unroll
      for (int i = 0; i < 16; i++) de.dst[64 * i] = x[i];
    }
  }
}

}  // namespace
}  // namespace chd

using namespace chd;

extern "C" int chd_k_switch_cols(const chd_tables *t, const chd_limb_map *m,
                                 const chd_switch_job *jobs, int num_jobs,
                                 void *stream) {
  if (!t || !m || !jobs || num_jobs < 1 || num_jobs > CHD_MAX_BCONV_JOBS)
    return set_error(CHD_ERR_ARG, "chd_k_switch_cols: invalid argument");
  SwitchBatch b{};
  int max_src = 0, max_dst = 0;
  for (int j = 0; j < num_jobs; j++) {
    const chd_switch_job &jb = jobs[j];
    if (!jb.dst || !jb.src || !jb.src_cst || !jb.table || jb.src_len < 1 ||
        jb.src_len > kMaxSrc || jb.dst_len < 1 || jb.skip_len < 0)
      return set_error(CHD_ERR_ARG, "chd_k_switch_cols: invalid job");
    b.job[j] = jb;
    max_src = std::max(max_src, jb.src_len);
    max_dst = std::max(max_dst, jb.dst_len);
  }
  // Limbs a workgroup holds: with more workgroups than CUs, half a CU's LDS
  // (two workgroups per CU), otherwise all of it. What does not fit runs as
  // parts of whole 16-destination tiles, each with its own copy of the
  // sources (two parts of a product's launches took 82.4 against 81.7 us).
  constexpr int kLimbBytes = kW * kColWords * 4;
  constexpr int kLds = 160 << 10;
  const int half_limbs = kLds / 2 / kLimbBytes, all_limbs = kLds / kLimbBytes;
  int limbs = kTiles * num_jobs > 256 ? half_limbs : all_limbs;
  if (limbs < max_src + std::min(16, max_dst)) limbs = all_limbs;
  int per = max_dst;
  if (max_src + max_dst > limbs) {
    const int fit = (limbs - max_src) / 16 * 16;
    const int parts = (max_dst + fit - 1) / fit;
    per = ((max_dst + parts - 1) / parts + 15) / 16 * 16;
  }
  const dim3 g(kTiles, num_jobs, (max_dst + per - 1) / per);
  const size_t lds = static_cast<size_t>(max_src + per) * kLimbBytes;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (max_src <= kChunkSrc)
    hipLaunchKernelGGL(switch_cols<1>, g, dim3(kThreads), lds, s, *t, *m, b,
                       per);
  else
    hipLaunchKernelGGL(switch_cols<2>, g, dim3(kThreads), lds, s, *t, *m, b,
                       per);
  return check_launch("chd_k_switch_cols");
}
