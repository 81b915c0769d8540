// The volcano factor of the reference's -A mode with any rank: X_nm = +-1,
// M = X diag(w) X^T with w_m = (-1)^m / N (makeu1 / makeu2 / m1 / m2,
// kuramoto.cu:62-143).  The reference regenerates the signs from Philox
// counters inside m1 / m2 and never stores them; here they are drawn once on
// the device from the library's own counter-based Philox stream (the same
// bits as the host generator sign_factor in kmt_rng.h: element e = n K + m is
// bit e mod 128 of block e / 128) and kept packed at one bit per entry, once
// per int8 pass, in that pass's tile order (sign_tile_word):
//   pass 2 tiles: row n, word q: m = 32 q + b in bit b (zero past K)
//   pass 1 tiles: row m, word q: n = 32 q + b in bit b (zero past N)
// (1.25 GB each at N = K = 10^5, against 40 GB for X in FP32), each with one
// more row of ones (k < the pass's k range) and zero rows up to its padded
// row count.
//
// Coupling on the int8 matrix cores with exact integer sums, four launches
// per stage (a stand-alone RHS: five).  (cos, sin)_n as 56-bit fixed point
// (2^-54 units) in 7 signed base-256 digits each are the B operand of pass 1,
// written by the launch that forms the vector (sign_stage_kernel,
// sign_emit_kernel) or, for a given vector, by sign_limbs_kernel:
//   sign_mfma_kernel   pass 1 over the pass-1 tiles: P_m = sum_n bit(m, n) * digit(n),
//                      per digit and per range of n, plus T = sum_n digit(n)
//   sign_gram_kernel   sum_n X_nm v_n = 2 P_m - T (X = 2 bit - 1) combined to
//                      double, G_m = w_m * that, and G as digits: the B
//                      operand of pass 2
//   sign_mfma_kernel   pass 2 over the pass-2 tiles: the same with rows n, k = m
//   sign_stage_kernel  C_n, S_n = 2 P_n - T combined, then the stage epilogue
// Each digit's sum over k is exact in int32 (|sum| <= 128 k < 2^31 for
// k < 2^24), so every coupling sum is the exact sum of the fixed-point
// inputs rounded once to double: of the oracle's factored path (kuramoto.cu:
// 62-101 restated) it differs only by the inputs' rounding to 2^-54 (cos,
// sin and |G_m| <= 1, as w_m = +-1/N) and by the oracle's own rounding of its
// sequential double additions.  Deterministic.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "kmt_kernels.hpp"

namespace kmt {

constexpr uint32_t kSignKeyTag = 0x4B4D5441u;     // the host generator's key tag
constexpr uint32_t kSignStream = 0x52410000u;     // its Rademacher stream

// Philox4x32-10 (Salmon et al., SC'11), the host generator's round function.
__device__ __forceinline__ void philox10(uint32_t x[4], uint32_t k0, uint32_t k1) {
#pragma unroll
  for (int round = 0; round < 10; ++round) {
    const uint32_t hb = __umulhi(0xCD9E8D57u, x[2]), lb = 0xCD9E8D57u * x[2];
    const uint32_t ha = __umulhi(0xD2511F53u, x[0]), la = 0xD2511F53u * x[0];
    x[0] = hb ^ x[1] ^ k0;
    x[1] = lb;
    x[2] = ha ^ x[3] ^ k1;
    x[3] = la;
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
}

// Word W of the sign stream: elements 32 W .. 32 W + 31 (bit b -> element 32 W + b).
__device__ __forceinline__ uint32_t sign_stream_word(uint64_t W, uint32_t seed) {
  uint32_t x[4] = {(uint32_t)(W >> 2), (uint32_t)(W >> 34), kSignStream, 0u};
  philox10(x, seed, kSignKeyTag);
  const uint32_t sel = (uint32_t)(W & 3);
  return sel == 0 ? x[0] : sel == 1 ? x[1] : sel == 2 ? x[2] : x[3];
}

// Tile order of a pass's bits: rows in groups of 256 (a workgroup's four waves
// of four 16-row MFMA tiles), words in pairs of 32 (1024 k, two super-blocks);
// the group's 256 rows x 32 words of pair P are 32 KB of consecutive memory,
// 8 KB per wave in the order it loads them: load (t, s) of lane (g, rl) is the
// 16 bytes of row 16 t + rl of the wave, words 32 P + 8 g + 4 s .. + 3, at
// 16-byte slot (2 t + s) 64 + 16 g + rl.  A workgroup thus streams one
// contiguous run as P advances (row-major bits gave each lane's row 128 bytes
// every pair, rows 12.5 KB apart at N = 10^5, and HBM served that at about
// half its rate; 8 KB runs per wave, 800 KB apart, were 2.5% slower).
__host__ __device__ __forceinline__ size_t sign_tile_word(long r, long q, long npairs) {
  const long rgb = r >> 8, w = (r >> 6) & 3, t = (r >> 4) & 3, rl = r & 15;
  const long P = q >> 5, g = (q >> 3) & 3, s = (q >> 2) & 1, e = q & 3;
  return (((((size_t)rgb * npairs + P) * 4 + w) * 8 + (2 * t + s)) * 64 + (16 * g + rl)) * 4 + e;
}

// Row n of the pass-2 tiles, word q: signs of m = 32 q .. 32 q + 31 (m < K):
// stream elements n K + 32 q + b, i.e. 32 consecutive stream bits from
// position e0 = n K + 32 q (at most two stream words).  One thread per word
// of the rows n < N, in tile order (coalesced stores).
[[maybe_unused]] static __global__ __launch_bounds__(kBlock) void gen_sign_bits_kernel(uint32_t *tiles, long N, long K,
                                                                                      long npairs, uint32_t seed) {
  const long o = (long)blockIdx.x * kBlock + threadIdx.x;
  if (o >= (N + 255) / 256 * npairs * 8192) return;
  const long piece = o >> 2, lane = piece & 63, ts = (piece >> 6) & 7, w = (piece >> 9) & 3, tile = piece >> 11;
  const long n = 256 * (tile / npairs) + 64 * w + 16 * (ts >> 1) + (lane & 15);
  const long q = 32 * (tile % npairs) + 8 * (lane >> 4) + 4 * (ts & 1) + (o & 3);
  if (n >= N) return;  // the ones row and zero rows are written separately
  uint32_t word = 0;
  if (32 * q < K) {
    const long nb = K - 32 * q < 32 ? K - 32 * q : 32;
    const uint64_t e0 = (uint64_t)n * (uint64_t)K + (uint64_t)(32 * q);
    const uint32_t sh = (uint32_t)(e0 & 31);
    word = sign_stream_word(e0 >> 5, seed) >> sh;
    if (sh != 0 && sh + nb > 32) word |= sign_stream_word((e0 >> 5) + 1, seed) << (32 - sh);
    if (nb < 32) word &= (1u << nb) - 1u;
  }
  tiles[o] = word;
}

// The ones row (row `rows`) of a pass's tiles: word q = ones[q].
[[maybe_unused]] static __global__ __launch_bounds__(kBlock) void sign_tile_ones_kernel(uint32_t *tiles, long rows,
                                                                                       const uint32_t *ones,
                                                                                       long npairs) {
  const long q = (long)blockIdx.x * kBlock + threadIdx.x;
  if (q < 32 * npairs) tiles[sign_tile_word(rows, q, npairs)] = ones[q];
}

// Pass-1 tiles from pass-2 tiles, 32 x 64 bit blocks: lane l holds row
// n0 + l's word q; the ballot of bit b over the wave is column m = 32 q + b
// for those 64 rows, i.e. words n0 / 32 and n0 / 32 + 1 of pass-1 row m.
// Lane b (< 32) writes row m = 32 q + b (rows m >= K get zero words; the
// ones row is written afterwards).
[[maybe_unused]] static __global__ __launch_bounds__(kBlock) void transpose_sign_bits_kernel(const uint32_t *tiles2, long N,
                                                                                            long npairs2, long Kw,
                                                                                            uint32_t *tiles1,
                                                                                            long npairs1) {
  const long wave = ((long)blockIdx.x * kBlock + threadIdx.x) / kWave;
  const int lane = threadIdx.x & (kWave - 1);
  const long nblk = (N + 63) / 64;
  if (wave >= nblk * Kw) return;  // whole waves: the ballot needs every lane
  const long q = wave / nblk, n0 = (wave % nblk) * 64;
  const uint32_t w = (n0 + lane < N) ? tiles2[sign_tile_word(n0 + lane, q, npairs2)] : 0u;
  uint32_t lo = 0, hi = 0;
#pragma unroll
  for (int b = 0; b < 32; ++b) {
    const unsigned long long m = __ballot((w >> b) & 1u);
    if (lane == b) {
      lo = (uint32_t)m;
      hi = (uint32_t)(m >> 32);
    }
  }
  if (lane < 32) {
    const long m = 32 * q + lane, c = n0 / 32;
    tiles1[sign_tile_word(m, c, npairs1)] = lo;
    if (c + 1 < 32 * npairs1) tiles1[sign_tile_word(m, c + 1, npairs1)] = hi;
  }
}

// ---------------------------------------------------------------------
// The int8 passes.  An MFMA v_mfma_i32_16x16x64_i8 multiplies a 16 x 64 int8
// A tile by a 64 x 16 int8 B tile into 16 x 16 int32: lane l holds A row l%16
// and B column l%16 with 16 bytes each for its quarter g = l/16 of the 64 k,
// and D rows 4g..4g+3 of column l%16.  A = the bits as bytes 0/1; B = 16
// columns: the 7 digits of the cos (or G_c) value in 0..6, of sin (G_s) in
// 7..13, zero in 14 and 15.
//
// k is walked in pairs of 512-wide super-blocks (32 bit words = 128 bytes
// per row).  Lane (row, g) loads words 32 P + 8 g .. + 7 of its row as two
// 16-byte vectors from the pass's tiles (sign_tile_word: the wave's 8 KB of
// the pair are consecutive); super-block S = 2 P + s takes words
// 32 P + 8 g + 4 s + u, u = 0..3.  For bit j = 0..3 of half h = 0, 1 the A
// operand is the four dwords (word u >> 4 h) & (0x01010101 << j): byte i of
// dword u is 2^j times bit 8 i + 4 h + j, k = 32 (32 P + 8 g + 4 s + u) + 8 i
// + 4 h + j.  The bits are not moved to the bytes' low end (that costs a shift
// per dword more): the four j accumulate apart, each a sum times 2^j, at most
// 2^3 2^7 2^20 / 4 < 2^29, and are shifted and added once at the end.  The B
// operand of (S, j, h) is stored in exactly that order (sign_bfrag_offset),
// 1 KB per MFMA, 8 KB per super-block, so the expansion of the bits costs a
// little over one VALU operation per 4 entries and no lane exchange.
// ---------------------------------------------------------------------
typedef int i32x4_t __attribute__((ext_vector_type(4)));
// Register sets of the pass's ring: one pair in use, kSignPF - 1 in flight.
constexpr int kSignPF = 2;

template <int I, int U, class F> __device__ __forceinline__ void sign_unroll(F &&f) {
  if constexpr (I < U) {
    f(std::integral_constant<int, I>{});
    sign_unroll<I + 1, U>(f);
  }
}
constexpr int kSignSB = 512;                          // k per super-block
constexpr long kSignBias = 0x80808080808080LL;        // 128 * sum_l 256^l, l < 7
constexpr double kSignScale = 0x1p54;                 // fixed point: 2^-54 units
// Largest N and K: a digit sum over k (2 P - T) is at most 3 * 128 k in
// magnitude, 384 * 2^20 < 2^28.6 here, which keeps sign_combine exact.
constexpr long kSignMaxDim = 1L << 20;

// byte of column c (0..15) for index k in the B fragments
__device__ __forceinline__ size_t sign_bfrag_offset(long k, int c) {
  const long q = k >> 5;
  const long S = 2 * (q >> 5) + ((q >> 2) & 1);
  const int g = (int)((q >> 3) & 3), u = (int)(q & 3);
  const int b = (int)(k & 31), i = b >> 3, h = (b >> 2) & 1, j = b & 3;
  return ((((size_t)S * 4 + j) * 2 + h) * 64 + (c + 16 * g)) * 16 + u * 4 + i;
}

// The 7 signed base-256 digits of round(v 2^54), |v| <= 1: e = d + bias is
// non-negative and below 2^56, and digit l = byte l of e minus 128 (as a
// byte: byte ^ 0x80), so that d = sum_l digit_l 256^l.  Bytes 0 .. 6 of the
// result (byte 7 zero).
__device__ __forceinline__ uint64_t sign_digits(double v) {
  const uint64_t e = (uint64_t)(__double2ll_rn(v * kSignScale) + kSignBias);
  return (e ^ 0x80808080808080ull) & 0xFFFFFFFFFFFFFFull;
}

// One k's 16 columns (digits of c in 0..6, of s in 7..13) of every thread of
// a workgroup, k = kBlock blockIdx.x + thread, into the B fragments: through
// LDS, so that each thread stores the 16 consecutive bytes of one (j, h,
// column) of a 128-wide stretch of k (a byte at a time, 16 stores 16 bytes
// apart, took most of the 4 us that a launch of its own spent on the digits
// at N = 10^4; with them in the launch that forms the vector, and the sums'
// 16-byte loads, an attempt there went from 237 to 212-225 us).
__device__ __forceinline__ void sign_write_frags(double c, double s, bool zero, uint32_t (&sh)[kBlock][4],
                                                 uint8_t *__restrict__ bfrag) {
  const int tid = threadIdx.x;
  uint64_t lo = 0, hi = 0;
  if (!zero) {
    const uint64_t dc = sign_digits(c), ds = sign_digits(s);
    lo = dc | ds << 56;
    hi = ds >> 8;
  }
  *reinterpret_cast<u32x4 *>(sh[tid]) = u32x4{(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)};
  __syncthreads();
  const int grp = tid >> 7, j = (tid >> 5) & 3, h = (tid >> 4) & 1, col = tid & 15;
  const uint8_t *src = reinterpret_cast<const uint8_t *>(sh) + (grp * 128 + 4 * h + j) * 16 + col;
  uint32_t w[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    w[u] = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) w[u] |= (uint32_t)src[(32 * u + 8 * i) * 16] << (8 * i);
  }
  const long k = (long)blockIdx.x * kBlock + grp * 128 + 4 * h + j;
  *reinterpret_cast<u32x4 *>(bfrag + sign_bfrag_offset(k, col)) = u32x4{w[0], w[1], w[2], w[3]};
}

// sum_l s_l 256^l 2^-54 rounded once to double: |s_l| < 2^28.6, so the low
// four digits (< 2^52.6) and the high three (< 2^44.6) are exact int64 and
// exact doubles, and one fma rounds their sum.
__device__ __forceinline__ double sign_combine(const long long (&s)[7]) {
  const long long lo = s[0] + s[1] * 256LL + s[2] * 65536LL + s[3] * 16777216LL;
  const long long hi = s[4] + s[5] * 256LL + s[6] * 65536LL;
  return __builtin_fma((double)hi, 0x1p32, (double)lo) * 0x1p-54;
}

// B fragments of pass 1 from a given vector pair: one thread per k = n (zero
// columns 14, 15 and zero rows for k >= N up to the grid's end; past it the
// buffer stays as cleared).
template <class R>
__global__ __launch_bounds__(kBlock) void sign_limbs_kernel(const R *__restrict__ vc, const R *__restrict__ vs, long N,
                                                             uint8_t *__restrict__ bfrag) {
  __shared__ __align__(16) uint32_t sh[kBlock][4];
  const long k = (long)blockIdx.x * kBlock + threadIdx.x;
  const long kk = k < N ? k : N - 1;
  sign_write_frags((double)vc[kk], (double)vs[kk], k >= N, sh, bfrag);
}

// The line of `units` (row group, pair) units over G workgroups: workgroup b
// owns [sign_first_unit(b), sign_first_unit(b + 1)); the owner of unit u.
__host__ __device__ __forceinline__ long sign_first_unit(long b, long units, long G) { return b * units / G; }
__host__ __device__ __forceinline__ long sign_unit_owner(long u, long units, long G) { return ((u + 1) * G - 1) / units; }

// The A operand of class (j, h): bit 4 h + j of every byte of the lane's four
// words, kept in place after the shift by 4 h, so every byte is 0 or 2^j.
__device__ __forceinline__ i32x4_t sign_class(const u32x4 w, int j, int h) {
  const uint32_t m = 0x01010101u << j;
  return i32x4_t{(int)((w.x >> (4 * h)) & m), (int)((w.y >> (4 * h)) & m), (int)((w.z >> (4 * h)) & m),
                 (int)((w.w >> (4 * h)) & m)};
}

// One pass: part[sp][r][c] = the sum of slot sp's share of k over bit(r, k) *
// B[k][c], for the rows r < ldp of the pass's tiles (its bit rows, then the
// ones row: T_c = sum_k B[k][c], then zero rows).  The work is a line of
// units (row group of 256 rows, pair of super-blocks), row group major, cut
// into gridDim.x equal stretches: a workgroup takes its stretch in order and
// writes its sums whenever a row group or the stretch ends, into the slot
// that counts the workgroups of that row group (sums are exact integers, so
// the cut does not change a result; slots that a row group does not reach
// stay zero).  Equal stretches because no split count fits every size: one
// (row group, range of k) per workgroup left 1.53 rounds of resident
// workgroups at N = K = 10^5.
// A workgroup = 4 waves, wave w on NT 16-row tiles of the row group.  The B
// fragments of a pair (16 KB) are loaded once per workgroup, 64 bytes per
// thread, and shared through LDS (double-buffered, one barrier per pair);
// every thread's loads for pair P + kSignPF (its share of the B fragments
// before the MFMAs of pair P, its rows' bit words after them) are issued in
// the order they are used, so kSignPF - 1 pairs stay in flight behind the one
// in use.
// Bound: the stream of bits (1.25 GB per pass at N = K = 10^5) together with
// VALU issue.  With the bits expanded to bytes 0 / 1 (7.5 instructions per
// MFMA, VALU busy 61% of the time) a pass took 249 us, 5.0 TB/s; leaving each
// bit at its place (4.5 instructions, four accumulator sets, 231 VGPRs, 2
// waves per SIMD), a row group's pair 32 KB of consecutive memory and equal
// stretches: 233 us, 5.4 TB/s.  One right-hand side: 527 -> 497 us; N = K =
// 65535 245 -> 223; an attempt at N = K = 10^4 is unchanged by this kernel
// (400 units, 7.5 us, latency).
template <class R, int NT>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2, 2))) void sign_mfma_kernel(
    const u32x4 *__restrict__ tiles, const u32x4 *__restrict__ bfrag, int npairs, long units,
    int32_t *__restrict__ part, long ldp, const State<R> *st, int check_state) {
  constexpr int NW = kBlock / kWave;
  constexpr int BPT = 2 * 8 * kWave / kBlock;  // 16-byte B pieces per thread and pair
  __shared__ u32x4 bsh[2][2 * 8 * kWave];
  if (check_state && (!st->active || st->commit_pending)) return;
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const long G = gridDim.x, u0 = sign_first_unit(blockIdx.x, units, G), u1 = sign_first_unit(blockIdx.x + 1, units, G);
  if (u0 >= u1) return;
  const int g = lane >> 4, rl = lane & 15;
  static_assert(NT == 4, "tile order: 64 rows per wave");
  // the wave's 8 KB of unit u start at tw + 2048 u (16-byte slots); every
  // lane loads (no divergent branch around the loads, which would make the
  // compiler wait for every load in flight)
  const u32x4 *tw = tiles + (size_t)wave * 512 + lane;
  i32x4_t acc[4][NT];  // [j]: sums with bits as 2^j
  auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[j][t] = i32x4_t{0, 0, 0, 0};
  };
  // unit u: the rows' bit words; pair P: this thread's pieces of the pair's B
  // fragments (piece f = tid + kBlock j of the pair's 1024, in the pair's
  // order: super-block s, (j, h), lane).  Nothing here consumes a value.
  auto load_w = [&](long u, u32x4 (&W)[NT][2]) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      W[t][0] = tw[(size_t)u * NW * 512 + (2 * t) * 64];
      W[t][1] = tw[(size_t)u * NW * 512 + (2 * t + 1) * 64];
    }
  };
  auto load_b = [&](int P, u32x4 (&Bst)[BPT]) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < BPT; ++j) Bst[j] = bfrag[(size_t)P * 2 * 8 * kWave + tid + kBlock * j];
  };
  // the MFMAs of super-block s of a pair, B fragments from LDS buffer buf
  auto multiply = [&](const u32x4 (&W)[NT][2], int s, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const i32x4_t b = __builtin_bit_cast(i32x4_t, bsh[buf][(s * 8 + j * 2 + h) * kWave + lane]);
#pragma unroll
        for (int t = 0; t < NT; ++t)
          acc[j][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(sign_class(W[t][s], j, h), b, acc[j][t], 0, 0, 0);
      }
  };
  // One row group's part of the stretch at a time, pairs [p0, p1).  Ring of
  // kSignPF register sets, slot d holding pair P + d; loads past the end
  // re-read the last pair (harmless, and no branch).  (Carrying the ring over
  // into the next row group, with the sums written inside the pair loop, was
  // 6% slower per pair.)
  u32x4 W[kSignPF][NT][2], Bst[kSignPF][BPT];
#pragma unroll 1
  for (long u = u0; u < u1;) {
    const long rgb = u / npairs, base = rgb * npairs;
    const int p0 = (int)(u - base), p1 = u1 - base < npairs ? (int)(u1 - base) : npairs, plast = p1 - 1;
    auto cl = [&](int p) __attribute__((always_inline)) { return p < plast ? p : plast; };
    sign_unroll<0, kSignPF>([&](auto i) __attribute__((always_inline)) {
      constexpr int d = decltype(i)::value;
      load_b(cl(p0 + d), Bst[d]);
      load_w(base + cl(p0 + d), W[d]);
    });
    clear();
    // pair P + d from slot d: its B fragments to LDS and a barrier, the slot's
    // B pieces refilled with pair P + d + kSignPF, the pair's MFMAs, then the
    // slot's bit words refilled (after the MFMAs that read them)
    auto pair = [&](auto i, int P, bool refill) __attribute__((always_inline)) {
      constexpr int d = decltype(i)::value;
      const int buf = (P + d - p0) & 1;
#pragma unroll
      for (int j = 0; j < BPT; ++j) bsh[buf][tid + kBlock * j] = Bst[d][j];
      __syncthreads();
      if (refill) load_b(cl(P + d + kSignPF), Bst[d]);
      __builtin_amdgcn_sched_barrier(0);
      multiply(W[d], 0, buf);
      multiply(W[d], 1, buf);
      __builtin_amdgcn_sched_barrier(0);
      if (refill) load_w(base + cl(P + d + kSignPF), W[d]);
      __builtin_amdgcn_sched_barrier(0);
    };
    int P = p0;
    for (; P + kSignPF <= p1; P += kSignPF)
      sign_unroll<0, kSignPF>([&](auto i) __attribute__((always_inline)) { pair(i, P, true); });
    sign_unroll<0, kSignPF - 1>([&](auto i) __attribute__((always_inline)) {
      if (P + decltype(i)::value < p1) pair(i, P, false);
    });
    __syncthreads();  // the next row group starts at buffer 0 again
    const long slot = blockIdx.x - sign_unit_owner(base, units, G);
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const long r = (rgb * NW + wave) * 16 * NT + 16 * t + 4 * g + v;
        // acc[j] is 2^j times its classes' sum: exact shifts
        part[((size_t)slot * ldp + r) * 16 + rl] =
            acc[0][t][v] + (acc[1][t][v] >> 1) + (acc[2][t][v] >> 2) + (acc[3][t][v] >> 3);
      }
    u = base + p1;
  }
}

// The 14 digit sums of row r (2 P - T over the slots), exact in int64.
__device__ __forceinline__ void sign_row_sums(const int32_t *__restrict__ part, int nsplit, long ldp, long r,
                                              long trow, long long (&sc)[7], long long (&ss)[7]) {
#pragma unroll
  for (int l = 0; l < 7; ++l) { sc[l] = 0; ss[l] = 0; }
#pragma unroll 2
  for (int sp = 0; sp < nsplit; ++sp) {
    const i32x4_t *pr = reinterpret_cast<const i32x4_t *>(part + ((size_t)sp * ldp + r) * 16);
    const i32x4_t *pt = reinterpret_cast<const i32x4_t *>(part + ((size_t)sp * ldp + trow) * 16);
    int32_t p[16], t[16];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const i32x4_t x = pr[q], y = pt[q];
      p[4 * q] = x.x, p[4 * q + 1] = x.y, p[4 * q + 2] = x.z, p[4 * q + 3] = x.w;
      t[4 * q] = y.x, t[4 * q + 1] = y.y, t[4 * q + 2] = y.z, t[4 * q + 3] = y.w;
    }
#pragma unroll
    for (int l = 0; l < 7; ++l) {
      sc[l] += 2LL * p[l] - t[l];
      ss[l] += 2LL * p[7 + l] - t[7 + l];
    }
  }
}

// G_m = w_m sum_n X_nm (cos, sin)_n from the pass-1 sums, written as the B
// fragments of pass 2 (one thread per k = m, zero past K).
template <class R>
__global__ __launch_bounds__(kBlock) void sign_gram_kernel(const int32_t *__restrict__ part, int nsplit, long ldp,
                                                            const R *__restrict__ w, long K,
                                                            uint8_t *__restrict__ bfrag, const State<R> *st,
                                                            int check_state) {
  if (check_state && (!st->active || st->commit_pending)) return;
  __shared__ __align__(16) uint32_t sh[kBlock][4];
  const long m = (long)blockIdx.x * kBlock + threadIdx.x;
  double c = 0.0, s = 0.0;
  if (m < K) {
    long long sc[7], ss[7];
    const double wm = (double)w[m];
    sign_row_sums(part, nsplit, ldp, m, K, sc, ss);
    c = sign_combine(sc) * wm;
    s = sign_combine(ss) * wm;
  }
  sign_write_frags(c, s, m >= K, sh, bfrag);
}

// C_n, S_n from the pass-2 sums, then the stage epilogue of row n; stages 2..6
// also write the digits of their output vector (the next pass 1's B operand),
// stage 7 one error partial per workgroup.
template <class R, int KIND>
__global__ __launch_bounds__(kBlock) void sign_stage_kernel(const int32_t *__restrict__ part, int nsplit, long ldp,
                                                             Vecs<R> v, uint8_t *__restrict__ bfrag) {
  const long i = (long)blockIdx.x * kBlock + threadIdx.x;
  // the epilogue's operands are in flight before the state check and the sums
  const RowOps<R, KIND> ops = row_load<R, KIND>(v, i < v.N ? i : v.N - 1);
  asm volatile("" ::: "memory");
  if constexpr (KIND >= 2) {
    if (v.check_state && (!v.st->active || v.st->commit_pending)) return;
  }
  __shared__ double errsq[kBlock];
  double sq = 0.0;
  R c = 0, s = 0;
  if (i < v.N) {
    double C = 0.0, S = 0.0;
    if (nsplit > 0) {
      long long sc[7], ss[7];
      sign_row_sums(part, nsplit, ldp, i, v.N, sc, ss);
      C = sign_combine(sc);
      S = sign_combine(ss);
    }
    sq = row_finish<R, KIND>(v, i, ops, (R)C, (R)S, &c, &s);
  }
  if constexpr (KIND >= 2 && KIND < 7) {
    __shared__ __align__(16) uint32_t sh[kBlock][4];
    if (bfrag) sign_write_frags((double)c, (double)s, i >= v.N, sh, bfrag);
  }
  if constexpr (KIND == 7) {
    const double tot = block_sum(sq, errsq);
    if (threadIdx.x == 0) v.err_part[blockIdx.x] = tot;
  }
}

// emit_commit_kernel that also writes the digits of the stage-2 vector.
template <class R>
__global__ __launch_bounds__(kBlock) void sign_emit_kernel(const EmitArgs<R> a, uint8_t *__restrict__ bfrag) {
  __shared__ __align__(16) uint32_t sh[kBlock][4];
  const long i = (long)blockIdx.x * kBlock + threadIdx.x;
  R c = 0, s = 0;
  if (emit_commit<R>(a, i, c, s)) sign_write_frags((double)c, (double)s, i >= a.N, sh, bfrag);
}

// Dense rows from the packed signs with the dense generator's chain
// (gen_adj_kernel): M_ij = sum_m fma(w_m, X_im X_jm, acc) in the working
// precision, X_im X_jm = +1 where the two bits agree, -1 where they differ.
// A workgroup owns ROWS rows and 256 columns; each thread reads its column's
// bit row (from the pass-2 tiles) one word (32 m) at a time, the rows'
// words are the same in every lane.
template <class R, class S, int ROWS>
__global__ __launch_bounds__(kBlock) void gen_adj_sign_kernel(const uint32_t *tiles, long npairs, const R *w, long K,
                                                               long N, long row0, long nrows, S *A, long lda,
                                                               R inv_scale) {
  const long i0 = row0 + (long)blockIdx.y * ROWS;
  const long j = (long)blockIdx.x * kBlock + threadIdx.x;
  const long jj = j < N ? j : N - 1;
  R acc[ROWS];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) acc[r] = (R)0;
  const long kw = (K + 31) / 32;
  for (long q = 0; q < kw; ++q) {
    const uint32_t wj = tiles[sign_tile_word(jj, q, npairs)];
    uint32_t wi[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      const long i = i0 + r < N ? i0 + r : N - 1;
      wi[r] = tiles[sign_tile_word(i, q, npairs)];
    }
    const int nb = K - 32 * q < 32 ? (int)(K - 32 * q) : 32;
    for (int b = 0; b < nb; ++b) {
      const R wm = w[32 * q + b];
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        const R x = (((wi[r] ^ wj) >> b) & 1u) ? (R)-1 : (R)1;
        acc[r] = rfma<R>(wm, x, acc[r]);
      }
    }
  }
  if (j < N) {
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
      if (i0 + r < row0 + nrows && i0 + r < N)
        A[(size_t)(i0 + r - row0) * lda + j] = store_value<R, S>(acc[r], inv_scale);
  }
}

}  // namespace kmt
