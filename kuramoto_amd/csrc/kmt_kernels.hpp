// HIP device code of the integrator (gfx950 / CDNA4, wave64).
//
// One DP45 attempt is 8 launches on one stream (captured in a hipGraph):
//   stage_kernel<2..7>  A streamed from HBM once per stage for both cos and
//                       sin; the epilogue writes k_s and the next stage's
//                       (cos, sin) of y + h*sum a_{s+1,j} k_j (stage 6 also
//                       keeps the 5th-order solution; stage 7 forms the
//                       embedded error and a per-workgroup sum of squares)
//   control_kernel      error norm, accept/reject, step-size update,
//                       accepted-step log, output times crossed, ring and
//                       output bookkeeping, end-of-run detection; also the
//                       order parameter of the rows the previous attempt
//                       emitted
//   emit_commit_kernel  dense output at the crossed output times + order
//                       parameter partial sums, then commit (ylast <- y,
//                       y <- y5, k1 <- k7) and the next attempt's stage-2
//                       (cos, sin)
// and after the last attempt of a graph
//   finalize_kernel     order parameter of the rows that attempt emitted
// Reference counterparts: dp45.cu:34-164 (stages, error, controller, FSAL,
// interpolation) and kuramoto.cu:42-55, :104-126, :164-249 (RHS, order
// parameter, output grid).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace kmt {

constexpr int kBlock = 256;  // threads per workgroup (4 waves of 64)
constexpr int kWave = 64;

// ---------------------------------------------------------------------
// Dormand–Prince 4(5) coefficients (dp45.cu:5-21).  Each entry is the same
// double expression as the reference, rounded to the working precision.
// ---------------------------------------------------------------------
namespace tab {
constexpr double A[6][6] = {
    {1.0 / 5, 0, 0, 0, 0, 0},
    {3.0 / 40, 9.0 / 40, 0, 0, 0, 0},
    {44.0 / 45, -56.0 / 15, 32.0 / 9, 0, 0, 0},
    {19372.0 / 6561, -25360.0 / 2187, 64448.0 / 6561, -212.0 / 729, 0, 0},
    {9017.0 / 3168, -355.0 / 33, 46732.0 / 5247, 49.0 / 176, -5103.0 / 18656, 0},
    {35.0 / 384, 0, 500.0 / 1113, 125.0 / 192, -2187.0 / 6784, 11.0 / 84}};
constexpr double E[7] = {-71.0 / 57600, 0, 71.0 / 16695, -71.0 / 1920, 17253.0 / 339200, -22.0 / 525, 1.0 / 40};
constexpr double P[7][4] = {
    {1.0, -8048581381.0 / 2820520608, 8663915743.0 / 2820520608, -12715105075.0 / 11282082432},
    {0, 0, 0, 0},
    {0, 131558114200.0 / 32700410799, -68118460800.0 / 10900136933, 87487479700.0 / 32700410799},
    {0, -1754552775.0 / 470086768, 14199869525.0 / 1410260304, -10690763975.0 / 1880347072},
    {0, 127303824393.0 / 49829197408, -318862633887.0 / 49829197408, 701980252875.0 / 199316789632},
    {0, -282668133.0 / 205662961, 2019193451.0 / 616988883, -1453857185.0 / 822651844},
    {0, 40617522.0 / 29380423, -110615467.0 / 29380423, 69997945.0 / 29380423}};
}  // namespace tab

// ---------------------------------------------------------------------
// Device-resident integrator state (one per context).
// ---------------------------------------------------------------------
template <class R> struct State {
  R t, h, t_last, t1;
  R atl, rtl;
  int active;          // run in progress
  int commit_pending;  // accepted step awaiting output emission + commit
  int pend_lo, pend_hi;
  int eval_i, n_eval;
  int ring_count, ring_cap;
  int times_count, times_cap;
  int fixed;
  int last_accept;
  int error;
  // what emit_commit_kernel has to do for the attempt just controlled: rows
  // t_eval[job_lo .. job_lo + job_n) into ring slots from job_slot, then
  // job_mode; the rows' order parameters follow in the next control_kernel
  // (or finalize_kernel), which then clears fin_n
  int job_mode, job_lo, job_n, job_slot;
  int fin_n;
  long long accepted, rejected, attempts, rhs_evals;
  double norm;
};
constexpr int JOB_NONE = 0;    // nothing (run finished)
constexpr int JOB_STAGE2 = 1;  // rejected step or start of a run: stage-2 vector from (y, k1)
constexpr int JOB_EMIT = 2;    // outputs only (the ring is full before the last one)
constexpr int JOB_COMMIT = 3;  // outputs, commit, stage-2 vector

// Storage tags for the adjacency.
struct bf16_t { uint16_t bits; };
struct f16_t { uint16_t bits; };

// VEC: stored values per 16-byte load; Val: the type a stored value unpacks
// to; Acc: the type the coupling sums accumulate in.  Native FP32 storage
// accumulates in double: the sums are then the correctly rounded float of
// the exact sums up to the double rounding (the oracle rounds its double
// sums the same way), so FP32 runs do not depend on the summation order.
// 16-bit storage keeps FP32 accumulation.
template <class S> struct Store;
template <> struct Store<float> { static constexpr int VEC = 4; using Val = float; using Acc = double; };
template <> struct Store<double> { static constexpr int VEC = 2; using Val = double; using Acc = double; };
template <> struct Store<bf16_t> { static constexpr int VEC = 8; using Val = float; using Acc = float; };
template <> struct Store<f16_t> { static constexpr int VEC = 8; using Val = float; using Acc = float; };

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
// Note: reinterpret a loaded 16-byte vector as a whole (u32x4 -> f32x4) or
// copy an element into a scalar first.  hipcc 7.2 mis-compiles
// __builtin_bit_cast(float, v[q]) applied directly to a vector element (it
// reads lane 0 for every q).

__device__ __forceinline__ float bf16_lo(uint32_t w) { return __builtin_bit_cast(float, w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __builtin_bit_cast(float, w & 0xFFFF0000u); }
__device__ __forceinline__ float f16_lo(uint32_t w) { return (float)__builtin_bit_cast(_Float16, (uint16_t)(w & 0xFFFFu)); }
__device__ __forceinline__ float f16_hi(uint32_t w) { return (float)__builtin_bit_cast(_Float16, (uint16_t)(w >> 16)); }

// 16 bytes of the adjacency -> VEC values.
template <class S> __device__ __forceinline__ void unpack(const u32x4 v, typename Store<S>::Val *out);
template <> __device__ __forceinline__ void unpack<float>(const u32x4 v, float *o) {
  const f32x4 f = __builtin_bit_cast(f32x4, v);
  o[0] = f.x; o[1] = f.y; o[2] = f.z; o[3] = f.w;
}
template <> __device__ __forceinline__ void unpack<double>(const u32x4 v, double *o) {
  const uint32_t w0 = v.x, w1 = v.y, w2 = v.z, w3 = v.w;
  o[0] = __builtin_bit_cast(double, ((uint64_t)w1 << 32) | w0);
  o[1] = __builtin_bit_cast(double, ((uint64_t)w3 << 32) | w2);
}
template <> __device__ __forceinline__ void unpack<bf16_t>(const u32x4 v, float *o) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int q = 0; q < 4; ++q) { o[2 * q] = bf16_lo(w[q]); o[2 * q + 1] = bf16_hi(w[q]); }
}
template <> __device__ __forceinline__ void unpack<f16_t>(const u32x4 v, float *o) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int q = 0; q < 4; ++q) { o[2 * q] = f16_lo(w[q]); o[2 * q + 1] = f16_hi(w[q]); }
}

// VEC consecutive reals (16- or 32-byte aligned).
template <class R, int VEC> __device__ __forceinline__ void load_reals(const R *p, R *o) {
  constexpr int W = (int)(VEC * sizeof(R) / 16);
  static_assert(W >= 1, "vector load width");
#pragma unroll
  for (int w = 0; w < W; ++w) {
    const u32x4 v = *reinterpret_cast<const u32x4 *>(reinterpret_cast<const char *>(p) + 16 * w);
    unpack<R>(v, o + (16 / sizeof(R)) * w);
  }
}

// Working-precision math.  FP32 cos / sin are the float roundings of the
// double functions (within 1 ulp of the exact value), i.e. the correctly
// rounded float except within 2^-29 relative of a rounding boundary: FP32
// runs then do not depend on one float libm's last bit (the oracle rounds
// the same way).  With Cauchy frequencies the fast oscillators' phases
// reach 1e4, where one float ulp is 1e-3 rad, and a last-bit difference of
// a cos or sin moves the whole population by ~1e-4 within t = 1.
// Both come from one sincos: the same bits as cos() and sin() (compared over
// 2^31 arguments of every range), which each reduce the argument again (214
// against 111 double operations).
template <class R> __device__ __forceinline__ void rsincos(R x, R &c, R &s) {
  double ds, dc;
  sincos((double)x, &ds, &dc);
  c = (R)dc;
  s = (R)ds;
}
template <class R> __device__ __forceinline__ R rabs(R x) {
  if constexpr (sizeof(R) == 4) return fabsf(x); else return fabs(x);
}
template <class R> __device__ __forceinline__ R rfma(R a, R b, R c) {
  if constexpr (sizeof(R) == 4) return __builtin_fmaf(a, b, c); else return __builtin_fma(a, b, c);
}
template <class R> __device__ __forceinline__ R rmax(R a, R b) {
  if constexpr (sizeof(R) == 4) return fmaxf(a, b); else return fmax(a, b);
}

// Exchanges between the lanes of a wave (all 64 active) in registers: the
// swaps of the wave's halves and of its rows of 16, and DPP moves inside a
// row.  Through LDS (a lane permute) every level of a sum waits for an LDS
// round trip.
template <class T, class F> __device__ __forceinline__ T lane_words(T v, F f) {
  if constexpr (sizeof(T) == 4) {
    return __builtin_bit_cast(T, f(__builtin_bit_cast(uint32_t, v)));
  } else {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    return __builtin_bit_cast(T, (uint64_t)f((uint32_t)(u >> 32)) << 32 | f((uint32_t)u));
  }
}
template <int CTRL> __device__ __forceinline__ uint32_t dpp_move(uint32_t w) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)w, CTRL, 0xF, 0xF, true);
}
// the value of lane ^ OFF (OFF = 8, 4, 2, 1)
template <int OFF, class T> __device__ __forceinline__ T lane_xor(T v) {
  return lane_words(v, [](uint32_t w) {
    if constexpr (OFF == 8) return dpp_move<0x128>(w);                        // row rotated by 8
    else if constexpr (OFF == 4) return dpp_move<0x1B>(dpp_move<0x141>(w));  // halves mirrored (^ 7), quads mirrored (^ 3)
    else if constexpr (OFF == 2) return dpp_move<0x4E>(w);                    // quads 2 3 0 1
    else return dpp_move<0xB1>(w);                                            // quads 1 0 3 2
  });
}
// OFF = 32, 16: lanes with the bit clear get a[l] + a[l ^ OFF], the others
// b[l ^ OFF] + b[l]
template <int OFF, class T> __device__ __forceinline__ T lane_swap_sum(T a, T b) {
  auto swap = [](uint32_t &x, uint32_t &y) {
    if constexpr (OFF == 32) {
      const auto r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
      x = r[0], y = r[1];
    } else {
      const auto r = __builtin_amdgcn_permlane16_swap(x, y, false, false);
      x = r[0], y = r[1];
    }
  };
  if constexpr (sizeof(T) == 4) {
    uint32_t x = __builtin_bit_cast(uint32_t, a), y = __builtin_bit_cast(uint32_t, b);
    swap(x, y);
    return __builtin_bit_cast(T, x) + __builtin_bit_cast(T, y);
  } else {
    const uint64_t u = __builtin_bit_cast(uint64_t, a), w = __builtin_bit_cast(uint64_t, b);
    uint32_t xl = (uint32_t)u, yl = (uint32_t)w, xh = (uint32_t)(u >> 32), yh = (uint32_t)(w >> 32);
    swap(xl, yl);
    swap(xh, yh);
    return __builtin_bit_cast(T, (uint64_t)xh << 32 | xl) + __builtin_bit_cast(T, (uint64_t)yh << 32 | yl);
  }
}
// v + the partner's v at distance OFF
template <int OFF, class T> __device__ __forceinline__ T lane_pair_sum(T v) {
  if constexpr (OFF >= 16) return lane_swap_sum<OFF>(v, v);
  else return v + lane_xor<OFF>(v);
}
template <class T, int OFF = kWave / 2> __device__ __forceinline__ T wave_sum(T v) {
  if constexpr (OFF > 0) return wave_sum<T, OFF / 2>(lane_pair_sum<OFF>(v));
  else return v;
}

// The NV values v[0..NV) of every lane, each summed over the wave in
// wave_sum's order (the same bits): lane l returns the sum of value
// wave_slot<NV>(l).  At each distance half of the remaining values go to the
// partner lane, so NV = 16 takes 8 + 4 + 2 + 1 + 1 + 1 exchanges instead of
// 16 x 6.
template <int NV> __device__ __forceinline__ int wave_slot(int lane) {
  int slot = 0;
#pragma unroll
  for (int half = NV / 2, off = kWave / 2; half > 0; half /= 2, off /= 2) slot += (lane & off) ? half : 0;
  return slot;
}
template <class T, int HALF, int OFF, int NV> __device__ __forceinline__ T wave_reduce_from(T (&v)[NV], int lane) {
  if constexpr (HALF > 0) {
    const bool up = lane & OFF;
#pragma unroll
    for (int k = 0; k < HALF; ++k) {
      if constexpr (OFF >= 16) {
        v[k] = lane_swap_sum<OFF>(v[k], v[k + HALF]);
      } else {
        const T keep = up ? v[k + HALF] : v[k], send = up ? v[k] : v[k + HALF];
        v[k] = keep + lane_xor<OFF>(send);
      }
    }
    return wave_reduce_from<T, HALF / 2, OFF / 2>(v, lane);
  } else {
    return wave_sum<T, OFF>(v[0]);
  }
}
template <class T, int NV> __device__ __forceinline__ T wave_reduce(T (&v)[NV], int lane) {
  static_assert(NV >= 1 && NV <= kWave && (NV & (NV - 1)) == 0, "a power of two");
  return wave_reduce_from<T, NV / 2, kWave / 2>(v, lane);
}

// Deterministic sum of one double per thread of a workgroup, in a fixed tree:
// x[t] + x[t + 128], then + 64, 32, ... 1.  The first two levels are read
// from LDS by one wave, the others are lane exchanges (a barrier per level
// took about three times as long): block_tree is the wave's part, over the
// 256 values at sh; every lane of the wave returns the sum.
__device__ __forceinline__ double block_tree(const double *sh) {
  const int lane = threadIdx.x & (kWave - 1);
  static_assert(kBlock == 4 * kWave, "two LDS levels");
  return wave_sum((sh[lane] + sh[lane + 2 * kWave]) + (sh[lane + kWave] + sh[lane + 3 * kWave]));
}
__device__ __forceinline__ double block_sum(double v, double *sh) {
  const int tid = threadIdx.x;
  sh[tid] = v;
  __syncthreads();
  if (tid < kWave) {
    const double r = block_tree(sh);
    if (tid == 0) sh[0] = r;
  }
  __syncthreads();
  const double r = sh[0];
  __syncthreads();
  return r;
}

// ---------------------------------------------------------------------
// Shared epilogue of every RHS evaluation.
// ---------------------------------------------------------------------
template <class R> struct Vecs {
  const R *cs_in;  // cos at [0, ldv), sin at [ldv, 2 ldv)
  R *cs_out;
  long ldv;        // padded vector length
  long N;
  const R *omega;
  R *y;
  R *k[7];
  R *ynew;         // 5th-order solution of the current attempt
  R *f_out;        // KIND_RHS output
  R *cs_pairs;     // interleaved (C_i, S_i), or nullptr
  R c1;
  State<R> *st;
  double *err_part;  // one per workgroup (stage 7)
  int check_state;   // stage kernels: skip unless an attempt is live
};

constexpr int KIND_RHS = 0;       // f = RHS(theta), optional couplings
constexpr int KIND_COUPLING = 1;  // couplings only
// KIND 2..7 = DP45 stage s

// kuramoto.cu:45: f = w + c1 (sin th C - cos th S), contracted as
// fma(c1, fma(sin, C, -(cos S)), w).
template <class R> __device__ __forceinline__ R rhs_value(R om, R c1, R cs, R sn, R C, R S) {
  return rfma<R>(c1, rfma<R>(sn, C, -(cs * S)), om);
}

// What the row epilogue of oscillator i reads besides C and S.  Loaded on
// its own so that kernels can have these loads in flight while they reduce
// the coupling sums (a dependent load costs 1-2 us between short kernels).
template <class R, int KIND> struct RowOps {
  static constexpr int NK = KIND >= 2 ? KIND - 1 : 0;  // k_1 .. k_{s-1}
  R cs, sn, om, y, yn, h, atl, rtl;
  R k[NK > 0 ? NK : 1];
};
template <class R, int KIND> __device__ __forceinline__ RowOps<R, KIND> row_load(const Vecs<R> &a, long i) {
  RowOps<R, KIND> o;
  o.cs = a.cs_in[i];
  o.sn = a.cs_in[a.ldv + i];
  o.om = a.omega[i];
  if constexpr (KIND >= 2) {
#pragma unroll
    for (int j = 0; j < KIND - 1; ++j) o.k[j] = a.k[j][i];
    o.y = a.y[i];
    o.h = a.st->h;
  }
  if constexpr (KIND == 7) {
    o.yn = a.ynew[i];
    o.rtl = a.st->rtl;
    o.atl = a.st->atl;
  }
  return o;
}

// Row epilogue for oscillator i.  Returns the squared scaled error of
// stage 7 (0 otherwise).  Stage combinations follow dp45.cu:34-69 with the
// contraction acc = k1*a0; acc = fma(k_j, a_j, acc); y + h*acc -> fma(acc, h, y).
// Stages 2..6 also hand back the (cos, sin) they write.
template <class R, int KIND>
__device__ __forceinline__ double row_finish(const Vecs<R> &a, long i, const RowOps<R, KIND> &o, R C, R S,
                                             R *c_out = nullptr, R *s_out = nullptr) {
  const R f = rhs_value<R>(o.om, a.c1, o.cs, o.sn, C, S);
  if constexpr (KIND == KIND_RHS) {
    a.f_out[i] = f;
    if (a.cs_pairs) { a.cs_pairs[2 * i] = C; a.cs_pairs[2 * i + 1] = S; }
    return 0.0;
  } else if constexpr (KIND == KIND_COUPLING) {
    a.cs_pairs[2 * i] = C;
    a.cs_pairs[2 * i + 1] = S;
    return 0.0;
  } else {
    constexpr int s = KIND;  // stage 2..7, k_s = f
    a.k[s - 1][i] = f;
    if constexpr (s < 7) {
      // coefficients of stage s+1 over k_1..k_s
      R acc = o.k[0] * (R)tab::A[s - 1][0];
#pragma unroll
      for (int j = 1; j < s; ++j) acc = rfma<R>(j == s - 1 ? f : o.k[j < s - 1 ? j : 0], (R)tab::A[s - 1][j], acc);
      const R yt = rfma<R>(acc, o.h, o.y);
      if constexpr (s + 1 == 7) a.ynew[i] = yt;
      R c, sn1;
      rsincos<R>(yt, c, sn1);
      a.cs_out[i] = c;
      a.cs_out[a.ldv + i] = sn1;
      if (c_out) { *c_out = c; *s_out = sn1; }
      return 0.0;
    } else {
      // embedded error, dp45.cu:79-84
      R acc = o.k[0] * (R)tab::E[0];
#pragma unroll
      for (int j = 1; j < 7; ++j) acc = rfma<R>(j == 6 ? f : o.k[j < 6 ? j : 0], (R)tab::E[j], acc);
      const R num = o.h * acc;
      const R den = rfma<R>(o.rtl, rmax<R>(rabs<R>(o.y), rabs<R>(o.yn)), o.atl);
      const R e = num / den;
      return (double)e * (double)e;
    }
  }
}
template <class R, int KIND>
__device__ __forceinline__ double row_epilogue(const Vecs<R> &a, long i, R C, R S) {
  return row_finish<R, KIND>(a, i, row_load<R, KIND>(a, i), C, S);
}

// ---------------------------------------------------------------------
// Fused gemv-pair stage kernel (dense adjacency).
// Each workgroup owns ROWS consecutive rows; all 256 threads sweep the
// columns with 16-byte loads (two chunks in flight per row), reuse each
// (cos, sin) chunk for all ROWS rows from registers, then reduce across
// the workgroup (wave shuffles + LDS) in a fixed order.
// ---------------------------------------------------------------------
template <class R, class S> struct DenseArgs {
  const S *A;
  long lda;     // row stride (elements), multiple of 64
  R mscale;     // M = mscale * stored
  Vecs<R> v;
};

// Row sums of one group of ROWS rows [row0, row_end): the wave sums
// (wave_reduce), then the 4 wave sums in wave order (fixed tree), scale, row
// epilogue, its operands loaded before the reduction.  Returns (in thread 0)
// the group's sum of squared scaled errors for stage 7.
template <class R, class Acc, int ROWS, int KIND>
__device__ __forceinline__ double finish_group(Acc (&accC)[ROWS], Acc (&accS)[ROWS], long row0, long row_end,
                                               R mscale, const Vecs<R> &v) {
  __shared__ Acc red[kBlock / kWave][2 * ROWS];
  __shared__ double errsq[ROWS];
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1), wave = tid / kWave;
  const long i = row0 + tid;
  // every lane loads (a row it shares with others): no branch around loads
  const long il = row0 + tid % ROWS;
  const RowOps<R, KIND> ops = row_load<R, KIND>(v, il < row_end ? il : row_end - 1);
  Acc val[2 * ROWS];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) { val[r] = accC[r]; val[ROWS + r] = accS[r]; }
  const Acc tot = wave_reduce<Acc, 2 * ROWS>(val, lane);
  red[wave][wave_slot<2 * ROWS>(lane)] = tot;  // the lanes of a slot hold the same sum
  __syncthreads();
  if (tid < ROWS) {
    double sq = 0.0;
    if (i < row_end) {
      Acc C = red[0][tid], Sv = red[0][ROWS + tid];
#pragma unroll
      for (int w = 1; w < kBlock / kWave; ++w) { C += red[w][tid]; Sv += red[w][ROWS + tid]; }
      sq = row_finish<R, KIND>(v, i, ops, (R)C * mscale, (R)Sv * mscale);
    }
    if constexpr (KIND == 7) errsq[tid] = sq;
  }
  double s = 0.0;
  if constexpr (KIND == 7) {
    __syncthreads();
    if (tid == 0) {
#pragma unroll
      for (int r = 0; r < ROWS; ++r) s += errsq[r];
    }
  }
  return s;
}

// One group per workgroup: rows [row0, min(row0 + ROWS, N)); stage 7 writes
// one error partial per workgroup.
template <class R, class Acc, int ROWS, int KIND>
__device__ __forceinline__ void finish_rows(Acc (&accC)[ROWS], Acc (&accS)[ROWS], long row0, R mscale,
                                            const Vecs<R> &v) {
  const double s = finish_group<R, Acc, ROWS, KIND>(accC, accS, row0, v.N, mscale, v);
  if constexpr (KIND == 7) {
    if (threadIdx.x == 0) v.err_part[blockIdx.x] = s;
  }
}

// BAL = false: workgroup b owns rows [b ROWS, b ROWS + ROWS).
// BAL = true ("balanced"): the grid is one round of resident workgroups and
// workgroup b owns the contiguous rows [b N / G, (b + 1) N / G), walked in
// groups of ROWS, so every workgroup streams the same number of rows (±1)
// and the launch has no tail round.  Rows past the end of a short group
// re-read the group's last row (cache hits) and are discarded.  Every row is
// summed in the same order in every variant.
template <class R, class S, int ROWS, int KIND, bool NT, bool BAL>
__global__ __launch_bounds__(kBlock) void stage_kernel(const DenseArgs<R, S> a) {
  if constexpr (KIND >= 2) {
    if (a.v.check_state && (!a.v.st->active || a.v.st->commit_pending)) return;
  }
  using Acc = typename Store<S>::Acc;
  using Val = typename Store<S>::Val;
  constexpr int VEC = Store<S>::VEC;
  constexpr long STRIDE = (long)kBlock * VEC;
  const int tid = threadIdx.x;
  const long N = a.v.N;
  long rb, re;
  if constexpr (BAL) {
    rb = (long)blockIdx.x * N / gridDim.x;
    re = (long)(blockIdx.x + 1) * N / gridDim.x;
  } else {
    rb = (long)blockIdx.x * ROWS;
    re = rb + ROWS < N ? rb + ROWS : N;
  }
  const R *cosv = a.v.cs_in;
  const R *sinv = a.v.cs_in + a.v.ldv;
  auto load_row = [&](const S *p) -> u32x4 {
    if constexpr (NT) return __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(p));
    else return *reinterpret_cast<const u32x4 *>(p);
  };
  double esum = 0.0;
  for (long row0 = rb; row0 < re; row0 += ROWS) {
    const long nr = re - row0 < ROWS ? re - row0 : ROWS;
    // rows past N of the last group (non-balanced grid) are zero padding rows
    // of the allocation; the balanced grid re-reads the group's last row
    const S *rowp[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) rowp[r] = a.A + (row0 + (BAL ? (r < nr ? r : nr - 1) : r)) * a.lda;

    Acc accC[ROWS], accS[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) { accC[r] = 0; accS[r] = 0; }

    long c = (long)tid * VEC;
    for (; c + STRIDE < a.lda; c += 2 * STRIDE) {
      R cv0[VEC], sv0[VEC], cv1[VEC], sv1[VEC];
      u32x4 raw0[ROWS], raw1[ROWS];
      // issue order: the (cos, sin) chunks (L2 hits, needed by every row)
      // first, then all 2 ROWS adjacency loads, then the first use.  The
      // loads complete in issue order, so row r of the first chunk waits
      // only for its own load.  Without the scheduling barriers the
      // scheduler sinks the second chunk's loads next to their uses (one
      // load in flight per wave) to save registers.
      load_reals<R, VEC>(cosv + c, cv0);
      load_reals<R, VEC>(sinv + c, sv0);
      load_reals<R, VEC>(cosv + c + STRIDE, cv1);
      load_reals<R, VEC>(sinv + c + STRIDE, sv1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = 0; r < ROWS; ++r) raw0[r] = load_row(rowp[r] + c);
#pragma unroll
      for (int r = 0; r < ROWS; ++r) raw1[r] = load_row(rowp[r] + c + STRIDE);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        Val m[VEC];
        unpack<S>(raw0[r], m);
#pragma unroll
        for (int q = 0; q < VEC; ++q) {
          accC[r] = rfma<Acc>((Acc)m[q], (Acc)cv0[q], accC[r]);
          accS[r] = rfma<Acc>((Acc)m[q], (Acc)sv0[q], accS[r]);
        }
        unpack<S>(raw1[r], m);
#pragma unroll
        for (int q = 0; q < VEC; ++q) {
          accC[r] = rfma<Acc>((Acc)m[q], (Acc)cv1[q], accC[r]);
          accS[r] = rfma<Acc>((Acc)m[q], (Acc)sv1[q], accS[r]);
        }
      }
    }
    if (c < a.lda) {
      R cv0[VEC], sv0[VEC];
      u32x4 raw0[ROWS];
#pragma unroll
      for (int r = 0; r < ROWS; ++r) raw0[r] = load_row(rowp[r] + c);
      load_reals<R, VEC>(cosv + c, cv0);
      load_reals<R, VEC>(sinv + c, sv0);
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        Val m[VEC];
        unpack<S>(raw0[r], m);
#pragma unroll
        for (int q = 0; q < VEC; ++q) {
          accC[r] = rfma<Acc>((Acc)m[q], (Acc)cv0[q], accC[r]);
          accS[r] = rfma<Acc>((Acc)m[q], (Acc)sv0[q], accS[r]);
        }
      }
    }
    esum += finish_group<R, Acc, ROWS, KIND>(accC, accS, row0, row0 + nr, a.mscale, a.v);
    if constexpr (BAL) __syncthreads();  // the next group reuses the reduction buffers
  }
  if constexpr (KIND == 7) {
    if (tid == 0) a.v.err_part[blockIdx.x] = esum;
  }
}

// The same group pass with the adjacency streamed through a ring of two
// chunk buffers: chunk k + 1 of every row loads while chunk k is reduced,
// so each wave always has one to two chunks of loads in flight (the loop
// above issues a pair of chunks and then waits for all of it) with the
// same two register sets.  Rows and vectors are buffer resources of lda
// elements: the lanes of the last, partial chunk read zeros (no memory
// access) instead of branching, every load in the loop is unconditional,
// and each chunk's loads are issued before the previous chunk's products.
// Every row is summed in the same order as stage_kernel: chunk by chunk, VEC
// values each; a zero chunk adds +0 to sums that are never -0, so the
// results are the same bits.  One group per workgroup.
template <class R, class S, int ROWS, int KIND, bool NT>
__global__ __launch_bounds__(kBlock) void stage_ring_kernel(const DenseArgs<R, S> a) {
  if constexpr (KIND >= 2) {
    if (a.v.check_state && (!a.v.st->active || a.v.st->commit_pending)) return;
  }
  using Acc = typename Store<S>::Acc;
  using Val = typename Store<S>::Val;
  constexpr int VEC = Store<S>::VEC;
  constexpr long STRIDE = (long)kBlock * VEC;
  constexpr int WV = (int)(VEC * sizeof(R) / 16);  // 16-byte loads per vector chunk
  const int tid = threadIdx.x;
  const long row0 = (long)blockIdx.x * ROWS;
  const long nch = (a.lda + STRIDE - 1) / STRIDE;
  __amdgpu_buffer_rsrc_t rrow[ROWS];
#pragma unroll
  for (int r = 0; r < ROWS; ++r)
    rrow[r] = __builtin_amdgcn_make_buffer_rsrc(const_cast<S *>(a.A + (row0 + r) * a.lda), (short)0,
                                                (int)(a.lda * (long)sizeof(S)), 0x00020000);
  const __amdgpu_buffer_rsrc_t rcos = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<R *>(a.v.cs_in), (short)0, (int)(a.lda * (long)sizeof(R)), 0x00020000);
  const __amdgpu_buffer_rsrc_t rsin = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<R *>(a.v.cs_in + a.v.ldv), (short)0, (int)(a.lda * (long)sizeof(R)), 0x00020000);
  constexpr int AUX = NT ? 2 : 0;
  struct Chunk {
    u32x4 raw[ROWS];
    u32x4 cv[WV], sv[WV];
  };
  auto load = [&](long k, Chunk &ch) {
    const long c = k * STRIDE + (long)tid * VEC;
    const int vo = (int)(c * (long)sizeof(R));
#pragma unroll
    for (int w = 0; w < WV; ++w) {
      ch.cv[w] = __builtin_amdgcn_raw_buffer_load_b128(rcos, vo + 16 * w, 0, 0);
      ch.sv[w] = __builtin_amdgcn_raw_buffer_load_b128(rsin, vo + 16 * w, 0, 0);
    }
    const int mo = (int)(c * (long)sizeof(S));
#pragma unroll
    for (int r = 0; r < ROWS; ++r) ch.raw[r] = __builtin_amdgcn_raw_buffer_load_b128(rrow[r], mo, 0, AUX);
  };
  Acc accC[ROWS], accS[ROWS];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) { accC[r] = 0; accS[r] = 0; }
  auto reduce = [&](const Chunk &ch) {
    R cv[VEC], sv[VEC];
#pragma unroll
    for (int w = 0; w < WV; ++w) {
      unpack<R>(ch.cv[w], cv + (16 / sizeof(R)) * w);
      unpack<R>(ch.sv[w], sv + (16 / sizeof(R)) * w);
    }
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      Val m[VEC];
      unpack<S>(ch.raw[r], m);
#pragma unroll
      for (int q = 0; q < VEC; ++q) {
        accC[r] = rfma<Acc>((Acc)m[q], (Acc)cv[q], accC[r]);
        accS[r] = rfma<Acc>((Acc)m[q], (Acc)sv[q], accS[r]);
      }
    }
  };
  Chunk c0, c1;
  load(0, c0);
  // chunk pairs; the loads past the last chunk return zeros without memory
  // traffic, so the loop needs no condition around them
  long k = 0;
#pragma unroll 1
  for (; k + 1 < nch; k += 2) {
    __builtin_amdgcn_sched_barrier(0);
    load(k + 1, c1);
    __builtin_amdgcn_sched_barrier(0);
    reduce(c0);
    __builtin_amdgcn_sched_barrier(0);
    load(k + 2, c0);
    __builtin_amdgcn_sched_barrier(0);
    reduce(c1);
  }
  reduce(c0);  // chunk nch - 1 for an odd count, zeros otherwise
  finish_rows<R, Acc, ROWS, KIND>(accC, accS, row0, a.mscale, a.v);
}

// ---------------------------------------------------------------------
// -A with register-rebuilt adjacency tiles: M_ij = sum_m w_m (X_im X_jm)
// is formed in registers for every (row, column) pair of a stage from the
// transposed factor XT (K x ldv, zero columns past N) — no N x N matrix in
// HBM, (2K + 2) N^2 VALU operations per RHS (K products and K fmas per
// entry, two fmas into the double sums; FP32 adds the entry's conversion to
// double: 2K + 3).  Each entry uses the dense
// generator's formula and the columns are visited in the dense stage
// kernel's order (VEC per 16-byte chunk, chunks strided by kBlock VEC), so
// the result equals the dense FP32/FP64 path on the generated matrix bit
// for bit.
// ---------------------------------------------------------------------
template <class R> struct RebuildArgs {
  const R *XT;  // [K][ldv]
  const R *w;   // [K]
  int K;
  Vecs<R> v;
};

// KT: rank bound of the register arrays; EXACT: K == KT (no per-term
// guards in the unrolled inner loop).
template <class R, int ROWS, int KIND, int KT, bool EXACT>
__global__ __launch_bounds__(kBlock) void rebuild_stage_kernel(const RebuildArgs<R> a) {
  if constexpr (KIND >= 2) {
    if (a.v.check_state && (!a.v.st->active || a.v.st->commit_pending)) return;
  }
  constexpr int VEC = 16 / sizeof(R);
  constexpr long STRIDE = (long)kBlock * VEC;
  const long ldv = a.v.ldv;
  const long row0 = (long)blockIdx.x * ROWS;
  const int K = EXACT ? KT : a.K;
  // The row factors are the same in every lane; a lane shuffle gives them a
  // per-lane register copy (otherwise they sit in scalar registers that
  // spill, and every use in the inner loop reloads them).
  const int lane = threadIdx.x & (kWave - 1);
  R xi[ROWS][KT], wm[KT];
#pragma unroll
  for (int m = 0; m < KT; ++m) {
    wm[m] = __shfl(m < K ? a.w[m] : (R)0, lane, kWave);
#pragma unroll
    for (int r = 0; r < ROWS; ++r) xi[r][m] = __shfl(m < K ? a.XT[m * ldv + row0 + r] : (R)0, lane, kWave);
  }
  const R *cosv = a.v.cs_in;
  const R *sinv = a.v.cs_in + ldv;
  using Acc = typename Store<R>::Acc;  // the dense path's accumulation
  Acc accC[ROWS], accS[ROWS];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) { accC[r] = 0; accS[r] = 0; }
  struct Chunk {
    R cv[VEC], sv[VEC], xj[KT][VEC];
  };
  auto load = [&](long c, Chunk &ch) __attribute__((always_inline)) {
    load_reals<R, VEC>(cosv + c, ch.cv);
    load_reals<R, VEC>(sinv + c, ch.sv);
#pragma unroll
    for (int m = 0; m < KT; ++m)
      if (m < K) load_reals<R, VEC>(a.XT + m * ldv + c, ch.xj[m]);
  };
  // The next chunk's loads ahead of this one's products in the FP32 K = 5 form
  // (222 registers, 2 waves per SIMD either way): N = 200000 11.52 -> 10.88 ms,
  // N = 20000 151 -> 134 us, N = 60000 1049 -> 1006.  The others lose a wave or
  // spill into AGPRs for it: FP64 K = 5, N = 60000 1742 -> 1809 us; FP32 K = 8,
  // N = 20000 266 -> 282; FP64 K = 8 541 -> 628.
  constexpr bool AHEAD = EXACT && sizeof(R) == 4;
  long c = (long)threadIdx.x * VEC;
  Chunk cur, nxt;
  if (AHEAD && c < ldv) load(c, cur);
  for (; c < ldv; c += STRIDE) {
    if constexpr (AHEAD) {
      load(c + STRIDE < ldv ? c + STRIDE : c, nxt);
      __builtin_amdgcn_sched_barrier(0);
    } else {
      load(c, cur);
    }
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
      for (int q = 0; q < VEC; ++q) {
        R mij = 0;
#pragma unroll
        for (int m = 0; m < KT; ++m)
          if (m < K) mij = rfma<R>(wm[m], xi[r][m] * cur.xj[m][q], mij);
        accC[r] = rfma<Acc>((Acc)mij, (Acc)cur.cv[q], accC[r]);
        accS[r] = rfma<Acc>((Acc)mij, (Acc)cur.sv[q], accS[r]);
      }
    if constexpr (AHEAD) cur = nxt;
  }
  finish_rows<R, Acc, ROWS, KIND>(accC, accS, row0, (R)1, a.v);
}

// ---------------------------------------------------------------------
// Factored (-A) coupling: M = X diag(w) X^T (makecoupling's m1/m2 branch,
// kuramoto.cu:62-108).  G_m = w_m sum_n X_nm (cos_n, sin_n); C_n =
// sum_m X_nm G_m.  Three small launches per RHS; all sums in double.
// ---------------------------------------------------------------------
constexpr int kRankTile = 8;

template <class R>
__global__ __launch_bounds__(kBlock) void lowrank_partial_kernel(const R *X, int K, long N, const R *cs, long ldv,
                                                                 double *part, const State<R> *st, int check_state) {
  if (check_state && (!st->active || st->commit_pending)) return;
  __shared__ double sh[kBlock];
  const int m0 = blockIdx.y * kRankTile;
  double ac[kRankTile], as[kRankTile];
#pragma unroll
  for (int q = 0; q < kRankTile; ++q) { ac[q] = 0; as[q] = 0; }
  for (long n = (long)blockIdx.x * kBlock + threadIdx.x; n < N; n += (long)gridDim.x * kBlock) {
    const double cv = cs[n], sv = cs[ldv + n];
#pragma unroll
    for (int q = 0; q < kRankTile; ++q) {
      if (m0 + q < K) {
        const double x = X[n * K + m0 + q];
        ac[q] = __builtin_fma(x, cv, ac[q]);
        as[q] = __builtin_fma(x, sv, as[q]);
      }
    }
  }
#pragma unroll
  for (int q = 0; q < kRankTile; ++q) {
    const double tc = block_sum(ac[q], sh);
    const double ts = block_sum(as[q], sh);
    if (threadIdx.x == 0 && m0 + q < K) {
      part[((size_t)blockIdx.x * K + m0 + q) * 2] = tc;
      part[((size_t)blockIdx.x * K + m0 + q) * 2 + 1] = ts;
    }
  }
}

template <class R>
__global__ __launch_bounds__(kBlock) void lowrank_reduce_kernel(const double *part, int nblk, int K, const R *w,
                                                                double *G, const State<R> *st, int check_state) {
  if (check_state && (!st->active || st->commit_pending)) return;
  __shared__ double sh[kBlock];
  for (int v = 0; v < 2 * K; ++v) {
    double s = 0;
    for (int b = threadIdx.x; b < nblk; b += kBlock) s += part[(size_t)b * 2 * K + v];
    const double tot = block_sum(s, sh);
    if (threadIdx.x == 0) G[v] = (double)w[v / 2] * tot;
  }
}

template <class R, int KIND>
__global__ __launch_bounds__(kBlock) void lowrank_expand_kernel(const R *X, int K, const double *G, Vecs<R> v) {
  if constexpr (KIND >= 2) {
    if (v.check_state && (!v.st->active || v.st->commit_pending)) return;
  }
  __shared__ double errsq[kBlock];
  const long i = (long)blockIdx.x * kBlock + threadIdx.x;
  double sq = 0.0;
  if (i < v.N) {
    double C = 0, S = 0;
    for (int m = 0; m < K; ++m) {
      const double x = X[i * K + m];
      C = __builtin_fma(x, G[2 * m], C);
      S = __builtin_fma(x, G[2 * m + 1], S);
    }
    sq = row_epilogue<R, KIND>(v, i, (R)C, (R)S);
  }
  if constexpr (KIND == 7) {
    const double tot = block_sum(sq, errsq);
    if (threadIdx.x == 0) v.err_part[blockIdx.x] = tot;
  }
}

// ---------------------------------------------------------------------
// Low-rank coupling, one launch per RHS (K <= kLrMaxRank).
//   G = w .* X^T (cos, sin) is formed in two halves: the launch that writes
//   a stage vector also writes partial sums of X^T (cos, sin); the next
//   launch starts with every workgroup adding those partials (the same order
//   in each, so all of them hold the same G), then computes C_i = sum_m X_im
//   G_c[m], S_i likewise and the row epilogue of its stage.  The stage-2
//   vector's partials come from lowrank_emit_kernel; lowrank_gram_kernel
//   writes those of a given vector (a stand-alone RHS).  No cross-workgroup
//   synchronisation inside a launch; partial buffers alternate between
//   consecutive launches.
// Every sum has an order that follows from N alone (the error norm feeds the
// step size, which feeds the phases: with fast oscillators the last bit of
// one sum is another sequence of steps a few attempts later, so neither the
// card's CU count nor the launch's shape may enter).  The rows are split into
// `blocks` of kBlock lanes, at most kLrMaxBlocks, lane t of block b taking
// rows kBlock b + t, + kBlock blocks, ...: one partial per block (its four
// waves' sums in wave order), one error partial per block and one order
// partial per kBlock consecutive rows (block_tree both).
// The few MB it moves stay in the caches, so a launch is bound by latency:
// one dependent round trip after another.  A workgroup holds one block, or
// two (LrPlace) once there are more blocks than a card has CUs, so that the
// partials are read once for both and each half sums half of the values; the
// row's X (from the transposed factor: coalesced), its epilogue operands and
// the partials are all loaded before the first of them is needed; the rank is
// a template argument up to 8 (no guards).  One attempt, FP32, K = 5, against
// workgroups of one block with guarded ranks and row-major X: N = 9000 66 ->
// 27 us, N = 100000 82 -> 35, N = 200000 109 -> 41, N = 10^6 225 -> 96; K = 16,
// N = 200000 357 -> 74; FP64, K = 5, N = 200000 121 -> 51.
// ---------------------------------------------------------------------
constexpr int kLrMaxRank = 16;
constexpr int kLrMaxBlocks = 512;
constexpr int kLrPairedBlocks = 256;       // more blocks than this: two per workgroup
constexpr int kLrThreads = 2 * kBlock;     // at most
constexpr int kLrBlockWaves = kBlock / kWave;
constexpr int lr_pow2(int n) { return n <= 1 ? 1 : 2 * lr_pow2((n + 1) / 2); }
static_assert(kLrMaxBlocks <= 2 * kBlock, "a lane adds at most two partials of a value");

template <class R> struct LrArgs {
  const R *XT;  // [K][ldv], zero past N
  const R *w;   // [K]
  int K;
  int blocks;
  const double *part_in;  // [2K][blocks]
  double *part_out;       // [2K][blocks]
};

// The block of this thread's half of the workgroup: b, and with two halves
// the other end's blocks - 1 - b (with more than one row per lane the first
// blocks hold one row more than the last ones).
struct LrPlace {
  int half, tid, wave;  // thread and wave within the block
  int blk;
  bool live;            // an odd count leaves the last workgroup's second half empty
  __device__ __forceinline__ LrPlace(int blocks)
      : half((int)threadIdx.x / kBlock), tid((int)threadIdx.x % kBlock), wave(tid / kWave),
        blk(half ? blocks - 1 - (int)blockIdx.x : (int)blockIdx.x), live(!half || blk > (int)blockIdx.x) {}
  __device__ __forceinline__ long first(long N) const { return live ? (long)blk * kBlock + tid : N; }
};

// A block's sums of acc (2K values, interleaved c / s) -> part[q][block]
template <int KT>
__device__ __forceinline__ void lr_write_partials(const LrPlace &pl, const double (&acc)[2 * KT], int K, int blocks,
                                                  double *part) {
  constexpr int NV = lr_pow2(2 * KT);
  __shared__ double red[kLrThreads / kWave][NV];
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  double v[NV];
#pragma unroll
  for (int q = 0; q < NV; ++q) v[q] = q < 2 * KT ? acc[q < 2 * KT ? q : 0] : 0.0;
  const double t = wave_reduce<double, NV>(v, lane);
  red[wave][wave_slot<NV>(lane)] = t;
  __syncthreads();
  if (pl.tid < 2 * K && pl.live) {
    const int w0 = wave - pl.wave;
    double s = red[w0][pl.tid];
#pragma unroll
    for (int q = 1; q < kLrBlockWaves; ++q) s += red[w0 + q][pl.tid];
    part[(size_t)pl.tid * blocks + pl.blk] = s;
  }
}

// G (2K values, interleaved c / s) from the blocks' partials, into g (LDS):
// lane t < kBlock adds partials t and t + kBlock of a value, then the waves'
// sums in wave order.  With two blocks per workgroup the second half's lanes
// take values K .. 2K - 1.  lr_fetch issues the loads (before the launch's
// state check; every buffer is readable then).
template <class R, int KT> struct LrFetched {
  double p[2 * KT];
  R w;
};
template <class R, int KT>
__device__ __forceinline__ LrFetched<R, KT> lr_fetch(const LrArgs<R> &l, const LrPlace &pl, int K) {
  LrFetched<R, KT> f;
  const bool two = blockDim.x > kBlock;
#pragma unroll
  for (int j = 0; j < 2 * KT; ++j) {
    const int jj = j < KT ? j : j - KT;  // two: value jj of the half, partials t (j < KT) and t + kBlock
    const int q = two ? pl.half * K + jj : j, b = pl.tid + (two && j >= KT ? kBlock : 0);
    f.p[j] = (two ? jj < K : j < 2 * K) && b < l.blocks ? l.part_in[(size_t)q * l.blocks + b] : 0.0;
  }
  f.w = l.w[(int)threadIdx.x < 2 * K ? threadIdx.x >> 1 : 0];
  return f;
}
template <class R, int KT>
__device__ __forceinline__ void lr_reduce(const LrFetched<R, KT> &f, const LrPlace &pl, int K, double *g) {
  constexpr int NV = lr_pow2(2 * KT), NH = lr_pow2(KT);
  __shared__ double red[kLrBlockWaves][NV + NH];
  const int lane = threadIdx.x % kWave;
  if (blockDim.x > kBlock) {
    double v[NH];
#pragma unroll
    for (int j = 0; j < NH; ++j) v[j] = j < KT ? f.p[j < KT ? j : 0] + f.p[j < KT ? KT + j : 0] : 0.0;
    const double t = wave_reduce<double, NH>(v, lane);
    const int slot = wave_slot<NH>(lane);
    if (slot < K) red[pl.wave][pl.half * K + slot] = t;
  } else {
    double v[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) v[j] = j < 2 * KT ? f.p[j < 2 * KT ? j : 0] + 0.0 : 0.0;
    const double t = wave_reduce<double, NV>(v, lane);
    red[pl.wave][wave_slot<NV>(lane)] = t;
  }
  __syncthreads();
  if ((int)threadIdx.x < 2 * K) {
    double t = red[0][threadIdx.x];
#pragma unroll
    for (int q = 1; q < kLrBlockWaves; ++q) t += red[q][threadIdx.x];
    g[threadIdx.x] = t * (double)f.w;
  }
  __syncthreads();
}

template <class R, int KT, bool EXACT>
__device__ __forceinline__ void lr_load_row(const LrArgs<R> &l, int K, long ldv, long i, R (&x)[KT]) {
#pragma unroll
  for (int m = 0; m < KT; ++m) x[m] = EXACT || m < K ? l.XT[m * ldv + i] : (R)0;
}
// acc += x (c, s) of one row; with a rank below KT the rows past it stay zero
template <class R, int KT, bool EXACT>
__device__ __forceinline__ void lr_accumulate(const R (&x)[KT], int K, R c, R s, double (&acc)[2 * KT]) {
#pragma unroll
  for (int m = 0; m < KT; ++m)
    if (EXACT || m < K) {
      acc[2 * m] = __builtin_fma((double)x[m], (double)c, acc[2 * m]);
      acc[2 * m + 1] = __builtin_fma((double)x[m], (double)s, acc[2 * m + 1]);
    }
}

template <class R, int KT, bool EXACT>
__global__ __launch_bounds__(kLrThreads) void lowrank_gram_kernel(const LrArgs<R> l, long N, const R *cs, long ldv) {
  const int K = EXACT ? KT : l.K;
  const LrPlace pl(l.blocks);
  double acc[2 * KT] = {};
  for (long i = pl.first(N); i < N; i += (long)l.blocks * kBlock) {
    R x[KT];
    lr_load_row<R, KT, EXACT>(l, K, ldv, i, x);
    lr_accumulate<R, KT, EXACT>(x, K, cs[i], cs[ldv + i], acc);
  }
  lr_write_partials<KT>(pl, acc, K, l.blocks, l.part_out);
}

template <class R, int KIND, int KT, bool EXACT>
__global__ __launch_bounds__(kLrThreads) void lowrank_stage_kernel(const LrArgs<R> l, const Vecs<R> v) {
  constexpr bool NEXT = KIND >= 2 && KIND < 7;  // also the partials of the vector this stage writes
  __shared__ double gs[2 * KT];
  const int K = EXACT ? KT : l.K;
  const LrPlace pl(l.blocks);
  // everything the first row needs is in flight before the state check and
  // the reduction of G (rows past N re-read row N - 1, never used)
  const long stride = (long)l.blocks * kBlock;
  long i = pl.first(v.N);
  const LrFetched<R, KT> fetched = lr_fetch<R, KT>(l, pl, K);
  R x[KT];
  const long i0 = i < v.N ? i : v.N - 1;
  lr_load_row<R, KT, EXACT>(l, K, v.ldv, i0, x);
  RowOps<R, KIND> ops = row_load<R, KIND>(v, i0);
  asm volatile("" ::: "memory");
  if constexpr (KIND >= 2) {
    if (v.check_state && (!v.st->active || v.st->commit_pending)) return;
  }
  lr_reduce<R, KT>(fetched, pl, K, gs);
  double acc[2 * KT] = {};
  double sq = 0.0;
  while (i < v.N) {
    // the next row's operands are in flight while this row is computed
    R xn[KT];
    RowOps<R, KIND> opsn;
    const bool more = i + stride < v.N;
    if (more) {
      lr_load_row<R, KT, EXACT>(l, K, v.ldv, i + stride, xn);
      opsn = row_load<R, KIND>(v, i + stride);
    }
    asm volatile("" ::: "memory");  // G is re-read from LDS for every row: in registers it would cost 4K of them
    double C = 0, S = 0;
#pragma unroll
    for (int m = 0; m < KT; ++m)
      if (EXACT || m < K) {
        C = __builtin_fma((double)x[m], gs[2 * m], C);
        S = __builtin_fma((double)x[m], gs[2 * m + 1], S);
      }
    R c = 0, s = 0;
    sq += row_finish<R, KIND>(v, i, ops, (R)C, (R)S, &c, &s);
    if constexpr (NEXT) lr_accumulate<R, KT, EXACT>(x, K, c, s, acc);
    i += stride;
    if (more) {
#pragma unroll
      for (int m = 0; m < KT; ++m) x[m] = xn[m];
      ops = opsn;
    }
  }
  if constexpr (KIND == 7) {
    __shared__ double errsq[2][kBlock];
    errsq[pl.half][pl.tid] = sq;
    __syncthreads();
    if (pl.wave == 0) {
      const double tot = block_tree(errsq[pl.half]);
      if (pl.tid == 0 && pl.live) v.err_part[pl.blk] = tot;
    }
  }
  if constexpr (NEXT) lr_write_partials<KT>(pl, acc, K, l.blocks, l.part_out);
}

// r = sqrt((X/N)^2 + (Y/N)^2) in the working precision (kuramoto.cu:220:
// pow((X/N*X/N + Y/N*Y/N), 0.5) with X, Y the sums of cos and sin).
template <class R> __device__ __forceinline__ R order_value(double X, double Y, long N) {
  const R XR = (R)X, YR = (R)Y, NR = (R)N;
  return (R)pow((double)(XR / NR * XR / NR + YR / NR * YR / NR), 0.5);
}

// Order parameters of n emitted rows from their workgroups' partial sums
// (nblk pairs a row), one wave per row: the sum over partials b, b + 256, ...
// of each b < 256, then block_tree's order.
template <class R>
__device__ __forceinline__ void order_rows(int n, const double *part, int nblk, long N, R *r) {
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  for (int q = wave; q < n; q += kBlock / kWave) {
    const double2 *p = reinterpret_cast<const double2 *>(part) + (size_t)q * nblk;
    double x[4] = {0, 0, 0, 0}, y[4] = {0, 0, 0, 0};
#pragma unroll
    for (int v = 0; v < 4; ++v)
      for (int b = lane + v * kWave; b < nblk; b += kBlock) {
        const double2 e = p[b];
        x[v] += e.x;
        y[v] += e.y;
      }
    const double X = wave_sum((x[0] + x[2]) + (x[1] + x[3]));
    const double Y = wave_sum((y[0] + y[2]) + (y[1] + y[3]));
    if (lane == 0) r[q] = order_value<R>(X, Y, N);
  }
}

// ---------------------------------------------------------------------
// Controller (dp45.cu:117-138), in registers: every lane of one wave holds
// the state S and updates it the same way.  err: sum of the squared scaled
// errors (unused with a fixed step); te: output time e0 + lane, with e0 =
// first pending or next output (NaN past the grid: never reached).  Lane 0
// appends to the accepted-step log.
// ---------------------------------------------------------------------
template <class R> __device__ __forceinline__ int control_first_output(const State<R> &S) {
  return S.commit_pending ? S.pend_lo : S.eval_i;
}
template <class R>
__device__ __forceinline__ void control_decide(State<R> &S, double err, long N, const R *t_eval, R te, R *times,
                                               int lane) {
  S.job_mode = JOB_NONE;
  S.job_n = S.fin_n = 0;
  if (!S.active) return;
  if (!S.commit_pending) {
    const R h = S.h;
    int accept;
    R hnext = h;
    S.attempts += 1;
    S.rhs_evals += 6;
    if (S.fixed) {
      accept = 1;
    } else {
      const R nrm = (R)sqrt(err);                                // {S,D}nrm2
      const R norm = (R)((double)nrm / sqrt((double)N));        // dp45.cu:119
      R factor = (R)(0.9 * pow((double)norm, -0.2));            // dp45.cu:120
      S.norm = (double)norm;
      if (norm < (R)1) {
        accept = 1;
        if (factor > (R)10) factor = (R)10;
        hnext = h * factor;
      } else {
        accept = 0;
        if (factor < (R)1) {
          if ((double)factor < 0.2) factor = (R)0.2;
          hnext = h * factor;
        }
        if (isnan((double)norm)) {  // the reference would loop forever here
          S.error = 1;
          S.active = 0;
        }
      }
    }
    S.last_accept = accept;
    S.h = hnext;
    if (!accept) {
      S.rejected += 1;
      if (S.active) S.job_mode = JOB_STAGE2;
      return;
    }
    const R tn = S.t + h;
    S.t_last = S.t;
    S.t = tn;
    S.accepted += 1;
    if (S.times_count < S.times_cap) {
      if (lane == 0) {
        times[2 * S.times_count] = tn;
        times[2 * S.times_count + 1] = hnext;
      }
      S.times_count += 1;
    }
    // output times crossed by this step (kuramoto.cu:205-212): up to the
    // first one not reached, 64 at a time
    int hi = S.eval_i;
    for (;;) {
      const unsigned long long miss = ~__ballot(tn >= te);
      hi += miss ? __ffsll((long long)miss) - 1 : kWave;
      if (miss) break;
      te = hi + lane < S.n_eval ? t_eval[hi + lane] : (R)NAN;
    }
    S.pend_lo = S.eval_i;
    S.pend_hi = hi;
    S.commit_pending = 1;
  }
  const int pend = S.pend_hi - S.pend_lo, room = S.ring_cap - S.ring_count;
  S.job_n = S.fin_n = pend < room ? pend : room;
  S.job_lo = S.pend_lo;
  S.job_slot = S.ring_count;
  S.job_mode = JOB_EMIT;
  S.ring_count += S.job_n;
  S.pend_lo += S.job_n;
  if (S.job_n == pend) {
    S.job_mode = JOB_COMMIT;
    S.commit_pending = 0;
    S.eval_i = S.pend_hi;
    if (!(S.t < S.t1)) S.active = 0;
  }
}

// One workgroup, bound by the latency of its chain of loads and of the
// norm's pow: the state is read once at the start, with the error partials
// and then the next 64 output times in flight beside it, and written back
// once.
template <class R>
__global__ __launch_bounds__(kBlock) void control_kernel(State<R> *st, const double *err_part, int nparts, long N,
                                                         const R *t_eval, R *times, const double *ord_part, int nblk,
                                                         R *r_ring) {
  __shared__ double sh[kBlock];
  double s = 0.0;
#pragma unroll 8
  for (int b = threadIdx.x; b < nparts; b += kBlock) s += err_part[b];
  sh[threadIdx.x] = s;
  State<R> S = *st;
  const int lane = threadIdx.x % kWave;
  const int e = control_first_output(S) + lane;
  const R te = e < S.n_eval ? t_eval[e] : (R)NAN;
  if (S.fin_n > 0)  // the previous attempt's rows
    order_rows<R>(S.fin_n, ord_part + (size_t)S.job_slot * nblk * 2, nblk, N, r_ring + S.job_slot);
  __syncthreads();
  if (threadIdx.x >= kWave) return;
  control_decide<R>(S, block_tree(sh), N, t_eval, te, times, lane);
  if (lane == 0) *st = S;
}

// The order parameters control_kernel has not computed yet (after the last
// attempt before the host reads the ring).
template <class R>
__global__ __launch_bounds__(kBlock) void finalize_kernel(State<R> *st, const double *ord_part, int nblk, long N,
                                                          R *r_ring) {
  const int n = st->fin_n, slot = st->job_slot;
  if (n <= 0) return;
  order_rows<R>(n, ord_part + (size_t)slot * nblk * 2, nblk, N, r_ring + slot);
  __syncthreads();
  if (threadIdx.x == 0) st->fin_n = 0;
}

// ---------------------------------------------------------------------
// Dense output + order-parameter partials + commit + next stage-2 vector.
// ---------------------------------------------------------------------
template <class R> struct EmitArgs {
  State<R> *st;
  long N, ldv;
  R *y, *ylast, *ynew;
  R *k[7];
  R *cs_out;          // stage-2 (cos, sin) for the next attempt
  const R *t_eval;
  R *ring;            // ring_cap x ldv rows (or nullptr)
  double *ord_part;   // ring_cap x gridDim.x x 2
};

template <class R> __device__ __forceinline__ void dense_coeffs(const R *kv, R Q[4]) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    R acc = kv[0] * (R)tab::P[0][q];
#pragma unroll
    for (int j = 1; j < 7; ++j) acc = rfma<R>(kv[j], (R)tab::P[j][q], acc);
    Q[q] = acc;
  }
}

// ylast + (hh x) (Q0 + x (Q1 + x (Q2 + x Q3))),  x = (te - t_last) / hh
template <class R> __device__ __forceinline__ R dense_value(const R Q[4], R yl, R hh, R x) {
  R in = rfma<R>(x, Q[3], Q[2]);
  in = rfma<R>(x, in, Q[1]);
  in = rfma<R>(x, in, Q[0]);
  return rfma<R>(hh * x, in, yl);
}

template <class R>
__device__ __forceinline__ void stage2_vector(const EmitArgs<R> &a, long i, R y, R k1, R h, R &c, R &s) {
  const R yt = rfma<R>(k1 * (R)tab::A[0][0], h, y);
  rsincos<R>(yt, c, s);
  a.cs_out[i] = c;
  a.cs_out[a.ldv + i] = s;
}

// n output rows of one dense-output interval, for each kBlock threads of a
// workgroup: te(q) the q-th output time, put(q, value) keeps this thread's
// value, part(q, sums) the row's partial sums of these threads.  Four rows at
// a time: their cos / sin, then one wave sums each row (block_tree), so a
// group of rows costs two barriers and one chain of latencies (one row at a
// time: 12 rows of N = 10^4 took 21 us).
constexpr int kEmitRows = kBlock / kWave;
template <class R, class TE, class PUT, class PART>
__device__ __forceinline__ void emit_rows(int n, bool valid, const R Q[4], R yl, R tl, R hh,
                                          double (&sh)[kEmitRows][2][kBlock], TE te, PUT put, PART part) {
  const int tid = threadIdx.x % kBlock, wave = tid / kWave;
  for (int q0 = 0; q0 < n; q0 += kEmitRows) {
    const int m = n - q0 < kEmitRows ? n - q0 : kEmitRows;
#pragma unroll
    for (int r = 0; r < kEmitRows; ++r) {
      if (r >= m) break;
      R c = 0, s = 0;
      if (valid) {
        const R x = (te(q0 + r) - tl) / hh;
        const R val = dense_value<R>(Q, yl, hh, x);
        put(q0 + r, val);
        rsincos<R>(val, c, s);
      }
      sh[r][0][tid] = (double)c;
      sh[r][1][tid] = (double)s;
    }
    __syncthreads();
    if (wave < m) {
      const double bc = block_tree(sh[wave][0]), bs = block_tree(sh[wave][1]);
      if (tid % kWave == 0) part(q0 + wave, make_double2(bc, bs));
    }
    __syncthreads();
  }
}

// The emit launch for oscillator i; true if the stage-2 vector was written
// (the same for every thread), with this thread's part in c, s.
template <class R> __device__ __forceinline__ bool emit_commit(const EmitArgs<R> &a, long i, R &c, R &s) {
  const State<R> *st = a.st;
  const int mode = st->job_mode;
  if (mode == JOB_NONE) return false;
  __shared__ double sh[kEmitRows][2][kBlock];
  const bool valid = i < a.N;
  const R h = st->h;
  if (mode == JOB_STAGE2) {
    if (valid) stage2_vector<R>(a, i, a.y[i], a.k[0][i], h, c, s);
    return true;
  }
  // every operand of the commit is in flight before the outputs are formed
  R yo = 0, yn = 0, k7 = 0;
  if (valid) yo = a.y[i], yn = a.ynew[i], k7 = a.k[6][i];
  const int n_emit = st->job_n, slot0 = st->job_slot, lo = st->job_lo;
  if (n_emit > 0) {
    const R tl = st->t_last, hh = st->t - tl;
    R Q[4] = {0, 0, 0, 0};
    if (valid) {
      R kv[7];
#pragma unroll
      for (int j = 0; j < 7; ++j) kv[j] = a.k[j][i];
      dense_coeffs<R>(kv, Q);
    }
    emit_rows<R>(
        n_emit, valid, Q, yo, tl, hh, sh, [&](int q) { return a.t_eval[lo + q]; },
        [&](int q, R val) {
          if (a.ring) a.ring[(size_t)(slot0 + q) * a.ldv + i] = val;
        },
        [&](int q, double2 sums) {
          reinterpret_cast<double2 *>(a.ord_part)[(size_t)(slot0 + q) * gridDim.x + blockIdx.x] = sums;
        });
  }
  if (mode == JOB_COMMIT && valid) {
    // commit (dp45.cu:123-125, FSAL copy :160) and the next stage-2 vector
    a.ylast[i] = yo;
    a.y[i] = yn;
    a.k[0][i] = k7;
    stage2_vector<R>(a, i, yn, k7, h, c, s);
  }
  return mode == JOB_COMMIT;
}
template <class R>
__global__ __launch_bounds__(kBlock) void emit_commit_kernel(const EmitArgs<R> a) {
  R c = 0, s = 0;
  (void)emit_commit<R>(a, (long)blockIdx.x * kBlock + threadIdx.x, c, s);
}

// emit_commit_kernel for the low-rank path, on its blocks, with the partials
// of X^T (cos, sin) of the stage-2 vector it writes.  nblk: order partials of
// an output row (one per kBlock rows).
template <class R, int KT, bool EXACT>
__global__ __launch_bounds__(kLrThreads) void lowrank_emit_kernel(const EmitArgs<R> a, const LrArgs<R> l, int nblk) {
  const State<R> *st = a.st;
  const int mode = st->job_mode;
  if (mode == JOB_NONE) return;
  __shared__ double sh[2][kEmitRows][2][kBlock];
  const int K = EXACT ? KT : l.K;
  const LrPlace pl(l.blocks);
  const long stride = (long)l.blocks * kBlock, first = pl.first(a.N);
  const R h = st->h;
  const int n_emit = mode == JOB_STAGE2 ? 0 : st->job_n, slot0 = st->job_slot, lo = st->job_lo;
  const R tl = st->t_last, hh = st->t - tl;
  double acc[2 * KT] = {};
  // the first half's block reaches as far as the second's: the same passes for both
  for (long p = 0; (long)blockIdx.x * kBlock + p * stride < a.N; ++p) {
    const long i = first + p * stride;
    const bool valid = i < a.N;
    R x[KT], y = 0, k1 = 0, yn = 0, k7 = 0;
    if (valid) {
      lr_load_row<R, KT, EXACT>(l, K, a.ldv, i, x);
      y = a.y[i], k1 = a.k[0][i], yn = a.ynew[i], k7 = a.k[6][i];
    }
    if (n_emit > 0) {
      R Q[4] = {0, 0, 0, 0};
      if (valid) {
        R kv[7];
        kv[0] = k1, kv[6] = k7;
#pragma unroll
        for (int j = 1; j < 6; ++j) kv[j] = a.k[j][i];
        dense_coeffs<R>(kv, Q);
      }
      const long blk = pl.blk + p * l.blocks;
      emit_rows<R>(
          n_emit, valid, Q, y, tl, hh, sh[pl.half], [&](int q) { return a.t_eval[lo + q]; },
          [&](int q, R val) {
            if (a.ring) a.ring[(size_t)(slot0 + q) * a.ldv + i] = val;
          },
          [&](int q, double2 sums) {
            if (pl.live && blk < nblk) reinterpret_cast<double2 *>(a.ord_part)[(size_t)(slot0 + q) * nblk + blk] = sums;
          });
    }
    if (mode == JOB_EMIT || !valid) continue;
    if (mode == JOB_COMMIT) {
      // commit (dp45.cu:123-125, FSAL copy :160)
      a.ylast[i] = y;
      a.y[i] = y = yn;
      a.k[0][i] = k1 = k7;
    }
    R c, s;
    stage2_vector<R>(a, i, y, k1, h, c, s);
    lr_accumulate<R, KT, EXACT>(x, K, c, s, acc);
  }
  if (mode != JOB_EMIT) lr_write_partials<KT>(pl, acc, K, l.blocks, l.part_out);
}

// ---------------------------------------------------------------------
// Small networks: whole attempts in one workgroup.
// Between launches of 25 workgroups (N = 200) a stage is 3.6 us of latency:
// a launch, the state check, one round trip for the rows, one for the
// epilogue.  Up to N = 256 (FP32) or 128 (FP64) the whole matrix fits the
// registers of one workgroup of 8 waves (G groups of 8 rows per wave, one
// 16-byte piece per lane and row), so one workgroup runs attempt after
// attempt in one launch: oscillator i's phase and k_j stay in thread i's
// registers, the stage vectors in LDS, a stage is two barriers, and
// kmt_advance needs no graph.  (Streaming a larger matrix into the one CU
// from its L2 was slower than the launches: N=300 FP32 96 us per attempt
// against 27.)  Sums, error partials, output rows and the controller follow
// the launched kernels' order exactly (lane l's columns are those of thread l
// of stage_ring_kernel, the only ones that see a column < 64 VEC; 8 rows per
// error partial; 256 oscillators per order partial), so results are the same
// bits.
// ---------------------------------------------------------------------
constexpr int kSmallThreads = 512;
constexpr int kSmallWaves = kSmallThreads / kWave;
template <class R> constexpr int kSmallMaxN = kWave * 16 / (int)sizeof(R);  // columns of one wave
template <class R> constexpr int kSmallMaxGroups = kSmallMaxN<R> / (8 * kSmallWaves);

template <class R> struct SmallArgs {
  const R *A;
  long lda, N, ldv;
  const R *omega;
  R *y, *ylast, *ynew;
  R *k[7];
  R *cs;  // the stage-2 vector between launches
  R c1;
  State<R> *st;
  const R *t_eval;
  R *times, *ring, *r_ring;
};

template <int I, int U, class F> __device__ __forceinline__ void small_unroll(F &&f) {
  if constexpr (I < U) {
    f(std::integral_constant<int, I>{});
    small_unroll<I + 1, U>(f);
  }
}

// The wave's rows: groups wave, wave + 8, ... of 8 rows, zero past the matrix
template <class R, int G>
__device__ __forceinline__ void small_load_rows(const SmallArgs<R> &a, u32x4 (&rows)[G][8]) {
  const int wave = threadIdx.x / kWave, c = threadIdx.x % kWave * (16 / (int)sizeof(R));
  small_unroll<0, G>([&](auto gi) {
    constexpr int g = decltype(gi)::value;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const long row = (long)(g * kSmallWaves + wave) * 8 + r;
      const bool in = c < a.lda && row < a.N;
      const u32x4 raw = *reinterpret_cast<const u32x4 *>(a.A + (in ? row * a.lda + c : 0));
      rows[g][r] = in ? raw : u32x4{0, 0, 0, 0};
    }
  });
}

// C, S of every row against the stage vector v (zero past N) -> sum
template <class R, int G>
__device__ __forceinline__ void small_row_sums(u32x4 (&rows)[G][8], const R (&v)[2][kSmallMaxN<R>],
                                               double (&sum)[2][kSmallMaxN<R>]) {
  constexpr int VEC = 16 / sizeof(R), ROWS = 8;
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  R cv[VEC], sv[VEC];
  load_reals<R, VEC>(v[0] + lane * VEC, cv);
  load_reals<R, VEC>(v[1] + lane * VEC, sv);
  small_unroll<0, G>([&](auto gi) {
    constexpr int g = decltype(gi)::value;
    double acc[2 * ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      // opaque: the conversions to double stay here (kept across stages they
      // take twice the matrix's registers)
      asm volatile("" : "+v"(rows[g][r]));
      R m[VEC];
      unpack<R>(rows[g][r], m);
      acc[r] = acc[ROWS + r] = 0.0;
#pragma unroll
      for (int q = 0; q < VEC; ++q) {
        acc[r] = __builtin_fma((double)m[q], (double)cv[q], acc[r]);
        acc[ROWS + r] = __builtin_fma((double)m[q], (double)sv[q], acc[ROWS + r]);
      }
    }
    const double t = wave_reduce<double, 2 * ROWS>(acc, lane);
    const int slot = wave_slot<2 * ROWS>(lane);
    sum[slot / ROWS][(g * kSmallWaves + wave) * ROWS + slot % ROWS] = t;
    __builtin_amdgcn_sched_barrier(0);  // one group's sums in registers at a time
  });
}

template <class R, int G>
__global__ __launch_bounds__(kSmallThreads) void small_attempts_kernel(const SmallArgs<R> a, int attempts) {
  constexpr int NMAX = kSmallMaxN<R>;
  static_assert(NMAX <= kBlock && NMAX % 8 == 0, "one order partial; whole groups of rows");
  __shared__ __align__(16) R v[2][2][NMAX];  // stage vectors (cos, sin), used alternately
  __shared__ double sum[2][NMAX];            // C, S; squared errors
  __shared__ double part[2][kBlock];         // error partials; (cos, sin) of an output row
  __shared__ State<R> S;
  u32x4 rows[G][8];
  small_load_rows<R, G>(a, rows);
  const int tid = threadIdx.x, lane = tid % kWave, N = (int)a.N;
  const bool mine = tid < N;
  R y = 0, yl = 0, yn = 0, om = 0, k[7] = {};
  if (tid == 0) S = *a.st;
  if (mine) {
    y = a.y[tid], yl = a.ylast[tid], yn = a.ynew[tid], om = a.omega[tid];
#pragma unroll
    for (int j = 0; j < 7; ++j) k[j] = a.k[j][tid];
  }
  if (tid < NMAX) {
    v[0][0][tid] = mine ? a.cs[tid] : (R)0;
    v[0][1][tid] = mine ? a.cs[a.ldv + tid] : (R)0;
    v[1][0][tid] = v[1][1][tid] = (R)0;
  }
  __syncthreads();
  auto set_vector = [&](R yt, int buf) {
    R c, s;
    rsincos<R>(yt, c, s);
    v[buf][0][tid] = c;
    v[buf][1][tid] = s;
  };
  for (int at = 0; at < attempts; ++at) {
    const int active = S.active, pending = S.commit_pending;
    const R h = S.h;
    __syncthreads();  // S is read by all before the controller rewrites it
    if (!active) break;
    if (!pending) {
      // stages 2..7, one copy of the row sums: f of the vector in buffer
      // s & 1 is k_s; the next vector goes to the other buffer
      R err = 0;
#pragma unroll 1
      for (int s = 2; s <= 7; ++s) {
        small_row_sums<R, G>(rows, v[s & 1], sum);
        __syncthreads();
        const int t = mine ? tid : 0;
        const R f = rhs_value<R>(om, a.c1, v[s & 1][0][t], v[s & 1][1][t], (R)sum[0][t], (R)sum[1][t]);
        R acc = 0;
        small_unroll<2, 8>([&](auto stage) {
          constexpr int S1 = decltype(stage)::value;
          if (s != S1) return;
          k[S1 - 1] = f;
          acc = k[0] * (R)(S1 < 7 ? tab::A[S1 < 7 ? S1 - 1 : 0][0] : tab::E[0]);
#pragma unroll
          for (int j = 1; j < S1; ++j)
            acc = rfma<R>(k[j], (R)(S1 < 7 ? tab::A[S1 < 7 ? S1 - 1 : 0][j] : tab::E[j]), acc);
        });
        if (s < 7) {
          const R yt = rfma<R>(acc, h, y);
          if (s == 6) yn = yt;
          if (mine) set_vector(yt, (s + 1) & 1);
        } else {
          err = acc;
        }
        __syncthreads();
      }
      const R num = h * err;
      const R den = rfma<R>(S.rtl, rmax<R>(rabs<R>(y), rabs<R>(yn)), S.atl);
      const R e = num / den;
      if (tid < NMAX) sum[0][tid] = mine ? (double)e * (double)e : 0.0;
      __syncthreads();
      if (tid < kBlock) {
        double p = 0.0;
        if (8 * tid < N) {
          double q = 0.0;
#pragma unroll
          for (int r = 0; r < 8; ++r) q += sum[0][8 * tid + r];
          p += q;
        }
        part[0][tid] = p;
      }
      __syncthreads();
    }
    if (tid < kWave) {
      State<R> W = S;
      const int o = control_first_output(W) + lane;
      const R te = o < W.n_eval ? a.t_eval[o] : (R)NAN;
      control_decide<R>(W, block_tree(part[0]), N, a.t_eval, te, a.times, lane);
      W.fin_n = 0;  // the rows' order parameters follow here
      if (lane == 0) S = W;
    }
    __syncthreads();
    const int mode = S.job_mode, n_emit = S.job_n, slot0 = S.job_slot;
    if (n_emit > 0) {
      const R tl = S.t_last, hh = S.t - tl;
      R Q[4];
      dense_coeffs<R>(k, Q);
      for (int q = 0; q < n_emit; ++q) {
        R c = 0, s = 0;
        if (mine) {
          const R val = dense_value<R>(Q, y, hh, (a.t_eval[S.job_lo + q] - tl) / hh);
          if (a.ring) a.ring[(size_t)(slot0 + q) * a.ldv + tid] = val;
          rsincos<R>(val, c, s);
        }
        if (tid < kBlock) {
          part[0][tid] = (double)c;
          part[1][tid] = (double)s;
        }
        __syncthreads();
        if (tid < kWave) {
          const double X = block_tree(part[0]), Y = block_tree(part[1]);
          if (lane == 0) a.r_ring[slot0 + q] = order_value<R>(X, Y, N);
        }
        __syncthreads();
      }
    }
    if (mode == JOB_COMMIT) yl = y, y = yn, k[0] = k[6];
    if (mine && (mode == JOB_COMMIT || mode == JOB_STAGE2)) set_vector(rfma<R>(k[0] * (R)tab::A[0][0], S.h, y), 0);
    __syncthreads();
    if (mode == JOB_EMIT) break;  // the ring is full: only the host can go on
  }
  if (tid == 0) *a.st = S;
  if (mine) {
    a.y[tid] = y, a.ylast[tid] = yl, a.ynew[tid] = yn;
#pragma unroll
    for (int j = 0; j < 7; ++j) a.k[j][tid] = k[j];
    a.cs[tid] = v[0][0][tid];
    a.cs[a.ldv + tid] = v[0][1][tid];
  }
}

// XT[m][i] = X[i][m] (XT cleared past N by its allocation)
template <class R>
__global__ __launch_bounds__(kBlock) void transpose_factor_kernel(const R *X, int K, long N, long ldv, R *XT) {
  const long i = (long)blockIdx.x * kBlock + threadIdx.x;
  if (i < N)
    for (int m = 0; m < K; ++m) XT[m * ldv + i] = X[i * K + m];
}

// ---------------------------------------------------------------------
// Small helpers: sin/cos of a phase vector, stand-alone order parameter,
// interpolation over the last accepted step, adjacency generation and
// conversion.
// ---------------------------------------------------------------------
template <class R>
__global__ __launch_bounds__(kBlock) void sincos_kernel(const R *y, long N, long ldv, R *cs) {
  const long i = (long)blockIdx.x * kBlock + threadIdx.x;
  if (i < N) {
    R c, s;
    rsincos<R>(y[i], c, s);
    cs[i] = c;
    cs[ldv + i] = s;
  }
}

// The same over the padded length: zeros at [N, ldv) of both halves, for a
// (cos, sin) buffer that other calls with other N share.
template <class R>
__global__ __launch_bounds__(kBlock) void sincos_pad_kernel(const R *y, long N, long ldv, R *cs) {
  const long i = (long)blockIdx.x * kBlock + threadIdx.x;
  if (i < ldv) {
    R c = 0, s = 0;
    if (i < N) rsincos<R>(y[i], c, s);
    cs[i] = c;
    cs[ldv + i] = s;
  }
}

template <class R>
__global__ __launch_bounds__(kBlock) void order_partial_kernel(const R *y, long N, double *part) {
  __shared__ double sh[kBlock];
  const long i = (long)blockIdx.x * kBlock + threadIdx.x;
  double c = 0, s = 0;
  if (i < N) {
    R cy, sy;
    rsincos<R>(y[i], cy, sy);
    c = (double)cy;
    s = (double)sy;
  }
  const double bc = block_sum(c, sh);
  const double bs = block_sum(s, sh);
  if (threadIdx.x == 0) { part[2 * blockIdx.x] = bc; part[2 * blockIdx.x + 1] = bs; }
}

template <class R>
__global__ __launch_bounds__(kBlock) void order_final_kernel(const double *part, int nblk, long N, double *out) {
  __shared__ double sh[kBlock];
  double sx = 0, sy = 0;
  for (int b = threadIdx.x; b < nblk; b += kBlock) { sx += part[2 * b]; sy += part[2 * b + 1]; }
  const double X = block_sum(sx, sh);
  const double Y = block_sum(sy, sh);
  if (threadIdx.x == 0) out[0] = (double)order_value<R>(X, Y, N);
}

// dp45_eval (dp45.cu:143-146) over the last accepted step.
template <class R>
__global__ __launch_bounds__(kBlock) void interp_kernel(const State<R> *st, long N, const R *ylast,
                                                        const R *k0, const R *k1, const R *k2, const R *k3,
                                                        const R *k4, const R *k5, const R *k6, R t_eval, R *out) {
  const long i = (long)blockIdx.x * kBlock + threadIdx.x;
  if (i >= N) return;
  const R tl = st->t_last;
  const R hh = st->t - tl;
  const R x = (t_eval - tl) / hh;
  const R kv[7] = {k0[i], k1[i], k2[i], k3[i], k4[i], k5[i], k6[i]};
  R Q[4];
  dense_coeffs<R>(kv, Q);
  out[i] = dense_value<R>(Q, ylast[i], hh, x);
}

__device__ __forceinline__ uint16_t to_bf16_rne(float f) {
  uint32_t u = __builtin_bit_cast(uint32_t, f);
  if ((u & 0x7FFFFFFFu) > 0x7F800000u) return (uint16_t)0x7FC0u;  // NaN
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

template <class R, class S> __device__ __forceinline__ S store_value(R v, R inv_scale);
template <> __device__ __forceinline__ float store_value<float, float>(float v, float) { return v; }
template <> __device__ __forceinline__ double store_value<double, double>(double v, double) { return v; }
template <> __device__ __forceinline__ bf16_t store_value<float, bf16_t>(float v, float s) {
  return bf16_t{to_bf16_rne(v * s)};
}
template <> __device__ __forceinline__ f16_t store_value<float, f16_t>(float v, float s) {
  return f16_t{__builtin_bit_cast(uint16_t, (_Float16)(v * s))};
}

// FP64 working precision with 16-bit storage: the scaled value is rounded
// to FP32 first, then to 16 bits (two roundings; the stored matrix is what
// the integration uses and what kmt_get_adjacency_rows returns).
template <> __device__ __forceinline__ bf16_t store_value<double, bf16_t>(double v, double s) {
  return bf16_t{to_bf16_rne((float)(v * s))};
}
template <> __device__ __forceinline__ f16_t store_value<double, f16_t>(double v, double s) {
  return f16_t{__builtin_bit_cast(uint16_t, (_Float16)(float)(v * s))};
}

template <class R, class S> __device__ __forceinline__ R load_value(S v, R scale);
template <> __device__ __forceinline__ float load_value<float, float>(float v, float) { return v; }
template <> __device__ __forceinline__ double load_value<double, double>(double v, double) { return v; }
template <> __device__ __forceinline__ float load_value<float, bf16_t>(bf16_t v, float s) {
  return __builtin_bit_cast(float, (uint32_t)v.bits << 16) * s;
}
template <> __device__ __forceinline__ float load_value<float, f16_t>(f16_t v, float s) {
  return (float)__builtin_bit_cast(_Float16, v.bits) * s;
}
template <> __device__ __forceinline__ double load_value<double, bf16_t>(bf16_t v, double s) {
  return (double)__builtin_bit_cast(float, (uint32_t)v.bits << 16) * s;
}
template <> __device__ __forceinline__ double load_value<double, f16_t>(f16_t v, double s) {
  return (double)(float)__builtin_bit_cast(_Float16, v.bits) * s;
}

// getadj (kuramoto.cu:145-161) from the stored factor: one workgroup per
// row, M_ij = sum_m fma(w_m, X_im X_jm, acc) (exactly symmetric).
template <class R, class S>
__global__ __launch_bounds__(kBlock) void gen_adj_kernel(const R *X, const R *w, int K, long N, long row0, S *A,
                                                         long lda, R inv_scale) {
  const long i = row0 + blockIdx.x;
  if (i >= N) return;
  const R *Xi = X + i * K;
  S *Ai = A + (size_t)blockIdx.x * lda;
  for (long j = threadIdx.x; j < N; j += kBlock) {
    const R *Xj = X + j * K;
    R acc = 0;
    for (int m = 0; m < K; ++m) acc = rfma<R>(w[m], Xi[m] * Xj[m], acc);
    Ai[j] = store_value<R, S>(acc, inv_scale);
  }
}

// Host-supplied rows (real) -> stored rows.
template <class R, class S>
__global__ __launch_bounds__(kBlock) void convert_rows_kernel(const R *src, long ld_src, long ncols, long nrows, S *dst,
                                                              long lda, R inv_scale) {
  const long r = blockIdx.y;
  if (r >= nrows) return;
  for (long j = (long)blockIdx.x * kBlock + threadIdx.x; j < ncols; j += (long)gridDim.x * kBlock)
    dst[(size_t)r * lda + j] = store_value<R, S>(src[(size_t)r * ld_src + j], inv_scale);
}

// Stored rows -> real rows (dequantized).
template <class R, class S>
__global__ __launch_bounds__(kBlock) void read_rows_kernel(const S *A, long lda, long ncols, long nrows, R scale,
                                                           R *dst) {
  const long r = blockIdx.y;
  if (r >= nrows) return;
  for (long j = (long)blockIdx.x * kBlock + threadIdx.x; j < ncols; j += (long)gridDim.x * kBlock)
    dst[(size_t)r * ncols + j] = load_value<R, S>(A[(size_t)r * lda + j], scale);
}

}  // namespace kmt
