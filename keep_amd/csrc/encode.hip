// Nearest-codeword encoders on gfx950: E8P (16-bit codes) and the 8-bit E8
// table, under an optional diagonal metric w (one shared [8], or one [8] per
// vector), the data-free RTN quantiser of src/keep/quant/rtn.py:270-318 and
// the weighted search of src/keep/vq/e8.py:367-539.
//
// The answer is defined as the exhaustive scan's: the codeword minimising
//   D = ((q0 + q1) + (q2 + q3)) + ((q4 + q5) + (q6 + q7)),  q_d = w_d ((v_d - c_d)^2)
// in double precision, ties to the lowest code. The E8P search is factored
// instead of scanning 65,536 codewords: for each shift (+1/4 with even stored
// sign parity, -1/4 with odd) and each of the 256 abs rows, the signs that
// follow the target's are optimal; an odd sign count is fixed by the single
// flip of least distance (ties: the lowest stored signs), and dimensions whose
// sign is free (w_d |t_d| = 0) take the lowest stored signs that satisfy the
// parity. Every candidate's D is the same tree over the same exact terms as
// the scan's (|v_d - c_d| = | |t_d| -+ a_d | exactly in double), so the two
// agree bit for bit except where distinct codewords' D differ by less than
// its rounding. With a metric every row is measured, one thread per vector,
// the 256 rows in LDS, every lane of a wave reading the same row (a
// broadcast): fp64 VALU-bound. Without one, k_encode_bounds measures only the
// rows that bounds from the matrix cores leave.
#include <algorithm>

#include "common.h"

namespace keep {

constexpr int ENC_THREADS = 256;
__constant__ int kEncShuffle[8] = {0, 4, 1, 5, 2, 6, 3, 7};  // dim d reads packed nibble kEncShuffle[d]

__device__ __forceinline__ double enc_tree8(const double (&q)[8]) {
#pragma clang fp contract(off)
  return ((q[0] + q[1]) + (q[2] + q[3])) + ((q[4] + q[5]) + (q[6] + q[7]));
}

// The vector (divided by its scale, correctly rounded to fp32) and its weights.
template <int WMODE>
__device__ __forceinline__ void enc_load(const float* x, const float* w, const float* scales, int64_t vps, int64_t i,
                                         float (&v)[8], double (&wd)[8]) {
  const float4* xp = (const float4*)(x + i * 8);
  const float4 a = xp[0], b = xp[1];
  const float xs[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
  const double s = scales ? (double)scales[i / vps] : 1.0;
#pragma unroll
  for (int d = 0; d < 8; ++d) v[d] = scales ? (float)((double)xs[d] / s) : xs[d];
#pragma unroll
  for (int d = 0; d < 8; ++d) wd[d] = WMODE == 0 ? 1.0 : (double)w[(WMODE == 2 ? i * 8 : 0) + d];
}

// One shift of the E8P search: |t| per dimension, the packed sign bits of t and
// of the dimensions whose sign is free (w |t| = 0).
struct EncShift {
  double at[8];
  uint32_t tneg, freem;
};
__device__ __forceinline__ EncShift enc_shift(const float (&v)[8], const double (&wd)[8], uint32_t p) {
#pragma clang fp contract(off)
  const double sig = p ? -0.25 : 0.25;
  EncShift s;
  s.tneg = s.freem = 0;
#pragma unroll
  for (int d = 0; d < 8; ++d) {
    const double t = (double)v[d] - sig;
    s.at[d] = fabs(t);
    if (t < 0.0) s.tneg |= 1u << kEncShuffle[d];
    if (wd[d] * s.at[d] == 0.0) s.freem |= 1u << kEncShuffle[d];
  }
  return s;
}

// The best codeword of abs row r (magnitudes a, packed sign bits neg) under shift p: its distance and code.
__device__ __forceinline__ double enc_row(const EncShift& s, const double (&wd)[8], uint32_t p, uint32_t r,
                                          const float (&a)[8], uint32_t neg, uint32_t& code) {
#pragma clang fp contract(off)
  double q[8];
#pragma unroll
  for (int d = 0; d < 8; ++d) {
    const double df = s.at[d] - (double)a[d];
    q[d] = wd[d] * (df * df);
  }
  double D = enc_tree8(q);
  const uint32_t E = s.tneg ^ neg;  // dims to negate so that every value follows its target's sign
  uint32_t S = E ^ p;               // stored signs (decode: eff = signs ^ parity on bit 0)
  if (s.freem) {
    uint32_t sf = S & ~s.freem;
    if ((uint32_t)(__builtin_popcount(sf) & 1) != p) sf |= s.freem & (0u - s.freem);
    S = sf;
  } else if (__builtin_popcount(E) & 1u) {
    double bd = __builtin_inf();
    uint32_t bs = 0xFFFFu;
#pragma unroll
    for (int f = 0; f < 8; ++f) {
      const double keep = q[f];
      const double df = s.at[f] + (double)a[f];
      q[f] = wd[f] * (df * df);
      const double Df = enc_tree8(q);
      q[f] = keep;
      const uint32_t Sf = S ^ (1u << kEncShuffle[f]);
      if (Df < bd || (Df == bd && Sf < bs)) {
        bd = Df;
        bs = Sf;
      }
    }
    D = bd;
    S = bs;
  }
  code = (r << 8) | S;
  return D;
}

__device__ __forceinline__ void enc_magnitudes(const float* row, float (&a)[8]) {
  const float4 lo = *(const float4*)row, hi = *(const float4*)(row + 4);
  a[0] = lo.x; a[1] = lo.y; a[2] = lo.z; a[3] = lo.w; a[4] = hi.x; a[5] = hi.y; a[6] = hi.z; a[7] = hi.w;
}

// Row e of the table in LDS: magnitudes and packed sign bits (E8P), or the signed values (8-bit E8).
template <bool E8P>
__device__ __forceinline__ uint32_t enc_table_row(uint32_t word, float (&a)[8]) {
  uint32_t neg = 0;
#pragma unroll
  for (int d = 0; d < 8; ++d) {
    const int s = E8P ? kEncShuffle[d] : d;
    const int m = (int)((word >> (4 * s)) & 15u) - 8;
    a[d] = E8P ? fabsf((float)m * 0.5f) : (float)m * 0.5f;
    if (E8P && m < 0) neg |= 1u << s;
  }
  return neg;
}

// Weighted search: every row of both shifts, one thread per vector.
template <int WMODE>
__global__ __launch_bounds__(ENC_THREADS) void k_e8p_encode(const float* x, int64_t n, const float* w,
                                                           const uint32_t* table, const float* scales, int64_t vps,
                                                           uint16_t* out) {
  __shared__ __attribute__((aligned(16))) float sa[256][8];
  __shared__ uint32_t sneg[256];
  {
    float a[8];
    sneg[threadIdx.x] = enc_table_row<true>(table[threadIdx.x], a);
#pragma unroll
    for (int d = 0; d < 8; ++d) sa[threadIdx.x][d] = a[d];
  }
  __syncthreads();
  const int64_t i = (int64_t)blockIdx.x * ENC_THREADS + threadIdx.x;
  if (i >= n) return;
  float v[8];
  double wd[8];
  enc_load<WMODE>(x, w, scales, vps, i, v, wd);
  double best = __builtin_inf();
  uint32_t best_code = 0xFFFFFFFFu;
  for (uint32_t p = 0; p < 2; ++p) {
    const EncShift s = enc_shift(v, wd, p);
    for (uint32_t r = 0; r < 256; ++r) {
      float a[8];
      enc_magnitudes(sa[r], a);
      uint32_t code;
      const double D = enc_row(s, wd, p, r, a, sneg[r], code);
      if (D < best || (D == best && code < best_code)) {
        best = D;
        best_code = code;
      }
    }
  }
  out[i] = (uint16_t)best_code;
}

// 8-bit E8 distance to a signed row.
__device__ __forceinline__ double enc_dist8(const float (&v)[8], const float (&c)[8]) {
#pragma clang fp contract(off)
  double q[8];
#pragma unroll
  for (int d = 0; d < 8; ++d) {
    const double df = (double)v[d] - (double)c[d];
    q[d] = df * df;
  }
  return enc_tree8(q);
}

// Weighted 8-bit E8: the 256 entries scanned in order (a tie keeps the lower index).
template <int WMODE>
__global__ __launch_bounds__(ENC_THREADS) void k_e8_encode(const float* x, int64_t n, const float* w,
                                                          const uint32_t* table, const float* scales, int64_t vps,
                                                          uint8_t* out) {
#pragma clang fp contract(off)
  __shared__ __attribute__((aligned(16))) float sc[256][8];
  {
    float a[8];
    (void)enc_table_row<false>(table[threadIdx.x], a);
#pragma unroll
    for (int d = 0; d < 8; ++d) sc[threadIdx.x][d] = a[d];
  }
  __syncthreads();
  const int64_t i = (int64_t)blockIdx.x * ENC_THREADS + threadIdx.x;
  if (i >= n) return;
  float v[8];
  double wd[8];
  enc_load<WMODE>(x, w, scales, vps, i, v, wd);
  double best = __builtin_inf();
  uint32_t best_code = 0;
  for (uint32_t r = 0; r < 256; ++r) {
    double q[8];
#pragma unroll
    for (int d = 0; d < 8; ++d) {
      const double df = (double)v[d] - (double)sc[r][d];
      q[d] = wd[d] * (df * df);
    }
    const double D = enc_tree8(q);
    if (D < best) {
      best = D;
      best_code = r;
    }
  }
  out[i] = (uint8_t)best_code;
}

// Unweighted search: the matrix cores bound every row's distance, and only the
// rows that could be nearest are measured in double.
//
// With C = |a_r|^2 / 2, half the distance to row r is |t|^2 / 2 - t . a_r + C
// (E8P: t the magnitudes |v -+ 1/4|, plus at least 2 min_d |t_d| min_d a_rd
// where the signs need a flip: a flip of dim f adds 2 |t_f| a_rf). A wave takes
// 64 vectors, one per lane, as two sets of 32 columns of 32x32x16 fp16 MFMAs,
// and 32 rows of the table at a time: t is split into hi + lo / 2048 fp16
// halves (one permlane swap lays the hi of a set in the lower lanes and its lo
// in the upper: rows a and a / 2048), and a second MFMA adds C, the flip bound
// and |t|^2 / 2 (both as hi + lo), so an accumulator is the lower bound of (row,
// vector) itself, off by less than EST = 2^-16 (|t|^2 / 2 + 64): 21 bits of
// every factor, at most 48 additions of terms summing below 2 (|t|^2 / 2 + 64).
// The bounds carry EST on top, so they are positive and order as their bits;
// the low 8 bits make way for the row's place. Cleared they only lower a bound;
// with the place in them a bound may stand up to 255 ulp higher, so the place
// orders the bounds but is cleared again before one is held against a distance.
// Each lane keeps its two least (three operations per bound); the least of both
// halves is measured exactly (enc_row / enc_dist8, the scan's own arithmetic),
// and a row whose bound is within the error of that distance (one vector in
// 65 of an RTN weight has any) is queued, for the wave's lanes to measure side
// by side, least distance and then least code kept per vector in LDS. Where
// a lane's second least passes too, its 32 vectors' bounds are formed again and
// all that pass are queued. A nearest row's bound is never above the measured
// distance plus its error, so ties and all, the answer is the full scan's.
// Vectors beyond +-64 (where the fp16 halves would overflow) and non-finite
// ones take the scan. VALU-bound; 1M vectors of an RTN weight:
// 150 us (the scan: 2,325 us).
typedef _Float16 enc_h8 __attribute__((ext_vector_type(8)));
typedef float enc_f16v __attribute__((ext_vector_type(16)));

constexpr int ENC_Q = 64 + 512;  // queue: under 64 waiting, plus half of a tile's 32 rows of 32 vectors

// LDS written by some lanes of a wave, read by others: its LDS operations complete in order, so only the compiler's
// order matters.
__device__ __forceinline__ void enc_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// (x, y) -> (x of the lower lanes | y of the lower lanes moved up, x of the upper lanes moved down | y of the upper).
__device__ __forceinline__ void enc_swap(uint32_t& x, uint32_t& y) {
  const auto r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
  x = r[0];
  y = r[1];
}
__device__ __forceinline__ void enc_swap(enc_h8& x, enc_h8& y) {
  typedef uint32_t u4 __attribute__((ext_vector_type(4)));
  u4 a = __builtin_bit_cast(u4, x), b = __builtin_bit_cast(u4, y);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t p = a[i], q = b[i];
    enc_swap(p, q);
    a[i] = p;
    b[i] = q;
  }
  x = __builtin_bit_cast(enc_h8, a);
  y = __builtin_bit_cast(enc_h8, b);
}

template <bool E8P, typename OUT>
__global__ __launch_bounds__(ENC_THREADS, 4) void k_encode_bounds(const float* x, int64_t n, const uint32_t* table,
                                                                  const float* scales, int64_t vps, OUT* out) {
  constexpr int WAVES = ENC_THREADS / 64;
  constexpr int NP = E8P ? 2 : 1;
  __shared__ __attribute__((aligned(16))) float sa[256][8];
  __shared__ uint32_t sneg[256];
  __shared__ enc_h8 sA[8][64], sA2[8][32];  // A operands of the eight 32-row tiles, by lane (sA2: lane % 32)
  __shared__ __attribute__((aligned(16))) float sv[WAVES][64][8];
  __shared__ unsigned long long sbest[WAVES][64];
  __shared__ uint32_t scode[WAVES][64];
  __shared__ uint16_t squeue[WAVES][ENC_Q];
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5, wv = threadIdx.x >> 6;
  {
    // one row per thread: its values, and its A operands
    const int r = threadIdx.x;
    float a[8];
    const uint32_t neg = enc_table_row<E8P>(table[r], a);
    float nn = 0.f, amin = fabsf(a[0]);
    enc_h8 hi, lo, a2v;
#pragma unroll
    for (int d = 0; d < 8; ++d) {
      sa[r][d] = a[d];
      hi[d] = (_Float16)a[d];
      lo[d] = (_Float16)(a[d] * 0.00048828125f);
      nn = fmaf(a[d], a[d], nn);
      amin = fminf(amin, fabsf(a[d]));
    }
    const bool odd = __builtin_popcount(neg) & 1;
    const float P = E8P && odd ? 2.f * amin : 0.f, N = E8P && !odd ? 2.f * amin : 0.f;
    const float a2[8] = {0.5f * nn, P, P * 0.00048828125f, N, N * 0.00048828125f, 1.f, 0.00048828125f, 0.f};
#pragma unroll
    for (int d = 0; d < 8; ++d) a2v[d] = (_Float16)a2[d];
    sneg[r] = neg;
    sA[r >> 5][r & 31] = hi;
    sA[r >> 5][32 + (r & 31)] = lo;
    sA2[r >> 5][r & 31] = a2v;
  }
  __syncthreads();
  const double one[8] = {1.0, 1.0, 1.0, 1.0, 1.0, 1.0, 1.0, 1.0};
  // f >= 0 -> a normal fp16 hi and 2048 x the rest
  auto split = [](float f, float& hi, float& lo) {
    hi = (float)__builtin_amdgcn_cvt_pkrtz(fmaxf(f, 6.103515625e-05f), 0.f)[0];
    lo = (f - hi) * 2048.f;
  };
  const int64_t groups = (n + 63) / 64;
  for (int64_t g = (int64_t)blockIdx.x * WAVES + wv; g < groups; g += (int64_t)gridDim.x * WAVES) {
    float v[8];
    {
      const int64_t i = min(g * 64 + lane, n - 1);
      enc_magnitudes(x + i * 8, v);
      if (scales) {
        const float s = scales[i / vps];
#pragma unroll
        for (int d = 0; d < 8; ++d) v[d] = v[d] / s;  // correctly rounded
      }
      *(float4*)&sv[wv][lane][0] = make_float4(v[0], v[1], v[2], v[3]);
      *(float4*)&sv[wv][lane][4] = make_float4(v[4], v[5], v[6], v[7]);
    }
    bool bad = false;
#pragma unroll
    for (int d = 0; d < 8; ++d) bad |= !(fabsf(v[d]) <= 64.f);
    enc_h8 B[2][NP], B2[2][NP];  // of the two sets of 32 vectors
    float slack = 0.f;
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      float nn = 0.f, tmin = 3.4e38f;
      uint32_t odd = 0;
      enc_h8 vh, vl;
#pragma unroll
      for (int d = 0; d < 8; ++d) {
        const float t = bad ? 0.f : E8P ? v[d] - (p ? -0.25f : 0.25f) : v[d];
        const float f = fabsf(t);
        nn = fmaf(f, f, nn);
        tmin = fminf(tmin, f);
        float hi, lo;
        split(f, hi, lo);
        if (E8P) odd ^= __float_as_uint(t);  // sign bits (-0: t == 0, where the flip bound is 0 either way)
        vh[d] = (_Float16)(!E8P && t < 0.f ? hi : -hi);
        vl[d] = (_Float16)(!E8P && t < 0.f ? lo : -lo);
      }
      const bool flip = odd >> 31;
      const float eps = (0.5f * nn + 64.f) * 1.52587890625e-05f;
      float nh, nl, mh = 0.f, ml = 0.f;
      split(0.5f * nn + eps, nh, nl);
      if (E8P) split(tmin, mh, ml);
      const float b2[8] = {1.f, flip ? 0.f : mh, flip ? 0.f : ml, flip ? mh : 0.f, flip ? ml : 0.f, nh, nl, 0.f};
#pragma unroll
      for (int d = 0; d < 8; ++d) B2[0][p][d] = (_Float16)b2[d];
      B[0][p] = vh;
      B[1][p] = vl;
      B2[1][p] = B2[0][p];
      enc_swap(B[0][p], B[1][p]);
      enc_swap(B2[0][p], B2[1][p]);
      if (h) B2[0][p] = B2[1][p] = enc_h8{};  // the second MFMA's terms are in the lower lanes
      slack = fmaxf(slack, eps);
    }
    auto bounds = [&](const enc_h8& b, const enc_h8& b2, int t) -> enc_f16v {
      const enc_f16v z = __builtin_amdgcn_mfma_f32_32x32x16_f16(sA2[t][c], b2, enc_f16v{}, 0, 0, 0);
      return __builtin_amdgcn_mfma_f32_32x32x16_f16(sA[t][lane], b, z, 0, 0, 0);
    };
    // the two least bounds of each lane, place p * 128 + t * 16 + u in the low bits (accumulator u of tile t is row
    // 32 t + 8 (u / 4) + 4 h + u % 4)
    uint32_t m1[2] = {0x7f800000u, 0x7f800000u}, m2[2] = {0x7f800000u, 0x7f800000u};
    uint32_t keep = 0xffffff00u;
    asm volatile("" : "+v"(keep));  // in a register: and-or takes one scalar
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll 1
      for (int t = 0; t < 8; ++t) {
        enc_f16v b[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) b[q] = bounds(B[q][p], B2[q][p], t);
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          uint32_t u1 = 0x7f800000u, u2 = 0x7f800000u;
#pragma unroll
          for (int u = 0; u < 16; ++u) {
            const uint32_t k = (__float_as_uint(b[q][u]) & keep) | (uint32_t)u;
            u2 = min(max(u1, k), u2);
            u1 = min(u1, k);
          }
          u1 |= (uint32_t)(p * 128 + t * 16);
          u2 |= (uint32_t)(p * 128 + t * 16);
          m2[q] = min(min(m2[q], u2), max(m1[q], u1));
          m1[q] = min(m1[q], u1);
        }
      }
    // lane c < 32 holds a vector of set 0, lane 32 + c one of set 1: its two lane halves' least and second least
    enc_swap(m1[0], m1[1]);
    enc_swap(m2[0], m2[1]);
    auto row_of = [&](uint32_t m, uint32_t half) -> uint32_t {  // shift * 256 + row
      return ((m & 0xf0u) << 1) + ((m & 0xcu) << 1) + 4u * half + (m & 3u);
    };
    auto measure = [&](const float (&vv)[8], uint32_t pr, uint32_t& code) -> double {
      const uint32_t p = pr >> 8, r = pr & 255u;
      float a[8];
      enc_magnitudes(sa[r], a);
      if constexpr (E8P) {
        return enc_row(enc_shift(vv, one, p), one, p, r, a, sneg[r], code);
      } else {
        code = r;
        return enc_dist8(vv, a);
      }
    };
    const bool upper = m1[1] < m1[0];
    uint32_t code;
    {
      const double D0 = measure(v, row_of(upper ? m1[1] : m1[0], upper), code);
      sbest[wv][lane] = (unsigned long long)__double_as_longlong(D0);
      scode[wv][lane] = code;
      slack = bad ? -3.4e38f : (float)(0.5 * D0) + 2.f * slack;  // the most that a nearest row's bound can be
    }
    const float thr = slack;
    enc_wave_sync();
    // the queued rows, measured 64 at a time
    uint32_t cnt = 0;
    auto drain = [&]() {
#pragma unroll 1
      for (uint32_t o = 0; o < cnt; o += 64) {
        enc_wave_sync();
        const bool on = o + (uint32_t)lane < cnt;
        const uint32_t ent = on ? squeue[wv][o + lane] : 0u;
        const uint32_t k = ent & 63u;
        float vv[8];
        enc_magnitudes(sv[wv][k], vv);
        uint32_t cd = 0;
        const double D = on ? measure(vv, ent >> 6, cd) : 0.0;
        const unsigned long long db = (unsigned long long)__double_as_longlong(D);  // D >= 0: ordered as its bits
        const unsigned long long before = sbest[wv][k];
        enc_wave_sync();
        if (on) atomicMin(&sbest[wv][k], db);
        enc_wave_sync();
        const unsigned long long now = sbest[wv][k];
        if (on && now < before) scode[wv][k] = 0xFFFFFFFFu;
        enc_wave_sync();
        if (on && db == now) atomicMin(&scode[wv][k], cd);
        enc_wave_sync();
      }
      cnt = 0;
    };
    auto append = [&](bool in, uint32_t ent) {
      const unsigned long long hit = __ballot(in);
      if (hit) {
        const uint32_t at = cnt + __builtin_amdgcn_mbcnt_hi((uint32_t)(hit >> 32),
                                                            __builtin_amdgcn_mbcnt_lo((uint32_t)hit, 0u));
        if (in) squeue[wv][at] = (uint16_t)ent;
        cnt += (uint32_t)__popcll(hit);
      }
    };
    const uint32_t other = upper ? m1[0] : m1[1];  // the other half's least
    append(__uint_as_float(other & keep) <= thr, row_of(other, !upper) << 6 | (uint32_t)lane);
    const unsigned long long again = __ballot(__uint_as_float(min(m2[0], m2[1]) & keep) <= thr);
    uint32_t sets = ((uint32_t)again != 0u ? 1u : 0u) | ((uint32_t)(again >> 32) != 0u ? 2u : 0u);
    while (cnt || sets) {
      if (cnt >= 64 || !sets) drain();
      if (!sets) break;
      const int q = (int)(sets & 1u) ^ 1;
      sets &= sets - 1u;
      const float tq = __shfl(thr, 32 * q + c, 64);
#pragma unroll 1
      for (int pt = 0; pt < NP * 8; ++pt) {
        const bool p1 = NP > 1 && pt >= 8;
        const enc_h8 b0 = q ? B[1][0] : B[0][0], b1 = q ? B[1][NP - 1] : B[0][NP - 1];
        const enc_h8 c0 = q ? B2[1][0] : B2[0][0], c1 = q ? B2[1][NP - 1] : B2[0][NP - 1];
        const enc_f16v b = bounds(p1 ? b1 : b0, p1 ? c1 : c0, pt & 7);
#pragma unroll 1
        for (int half = 0; half < 2; ++half) {
          if (cnt >= 64) drain();
#pragma unroll
          for (int u = 0; u < 8; ++u)
            append(__uint_as_float(__float_as_uint(half ? b[8 + u] : b[u]) & keep) <= tq,
                   row_of((uint32_t)(pt * 16 + 8 * half + u), (uint32_t)h) << 6 | (uint32_t)(32 * q + c));
        }
      }
    }
    enc_wave_sync();
    code = scode[wv][lane];
    if (bad) {  // the scan
      double best = __builtin_inf();
      code = E8P ? 0xFFFFFFFFu : 0u;
#pragma unroll 1
      for (uint32_t pr = 0; pr < NP * 256u; ++pr) {
        uint32_t cd;
        const double D = measure(v, pr, cd);
        if (D < best || (E8P && D == best && cd < code)) {
          best = D;
          code = cd;
        }
      }
    }
    if (g * 64 + lane < n) out[g * 64 + lane] = (OUT)code;
    enc_wave_sync();
  }
}

// Per (row, group) max |x| / divisor in fp32 (the max_abs estimator,
// src/keep/quant/rtn.py:253-264): one wave per group, 16-byte loads where the
// groups allow them. Any output may be null: the scales, the divisors of the
// encoder (1 where a scale is not positive), the stored fp16 scales.
__global__ __launch_bounds__(256) void k_group_absmax(const float* x, int64_t groups_total, int64_t group_size,
                                                      float divisor, int quads, float* scales, float* safe,
                                                      _Float16* stored) {
  const int64_t g = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (g >= groups_total) return;
  const float* p = x + g * group_size;
  float m = 0.f;
  if (quads) {
    for (int64_t j = lane; j < group_size / 4; j += 64) {
      const float4 q = ((const float4*)p)[j];
      m = fmaxf(fmaxf(fmaxf(m, fabsf(q.x)), fmaxf(fabsf(q.y), fabsf(q.z))), fabsf(q.w));
    }
  } else {
    for (int64_t j = lane; j < group_size; j += 64) m = fmaxf(m, fabsf(p[j]));
  }
  for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
  if (lane == 0) {
    const float s = (float)((double)m / (double)divisor);  // the correctly rounded fp32 quotient
    if (scales) scales[g] = s;
    if (safe) safe[g] = s > 0.f ? s : 1.f;
    if (stored) stored[g] = (_Float16)s;
  }
}

template <int WMODE>
static void launch_weighted(int code_bits, const float* x, int64_t n, const float* w, const uint32_t* table,
                            const float* scales, int64_t vps, void* out, hipStream_t s) {
  const dim3 grid((unsigned)((n + ENC_THREADS - 1) / ENC_THREADS)), blk(ENC_THREADS);
  if (code_bits == 16)
    hipLaunchKernelGGL((k_e8p_encode<WMODE>), grid, blk, 0, s, x, n, w, table, scales, vps, (uint16_t*)out);
  else
    hipLaunchKernelGGL((k_e8_encode<WMODE>), grid, blk, 0, s, x, n, w, table, scales, vps, (uint8_t*)out);
}

// Persistent waves of 64 vectors at a time: the table's operands are built once per wave.
static void launch_bounds(int code_bits, const float* x, int64_t n, const uint32_t* table, const float* scales,
                          int64_t vps, void* out, hipStream_t s) {
  const int64_t blocks = std::min<int64_t>((n + 255) / 256, 256 * 4);
  const dim3 grid((unsigned)blocks), blk(ENC_THREADS);
  if (code_bits == 16)
    hipLaunchKernelGGL((k_encode_bounds<true, uint16_t>), grid, blk, 0, s, x, n, table, scales, vps, (uint16_t*)out);
  else
    hipLaunchKernelGGL((k_encode_bounds<false, uint8_t>), grid, blk, 0, s, x, n, table, scales, vps, (uint8_t*)out);
}

}  // namespace keep

using namespace keep;

extern "C" int keep_vq_encode(const float* vectors, int64_t n, int code_bits, const float* diagonal, int diag_mode,
                              const uint32_t* table, const float* scales, int64_t vectors_per_scale, void* codes,
                              void* stream) {
  KEEP_REQUIRE_DIMS(n, vectors_per_scale);
  KEEP_REQUIRE(code_bits == 8 || code_bits == 16, "code_bits must be 8 or 16, got %d", code_bits);
  KEEP_REQUIRE(diag_mode >= 0 && diag_mode <= 2, "diag_mode must be 0 (none), 1 (shared [8]) or 2 (per vector)");
  KEEP_REQUIRE(n >= 0, "n must be >= 0");
  if (n == 0) return KEEP_OK;
  KEEP_REQUIRE(vectors && table && codes && (diag_mode == 0 || diagonal), "null pointer argument");
  KEEP_REQUIRE(aligned(vectors, 16), "vectors must be 16-byte aligned");
  KEEP_REQUIRE(!scales || vectors_per_scale >= 1, "vectors_per_scale must be >= 1");
  KEEP_REQUIRE((n + ENC_THREADS - 1) / ENC_THREADS <= 0x7fffffffLL, "too many vectors");
  hipStream_t s = (hipStream_t)stream;
  if (diag_mode == 0) launch_bounds(code_bits, vectors, n, table, scales, vectors_per_scale, codes, s);
  else if (diag_mode == 1)
    launch_weighted<1>(code_bits, vectors, n, diagonal, table, scales, vectors_per_scale, codes, s);
  else launch_weighted<2>(code_bits, vectors, n, diagonal, table, scales, vectors_per_scale, codes, s);
  return launch_status("keep_vq_encode");
}

static int group_scales(const char* what, const float* x, int64_t groups_total, int64_t group_size, float divisor,
                        float* scales, float* safe, void* stored, void* stream) {
  KEEP_REQUIRE(groups_total >= 0 && group_size >= 1, "bad group sizes");
  KEEP_REQUIRE(divisor > 0.f, "divisor must be positive");
  if (groups_total == 0) return KEEP_OK;
  KEEP_REQUIRE(x && (scales || (safe && stored)), "null pointer argument");
  const int64_t blocks = (groups_total + 3) / 4;
  KEEP_REQUIRE(blocks <= 0x7fffffffLL, "too many groups");
  const int quads = group_size % 4 == 0 && aligned(x, 16);
  hipLaunchKernelGGL(k_group_absmax, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, x, groups_total,
                     group_size, divisor, quads, scales, safe, (_Float16*)stored);
  return launch_status(what);
}

extern "C" int keep_group_absmax(const float* x, int64_t groups_total, int64_t group_size, float divisor,
                                 float* scales, void* stream) {
  KEEP_REQUIRE_DIMS(groups_total, group_size);
  return group_scales("keep_group_absmax", x, groups_total, group_size, divisor, scales, nullptr, nullptr, stream);
}

extern "C" int keep_rtn_scales(const float* x, int64_t groups_total, int64_t group_size, float divisor, float* safe,
                               void* stored, void* stream) {
  KEEP_REQUIRE_DIMS(groups_total, group_size);
  return group_scales("keep_rtn_scales", x, groups_total, group_size, divisor, nullptr, safe, stored, stream);
}
