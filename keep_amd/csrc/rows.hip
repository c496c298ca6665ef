// Routed VQ mat-vecs on the matrix cores: out[route] = W[expert] . x[row] for
// verify windows (routes grouped by expert in tiles of up to 16), single
// routes, and one matrix against a few rows; 8-bit E8 codes with fp16 or bf16
// rows, E8P codes with fp16 rows. Replaces the lane-per-chunk mat-vecs of
// matvec.hip where K and the scale group allow it (gather_vqmm_verify_rows,
// src/ramp/ops/vq_switch.py:286-377, and gather_vqmm's direct routes).
//
// A block's 16 waves form groups of K / CK waves, CK = 512 (8-bit) or 256
// (E8P); wave s of a group owns K slice s. Lane (c, q) of a 16x16x32 MFMA holds
// A row c (a route's x) and W row c, and of the slice the codewords of quarter
// q: 16 bytes of codes, one load. At step s the B operand is codeword s of
// them, straight from the block's LDS image: 8-bit codes look up eight weights
// x 4 ready in the rows' 16-bit type (one permute, one 16-byte lookup), E8P
// codes T' ^ M and a conversion (as gemm_q8.hip). The A operands of a tile stay
// in registers; a group streams the tile's W rows in units of 32, the codes of
// the next two units in flight (nothing else is loaded inside the loop: loads
// retire in order, and an x load behind a code load would wait for it), each
// unit's slice sums scaled and added over the waves, in slice order, through
// LDS. Per codeword that is 2 VALU operations for all the routes of a tile,
// against 7 per route on the mat-vec, whose lookups also collide in LDS (one
// 4 KiB table; here lane l reads copy l % 16 of each entry).
//
// A row's result depends on its own x and codes only, in slice order, whatever
// tile it falls in: grouped, flat and single calls agree bit for bit. Up to 128
// routes every block groups them itself (plan_small_to): no plan launch, no
// gather of the routes' rows.
//
// Bound: waiting. 8 fp16 rows, top-6 of 256 8-bit experts 4096 -> 2048, groups of
// 512 (48 MB): 24 us, against 128 on the mat-vec in tiles of 4 routes it replaces
// and 55 on single routes; the codes alone would take 9.5. Its waves wait 54% of
// the time (the first codes and x of each block's six units, the barrier of
// each) with the VALU busy 37%, LDS 29%, the matrix cores 23%. 333 bf16 rows of
// the same, 143 us: 48%, 46% and 37%, waves waiting 50%; a third of its units
// are those of a plan's empty tiles. One matrix 4096 x 4096, 16 rows, 14 us
// against 37.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "moe_dev.h"
#include "plan_dev.h"
#include "q8_dev.h"
#include "route_dev.h"

namespace keep {

constexpr int VR_THREADS = 1024;
constexpr int VR_M = 16;     // routes per tile
constexpr int VR_RT = 2;     // 16-row tiles of W per unit
constexpr int VR_UNIT = 16 * VR_RT;
constexpr int VR_DEPTH = 2;  // units in flight

struct RowsArgs {
  const void* x;
  int64_t x_rows;
  const uint8_t* codes;
  const void* scales;
  int sdt;
  const void* table;  // E8P: T and M (keep_e8p_prepare); E8: the packed 8-bit table
  const int32_t *rhs, *lhs;
  int64_t routes, x_div;
  int64_t E, N, K, G;
  int spg;                             // K slices per scale group
  const int32_t *order, *te, *to, *tc; // tiles of a route plan (null: planned here, or none)
  int64_t n_tiles;                     // of te, or routes (flat), or rows / 16 (one matrix)
  int local, planned;                  // routes <= PLAN_SMALL_R: tiles in LDS, of one route each or grouped here
  int nsl, groups;                     // K slices, and groups of that many waves per block
  int upt;                             // units per tile
  void* out;
  int odt;
};

typedef _Float16 vr_h8 __attribute__((ext_vector_type(8)));
typedef float vr_f4 __attribute__((ext_vector_type(4)));

template <bool BF>
__device__ __forceinline__ vr_f4 vr_mfma(uint4 a, uint4 b, vr_f4 c) {
  typedef __bf16 b8 __attribute__((ext_vector_type(8)));
  if constexpr (BF)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8, a), __builtin_bit_cast(b8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(vr_h8, a), __builtin_bit_cast(vr_h8, b), c, 0, 0, 0);
}

template <int CB, typename XT>
__global__ __launch_bounds__(VR_THREADS) void k_vq_rows(RowsArgs a) {
  constexpr bool BF = std::is_same<XT, bf16s>::value;
  constexpr bool E8 = CB == 8;
  static_assert(E8 || !BF, "E8P rows are fp16");
  constexpr int SPL = E8 ? 16 : 8;  // codewords of a lane's 16 bytes
  constexpr int CK = SPL * 32;      // K per slice
  constexpr int D = VR_DEPTH;
  // the image first: its lookups' offsets then fit the instruction
  __shared__ struct {
    uint4 img[256 * 16];
    float red[2][16][VR_RT][VR_M][20];  // [parity][wave][row tile][route][row]: quarters 16 banks apart
  } S;
  auto& img = S.img;
  auto& red = S.red;
  __shared__ int32_t s_r[PLAN_SMALL_R], s_b[PLAN_SMALL_R], s_order[PLAN_SMALL_R], s_te[PLAN_SMALL_R],
      s_to[PLAN_SMALL_R], s_tc[PLAN_SMALL_R], s_nt[2];
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, q = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  // the image entry's table words first: loads retire in order, so behind the codes they would wait for HBM
  const int en = tid >> 2;
  uint32_t p8 = 0;
  uint2 tt = make_uint2(0u, 0u), tm = tt;
  if constexpr (E8) {
    p8 = ((const uint32_t*)a.table)[en];
  } else {
    tt = ((const uint2*)a.table)[en];
    tm = ((const uint2*)a.table)[256 + en];
  }
  int nt = (int)a.n_tiles;
  if (a.local) {
    if (tid < a.routes) {
      const int e = a.rhs[tid];
      s_r[tid] = s_te[tid] = e;
      s_order[tid] = s_to[tid] = tid;
      s_tc[tid] = 1;
    }
    __syncthreads();
    if (a.planned) {
      const PlanSmallOut o{nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 0,
                           s_order, s_te, s_to, s_tc};
      plan_small_to([&](int r) { return s_r[r]; }, (int)a.routes, (int)a.E, VR_M, o, s_b, s_nt);
      nt = s_nt[0];  // the routes of invalid experts too: their rows are NaN
    }
  }
  // this wave's group and K slice; the groups of the grid share the units evenly, in contiguous runs
  const int grp = wv / a.nsl, sl = wv - grp * a.nsl;
  const bool work = grp < a.groups;
  const int U = nt * a.upt, ng = (int)gridDim.x * a.groups;
  const int per = (U + ng - 1) / ng;
  const int u0 = min(U, (grp * (int)gridDim.x + (int)blockIdx.x) * per);
  const int u1 = work ? min(U, u0 + per) : u0;
  if (U == 0) return;
  const int64_t C = a.K >> 3;
  const int64_t sbytes = a.sdt == KEEP_F32 ? 4 : 2;
  const int64_t gsl = (work ? sl : 0) / a.spg;
  // x past the end reads as zeros without memory traffic (rows with no route)
  const __amdgpu_buffer_rsrc_t xres =
      __builtin_amdgcn_make_buffer_rsrc((void*)a.x, (short)0, (int)(a.x_rows * a.K * 2), 0x00020000);

  // a tile's expert row (-1: none valid) and, for lane c, its route and A row
  auto expert_of = [&](int tile) -> int64_t {
    const int64_t e = a.local ? s_te[tile] : a.te ? a.te[tile] : a.rhs ? a.rhs[tile] : 0;
    return e < 0 || e >= a.E ? -1 : e;
  };
  struct Tile {
    int m, route;  // route of lane c, -1 - route where its row is NaN
    uint32_t ao;
  };
  auto tile_of = [&](int tile, int64_t e) -> Tile {
    int64_t off = tile;
    Tile t{1, 0, 0x80000000u};
    if (a.local) {
      off = s_to[tile];
      t.m = s_tc[tile];
    } else if (a.te) {
      off = a.to[tile];
      t.m = a.tc[tile];
      if (off < 0 || off + t.m > a.routes) t.m = 0;
    } else if (!a.rhs) {
      off = (int64_t)tile * VR_M;
      t.m = (int)min((int64_t)VR_M, a.routes - off);
    }
    t.m = min(t.m, VR_M);
    if (c < t.m) {
      t.route = (int)off + c;
      if (a.local) t.route = s_order[t.route];
      else if (a.order) t.route = a.order[t.route];
      const int64_t xr = a.lhs ? (int64_t)a.lhs[t.route] : t.route / a.x_div;
      if (xr < 0 || xr >= a.x_rows || e < 0) t.route = -1 - t.route;
      else t.ao = (uint32_t)((xr * a.K + (work ? sl : 0) * CK + q * (SPL * 8)) * 2);
    }
    return t;
  };
  struct Buf {
    uint4 q[VR_RT];
    uint32_t s[VR_RT];
  };
  // the unit last loaded (past the group's end its last unit again), and the one being computed
  int lu = u0, ltile = u0 < u1 ? u0 / a.upt : 0, lk = u0 < u1 ? u0 - ltile * a.upt : 0;
  int tile = ltile, k = lk;
  int64_t e = expert_of(tile), lrow = max(e, (int64_t)0) * a.N;
  auto load_unit = [&](Buf& b) {
#pragma unroll
    for (int rt = 0; rt < VR_RT; ++rt) {
      const int64_t row = lrow + min((int64_t)lk * VR_UNIT + rt * 16 + c, a.N - 1);
      b.q[rt] = ldg16_q(a.codes + row * (C * (CB / 8)) + (work ? sl : 0) * 64 + q * 16);
      b.s[rt] = ldg4_q((const char*)a.scales + ((row * a.G + gsl) * sbytes & ~(int64_t)3));
    }
    if (lu + 1 < u1) {
      ++lu;
      if (++lk == a.upt) {
        lk = 0;
        ++ltile;
        lrow = max(expert_of(ltile), (int64_t)0) * a.N;
      }
    }
  };
  Tile t = tile_of(tile, e);
  uint4 A[SPL];
  auto load_a = [&]() {
#pragma unroll
    for (int s = 0; s < SPL; ++s) {
      const auto v = __builtin_amdgcn_raw_buffer_load_b128(xres, (int)(t.ao + 16 * s), 0, 0);
      A[s] = uint4{(uint32_t)v[0], (uint32_t)v[1], (uint32_t)v[2], (uint32_t)v[3]};
    }
  };
  load_a();
  Buf b[D];
#pragma unroll
  for (int i = 0; i < D; ++i) load_unit(b[i]);
  {  // the LDS image, while they land: sixteen copies of entry tid / 4, each 8 lanes' store to 8 different slots
    uint4 v;
    if constexpr (E8) {
      uint32_t w[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {  // 2 (nibble - 8) as 16-bit floats (encode_half_units(v): v / 2)
        const int lo = 4 * ((int)((p8 >> (8 * i)) & 15u) - 8), hi = 4 * ((int)((p8 >> (8 * i + 4)) & 15u) - 8);
        constexpr int PK = BF ? PAIR_BF16 : PAIR_F16;
        w[i] = encode_half_units<PK>(lo) | (encode_half_units<PK>(hi) << 16);
      }
      v = make_uint4(w[0], w[1], w[2], w[3]);
    } else {
      tt = q8_natural(tt);
      tm = q8_natural(tm);
      v = make_uint4(tt.x ^ 0x80808080u, tt.y ^ 0x80808080u, tm.x, tm.y);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) img[en * 16 + (((tid & 3) * 4 + en + i) & 15)] = v;
  }
  rt_lds_barrier();
  const char* im = (const char*)img;
  const Q8Keys keys = q8_keys(lane);
  auto lookup = [&](const uint4& w, int s) -> uint4 {  // codeword s of the lane's 16 bytes
    if constexpr (E8) {
      const uint32_t d = s < 4 ? w.x : s < 8 ? w.y : s < 12 ? w.z : w.w;
      return *(const uint4*)(im + __builtin_amdgcn_perm(d, (uint32_t)c << 4, 0x0c0c0400u + ((uint32_t)(s & 3) << 8)));
    } else {
      const uint32_t d = s < 2 ? w.x : s < 4 ? w.y : s < 6 ? w.z : w.w;
      const bool hi = (s & 1) != 0;
      const uint2 x1 = *(const uint2*)(im + __builtin_amdgcn_perm(d, keys.base1, hi ? keys.s1hi : keys.s1lo));
      const uint2 x2 = *(const uint2*)(im + __builtin_amdgcn_perm(d, keys.base2, hi ? keys.s2hi : keys.s2lo));
      return __builtin_bit_cast(uint4, q8_f16_of_bytes(make_uint2(x1.x ^ x2.x, x1.y ^ x2.y)));
    }
  };
  auto unit = [&](int u, Buf& bu, int par) {
    if (k == a.upt && u < u1) {  // the next tile (wave-uniform)
      k = 0;
      ++tile;
      e = expert_of(tile);
      t = tile_of(tile, e);
      load_a();
    }
    vr_f4 acc[VR_RT];
#pragma unroll
    for (int rt = 0; rt < VR_RT; ++rt) acc[rt] = vr_f4{0.f, 0.f, 0.f, 0.f};
    if (u < u1) {  // wave-uniform; no loads inside, so their order stays known
#pragma unroll
      for (int s = 0; s < SPL; ++s)
#pragma unroll
        for (int rt = 0; rt < VR_RT; ++rt) acc[rt] = vr_mfma<BF>(A[s], lookup(bu.q[rt], s), acc[rt]);
    }
    float sc[VR_RT];
#pragma unroll
    for (int rt = 0; rt < VR_RT; ++rt) {
      // the scale's half of its word: units start at even rows
      const uint32_t half = (uint32_t)gsl + (a.G & 1 ? (uint32_t)(max(e, (int64_t)0) * a.N) + c : 0u);
      sc[rt] = 0.25f * scale_cvt(bu.s[rt], a.sdt, half);
      asm volatile("" : "+v"(sc[rt]));  // done with the unit's words before they are loaded again
    }
    load_unit(bu);
#pragma unroll
    for (int rt = 0; rt < VR_RT; ++rt)
#pragma unroll
      for (int v = 0; v < 4; ++v) red[par][wv][rt][4 * q + v][c] = acc[rt][v] * sc[rt];
    rt_lds_barrier();  // LDS only: the codes in flight are not waited for
    // the unit's outputs, 32 columns per route, by the group's threads
    const int64_t n0 = (int64_t)k * VR_UNIT;
    const int rel = sl * 64 + lane;
    if (u < u1)
      for (int o = rel; o < t.m * VR_UNIT; o += a.nsl * 64) {
        const int r = o / VR_UNIT, col = o % VR_UNIT;
        float v = 0.f;
        for (int s = 0; s < a.nsl; ++s) v += red[par][grp * a.nsl + s][col >> 4][r][col & 15];
        const int ro = __shfl(t.route, r, 64);
        if (ro < 0) v = __builtin_nanf("");
        if (n0 + col < a.N) {
          const int64_t at = (int64_t)(ro < 0 ? -1 - ro : ro) * a.N + n0 + col;
          if (a.odt == KEEP_F32) ((float*)a.out)[at] = v;
          else if (a.odt == KEEP_BF16) ((uint16_t*)a.out)[at] = from_float<bf16s>(v).bits;
          else ((_Float16*)a.out)[at] = (_Float16)v;
        }
      }
    ++k;
  };
  // every wave of the block runs the same number of units (the barriers)
  for (int i = 0; i < per; i += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (i + d >= per) break;
      unit(u0 + i + d, b[d], (i + d) & 1);
    }
  }
}

}  // namespace keep

using namespace keep;

extern "C" int keep_vq_rows_supported(int x_dtype, int code_bits, int64_t K, int64_t group_size) {
  if (!::keep::dims_ok({K, group_size})) return 0;
  const int64_t ck = code_bits == 8 ? 512 : 256, waves = 16;
  return (code_bits == 8 || code_bits == 16) &&
                 (x_dtype == KEEP_F16 || (x_dtype == KEEP_BF16 && code_bits == 8)) && K > 0 && group_size > 0 &&
                 K % ck == 0 && K / ck <= waves && group_size % ck == 0 && K % group_size == 0
             ? 1
             : 0;
}

extern "C" int keep_vq_rows(const void* x, int x_dtype, int64_t x_rows, const void* codes, int code_bits,
                            const void* scales, int scale_dtype, const void* tables, const int32_t* rhs,
                            const int32_t* lhs, int64_t routes, int64_t x_div, int grouped, const int32_t* order,
                            const int32_t* tile_expert, const int32_t* tile_offset, const int32_t* tile_count,
                            int64_t n_tiles, int64_t num_experts, int64_t N, int64_t K, int64_t group_size, void* out,
                            int out_dtype, void* stream) {
  KEEP_REQUIRE_DIMS(x_rows, routes, x_div, n_tiles, num_experts, N, K, group_size);
  KEEP_REQUIRE(dtype_ok(scale_dtype) && dtype_ok(out_dtype), "bad dtype enum");
  KEEP_REQUIRE(keep_vq_rows_supported(x_dtype, code_bits, K, group_size),
               "matrix-core rows need fp16 rows (8-bit codes: or bf16), K and the scale group multiples of %d",
               code_bits == 8 ? 512 : 256);
  KEEP_REQUIRE(N > 0 && num_experts > 0 && x_rows <= 0x40000000LL / K, "bad sizes (x must be under 2 GiB)");
  if (routes == 0) return KEEP_OK;
  KEEP_REQUIRE(x && codes && scales && tables && out && x_rows > 0, "null pointer argument");
  KEEP_REQUIRE(rhs || (num_experts == 1 && !grouped), "rhs may be NULL only for one matrix (num_experts == 1)");
  KEEP_REQUIRE(lhs || x_div > 0, "x_div must be > 0 without lhs");
  KEEP_REQUIRE(!grouped || routes <= PLAN_SMALL_R || (order && tile_expert && tile_offset && tile_count),
               "more than %d grouped routes need a route plan", PLAN_SMALL_R);
  KEEP_REQUIRE(aligned(x, 16) && aligned(codes, 16) && aligned(scales, 4) && aligned(tables, 16),
               "x, codes and tables must be 16-byte aligned, scales 4 bytes");
  RowsArgs a{};
  a.x = x; a.x_rows = x_rows; a.codes = (const uint8_t*)codes; a.scales = scales; a.sdt = scale_dtype;
  a.table = code_bits == 16 ? (const char*)tables + TQ_OFFSET : (const char*)tables;
  a.rhs = rhs; a.lhs = lhs; a.routes = routes; a.x_div = x_div > 0 ? x_div : 1;
  a.E = num_experts; a.N = N; a.K = K; a.G = K / group_size;
  const int64_t ck = code_bits == 8 ? 512 : 256;
  a.spg = (int)(group_size / ck);
  a.nsl = (int)(K / ck);
  a.groups = VR_THREADS / 64 / a.nsl;
  a.upt = (int)((N + VR_UNIT - 1) / VR_UNIT);
  a.out = out; a.odt = out_dtype;
  a.local = rhs && routes <= PLAN_SMALL_R;
  if (a.local) {
    a.planned = grouped;
    a.n_tiles = routes;
  } else if (grouped) {
    a.order = order; a.te = tile_expert; a.to = tile_offset; a.tc = tile_count;
    a.n_tiles = n_tiles;
  } else {
    a.n_tiles = rhs ? routes : (routes + VR_M - 1) / VR_M;
  }
  KEEP_REQUIRE(a.n_tiles <= 0x7fffffffLL / a.upt, "too many units");
  const dim3 grid((unsigned)std::max<int64_t>(1, std::min<int64_t>(a.n_tiles * a.upt, 256)));
  hipStream_t s = (hipStream_t)stream;
  if (code_bits == 16) hipLaunchKernelGGL((k_vq_rows<16, _Float16>), grid, dim3(VR_THREADS), 0, s, a);
  else if (x_dtype == KEEP_F16) hipLaunchKernelGGL((k_vq_rows<8, _Float16>), grid, dim3(VR_THREADS), 0, s, a);
  else hipLaunchKernelGGL((k_vq_rows<8, bf16s>), grid, dim3(VR_THREADS), 0, s, a);
  return launch_status("keep_vq_rows");
}
