// Q4_0 GEMM for any number of activation rows and any K % 32 == 0 on MFMA:
// prompts of a few dozen to a few hundred rows, and the batched decode rows of
// linears whose K is not a multiple of 64.
//
// Y[m][n] = sum_k X[m][k] * W[n][k], W in GGUF Q4_0 blocks (fp16 d, 16 bytes
// of nibbles, value d * (nibble - 8)), bf16 X and Y, fp32 accumulation.
//
// What bounds it: at these sizes neither the matrix cores nor HBM but latency
// and the conversion of the weights, so
//  * the weights go from the GGUF stream to MFMA B operands in registers, with
//    no bf16 copy of the matrix in memory (dequantising it first and
//    multiplying after writes and reads 64 bytes per 18-byte block);
//  * a wave holds an MT x NT tile of 16 x 16 outputs over ALL of its rows, so a
//    weight is converted once per MT row tiles;
//  * WK groups of waves split K (128-element tiles t = wk, wk + WK, ...) and meet
//    in LDS at the end, so a few hundred output columns already fill the chip;
//  * activations are staged in LDS, a tile's 16 MT rows x 256 bytes per group,
//    loaded one tile ahead: with WN = 1 the slice is the wave's own and the loop
//    has no barrier, with more the WN waves of a group share it, one barrier a
//    tile.  (Read straight from memory in operand layout, 16 rows a load, 48 rows
//    of 6144 x 2560 took 13.5 us against 11.4.)
//
// Weights: lane 16 j + n loads block 4 t + j of weight row n (16 bytes of
// nibbles at 2-byte alignment, 2 of scale); a 4x4 transpose across the lanes
// n + 16 j gives lane (n, g) the k-group g of the tile's four blocks, group g
// being elements 8 g .. 8 g + 7 (the low nibbles of qs[8 g ..] for g < 2, the
// high ones of qs[8 (g - 2) ..] otherwise).  Then
//  * EXACT (m <= 16): B = nibble - 8, exact in bf16, and the block's sum is
//    scaled by d in fp32, the GEMV's arithmetic;
//  * else B = RNE_bf16(d * (nibble - 8)), the value q4_0_dequant_kernel writes
//    (its zeros of a negative d are -0, here +0, which no sum tells apart).
#include <limits.h>
#include <math.h>

#include <type_traits>

#include "smx_common.h"
#include "smx_launch.h"

namespace smx {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32_a2 __attribute__((aligned(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

// pack_bf16x2 as one v_cvt_pk_bf16_f32 (it compiles to two conversions, shifted
// and joined); the same bits.  Half of this kernel's operations are conversions.
__device__ __forceinline__ uint32_t cvt_pk_bf16(float lo, float hi) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{lo, hi}), bf16x2));
}

// fp32 product of the fp16 values in the low or high halves of a and d
// (v_fma_mix_f32 with a zero addend, so a zero product is +0; exact: 4 + 11 bits)
template <bool A_HI, bool D_HI>
__device__ __forceinline__ float mul_mix(uint32_t a, uint32_t d) {
  float r;
  if constexpr (A_HI && D_HI)
    __asm__("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[1,1,0] op_sel_hi:[1,1,0]" : "=v"(r) : "v"(a), "v"(d));
  else if constexpr (A_HI)
    __asm__("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[1,0,0] op_sel_hi:[1,1,0]" : "=v"(r) : "v"(a), "v"(d));
  else if constexpr (D_HI)
    __asm__("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[0,1,0] op_sel_hi:[1,1,0]" : "=v"(r) : "v"(a), "v"(d));
  else
    __asm__("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[0,0,0] op_sel_hi:[1,1,0]" : "=v"(r) : "v"(a), "v"(d));
  return r;
}

// The 8 nibbles of a k-group (bytes 0..3 of lo, then of hi) as an MFMA operand.
template <bool EXACT, bool D_HI>
__device__ __forceinline__ bf16x8 group_operand(uint32_t lo, uint32_t hi, uint32_t d) {
  uint32_t r[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t b = i < 2 ? lo : hi;
    // fp16 pair (1024 + nibble), minus 1032
    const f16x2 t = __builtin_bit_cast(
        f16x2, perm_b32(0x64646464u, b, (i & 1) ? 0x04030402u : 0x04010400u));
    const f16x2 v = t - f16x2{(_Float16)1032.0f, (_Float16)1032.0f};
    if constexpr (EXACT) {
      r[i] = cvt_pk_bf16((float)v[0], (float)v[1]);
    } else {
      const uint32_t vu = __builtin_bit_cast(uint32_t, v);
      r[i] = cvt_pk_bf16(mul_mix<false, D_HI>(vu, d), mul_mix<true, D_HI>(vu, d));
    }
  }
  return __builtin_bit_cast(bf16x8, r);
}

// One workgroup: WN x WK waves (wave = wk * WN + wn) over 16 MT rows and
// 16 NT WN columns; wave (wn, wk) computes its 16 NT columns over the tiles
// t = wk, wk + WK, ...  The WN waves of one wk share the tile's activations in
// LDS: each loads a part of the rows, and with WN > 1 two buffers alternate, so
// one barrier a tile is enough (WN == 1: the slice is the wave's own, no barrier).
template <int MT, int NT, int WN, int WK, bool EXACT>
__global__ __launch_bounds__(64 * WN * WK) void q4_0_gemm_rows_kernel(
    const uint8_t* w, const uint16_t* x, int nb, int n_out, int m, uint16_t* y, int vec) {
  static_assert(4 * MT % WN == 0, "whole activation loads per wave");
  constexpr int XL = 4 * MT / WN;  // this wave's activation loads per tile
  constexpr int SLICE = 256 * MT;  // 16-byte chunks of a tile's activations
  // [WK][buffers][16 MT rows x 16 chunks of 16 bytes]; the waves' sums at the end
  extern __shared__ u32x4 lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wn = wave % WN, wk = wave / WN;
  const int n = lane & 15, j = lane >> 4;  // j: the lane's block, then its k-group
  const int n0 = blockIdx.x * (16 * NT * WN), m0 = blockIdx.y * (16 * MT);
  const int ntiles = (nb + 3) >> 2;
  const uint32_t hshift = (uint32_t)(j >> 1) * 4u;  // high nibbles for k-groups 2 and 3

  // A block starts on a 4-byte boundary or 2 bytes past one (w % 4 == 0), the
  // same for all of a lane's blocks of a row.  It is read as the 5 dwords from
  // the boundary on, which hold all of its 18 bytes: (d, qs[0..1]), ..., or
  // (., d), qs[0..3], ....  (A 16-byte load 2 bytes off costs the L1 over 100
  // accesses a wave.)  In the first form the fifth dword ends 2 bytes past the
  // block; for the last block of the matrix it is read 2 bytes earlier instead.
  const uint8_t* wr[NT];
  uint32_t qsel[NT], dshift[NT];
  int off[NT], last4[NT];
  // this lane's last block of the parity of its own (its alignment then holds
  // for every tile; blocks past the row's end are read there and not used)
  const int bend = nb - 1 - (((nb - 1) ^ j) & 1);
  const int bmax = max(bend, 0);
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    const int row = min(n0 + 16 * (wn * NT + i) + n, n_out - 1);
    off[i] = ((uint32_t)row * (uint32_t)nb + (bend < 0 ? 0u : (uint32_t)j)) & 1u ? 2 : 0;
    wr[i] = w + (int64_t)row * (nb * 18);
    qsel[i] = off[i] ? 0x07060504u : 0x05040302u;
    dshift[i] = off[i] ? 16u : 0u;
    last4[i] = (int)min((int64_t)(n_out - row) * (nb * 18) - 4, (int64_t)INT_MAX);
  }
  u32x4 q[NT];
  uint32_t q4[NT], q4shift[NT];
  auto load_w = [&](int t) {
    const int o = 18 * min(4 * t + j, bmax);
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int oi = o - off[i], o4 = min(oi + 16, last4[i]);
      q[i] = *reinterpret_cast<const u32x4_a4*>(wr[i] + oi);
      q4[i] = *reinterpret_cast<const u32_a2*>(wr[i] + o4);
      q4shift[i] = 8u * (uint32_t)(oi + 16 - o4);
    }
  };
  // Load i of a tile's activations: rows 4 (wn XL + i) + j, chunk n of their 16
  // (rows past m repeat the last row: they only feed outputs that are not
  // stored; chunks past the row's end repeat its last block and are not used).
  uint32_t xo[XL];  // byte offsets of those rows (m * k * 2 < 2^31)
#pragma unroll
  for (int i = 0; i < XL; ++i)
    xo[i] = (uint32_t)min(m0 + 4 * (wn * XL + i) + j, m - 1) * (uint32_t)(nb * 64);
  u32x4 sv[XL];
  auto load_x = [&](int t) {
    const uint32_t o = 64u * (uint32_t)min(4 * t + (n >> 2), nb - 1) + 16u * (n & 3);
#pragma unroll
    for (int i = 0; i < XL; ++i)
      sv[i] = *reinterpret_cast<const u32x4*>(reinterpret_cast<const char*>(x) + (xo[i] + o));
  };
  // Chunk c of row r sits at chunk c ^ (r & 15) of the row's 256 bytes, so the
  // 16 rows of an operand read fall in different banks.
  u32x4* sl = lds + wk * (WN > 1 ? 2 * SLICE : SLICE);
  auto own_slice_fence = [&]() {
    // a slice of the wave's own: its LDS operations complete in order, so only
    // the compiler has to be kept from reordering
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  auto stage_x = [&]() {
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      const int r = 4 * (wn * XL + i) + j;
      sl[16 * r + (n ^ (r & 15))] = sv[i];
    }
    if constexpr (WN > 1) __syncthreads();
    else own_slice_fence();
  };

  f32x4 acc[MT][NT];
#pragma unroll
  for (int a = 0; a < MT; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};

  uint32_t qa[NT][4], qb[NT][4], dk[NT][2];  // a tile's operands by block (scales: two a word)
  auto spread = [&]() {
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      qa[i][0] = qa[i][2] = perm_b32(q[i].y, q[i].x, qsel[i]);
      qb[i][0] = qb[i][2] = perm_b32(q[i].z, q[i].y, qsel[i]);
      qa[i][1] = qa[i][3] = perm_b32(q[i].w, q[i].z, qsel[i]);
      qb[i][1] = qb[i][3] = perm_b32(q4[i] >> q4shift[i], q[i].w, qsel[i]);
      const uint32_t dl = q[i].x >> dshift[i];
      transpose_rows4(qa[i][0], qa[i][1], qa[i][2], qa[i][3]);
      transpose_rows4(qb[i][0], qb[i][1], qb[i][2], qb[i][3]);
      const auto a = __builtin_amdgcn_permlane16_swap(dl, dl, false, false);
      const uint32_t p = perm_b32(a[1], a[0], 0x05040100u);  // (d0, d1) in rows 0-1, (d2, d3) in rows 2-3
      const auto c = __builtin_amdgcn_permlane32_swap(p, p, false, false);
      dk[i][0] = c[0];
      dk[i][1] = c[1];
    }
  };
  auto block = [&](auto bc) {
    constexpr int b = decltype(bc)::value;
    bf16x8 B[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i)
      B[i] = group_operand<EXACT, (b & 1) != 0>((qa[i][b] >> hshift) & 0x0F0F0F0Fu,
                                                (qb[i][b] >> hshift) & 0x0F0F0F0Fu, dk[i][b >> 1]);
#pragma unroll
    for (int a = 0; a < MT; ++a) {
      const bf16x8 A = __builtin_bit_cast(bf16x8, sl[16 * (16 * a + n) + ((4 * b + j) ^ n)]);
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        if constexpr (EXACT) {
          const f32x4 c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              A, B[i], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
          const float d = f16_bits_to_f32((b & 1) ? dk[i][b >> 1] >> 16 : dk[i][b >> 1] & 0xffffu);
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[a][i][r] = fmaf(d, c[r], acc[a][i][r]);
        } else {
          acc[a][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A, B[i], acc[a][i], 0, 0, 0);
        }
      }
    }
  };
  using std::integral_constant;
  auto whole_tile = [&]() {
    block(integral_constant<int, 0>{});
    block(integral_constant<int, 1>{});
    block(integral_constant<int, 2>{});
    block(integral_constant<int, 3>{});
  };

  // Every wave runs the same number of iterations (a barrier each); past the
  // row's end it loads the last tile again and computes nothing.
  load_w(min(wk, ntiles - 1));
  load_x(min(wk, ntiles - 1));
  int buf = 0;
  for (int t0 = 0; t0 < ntiles; t0 += WK) {
    const int t = t0 + wk;
    spread();
    stage_x();
    __builtin_amdgcn_sched_barrier(0);  // the loads below reuse the registers just read
    load_w(min(t + WK, ntiles - 1));
    load_x(min(t + WK, ntiles - 1));
    if (4 * t + 4 <= nb) {
      whole_tile();
    } else {  // the 0..3 blocks after the last whole tile
      if (4 * t < nb) block(integral_constant<int, 0>{});
      if (4 * t + 1 < nb) block(integral_constant<int, 1>{});
      if (4 * t + 2 < nb) block(integral_constant<int, 2>{});
    }
    if constexpr (WN > 1) {
      sl += buf ? -SLICE : SLICE;
      buf ^= 1;
    } else {
      own_slice_fence();
    }
  }

  // Sum over the WK waves of a column group, one row tile at a time.  C layout:
  // lane l holds rows 4 (l >> 4) + r of column l & 15; a thread sums and stores
  // 4 columns of a row.
  f32x4* red = reinterpret_cast<f32x4*>(lds);  // [WK][WN NT][64]
  constexpr int CT = WN * NT, NTHR = 64 * WN * WK;
#pragma unroll
  for (int a = 0; a < MT; ++a) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NT; ++i) red[(wave * NT + i) * 64 + lane] = acc[a][i];
    __syncthreads();
#pragma unroll
    for (int e0 = 0; e0 < 64 * CT; e0 += NTHR) {
      const int e = e0 + (int)threadIdx.x;
      if (64 * CT % NTHR != 0 && e >= 64 * CT) break;
      const int row = e / (4 * CT), cq = e % (4 * CT);
      const int mr = m0 + 16 * a + row, o = n0 + 4 * cq;
      if (mr < m && o < n_out) {
        const int l0 = 16 * (row >> 2) + (cq & 3) * 4;
        float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int v = 0; v < WK; ++v)
#pragma unroll
          for (int c = 0; c < 4; ++c) s[c] += red[(v * CT + (cq >> 2)) * 64 + l0 + c][row & 3];
        uint16_t* yo = y + (int64_t)mr * n_out + o;
        if (vec) {  // n_out % 4 == 0 and y 8-byte aligned
          st_agent(reinterpret_cast<u32x2*>(yo), u32x2{cvt_pk_bf16(s[0], s[1]), cvt_pk_bf16(s[2], s[3])});
        } else {
#pragma unroll
          for (int c = 0; c < 4; ++c)
            if (o + c < n_out) st_agent(yo + c, f32_to_bf16(s[c]));
        }
      }
    }
  }
  stores_done();
}

template <int MT, int NT, int WN, int WK, bool EXACT = false>
hipError_t launch_rows(hipStream_t s, const void* x, const void* w, void* y, int m, int n, int nb) {
  constexpr int SLICES = WN > 1 ? 2 * WK : WK;
  constexpr size_t lds = 1024 * (SLICES * 4 * MT > WN * WK * NT ? SLICES * 4 * MT : WN * WK * NT);
  static_assert(lds <= 160 * 1024, "LDS of a CU");
  const int vec = n % 4 == 0 && (uintptr_t)y % 8 == 0;
  constexpr int BN = 16 * NT * WN;
  const dim3 grid((unsigned)((n + BN - 1) / BN), (unsigned)((m + 16 * MT - 1) / (16 * MT)));
  SMX_LAUNCH((q4_0_gemm_rows_kernel<MT, NT, WN, WK, EXACT>), grid, dim3(64 * WN * WK), lds, s,
             (const uint8_t*)w, (const uint16_t*)x, nb, n, m, (uint16_t*)y, vec);
  return hipGetLastError();
}

// Launch shapes for more than 16 rows, each with the time of one round of
// workgroups (at most one per CU) as measured: fixed + per_tile us for each 128
// elements of K.  The smallest tiles spread a small product over the chip (8
// waves share a workgroup's K); larger ones convert a weight for more rows and
// read the activations less often, so they win once the small ones need
// several rounds (9728 x 2560 at 193 rows: <5, 2, 4, 2> 228 workgroups, 31.7 us;
// <7, 1, 4, 2> 304 workgroups in two rounds, 43.4; <2, 2, 1, 8> 50 and more).
struct RowsShape {
  int mt, nt, wn, wk;
  float fixed, per_tile;
};
constexpr RowsShape kRowsShapes[] = {
    {2, 1, 1, 8, 4.6f, 0.11f}, {2, 2, 1, 8, 5.6f, 0.18f}, {3, 1, 1, 8, 5.6f, 0.16f},
    {3, 2, 1, 8, 6.7f, 0.23f}, {4, 1, 1, 8, 7.1f, 0.20f}, {4, 2, 1, 8, 7.8f, 0.28f},
    {2, 2, 2, 4, 3.7f, 0.46f}, {3, 2, 2, 4, 4.7f, 0.56f}, {4, 2, 2, 4, 5.2f, 0.61f},
    {7, 1, 4, 2, 5.0f, 0.94f}, {4, 2, 4, 2, 5.0f, 1.19f}, {5, 2, 4, 2, 5.0f, 1.33f},
    {6, 2, 4, 2, 5.0f, 1.46f}, {7, 2, 4, 2, 5.0f, 1.59f}};
constexpr int kNumRowsShapes = sizeof(kRowsShapes) / sizeof(kRowsShapes[0]);

// Estimated us of a shape: rounds of 256 workgroups (the first shape runs two
// per CU, so its rounds overlap).
float rows_cost(const RowsShape& c, int64_t m, int64_t n, int64_t nb) {
  const int64_t wgs = ((n + 16 * c.nt * c.wn - 1) / (16 * c.nt * c.wn)) *
                      ((m + 16 * c.mt - 1) / (16 * c.mt));
  const float one = c.fixed + c.per_tile * (float)((nb + 3) / 4);
  const float rounds = (float)wgs / 256.0f;
  return one * (c.mt * c.nt == 2 ? (rounds > 1.0f ? rounds : 1.0f) : ceilf(rounds));
}

int rows_pick(int64_t m, int64_t n, int64_t nb, float* cost) {
  int best = 0;
  *cost = rows_cost(kRowsShapes[0], m, n, nb);
  for (int i = 1; i < kNumRowsShapes; ++i) {
    const float c = rows_cost(kRowsShapes[i], m, n, nb);
    if (c < *cost) {
      *cost = c;
      best = i;
    }
  }
  return best;
}

template <int I>
hipError_t launch_shape(int pick, hipStream_t s, const void* x, const void* w, void* y, int m,
                        int n, int nb) {
  if constexpr (I < kNumRowsShapes) {
    constexpr RowsShape c = kRowsShapes[I];
    if (pick == I) return launch_rows<c.mt, c.nt, c.wn, c.wk>(s, x, w, y, m, n, nb);
    return launch_shape<I + 1>(pick, s, x, w, y, m, n, nb);
  }
  return hipErrorInvalidValue;
}

hipError_t rows_dispatch(hipStream_t s, const void* x, const void* w, void* y, int m, int n,
                         int nb) {
  if (m <= 16) return launch_rows<1, 1, 1, 8, true>(s, x, w, y, m, n, nb);
  float cost;
  int pick = rows_pick(m, n, nb, &cost);
  if (const char* e = tuning_env("SMX_ROWS_SHAPE")) {  // tuning sweeps
    const int v = atoi(e);
    if (v >= 0 && v < kNumRowsShapes) pick = v;
  }
  return launch_shape<0>(pick, s, x, w, y, m, n, nb);
}

}  // namespace
}  // namespace smx

#include "smx_abi_util.h"

extern "C" int smx_q4_0_gemm_rows(void* stream, const void* x, const void* w, void* y, int64_t m,
                                  int64_t n, int64_t k) {
  SMX_REQUIRE(x && w && y, "null pointer argument");
  SMX_REQUIRE(n >= 1 && n <= (1ll << 30), "bad output size");
  SMX_REQUIRE(k >= 32 && k % 32 == 0 && k <= (1 << 20), "k must be a multiple of 32 in [32, 2^20]");
  SMX_REQUIRE(m >= 1 && m <= (1 << 20) && m * k < (1ll << 30), "m * k must be below 2^30");
  SMX_REQUIRE((uintptr_t)x % 16 == 0 && (uintptr_t)w % 4 == 0 && (uintptr_t)y % 2 == 0,
              "x must be 16-byte aligned, w 4-byte and y 2-byte aligned");
  return (int)smx::rows_dispatch((hipStream_t)stream, x, w, y, (int)m, (int)n, (int)(k / 32));
}

// 1 where the fused kernel is the faster way to an [m, n] product with bf16
// weight roundings (m > 16), 0 where dequantising the matrix and multiplying
// with a library GEMM is.  That way grows slower with m, as the fused kernel
// pays for the conversion once per row group.  Its estimate is a fit to both
// ways measured at 18 row counts of 61 sizes: a launch and a half, the matrix
// written and read back (dearer once its bf16 form leaves the last-level cache
// at 100 million weights), less for the outputs a short K has many of.  Of the
// 793 sizes it picks the fused kernel for, 5 are slower by it, at most 12 %
// (22016 x 4096 at 128 rows 77.7 us against 69.6; 19456 x 2560 at 128 rows 50.8,
// 48.4); of 244 at 16 sizes it was not fitted to, 6, at most 6 %.  us, fused and
// library:
//   6144 x 2560    48 rows 12.4, 29.9   256 rows 29.2, 40.2   512 rows 37.2, 36.0
//   9728 x 2560    64 rows 18.5, 32.8   193 rows 33.1, 39.5   512 rows 62.9, 47.9
//   19456 x 2560   96 rows 35.1, 46.4   256 rows 67.3, 59.5
//   2560 x 4096   128 rows 14.9, 32.3   320 rows 26.3, 27.7   512 rows 34.8, 29.3
//   20000 x 160    64 rows  8.7, 12.1   256 rows 20.9, 17.3
extern "C" int smx_q4_0_gemm_rows_preferred(int64_t m, int64_t n, int64_t k) {
  if (m < 17 || m > 512 || n < 1 || n > (1ll << 30) || k < 32 || k % 32 != 0 ||
      k > (1 << 20) || m * k >= (1ll << 30))
    return 0;
  float fused;
  smx::rows_pick(m, n, k / 32, &fused);
  const float mw = 1e-6f * (float)n * (float)k, mo = 1e-6f * (float)m * (float)n;
  return fused < 15.2f + 0.86f * fminf(mw, 12.0f) + mw * (0.7f + 0.0003f * (float)m) +
                     0.6f * fmaxf(mw - 100.0f, 0.0f) - 2.2f * mo;
}
