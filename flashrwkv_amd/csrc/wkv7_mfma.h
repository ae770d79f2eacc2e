// MFMA and LDS-tile helpers for the chunked WKV7 kernels (gfx950, wave64).
//
// Every matrix product in the chunked kernels is a sum of 16x16x16 bf16 MFMA
// tiles (v_mfma_f32_16x16x16_bf16, fp32 accumulate). With lane l, g = l / 16
// and n = l % 16 the register layouts are:
//   A operand (4 bf16): A[m = n][k = 4g + e],  e = 0..3
//   B operand (4 bf16): B[k = 4g + e][n]
//   C / D     (4 fp32): C[m = 4g + j][n],      j = 0..3
// so an accumulator tile in C layout is, after conversion to bf16, directly
// the B operand of a product contracting over its rows, and the A operand of
// a product contracting over its columns with its transpose. Kernels chain
// products through registers this way and only stage operands that several
// waves share through LDS.
//
// LDS tiles are 64 x 64 bf16 with a padded row stride of 72 elements
// (144 bytes = 36 banks): the 16 rows an operand read touches start in 16
// distinct bank groups, so 8-byte operand reads are conflict-free within each
// 16-lane group.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace frwkv {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef short i16x4 __attribute__((ext_vector_type(4)));

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

// Buffer resource over [base, base + bytes): loads beyond the range return
// zero and stores beyond it are dropped by the hardware. Descriptor word 3
// for gfx9-family raw buffers.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_rsrc(const void* base,
                                                              uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0,
                                           static_cast<int>(bytes), 0x00020000);
}

constexpr int kTileStride = 72;                  // bf16 elements per LDS row
constexpr int kTileElems = 64 * kTileStride;     // one 64 x 64 tile

typedef short i16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ f32x4 mfma16(i16x4 a, i16x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// v_mfma_f32_16x16x32_bf16: same issue cost as the 16x16x16 form on gfx950
// for twice the work. An accumulator chain must keep one MFMA shape: with
// this toolchain, a 16x16x16 MFMA taking a 16x16x32 result as its
// accumulator a few instructions later produced wrong sums on MI355X (the
// wait states between the two were too few), so single 16-blocks are fed as
// zero-padded 32-wide steps instead. Operand register e of lane (g, n) carries
// k = 4g + e (e < 4) and k = 16 + 4g + (e - 4) (e >= 4) of the 32-wide K
// block: two 16-row blocks in C layout concatenate into one operand, and an
// LDS operand is two 8-byte reads 16 columns apart.
__device__ __forceinline__ f32x4 mfma32(i16x8 a, i16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

__device__ __forceinline__ i16x8 cat(i16x4 lo, i16x4 hi) {
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

__device__ __forceinline__ f32x4 zero4() { return f32x4{0.f, 0.f, 0.f, 0.f}; }

// Round-to-nearest-even fp32 -> bf16 bits.
__device__ __forceinline__ uint16_t to_bf16_bits(float x) {
  __bf16 h = static_cast<__bf16>(x);
  uint16_t bits;
  __builtin_memcpy(&bits, &h, 2);
  return bits;
}

__device__ __forceinline__ float bf16_float(uint16_t bits) {
  return __uint_as_float(static_cast<uint32_t>(bits) << 16);
}

// Two fp32 -> two round-to-nearest-even bf16 in one dword (lo in bits
// 0..15). The vector conversion selects one v_cvt_pk_bf16_f32 with both
// sources; converting the halves one by one costs a conversion per value plus
// the shift/mask/or to pack them.
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  const f32x2 v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

// Two fp32 split into bf16 pairs x = hi + lo: .x packs hi = bf16(x), .y packs
// lo = bf16(x - hi) (x - hi is exact in fp32), leaving a relative error of
// about 2^-17 where bf16 alone leaves 2^-9.
__device__ __forceinline__ uint2 split_bf16x2(float x0, float x1) {
  const uint32_t hi = pack_bf16x2(x0, x1);
  const float h0 = __uint_as_float(hi << 16);
  const float h1 = __uint_as_float(hi & 0xffff0000u);
  return make_uint2(hi, pack_bf16x2(x0 - h0, x1 - h1));
}

// The same in three parts, x = hi + mid + lo exactly (8 bits of the significand
// each), for finite x whose low parts are normal numbers.
__device__ __forceinline__ uint3 split3_bf16x2(float x0, float x1) {
  const uint32_t hi = pack_bf16x2(x0, x1);
  const uint2 rest = split_bf16x2(x0 - __uint_as_float(hi << 16),
                                  x1 - __uint_as_float(hi & 0xffff0000u));
  return make_uint3(hi, rest.x, rest.y);
}

// C-layout accumulator -> bf16 operand registers (two packed conversions;
// a single 4-wide vector conversion is split into per-value conversions plus
// byte permutes when its result feeds an MFMA operand directly).
__device__ __forceinline__ i16x4 to_operand(f32x4 c) {
  const u32x2 q = {pack_bf16x2(c[0], c[1]), pack_bf16x2(c[2], c[3])};
  return __builtin_bit_cast(i16x4, q);
}

// The same as a split pair of operands, c = hi + lo (see split_bf16x2).
__device__ __forceinline__ void to_operand_split(f32x4 c, i16x4& hi, i16x4& lo) {
  const uint2 p01 = split_bf16x2(c[0], c[1]);
  const uint2 p23 = split_bf16x2(c[2], c[3]);
  const u32x2 h = {p01.x, p23.x}, l = {p01.y, p23.y};
  hi = __builtin_bit_cast(i16x4, h);
  lo = __builtin_bit_cast(i16x4, l);
}
__device__ __forceinline__ void to_operand_split3(f32x4 c, i16x4& hi, i16x4& mid, i16x4& lo) {
  const uint3 p01 = split3_bf16x2(c[0], c[1]);
  const uint3 p23 = split3_bf16x2(c[2], c[3]);
  hi = __builtin_bit_cast(i16x4, u32x2{p01.x, p23.x});
  mid = __builtin_bit_cast(i16x4, u32x2{p01.y, p23.y});
  lo = __builtin_bit_cast(i16x4, u32x2{p01.z, p23.z});
}

// Inverses of I - L for a strictly lower 16 x 16 L, as every chunk form needs
// of its diagonal blocks. Registers: X_R "lane (g, n) holds X[n][4g + j]" (A
// operand of X, C layout of X^T) and X_C the C layout of X (B operand of X); a
// product Z = X Y is Z_C = mfma(X_R, Y_C) and Z_R = mfma(Y_C, X_R).
//
// Block substitution: the four 4 x 4 diagonal blocks by substitution in fp32
// (a block's rows lie in one quad of lanes), then twice
//   T <- T + T E T,  E the part of L that joins pairs of inverted blocks
// (E T E = 0, so this is exact). No power of L is formed: the product
// (I + L)(I + L^2)(I + L^4)(I + L^8) has intermediate entries up to
// C(14, 7) = 3432 for the L of repeated keys (every entry near -1) that must
// cancel to the entries of T, near 1, and in bf16 they do not: states were off
// by a factor of 1e10 after 256 tokens of one key, and are 2e-3 off with this
// form; random keys are the same to two digits (3.7e-3).
template <int kLane>
__device__ __forceinline__ float quad_lane(float x) {
  return __int_as_float(
      __builtin_amdgcn_mov_dpp(__float_as_int(x), 0x55 * kLane, 0xf, 0xf, true));
}

// Lane masks that depend on (g, n) alone are constants. The empty asm has them
// written to scalar registers where they are used: hoisted out of a chunk loop,
// as compares or as constants, they spill there (prefill 2 to 3% slower).
template <typename F>
constexpr uint64_t lanes_where(F f) {
  uint64_t mask = 0;
  for (int lane = 0; lane < 64; ++lane) {
    if (f(lane >> 4, lane & 15)) mask |= uint64_t{1} << lane;
  }
  return mask;
}
__device__ __forceinline__ bool in_lanes(uint64_t mask) {
  uint32_t lo = static_cast<uint32_t>(mask), hi = static_cast<uint32_t>(mask >> 32);
  asm volatile("" : "+s"(lo), "+s"(hi));
  return __builtin_amdgcn_inverse_ballot_w64(static_cast<uint64_t>(hi) << 32 | lo);
}
// Strict lower triangle of the 4 x 4 diagonal blocks: element j of a lane of
// X_R (rows i > j) and of X_C (columns i < j), i = n - 4g.
template <int j>
constexpr uint64_t kRowBelow = lanes_where([](int g, int n) {
  return n - 4 * g > j && n - 4 * g < 4;
});
template <int j>
constexpr uint64_t kColumnBelow = lanes_where([](int g, int n) {
  return n - 4 * g >= 0 && n - 4 * g < j;
});
template <int j>
constexpr uint64_t kOnDiagonal = lanes_where([](int g, int n) { return n == 4 * g + j; });
// Lanes of X_C that join 4 x 4 blocks to 8 x 8 ones, and those to 16 x 16.
constexpr uint64_t kJoins8 = lanes_where([](int g, int n) {
  return g % 2 == 1 && n / 4 == g - 1;
});
constexpr uint64_t kJoins16 = lanes_where([](int g, int n) { return g / 2 > n / 8; });

// N with I + N the inverse of the 4 x 4 diagonal blocks, in both layouts, zero
// elsewhere. Of l_r and l_c only the strict lower triangle is read.
__device__ __forceinline__ void invert_diagonal4(f32x4 l_r, f32x4 l_c, f32x4& n_r, f32x4& n_c) {
  // Rows: row i of the block in lane i of the quad, rows before it broadcast.
  n_r = f32x4{in_lanes(kRowBelow<0>) ? l_r[0] : 0.0f, in_lanes(kRowBelow<1>) ? l_r[1] : 0.0f,
              in_lanes(kRowBelow<2>) ? l_r[2] : 0.0f, 0.0f};
  const float c1 = n_r[1], c2 = n_r[2];
  n_r[0] += c1 * quad_lane<1>(n_r[0]);
  const float r0 = quad_lane<2>(n_r[0]), r1 = quad_lane<2>(n_r[1]);
  n_r[0] += c2 * r0;
  n_r[1] += c2 * r1;
  // Columns: column c in lane c, L's further columns broadcast.
  n_c = f32x4{0.0f, in_lanes(kColumnBelow<1>) ? l_c[1] : 0.0f,
              in_lanes(kColumnBelow<2>) ? l_c[2] : 0.0f,
              in_lanes(kColumnBelow<3>) ? l_c[3] : 0.0f};
  const float l2 = n_c[2], l3 = n_c[3];
  n_c[2] += quad_lane<1>(l2) * n_c[1];
  n_c[3] += quad_lane<1>(l3) * n_c[1];
  n_c[3] += quad_lane<2>(l3) * n_c[2];
}

// T_R of (I - L)^{-1} with bf16 operands (see above), by T <- (I + T E) T: five
// matrix products, four of them in a chain. The identity goes into operands
// whose diagonal is zero; of l_r and l_c only the strict lower triangle is read.
__device__ __forceinline__ f32x4 invert_unit_lower(f32x4 l_r, f32x4 l_c) {
  f32x4 n_r, n_c;
  invert_diagonal4(l_r, l_c, n_r, n_c);
  const u32x2 one = {
      (in_lanes(kOnDiagonal<0>) ? 0x3f80u : 0u) | (in_lanes(kOnDiagonal<1>) ? 0x3f800000u : 0u),
      (in_lanes(kOnDiagonal<2>) ? 0x3f80u : 0u) | (in_lanes(kOnDiagonal<3>) ? 0x3f800000u : 0u)};
  auto plus_one = [&](f32x4 x) {
    return __builtin_bit_cast(i16x4, __builtin_bit_cast(u32x2, to_operand(x)) | one);
  };
  const i16x4 zero = {0, 0, 0, 0};
  const i16x4 l = to_operand(l_c), t4_r = plus_one(n_r), t4_c = plus_one(n_c);
  const i16x4 x = plus_one(mfma16(in_lanes(kJoins8) ? l : zero, t4_r, zero4()));
  const f32x4 t8_r = mfma16(t4_c, x, zero4()), t8_c = mfma16(x, t4_c, zero4());
  const i16x4 y = plus_one(mfma16(in_lanes(kJoins16) ? l : zero, to_operand(t8_r), zero4()));
  return mfma16(to_operand(t8_c), y, zero4());
}

// Operand read from an LDS tile: 4 consecutive bf16 of row `row` starting at
// column `col` (8-byte aligned). Serves as A operand (row = m, col = k0) or
// as B operand of a tile stored [n][k] (row = n, col = k0).
template <int Stride = kTileStride>
__device__ __forceinline__ i16x4 lds_operand(const uint16_t* tile, int row, int col) {
  return *reinterpret_cast<const i16x4*>(tile + row * Stride + col);
}

// 32-wide K operand from an LDS tile: columns col + 4g .. +3 and
// col + 16 + 4g .. +3 of row `row` (lane group g), matching mfma32's K order.
template <int Stride = kTileStride>
__device__ __forceinline__ i16x8 lds_operand32(const uint16_t* tile, int row, int col, int g) {
  return cat(lds_operand<Stride>(tile, row, col + 4 * g),
             lds_operand<Stride>(tile, row, col + 16 + 4 * g));
}

// B operand over tokens from a row-major [t][col] LDS tile via the gfx950
// transpose read (ds_read_b64_tr_b16): lane (g, n) receives
// X[t0 + 4g + e][c0 + n], e = 0..3, i.e. the MFMA operand layout for
// K = tokens t0 .. t0 + 15. Within a 16-lane group, lane i's element e
// comes from the 8 bytes addressed by lane 4e + i / 4, element i % 4, so
// lane j addresses row t0 + 4g + j / 4, columns c0 + 4 (j % 4) .. +3. The
// row stride (elements) must keep those addresses 8-byte aligned.
template <int Stride>
__device__ __forceinline__ i16x4 lds_operand_tr(const uint16_t* tile, int t0, int c0, int g,
                                                int n) {
  typedef short v4i16 __attribute__((ext_vector_type(4)));
  static_assert((Stride * 2) % 8 == 0, "rows must be 8-byte aligned");
  const uint16_t* src = tile + (t0 + 4 * g + (n >> 2)) * Stride + c0 + 4 * (n & 3);
  const v4i16 x = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) v4i16*)(src));
  i16x4 r;
  r[0] = x[0];
  r[1] = x[1];
  r[2] = x[2];
  r[3] = x[3];
  return r;
}

// Stores a C-layout tile transposed: lane (g, n) writes its 4 values to
// dst[n][4g .. 4g+3] of a tile with the given row stride (one 8-byte write).
__device__ __forceinline__ void lds_store_transposed(uint16_t* dst, int stride,
                                                     int g, int n, f32x4 c) {
  uint2 q;
  q.x = pack_bf16x2(c[0], c[1]);
  q.y = pack_bf16x2(c[2], c[3]);
  *reinterpret_cast<uint2*>(dst + n * stride + 4 * g) = q;
}

// lds_store_transposed of the split pair c = hi + lo into two tiles.
__device__ __forceinline__ void lds_store_transposed_split(uint16_t* dst_hi, uint16_t* dst_lo,
                                                           int stride, int g, int n, f32x4 c) {
  const uint2 p01 = split_bf16x2(c[0], c[1]);
  const uint2 p23 = split_bf16x2(c[2], c[3]);
  *reinterpret_cast<uint2*>(dst_hi + n * stride + 4 * g) = make_uint2(p01.x, p23.x);
  *reinterpret_cast<uint2*>(dst_lo + n * stride + 4 * g) = make_uint2(p01.y, p23.y);
}

}  // namespace frwkv
