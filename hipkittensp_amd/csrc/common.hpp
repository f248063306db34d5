// Shared device/host helpers for the MXFP6 GEMM kernels (gfx950 only).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mxfp6 {

typedef int v12i __attribute__((ext_vector_type(12)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

#define MXFP6_LDS __attribute__((address_space(3)))

// Output element traits: the kernels are instantiated for bf16 (the operator) and float (the
// unrounded accumulators, used to state the accuracy contract before the bf16 rounding).
struct OutBf16 { typedef uint16_t type; };
struct OutF32 { typedef float type; };
struct OutFp6 { typedef uint8_t type; };  // C re-quantised to MXFP6: packed [M, 3N/4] + E8M0 [M, N/32]

// E8M0 byte of a 32-block with largest magnitude amax (floor(log2(amax)) - emax, clamped; 0 for an all-zero block)
__device__ __forceinline__ int e8m0_of_amax(float amax, int emax) {
  if (!(amax > 0.f)) return 0;
  const uint32_t u = __float_as_uint(amax);
  const int be = (int)(u >> 23);
  const int fl = be ? be - 127 : (31 - __clz((int)u)) - 149;  // fp32 subnormals included
  const int sb = fl - emax + 127;
  return sb < 0 ? 0 : (sb > 254 ? 254 : sb);
}

// A 32-block of bf16 (64 bytes) quantised to FMT: six dwords and its E8M0 byte.  The instruction divides by the power of two and
// rounds (nearest even, saturating).
// The conversions read their sources over several passes and write the result meanwhile: registers that the two share come out
// wrong (v[0:5] from v[18:33], v[2:17]: the third dword on).  The compiler does not know, so every source is kept in use until
// behind the instruction.
typedef uint32_t u32x6 __attribute__((ext_vector_type(6)));
template <int FMT>
__device__ __forceinline__ u32x6 quantise_block_bf16(const v4i (&x)[4], int& sb) {
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) {
      amax = fmaxf(amax, fabsf(__int_as_float(x[i][j] << 16)));
      amax = fmaxf(amax, fabsf(__int_as_float(x[i][j] & (int)0xffff0000)));
    }
  sb = e8m0_of_amax(amax, FMT == 2 ? 2 : 4);
  const float scale = __uint_as_float((uint32_t)sb << 23);  // 2^(sb - 127); the instruction uses the exponent field
  typedef __bf16 v32bf __attribute__((ext_vector_type(32)));
  typedef int v16i __attribute__((ext_vector_type(16)));
  v16i raw;
#pragma unroll
  for (int i = 0; i < 16; i++) raw[i] = x[i / 4][i & 3];
  const v32bf xb = __builtin_bit_cast(v32bf, raw);
  u32x6 w;
  if constexpr (FMT == 2) w = __builtin_amdgcn_cvt_scalef32_pk32_fp6_bf16(xb, scale);
  else w = __builtin_amdgcn_cvt_scalef32_pk32_bf6_bf16(xb, scale);
  asm volatile("" : "+v"(w) : "v"(raw), "v"(scale));
  return w;
}

// The same for a 32-block of fp32 (128 bytes)
template <int FMT>
__device__ __forceinline__ u32x6 quantise_block_f32(const v4i (&x)[8], int& sb) {
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < 8; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) amax = fmaxf(amax, fabsf(__int_as_float(x[i][j])));
  sb = e8m0_of_amax(amax, FMT == 2 ? 2 : 4);
  const float scale = __uint_as_float((uint32_t)sb << 23);  // 2^(sb - 127); the instruction uses the exponent field
  v16f ev, od;
#pragma unroll
  for (int i = 0; i < 16; i++) ev[i] = __int_as_float(x[i / 2][(2 * i) & 3]), od[i] = __int_as_float(x[i / 2][(2 * i + 1) & 3]);
  u32x6 w;
  if constexpr (FMT == 2) w = __builtin_amdgcn_cvt_scalef32_2xpk16_fp6_f32(ev, od, scale);
  else w = __builtin_amdgcn_cvt_scalef32_2xpk16_bf6_f32(ev, od, scale);
  asm volatile("" : "+v"(w) : "v"(ev), "v"(od), "v"(scale));
  return w;
}

// The same for a 32-block of fp32 as two lanes of an MFMA tile hold it: column 8 (k / 4) + k % 4 of the block in p0[k], that + 4 in
// p1[k].  fmt (2 or 3) is uniform.
__device__ __forceinline__ u32x6 quantise_block_acc(const float (&p0)[16], const float (&p1)[16], int fmt, int& sb) {
  float amax = 0.f;
#pragma unroll
  for (int k = 0; k < 16; k++) amax = fmaxf(amax, fmaxf(fabsf(p0[k]), fabsf(p1[k])));
  sb = e8m0_of_amax(amax, fmt == 2 ? 2 : 4);
  const float scale = __uint_as_float((uint32_t)sb << 23);
  v16f ev, od;  // even and odd columns: column n = 8 q + r is p0[4 q + r] for r < 4, p1[4 q + r - 4] otherwise
#pragma unroll
  for (int t = 0; t < 16; t++) {
    const int ne = 2 * t, no = 2 * t + 1;
    ev[t] = (ne & 4) ? p1[4 * (ne >> 3) + (ne & 3)] : p0[4 * (ne >> 3) + (ne & 3)];
    od[t] = (no & 4) ? p1[4 * (no >> 3) + (no & 3)] : p0[4 * (no >> 3) + (no & 3)];
  }
  u32x6 w;
  if (fmt == 2) {
    w = __builtin_amdgcn_cvt_scalef32_2xpk16_fp6_f32(ev, od, scale);
    asm volatile("" : "+v"(w) : "v"(ev), "v"(od), "v"(scale));
  } else {
    w = __builtin_amdgcn_cvt_scalef32_2xpk16_bf6_f32(ev, od, scale);
    asm volatile("" : "+v"(w) : "v"(ev), "v"(od), "v"(scale));
  }
  return w;
}

// Two 32 x 32 accumulator tiles side by side (a band of 32 rows), re-quantised along N and stored as blocks blk0 and blk0 + 1 of
// row m of an fp6 operand with nkb blocks a row.  A 32-block of row m is the 16 values of lane (m, h = 0) and the 16 of lane
// (m, h = 1) of one tile.  The two tiles are traded with v_permlane32_swap, register by register, after which the lower lane holds
// all of the first block and the upper lane all of the second: then exactly the quantiser, 24 bytes and a scale byte per lane.
__device__ __forceinline__ void store_fp6_band(const v16f& c0, const v16f& c1, int fmt, uint8_t* packed, uint8_t* scales, long m, int M, int blk0, int nkb) {
  float p0[16], p1[16];
#pragma unroll
  for (int k = 0; k < 16; k++) {
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(c0[k]), __float_as_uint(c1[k]), false, false);
    p0[k] = __uint_as_float(sw[0]), p1[k] = __uint_as_float(sw[1]);
  }
  int sb;
  const u32x6 w = quantise_block_acc(p0, p1, fmt, sb);
  const int blk = blk0 + ((threadIdx.x >> 5) & 1);
  if (m < M && blk < nkb) {
    u32x2* dst = reinterpret_cast<u32x2*>(packed + (m * nkb + blk) * 24);
#pragma unroll
    for (int c = 0; c < 3; c++) dst[c] = u32x2{w[2 * c], w[2 * c + 1]};
    scales[m * nkb + blk] = (uint8_t)sb;
  }
}

// fp32 -> bf16, round to nearest even (v_cvt_pk_bf16_f32 on gfx950).
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
  typedef float f2 __attribute__((ext_vector_type(2)));
  f2 v = {lo, hi};
  bf2 r = __builtin_convertvector(v, bf2);
  return __builtin_bit_cast(uint32_t, r);
}

// Store 4 consecutive outputs (n .. n+3) of one row.
__device__ __forceinline__ void store4(uint16_t* p, float a, float b, float c, float d) {
  u32x2 v = {pack_bf16x2(a, b), pack_bf16x2(c, d)};
  *reinterpret_cast<u32x2*>(p) = v;
}
__device__ __forceinline__ void store4(float* p, float a, float b, float c, float d) {
  v4f v = {a, b, c, d};
  *reinterpret_cast<v4f*>(p) = v;
}
__device__ __forceinline__ void store1(uint16_t* p, float a) { *p = (uint16_t)(pack_bf16x2(a, 0.f) & 0xffffu); }
__device__ __forceinline__ void store1(float* p, float a) { *p = a; }

// Whole lines for the stores of an MFMA tile.  A lane holds 16 bytes of row l % 32 in each register, the upper half of the wave the 16
// bytes behind the lower half's: a store of them touches 32 rows, 32 bytes each, and a line is whole after four stores.  The L2s put that
// together, but keep all of it until the write-back at the end of the kernel, which nothing runs beside; sent out early, in parts, it
// takes longer still.  With whole lines, sent out at once (store_c), C leaves under the rest of the kernel: us, before / after, tiled 256 x 256
// and block kernel, tile-major operands: 8192 x 2048 x 512 17.1 / 12.2, 19.6 / 13.7; 1024 x 23552 x 512 26.2 / 22.2, 27.6 / 22.5; 6255 x 1920 x 1536
// 24.3 / 21.5, 28.0 / 24.9; 4530 x 7936 x 2048 71.7 / 67.3, 78.5 / 75.0; 8192^3 287 / 280 (tiled).  (The same non-temporal in parts of 32 bytes: 19.7, 36.2;
// 34.7, 56.6; 27.2, 35.7; 91, 95; 307; in parts of 64: 16.0, 16.1; 25.8, 26.2; 21.4, 25.1; 70, 78; 297.  Whole lines without it: 16.6, 19.0; 25.8, 27.2; 24.3,
// 27.1; 71.1, 76.3; 284.)
// Little C is stored as it comes: the lanes' trades and the way to memory cost such a call more than they give (block_c_form, ragged_c_form; of the time as it
// comes, whole lines non-temporally on the block kernel, by C's size below 1 MB, 1 to 2, 2 to 4 MB: rows on lines 1.01, 1.00, 0.98, others 1.07, 1.03, 1.02).
// A program whose next kernel reads C keeps most of the gain (us, in pieces / as it is now, the quantiser or an elementwise add behind the kernel that the choice
// takes): 512 x 2048 x 2048 12.6 / 12.6, 11.8 / 11.8; 1024 x 4096 x 1024 12.9 / 11.7, 12.4 / 11.6; 2048 x 4096 x 1024 17.5 / 15.6, 18.5 / 17.2; 4096 x 4096 x 2048
// 35.2 / 33.2, 37.9 / 37.7; tiled 256 x 256, 2048 x 14336 x 1024 45.5 / 43.2, 50.6 / 51.7, 4096 x 14336 x 1024 87.1 / 81.0, 97.4 / 97.1.
// How a tile kernel stores C: 16 bytes of 32 rows at a time, as the accumulators hold them; whole lines, through the L2s; whole lines, non-temporally
enum CStore : int { kCPieces, kCKept, kCOut };
// pair_rows: y holds what lies 32 bytes behind x's.  Afterwards x holds 64 contiguous bytes of rows 0 - 15 and y those of rows 16 - 31:
// row l % 16, 16-byte piece 2 (l / 16 % 2) + l / 32 of the four.
__device__ __forceinline__ void pair_rows(v4i& x, v4i& y) {
#pragma unroll
  for (int c = 0; c < 4; c++) {
    const auto sw = __builtin_amdgcn_permlane16_swap(x[c], y[c], false, false);
    x[c] = sw[0], y[c] = sw[1];
  }
}
// join_lines: x and y as pair_rows leaves them (the same 16 rows), y's bytes 64 behind x's.  Afterwards x holds 128 contiguous bytes of rows 0
// - 7 and y those of rows 8 - 15: row l % 8, half l / 8 % 2, piece as before.
__device__ __forceinline__ void join_lines(v4i& x, v4i& y) {
#pragma unroll
  for (int c = 0; c < 4; c++) {
    constexpr int kRowRor8 = 0x128;
    const int lower = __builtin_amdgcn_update_dpp(x[c], y[c], kRowRor8, 0xf, 0xc, false);
    y[c] = __builtin_amdgcn_update_dpp(y[c], x[c], kRowRor8, 0xf, 0x3, false);
    x[c] = lower;
  }
}
// A lane's place in what pair_rows leaves (LINE 0) or join_lines (LINE 1): its row, and the 16-byte pieces in front of its own in the row
template <int LINE>
__device__ __forceinline__ int line_row(int lane) { return lane & (LINE ? 7 : 15); }
template <int LINE>
__device__ __forceinline__ int line_piece(int lane) { return (LINE ? lane >> 1 & 4 : 0) + (lane >> 3 & 2) + (lane >> 5); }

// Stores 16 bytes per lane, non-temporal: lines that are whole go out to memory at once, under the rest of the kernel, and do not wait in the
// L2s for the write-back at its end.  STREAM false: the same through the L2s.
// The registers stay as they are for four more cycles: a store of 16 bytes reads its data a little after it has been issued.  Where it has a scalar
// offset, as half of these have, the compiler lets the next instruction write them (the instruction set's table of required waits excepts such
// stores), and here a v_mov of the first dword right behind one changed what the last four of every sixteen lanes stored, now and then.  Where it has none --
// the 16-byte stores through a pointer, in every kernel -- the compiler leaves two cycles, which is the table's wait, and no such store was seen to go
// wrong.  A test disassembles the library for both distances.
template <bool STREAM>
__device__ __forceinline__ void store_c(v4i v, const __amdgpu_buffer_rsrc_t& rsrc, int voff, int soff) {
  constexpr int kNonTemporal = 2;
  __builtin_amdgcn_raw_buffer_store_b128(v, rsrc, voff, soff, STREAM ? kNonTemporal : 0);
  asm volatile("s_nop 3" ::"v"(v) : "memory");
}
// Whether C in whole lines, `rows` rows of `row` bytes, leaves non-temporally: where its rows start on lines, and up to 16 MB.  Rows that start inside a
// line leave every line to two stores, and of a large C the L2s send out the first part before the second has come.  Through the L2s / non-temporally,
// of the time in pieces, over 110 drawn shapes with such rows, block kernel: bf16 4 to 12 MB 0.99 / 0.97, 16 to 24 MB 0.98 / 1.02, above 0.98 / 1.02 (up to 1.3);
// fp32 1.01 / 0.98, 0.99 / 1.03, above 0.97 / 1.27 (up to 1.9).
constexpr size_t kLeavingPartLines = (size_t)16 << 20;
__host__ __device__ inline bool c_leaves(const void* C, int rows, size_t row) { return (((uintptr_t)C | row) & 127) == 0 || rows * row <= kLeavingPartLines; }

// Optional work fused into every kernel's epilogue, in fp32 before the output rounding:
//   y = act(acc * row_scale[m] * col_scale[n] + bias[n])        (each factor / term only if its pointer is set)
// act: 0 none, 1 relu, 2 gelu (erf form), 3 silu.  bias is float or bf16 (bias_bf16).
struct Epilogue {
  const void* bias = nullptr;
  const float* row_scale = nullptr;
  const float* col_scale = nullptr;
  int bias_bf16 = 0;
  int act = 0;
};
__host__ __device__ __forceinline__ bool epilogue_any(const Epilogue& e) { return e.bias || e.row_scale || e.col_scale || e.act; }
__device__ __forceinline__ float bf16_bits_to_f32(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }
// The activations in a handful of instructions each (they are unrolled over every accumulator of a tile, and their VALU time is
// what the tile kernels' epilogues wait for): silu with the hardware exp2 / reciprocal (~1e-6 relative); gelu as y Phi(y), Phi(-|y|) = erfc(|y| /
// sqrt 2) / 2 = exp2(P(|y|)), P of degree 8 fitted to the logarithm with Phi as the weight on [0, 7] (from there on it falls without end, so that
// Phi is zero).  Against 64 bits, y from -12 to 12: 4.0e-7 at most, 3.9e-8 rms, and 2.6e-6 of the value down to y = -3; erf by Abramowitz & Stegun 7.1.26
// with a reciprocal more, as this was before: 4.7e-7, 7.2e-8, 6.2e-5, and 22 VALU cycles for every lane of an output where this takes 16 (us, with
// gelu, before / after: 8192 x 5120 x 1408 78.2 / 73.0, with MXFP6 output 77.6 / 71.8, 4530 x 7936 x 2048 with MXFP6 output 86.2 / 78.7, 2048 x 14336 x 4096
// 103.5 / 99.1).
__device__ __forceinline__ float act_relu(float y) { return y > 0.f ? y : 0.f; }
__device__ __forceinline__ float act_silu(float y) { return y * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-1.4426950408889634f * y)); }
__device__ __forceinline__ float act_gelu(float y) {
  const float a = fabsf(y);
  float p = -2.77202492e-06f;
  p = fmaf(p, a, 3.86205185e-05f);
  p = fmaf(p, a, -1.82546781e-04f);
  p = fmaf(p, a, -1.45871528e-04f);
  p = fmaf(p, a, 7.07547287e-03f);
  p = fmaf(p, a, -5.25050290e-02f);
  p = fmaf(p, a, -4.59204907e-01f);
  p = fmaf(p, a, -1.15110572e+00f);
  p = fmaf(p, a, -9.99999978e-01f);
  const float tail = __builtin_amdgcn_exp2f(p);  // Phi(-|y|)
  return y * (y >= 0.f ? 1.f - tail : tail);
}
__device__ __forceinline__ float epilogue_act(float y, int act) {
  if (act == 1) return act_relu(y);
  if (act == 2) return act_gelu(y);
  if (act == 3) return act_silu(y);
  return y;
}
// one element; m < M and n < N are the caller's business
__device__ __forceinline__ float epilogue_apply(const Epilogue& e, float v, long m, long n) {
  if (e.row_scale) v *= e.row_scale[m];
  if (e.col_scale) v *= e.col_scale[n];
  if (e.bias) v += e.bias_bf16 ? bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(e.bias)[n]) : reinterpret_cast<const float*>(e.bias)[n];
  return epilogue_act(v, e.act);
}

// Raw buffer resource over [base, base + bytes): out-of-range lanes of a buffer load read 0.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
}

// D(32x32, fp32) += SA(32 x 64) . SB(32 x 64)^T with per-lane E8M0 block scales.
//   lane l supplies row l%32, K-block l/32 (32 fp6 values = 6 dwords) of each source;
//   result register v of lane l is D[8*(v/4) + 4*(l/32) + v%4][l%32]   (row from SA, column from SB).
//   OPA/OPB select which byte of the scale dword is used.
template <int FMT_SA, int FMT_SB, int OPA, int OPB>
__device__ __forceinline__ v16f mfma_fp6(v8i sa, v8i sb, v16f acc, int scale_sa, int scale_sb) {
  return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(sa, sb, acc, FMT_SA, FMT_SB, OPA, scale_sa, OPB, scale_sb);
}

// Workgroup -> output tile of the LDS-tiled kernels.  Workgroup `bid` of a launch works on tiles bid, bid + grid, ... of a
// logical order in which the round-robin placement of workgroups on the 8 XCDs (workgroup b runs on XCD b % 8) is
// undone, so that each XCD gets a contiguous run of logical tiles (xcd_remap; the idea of chiplet_transform_chunked,
// include/common/util.cuh:78-101, as an exact bijection for any tile count), and the raster walks group_m tile rows at a
// time down the columns (analysis/bf16_gemm/mi325x/kernel_8192.cpp:45-61): the tiles an XCD works on at once share
// operand rows in its L2.  Returns pm | pn << 16, or -1 past the last tile.
__host__ __device__ __forceinline__ int tile_order(int bid, int tiles_m, int tiles_n, int group_m, int xcd_remap) {
  const int nb = tiles_m * tiles_n;
  if (bid >= nb) return -1;
  int L = bid;
  if (xcd_remap) {
    const int xcd = bid & 7, idx = bid >> 3;
    const int per = nb >> 3, rem = nb & 7;
    L = (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + idx;
  }
  const int width = group_m * tiles_n, group = L / width, first = group * group_m;
  const int gsz = tiles_m - first < group_m ? tiles_m - first : group_m, in = L - group * width;
  return (first + in % gsz) | (in / gsz) << 16;
}

// K split between workgroups: position of workgroup `bid` (of `total` = tiles x shares) in share-major order, share s of
// tile i at s * tiles + i.  The hardware deals workgroups to the eight XCDs round-robin; this hands XCD x the x-th
// eighth of that order, so that with eight shares or more an XCD's workgroups all work on the same K range: they pull
// that eighth of A and of B through the XCD's L2 once, where tile-by-tile order has every XCD fetch all of A for its
// tiles (256 x 8192 x 28672, eight shares: 263 MB of L2 misses for 189 MB of operands; A alone is 5.5 MB against 4 MB
// of L2).  With fewer shares an XCD gets part of one share's tiles, the same volume as before.  A bijection on
// [0, total) when total % 8 == 0; the identity otherwise, with the remap switched off (xcd_remap 0) or with xcd_remap 2
// (measurement: tile-by-tile order, XCDs dealt by tile_order).
__host__ __device__ __forceinline__ bool ksplit_by_share(int total, int xcd_remap) { return xcd_remap == 1 && (total & 7) == 0; }
__host__ __device__ __forceinline__ int ksplit_order(int bid, int total, int xcd_remap) {
  return ksplit_by_share(total, xcd_remap) ? (bid & 7) * (total >> 3) + (bid >> 3) : bid;
}

// Floats per row of the partial matrices that a K split of a ragged product leaves (rows of whole, aligned 16 bytes)
__host__ __device__ __forceinline__ size_t ragged_pitch(int n) { return ((size_t)n + 3) & ~(size_t)3; }

// Byte offset of the partial sums that share `share` of a K split leaves for band `band` (32 rows) and column tile `ct` (32
// columns) of C: 4 KB in the order of the MFMA's accumulators, quad q of lane l (row l % 32, columns 8 q + 4 (l / 32) .. + 3)
// at 1024 q + 16 l, so that every store of the GEMM kernel and every load of the reduction is one contiguous KiB.  (Shares as
// row-major matrices, where a store touches 32 rows, 32 bytes each: 1 - 4 us more per call; 256 x 8192 x 28672, eight shares,
// 72.8 against 71.2 us, 512 x 4096 x 14336, four shares, 42.5 against 41.0.)
__host__ __device__ __forceinline__ size_t partial_offset(int share, int band, int ct, int M, int N) {
  const size_t bands = ((size_t)M + 31) / 32, cts = ((size_t)N + 31) / 32;
  return (((size_t)share * bands + band) * cts + ct) * 4096;
}

// Byte offset, inside a tile-major operand, of byte `b` (0 .. 3K/4) of row `row`; nkt = K / 128.
// Tiles are 32 rows x 96 bytes in the kernels' LDS image order (16-byte pieces, pairs swapped in
// rows with bit 3 set).
__host__ __device__ __forceinline__ size_t tile_major_offset(int row, int b, int nkt) {
  const int kt = b / 96, in = b - kt * 96, c = in >> 4, r = row & 31;
  return ((size_t)(row >> 5) * nkt + kt) * 3072 + (size_t)((r * 6 + (c ^ ((r >> 3) & 1))) * 16 + (in & 15));
}

// Byte offset, inside tile-major scales, of the E8M0 byte of K-block kb (32 elements) of row `row`; nk4 =
// ceil(K / 512).  The 16 scale bytes one row has for four K-tiles stay together, and the 32 rows of a row-tile
// are adjacent: 512-byte chunk (rt, g) at ((rt * nk4) + g) * 512, row r of the tile at r * 16 inside it.
__host__ __device__ __forceinline__ size_t tile_major_scale_offset(int row, int kb, int nk4) {
  return ((size_t)(row >> 5) * nk4 + (kb >> 4)) * 512 + (size_t)((row & 31) * 16 + (kb & 15));
}

}  // namespace mxfp6
