// fp32 -> MXFP6 quantise + pack on the GPU, the tile-major re-layout copies, and the zero fill used for K == 0.
// HBM-bound elementwise work: 4 B/element read, 0.78 B/element written.
#include "common.hpp"
#include "kernels.hpp"
#include "loader.hpp"

namespace mxfp6 {

// Quantiser.  One lane handles one 32-element block (128 bytes in, 24 bytes + 1 scale byte out), but the memory
// system wants consecutive lanes on consecutive bytes: a wave fetches 64 blocks (8 KB, contiguous) with eight
// direct-to-LDS loads of 16 bytes per lane into a private buffer and every lane reads its own block back.  The
// buffer is an image of memory with the eight 16-byte pieces of block b rotated: piece c lives in slot
// b * 8 + (c ^ (b & 7)), chosen by which global bytes each lane fetches (a direct load writes lane l at 16 l), so
// that the 16 lanes of a ds_read_b128 phase spread over all banks.  The conversion itself is the hardware's:
// v_cvt_scalef32_2xpk16_{fp6,bf6}_f32 divides 32 floats by a power of two and rounds them to e2m3 / e3m2 (nearest
// even, saturating, NaN -> largest magnitude, fp32 subnormals -> 0); its result interleaves its two sources,
// so they are the even and the odd elements of the block.  (With the rounding done by integer arithmetic, ~25
// instructions per element, the kernel was ALU-bound at 4.4 TB/s.)
// Row-major output: a wave's 64 blocks are consecutive (1536 contiguous output bytes).  Tile-major output: they are
// 16 rows x one K-tile (512 input bytes per row, four whole lines), which is half of a 3 KB output tile and again
// 1536 contiguous bytes.  The 1536 bytes are put together in the wave's buffer (a block's 24 bytes are three 8-byte writes:
// an aligned 8-byte run never straddles the 16-byte pieces the tile-major order permutes) and leave as 16 bytes per lane, whole
// lines in one and a half store instructions instead of three that touch every line three times.
// What bounds it is memory: 8192 x 28672 fp32 (940 MB in, 183 MB out) took 224 us (5.0 TB/s; a copy reaches 4.8, a
// read-only stream 6.05) with five workgroups per CU that each took many chunks in turn, the next one's loads under the
// stores; one chunk per wave and as many workgroups as that takes, so that the CUs' scheduler fills every gap: 214; past the last-level
// cache the input read and the output written with the non-temporal bit: 185 (6.1 TB/s; each alone 196 and 205).
// The input only from the size of that cache on: below it the bit gains nothing on an input from memory and loses where the program has
// just written it (us, plain / non-temporal, an input from memory: 128 MB of fp32 28.1 / 28.1, 192 MB 40.4 / 40.4, 256 MB 55.1 / 52.5, 128 MB of
// bf16 30.2 / 31.9; one in the cache 24.3 / 27.0, 35.1 / 40.4, 54.6 / 52.5, 28.9 / 31.9).
constexpr size_t kCacheBytes = (size_t)256 << 20;  // last-level cache
// Up to so many chunks, workgroups of one wave: four on one compute unit share its way to memory while other units have none.  us, four
// waves / one, replayed back to back: 23 x 14336 of bf16 (161 chunks) 2.56 / 2.40, 64 x 4096 2.51 / 2.39, 512 x 4096 (1024) 2.81 / 2.69, 64 x 4096 of
// fp32 2.80 / 2.52; at twice as many chunks level (1024 x 4096 3.30 / 3.31).
constexpr long kQFewChunks = 1024;
constexpr int kQWaves = 4;  // waves per workgroup; a wave fetches 64 blocks at a time (8 KB of fp32, 4 KB of bf16)


// In: float, or uint16_t for bf16 (the same values after the exact widening: the bf16 instruction
// v_cvt_scalef32_pk32_{fp6,bf6}_bf16 was checked against the fp32 one on 1 M values per format, no difference).
template <int FMT, typename In, int W>
__global__ __launch_bounds__(W * 64) void quantize_kernel(const In* __restrict__ X, uint8_t* __restrict__ packed,
                                                              uint8_t* __restrict__ scales, long nblocks, int nkb, int layout, int rows, int stream_in, int stream_out) {
  constexpr int BB = 32 * (int)sizeof(In), P = BB / 16;  // bytes and 16-byte pieces of a block
  constexpr int kChunk = 64 * BB, NLD = kChunk / 1024;   // bytes and direct loads of a chunk
  __shared__ __attribute__((aligned(1024))) uint8_t smem[W * kChunk];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t buf = (uint32_t)(uintptr_t)(MXFP6_LDS uint8_t*)smem + wave * kChunk;
  const int nkt = (nkb + 3) / 4;  // tile-major only: K-tiles per row (the last one padded with zeros)
  const long nchunks = layout ? (long)((rows + 15) / 16) * nkt : (nblocks + 63) / 64;
  const long stride = (long)gridDim.x * W;
  long chunk = (long)blockIdx.x * W + wave;

  // slot s = q * 64 + lane of load q holds piece (s % P) ^ (b % P) of the chunk's block b = s / P; tile-major:
  // block b is K-block b % 4 of row b / 4 of the chunk
  int voff[NLD];
#pragma unroll
  for (int q = 0; q < NLD; q++) {
    const int sl = q * 64 + lane, b = sl / P, c = (sl % P) ^ (b % P);
    voff[q] = layout ? (b >> 2) * (nkb * BB) + (b & 3) * BB + c * 16 : (b * P + c) * 16;
  }
  auto fetch = [&](long ch) __attribute__((always_inline)) {
    // the resource covers this chunk only (the whole input may exceed 4 GB); bytes past the end read as zero
    const uint8_t* base;
    uint32_t len;
    if (layout) {
      const long g16 = ch / nkt, kt = ch - g16 * nkt;
      base = reinterpret_cast<const uint8_t*>(X) + (g16 * 16 * nkb + kt * 4) * BB;
      len = (uint32_t)((min(16, rows - (int)g16 * 16) - 1) * nkb * BB + min(4, nkb - (int)kt * 4) * BB);  // rows past the last read as zeros
    } else {
      const long left = nblocks * BB - ch * kChunk;
      base = reinterpret_cast<const uint8_t*>(X) + ch * kChunk;
      len = (uint32_t)(left < kChunk ? left : kChunk);
    }
    const __amdgpu_buffer_rsrc_t r = make_rsrc(base, len);
    if (stream_in) {
#pragma unroll
      for (int q = 0; q < NLD; q++) dma16_nt(r, buf + q * 1024, voff[q], 0);
    } else {
#pragma unroll
      for (int q = 0; q < NLD; q++) dma16(r, buf + q * 1024, voff[q], 0);
    }
  };
  for (; chunk < nchunks; chunk += stride) {  // once, unless the chunks outnumber the largest grid
    fetch(chunk);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    v4i x[P];
#pragma unroll
    for (int c = 0; c < P; c++) x[c] = *reinterpret_cast<const v4i*>(smem + wave * kChunk + lane * BB + ((c ^ (lane % P)) * 16));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (layout && (nkb & 3) && (int)(chunk % nkt) * 4 + (lane & 3) >= nkb) {  // K-blocks past K
#pragma unroll
      for (int c = 0; c < P; c++) x[c] = v4i{0, 0, 0, 0};
    }

    int sb;
    u32x6 w;
    if constexpr (sizeof(In) == 4) w = quantise_block_f32<FMT>(x, sb);
    else w = quantise_block_bf16<FMT>(x, sb);
    // the chunk's 1536 output bytes in order, in the buffer its input has left
    uint8_t* const image = smem + wave * kChunk;
    const long g16 = layout ? chunk / nkt : 0;
    const int kt = layout ? (int)(chunk - g16 * nkt) : 0, row = (int)(g16 * 16) + (lane >> 2);
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const int byte = (lane & 3) * 24 + 8 * i, c = byte >> 4;
      const int at = layout ? (lane >> 2) * 96 + (c ^ ((row >> 3) & 1)) * 16 + (byte & 15) : lane * 24 + 8 * i;
      *reinterpret_cast<u32x2*>(image + at) = u32x2{w[2 * i], w[2 * i + 1]};
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    v4i out0 = *reinterpret_cast<const v4i*>(image + lane * 16), out1 = *reinterpret_cast<const v4i*>(image + 1024 + (lane & 31) * 16);
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(out0), "+v"(out1)::"memory");
    uint8_t* const dst = layout ? packed + ((g16 >> 1) * nkt + kt) * 3072 + (g16 & 1) * 1536 : packed + chunk * 1536;
    if (layout || (chunk + 1) * 64 <= nblocks) {
      v4i* const d = reinterpret_cast<v4i*>(dst) + lane;
      if (stream_out) {
        __builtin_nontemporal_store(out0, d);
        if (lane < 32) __builtin_nontemporal_store(out1, d + 64);
      } else {
        d[0] = out0;
        if (lane < 32) d[64] = out1;
      }
    } else if (chunk * 64 + lane < nblocks) {  // the last chunk's blocks one by one
#pragma unroll
      for (int i = 0; i < 3; i++) *reinterpret_cast<u32x2*>(dst + lane * 24 + 8 * i) = u32x2{w[2 * i], w[2 * i + 1]};
    }
    if (layout == 0) {
      if (chunk * 64 + lane < nblocks) scales[chunk * 64 + lane] = (uint8_t)sb;
    } else {
      uint8_t* const sp = scales + tile_major_scale_offset(row, kt * 4 + (lane & 3), (nkt + 3) / 4);
      *sp = (uint8_t)sb;
      if (kt == nkt - 1)  // the bytes of K-blocks past K (K % 512 != 0) are zeros
        for (int b = 4; b < 16 - ((nkt * 4 - 4) & 15); b += 4) sp[b] = 0;
    }
  }
}

hipError_t launch_quantize(const void* X, int x_bf16, uint8_t* packed, uint8_t* scales, int rows, int K, int fmt, int layout, hipStream_t s) {
  const long nblocks = (long)rows * (K / 32);
  if (nblocks == 0) return hipSuccess;
  const long nchunks = layout ? (long)((rows + 15) / 16) * ((K + 127) / 128) : (nblocks + 63) / 64;
  const int waves = nchunks <= kQFewChunks ? 1 : kQWaves;
  const long want = (nchunks + waves - 1) / waves, most = 0xffffffffL / (waves * 64);  // a launch has less than 2^32 work-items; the chunks past them are the grid's next round
  const unsigned grid = (unsigned)(want < most ? want : most);
  const int stream_in = (size_t)rows * K * (x_bf16 ? 2 : 4) >= kCacheBytes, stream_out = (size_t)rows * (K / 4 * 3) >= kStreamBytes;
#define MXFP6_QW(FMT, T, W) quantize_kernel<FMT, T, W><<<grid, W * 64, 0, s>>>((const T*)X, packed, scales, nblocks, K / 32, layout, rows, stream_in, stream_out)
#define MXFP6_Q(FMT, T) do { if (waves == 1) MXFP6_QW(FMT, T, 1); else MXFP6_QW(FMT, T, kQWaves); } while (0)
  if (fmt == 2) { if (x_bf16) MXFP6_Q(2, uint16_t); else MXFP6_Q(2, float); }
  else { if (x_bf16) MXFP6_Q(3, uint16_t); else MXFP6_Q(3, float); }
#undef MXFP6_Q
#undef MXFP6_QW
  return hipGetLastError();
}

// row-major <-> tile-major.  A workgroup moves 32 rows x four K-tiles: 384 row-major bytes per row (three whole cache
// lines) against four whole 3 KB tiles, so both sides are touched in whole lines by one workgroup (one 16-byte piece
// per lane in row-major order over the whole operand ran at 3.9 TB/s, this at 5.8).
__global__ __launch_bounds__(256) void tile_operand_kernel(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst, int nkt, int nk4,
                                                          int tile) {
  const int rt = blockIdx.x / nk4, g = blockIdx.x - rt * nk4;  // row-tile, group of four K-tiles
  const int ntile = min(4, nkt - 4 * g);
  const size_t rm0 = ((size_t)rt * 32 * nkt + 4 * g) * 96, tm0 = ((size_t)rt * nkt + 4 * g) * 3072;
#pragma unroll
  for (int i = 0; i < 3; i++) {
    const int p = threadIdx.x + 256 * i, r = p / 24, q = p - r * 24;  // piece q of the row's 384 bytes
    const int tg = q / 6, c = q - tg * 6;
    if (tg >= ntile) continue;
    const size_t rm = rm0 + (size_t)r * nkt * 96 + q * 16, tm = tm0 + tg * 3072 + (r * 6 + (c ^ ((r >> 3) & 1))) * 16;
    *reinterpret_cast<v4i*>(dst + (tile ? tm : rm)) = *reinterpret_cast<const v4i*>(src + (tile ? rm : tm));
  }
}

hipError_t launch_tile_operand(const uint8_t* src, uint8_t* dst, int rows, int K, int tile, hipStream_t s) {
  const int nkt = K / 128, nk4 = (nkt + 3) / 4;
  const long blocks = (long)(rows / 32) * nk4;
  if (blocks == 0) return hipSuccess;
  tile_operand_kernel<<<(unsigned)blocks, 256, 0, s>>>(src, dst, nkt, nk4, tile);
  return hipGetLastError();
}

// scales [rows, K/32] row-major <-> tile-major: one lane moves the (up to) 16 bytes one row has for four K-tiles;
// K-blocks past K (K % 512 != 0) are written as zero in the tile-major direction
__global__ __launch_bounds__(256) void tile_scales_kernel(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst, long nchunks,
                                                         int nkb, int nk4, int tile) {
  const long s = (long)blockIdx.x * 256 + threadIdx.x;
  if (s >= nchunks) return;
  const int row = (int)(s / nk4), g = (int)(s - (long)row * nk4);
  const int nvalid = min(16, nkb - g * 16);  // a multiple of 4: K % 128 == 0
  const size_t rm = (size_t)row * nkb + (size_t)g * 16, tm = tile_major_scale_offset(row, g * 16, nk4);
#pragma unroll
  for (int i = 0; i < 4; i++) {
    if (tile) {
      *reinterpret_cast<uint32_t*>(dst + tm + 4 * i) = 4 * i < nvalid ? *reinterpret_cast<const uint32_t*>(src + rm + 4 * i) : 0u;
    } else if (4 * i < nvalid) {
      *reinterpret_cast<uint32_t*>(dst + rm + 4 * i) = *reinterpret_cast<const uint32_t*>(src + tm + 4 * i);
    }
  }
}

hipError_t launch_tile_scales(const uint8_t* src, uint8_t* dst, int rows, int K, int tile, hipStream_t s) {
  const int nkb = K / 32, nk4 = (nkb + 15) / 16;
  const long nchunks = (long)rows * nk4;
  if (nchunks == 0) return hipSuccess;
  tile_scales_kernel<<<(unsigned)((nchunks + 255) / 256), 256, 0, s>>>(src, dst, nchunks, nkb, nk4, tile);
  return hipGetLastError();
}

// Row-major -> tile-major for up to two operands (packed bytes and scales) of any size and alignment in one launch, K padded to
// whole K-tiles and the rows to whole row-tiles, zeros in both: the pre-pass of large and of ragged products, where every extra launch
// would cost as much as part of the copy.  A workgroup copies 32 rows x four K-tiles (384 source bytes per row = three whole cache
// lines; a single K-tile's 96 bytes straddle lines, and lines shared between workgroups on different XCDs were fetched twice: 1.64x
// read traffic) in source order, all three loads of a lane in flight: consecutive lanes read consecutive 16-byte pieces of a row and
// write runs of 96 bytes into the four 3 KB tiles.  Other workgroups move the 16 scale bytes one row has for four K-tiles, one row per lane; a
// row's scales start at any byte: five aligned dwords (the last one that is read holds the tensor's last byte) are shifted into
// place.  Bound by memory: both operands of 8192^3, 200 MB moved, about 30 us; level there with a form for whole row- and K-tiles only.
struct PadJob {
  const uint8_t *src, *ssrc;
  uint8_t *dst, *sdst;
  int rows;
  unsigned pblocks, sblocks;
};
__global__ __launch_bounds__(256) void pad_both_kernel(PadJob j0, PadJob j1, int nkb, int nkt, int nk4) {
  unsigned bid = blockIdx.x;
  const bool second = bid >= j0.pblocks + j0.sblocks;
  if (second) bid -= j0.pblocks + j0.sblocks;
  const PadJob& j = second ? j1 : j0;
  const int rowbytes = nkb * 24;
  if (bid < j.pblocks) {
    const int rt = bid / nk4, g = bid - rt * nk4, ntile = min(4, nkt - 4 * g);
    const __amdgpu_buffer_rsrc_t r = make_rsrc(j.src + (size_t)rt * 32 * rowbytes, (uint32_t)min(32, j.rows - rt * 32) * rowbytes);
    uint8_t* const dst = j.dst + ((size_t)rt * nkt + 4 * g) * 3072;
    v4i v[3];
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const int p = threadIdx.x + 256 * i, row = p / 24, q = p - row * 24, at = g * 384 + q * 16;
      v[i] = at < rowbytes ? __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(r, row * rowbytes + at, 0, 0)) : v4i{0, 0, 0, 0};
      if (at + 16 > rowbytes) v[i][2] = v[i][3] = 0;  // rows are whole runs of 8 bytes
    }
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const int p = threadIdx.x + 256 * i, row = p / 24, q = p - row * 24, tg = q / 6, c = q - tg * 6;
      if (tg < ntile) *reinterpret_cast<v4i*>(dst + tg * 3072 + (row * 6 + (c ^ ((row >> 3) & 1))) * 16) = v[i];
    }
  } else {
    const long s = (long)(bid - j.pblocks) * 256 + threadIdx.x;
    const long row = s / nk4;
    const int g = (int)(s - row * nk4);
    if (row >= ((j.rows + 31) & ~31)) return;
    v4i out = {0, 0, 0, 0};
    if (row < j.rows) {
      const size_t at = (size_t)row * nkb + g * 16, end = ((uintptr_t)j.ssrc + (size_t)j.rows * nkb + 3) & ~(uintptr_t)3;
      const uintptr_t from = (uintptr_t)j.ssrc + at;
      const uint32_t* const d = reinterpret_cast<const uint32_t*>(from & ~(uintptr_t)3);
      uint32_t w[5];
#pragma unroll
      for (int i = 0; i < 5; i++) w[i] = (uintptr_t)(d + i) < end ? d[i] : 0u;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int valid = nkb - g * 16 - 4 * i;
        const uint32_t keep = valid >= 4 ? ~0u : valid <= 0 ? 0u : (1u << (8 * valid)) - 1;
        out[i] = (int)(__builtin_amdgcn_alignbyte(w[i + 1], w[i], (uint32_t)from) & keep);
      }
    }
    *reinterpret_cast<v4i*>(j.sdst + tile_major_scale_offset((int)row, g * 16, nk4)) = out;
  }
}

// rows1 == 0: only the first operand
hipError_t launch_pad_both(const uint8_t* src0, uint8_t* dst0, const uint8_t* ssrc0, uint8_t* sdst0, int rows0, const uint8_t* src1, uint8_t* dst1, const uint8_t* ssrc1,
                           uint8_t* sdst1, int rows1, int K, hipStream_t s) {
  const int nkb = K / 32, nkt = (nkb + 3) / 4, nk4 = (nkt + 3) / 4;
  auto job = [&](const uint8_t* src, uint8_t* dst, const uint8_t* ssrc, uint8_t* sdst, int rows) {
    const long tiles = ((long)rows + 31) / 32;
    return PadJob{src, ssrc, dst, sdst, rows, (unsigned)(tiles * nk4), (unsigned)((tiles * 32 * nk4 + 255) / 256)};
  };
  const PadJob j0 = job(src0, dst0, ssrc0, sdst0, rows0), j1 = job(src1, dst1, ssrc1, sdst1, rows1);
  const unsigned blocks = j0.pblocks + j0.sblocks + j1.pblocks + j1.sblocks;
  if (blocks == 0) return hipSuccess;
  pad_both_kernel<<<blocks, 256, 0, s>>>(j0, j1, nkb, nkt, nk4);
  return hipGetLastError();
}

__global__ void fill_zero_kernel(uint8_t* p, size_t n) {
  size_t i = (size_t)blockIdx.x * 256 + threadIdx.x, st = (size_t)gridDim.x * 256;
  for (; i < n; i += st) p[i] = 0;
}

hipError_t launch_fill_zero(void* p, size_t bytes, hipStream_t s) {
  size_t blocks = (bytes + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  if (blocks == 0) return hipSuccess;
  fill_zero_kernel<<<(unsigned)blocks, 256, 0, s>>>((uint8_t*)p, bytes);
  return hipGetLastError();
}

}  // namespace mxfp6
