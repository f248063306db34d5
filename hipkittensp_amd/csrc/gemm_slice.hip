// MXFP6 GEMM for small problems: output tiles of 32 or 64 rows and columns, the K range dealt to the waves of a workgroup.
//
// A GEMM of a few microseconds is latency: its launch, one trip to memory, and, on a kernel that walks K with a barrier per
// K-tile, a chain of steps that leaves most of the chip idle (256 x 1024 x 1024 is 16 tiles of 128 x 128 with eight steps
// each).  Here the chain is cut instead: a workgroup owns a tile of (32 TA) x (32 TB) outputs, so that small problems still
// give every compute unit one, and its waves take chunks of two K-tiles (192 bytes per row) in turn, each through a buffer of
// its own with all of the chunk's loads in flight at once.  No wave waits for another before the sums of the waves meet in
// LDS; where the tiles alone leave compute units idle, the K range is split between workgroups as well, and the workgroup of
// a tile that arrives last adds the shares' sums up in share order (no second launch; bit-reproducible).
//
// Any M, N, K % 32 == 0, either layout and every alignment the entry points take, in one instantiation: rows of 24 bytes
// per K-block start at multiples of 4 at least, which a direct load of 16 bytes accepts; a row's scales start at any byte, a
// lane fetches the 16 bytes of aligned dwords around the eight a chunk needs and the reader shifts them into place
// (v_alignbyte_b32).  All offsets ride in the per-lane offset, which the hardware checks against the end of the resource:
// rows past M or N and K-tiles past the last row's end read as zeros.  A partial last K-tile brings in the head of the next
// row, or of the next row-tile; the scale bytes of K-blocks past K are zeros for both operands, and the products of what
// stands there, 28 * 28 * 32 * 2^-254 at most, are nothing to an fp32 sum, whose last place is 2^-149 at least.
//
// LDS image of a chunk (a wave's buffer): 32-row tiles of 6 KB.  Row-major: rows of 192 bytes, 16-byte piece p of row r at
// r * 192 + (p ^ ((r >> 2) & 3)) * 16 (the 16 rows of a ds_read_b128 phase fall into different banks); tile-major: the two
// K-tiles' 3 KB as they are stored.  MFMA operand map as in the other kernels (common.hpp).
//
// Activations (XT = uint16_t for bf16, float): A is not packed yet, and every wave quantises the part of it that its chunk
// needs: XR rows x 256 elements come into LDS in front of the chunk's B, and while B is on its way every lane turns 32-blocks
// into A's image (the quantiser's own conversion, so the operand has the same bits).  A linear layer of few rows is then one
// launch: the quantiser's is 2.5 us and more of GPU time, of 6 to 9 in all (8 x 4096 x 4096 8.2 -> 6.1 us, 61 x 512 x 2048 7.4 -> 4.8).
// What it costs: every column tile reads and quantises the activations anew, about 300 clocks of a SIMD per 64 blocks, so that it
// pays for few rows (choose_linear_kernel).
#include <type_traits>

#include "kernels.hpp"
#include "loader.hpp"

namespace mxfp6 {
namespace {

constexpr int kSliceTile = 6144;      // bytes of 32 rows of a chunk (two K-tiles)
constexpr int kSliceMaxShares = 16;   // workgroups that share an output tile at most

struct SliceArgs {
  const uint8_t *A, *B, *As, *Bs;  // XT: A are the activations, As is not used
  void* C;
  uint8_t* C_scale;  // fp6 output only
  float* part;       // nsplit > 1: the shares' sums, [tile][share][TA TB tiles of 4 KB]
  unsigned* counters;  // nsplit > 1: one arrival counter per output tile, zero between launches
  int M, N, K, layout_a, layout_b, col_tiles, m_blocks, nsplit;
  int stream;  // B is read with the non-temporal bit (kStreamBytes)
  int vec;     // C takes four outputs of a row at a time
  int fmt_c;
  Epilogue ep;
};

struct PackedA {};  // XT of a packed A
template <int FA, int FB, typename Out, int TA, int TB, int NW, typename XT = PackedA, int XR = 32>
__global__ __launch_bounds__(NW * 64) void gemm_slice_kernel(const SliceArgs args) {
  typedef typename Out::type OutT;
  static_assert((TA == 1 || TA == 2) && (TB == 1 || TB == 2) && NW % 2 == 0, "tile, waves (the chunks of a wave keep their place in a group of four K-tiles)");
  constexpr bool XQ = !std::is_same_v<XT, PackedA>;
  static_assert(XQ ? TA == 1 && XR % 8 == 0 && XR >= 8 && XR <= 32 : XR == 32, "rows of activations");
  constexpr int TT = TA * TB, kRowsA = TA * XR;
  constexpr int kA = TA * XR * 192, kB = TB * kSliceTile, kScA = kA + kB, kScB = kScA + (XQ ? 512 : 1024), kX = kScB + 1024;
  constexpr int kXBlock = XQ ? 32 * (int)sizeof(XT) : 0, kXRow = 8 * kXBlock;  // bytes of activations: of a block, of a row's chunk
  constexpr int kBuf = kX + XR * kXRow;
  constexpr int NAL = XQ ? 1 : kA / 1024, NBL = kB / 1024, NXL = XR * kXRow / 1024;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[NW * kBuf];
  static_assert(NW * kBuf <= 163840 && NW * kBuf >= NW * TT * 4096 + 64, "LDS budget (the buffers double as the reduction buffer)");

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, r32 = lane & 31;
  const int K = args.K, layout_a = args.layout_a, layout_b = args.layout_b;
  const int sbytes = K / 32, rowbytes = sbytes * 24, nkt = (K + 127) / 128, nk4 = (nkt + 3) / 4;

  // workgroup -> (share of K, column tile, block of rows): the round-robin placement on the eight XCDs undone, so that an XCD's
  // workgroups are a contiguous run in which the blocks of rows that read the same rows of B sit side by side
  const int tiles = args.col_tiles * args.m_blocks, total = tiles * args.nsplit;
  const int xcd = blockIdx.x & 7, per = total >> 3, rem = total & 7;
  const int order = (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + (blockIdx.x >> 3);
  const int share = order / tiles, tile = order - share * tiles;
  const int ct = tile / args.m_blocks, mb = tile - ct * args.m_blocks;
  const int m0 = mb * kRowsA, n0 = ct * (32 * TB);
  const int rows_a = min(kRowsA, args.M - m0), rows_b = min(32 * TB, args.N - n0);

  // (a tile-major operand may end in a partial row-tile: its rows past the end are there, of no meaning)
  const __amdgpu_buffer_rsrc_t rA = XQ ? make_rsrc(args.A + (size_t)m0 * sbytes * kXBlock, (uint32_t)rows_a * sbytes * kXBlock)
                                       : make_rsrc(args.A + (size_t)m0 * rowbytes, (uint32_t)(layout_a ? (rows_a + 31) & ~31 : rows_a) * rowbytes);
  const __amdgpu_buffer_rsrc_t rB = make_rsrc(args.B + (size_t)n0 * rowbytes, (uint32_t)(layout_b ? (rows_b + 31) & ~31 : rows_b) * rowbytes);
  // scales: the resource starts and ends at aligned dwords (which hold at least one byte of the tensor each)
  const uint8_t* const sa0 = args.As + (layout_a ? (size_t)(m0 >> 5) * nk4 * 512 : (size_t)m0 * sbytes);
  const uint8_t* const sb0 = args.Bs + (layout_b ? (size_t)(n0 >> 5) * nk4 * 512 : (size_t)n0 * sbytes);
  const uint32_t mis_a = (uint32_t)(uintptr_t)sa0 & 3, mis_b = (uint32_t)(uintptr_t)sb0 & 3;
  const uint32_t len_a = layout_a ? (uint32_t)((rows_a + 31) / 32) * nk4 * 512 : (uint32_t)rows_a * sbytes;
  const uint32_t len_b = layout_b ? (uint32_t)((rows_b + 31) / 32) * nk4 * 512 : (uint32_t)rows_b * sbytes;
  const __amdgpu_buffer_rsrc_t rAs = make_rsrc(sa0 - mis_a, (len_a + mis_a + 3) & ~3u), rBs = make_rsrc(sb0 - mis_b, (len_b + mis_b + 3) & ~3u);

  // chunks of this workgroup: [c0, c1); of this wave: c0 + wave, c0 + wave + NW, ...
  const int nchunks = (nkt + 1) / 2, cps = (nchunks + args.nsplit - 1) / args.nsplit;
  const int c0 = share * cps, c1 = min(nchunks, c0 + cps), first = c0 + wave;

  // per-lane offsets of the next chunk's loads: load i fills LDS bytes [i * 1024, + 1024) of the operand's part of the buffer
  int voff_a[NAL], voff_b[NBL];
  auto load_offset = [&](int i, int layout) __attribute__((always_inline)) {
    const int o = i * 64 + lane, r = o / 12, p = (o - r * 12) ^ ((r >> 2) & 3);
    return layout ? (o / 384) * (nkt * 3072) + (o % 384) * 16 + first * 6144 : r * rowbytes + p * 16 + first * 192;
  };
  if constexpr (!XQ) {
#pragma unroll
    for (int i = 0; i < NAL; i++) voff_a[i] = load_offset(i, layout_a);
  }
#pragma unroll
  for (int i = 0; i < NBL; i++) voff_b[i] = load_offset(i, layout_b);
  const int kstep_a = layout_a ? NW * 6144 : NW * 192, kstep_b = layout_b ? NW * 6144 : NW * 192;
  // scales: lane l fetches those of row l (one 32-row tile: of row l % 32)
  auto scale_offset = [&](int row, int layout, uint32_t mis) __attribute__((always_inline)) {
    return layout ? (row >> 5) * (nk4 * 512) + (row & 31) * 16 + (first >> 1) * 512 + (first & 1) * 8 : ((row * sbytes + (int)mis) & ~3) + first * 8;
  };
  int voff_sa = scale_offset(TA == 2 ? lane : r32, layout_a, mis_a), voff_sb = scale_offset(TB == 2 ? lane : r32, layout_b, mis_b);
  // activations: load i fills LDS bytes [i * 1024, + 1024); the 16-byte pieces of a block are rotated by its place among the 16
  // blocks of two rows, so that the 16 lanes of a ds_read_b128 phase, each on a block of its own, fall into different banks
  constexpr int kXPieces = XQ ? kXBlock / 16 : 1, kXSame = XQ ? 16 / kXPieces : 1;  // blocks next to each other that cover all banks
  auto x_rotate = [](int block) __attribute__((always_inline)) { return (block & 15) / kXSame; };
  [[maybe_unused]] int voff_x[XQ ? NXL : 1];
  if constexpr (XQ) {
#pragma unroll
    for (int i = 0; i < NXL; i++) {
      const int o = i * 64 + lane, b = o / kXPieces, c = (o ^ x_rotate(b)) & (kXPieces - 1);
      voff_x[i] = (b >> 3) * sbytes * kXBlock + (b & 7) * kXBlock + c * 16 + first * kXRow;
    }
  }
  const int sstep_a = layout_a ? NW / 2 * 512 : NW * 8, sstep_b = layout_b ? NW / 2 * 512 : NW * 8;
  // how many bytes a row's scales start behind the aligned dwords fetched for it (taken modulo 4; rows 32 apart share it)
  const uint32_t shift_a = XQ ? 0 : mis_a + (layout_a ? 0 : r32 * sbytes), shift_b = mis_b + (layout_b ? 0 : r32 * sbytes);

  const uint32_t buf = lds_address(smem) + wave * kBuf;
  const uint8_t* const bufp = smem + wave * kBuf;
  [[maybe_unused]] auto issue_x = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < (XQ ? NXL : 0); i++) dma16(rA, buf + kX + i * 1024, voff_x[i], 0);
#pragma unroll
    for (int i = 0; i < (XQ ? NXL : 0); i++) voff_x[i] += NW * kXRow;
  };
  auto issue = [&]() __attribute__((always_inline)) {
    dma16(rBs, buf + kScB, voff_sb, 0);
    if constexpr (!XQ) dma16(rAs, buf + kScA, voff_sa, 0);
    voff_sa += sstep_a, voff_sb += sstep_b;
    if (args.stream) {
#pragma unroll
      for (int i = 0; i < NBL; i++) dma16_nt(rB, buf + kA + i * 1024, voff_b[i], 0);
    } else {
#pragma unroll
      for (int i = 0; i < NBL; i++) dma16(rB, buf + kA + i * 1024, voff_b[i], 0);
    }
    if constexpr (!XQ) {
#pragma unroll
      for (int i = 0; i < NAL; i++) dma16(rA, buf + i * 1024, voff_a[i], 0);
#pragma unroll
      for (int i = 0; i < NAL; i++) voff_a[i] += kstep_a;
    }
#pragma unroll
    for (int i = 0; i < NBL; i++) voff_b[i] += kstep_b;
  };
  // Lane l of pass p quantises block (64 p + l) % 8 of row (64 p + l) / 8 of the chunk's activations.  All of them go into registers
  // first, so that the next chunk's are on their way while this one's are quantised and multiplied.
  [[maybe_unused]] auto quantise = [&](bool more) __attribute__((always_inline)) {
    uint8_t* const own = smem + wave * kBuf;
    v4i x[XR / 8][kXPieces];
#pragma unroll
    for (int p = 0; p < XR / 8; p++)
#pragma unroll
      for (int c = 0; c < kXPieces; c++) {
        const int b = p * 64 + lane;
        x[p][c] = *reinterpret_cast<const v4i*>(own + kX + b * kXBlock + ((c ^ x_rotate(b)) & (kXPieces - 1)) * 16);
      }
    wait_lds_reads();
#pragma unroll
    for (int p = 0; p < XR / 8; p++)
#pragma unroll
      for (int c = 0; c < kXPieces; c++) asm volatile("" : "+v"(x[p][c]));
    if (more) issue_x();
#pragma unroll
    for (int p = 0; p < XR / 8; p++) {
      const int b = p * 64 + lane, row = b >> 3, blk = b & 7;
      int sb;
      u32x6 w;
      if constexpr (kXBlock == 64) w = quantise_block_bf16<FA>(x[p], sb);
      else if constexpr (XQ) w = quantise_block_f32<FA>(x[p], sb);
#pragma unroll
      for (int i = 0; i < 3; i++) {
        const int byte = blk * 24 + 8 * i;
        *reinterpret_cast<u32x2*>(own + row * 192 + ((byte >> 4) ^ ((row >> 2) & 3)) * 16 + (byte & 15)) = u32x2{w[2 * i], w[2 * i + 1]};
      }
      own[kScA + row * 16 + blk] = (uint8_t)sb;
    }
    wait_lds_reads();  // (writes too)
  };
  if (first < c1) {
    if constexpr (XQ) issue_x();  // in front of B: quantised while B is on its way
    issue();
  }

  int a_rd[2][3], b_rd[2][3];  // K-tile u of a chunk, piece 3h + c of the row's 96 bytes
#pragma unroll
  for (int u = 0; u < 2; u++)
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const int row = r32 * 192 + ((6 * u + 3 * h + c) ^ ((r32 >> 2) & 3)) * 16, til = u * 3072 + r32 * 96 + ((3 * h + c) ^ ((r32 >> 3) & 1)) * 16;
      const int ra = XQ ? r32 % XR : r32, rowx = ra * 192 + ((6 * u + 3 * h + c) ^ ((ra >> 2) & 3)) * 16;
      a_rd[u][c] = XQ ? rowx : layout_a ? til : row;  // rows past the XR that are staged mirror those; their outputs are not stored
      b_rd[u][c] = kA + (layout_b ? til : row);
    }

  v16f acc[TA][TB];
#pragma unroll
  for (int t = 0; t < TA; t++)
#pragma unroll
    for (int s = 0; s < TB; s++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[t][s][e] = 0.f;

  for (int c = first; c < c1; c += NW) {
    if constexpr (XQ) {
      wait_vmcnt<NBL + 1>();
      quantise(c + NW < c1);
      if (c + NW < c1) wait_vmcnt<NXL>();
      else wait_vmcnt<0>();
    } else {
      wait_vmcnt<0>();
    }
    v4i fa[TA][2][3], fb[TB][2][3], raw_a[TA], raw_b[TB];
#pragma unroll
    for (int s = 0; s < TB; s++) {
      raw_b[s] = *reinterpret_cast<const v4i*>(bufp + kScB + (s * 32 + r32) * 16);
#pragma unroll
      for (int u = 0; u < 2; u++)
#pragma unroll
        for (int p = 0; p < 3; p++) fb[s][u][p] = *reinterpret_cast<const v4i*>(bufp + b_rd[u][p] + s * kSliceTile);
    }
#pragma unroll
    for (int t = 0; t < TA; t++) {
      raw_a[t] = *reinterpret_cast<const v4i*>(bufp + kScA + (t * 32 + (XQ ? r32 % XR : r32)) * 16);
#pragma unroll
      for (int u = 0; u < 2; u++)
#pragma unroll
        for (int p = 0; p < 3; p++) fa[t][u][p] = *reinterpret_cast<const v4i*>(bufp + a_rd[u][p] + t * kSliceTile);
    }
    wait_lds_reads();  // the buffer is about to be refilled: its reads must have left LDS
    __builtin_amdgcn_sched_barrier(0);
    if (c + NW < c1) issue();
#pragma unroll
    for (int u = 0; u < 2; u++) {
      // a lane's two scale bytes of the K-tile are blocks 2h, 2h + 1 of its four; those past K count as zeros
      const int valid = sbytes - c * 8 - u * 4;
      const uint32_t keep = valid >= 4 ? ~0u : valid <= 0 ? 0u : (1u << (8 * valid)) - 1;
      int sa[TA], sb[TB];
#pragma unroll
      for (int t = 0; t < TA; t++) sa[t] = (int)((__builtin_amdgcn_alignbyte(raw_a[t][u + 1], raw_a[t][u], shift_a) & keep) >> (16 * h));
#pragma unroll
      for (int s = 0; s < TB; s++) sb[s] = (int)((__builtin_amdgcn_alignbyte(raw_b[s][u + 1], raw_b[s][u], shift_b) & keep) >> (16 * h));
#pragma unroll
      for (int t = 0; t < TA; t++)
#pragma unroll
        for (int s = 0; s < TB; s++) {
          const v8i b0 = __builtin_shufflevector(fb[s][u][0], fb[s][u][1], 0, 1, 2, 3, 4, 5, -1, -1);
          const v8i a0 = __builtin_shufflevector(fa[t][u][0], fa[t][u][1], 0, 1, 2, 3, 4, 5, -1, -1);
          acc[t][s] = mfma_fp6<FB, FA, 0, 0>(b0, a0, acc[t][s], sb[s], sa[t]);
        }
#pragma unroll
      for (int t = 0; t < TA; t++)
#pragma unroll
        for (int s = 0; s < TB; s++) {
          const v8i b1 = __builtin_shufflevector(fb[s][u][1], fb[s][u][2], 2, 3, 4, 5, 6, 7, -1, -1);
          const v8i a1 = __builtin_shufflevector(fa[t][u][1], fa[t][u][2], 2, 3, 4, 5, 6, 7, -1, -1);
          acc[t][s] = mfma_fp6<FB, FA, 1, 1>(b1, a1, acc[t][s], sb[s], sa[t]);
        }
    }
  }

  // ---- the waves' sums meet in LDS.  Quad q of lane l of tile (t, s) is C[32 t + l % 32][32 s + 8 q + 4 (l / 32) .. + 3], kept
  // at quad_at(w, tile, l % 32, 2 q + l / 32): 16 bytes each, the rows rotated by twice the quad's number inside their 32
  // places, so that eight lanes on the quads of one row (and the next row's eight) fall into different banks.
  v4f* const sums = reinterpret_cast<v4f*>(smem);
  auto quad_at = [&](int w, int t, int m, int quad) __attribute__((always_inline)) { return (w * TT + t) * 256 + quad * 32 + ((m + 2 * quad) & 31); };
  __syncthreads();  // every wave is out of its buffer
#pragma unroll
  for (int t = 0; t < TA; t++)
#pragma unroll
    for (int s = 0; s < TB; s++)
#pragma unroll
      for (int q = 0; q < 4; q++) sums[quad_at(wave, t * TB + s, r32, 2 * q + h)] = v4f{acc[t][s][4 * q], acc[t][s][4 * q + 1], acc[t][s][4 * q + 2], acc[t][s][4 * q + 3]};
  __syncthreads();
  // thread -> (tile, row, quad): eight lanes side by side own a row's 32 outputs
  constexpr int kItems = (TT * 256 + NW * 64 - 1) / (NW * 64);
  v4f sum[kItems];
#pragma unroll
  for (int k = 0; k < kItems; k++) {
    const int item = tid + k * (NW * 64), t = item >> 8, m = (item >> 3) & 31, quad = item & 7;
    if (item >= TT * 256) continue;
    sum[k] = sums[quad_at(0, t, m, quad)];
#pragma unroll
    for (int w = 1; w < NW; w++) sum[k] += sums[quad_at(w, t, m, quad)];
  }
  if (args.nsplit > 1) {
    // Partial tiles and counter are written and read with device-scope atomic accesses, which go past the XCDs' own L2s (see the
    // ring kernel); the counter wraps to zero at the last share's arrival, so that the next launch finds it as this one did.
    uint64_t* const mine = reinterpret_cast<uint64_t*>(args.part + ((size_t)tile * args.nsplit + share) * (TT * 1024));
#pragma unroll
    for (int k = 0; k < kItems; k++) {
      const int item = tid + k * (NW * 64);
      if (item >= TT * 256) continue;
#pragma unroll
      for (int i = 0; i < 2; i++)
        __hip_atomic_store(mine + item * 2 + i, (uint64_t)__float_as_uint(sum[k][2 * i]) | (uint64_t)__float_as_uint(sum[k][2 * i + 1]) << 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    wait_vmcnt<0>();  // stores count there too: the partial tile has arrived before the counter moves
    __syncthreads();
    int* const last = reinterpret_cast<int*>(smem + NW * TT * 4096);  // behind the sums
    if (tid == 0) *last = atomicInc(args.counters + tile, args.nsplit - 1) == (unsigned)args.nsplit - 1;
    __syncthreads();
    if (!*last) return;
    const uint64_t* const all = reinterpret_cast<const uint64_t*>(args.part + (size_t)tile * args.nsplit * (TT * 1024));
#pragma unroll
    for (int k = 0; k < kItems; k++) {
      const int item = tid + k * (NW * 64);
      if (item >= TT * 256) continue;
      // all shares' loads go out before the first sum; added in share order whoever adds
      uint64_t v[kSliceMaxShares][2];
#pragma unroll
      for (int s = 0; s < kSliceMaxShares; s++)
        if (s < args.nsplit) {
#pragma unroll
          for (int i = 0; i < 2; i++) v[s][i] = __hip_atomic_load(all + s * (TT * 512) + item * 2 + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
#pragma unroll
      for (int s = 0; s < kSliceMaxShares; s++)
        if (s < args.nsplit) {
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const float x = __uint_as_float((uint32_t)(v[s][e >> 1] >> (32 * (e & 1))));
            sum[k][e] = s == 0 ? x : sum[k][e] + x;
          }
        }
    }
  }

  // ---- output
  const int M = args.M, N = args.N;
  const bool has_ep = epilogue_any(args.ep);
#pragma unroll
  for (int k = 0; k < kItems; k++) {
    const int item = tid + k * (NW * 64), t = item >> 8, row = (item >> 3) & 31, quad = item & 7;
    const long m = (long)m0 + (t / TB) * 32 + row, n = (long)n0 + (t % TB) * 32 + quad * 4;
    if (item >= TT * 256 || (XR < 32 && row >= XR)) continue;
    if (has_ep && m < M) {
#pragma unroll
      for (int e = 0; e < 4; e++)
        if (n + e < N) sum[k][e] = epilogue_apply(args.ep, sum[k][e], m, n + e);
    }
    if constexpr (sizeof(OutT) == 1) {
      sums[quad_at(0, t, row, quad)] = sum[k];  // where this thread alone has read
    } else if (m < M) {
      OutT* const c = reinterpret_cast<OutT*>(args.C) + (size_t)m * N + n;
      if (args.vec) {
        if (n < N) store4(c, sum[k][0], sum[k][1], sum[k][2], sum[k][3]);
      } else {
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (n + e < N) store1(c + e, sum[k][e]);
      }
    }
  }
  if constexpr (sizeof(OutT) == 1) {  // C re-quantised to MXFP6 along N (N % 32 == 0): a thread per 32-block
    __syncthreads();
    const int t = tid >> 5, row = tid & 31;
    const long m = (long)m0 + (t / TB) * 32 + row;
    const int blk = ct * TB + t % TB, nkb = N / 32;
    if (t < TT && m < M && blk < nkb) {
      float p0[16], p1[16];
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const v4f a = sums[quad_at(0, t, row, 2 * q)], b = sums[quad_at(0, t, row, 2 * q + 1)];
#pragma unroll
        for (int e = 0; e < 4; e++) p0[4 * q + e] = a[e], p1[4 * q + e] = b[e];
      }
      int sb;
      const u32x6 w = quantise_block_acc(p0, p1, args.fmt_c, sb);
      u32x2* const dst = reinterpret_cast<u32x2*>(reinterpret_cast<uint8_t*>(args.C) + ((size_t)m * nkb + blk) * 24);
#pragma unroll
      for (int i = 0; i < 3; i++) dst[i] = u32x2{w[2 * i], w[2 * i + 1]};
      args.C_scale[(size_t)m * nkb + blk] = (uint8_t)sb;
    }
  }
}

}  // namespace

// Which calls: any size, layout and alignment of the entry points up to 32-bit offsets inside a tile
bool gemm_slice_supports(const GemmArgs& g) {
  return g.M > 0 && g.N > 0 && g.K >= 32 && g.K % 32 == 0 && (long)64 * (g.K / 4 * 3) < (1L << 31) - (1 << 20) && (long)g.M * g.N < (1L << 31) && !g.no_alloc;
}

// Workspace of the K split: bytes of partial tiles and arrival counters
void slice_workspace(const GemmArgs& g, const SlicePlan& p, size_t* part_bytes, size_t* counters) {
  const int rows = p.xrows ? p.xrows : 32 * p.ta;
  *counters = (size_t)((g.M + rows - 1) / rows) * ((g.N + 32 * p.tb - 1) / (32 * p.tb));
  *part_bytes = *counters * p.shares * p.ta * p.tb * 4096;
}

template <int FA, int FB, typename Out>
static hipError_t launch(const GemmArgs& g, const SlicePlan& p, hipStream_t s) {
  const int rows = p.xrows ? p.xrows : 32 * p.ta, col_tiles = (g.N + 32 * p.tb - 1) / (32 * p.tb), m_blocks = (g.M + rows - 1) / rows;
  const int nchunks = ((g.K + 127) / 128 + 1) / 2, shares = p.shares > 1 && g.ks_part && g.ks_counters ? p.shares : 1;
  if (shares > kSliceMaxShares || (shares - 1) * ((nchunks + shares - 1) / shares) >= nchunks) return hipErrorInvalidValue;  // no empty share
  constexpr size_t out = sizeof(typename Out::type);
  // (B with the non-temporal bit, kStreamBytes: not row-major rows that start inside a line, which two chunks read: us, with / without, 8 x 16866 x 16960
  // 68.8 / 64.7, 5 x 34000 x 7008 48.9 / 45.8)
  const SliceArgs a{g.A, g.B, g.As, g.Bs, g.C, g.C_scale, g.ks_part, reinterpret_cast<unsigned*>(g.ks_counters), g.M, g.N, g.K, g.layout_a, g.layout_b, col_tiles, m_blocks, shares,
                    m_blocks == 1 && (g.layout_b || g.K % 512 == 0) && (size_t)g.N * (g.K / 4 * 3) >= kStreamBytes, g.N % 4 == 0 && ((uintptr_t)g.C & (4 * out - 1)) == 0, g.fmt_c, g.ep};
  const unsigned grid = (unsigned)col_tiles * m_blocks * shares;
  if (p.xrows) {
    if constexpr (out == 2) {
      SliceArgs x = a;
      x.A = static_cast<const uint8_t*>(g.X), x.As = g.Bs, x.layout_a = 0;
#define MXFP6_SLICE_X(T, BF16, XR, TB, NW) \
  if (g.x_bf16 == BF16 && p.xrows == XR && p.tb == TB && p.waves == NW) { \
    gemm_slice_kernel<FA, FB, Out, 1, TB, NW, T, XR><<<grid, NW * 64, 0, s>>>(x); \
    return hipGetLastError(); \
  }
      MXFP6_SLICE_X(uint16_t, 1, 8, 1, 4) MXFP6_SLICE_X(uint16_t, 1, 8, 1, 8) MXFP6_SLICE_X(uint16_t, 1, 8, 2, 4) MXFP6_SLICE_X(uint16_t, 1, 8, 2, 8)
      MXFP6_SLICE_X(uint16_t, 1, 16, 1, 4) MXFP6_SLICE_X(uint16_t, 1, 16, 1, 8) MXFP6_SLICE_X(uint16_t, 1, 16, 2, 4) MXFP6_SLICE_X(uint16_t, 1, 16, 2, 6)
      MXFP6_SLICE_X(uint16_t, 1, 32, 1, 4) MXFP6_SLICE_X(uint16_t, 1, 32, 2, 4)
      MXFP6_SLICE_X(float, 0, 8, 1, 4) MXFP6_SLICE_X(float, 0, 8, 1, 8) MXFP6_SLICE_X(float, 0, 8, 2, 4) MXFP6_SLICE_X(float, 0, 8, 2, 6)
      MXFP6_SLICE_X(float, 0, 16, 1, 4) MXFP6_SLICE_X(float, 0, 16, 2, 4) MXFP6_SLICE_X(float, 0, 24, 1, 4)
#undef MXFP6_SLICE_X
    }
    return hipErrorInvalidValue;
  }
#define MXFP6_SLICE(TA, TB, NW) \
  if (p.ta == TA && p.tb == TB && p.waves == NW) { \
    gemm_slice_kernel<FA, FB, Out, TA, TB, NW><<<grid, NW * 64, 0, s>>>(a); \
    return hipGetLastError(); \
  }
  MXFP6_SLICE(1, 1, 4) MXFP6_SLICE(1, 1, 8) MXFP6_SLICE(1, 2, 4) MXFP6_SLICE(1, 2, 8) MXFP6_SLICE(2, 2, 6)
#undef MXFP6_SLICE
  return hipErrorInvalidValue;
}

hipError_t launch_gemm_slice(const GemmArgs& g, const SlicePlan& p, hipStream_t s) {
#define MXFP6_CASE(FA, FB) \
  if (g.fmt_a == FA && g.fmt_b == FB) return g.fmt_c ? launch<FA, FB, OutFp6>(g, p, s) : g.f32out ? launch<FA, FB, OutF32>(g, p, s) : launch<FA, FB, OutBf16>(g, p, s);
  MXFP6_CASE(2, 2) MXFP6_CASE(2, 3) MXFP6_CASE(3, 2) MXFP6_CASE(3, 3)
#undef MXFP6_CASE
  return hipErrorInvalidValue;
}

}  // namespace mxfp6
