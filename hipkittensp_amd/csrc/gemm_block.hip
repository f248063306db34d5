// MXFP6 GEMM for a few hundred to a few thousand rows of A: output tiles of 128 x 128, four waves in step.
//
// The 8-wave ping-pong kernel (gemm_tiled.hip) alternates two wave groups between a memory cluster and a compute
// cluster, which pays when a compute cluster is as long as a memory cluster: 16 MFMAs per wave and K-tile at 256 x 256.
// With the small tiles that fill the machine at a few hundred rows of A a compute cluster is 4 MFMAs, and a K-tile costs
// the two memory clusters one after the other: the operand fragments' way from LDS into registers, twice, plus two
// barriers.  Here nothing alternates.  Every wave owns a 64 x 64 corner of the tile (2 x 2 MFMA tiles, both K-steps of a
// K-tile: 8 MFMAs per K-tile) and keeps two sets of fragment registers: while the MFMAs of K-tile k run on one set, the
// LDS reads of K-tile k+1 fill the other and the direct loads of K-tile k+3 go out; one barrier per K-tile.  48 KB of LDS
// reads per K-tile and workgroup (the 8-wave kernel's 128 x 128 shape: 72 KB).  80 KB of LDS: two workgroups per CU,
// one's waits are the other's work.  That is the ring of three slots of one K-tile, described below; where a CU gets one
// workgroup anyway, or both operands are row-major, the ring is three slots of two K-tiles each (PAIR below, block_stages), and
// tiles of 128 x 256 with eight waves have four slots of one.
//
// Same operand formats, LDS image, lane mapping and raster as the tiled kernel (common.hpp, gemm_tiled.hip): row-major
// or tile-major operands and scales, any M and N (edge tiles: rows past M or N lie beyond the end of their buffer
// resource and read as zeros, stores are predicated), K % 128 == 0, bf16 or fp32 output, fused scales / bias / activation
// (separate instantiations); fp6 output; any size and alignment in instantiations of their own (RAGGED below).
//   ring: three slots of 24 KB (A's 128 rows x 96 bytes, then B's); K-tile k lives in slot k % 3
//   scales: the 16 bytes a row has for four K-tiles, two buffers of (128 + 128) rows x 16 bytes, group g in buffer g % 2
//   step k: loads of K-tile k+3 into the slot K-tile k has left (its fragments are in registers since step k-1), LDS
//           reads of K-tile k+1, MFMAs of K-tile k, wait for the LDS reads and for every load older than this step's,
//           barrier.  A load has two steps to land.
#include "kernels.hpp"
#include "loader.hpp"

namespace mxfp6 {
namespace {

constexpr int kBM = 128, kBK = 128;
constexpr int kATile = kBM * 96;  // bytes of A's tile in a ring slot
constexpr int kScA = kBM * 16;    // bytes of A's scales for four K-tiles
constexpr int kGroupM = 8;        // tile rows per raster group


struct BlockArgs {
  const uint8_t *A, *B, *As, *Bs;
  void* C;
  int M, N, K, tiles_m, tiles_n, layout_a, layout_b, group_m, xcd_remap;
  int nsplit;  // workgroups that share an output tile, each over the same number of whole groups of four K-tiles (the last one over what is left); 1 = no split
  Epilogue ep;  // FUSED instantiations: scales / bias / activation on the accumulators before the output rounding
  uint8_t* C_scale;  // fp6 output only
  int fmt_c;
};

int cu_count_of_device() {
  static int cus[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  if (cus[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) return 0;
    cus[dev] = n;
  }
  return cus[dev];
}

// Chunks of two K-tiles (PAIR, one workgroup per CU) or three slots of one K-tile (two workgroups per CU, one's waits are the
// other's work).  While no CU gets a second workgroup: PAIR, but for K up to 1024, where filling its slots takes a good part of
// the eight K-tiles there are (us, three slots / PAIR: 256 x 4096 x 512 5.9 / 6.4, 256^3 4.4 / 5.0, 384 x 2048 x 1024 7.4 / 7.4 and
// 6.7 / 7.1 tile-major; 256 x 8192 x 1536 12.1 / 11.0, 512 x 4096 x 2048 15.4 / 13.3, tile-major 11.7 / 11.5; 32 x 20608 x 5632
// 27.6 / 23.4 and 22.2 / 18.4), and up to 2048 with both operands tile-major (512 x 8192 x 2048 12.9 / 13.3, 512 x 4096 x 4096 17.9 /
// 16.8).  Beyond: PAIR where its fewer line requests outweigh the second workgroup, with both operands row-major from K = 4096 on
// (2048 x 4096 x 4096 49.5 / 43.8, 1536 x 4096 x 4096 41.2 / 41.1, 640 x 8192 x 2048 23.6 / 25.1), with one from 8192 on (1024 x 8192 x 8192
// 70.1 / 64.9, 256 x 28672 x 8192 81.0 / 73.0, 2048 x 4096 x 4096 39.2 / 40.3), with none never (31.5 / 36.4).
// (launch's and launch_fp6's `stages` = 3 or 6 forces one, for measurement.)
int block_stages(const GemmArgs& g, int grid, int cus) {
  const int row_major = !g.layout_a + !g.layout_b;
  const int min_k = grid <= cus ? (row_major ? 1025 : 2049) : row_major == 2 ? 4096 : row_major == 1 ? 8192 : 0x7fffffff;
  return g.K >= min_k ? 6 : 3;
}
int forced_stages(const GemmArgs& g) { return g.tile_rows == 3 || g.tile_rows == 6 ? g.tile_rows : 0; }

}  // namespace

#ifdef MXFP6_BLOCK_FMT  // ------------------------------------------------------------------------ one pair of operand formats

namespace {

// STAGES: ring slots, 3 (80 KB of LDS, two workgroups per CU), 4 (128 x 256 tiles) or 6, which is PAIR.  Loads run STAGES K-tiles
// ahead of the MFMAs and have STAGES - 1 steps to land.
// PAIR: three slots of two K-tiles (a chunk) each, 152 KB, one workgroup per CU.  What it is for is a row-major operand: the 96
// bytes that a row has in one K-tile straddle 128-byte lines, six line requests for the three lines of four K-tiles, and requests
// are what bounds the way from L2; 192 bytes at a time are four.  A's part of a chunk is loaded in one step and B's in the next,
// three chunks ahead, and there is one wait and one barrier per chunk.  LDS image of a row-major part: rows of 192 bytes, 16-byte
// pieces permuted inside groups of four (piece p of row r at r * 192 + (p ^ ((r >> 2) & 3)) * 16: the 16 rows of a ds_read_b128
// phase fall into different banks); of a tile-major one: two sets of four 3 KB tiles.  us, six slots of one K-tile / PAIR,
// both operands row-major, B tile-major, both: 512 x 8192 x 8192 49.5 / 39.8, 42.4 / 34.6, 33.4 / 31.6; 1024 x 4096 x 14336
// 80.2 / 65.2, 67.5 / 58.9, 52.3 / 51.3; 512 x 2048 x 2048 15.6 / 12.7, 13.6 / 11.6, 11.2 / 10.8.
// WN: waves side by side along N, 2 (tile of 128 x 128, four waves) or 4 (128 x 256, eight waves: waves 0-3 load A's tile
// and half of B's, six loads per K-tile, waves 4-7 the other half of B's, three loads).
// FUSED: the epilogue applies args.ep (a separate instantiation, so that unfused calls carry none of it).
// RAGGED: any M, N, K (K % 32 == 0) and any alignment the entry points take.  What differs from the aligned instantiations:
//   * rows of 24 bytes per K-block start at multiples of 8 (4 at least), which a direct load of 16 bytes accepts; the
//     K-tile's offset rides in the per-lane offset, so that the last K-tile of the last row is cut off at the end of the
//     resource.  Elsewhere a partial last K-tile brings in the head of the next row, and the reader puts 0 for both
//     operands' scale bytes of the K-blocks past K: the products of what stands there, 28 * 28 * 32 * 2^-254 at most, are
//     nothing to an fp32 sum, whose last place is 2^-149 at least.  (Zeroing A's fragments instead: 24 v_and a K-tile behind
//     the wait for the LDS reads, 3 us of 20 at 500 x 5003 x 2880, and in a branch the compiler spills them.)
//   * a row's scales start at any byte: a lane fetches the 20 bytes of aligned dwords around its 16 (one load of 16 bytes and
//     one of 4) and the reader shifts them into place (v_alignbyte_b32, once per four K-tiles).  With three slots one scale
//     buffer serves (a group's scales are in registers, and a barrier passed, before the next group's are fetched): 77 KB
//   * C's rows start at any element: 16-byte stores at element alignment, and single elements where a run of eight (bf16) or
//     four (fp32) outputs crosses N.  Eight lanes' runs can be 128 bytes of a row as in the aligned instantiations, if not one line
// STREAM: B is read with the non-temporal bit: tile-major weights of kStreamBytes and more against one tile row, which nothing reads again.  us,
// plain / non-temporal, layers' weights in turn, one set of activations (and one for each layer): K split, 128 x 8192 x 28672 44.8 / 44.3 (50.3 / 44.2),
// 96 rows (45.2 / 41.2); unsplit, 128 x 28672 x 8192 (48.8 / 40.2); 24 linear layers of these two shapes one after the other, a layer, 128 rows 47.6 / 44.4, 80
// rows 44.1 / 40.8.  What it costs stands at kStreamBytes.  Not row-major weights: 50.6 / 51.8, 96 rows 47.7 / 49.4, 128 x 8192 x 24576 45.0 / 47.5, unsplit 49.7 / 50.5 (with
// activations for each layer 53.8 / 51.6, but 54.0 / 55.0 over 24 layers).  (An instantiation of its own: picked as the kernel runs, 1024 x 4096 x 14336
// paid 58.6 / 59.5 for it.)
// CFORM: how C is stored (CStore; block_c_form), one form to an instantiation: a choice at each store costs a short fp32 product 3 %, and of two copies
// one comes through the instruction cache in vain (aligned rows, C of 4 to 12 MB, of the time as it comes: two copies 0.975, one 0.957).
// 500 x 5003 x 2880: 17.0 us against 148.5 on the one-wave-per-tile kernel, which fetches every operand row again for each of
// its 32 x 32 tiles, 4 bytes per lane.
template <int FA, int FB, typename Out, int STAGES, int WN, bool FUSED, bool RAGGED = false, bool STREAM = false, int CFORM = kCPieces>
__global__ __launch_bounds__(2 * WN * 64, STAGES <= 3 ? 2 : WN / 2) void gemm_block_kernel(const BlockArgs args) {
  typedef typename Out::type OutT;
  static_assert((STAGES == 3 || STAGES == 4 || STAGES == 6) && (WN == 2 || WN == 4), "ring depth, tile width");
  constexpr bool PAIR = STAGES == 6;
  static_assert(!RAGGED || (WN == 2 && FUSED), "one tile width, one epilogue");
  static_assert(!PAIR || WN == 2, "three slots of two K-tiles");
  static_assert(!STREAM || (PAIR && !RAGGED), "three slots of two K-tiles");
  static_assert(sizeof(OutT) != 1 || (FUSED && !RAGGED), "fp6 output: one epilogue, whole 32-blocks");
  constexpr int NW = 2 * WN, kBN = WN * 64, kSlot = kATile + kBN * 96, kScRows = kScA + kBN * 16;
  constexpr int kScBuf = kScRows + (RAGGED ? (kBM + kBN) * 4 : 0);  // RAGGED: 4 more bytes per row behind the rows' 16
  constexpr int kStages = STAGES;
  constexpr int kScBufs = RAGGED && !PAIR ? 1 : 2;
  constexpr int kScLoads = RAGGED ? 2 : 1;  // loads per group of scales
  constexpr int kScBase = kStages * kSlot, kLdsBytes = kScBase + kScBufs * kScBuf;
  static_assert(kLdsBytes <= (STAGES <= 3 && WN == 2 ? 81920 : 163840), "LDS budget");
  __shared__ __attribute__((aligned(1024))) uint8_t smem[kLdsBytes];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(MXFP6_LDS uint8_t*)smem;
  const int K = args.K, layout_a = args.layout_a, layout_b = args.layout_b;
  const int rowbytes = K / 32 * 24, sbytes = K / 32, nkt_all = RAGGED ? (K + kBK - 1) / kBK : K / kBK, nk4_all = (nkt_all + 3) / 4;  // tile-major scales: one 512-byte chunk per 32 rows and group of four K-tiles, the last one padded
  // K split: workgroup b takes share l / tiles of tile l % tiles, l = ksplit_order(b) -- the same number of whole groups
  // of four K-tiles for every share, the last one what is left of K (at least one K-tile: the launcher sees to that) --
  // and leaves its fp32 sums in args.C, then a workspace (partial_offset; RAGGED: nsplit matrices; the reduction adds them up)
  const int ntiles = args.tiles_m * args.tiles_n;
  const bool by_share = args.nsplit > 1 && ksplit_by_share(ntiles * args.nsplit, args.xcd_remap);  // the XCDs are dealt by ksplit_order, not by tile_order
  const int order = args.nsplit > 1 ? ksplit_order(blockIdx.x, ntiles * args.nsplit, args.xcd_remap) : blockIdx.x, share = order / ntiles;
  const int share_groups = (nk4_all + args.nsplit - 1) / args.nsplit, kt0 = share * share_groups * 4;
  const int nkt = min(nkt_all - kt0, share_groups * 4), nk4 = (nkt + 3) / 4;

  const int tile = tile_order(order - share * ntiles, args.tiles_m, args.tiles_n, args.group_m, by_share ? 0 : args.xcd_remap);
  if (tile < 0) return;  // never: the grid is the tile count times the shares
  const int pm = tile & 0xffff, pn = tile >> 16;
  const int rows_a = min(kBM, args.M - pm * kBM), rows_b = min(kBN, args.N - pn * kBN);

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const bool loads_a = wave < 4;  // this wave loads row-tile `wave` of A's tile (every wave loads row-tile `wave` of B's)
  const int h = lane >> 5, r32 = lane & 31;

  // operand rows of this tile; rZ: a resource of length zero, loads through it fetch nothing (K-tiles past the end)
  // (a share's resources start at its first K-tile, 96 or 3072 bytes times kt0 into a row or row-tile, and end that much
  // earlier, so that rows past the tile's last still lie beyond the end)
  const uint32_t oa = (uint32_t)kt0 * (layout_a ? 3072 : 96), ob = (uint32_t)kt0 * (layout_b ? 3072 : 96);
  // (a tile-major operand may end in a partial row-tile: its rows past the end are there, of no meaning)
  const __amdgpu_buffer_rsrc_t rA = make_rsrc(args.A + (size_t)pm * kBM * rowbytes + oa, (uint32_t)(layout_a ? (rows_a + 31) & ~31 : rows_a) * rowbytes - oa);
  const __amdgpu_buffer_rsrc_t rB = make_rsrc(args.B + (size_t)pn * kBN * rowbytes + ob, (uint32_t)(layout_b ? (rows_b + 31) & ~31 : rows_b) * rowbytes - ob);
  const __amdgpu_buffer_rsrc_t rZ = make_rsrc(args.A, 0);
  // scales: the first half of the waves fetch A's (rows 0-63, 64-127 of the tile; with eight waves, waves 2, 3 fetch what
  // waves 0, 1 fetch, into the same place, so that every wave issues one scale load per group), the second half B's, 64
  // rows each; a lane fetches the 16 bytes one row has for four K-tiles
  const bool sc_a = wave < NW / 2;
  const int slay = sc_a ? layout_a : layout_b, srows = sc_a ? rows_a : rows_b, stile = sc_a ? pm : pn;
  const uint8_t* sp = sc_a ? args.As : args.Bs;
  const int sheight = sc_a ? kBM : kBN;  // rows per tile of the operand whose scales these are
  const uint32_t os = (uint32_t)(kt0 >> 2) * (slay ? 512 : 16);  // the share's first group of four K-tiles
  const uint8_t* const sbase = sp + (size_t)stile * (sheight / 32) * (slay ? nk4_all * 512 : 32 * sbytes) + os;
  const uint32_t slen = (uint32_t)(slay ? (srows + 31) / 32 * nk4_all * 512 : srows * sbytes) - os;
  // RAGGED: the resource starts and ends at aligned dwords (which hold at least one byte of the tensor each)
  const uint32_t smis = RAGGED ? (uint32_t)(uintptr_t)sbase & 3 : 0;
  const __amdgpu_buffer_rsrc_t rS = RAGGED ? make_rsrc(sbase - smis, (slen + smis + 3) & ~3u) : make_rsrc(sbase, slen);
  const int spart = sc_a ? wave & 1 : wave - NW / 2;  // which 64 rows
  const int srow = spart * 64 + lane;
  const int voff_row = slay ? (srow >> 5) * nk4_all * 512 + (srow & 31) * 16 : srow * sbytes;
  const int voff_s = RAGGED ? (voff_row + (int)smis) & ~3 : voff_row;
  const int sstep = slay ? 512 : 16;
  const uint32_t sdst = lds0 + kScBase + (sc_a ? 0 : kScA) + spart * 1024;
  const uint32_t sdst_tail = lds0 + kScBase + kScRows + (sc_a ? 0 : kBM * 4) + spart * 256;  // RAGGED: bytes 16 .. 19 of a row's dwords

  // per-lane global byte offsets of the direct loads: load q = 3 wave + i fills LDS bytes [q * 1024, + 1024) of an
  // operand's tile.  Row-major: 16-byte slot o holds piece (o % 6) ^ ((row >> 3) & 1) of row o / 6.  Tile-major: the
  // 3072-byte tile of 32 rows is stored in this order; wave w loads row-tile w.
  // PAIR: load q = 6 wave + i of two K-tiles: slot o holds piece (o % 12) ^ ((row >> 2) & 3) of row o / 12; tile-major: K-tile
  // q / 12's four tiles one after the other.
  constexpr int kLoads = PAIR ? 6 : 3;
  int voff_a[kLoads], voff_b[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; i++) {
    if constexpr (PAIR) {
      const int q = wave * 6 + i, o = q * 64 + lane, r = o / 12, c = (o - r * 12) ^ ((r >> 2) & 3);
      const int vrow = r * rowbytes + c * 16, vtile = (q % 12 / 3) * (nkt_all * 3072) + (q / 12) * 3072 + (q % 3) * 1024 + lane * 16;
      voff_a[i] = layout_a ? vtile : vrow;
      voff_b[i] = layout_b ? vtile : vrow;
      continue;
    }
    const int q = wave * 3 + i, o = q * 64 + lane;
    const int r = o / 6, c = (o - r * 6) ^ ((r >> 3) & 1);
    const int vrow = r * rowbytes + c * 16, vtile = wave * (nkt_all * 3072) + i * 1024 + lane * 16;
    voff_a[i] = layout_a ? vtile : vrow;
    voff_b[i] = layout_b ? vtile : vrow;
  }
  const int kstep_a = layout_a ? 3072 : 96, kstep_b = layout_b ? 3072 : 96;

  // per-lane LDS read offsets inside a slot: the lane's three 16-byte pieces 3h .. 3h + 2 of its row
  const int sw = (r32 >> 3) & 1;
  int a_rd[3], b_rd[3];
#pragma unroll
  for (int c = 0; c < 3; c++) {
    a_rd[c] = (wm * 64 + r32) * 96 + ((3 * h + c) ^ sw) * 16;
    b_rd[c] = kATile + (wn * 64 + r32) * 96 + ((3 * h + c) ^ sw) * 16;
  }
  // PAIR: pieces 6 u + 3 h .. + 2 of the row's two K-tiles (u: which), and the step from a 32-row tile to the next
  [[maybe_unused]] int a_rd2[2][3], b_rd2[2][3];
  [[maybe_unused]] const int a_next = layout_a ? 3072 : 6144, b_next = layout_b ? 3072 : 6144;
  if constexpr (PAIR) {
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int c = 0; c < 3; c++) {
        const int row = r32 * 192 + ((6 * u + 3 * h + c) ^ ((r32 >> 2) & 3)) * 16, tile = u * 12288 + r32 * 96 + ((3 * h + c) ^ sw) * 16;
        a_rd2[u][c] = wm * 2 * a_next + (layout_a ? tile : row);
        b_rd2[u][c] = 2 * kATile + wn * 2 * b_next + (layout_b ? tile : row);
      }
  }
  const int sa_rd = kScBase + (wm * 64 + r32) * 16, sb_rd = kScBase + kScA + (wn * 64 + r32) * 16;
  const int sc_shift = 16 * h;  // a lane's two scale bytes of a K-tile: bytes 2h, 2h + 1 of the K-tile's four

  v16f acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[i][j][e] = 0.f;
  v12i fa[2][2], fb[2][2];  // [set][tile]: a lane's 48 bytes of a 32-row tile, dwords 0-5 the first MFMA's operand, 6-11 the second's
  int sca[2][4], scb[2][4];  // [tile][K-tile of the group]: scale bytes in bytes 0, 1
  v4i raw_a[2], raw_b[2];
  [[maybe_unused]] int tail_a[2], tail_b[2];
  // RAGGED: how many bytes a row's scales start behind the aligned dwords fetched for it (v_alignbyte_b32 takes it modulo 4;
  // rows 32 apart share it)
  [[maybe_unused]] const uint32_t shift_a = (uint32_t)(uintptr_t)args.As + (layout_a ? 0 : r32 * sbytes);
  [[maybe_unused]] const uint32_t shift_b = (uint32_t)(uintptr_t)args.Bs + (layout_b ? 0 : r32 * sbytes);

  // load n of this wave's for K-tile t: 0-2 the three of row-tile `wave` of A's tile (LA: this wave loads A at all), 3-5 of B's
  auto load_one = [&]<bool LA>(int t, int slot, int n) __attribute__((always_inline)) {
    const bool in = t < nkt;
    const uint32_t dst = lds0 + slot * kSlot + wave * 3072;
    if (n < 3) {
      if constexpr (LA) dma16(in ? rA : rZ, dst + n * 1024, voff_a[n], RAGGED ? 0 : t * kstep_a);
      if constexpr (RAGGED) voff_a[n] += kstep_a;  // the loads come in the order of t
    } else {
      dma16(in ? rB : rZ, dst + kATile + (n - 3) * 1024, voff_b[n - 3], RAGGED ? 0 : t * kstep_b);
      if constexpr (RAGGED) voff_b[n - 3] += kstep_b;
    }
  };
  // PAIR: load n of this wave's six of A's or B's part of chunk c (K-tiles 2c, 2c + 1).  The chunk's offset rides in the per-lane
  // offset, which the hardware checks against the end of the resource: past the last row's last K-tile it fetches nothing.
  [[maybe_unused]] const int nchunks = (nkt + 1) / 2;
  auto load_pair = [&]<bool OF_A>(int c, int slot, int n) __attribute__((always_inline)) {
    const uint32_t dst = lds0 + slot * (2 * kSlot) + (OF_A ? 0 : 2 * kATile) + (wave * 6 + n) * 1024;
    if constexpr (OF_A) dma16(c < nchunks ? rA : rZ, dst, voff_a[PAIR ? n : 0] + c * (2 * kstep_a), 0);
    else if constexpr (STREAM) dma16_nt(c < nchunks ? rB : rZ, dst, voff_b[PAIR ? n : 0] + c * (2 * kstep_b), 0);
    else dma16(c < nchunks ? rB : rZ, dst, voff_b[PAIR ? n : 0] + c * (2 * kstep_b), 0);
  };
  auto load_tile = [&]<bool LA>(int t, int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < 6; n++) load_one.template operator()<LA>(t, slot, n);
  };
  // (the group's offset goes into the per-lane offset, which the hardware checks against the end of the resource: with
  // K % 512 != 0 the last group of a row-major row is shorter than 16 bytes, and the last row's must not read past the tensor)
  auto load_scales = [&](int grp) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t rs = grp < nk4 ? rS : rZ;
    dma16(rs, sdst + (grp & (kScBufs - 1)) * kScBuf, voff_s + grp * sstep, 0);
    if constexpr (RAGGED) dma4(rs, sdst_tail + (grp & (kScBufs - 1)) * kScBuf, voff_s + grp * sstep + 16, 0);
  };
  auto read_tile = [&]<int SET>(int slot) __attribute__((always_inline)) {
    const uint8_t* st = smem + slot * kSlot;
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int c = 0; c < 3; c++) {
        const v4i p = *reinterpret_cast<const v4i*>(st + b_rd[c] + j * 3072);
#pragma unroll
        for (int e = 0; e < 4; e++) fb[SET][j][4 * c + e] = p[e];
      }
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int c = 0; c < 3; c++) {
        const v4i p = *reinterpret_cast<const v4i*>(st + a_rd[c] + i * 3072);
#pragma unroll
        for (int e = 0; e < 4; e++) fa[SET][i][4 * c + e] = p[e];
      }
  };
  auto read_pair = [&]<int SET, int U>(int slot) __attribute__((always_inline)) {  // PAIR: K-tile U of a chunk
    const uint8_t* st = smem + slot * (2 * kSlot);
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int c = 0; c < 3; c++) {
        const v4i p = *reinterpret_cast<const v4i*>(st + b_rd2[U][c] + j * b_next);
#pragma unroll
        for (int e = 0; e < 4; e++) fb[SET][j][4 * c + e] = p[e];
      }
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int c = 0; c < 3; c++) {
        const v4i p = *reinterpret_cast<const v4i*>(st + a_rd2[U][c] + i * a_next);
#pragma unroll
        for (int e = 0; e < 4; e++) fa[SET][i][4 * c + e] = p[e];
      }
  };
  auto read_scales = [&](int grp) __attribute__((always_inline)) {
    const uint8_t* sc = smem + (grp & (kScBufs - 1)) * kScBuf;
#pragma unroll
    for (int i = 0; i < 2; i++) raw_a[i] = *reinterpret_cast<const v4i*>(sc + sa_rd + i * 512);
#pragma unroll
    for (int j = 0; j < 2; j++) raw_b[j] = *reinterpret_cast<const v4i*>(sc + sb_rd + j * 512);
    if constexpr (RAGGED) {
#pragma unroll
      for (int i = 0; i < 2; i++) {
        tail_a[i] = *reinterpret_cast<const int*>(sc + kScBase + kScRows + (wm * 64 + i * 32 + r32) * 4);
        tail_b[i] = *reinterpret_cast<const int*>(sc + kScBase + kScRows + kBM * 4 + (wn * 64 + i * 32 + r32) * 4);
      }
    }
  };
  auto take_scales = [&]([[maybe_unused]] int grp) __attribute__((always_inline)) {
    if constexpr (RAGGED) {
#pragma unroll
      for (int km = 0; km < 4; km++) {
        // K-blocks this K-tile has; a lane's two are blocks 2h, 2h + 1
        const int nvalid = sbytes - ((kt0 >> 2) + grp) * 16 - 4 * km;
        const uint32_t keep = (2 * h < nvalid ? 0xffu : 0u) | (2 * h + 1 < nvalid ? 0xff00u : 0u);
#pragma unroll
        for (int i = 0; i < 2; i++) {
          const uint32_t wa = __builtin_amdgcn_alignbyte(km < 3 ? raw_a[i][km + 1] : tail_a[i], raw_a[i][km], shift_a);
          const uint32_t wb = __builtin_amdgcn_alignbyte(km < 3 ? raw_b[i][km + 1] : tail_b[i], raw_b[i][km], shift_b);
          sca[i][km] = (int)(wa >> sc_shift & keep), scb[i][km] = (int)(wb >> sc_shift & keep);
        }
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int km = 0; km < 4; km++) sca[i][km] = (int)((uint32_t)raw_a[i][km] >> sc_shift), scb[i][km] = (int)((uint32_t)raw_b[i][km] >> sc_shift);
  };
  // first source = B rows (index n), second = A rows (index m): a lane ends up owning 4 consecutive n of row m = lane % 32,
  // four times per 32 x 32 tile
  // between(q) runs after the q-th of the eight MFMAs
  auto mma_tile = [&]<int SET, int KM>(auto&& between) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const v8i a0 = __builtin_shufflevector(fa[SET][i], fa[SET][i], 0, 1, 2, 3, 4, 5, -1, -1);
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const v8i b0 = __builtin_shufflevector(fb[SET][j], fb[SET][j], 0, 1, 2, 3, 4, 5, -1, -1);
        acc[i][j] = mfma_fp6<FB, FA, 0, 0>(b0, a0, acc[i][j], scb[j][KM], sca[i][KM]);
        between(i * 2 + j);
      }
    }
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const v8i a1 = __builtin_shufflevector(fa[SET][i], fa[SET][i], 6, 7, 8, 9, 10, 11, -1, -1);
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const v8i b1 = __builtin_shufflevector(fb[SET][j], fb[SET][j], 6, 7, 8, 9, 10, 11, -1, -1);
        acc[i][j] = mfma_fp6<FB, FA, 1, 1>(b1, a1, acc[i][j], scb[j][KM], sca[i][KM]);
        between(4 + i * 2 + j);
      }
    }
  };

  // slot[i]: ring slot of K-tile k + i
  int slot[kStages];
#pragma unroll
  for (int i = 0; i < kStages; i++) slot[i] = i;
  // LA: this wave loads A's tile too (six loads per K-tile, else three); instantiated per wave class, so that no branch
  // sits between the MFMAs (a branch there makes the compiler keep a second copy of the accumulators)
  auto step = [&]<int KM, bool LA>(int k) __attribute__((always_inline)) {
    constexpr int CUR = KM & 1, NXT = CUR ^ 1;
    // LDS reads of K-tile k + 1 first, then the MFMAs of K-tile k with the direct loads of K-tile k + STAGES (into K-tile
    // k's slot) between them, one after each of the first six, and after the seventh the scales of a later group of four
    // (with a group's first K-tile): the loads wait for the address unit behind an MFMA instead of in front of the LDS reads
    // PAIR: slot[0 .. 2] hold chunks k / 2 .. + 2
    if constexpr (PAIR) read_pair.template operator()<NXT, NXT>(slot[KM & 1]);
    else read_tile.template operator()<NXT>(slot[1]);
    if (KM == 3) read_scales((k >> 2) + 1);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
    mma_tile.template operator()<CUR, KM>([&](int q) __attribute__((always_inline)) {
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (PAIR) {  // B's part of chunk k / 2 + 2 in even steps, A's of chunk k / 2 + 3 in odd ones
        if (q < 6 && (KM & 1) == 0) load_pair.template operator()<false>((k >> 1) + 2, slot[2], q);
        if (q < 6 && (KM & 1) == 1) load_pair.template operator()<true>((k >> 1) + 3, slot[0], q);
      } else {
        if (q < 6) load_one.template operator()<LA>(k + kStages, slot[0], q);
      }
      if (q == 6 && KM == 0) load_scales((k >> 2) + 1);
      __builtin_amdgcn_sched_barrier(0);
    });
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
    wait_lds_reads();
#pragma unroll
    for (int i = 0; i < 2; i++) asm volatile("" : "+v"(fa[NXT][i]));
#pragma unroll
    for (int j = 0; j < 2; j++) asm volatile("" : "+v"(fb[NXT][j]));
    if (KM == 3) take_scales((k >> 2) + 1);
    if constexpr (PAIR) {
      // Chunk c's places are free once its second K-tile is in registers (the barrier of step 2c), and chunk c + 1 must be there
      // for step 2c + 1: one wait and barrier per chunk.  Younger than the last of chunk c + 1's loads (step 2c - 2): A's of step
      // 2c - 1, B's of this step, six each, and this step's scales; those of step 2c - 2 must have landed (read in step 2c + 1).
      if constexpr ((KM & 1) == 0) {
        wait_vmcnt<12 + (KM == 0 ? kScLoads : 0)>();
        barrier();
      } else {
        const int t = slot[0];
        slot[0] = slot[1], slot[1] = slot[2], slot[2] = t;
      }
      return;
    }
    // K-tile k + 2 has landed: everything older than the loads of the last STAGES - 2 steps (six each, and a scale load
    // in steps with KM == 0)
    constexpr int kScalesInFlight = (KM % 4 == 0) + (STAGES == 4 && (KM + 3) % 4 == 0);
    wait_vmcnt<(LA ? 6 : 3) * (STAGES - 2) + kScLoads * kScalesInFlight>();
    barrier();
    const int t = slot[0];
#pragma unroll
    for (int i = 0; i + 1 < kStages; i++) slot[i] = slot[i + 1];
    slot[kStages - 1] = t;
  };

  // prologue (scales of the first group(s), K-tiles 0 .. STAGES - 1) and the K loop
  auto run = [&]<bool LA>() __attribute__((always_inline)) {
    constexpr int NL = LA ? 6 : 3;
    load_scales(0);
    if constexpr (PAIR) {  // chunks 0, 1 and A's part of chunk 2; step 0 goes on with B's
#pragma unroll
      for (int t = 0; t < 5; t++)
#pragma unroll
        for (int n = 0; n < 6; n++) {
          if (t & 1) load_pair.template operator()<false>(t >> 1, t >> 1, n);
          else load_pair.template operator()<true>(t >> 1, t >> 1, n);
        }
      wait_vmcnt<18>();
      barrier();
      read_pair.template operator()<0, 0>(0);
      read_scales(0);
      wait_lds_reads();
      take_scales(0);
    } else {
#pragma unroll
      for (int t = 0; t < kStages; t++) load_tile.template operator()<LA>(t, t);
      wait_vmcnt<NL * (STAGES - 1)>();
      barrier();
      read_tile.template operator()<0>(0);
      read_scales(0);
      wait_lds_reads();
      take_scales(0);
      wait_vmcnt<NL * (STAGES - 2)>();
      barrier();  // K-tile 1 is in place, and every wave has K-tile 0 in registers: its slot is free
    }
    int k = 0;
    for (; k + 4 <= nkt; k += 4) {
      step.template operator()<0, LA>(k);
      step.template operator()<1, LA>(k + 1);
      step.template operator()<2, LA>(k + 2);
      step.template operator()<3, LA>(k + 3);
    }
    // a last group of fewer than four K-tiles (K % 512 != 0): the same steps; their loads lie past the end and fetch nothing
    if (k < nkt) step.template operator()<0, LA>(k);
    if (k + 1 < nkt) step.template operator()<1, LA>(k + 1);
    if (k + 2 < nkt) step.template operator()<2, LA>(k + 2);
  };
  if constexpr (WN == 2) {
    run.template operator()<true>();
  } else {
    if (loads_a) run.template operator()<true>();
    else run.template operator()<false>();
  }
  wait_vmcnt<0>();  // no direct load may still be on its way into LDS when the workgroup gives the memory back

  // ---- epilogue, straight from the accumulators.  Register v of lane l is C[m][n] with m = l % 32 and
  // n = 8 (v / 4) + 4 (l / 32) + v % 4 inside a 32 x 32 tile.  bf16: after the conversion lanes l and l + 32 trade halves
  // (v_permlane32_swap), so that every lane owns 8 consecutive outputs, 16 bytes; then lanes trade for whole lines (pair_rows, join_lines).
  const int N = args.N, N2 = N * (int)sizeof(OutT);
  const bool edge = rows_a != kBM || rows_b != kBN;
  if constexpr (FUSED) {
    // y = act(acc * row_scale[m] * col_scale[n] + bias[n]) in fp32.  Per 32 x 32 tile a lane owns row 32 i + lane % 32 of its
    // wave's rows and columns 8 q + 4 h .. + 3 for q = 0 .. 3; N % 8 == 0, so a run of four is inside or outside N as a whole
    const void* bias = args.ep.bias;
    const float *row_scale = args.ep.row_scale, *col_scale = args.ep.col_scale;
    const int act = args.ep.act, bias_bf16 = args.ep.bias_bf16;
    const long m0 = (long)pm * kBM + wm * 64 + r32, n0 = (long)pn * kBN + wn * 64 + 4 * h;
    float rs[2];
#pragma unroll
    for (int i = 0; i < 2; i++) rs[i] = row_scale && m0 + i * 32 < args.M ? row_scale[m0 + i * 32] : 1.f;
#pragma unroll
    for (int j = 0; j < 2; j++) {
      if (bias || row_scale || col_scale) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const long n = n0 + j * 32 + q * 8;
          v4f cs = {1.f, 1.f, 1.f, 1.f}, bi = {0.f, 0.f, 0.f, 0.f};
          if constexpr (RAGGED) {  // a run of four may cross N
#pragma unroll
            for (int e = 0; e < 4; e++) {
              const long ne = n + e < N ? n + e : N - 1;
              if (col_scale) cs[e] = col_scale[ne];
              if (bias) bi[e] = bias_bf16 ? bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(bias)[ne]) : reinterpret_cast<const float*>(bias)[ne];
            }
          } else if (n < N) {
            if (col_scale) cs = *reinterpret_cast<const v4f*>(col_scale + n);
            if (bias && bias_bf16) {
              const u32x2 b2 = *reinterpret_cast<const u32x2*>(reinterpret_cast<const uint16_t*>(bias) + n);
              bi = v4f{__uint_as_float(b2[0] << 16), __uint_as_float(b2[0] & 0xffff0000u), __uint_as_float(b2[1] << 16), __uint_as_float(b2[1] & 0xffff0000u)};
            } else if (bias) {
              bi = *reinterpret_cast<const v4f*>(reinterpret_cast<const float*>(bias) + n);
            }
          }
#pragma unroll
          for (int i = 0; i < 2; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) acc[i][j][4 * q + e] = fmaf(acc[i][j][4 * q + e] * rs[i], cs[e], bi[e]);
        }
      }
      // one branch per activation and tile, not one per element (that took 2 us of a 20 us call, with or without an activation)
#pragma unroll
      for (int i = 0; i < 2; i++) {
        if (act == 1) {
#pragma unroll
          for (int e = 0; e < 16; e++) acc[i][j][e] = act_relu(acc[i][j][e]);
        } else if (act == 2) {
#pragma unroll
          for (int e = 0; e < 16; e++) acc[i][j][e] = act_gelu(acc[i][j][e]);
        } else if (act == 3) {
#pragma unroll
          for (int e = 0; e < 16; e++) acc[i][j][e] = act_silu(acc[i][j][e]);
        }
        asm volatile("" : "+v"(acc[i][j]));
      }
    }
  }
  if constexpr (sizeof(OutT) == 1) {  // C re-quantised to MXFP6 along N (the next GEMM's K): a wave's two tiles of a band at a time
#pragma unroll
    for (int i = 0; i < 2; i++)
      store_fp6_band(acc[i][0], acc[i][1], args.fmt_c, (uint8_t*)args.C, args.C_scale, (long)pm * kBM + wm * 64 + i * 32 + r32, args.M, pn * (kBN / 32) + wn * 2, N / 32);
    return;
  }
  // RAGGED with a K split: the shares' matrices have rows of a multiple of four floats
  [[maybe_unused]] const size_t ldc = RAGGED && args.nsplit > 1 ? ragged_pitch(N) : N;
  const __amdgpu_buffer_rsrc_t rC = make_rsrc((OutT*)args.C + (size_t)share * args.M * N + (size_t)pm * kBM * N + (size_t)pn * kBN,
                                              (uint32_t)((rows_a - 1) * N + rows_b) * (uint32_t)sizeof(OutT));
  if constexpr (!RAGGED && sizeof(OutT) == 4) {
    if (args.nsplit > 1) {
      // this share's partial sums, in the accumulators' order (partial_offset)
      const int band0 = pm * (kBM / 32) + wm * 2, ct0 = pn * (kBN / 32) + wn * 2;
      float* const base = (float*)args.C + partial_offset(share, band0, ct0, args.M, N) / 4 + lane * 4;
      const size_t band_stride = ((size_t)N + 31) / 32 * 1024;
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
          if ((band0 + i) * 32 + r32 < args.M && (ct0 + j) * 32 < N) {
#pragma unroll
            for (int gq = 0; gq < 4; gq++)
              *reinterpret_cast<v4f*>(base + i * band_stride + j * 1024 + gq * 256) = v4f{acc[i][j][4 * gq], acc[i][j][4 * gq + 1], acc[i][j][4 * gq + 2], acc[i][j][4 * gq + 3]};
          }
      return;
    }
  }
  constexpr bool LINES = CFORM != kCPieces, OUT = CFORM == kCOut;
  constexpr int kRun = 16 / (int)sizeof(OutT);
  const int row_l = wm * 64 + (LINES ? line_row<1>(lane) : r32), col_l = wn * 64 + (LINES ? line_piece<1>(lane) : h) * kRun;
  const int voff = row_l * N2 + col_l * (int)sizeof(OutT);
  // RAGGED: `n` consecutive outputs of a row, 16 bytes of them at C's element alignment or, across N, one by one
  // (the lane's address once, the stores' places from it: 512 x 296 x 16960 19.6 / 19.0, 49 x 20832 x 672 fp32 7.8 / 7.5)
  [[maybe_unused]] OutT* const lane_c = (OutT*)args.C + ((size_t)share * args.M + (size_t)pm * kBM + row_l) * ldc + (size_t)pn * kBN + col_l;
  // 16 bytes of the lane, `row` rows and `col` columns on
  auto put = [&](v4i v, int row, int col) __attribute__((always_inline)) {
    const int m = row_l + row, n = col_l + col;
    if constexpr (!RAGGED) {
      if (!edge || (m < rows_a && n < rows_b)) store_c<OUT>(v, rC, voff + col * (int)sizeof(OutT), row * N2);
    } else {
      if (m >= rows_a || n >= rows_b) return;
      OutT* const p = lane_c + row * ldc + col;
      if (n + kRun <= rows_b) {
        typedef int v4i_element __attribute__((ext_vector_type(4), aligned(2)));
        if constexpr (OUT) __builtin_nontemporal_store((v4i_element)v, reinterpret_cast<v4i_element*>(p));
        else *reinterpret_cast<v4i_element*>(p) = (v4i_element)v;
      } else {
        OutT o[kRun];
        __builtin_memcpy(o, &v, 16);
#pragma unroll
        for (int e = 0; e + 1 < kRun; e++)
          if (n + e < rows_b) p[e] = o[e];
      }
    }
  };
  // four registers, 16 outputs (bf16) or 8 (fp32) of a row apart, of rows `row` on; `col` columns on
  auto put4 = [&](v4i (&v)[2][2], int row, int col) __attribute__((always_inline)) {
    constexpr int kApart = 2 * kRun;
    if constexpr (LINES) {
#pragma unroll
      for (int p = 0; p < 2; p++) pair_rows(v[p][0], v[p][1]);
#pragma unroll
      for (int t = 0; t < 2; t++) {
        join_lines(v[0][t], v[1][t]);
        put(v[0][t], row + t * 16, col);
        put(v[1][t], row + t * 16 + 8, col);
      }
    } else {
#pragma unroll
      for (int q = 0; q < 4; q++) put(v[q >> 1][q & 1], row, col + q * kApart);
    }
  };
  if constexpr (sizeof(OutT) == 2) {
#pragma unroll
    for (int i = 0; i < 2; i++) {
      uint32_t pk[2][8];
#pragma unroll
      for (int j = 0; j < 2; j++)
#pragma unroll
        for (int e = 0; e < 8; e++) pk[j][e] = pack_bf16x2(acc[i][j][2 * e], acc[i][j][2 * e + 1]);
#pragma unroll
      for (int j = 0; j < 2; j++)
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
          for (int c = 0; c < 2; c++) {
            // runs 2t and 2t+1 (dwords 4t+c and 4t+2+c): lower lanes keep run 2t and get the partner's, upper lanes run 2t+1
            const auto x = __builtin_amdgcn_permlane32_swap(pk[j][4 * t + c], pk[j][4 * t + 2 + c], false, false);
            pk[j][4 * t + c] = x[0], pk[j][4 * t + 2 + c] = x[1];
          }
      v4i v[2][2];
#pragma unroll
      for (int j = 0; j < 2; j++)
#pragma unroll
        for (int t = 0; t < 2; t++) v[j][t] = v4i{(int)pk[j][4 * t], (int)pk[j][4 * t + 1], (int)pk[j][4 * t + 2], (int)pk[j][4 * t + 3]};
      put4(v, i * 32, 0);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int j = 0; j < 2; j++) {
        v4i v[2][2];
#pragma unroll
        for (int q = 0; q < 4; q++)
#pragma unroll
          for (int e = 0; e < 4; e++) v[q >> 1][q & 1][e] = __float_as_int(acc[i][j][4 * q + e]);
        put4(v, i * 32, j * 32);
      }
  }
}

template <int FA, int FB, bool FUSED>
hipError_t launch(const GemmArgs& g, const BlockArgs& a, int tiles, int stages, hipStream_t s) {
  const int cus = cu_count_of_device();
  const bool f32 = g.f32out || a.nsplit > 1;  // shares leave fp32 partial sums
  const int grid = tiles * a.nsplit, form = block_c_form(g);
  if (stages == 0) stages = block_stages(g, grid, cus);
  auto with = [&]<typename Out, int STAGES, int WN, bool STREAM>() {
    constexpr int kThreads = 2 * WN * 64;
    if (form == kCOut) gemm_block_kernel<FA, FB, Out, STAGES, WN, FUSED, false, STREAM, kCOut><<<grid, kThreads, 0, s>>>(a);
    else if (form == kCPieces) gemm_block_kernel<FA, FB, Out, STAGES, WN, FUSED, false, STREAM, kCPieces><<<grid, kThreads, 0, s>>>(a);
    else gemm_block_kernel<FA, FB, Out, STAGES, WN, FUSED, false, false, kCKept><<<grid, kThreads, 0, s>>>(a);
  };
  auto with_out = [&]<typename Out>() {
    if (g.tile_cols == 256) with.template operator()<Out, 4, 4, false>();  // tiles of 128 x 256, eight waves, four slots
    else if ((sizeof(typename Out::type) == 2 || !FUSED) && block_streams_weights(g)) with.template operator()<Out, 6, 2, sizeof(typename Out::type) == 2 || !FUSED>();
    else if (stages == 6) with.template operator()<Out, 6, 2, false>();
    else with.template operator()<Out, 3, 2, false>();
  };
  if (f32) with_out.template operator()<OutF32>();
  else with_out.template operator()<OutBf16>();
  return hipGetLastError();
}
// RAGGED instantiations, the fused epilogue applied or not inside.  PAIR from K = 1920 on while no CU gets a second workgroup (us,
// three slots / PAIR: 64 x 3001 x 1888 11.1 / 11.1, 500 x 5003 x 1056 13.2 / 13.6, 100 x 5003 x 2016 17.8 / 16.1), from 6144 on
// beyond (2000 x 8191 x 4128 107.5 / 105.0, 1000 x 4097 x 4128 47.3 / 48.6, 572 x 22563 x 13760 295 / 266).
template <int FA, int FB>
hipError_t launch_ragged(const GemmArgs& g, const BlockArgs& a, int tiles, hipStream_t s) {
  const int grid = tiles * a.nsplit, cus = cu_count_of_device();
  const bool deep = g.K >= (grid <= cus ? 1920 : 6144);
  auto with = [&]<typename Out, int CFORM>() {
    if (deep) gemm_block_kernel<FA, FB, Out, 6, 2, true, true, false, CFORM><<<grid, 256, 0, s>>>(a);
    else gemm_block_kernel<FA, FB, Out, 3, 2, true, true, false, CFORM><<<grid, 256, 0, s>>>(a);
  };
  auto with_out = [&]<typename Out>(int form) {
    if (form == kCOut) with.template operator()<Out, kCOut>();
    else if (form == kCKept) with.template operator()<Out, kCKept>();
    else with.template operator()<Out, kCPieces>();
  };
  if (g.f32out || a.nsplit > 1) with_out.template operator()<OutF32>(block_c_form(g));
  else with_out.template operator()<OutBf16>(block_c_form(g));
  return hipGetLastError();
}
// fp6 output, the fused epilogue applied or not inside
template <int FA, int FB>
hipError_t launch_fp6(const GemmArgs& g, const BlockArgs& a, int tiles, int stages, hipStream_t s) {
  if (stages == 0) stages = block_stages(g, tiles, cu_count_of_device());
  if (g.tile_cols == 256) gemm_block_kernel<FA, FB, OutFp6, 4, 4, true><<<tiles, 512, 0, s>>>(a);
  else if (stages == 6) gemm_block_kernel<FA, FB, OutFp6, 6, 2, true><<<tiles, 256, 0, s>>>(a);
  else gemm_block_kernel<FA, FB, OutFp6, 3, 2, true><<<tiles, 256, 0, s>>>(a);
  return hipGetLastError();
}
template <int FA, int FB>
hipError_t launch(const GemmArgs& g, const BlockArgs& a, int tiles, int stages, hipStream_t s) {
  if (g.fmt_c && a.nsplit == 1) return launch_fp6<FA, FB>(g, a, tiles, stages, s);
  // a split leaves the epilogue to the reduction
  if (a.nsplit == 1 && epilogue_any(g.ep)) return launch<FA, FB, true>(g, a, tiles, stages, s);
  return launch<FA, FB, false>(g, a, tiles, stages, s);
}


}  // namespace

#define MXFP6_PASTE2(a, b) a##b
#define MXFP6_PASTE(a, b) MXFP6_PASTE2(a, b)
hipError_t MXFP6_PASTE(launch_gemm_block_fmt, MXFP6_BLOCK_FMT)(const GemmArgs& g, hipStream_t s) {
  constexpr int FA = MXFP6_BLOCK_FMT / 10, FB = MXFP6_BLOCK_FMT % 10;
  static_assert((FA == 2 || FA == 3) && (FB == 2 || FB == 3), "MXFP6_BLOCK_FMT: 22, 23, 32 or 33");
  const int bn = g.tile_cols == 256 ? 256 : 128, nsplit = g.ksplit > 1 ? g.ksplit : 1;
  BlockArgs a{g.A, g.B, g.As, g.Bs, nsplit > 1 ? (void*)g.ks_part : g.C, g.M, g.N, g.K, (g.M + kBM - 1) / kBM, (g.N + bn - 1) / bn, g.layout_a, g.layout_b,
              g.raster_group_m > 0 ? g.raster_group_m : kGroupM, g.raster_no_xcd_remap == 1 ? 0 : g.raster_no_xcd_remap == 2 ? 2 : 1, nsplit, g.ep, g.C_scale, g.fmt_c};
  const int tiles = a.tiles_m * a.tiles_n;
  if (g.ragged) {
    if (nsplit > 1) a.ep = Epilogue{};  // the reduction applies it
    return launch_ragged<FA, FB>(g, a, tiles, s);
  }
  return launch<FA, FB>(g, a, tiles, forced_stages(g), s);
}
#undef MXFP6_PASTE
#undef MXFP6_PASTE2

#else  // ---------------------------------------------------------------------------------------- the host-side object

bool gemm_block_supports(const GemmArgs& g) {
  // N % 8 keeps every run of 8 bf16 outputs whole and aligned; K in whole K-tiles; 32-bit byte offsets
  // inside one tile's operand rows and inside one tile's rows of C
  return g.M > 0 && g.N > 0 && g.K >= 128 && g.N % 8 == 0 && g.K % 128 == 0 && (long)128 * (g.K / 4 * 3) < (1L << 31) &&
         (long)128 * g.N * 4 < (1L << 31) && (long)((g.M + 127) / 128) <= 65535 && (long)((g.N + 127) / 128) <= 32767 &&
         (long)((g.M + 127) / 128) * ((g.N + 127) / 128) < (1L << 31) && ((uintptr_t)g.C % 16) == 0 && operands_aligned16(g) && !g.fmt_c &&
         !g.no_alloc;
}

// The RAGGED instantiations: whatever the entry points take, up to 32-bit offsets inside a tile
bool gemm_block_ragged_supports(const GemmArgs& g) {
  return g.M > 0 && g.N > 0 && g.K >= 32 && g.K % 32 == 0 && (long)128 * (g.K / 4 * 3) < (1L << 31) - 32768 && (long)((g.M + 127) / 128) <= 65535 &&
         (long)((g.N + 127) / 128) <= 32767 && (long)((g.M + 127) / 128) * ((g.N + 127) / 128) < (1L << 31) && !g.fmt_c;
}

bool block_streams_weights(const GemmArgs& g) {
  const int split = g.ksplit > 1 ? g.ksplit : 1;
  if (g.ragged || g.tile_cols == 256 || !g.layout_b || g.M > kBM || (size_t)g.N * (g.K / 4 * 3) < kStreamBytes || block_c_form(g) == kCKept) return false;
  if (split == 1 && (g.fmt_c || (g.f32out && epilogue_any(g.ep)))) return false;  // not built
  return (forced_stages(g) ? forced_stages(g) : block_stages(g, (g.N + 127) / 128 * split, cu_count_of_device())) == 6;
}

// How a RAGGED instantiation stores C.  As it comes where that is little: below 4 MB, up to 64 rows, and the sums of a K split's shares, which are
// read again at once (us, as it comes / whole lines through the L2s / whole lines non-temporal, fp32: 49 x 20832 x 672 7.45 / 7.75 / 7.5, 20 x 30001 x 672 7.35 /
// 7.65 / 7.8, 64 x 20001 x 2080 13.1 / 13.35 / 13.4; 191 x 664 x 18624 18.6 / 18.85 / 18.85, 512 x 296 x 16960 19.05 / 19.2 / 19.2).  Else non-temporally where
// its rows start on lines.  Where they do not, a line is two stores: bf16 up to 32 MB (1000 x 5003 x 1056, 9.5 MB, 17.1 / 17.1 / 16.6; 256 x 16001 x 1056 13.2 / 13.2 /
// 12.8; 2000 x 8191 x 1056, 31 MB, 38.5 / 38.4 / 37.2; not 6000 x 3001 x 672, 34 MB, 33.6 / 33.2 / 36.2, nor, through the L2s most with a short K, 3524 x 13814 x 288,
// 93 MB, 47.6 / 42.3); fp32 never (256 x 16001 x 1056, 16 MB, 13.4 / 12.2 /
// 16.3; 1000 x 5003 x 1056, 19 MB, 16.5 / 15.5 / 18.6; 2000 x 8191 x 1056 36.3 / 34.2 / 49.3).  Over 70 drawn shapes of each type, of the time as it comes: bf16
// 4 to 32 MB 1.00 / 0.97, above 1.00 / 1.04; fp32 8 to 12 MB 0.96 / 1.00, 12 to 20 MB 0.93 / 1.09, above 0.94 / 1.28.
static int ragged_c_form(const GemmArgs& g) {
  const size_t row = (size_t)g.N * (g.f32out ? 4 : 2), bytes = g.M * row;
  if (g.ksplit > 1 || g.M <= 64 || bytes < (size_t)4 << 20) return kCPieces;
  if ((((uintptr_t)g.C | row) & 127) == 0) return kCOut;
  return !g.f32out && bytes <= (size_t)32 << 20 ? kCOut : kCKept;
}
int block_c_form(const GemmArgs& g) {
  if (g.ragged) return ragged_c_form(g);
  if (g.ksplit > 1 || g.fmt_c) return kCPieces;
  const size_t row = (size_t)g.N * (g.f32out ? 4 : 2), bytes = g.M * row;
  const bool whole = (((uintptr_t)g.C | row) & 127) == 0;
  return bytes < (size_t)(whole ? 2 : 4) << 20 ? kCPieces : c_leaves(g.C, g.M, row) ? kCOut : kCKept;
}

hipError_t launch_gemm_block_fmt22(const GemmArgs& g, hipStream_t s);
hipError_t launch_gemm_block_fmt23(const GemmArgs& g, hipStream_t s);
hipError_t launch_gemm_block_fmt32(const GemmArgs& g, hipStream_t s);
hipError_t launch_gemm_block_fmt33(const GemmArgs& g, hipStream_t s);

// g.ksplit > 1 (with g.ks_part): the K range of every output tile split between that many workgroups, then
// ksplit_reduce_kernel (gemm_tiled.hip), which also applies a fused epilogue.  The caller has checked that the last share
// is not empty (block_split_shares, dispatch.hip).
hipError_t launch_gemm_block(const GemmArgs& g, hipStream_t s) {
  const hipError_t e = g.fmt_a == 2 ? (g.fmt_b == 2 ? launch_gemm_block_fmt22(g, s) : launch_gemm_block_fmt23(g, s))
                                    : (g.fmt_b == 2 ? launch_gemm_block_fmt32(g, s) : launch_gemm_block_fmt33(g, s));
  return e == hipSuccess && g.ksplit > 1 ? launch_ksplit_reduce(g, s) : e;
}

#endif  // MXFP6_BLOCK_FMT

}  // namespace mxfp6
