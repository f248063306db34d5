// Internal launcher interface between the C ABI (api.hip) and the kernel translation units.
#pragma once
#include "common.hpp"
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mxfp6 {

struct GemmArgs {
  const uint8_t *A, *B, *As, *Bs;  // packed operands and E8M0 scales (device)
  void* C;                         // bf16 or float [M, N]
  int M, N, K;
  int fmt_a, fmt_b;  // 2 = e2m3, 3 = e3m2
  bool f32out;
  int layout_a = 0, layout_b = 0;  // 0 = row-major, 1 = tile-major (operand: 32 rows x 128 elements in LDS image order; scales: 32 rows x 16 bytes)
  int tile_rows = 0;               // tiled kernel: rows of A per output tile, 128 or 256; 0 = chosen per shape
  int tile_cols = 0;               // ... and rows of B: 128 (with 128 rows of A only) or 256; 0 with tile_rows set = 256
  int skinny_geometry = 0;         // skinny kernel: 1 = 32 rows of B and all waves, 2 = 16 rows of B, 3 = half the waves, 4 - 9 = 1 or 2 with the K range split between 2 / 4 / 8 workgroups, 10 = two waves; 0 = by shape
  Epilogue ep;                     // fused bias / scales / activation (all optional)
  uint8_t* C_scale = nullptr;      // fp6 output (every kernel but the ragged and generic ones; skinny: gemm_skinny_stores_fp6): C is the packed operand [M, 3N/4], this its E8M0 bytes [M, N/32]
  int fmt_c = 0;                   // 2 / 3: format of the fp6 output; 0: bf16 / fp32 output
  int out_fp6 = 0;                 // kernel choice only: the fp32 sums (f32out) leave as MXFP6
  const void* X = nullptr;         // skinny and slice kernel: activations [M, K] that they quantise to fmt_a themselves, in place of A and As (gemm_skinny_takes_x, choose_linear_kernel)
  int x_bf16 = 0;                  // ... in bf16 (the skinny kernel takes no others), else fp32
  int raster_group_m = 0, raster_no_xcd_remap = 0;  // tiled kernel, measurement only: tile rows per raster group (0 = the default, 4), XCD remap off (1), or on with a K split's workgroups in tile-by-tile order (2)
  int ablation = 0;  // tiled kernel, measurement only: leave out LDS reads (1), loads (2), MFMAs (4); results are then meaningless
  uint32_t* clock_stamps = nullptr;  // tiled kernel, measurement only: four words for workgroup 0's clock / real-time counters at start and end
  int ragged = 0;                  // block kernel: its instantiations for any size and alignment (gemm_block_ragged_supports)
  int no_alloc = 0;                // skinny kernel: the K split keeps its partial tiles in the library's static scratch array instead of an allocated workspace
  int force_split = 0;             // skinny kernel, M <= 32: split K between this many workgroups (1, 2, 4, 8); 0 = by shape
  int ksplit = 0;                  // tiled, block and ring kernels: workgroups that share an output tile (KernelChoice::shares, ragged_shares); needs ks_part
  float* ks_part = nullptr;        // ... their partial sums: ksplit sets of 32 x 32 tiles (partial_offset), ragged: matrices [M, ragged_pitch(N)] of floats (ring and slice kernels: partial tiles)
  int* ks_counters = nullptr;      // K split of the ring and slice kernels: one arrival counter per tile of C, zero between launches
};

// the LDS-staged kernels fetch operands and scales 16 bytes per lane: all four tensors must be 16-byte aligned
inline bool operands_aligned16(const GemmArgs& g) {
  return (((uintptr_t)g.A | (uintptr_t)g.B | (uintptr_t)g.As | (uintptr_t)g.Bs) & 15) == 0;
}

// Weights (and the quantiser's output) of this many bytes and more are read (written) with the non-temporal bit: half of the 256 MB
// last-level cache, so that with the activations and the outputs little of them would be found there by the next read.  us, plain /
// non-temporal, N = 8192, tile-major weights, in turn from 640 MB of them (a program's layers): skinny kernel, 16 rows, 60 MB
// 15.3 / 14.3, 120 MB 25.7 / 23.8, 144 MB 30.2 / 27.5, 168 MB 33.8 / 31.0; ring kernel, 64 rows, 20.9 / 21.2, 33.1 / 30.5, 37.9 / 34.2, 42.3 /
// 38.2.  The same weights again in every call, which stay in that cache in part or, below the line, as a whole: skinny 13.2 / 12.0, 21.8 /
// 22.4, 25.2 / 26.2, 28.7 / 30.0; ring 19.0 / 19.6, 28.0 / 30.0, 31.8 / 33.6, 34.9 / 37.6.
// The tiled kernel's K split and the block kernel, tile-major weights of 176 MB that one tile row meets, N = 8192 (up: N = 28672, K = 8192):
//   * layers' weights in turn, one set of activations: tiled, 256 rows 67.9 / 66.0, 224 63.3 / 62.5; block, 128 rows 44.8 / 44.3; with activations for each of 2
//     to 8 layers 69.6 / 64.9, 50.2 / 44.1, up 48.7 / 40.0, for each of 24 69.9 / 69.8, 50.4 / 48.4, up 49.1 / 40.5.  (What B does not displace stays: activations,
//     partial sums, C.)
//   * 24 linear layers, up and down in turn, a layer: 128 rows 47.6 / 44.4, 80 rows 44.1 / 40.8, 160 60.7 / 60.2, 256 68.2 / 67.9; their first forward pass
//     49.2 / 48.9, 68.7 / 68.3
//   * the same weights in every call: 60.0 / 67.5, 39.9 / 46.2, up 36.2 / 40.2
//   * a first pass right behind the quantiser that made the weights, from a source that is 940 MB of new fp32: 85.4 / 88.6 (host clock), 58.5 / 62.5, up 59.2 /
//     63.1; from one that was there before: 94.2 / 88.2, 67.6 / 64.4, up 65.1 / 63.9; behind a copy of the weights 88.4 / 89.9, 59.2 / 58.8; behind 1 GB of other
//     stores 113 / 86, 92 / 64, up 93 / 59
// So it costs a program that runs one layer over and over, or quantises and multiplies once, up to a sixth, and gives one with layers up to a sixth.
constexpr size_t kStreamBytes = (size_t)128 << 20;

// ---- kernel choice (dispatch.hip): candidates of the automatic path, a time model per candidate, a calibration table
enum Candidate : int { kCandTiled256 = 0, kCandTiled128x256, kCandTiled128x128, kCandBlock, kCandBlockWide, kCandSkinny, kCandTiledSplit256, kCandTiledSplit128, kCandBlockSplit, kCandRing, kNumCandidates,
  kCandSlice = kNumCandidates,  // not calibrated: its own model against the best of the others (slice_plan)
  kCandSliceX };  // in candidate sets only: the slice kernel on a linear layer's activations (choose_linear_kernel)
struct SlicePlan {  // small problems: tiles of 32 ta x 32 tb outputs, K dealt to `waves` waves and to `shares` workgroups (gemm_slice.hip)
  int ta, tb, waves, shares;
  int xrows = 0;  // rows of activations a workgroup quantises itself (8, 16, 24, 32); 0: A is packed
};
struct KernelChoice {
  int cand;    // a Candidate, or -1: none of them takes the shape (ragged_shares says what does)
  int shares;  // K split: workgroups per output tile (1 = none)
  int rows;    // tiled kernel's split: rows of A per tile
  double us;   // modelled time x calibration factor
  SlicePlan slice = {};
};
int device_cus();
double candidate_model_us(const GemmArgs& g, int cand, int want_split, int cus, int* shares, int* rows);  // modelled microseconds; < 0: the candidate does not take the shape
KernelChoice choose_kernel(const GemmArgs& g, int want_split, bool allow_split, unsigned mask = ~0u);  // mask: bit per Candidate that may be chosen; want_split: 0 = by the model, 1 = never, n = n shares where a candidate splits; allow_split: a workspace is to be had
bool padded_pays(const GemmArgs& g, int want_split, unsigned mask, const KernelChoice& other, bool a_done, GemmArgs* t, KernelChoice* c);  // a ragged product on padded tile-major copies
KernelChoice choose_linear_kernel(const GemmArgs& g, int want_split, unsigned mask);  // g.X, g.x_bf16: the activations
int tiled_split_shares(const GemmArgs& g, int want, int cus, int bm);  // the tiled kernel's K split with tiles of bm (256 or 128) rows when it is to split: shares (1 = the shape has none)
int ragged_shares(const GemmArgs& g, int want, bool allow_split);  // shapes no candidate takes: shares of the block kernel's K split (1 = unsplit), 0 = the generic kernel
int block_split_shares(const GemmArgs& g, int want, int cus);             // ... the block kernel's

hipError_t launch_gemm_generic(const GemmArgs& g, hipStream_t s);
bool gemm_tiled_supports(const GemmArgs& g);
hipError_t launch_gemm_tiled(const GemmArgs& g, hipStream_t s);
bool tiled_streams_weights(const GemmArgs& g);  // whether launch_gemm_tiled reads B with the non-temporal bit
int tiled_c_form(const GemmArgs& g);            // how it stores C (CStore; kCPieces: a K split's sums, MXFP6)
bool gemm_tiled4_supports(const GemmArgs& g);  // the 4-wave variant of the tiled kernel (selectable, never chosen automatically)
hipError_t launch_gemm_tiled4(const GemmArgs& g, hipStream_t s);
bool gemm_block_supports(const GemmArgs& g);  // 128 x 128 tiles, four waves in step (a few hundred to a few thousand rows of A)
bool gemm_block_ragged_supports(const GemmArgs& g);  // with GemmArgs::ragged: any M, N, K % 32 == 0 and alignment
hipError_t launch_gemm_block(const GemmArgs& g, hipStream_t s);
bool block_streams_weights(const GemmArgs& g);  // whether launch_gemm_block reads B with the non-temporal bit
int block_c_form(const GemmArgs& g);            // how it stores C or, split, its shares' sums (CStore)
hipError_t launch_ksplit_reduce(const GemmArgs& g, hipStream_t s);  // sums g.ksplit shares' partial sums at g.ks_part into g.C, with the epilogue
bool gemm_ring_supports(const GemmArgs& g);  // batched decode: private streams of B per wave, A through a flag-guarded ring (no barrier per K-tile)
int ring_ksplit_plan(const GemmArgs& g, int want, size_t* part_bytes, size_t* counters);  // its K split for this problem (want: 0 = by shape, 1 = none, n = n shares): shares (1 = none), bytes of partial tiles, arrival counters
hipError_t launch_gemm_ring(const GemmArgs& g, hipStream_t s);
bool gemm_slice_supports(const GemmArgs& g);
void slice_workspace(const GemmArgs& g, const SlicePlan& p, size_t* part_bytes, size_t* counters);  // of its K split (shares > 1): g.ks_part, g.ks_counters
hipError_t launch_gemm_slice(const GemmArgs& g, const SlicePlan& p, hipStream_t s);  // without the workspace: unsplit
bool gemm_mid_supports(const GemmArgs& g);
hipError_t launch_gemm_mid(const GemmArgs& g, hipStream_t s);
bool gemm_skinny_supports(const GemmArgs& g);
bool gemm_skinny_stores_fp6(const GemmArgs& g);  // MXFP6 output without a workspace (N % 32, the workgroup's shape)
bool gemm_skinny_takes_x(const GemmArgs& g);  // M and K of a call whose activations the kernel can quantise itself
hipError_t launch_gemm_skinny(const GemmArgs& g, hipStream_t s);
bool gemm_skinny_scratch_fits(const GemmArgs& g);  // no_alloc: the K split this call would use fits the static scratch array
hipError_t release_split_workspaces();             // returns every K-split workspace to the stream-ordered allocator
hipError_t launch_quantize(const void* X, int x_bf16, uint8_t* packed, uint8_t* scales, int rows, int K, int fmt, int layout, hipStream_t s);
hipError_t launch_tile_operand(const uint8_t* src, uint8_t* dst, int rows, int K, int tile, hipStream_t s);
hipError_t launch_tile_scales(const uint8_t* src, uint8_t* dst, int rows, int K, int tile, hipStream_t s);
hipError_t launch_pad_both(const uint8_t* src0, uint8_t* dst0, const uint8_t* ssrc0, uint8_t* sdst0, int rows0, const uint8_t* src1, uint8_t* dst1, const uint8_t* ssrc1,
                           uint8_t* sdst1, int rows1, int K, hipStream_t s);  // any size and alignment -> padded tile-major; rows1 == 0: one operand
hipError_t launch_fill_zero(void* p, size_t bytes, hipStream_t s);
hipError_t launch_mfma_probe(const uint8_t* A, const uint8_t* B, const uint8_t* As, const uint8_t* Bs, int rows_a, int rows_b, int K, int fmt_a,
                             int fmt_b, int iters, int workgroups, float* sink, uint32_t* stats, hipStream_t s);
hipError_t launch_stream_probe(const uint8_t* buf, size_t bytes, int workgroups, int waves, uint32_t* stats, hipStream_t s);

}  // namespace mxfp6
