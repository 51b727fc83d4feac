// Device descriptors of the heightfield-fit problems and the launcher shared by the
// C ABI and the adjoint kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>

#include "wt_device.hpp"

namespace wt {

constexpr int kFitMaxWaves = 128;
constexpr int kFitMaxSnapshots = 32;
// The reduction: blocks of 16 rows (parameters, and the loss), 16 wavefronts of four parts
// each side by side.
constexpr int kReduceRows = 16, kReduceThreads = 1024;
inline int reduce_blocks(int W) { return (5 * W + 1 + kReduceRows - 1) / kReduceRows; }
// Classes of problems, a kernel each: few waves (adjoint_few_kernel), and W <= 64 and
// W <= 128: the chunks of 16 waves the adjoint kernel's LDS has room for. From 65 waves on
// the time table does not fit beside the rest.
constexpr int kFitClasses = 3;
constexpr int kFitClassChunks[kFitClasses] = {1, 4, 8};
constexpr int kFitWavefronts = 8;  // of an adjoint workgroup: two per SIMD, sharing the tables
constexpr int kFitFewWavefronts = 4;
// Few waves: up to 4 at any size, and up to 6 in a small problem (up to 512 tiles of 16
// pairs), which is bound by its chain of loads, set-up and one tile. Loss and gradient, us in
// a graph, matrix contraction / few-waves kernel: 64 x 64 x 4 snapshots with 1 wave 10.1 / 7.3,
// 4 waves 10.4 / 8.2, 6 waves 10.4 / 9.2; 512 x 512 x 16 with 4 waves 19.5 / 19.0; 200 problems
// of 256 x 256 x 16 with 1 wave 732 / 445, 4 waves 740 / 582. Sums of 8 waves pass its registers,
// and at 5 the matrix contraction of large problems is even.
constexpr int kFitFewWaves = 4, kFitFewWavesSmall = 6, kFitSmallTiles = 512;
// How a problem's work is cut into adjoint blocks: strips of columns, and per strip runs
// of tiles of consecutive (row, snapshot) pairs: 16, or 8 or 4 of few waves. It depends on
// the problem alone.
struct FitBlocks {
  int tile_pairs, tiles_per_block, blocks_per_strip, nblocks;
};
inline FitBlocks fit_blocks(int n, int S, int W) {
  const long long strips = (n + 63) / 64, pairs = (long long)n * S;
  const bool small = strips * ((pairs + 15) / 16) <= kFitSmallTiles;
  const bool few = W <= (small ? kFitFewWavesSmall : kFitFewWaves);
  FitBlocks b;
  b.tile_pairs = !few ? 16 : small ? 4 : 8;
  const long long tiles = (pairs + b.tile_pairs - 1) / b.tile_pairs, total = strips * tiles;
  // enough tiles per wavefront to pay for a block's set-up
  const int wavefronts = few ? kFitFewWavefronts : kFitWavefronts;
  long long per_block = std::min<long long>((total + 2047) / 2048, 8) * wavefronts;
  if (few && small) per_block = wavefronts;
  // a problem too small to fill the GPU's wavefronts that way is cut into parts of 4, 2 or 1
  // tiles, about one for each CU, and each tile then has more of a CU's load path to
  // itself: the eight tiles of a workgroup took 3.5 us to fetch on one CU (64 x 64, 8
  // snapshots, 16 waves: 14.0 us an iteration with 4 parts of 8 tiles, 11.3 with 32 of one;
  // 256 x 256, 16 snapshots, 64 waves: 23.0 with 128 of 8, 19.5 with 256 of 4)
  if (!few)
    for (; per_block > 1 && total <= per_block * 128; per_block /= 2) {
    }
  b.tiles_per_block = (int)per_block;
  b.blocks_per_strip = (int)((tiles + b.tiles_per_block - 1) / b.tiles_per_block);
  b.nblocks = (int)(strips * b.blocks_per_strip);
  return b;
}
inline bool fit_few(const FitBlocks& b) { return b.tile_pairs < 16; }
inline int fit_class(const FitBlocks& b, int W) { return fit_few(b) ? 0 : W <= 64 ? 1 : 2; }

// One adjoint workgroup: parts [part, part + parts) of one strip of a problem. A part's
// sums are the same whichever workgroup takes it; a workgroup of several parts sets the
// strip's tables up once, and takes parts of fewer tiles than it has wavefronts side by
// side.
struct FitUnit {
  int problem, strip, part, parts;
};

// One problem of a batch as the kernels see it. Device pointers are owned by the
// wt_fit handle except params and target, which the caller owns.
struct FitDesc {
  double spacing, x0, z0, t0, dt, g;
  const float* target;  // [S][n*n][3]
  float* params;        // [W][5] {A, L, alpha, Q, phi0}
  float* adam_m;        // [W*5]
  float* adam_v;        // [W*5]
  float* partials;      // [nblocks][W*5 + 1]: per-block sums of r . dd/dp and of |r|^2 / 2
  float* loss;          // [1] loss of the last evaluation
  int* step;            // [1] Adam step counter
  int n, S, W;
  int tile_pairs, tiles_per_block, blocks_per_strip, nblocks;  // FitBlocks
  long long reduce_offset;     // first block of this problem in the reduce grid
  long long param_out_offset;  // first parameter of this problem in a concatenated gradient
};

struct FitAdam {
  float lr, beta1, beta2, eps;
};

// Device tables of a batch: problems, adjoint units (grouped by class, class c at
// [class_begin[c], + class_blocks[c])), reduce block -> problem. At most two classes have
// units: that of up to 64 waves takes the few-waves units too. side: a stream beside the
// caller's on which the smaller class's launch runs (one's tail overlaps the other's
// blocks), forked and joined by events before the reduction; null for one class.
struct FitLaunch {
  const FitDesc* probs;
  const FitUnit* units;
  const int* reduce_prob;
  long long class_begin[kFitClasses];
  long long class_blocks[kFitClasses];
  long long reduce_blocks;
  bool mixed;  // class 1 holds units of few waves too
  hipStream_t side;
  hipEvent_t fork, join;
};

// mode 0: gradient + loss only (grad_out receives the concatenated gradients);
// mode 1: Adam step (the adjoint launch bumps each problem's step counter first).
hipError_t launch_fit_iteration(const FitLaunch& L, const FitAdam& adam, int mode, float* grad_out, float* loss_out,
                                hipStream_t st);

// Target of a problem from its own params (the hidden wave set) plus N(0, sigma) noise.
hipError_t launch_synthesize(const FitDesc& P, float* out, float sigma, unsigned long long seed, hipStream_t st);

// Zero n 32-bit words with a kernel (graph-capture safe).
hipError_t launch_zero_words(uint32_t* p, size_t n, hipStream_t st);

// Writes one problem's descriptor (passed by value) to d_desc, its units, one part each,
// to d_units, and zeroes zero_words 32-bit words at zero_begin (the row map, Adam state,
// loss and step counter), in one kernel: the set-up of a single-problem evaluation in
// memory the caller did not allocate per call.
hipError_t launch_fit_setup_single(const FitDesc& d, FitDesc* d_desc, FitUnit* d_units, size_t units,
                                   uint32_t* zero_begin, size_t zero_words, hipStream_t st);

// The device address of this library's fixed single-problem fit scratch on `device`
// (resolved once per device, with that device current), or null with a message.
void* static_fit_scratch(int device, std::string* error);
// Its size in bytes.
size_t static_fit_scratch_bytes();

}  // namespace wt
