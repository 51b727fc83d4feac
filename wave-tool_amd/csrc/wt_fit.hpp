// Device descriptors of the heightfield-fit problems and the launcher shared by the
// C ABI and the adjoint kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <string>

#include "wt_device.hpp"

namespace wt {

constexpr int kFitMaxWaves = 128;
constexpr int kFitMaxSnapshots = 32;
// The reduction: blocks of 16 rows (parameters, and the loss), 16 wavefronts of four parts
// each side by side.
constexpr int kReduceRows = 16, kReduceThreads = 1024;
inline int reduce_blocks(int W) { return (5 * W + 1 + kReduceRows - 1) / kReduceRows; }
// Wave-count classes W <= 64 and W <= 128: the chunks of 16 waves the adjoint kernel's LDS
// has room for. From 65 waves on the time table does not fit beside the rest.
constexpr int kFitClasses = 2;
constexpr int kFitClassChunks[kFitClasses] = {4, 8};
constexpr int kFitWavefronts = 8;  // of an adjoint workgroup: two per SIMD, sharing the tables
inline int fit_class(int W) { return W <= 64 ? 0 : 1; }
// How a problem's work is cut into adjoint blocks: strips of columns, and per strip runs
// of tiles of 16 (row, snapshot) pairs. It depends on the problem alone.
struct FitBlocks {
  int tiles_per_block, blocks_per_strip, nblocks;
};
inline FitBlocks fit_blocks(int n, int S) {
  const long long strips = (n + 63) / 64, tiles = ((long long)n * S + 15) / 16;
  // enough tiles per wavefront to pay for a block's set-up; a problem too small to fill
  // the GPU's wavefronts that way is cut into parts of 4, 2 or 1 tiles, about one for each
  // CU, and each tile then has more of a CU's load path to itself: the eight tiles of a
  // workgroup took 3.5 us to fetch on one CU (64 x 64, 8 snapshots, 16 waves: 14.0 us an
  // iteration with 4 parts of 8 tiles, 11.3 with 32 of one; 256 x 256, 16 snapshots, 64
  // waves: 23.0 with 128 of 8, 19.5 with 256 of 4)
  const long long total = strips * tiles;
  long long per_block = (total + 2047) / 2048 * kFitWavefronts;
  if (per_block > 8 * kFitWavefronts) per_block = 8 * kFitWavefronts;
  for (; per_block > 1 && total <= per_block * 128; per_block /= 2) {
  }
  FitBlocks b;
  b.tiles_per_block = (int)per_block;
  b.blocks_per_strip = (int)((tiles + b.tiles_per_block - 1) / b.tiles_per_block);
  b.nblocks = (int)(strips * b.blocks_per_strip);
  return b;
}

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
  int tiles_per_block, blocks_per_strip, nblocks;  // FitBlocks
  long long reduce_offset;     // first block of this problem in the reduce grid
  long long param_out_offset;  // first parameter of this problem in a concatenated gradient
};

struct FitAdam {
  float lr, beta1, beta2, eps;
};

// Device tables of a batch: problems, adjoint units (grouped by wave-count class, class c
// at [class_begin[c], + class_blocks[c])), reduce block -> problem.
// Streams beside the caller's on which the classes' adjoint launches run
// concurrently (one class's tail overlaps the next class's blocks), joined by events
// before the reduction.
constexpr int kFitSideStreams = 3;

struct FitLaunch {
  const FitDesc* probs;
  const FitUnit* units;
  const int* reduce_prob;
  long long class_begin[kFitClasses];
  long long class_blocks[kFitClasses];
  long long reduce_blocks;
  hipStream_t side[kFitSideStreams];  // null: every class on the caller's stream
  hipEvent_t fork;
  hipEvent_t join[kFitSideStreams];
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
