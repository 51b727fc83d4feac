// C-ABI of the heightfield fit: problem tables, Adam iterations (single or batched),
// gradient evaluation, target synthesis and the phase-storage policy.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/wt.h"
#include "wt_fit.hpp"

struct wt_ctx;

namespace wt {
wt_status ctx_fail(wt_ctx* ctx, wt_status s, const std::string& msg);
}

struct wt_fit {
  wt_ctx* ctx = nullptr;
  int count = 0;
  long long total_reduce = 0, total_params = 0;
  std::vector<wt::FitDesc> host;
  wt::FitDesc* d_desc = nullptr;
  wt::FitUnit* d_units = nullptr;
  int* d_rows = nullptr;    // reduce block -> problem
  char* d_state = nullptr;  // moments, partials, loss, step for every problem
  size_t state_bytes = 0;
  wt::FitLaunch launch{};
};

namespace {

wt_status hip_err(wt_ctx* ctx, hipError_t e, const char* where) {
  return wt::ctx_fail(ctx, WT_ERR_HIP, std::string(where) + ": " + hipGetErrorString(e));
}

bool problem_ok(const wt_fit_problem& p, std::string* why) {
  if (p.grid_side < 1 || p.grid_side > 8192) return *why = "grid_side must be in [1, 8192]", false;
  if (p.snapshots < 1 || p.snapshots > (uint32_t)wt::kFitMaxSnapshots) return *why = "snapshots must be in [1, 32]", false;
  if (p.wave_count < 1 || p.wave_count > (uint32_t)wt::kFitMaxWaves) return *why = "wave_count must be in [1, 128]", false;
  const double v[6] = {p.spacing, p.x0, p.z0, p.t0, p.dt, p.gravity};
  for (double x : v)
    if (!std::isfinite(x)) return *why = "problem scalars must be finite", false;
  if (!(p.spacing > 0.0) || !(p.gravity > 0.0)) return *why = "spacing and gravity must be positive", false;
  if (!p.target || !p.params) return *why = "target and params must be device pointers", false;
  return true;
}

}  // namespace

// ---------------------------------------------------------------- fixed scratch
// Device memory of wt_fit_loss_grad_static: one problem's descriptor, its block and row
// maps, Adam state it never steps, the loss, and the per-block partial sums, in a
// file-scope device array, so the entry point never allocates. Each device holds its own
// copy for the life of the process. Its address is resolved once per device with
// hipGetSymbolAddress (the array's name in host code is only a stand-in for the symbol);
// kernels receive that address.
namespace {

constexpr size_t kStaticFitScratchBytes = WT_FIT_STATIC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kStaticFitScratchBytes];

std::mutex g_scratch_mutex;
std::vector<void*> g_scratch_ptr;          // per device, once resolved
std::vector<std::string> g_scratch_error;  // per device, when resolving failed
std::vector<char> g_scratch_done;

constexpr size_t kStaticFitDescBytes = 144;  // of a problem's descriptor, as the limit counts it

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

// Layout of the scratch for a problem of `np` = 5 W parameters and `nblocks` adjoint
// blocks: descriptor | units | row map (np + 1 ints), m, v (np floats each), loss, step |
// partials ((np + 1) x nblocks floats). Returns the total bytes; offsets through the
// pointers.
size_t static_fit_layout(int np, int nblocks, size_t* units, size_t* rows, size_t* partials) {
  size_t off = align256(sizeof(wt::FitDesc));
  *units = off;
  off = align256(off + sizeof(wt::FitUnit) * (size_t)nblocks);
  *rows = off;
  off = align256(off + sizeof(float) * (3 * (size_t)np + 3));
  *partials = off;
  return off + sizeof(float) * (size_t)(np + 1) * nblocks;
}

// The bytes the entry point's documented limit counts, in blocks of 256 grid points (512
// for S <= 8): descriptor, maps, state and partials of that many blocks. The adjoint's own
// parts need less wherever this is near the limit.
size_t static_fit_limit(const wt_fit_problem& p) {
  const size_t V = (size_t)p.grid_side * p.grid_side, np = 5 * (size_t)p.wave_count;
  const size_t points = p.snapshots <= 8 ? 512 : 256, blocks = (V + points - 1) / points;
  size_t off = align256(kStaticFitDescBytes);
  off = align256(off + sizeof(int) * (blocks + np + 1));
  off = align256(off + sizeof(float) * (2 * np + 2));
  return off + sizeof(float) * (np + 1) * blocks;
}

}  // namespace

namespace wt {

size_t static_fit_scratch_bytes() { return kStaticFitScratchBytes; }

void* static_fit_scratch(int device, std::string* error) {
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (device < 0) {
    *error = "invalid device";
    return nullptr;
  }
  if ((size_t)device >= g_scratch_done.size()) {
    g_scratch_ptr.resize(device + 1, nullptr);
    g_scratch_error.resize(device + 1);
    g_scratch_done.resize(device + 1, 0);
  }
  if (!g_scratch_done[device]) {
    int cur = -1;
    hipError_t e = hipGetDevice(&cur);
    if (e == hipSuccess && cur != device) e = hipSetDevice(device);
    void* ptr = nullptr;
    if (e == hipSuccess) e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e == hipSuccess && !ptr) e = hipErrorInvalidSymbol;
    if (e == hipSuccess) {
      g_scratch_ptr[device] = ptr;
    } else {
      g_scratch_error[device] = std::string("fixed fit scratch: ") + hipGetErrorString(e);
    }
    if (cur >= 0 && cur != device) (void)hipSetDevice(cur);
    g_scratch_done[device] = 1;
  }
  if (!g_scratch_ptr[device]) *error = g_scratch_error[device];
  return g_scratch_ptr[device];
}

}  // namespace wt

extern "C" {

wt_status wt_fit_create(wt_ctx* ctx, const wt_fit_problem* problems, uint32_t count, wt_fit** out) {
  if (!ctx || !out) return WT_ERR_INVALID_ARG;
  *out = nullptr;
  if (!problems || count == 0) return wt::ctx_fail(ctx, WT_ERR_INVALID_ARG, "need at least one problem");
  wt_fit* f = new (std::nothrow) wt_fit();
  if (!f) return WT_ERR_OOM;
  f->ctx = ctx;
  f->count = (int)count;
  f->host.resize(count);
  // state layout per problem: m[W*5], v[W*5], partials[(W*5+1)*nblocks], loss, step
  std::vector<size_t> off(count);
  size_t bytes = 0;
  long long rounds = 0, parts = 0;  // tiles per wavefront over all blocks, and the blocks
  for (uint32_t i = 0; i < count; ++i) {
    std::string why;
    if (!problem_ok(problems[i], &why)) {
      delete f;
      return wt::ctx_fail(ctx, WT_ERR_INVALID_ARG, "problem " + std::to_string(i) + ": " + why);
    }
    const wt_fit_problem& p = problems[i];
    const wt::FitBlocks fb = wt::fit_blocks((int)p.grid_side, (int)p.snapshots, (int)p.wave_count);
    const int nblocks = fb.nblocks;
    const int np = (int)p.wave_count * 5;
    wt::FitDesc& d = f->host[i];
    d.spacing = p.spacing;
    d.x0 = p.x0;
    d.z0 = p.z0;
    d.t0 = p.t0;
    d.dt = p.dt;
    d.g = p.gravity;
    d.target = p.target;
    d.params = p.params;
    d.n = (int)p.grid_side;
    d.S = (int)p.snapshots;
    d.W = (int)p.wave_count;
    d.tile_pairs = fb.tile_pairs;
    d.tiles_per_block = fb.tiles_per_block;
    d.blocks_per_strip = fb.blocks_per_strip;
    d.nblocks = nblocks;
    d.reduce_offset = f->total_reduce;
    d.param_out_offset = f->total_params;
    rounds += ((long long)nblocks * fb.tiles_per_block + wt::kFitWavefronts - 1) / wt::kFitWavefronts;
    parts += nblocks;
    f->total_reduce += wt::reduce_blocks(d.W);
    f->total_params += np;
    off[i] = bytes;
    bytes += sizeof(float) * ((size_t)2 * np + (size_t)(np + 1) * nblocks + 1) + sizeof(int);
    bytes = (bytes + 255) & ~(size_t)255;
  }
  // adjoint units by class, the longest first (the dispatcher starts workgroups in index
  // order). A workgroup takes several parts of a strip where the batch has many more parts
  // than the GPU has room for workgroups (256 CUs, one or two on each, four of the
  // few-waves kernel), so that setting the strip's tables up is paid for by several rounds
  // of tiles. Problems of few waves beside ones of up to 64 go with these, whose kernel
  // takes both: a launch more, forked and joined, costs more than they do in any small
  // batch (24 problems of sides to 64 with 2-16 waves 29 us, so 19).
  const long long unit_rounds = std::min<long long>(16, std::max<long long>(1, rounds / 2048));
  auto own_class = [&](const wt::FitDesc& d) {
    return wt::fit_class(wt::FitBlocks{d.tile_pairs, d.tiles_per_block, d.blocks_per_strip, d.nblocks}, d.W);
  };
  const bool matrix = std::any_of(f->host.begin(), f->host.end(), [&](const wt::FitDesc& d) { return own_class(d) == 1; });
  std::vector<wt::FitUnit> units;
  long long unit_begin = 0;
  for (int c = 0; c < wt::kFitClasses; ++c) {
    for (uint32_t i = 0; i < count; ++i) {
      const wt::FitDesc& d = f->host[i];
      const int own = own_class(d);
      if ((own == 0 && matrix ? 1 : own) != c) continue;
      f->launch.mixed |= own != c;
      int per;
      if (own == 0) {
        // beside others two at a time, in a workgroup that has the CU to itself
        per = (int)(matrix ? 2 * std::min<long long>(8, std::max<long long>(1, parts / 512))
                           : std::min<long long>(16, (parts + 1023) / 1024));
      } else {
        // parts that run side by side share a workgroup once every CU has one
        const int side_by = std::max(1, wt::kFitWavefronts / d.tiles_per_block);
        const int part_rounds = std::max(1, d.tiles_per_block / wt::kFitWavefronts);
        per = unit_rounds > 1 ? (int)std::max<long long>(1, unit_rounds / part_rounds) * side_by
                              : (int)std::min<long long>(side_by, std::max<long long>(1, parts / 256));
      }
      const int strips = d.nblocks / d.blocks_per_strip;
      for (int st = 0; st < strips; ++st)
        for (int b = 0; b < d.blocks_per_strip; b += per)
          units.push_back(wt::FitUnit{(int)i, st, b, std::min(per, d.blocks_per_strip - b)});
      if (units.size() >= (1ull << 31)) break;
    }
    std::stable_sort(units.begin() + unit_begin, units.end(), [&](const wt::FitUnit& x, const wt::FitUnit& y) {
      auto pairs = [&](const wt::FitUnit& u) {
        return (long long)u.parts * f->host[u.problem].tiles_per_block * f->host[u.problem].tile_pairs;
      };
      return pairs(x) > pairs(y);
    });
    f->launch.class_begin[c] = unit_begin;
    f->launch.class_blocks[c] = (long long)units.size() - unit_begin;
    unit_begin = (long long)units.size();
  }
  if (units.size() >= (1ull << 31) || f->total_reduce >= (1ll << 31)) {
    delete f;
    return wt::ctx_fail(ctx, WT_ERR_UNSUPPORTED, "batch too large for one launch");
  }
  hipError_t e = hipMalloc(&f->d_state, bytes);
  if (e != hipSuccess) {
    delete f;
    return wt::ctx_fail(ctx, WT_ERR_OOM, "fit state allocation");
  }
  f->state_bytes = bytes;
  for (uint32_t i = 0; i < count; ++i) {
    wt::FitDesc& d = f->host[i];
    const int np = d.W * 5;
    float* base = reinterpret_cast<float*>(f->d_state + off[i]);
    d.adam_m = base;
    d.adam_v = base + np;
    d.partials = base + 2 * np;
    d.loss = d.partials + (size_t)(np + 1) * d.nblocks;
    d.step = reinterpret_cast<int*>(d.loss + 1);
  }
  std::vector<int> rows((size_t)f->total_reduce);
  for (uint32_t i = 0; i < count; ++i) {
    const wt::FitDesc& d = f->host[i];
    for (int r = 0; r < wt::reduce_blocks(d.W); ++r) rows[(size_t)d.reduce_offset + r] = (int)i;
  }
  e = hipMalloc(&f->d_desc, sizeof(wt::FitDesc) * count);
  if (e == hipSuccess) e = hipMalloc(&f->d_units, sizeof(wt::FitUnit) * units.size());
  if (e == hipSuccess) e = hipMalloc(&f->d_rows, sizeof(int) * rows.size());
  if (e == hipSuccess) e = hipMemcpy(f->d_desc, f->host.data(), sizeof(wt::FitDesc) * count, hipMemcpyHostToDevice);
  if (e == hipSuccess)
    e = hipMemcpy(f->d_units, units.data(), sizeof(wt::FitUnit) * units.size(), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(f->d_rows, rows.data(), sizeof(int) * rows.size(), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemset(f->d_state, 0, bytes);
  if (e == hipSuccess) e = hipDeviceSynchronize();
  if (e != hipSuccess) {
    wt_status s = hip_err(ctx, e, "wt_fit_create");
    wt_fit_destroy(f);
    return s;
  }
  f->launch.probs = f->d_desc;
  f->launch.units = f->d_units;
  f->launch.reduce_prob = f->d_rows;
  f->launch.reduce_blocks = f->total_reduce;
  // the side stream (default priority, not synchronising with the null stream) and its
  // fork / join events, for batches of two classes
  int classes = 0;
  for (int c = 0; c < wt::kFitClasses; ++c) classes += f->launch.class_blocks[c] > 0;
  if (classes > 1) {
    e = hipEventCreateWithFlags(&f->launch.fork, hipEventDisableTiming);
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&f->launch.side, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&f->launch.join, hipEventDisableTiming);
    if (e != hipSuccess) {
      wt_status s = hip_err(ctx, e, "wt_fit_create stream");
      wt_fit_destroy(f);
      return s;
    }
  }
  *out = f;
  return WT_OK;
}

void wt_fit_destroy(wt_fit* f) {
  if (!f) return;
  if (f->launch.side) (void)hipStreamDestroy(f->launch.side);
  if (f->launch.join) (void)hipEventDestroy(f->launch.join);
  if (f->launch.fork) (void)hipEventDestroy(f->launch.fork);
  if (f->d_desc) (void)hipFree(f->d_desc);
  if (f->d_units) (void)hipFree(f->d_units);
  if (f->d_rows) (void)hipFree(f->d_rows);
  if (f->d_state) (void)hipFree(f->d_state);
  delete f;
}

wt_status wt_fit_reset(wt_fit* f, void* stream) {
  if (!f) return WT_ERR_INVALID_ARG;
  // a fill kernel rather than hipMemsetAsync, so the reset may sit inside a captured graph
  hipError_t e = wt::launch_zero_words(reinterpret_cast<uint32_t*>(f->d_state), f->state_bytes / 4, (hipStream_t)stream);
  return e == hipSuccess ? WT_OK : hip_err(f->ctx, e, "wt_fit_reset");
}

wt_status wt_fit_iterate(wt_fit* f, const wt_adam_config* adam, uint32_t iterations, float* d_losses, void* stream) {
  if (!f || !adam) return WT_ERR_INVALID_ARG;
  if (!(adam->lr > 0.0f) || !(adam->beta1 >= 0.0f && adam->beta1 < 1.0f) || !(adam->beta2 >= 0.0f && adam->beta2 < 1.0f) ||
      !(adam->eps > 0.0f))
    return wt::ctx_fail(f->ctx, WT_ERR_INVALID_ARG, "Adam settings out of range");
  const wt::FitAdam a{adam->lr, adam->beta1, adam->beta2, adam->eps};
  for (uint32_t it = 0; it < iterations; ++it) {
    hipError_t e = wt::launch_fit_iteration(f->launch, a, 1, nullptr, d_losses, (hipStream_t)stream);
    if (e != hipSuccess) return hip_err(f->ctx, e, "fit iteration launch");
  }
  return WT_OK;
}

wt_status wt_fit_loss_grad(wt_fit* f, float* d_grad, float* d_losses, void* stream) {
  if (!f || !d_grad) return WT_ERR_INVALID_ARG;
  const wt::FitAdam a{0.0f, 0.0f, 0.0f, 0.0f};
  hipError_t e = wt::launch_fit_iteration(f->launch, a, 0, d_grad, d_losses, (hipStream_t)stream);
  return e == hipSuccess ? WT_OK : hip_err(f->ctx, e, "fit gradient launch");
}

wt_status wt_fit_loss_grad_static(wt_ctx* ctx, const wt_fit_problem* p, float* d_grad, float* d_loss, void* stream) {
  if (!ctx || !p || !d_grad) return WT_ERR_INVALID_ARG;
  std::string why;
  if (!problem_ok(*p, &why)) return wt::ctx_fail(ctx, WT_ERR_INVALID_ARG, why);
  const wt::FitBlocks fb = wt::fit_blocks((int)p->grid_side, (int)p->snapshots, (int)p->wave_count);
  const int cls = wt::fit_class(fb, (int)p->wave_count);
  const long long nblocks = fb.nblocks;
  const int np = (int)p->wave_count * 5;
  size_t off_units = 0, off_rows = 0, off_partials = 0;
  const size_t need =
      std::max(static_fit_limit(*p), static_fit_layout(np, (int)nblocks, &off_units, &off_rows, &off_partials));
  if (need > kStaticFitScratchBytes)
    return wt::ctx_fail(ctx, WT_ERR_INVALID_ARG,
                        "problem needs " + std::to_string(need) + " bytes of fixed scratch; the limit is " +
                            std::to_string(kStaticFitScratchBytes) + " (fewer grid points or waves, or wt_fit_create)");
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return hip_err(ctx, e, "wt_fit_loss_grad_static");
  void* base = wt::static_fit_scratch(dev, &why);
  if (!base) return wt::ctx_fail(ctx, WT_ERR_HIP, why);
  char* b = static_cast<char*>(base);
  wt::FitDesc d{};
  d.spacing = p->spacing;
  d.x0 = p->x0;
  d.z0 = p->z0;
  d.t0 = p->t0;
  d.dt = p->dt;
  d.g = p->gravity;
  d.target = p->target;
  d.params = p->params;
  int* rows = reinterpret_cast<int*>(b + off_rows);
  float* state = reinterpret_cast<float*>(rows + np + 1);
  d.adam_m = state;
  d.adam_v = state + np;
  d.loss = state + 2 * np;
  d.step = reinterpret_cast<int*>(state + 2 * np + 1);
  d.partials = reinterpret_cast<float*>(b + off_partials);
  d.n = (int)p->grid_side;
  d.S = (int)p->snapshots;
  d.W = (int)p->wave_count;
  d.tile_pairs = fb.tile_pairs;
  d.tiles_per_block = fb.tiles_per_block;
  d.blocks_per_strip = fb.blocks_per_strip;
  d.nblocks = (int)nblocks;
  d.reduce_offset = 0;
  d.param_out_offset = 0;
  const hipStream_t st = (hipStream_t)stream;
  wt::FitDesc* d_desc = reinterpret_cast<wt::FitDesc*>(b);
  wt::FitUnit* d_units = reinterpret_cast<wt::FitUnit*>(b + off_units);
  // the previous call's contents stay in the array: rewrite the descriptor and units and
  // clear the row map (problem 0) and the state words; every partial is overwritten by
  // the adjoint launch
  e = wt::launch_fit_setup_single(d, d_desc, d_units, (size_t)nblocks, reinterpret_cast<uint32_t*>(rows),
                                  3 * (size_t)np + 3, st);
  if (e != hipSuccess) return hip_err(ctx, e, "fixed-scratch set-up launch");
  wt::FitLaunch L{};
  L.probs = d_desc;
  L.units = d_units;
  L.reduce_prob = rows;
  L.class_begin[cls] = 0;
  L.class_blocks[cls] = nblocks;
  L.reduce_blocks = wt::reduce_blocks(d.W);
  const wt::FitAdam a{0.0f, 0.0f, 0.0f, 0.0f};
  e = wt::launch_fit_iteration(L, a, 0, d_grad, d_loss, st);
  return e == hipSuccess ? WT_OK : hip_err(ctx, e, "fit gradient launch");
}

wt_status wt_fit_synthesize(wt_ctx* ctx, const wt_fit_problem* p, float sigma, uint64_t seed, float* d_target,
                            void* stream) {
  if (!ctx || !p || !d_target) return WT_ERR_INVALID_ARG;
  wt_fit_problem q = *p;
  q.target = d_target;
  std::string why;
  if (!problem_ok(q, &why)) return wt::ctx_fail(ctx, WT_ERR_INVALID_ARG, why);
  if (!(sigma >= 0.0f) || !std::isfinite(sigma)) return wt::ctx_fail(ctx, WT_ERR_INVALID_ARG, "sigma must be >= 0");
  wt::FitDesc d{};
  d.spacing = q.spacing;
  d.x0 = q.x0;
  d.z0 = q.z0;
  d.t0 = q.t0;
  d.dt = q.dt;
  d.g = q.gravity;
  d.params = q.params;
  d.n = (int)q.grid_side;
  d.S = (int)q.snapshots;
  d.W = (int)q.wave_count;
  hipError_t e = wt::launch_synthesize(d, d_target, sigma, (unsigned long long)seed, (hipStream_t)stream);
  return e == hipSuccess ? WT_OK : hip_err(ctx, e, "synthesize launch");
}

wt_status wt_fit_phase_plan(const wt_fit_problem* p, uint64_t budget_bytes, uint64_t* phase_tensor_bytes,
                            int* recompute) {
  if (!p || !phase_tensor_bytes || !recompute) return WT_ERR_INVALID_ARG;
  const uint64_t V = (uint64_t)p->grid_side * p->grid_side;
  // (cos, sin) per snapshot x grid point x wave in FP32
  *phase_tensor_bytes = V * p->snapshots * p->wave_count * 8ull;
  // The kernels contract separable factors of (cos, sin), W (n + 64) values per row and
  // column where the tensor has S n^2 W: nothing is gained by storing it at any size. The
  // tensor size is reported so callers can see what storing would need against their
  // budget.
  (void)budget_bytes;
  *recompute = 1;
  return WT_OK;
}

}  // extern "C"
