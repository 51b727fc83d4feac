// Kernel argument blocks and launchers shared between the C-ABI layer and the kernels.
#pragma once

#include <hip/hip_runtime.h>

#include "wt_device.hpp"

namespace wt {

// Plain forward: one frame of one grid. Corner algebra in FP64:
// P(u, v) = BL + u (BR - BL) + v (TL - BL) + u v (TR - TL - BR + BL), the expanded form of
// mix(mix(BL, BR, u), mix(TL, TR, u), v) (water-grid.vert:87-91).
struct FwdParams {
  double bl_x, bl_z;
  double du_x, du_z;    // BR - BL
  double dv_x, dv_z;    // TL - BL
  double duv_x, duv_z;  // TR - TL - BR + BL
  double inv_nm1;       // 1 / (gridLength - 1)
  double time;
  int N, W;
  const wt_gerstner_wave* waves;
  EpilogueArgs ep;
};

struct LaunchShape {
  int split;          // S: wavefronts sharing a block of vertices, 1 or 2
  int steps;          // K: 4, 8, 16
  int lanes_per_row;  // LC: 64, 32, 16, 8
  int wave_chunk;     // waves per LDS pass (64 in this build)
  bool own = false;   // the library's own choice for the size: segments may be taken in halves
};

hipError_t launch_forward(const FwdParams& p, const LaunchShape& s, hipStream_t st);

// One patch of a batch on the device: the corner algebra of FwdParams, set on the host
// at batch creation or by the device projector (launch_projector).
struct PatchDesc {
  double bl_x, bl_z, du_x, du_z, dv_x, dv_z, duv_x, duv_z, inv_nm1;
  double time;
  float cam[3];
  float s_h, s_d, bounce, scroll_x, scroll_z;
  int N, W, wave_offset;
  int shape;                // segment shape of this patch in the batched kernel (kBatchShapes)
  long long vertex_offset;  // first vertex of the patch in the output arrays
  int active;               // 0: the patch's camera misses the water; its units write nothing
  // units [0, whole_groups) are of whole segments, whole_per_row to a row; the others of
  // the half segments that end the rows where their upper halves have no columns (row_cut;
  // 256 patches of sides 17 to 40: 15.0 -> 12.3 us). A batch's units fill the card, so
  // segments with columns in both halves stay whole: all in halves, 64 patches of sides 60
  // to 130 took 35.8 us against 30.9
  int whole_groups, whole_per_row;
};

// Corner algebra of a grid from its corners [4][4] (BL, TL, BR, TR; x and z used).
template <class D>
__host__ __device__ inline void set_corner_algebra(D& d, const double (*c)[4]) {
  d.bl_x = c[0][0];
  d.bl_z = c[0][2];
  d.du_x = c[2][0] - c[0][0];
  d.du_z = c[2][2] - c[0][2];
  d.dv_x = c[1][0] - c[0][0];
  d.dv_z = c[1][2] - c[0][2];
  d.duv_x = c[3][0] - c[1][0] - c[2][0] + c[0][0];
  d.duv_z = c[3][2] - c[1][2] - c[2][2] + c[0][2];
}

// Launches of up to this many workgroups whose shape is the library's own choice take
// segments of 8 steps and two wavefronts in halves of 4 steps, a pair of wavefronts each: they leave SIMDs idle, and a wavefront's
// chain of sums and vertices, which bounds them, is about half as long (the upper half
// repeats the lower one's sequence). Above, the repeated work costs more than the idle
// SIMDs. Whole / in halves, us per launch in a graph: 128 x 128 with 16 waves 5.9 / 5.1,
// 256 x 256 with 100 waves 16.4 / 13.1, 513 x 513 with 64 waves (513 workgroups) 17.0 / 15.0,
// 600 x 600 with 100 waves (600) 26.2 / 22.7; 700 x 700 with 100 waves (700) 28.0 / 28.8. Per
// launch with two frames in flight: 4.9 / 4.7, 9.9 / 8.0, 10.4 / 9.7, 16.2 / 15.7, and 512 x 512
// with 100 waves (256) 10.2 / 10.3; with three, 512 x 512 loses (8.4 / 9.7): what
// wt_autotune_forward_overlapped is for, which times whole segments too.
constexpr long long kHalvesBlocks = 640;

// Past that, rows that end in the lower half of a segment end in half segments
// (water_forward_tail_kernel), with these exceptions, where the sums past the edge, which
// the halves save, cost less than what they bring along. Per launch in a graph, with halves
// over whole:
// - up to kOneRoundBlocks workgroups, four to a CU, a map and few waves: all of whole segments
//   run at once there, and a second kind of workgroup is only more of them. 768 x 768 with 1
//   wave 9.6 / 9.3 us, 16 waves 10.9 / 10.1, 32 waves 12.5 / 12.6, 64 waves 16.3 / 18.6 (without
//   a map 5.9 / 6.3, 8.1 / 8.9 and 10.9 / 11.9: halves); 1025 x 1025 (1538
//   workgroups) with 1 wave 14.9 / 16.3, 16 waves 17.6 / 18.3.
// - few waves, bound by the stores: a row's end is then stored by another workgroup at
//   another time. Without a map and 3 or 4 outputs 1.03-1.11 up to 8 and 16 waves; where rows
//   are no whole 64-byte pieces, so that the two also share one, up to 12 and 24 waves
//   1.04-1.22 (2 outputs, sides past 1536: 1.00-1.10 up to 4 waves). Beyond these 0.89-0.97.
//   With a map, whose texels past the edge the halves save too, 0.86-1.03, but 4 outputs at
//   sides past 2048 in shared pieces 1.02-1.17 from 8 to 16 waves.
constexpr long long kOneRoundBlocks = 1024;
constexpr int kRowEndWaves = 32;
inline bool rows_end_in_halves(long long blocks, int N, int W, bool map, int outputs) {
  if (blocks <= kOneRoundBlocks) return !map || W >= kRowEndWaves;
  const bool pieces = N % 16 == 0;
  if (map) return pieces || outputs < 4 || N <= 2048 || W >= 24;
  return W >= 12 * (outputs - 2) && (pieces || W >= (8 << (outputs - 2)) || (outputs == 2 && N <= 1536));
}

// How the rows of a grid are cut in a shape of two wavefronts per segment: whole segments,
// and half segments at the rows' ends where the upper halves have no columns. Workgroups
// take two segments of either kind.
struct RowCut {
  int whole_per_row;
  long long whole_groups, end_groups;
};
inline RowCut row_cut(int N, const LaunchShape& s) {
  const int columns = s.lanes_per_row * s.steps, tail = N % columns;
  const long long rows = (N + 64 / s.lanes_per_row - 1) / (64 / s.lanes_per_row);
  const bool half = tail > 0 && tail <= columns / 2;
  RowCut c;
  c.whole_per_row = N / columns + (tail > 0 && !half ? 1 : 0);
  c.whole_groups = (c.whole_per_row * rows + 1) / 2;
  c.end_groups = half ? (rows + 1) / 2 : 0;
  return c;
}

// One workgroup's segment group of one patch.
struct BatchUnit {
  int patch;
  int group;
};

struct BatchArgs {
  const PatchDesc* patches;
  const BatchUnit* units;  // every unit of the batch
  long long unit_begin;    // this launch's units: [unit_begin, unit_begin + n_units)
  int n_units;
  double time_offset;  // added to every patch's time (frame clock)
  const wt_gerstner_wave* waves;
  const void* texels;
  int tex_w, tex_h, tex_fmt, tex_wrap;
  float* pos;
  float* nrm;
  float* tan;
  float* bit;
};

// Varyings pass (wt_vertex_varyings): one thread per vertex.
struct VaryingArgs {
  float vp[16];    // viewProjection, column-major
  float vyaw[16];  // viewMatOnlyYaw, column-major
  float cam[3];
  float s_h;
  double hm_off_s, hm_off_t;  // scroll offsets reduced to one wrap period
  const void* texels;
  int tex_w, tex_h, tex_fmt, tex_wrap;
  const float* pos;
  const float* nrm;
  long long count;
  float* clip;
  float* ndc0;
  float* view;
  float* nview;
  float* sample;
};
hipError_t launch_varyings(const VaryingArgs& a, hipStream_t st);

// Segment shapes the batched kernel chooses from, per patch (all K = 8, S = 2): 512 x 1
// for wide grids, 256 x 2 and 128 x 4 for narrower ones.
constexpr int kBatchShapes = WT_BATCH_SHAPES;
constexpr LaunchShape kBatchShape[kBatchShapes] = {{2, 8, 64, 64}, {2, 8, 32, 64}, {2, 8, 16, 64}};
// The shape with the fewest padded vertices for a grid of side N (ties to the wider
// shape).
int batch_shape_for(int N);

// Device projector: the reference projector in FP64 for every camera.
// corners (count x 16, row = corner BL, TL, BR, TR) and status (wt_status per camera)
// may be null; with patches set, patch i takes camera i's corner algebra and camera
// position and is switched off when its status is not WT_OK.
struct ProjectorArgs {
  const wt_camera* cameras;
  const float* amplitudes;
  int count;
  double* corners;
  int* status;
  PatchDesc* patches;
};
hipError_t launch_projector(const ProjectorArgs& a, hipStream_t st);

// Triangle index list of an n x n grid (n >= 2), 6 (n - 1)^2 entries, ids offset by base.
hipError_t launch_grid_indices(uint32_t n, uint32_t base, uint32_t* out, hipStream_t st);

// Launches the batched kernel, one workgroup per unit of a.
hipError_t launch_forward_batched(const BatchArgs& a, hipStream_t st);

// Fragment stage (wt_water_shade): the water program's fragment shader over a
// per-pixel fragment buffer. RGBA8 images are read as one 32-bit word per texel.
struct ShadeArgs {
  float fog[4];  // fogColourFarAtCurrentTime
  float fog_far, fog_near;
  float inv_fog_range;  // 1 / (fogDepthRadiusFar - fogDepthRadiusNear), used only between the radii
  int tint_off, soft_off;   // tintDeltaDepthThreshold / softEdgesDeltaDepthThreshold == 0
  float inv_tint, inv_soft;  // their reciprocals otherwise
  float sun[3];
  float shininess, strength, clarity, zfar, znear;
  float zfar_m_znear, inv_zfar;
  float inv_viewport_w, inv_viewport_h;  // 1 / viewportWidthHeight
  const float* depth;
  int depth_w, depth_h;
  const unsigned* refl;
  int refl_w, refl_h;
  const unsigned* refr;
  int refr_w, refr_h;
  const unsigned* sky;  // six faces, sky_len^2 texels each
  int sky_len;
  const float4* frags;  // three float4 per pixel
  const unsigned char* coverage;
  float4* colour;
  int width, count;  // count = width x height <= 2^30
  int blend;
};
hipError_t launch_shade(const ShadeArgs& a, hipStream_t st);

}  // namespace wt
