// Device projector: the reference's per-frame projector (src/render-engine.cpp:797-1042)
// for many cameras at once, in FP64. It writes corners, a status per camera, and/or
// re-aims the patches of a batch in place so a captured frame loop recomputes every
// patch's grid without a host round trip.
//
// One camera is a serial chain of FP64 divisions, square roots and trigonometry: its
// latency bounds small counts. Up to kWaveProjectorCameras cameras get a wavefront each,
// whose lanes take the parts that do not depend on each other (both inverses at once with
// a column per lane, the frustum corners, edges and grid corners, the trigonometry of yaw
// and pitch): a third of the instructions. Past that every SIMD has work either way and a
// thread per camera does less in all. Every value is formed by the same operations in
// both, so they agree bit for bit. Measured per launch in a graph, wavefront / thread per
// camera: 24 cameras 7.5 / 15.0 us, 512 8.2 / 15.1, 2048 11.6 / 15.2, 4096 20.0 / 15.2.
#include "wt_kernels.hpp"
#include "wt_projector.hpp"

namespace wt {

constexpr int kWaveProjectorCameras = 2048;

// ------------------------------------------------------------------ a thread per camera
constexpr int kProjectorThreads = 64;

__global__ __launch_bounds__(kProjectorThreads) void projector_kernel(ProjectorArgs a) {
  const int i = (int)blockIdx.x * kProjectorThreads + (int)threadIdx.x;
  if (i >= a.count) return;
  const wt_camera cam = a.cameras[i];
  const float amp = a.amplitudes[i];
  double c[4][4];
  int st = WT_ERR_INVALID_ARG;
  if (proj::camera_valid(cam) && __builtin_isfinite(amp) && amp >= 0.0f)
    st = proj::projector_corners(proj::camera_from(cam), (double)amp, c);
  if (a.corners) {
    double* o = a.corners + 16 * (size_t)i;
    for (int k = 0; k < 16; ++k) o[k] = st == WT_OK ? c[k / 4][k % 4] : __builtin_nan("");
  }
  if (a.status) a.status[i] = st;
  if (a.patches) {
    PatchDesc& d = a.patches[i];
    if (st == WT_OK) {
      set_corner_algebra(d, c);
      d.cam[0] = cam.position[0];
      d.cam[1] = cam.position[1];
      d.cam[2] = cam.position[2];
    }
    d.active = st == WT_OK;
  }
}

// ------------------------------------------------------------------ a wavefront per camera
#pragma clang fp contract(off)

// v of lane `lane` (the same for the whole wavefront), as a uniform value.
__device__ __forceinline__ double lane_value(double v, int lane) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, lane);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), lane);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// v of another lane of the row of 16, by a DPP control.
template <int kCtrl>
__device__ __forceinline__ double dpp(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)b, kCtrl, 0xf, 0xf, false);
  const unsigned hi = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)(b >> 32), kCtrl, 0xf, 0xf, false);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// v of lane kLane of each row of 16 lanes (row_newbcast).
template <int kLane>
__device__ __forceinline__ double row_value(double v) {
  return dpp<0x150 | kLane>(v);
}

__device__ __forceinline__ double lesser(double a, double b) { return b < a ? b : a; }
__device__ __forceinline__ double greater(double a, double b) { return b > a ? b : a; }

// Least and greatest of v over the lanes 0-31 that are `in`, as NdcBounds forms them one by
// one: NaN is passed over, unless the first lane holds it. Rows of 16 by DPP (quad_perm
// neighbours and pairs, row_half_mirror, row_mirror), then the two rows.
__device__ __forceinline__ void bounds(double v, bool in, int first, double* least, double* most) {
  const bool use = in && v == v;
  double a = use ? v : __builtin_inf(), b = use ? v : -__builtin_inf();
  a = lesser(a, dpp<0xB1>(a));
  b = greater(b, dpp<0xB1>(b));
  a = lesser(a, dpp<0x4E>(a));
  b = greater(b, dpp<0x4E>(b));
  a = lesser(a, dpp<0x141>(a));
  b = greater(b, dpp<0x141>(b));
  a = lesser(a, dpp<0x140>(a));
  b = greater(b, dpp<0x140>(b));
  const double lead = lane_value(v, first);
  *least = lead == lead ? lesser(lane_value(a, 0), lane_value(a, 16)) : lead;
  *most = lead == lead ? greater(lane_value(b, 0), lane_value(b, 16)) : lead;
}

// The matrix whose column c lane first + c holds.
__device__ __forceinline__ proj::Mat4 gather_columns(const double (&col)[4], int first) {
  proj::Mat4 m;
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int r = 0; r < 4; ++r) m.c[c][r] = lane_value(col[r], first + c);
  return m;
}

// Component r of column c of m, c differing between lanes.
__device__ __forceinline__ double pick_column(const proj::Mat4& m, int c, int r) {
  const double a = c == 1 ? m.c[1][r] : m.c[0][r], b = c == 3 ? m.c[3][r] : m.c[2][r];
  return c < 2 ? a : b;
}

// Column of a * b (proj::mat_mul) for b's column b_col.
__device__ __forceinline__ void mul_column(const proj::Mat4& a, const double (&b_col)[4], double (&out)[4]) {
#pragma unroll
  for (int row = 0; row < 4; ++row) {
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < 4; ++k) s += a.c[k][row] * b_col[k];
    out[row] = s;
  }
}

// Step kP of proj::mat_inverse with column c of the augmented matrix [A | I] in lane c of
// each row of 16 lanes: only the pivot column goes between lanes. False for a singular A.
template <int kP>
__device__ __forceinline__ bool eliminate(double (&a)[4]) {
  double f[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) f[r] = row_value<kP>(a[r]);
  int best = kP;
  double big = fabs(f[kP]);
#pragma unroll
  for (int r = kP + 1; r < 4; ++r)
    if (fabs(f[r]) > big) {
      best = r;
      big = fabs(f[r]);
    }
#pragma unroll
  for (int r = kP + 1; r < 4; ++r) {
    const bool swap = r == best;
    const double t = a[kP], g = f[kP];
    a[kP] = swap ? a[r] : t;
    a[r] = swap ? t : a[r];
    f[kP] = swap ? f[r] : g;
    f[r] = swap ? g : f[r];
  }
  a[kP] *= 1.0 / f[kP];
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (r != kP) a[r] = f[r] == 0.0 ? a[r] : a[r] - f[r] * a[kP];
  return big != 0.0;
}

// Camera::set_rotation and ::update_basis, with the yaw's trigonometry in the even lanes
// and the pitch's in the odd ones.
__device__ __forceinline__ proj::Mat4 aimed_view(double yaw, double pitch, const proj::Vec3& position, int lane,
                                                 double* yaw_deg, proj::Vec3* forward) {
  *yaw_deg = proj::glsl_mod(yaw, 360.0);
  const double pitch_deg = pitch < -89.0 ? -89.0 : (pitch > 89.0 ? 89.0 : pitch);
  const double angle = proj::radians((lane & 1) ? pitch_deg : *yaw_deg);
  const double c = cos(angle), s = sin(angle);
  const double cy = lane_value(c, 0), sy = lane_value(s, 0), cp = lane_value(c, 1), sp = lane_value(s, 1);
  *forward = proj::unit(proj::Vec3{cy * cp, sp, sy * cp});
  const proj::Vec3 right = proj::unit(proj::cross3(*forward, proj::Vec3{0, 1, 0}));
  const proj::Vec3 up = proj::unit(proj::cross3(right, *forward));
  return proj::look_at_rh(position, proj::add(position, *forward), up);
}

// proj::projector_corners of proj::camera_from(c): corner i (BL, TL, BR, TR) in lane 2 i.
__device__ __forceinline__ int projector_corners_wave(const wt_camera& c, double amp, int lane, proj::Vec3* corner) {
  using namespace proj;
  const Mat4 persp = perspective_rh(radians(c.fov_deg), c.aspect, c.near_clip, c.far_clip);
  const Vec3 eye{c.position[0], c.position[1], c.position[2]};
  double yaw_deg;
  Vec3 forward;
  const Mat4 view = aimed_view(c.yaw_deg, c.pitch_deg, eye, lane, &yaw_deg, &forward);

  // the projector: lifted above the slab and aimed at y = 0; without an aim point its
  // view is not used
  Vec3 pj_eye = eye;
  const bool underwater = eye.y < 0.0;
  const double min_height = amp + 1.0;
  if (eye.y < min_height)
    pj_eye = add(eye, Vec3{0.0, underwater ? min_height - 2.0 * eye.y : min_height - eye.y, 0.0});
  Vec3 fwd = forward;
  const double eps = 0.001;
  if (fabs(fwd.y) < eps) fwd.y = (fwd.y >= 0.0 ? 1.0 : -1.0) * eps;
  const bool looking_down = fwd.y < 0.0;
  const Vec3 ray = (looking_down != underwater) ? fwd : Vec3{fwd.x, -fwd.y, fwd.z};
  Vec3 aim1{0, 0, 0};
  const bool aim_ok = hit_plane_y(eye, add(eye, ray), 0.0, &aim1);
  Vec3 aim2 = add(eye, forward);
  aim2.y = 0.0;
  const double ay = fabs(fwd.y);
  const Vec3 nf = unit(sub(add(scale(aim2, 1.0 - ay), scale(aim1, ay)), pj_eye));
  double cosine = dot3(nf, unit(Vec3{nf.x, 0.0, nf.z}));
  cosine = cosine > 1.0 ? 1.0 : (cosine < -1.0 ? -1.0 : cosine);
  double pj_yaw;
  Vec3 pj_forward;
  const Mat4 pj_view = aimed_view(yaw_deg, -acos(cosine) * 180.0 / kPi, pj_eye, lane, &pj_yaw, &pj_forward);

  // both view-projections, column (lane & 3) of the camera's in lanes 0-15 and of the
  // projector's in lanes 16-31, and their inverses: columns 4-7 of [A | I] in lanes 4-7, 20-23
  double vp[4], a[4], b_col[4];
#pragma unroll
  for (int k = 0; k < 4; ++k)
    b_col[k] = (lane & 16) ? pick_column(pj_view, lane & 3, k) : pick_column(view, lane & 3, k);
  mul_column(persp, b_col, vp);
#pragma unroll
  for (int r = 0; r < 4; ++r) a[r] = (lane & 4) ? ((lane & 3) == r ? 1.0 : 0.0) : vp[r];
  bool regular = eliminate<0>(a);
  regular &= eliminate<1>(a);
  regular &= eliminate<2>(a);
  regular &= eliminate<3>(a);
  const unsigned long long regular_lanes = __ballot(regular);
  if (!(regular_lanes & 1)) return WT_ERR_DEGENERATE;

  // padded frustum corner (lane & 7)
  const Mat4 pvp = gather_columns(vp, 16);
  const double pad = 1.2;
  const double sx = (lane & 4) ? 1.0 : -1.0, sy = (lane & 2) ? 1.0 : -1.0, sz = (lane & 1) ? 1.0 : -1.0;
  const Vec4 h = mat_apply(gather_columns(a, 4), Vec4{sx * pad, sy * pad, sz, 1.0});
  const Vec3 fc{h.x / h.w, h.y / h.w, h.z / h.w};

  // points of the slab in the reference's order: edge lane / 2 on the upper and the lower
  // plane in lanes 0-23, frustum corner lane - 24 in lanes 24-31; edges as octal digits
  const int shift = 3 * (lane < 24 ? lane >> 1 : 0);
  const int e0 = (int)(0654432211000ull >> shift) & 7, e1 = (int)(0776576353421ull >> shift) & 7;
  const Vec3 p{__shfl(fc.x, e0), __shfl(fc.y, e0), __shfl(fc.z, e0)};
  const Vec3 q{__shfl(fc.x, e1), __shfl(fc.y, e1), __shfl(fc.z, e1)};
  const double plane = (lane & 1) ? -amp : amp;
  Vec3 point{0, 0, 0};
  bool inside = lane < 24 && fmin(p.y, q.y) <= plane && plane <= fmax(p.y, q.y) && hit_plane_y(p, q, plane, &point);
  if (lane >= 24 && lane < 32) {
    inside = -amp <= fc.y && fc.y <= amp;
    point = fc;
  }
  const unsigned long long points = __ballot(inside);
  if (points == 0) return WT_ERR_NO_INTERSECTION;
  if (!aim_ok || !((regular_lanes >> 16) & 1)) return WT_ERR_DEGENERATE;
  const Vec4 ndc = mat_apply(pvp, Vec4{point.x, 0.0, point.z, 1.0});
  const double nx = ndc.x / ndc.w, ny = ndc.y / ndc.w;
  double xmin, xmax, ymin, ymax;
  const int lead = __builtin_ctzll(points);
  bounds(nx, inside, lead, &xmin, &xmax);
  bounds(ny, inside, lead, &ymin, &ymax);

  // projector matrix: column (lane & 3) of inverse * range in each lane
  const int col = lane & 3;
  const double range_col[4] = {col == 0 ? xmax - xmin : (col == 3 ? xmin : 0.0),
                               col == 1 ? ymax - ymin : (col == 3 ? ymin : 0.0), col == 2 ? 1.0 : 0.0,
                               col == 3 ? 1.0 : 0.0};
  double m_col[4];
  mul_column(gather_columns(a, 20), range_col, m_col);
  // range-space corner i on the near plane in lane 2 i, on the far plane in lane 2 i + 1
  const double u = (lane & 4) ? 1.0 : 0.0, v = (lane & 2) ? 1.0 : 0.0;
  const Vec4 n = mat_apply(gather_columns(m_col, 0), Vec4{u, v, (lane & 1) ? 1.0 : -1.0, 1.0});
  const Vec3 end{n.x / n.w, n.y / n.w, n.z / n.w};
  const Vec3 far_end{__shfl_down(end.x, 1), __shfl_down(end.y, 1), __shfl_down(end.z, 1)};
  const bool hit = hit_plane_y(end, far_end, 0.0, corner);
  return (__ballot(hit) & 0x55) == 0x55 ? WT_OK : WT_ERR_DEGENERATE;
}

__global__ __launch_bounds__(64) void projector_wave_kernel(ProjectorArgs a) {
  const int i = (int)blockIdx.x, lane = (int)threadIdx.x;
  const wt_camera cam = a.cameras[i];
  const float amp = a.amplitudes[i];
  proj::Vec3 c{0, 0, 0};
  int st = WT_ERR_INVALID_ARG;
  if (proj::camera_valid(cam) && __builtin_isfinite(amp) && amp >= 0.0f)
    st = projector_corners_wave(cam, (double)amp, lane, &c);
  if (a.corners && lane < 8 && !(lane & 1)) {
    double* o = a.corners + 16 * (size_t)i + 2 * lane;
    const double nan = __builtin_nan("");
    o[0] = st == WT_OK ? c.x : nan;
    o[1] = st == WT_OK ? c.y : nan;
    o[2] = st == WT_OK ? c.z : nan;
    o[3] = st == WT_OK ? 1.0 : nan;
  }
  if (a.status && lane == 0) a.status[i] = st;
  if (a.patches) {
    double corners[4][4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      corners[k][0] = lane_value(c.x, 2 * k);
      corners[k][2] = lane_value(c.z, 2 * k);
    }
    PatchDesc& d = a.patches[i];
    if (lane == 0) {
      if (st == WT_OK) {
        set_corner_algebra(d, corners);
        d.cam[0] = cam.position[0];
        d.cam[1] = cam.position[1];
        d.cam[2] = cam.position[2];
      }
      d.active = st == WT_OK;
    }
  }
}

#pragma clang fp contract(fast)

hipError_t launch_projector(const ProjectorArgs& a, hipStream_t st) {
  if (a.count <= 0) return hipSuccess;
  if (a.count <= kWaveProjectorCameras) {
    hipLaunchKernelGGL(projector_wave_kernel, dim3((unsigned)a.count), dim3(64), 0, st, a);
  } else {
    const unsigned blocks = (unsigned)((a.count + kProjectorThreads - 1) / kProjectorThreads);
    hipLaunchKernelGGL(projector_kernel, dim3(blocks), dim3(kProjectorThreads), 0, st, a);
  }
  return hipGetLastError();
}

}  // namespace wt
