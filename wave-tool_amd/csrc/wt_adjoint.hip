// Adjoint of the heightfield fit and its Adam update (no reference counterpart).
//
// Model per wave (A, L, alpha, Q, phi0): w = 2 pi / L, omega = sqrt(g w),
// D = (cos alpha, sin alpha), theta = w D.x + omega t + phi0 (the reference's sign
// convention, assets/shaders/water-grid.vert:78), displacement
// d = (Q A Dx cos theta, A sin theta, Q A Dz cos theta) (water-grid.vert:79-81).
// Loss = 1 / (2 S V) * sum over snapshots and grid points of |d - target|^2.
//
// On a regular grid exp(i theta) splits into a column factor and a (row, snapshot) factor
// P = exp(i (kx x_mid + kz z_j + omega t_s + phi0)), x_mid the centre of a strip of 64
// columns. The columns pair up about the centre at the offsets +-delta, so the column
// factors are the real cos(kx delta) and sin(kx delta) of 32 offsets, and both passes are
// contractions for the matrix cores over the even and the odd part of what they act on:
//   forward   (d+ + d-) / 2 [delta, (j,s)] = sum over waves of cos(kx delta) x B, and
//             (d+ - d-) / 2 the same with sin and B', B and B' the coefficients times P;
//   backward  G[wave, (j,s)] = sum over offsets of cos(kx delta) x (r+ + r-) and of
//             sin(kx delta) x (r+ - r-), and the same weighted with the offset, from which
//             P gives every wave's sums of r cos theta and r sin theta.
// Folding halves the products of the plain split into 64 columns (a batch of 256 uneven
// problems on one MI355X: 1.3 ms an iteration against 1.5 ms).
// adjoint_kernel: a workgroup takes one strip and a run of (row, snapshot) pairs q = j S + s,
//   16 consecutive pairs (a tile) per wavefront at a time, so any snapshot count packs the
//   tiles without padding. The column factors sit in LDS as matrix fragments, built once
//   per workgroup; per tile a wavefront forms P and B in registers, contracts the forward
//   pass onto the negated targets, and contracts the backward pass with the residuals still
//   in the registers the forward pass left them in (the offset order of the backward
//   fragments is the accumulators' order). Chunks of 16 waves are looped over, not
//   unrolled: one body serves every wave count and stays in the instruction cache.
// Operands are FP32 values split into two FP16 halves, v = hi + lo with hi = fp16(v)
//   and lo = fp16(v - hi), multiplied as hi hi + hi lo + lo hi with FP32 accumulation
//   (about 2^-22 per product). Powers of two keep both halves in FP16's range: the column
//   factors are scaled by 2^4, the coefficients by their largest magnitude in the problem,
//   and the residuals by the largest of the wavefront's tile where that leaves the range.
//   Against the FP64 adjoint the gradients of 84 drawn problems (sides 32-400, 2-32
//   snapshots, 4-64 waves) are closer than with FP32 recurrences over the snapshots: rms of
//   the relative error 7.9e-8 against 1.3e-6, of 65-128 waves 6.4e-8 against 5.5e-7.
// What bounds it: VALU issue and the matrix cores together, which do not overlap on one
//   SIMD (two wavefronts of one SIMD, one issuing only matrix instructions and one only
//   FMAs, take the sum of their times): per tile of 64 waves about 1300 VALU instructions
//   and 216 matrix instructions of 16 cycles. With the reduction, in a graph: 512^2 x 16 x 32
//   21.5 us (66 us with FP32 recurrences over the snapshots on the VALU); the 256-problem batch
//   1.23 ms an iteration (3.67 ms).
//   Two wavefronts per SIMD at up to 256 VGPRs: a 32-column strip at three or four
//   wavefronts repeats P, B and the sums per point (1.7 ms), and a spilled register is a
//   round trip to cold scratch memory (5 us per workgroup).
// reduce_adam_kernel: one workgroup per 16 parameter rows of a problem: fixed-order sum of
//   the block partials in FP64, scaling to the mean misfit, and either an Adam step on the
//   parameters or a plain gradient / loss write-out. Bound by its memory round trips: the
//   rows are consecutive in memory and 64 parts are read side by side, so a sum over 256
//   parts is one round of loads (a workgroup per row took 58 us for the
//   256-problem batch, 24 so).
// adjoint_few_kernel: the same for problems of up to 4 waves (6 where they are small), on the
//   VALU (fit_few).
// All find their problem through a unit (reduce block) -> problem map built at
// creation, so one launch per wave-count class covers a whole batch; a single problem is
// a table of one. A problem's blocks and the order of every sum depend on the problem
// alone, so a batch repeats the bits of its problems run one by one.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>
#include <utility>

#include "wt_fit.hpp"

namespace wt {

typedef _Float16 Half2 __attribute__((ext_vector_type(2)));
typedef _Float16 Half8 __attribute__((ext_vector_type(8)));
typedef float Float4 __attribute__((ext_vector_type(4)));

// A wave's constants in the tile loop (zero for the padding up to a multiple of 16).
struct FitWaveLds {
  double kx, kz, c0, om;  // revolutions per metre along x and z, phase at t0 (fract), revolutions per second
};
// And those that turn its sums into parameter derivatives.
struct FitWaveGrad {
  float A, Q, Dx, Dz, w, wL, om2L;  // wL = w / L, om2L = omega / (2 L)
};

// One wave's constants from its parameters, in FP64, rounded once.
struct FitWave {
  FitWaveLds lds;
  FitWaveGrad grad;
  float bx, by, bz;  // Q A Dx, A, Q A Dz
  float2 dir;        // Q Dx, Q Dz
};
__device__ __forceinline__ FitWave fit_wave(const FitDesc& P, const float (&p)[5]) {
  const double A = p[0], L = p[1] > 1e-3f ? p[1] : 1e-3f, al = p[2], Q = p[3], ph0 = p[4];
  const double w = kTwoPi / L, om = sqrt(P.g * w);
  double sa, ca;
  sincos(al, &sa, &ca);
  FitWave o;
  o.lds.kx = w * ca * kInvTwoPi;
  o.lds.kz = w * sa * kInvTwoPi;
  o.lds.c0 = __builtin_amdgcn_fract(fma(om, P.t0, ph0) * kInvTwoPi);
  o.lds.om = om * kInvTwoPi;
  o.bx = (float)(Q * A * ca);
  o.by = (float)A;
  o.bz = (float)(Q * A * sa);
  o.dir = make_float2((float)(Q * ca), (float)(Q * sa));
  o.grad = FitWaveGrad{(float)A, (float)Q, (float)ca, (float)sa, (float)w, (float)(w / L), (float)(om / (2.0 * L))};
  return o;
}

// Sum over the 64 lanes of a wavefront with DPP moves (VALU only, fixed order); the
// total lands in lane 63. quad_perm [1,0,3,2] and [2,3,0,1] give quad sums,
// row_half_mirror and row_mirror row sums, row_bcast:15 / :31 the rest.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ float dpp_term(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROW_MASK, 0xf, false));
}
// The sum over each row of 16 lanes, in every lane of the row.
__device__ __forceinline__ float row_sum(float v) {
  v += dpp_term<0xB1, 0xf>(v);
  v += dpp_term<0x4E, 0xf>(v);
  v += dpp_term<0x141, 0xf>(v);
  v += dpp_term<0x140, 0xf>(v);
  return v;
}
__device__ __forceinline__ float wave_sum63(float v) {
  v = row_sum(v);
  v += dpp_term<0x142, 0xa>(v);
  v += dpp_term<0x143, 0xc>(v);
  return v;
}
// gfx950's lane swaps between two registers, summed lane by lane. With rows r0..r3 of
// 16 lanes,
//   swap32_sum(x, y) = [x.r0 + x.r2, x.r1 + x.r3, y.r0 + y.r2, y.r1 + y.r3],
//   swap16_sum(x, y) = [x.r0 + x.r1, y.r0 + y.r1, x.r2 + x.r3, y.r2 + y.r3],
// so four values are summed over the rows in two swap32 sums and one swap16 sum.
__device__ __forceinline__ float swap32_sum(float x, float y) {
  const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
  return __uint_as_float(p[0]) + __uint_as_float(p[1]);
}
__device__ __forceinline__ float swap16_sum(float x, float y) {
  const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
  return __uint_as_float(p[0]) + __uint_as_float(p[1]);
}
// The maximum of a non-negative value over the wavefront, wave-uniform.
__device__ __forceinline__ float wave_max(float v) {
  v = fmaxf(v, dpp_term<0xB1, 0xf>(v));
  v = fmaxf(v, dpp_term<0x4E, 0xf>(v));
  v = fmaxf(v, dpp_term<0x141, 0xf>(v));
  v = fmaxf(v, dpp_term<0x140, 0xf>(v));
  v = fmaxf(v, dpp_term<0x142, 0xa>(v));
  v = fmaxf(v, dpp_term<0x143, 0xc>(v));
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

// The power of two that takes magnitude m (>= 0) to [2^3, 2^4), as an exponent; clamped
// for m zero, denormal, infinite or NaN so that it, its inverse and (up to 2^60) what is
// multiplied by it stay floats.
__device__ __forceinline__ int scale_exponent(float m) {
  const int e = (int)((__float_as_uint(m) >> 23) & 0xffu) - 127;
  return min(max(3 - e, -110), 60);
}
__device__ __forceinline__ float pow2f(int e) { return __uint_as_float((uint32_t)(127 + e) << 23); }

// (a, b) as packed halves: hi = fp16, lo = fp16 of the rest (exact in FP32). The empty
// asm statements keep the remainder a fused a - hi from the packed word, which converts on
// the way in and out (v_fma_mixlo_f16 / v_fma_mixhi_f16: three instructions per pair).
__device__ __forceinline__ void split2(float a, float b, uint32_t& hi, uint32_t& lo) {
  const Half2 h = {(_Float16)a, (_Float16)b};
  hi = __builtin_bit_cast(uint32_t, h);
  asm("" : "+v"(hi));
  float minus = -1.0f;
  asm("" : "+s"(minus));
  const Half2 g = __builtin_bit_cast(Half2, hi);
  const Half2 l = {(_Float16)fmaf((float)g.x, minus, a), (_Float16)fmaf((float)g.y, minus, b)};
  lo = __builtin_bit_cast(uint32_t, l);
}

union Frag {  // one lane's 8 halves of a 16x16x32 operand
  uint32_t w[4];
  Half8 h;
};

__device__ __forceinline__ Float4 mma(const Half8& a, const Half8& b, const Float4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// One column factor (hi, lo) contracted with the three components of a residual part.
__device__ __forceinline__ void column_sums(const Half8& eh, const Half8& el, const Frag (&rh)[3], const Frag (&rl)[3],
                                            Float4 (&o)[3]) {
#pragma unroll
  for (int c = 0; c < 3; ++c) o[c] = mma(rh[c].h, eh, o[c]);
#pragma unroll
  for (int c = 0; c < 3; ++c) o[c] = mma(rl[c].h, eh, o[c]);
#pragma unroll
  for (int c = 0; c < 3; ++c) o[c] = mma(rh[c].h, el, o[c]);
}

// Consecutive floats at 4-byte alignment.
struct __attribute__((packed, aligned(4))) Target4 {
  float v[4];
};
struct __attribute__((packed, aligned(4))) Target3 {
  float v[3];
};

// cos and sin of 2 pi f for an FP64 phase f in revolutions: reduced in FP64 to r in
// [-1/8, 1/8] of a quarter turn's centre, then interpolating polynomials in r^2 through
// the Chebyshev nodes of [0, 1/64] (truncation below 1e-8), signs and order by quadrant.
// Worst error 9e-8, rms 2e-8, against 2e-7 and about 1e-7 for v_sin_f32 / v_cos_f32 with
// the argument's rounding corrected: one factor serves a whole row or column of products
// here, so its error does not average out, and with the hardware functions the gradients
// of few-snapshot problems were up to 1.6 times further from the FP64 adjoint.
__device__ __forceinline__ void sincos_turn(double f, float* c, float* s) {
  f = __builtin_amdgcn_fract(f);
  const double k = rint(4.0 * f);
  const float r = (float)fma(-0.25, k, f), u = r * r;
  const int quad = (int)k;
  const float sp = r * fmaf(fmaf(fmaf(-75.4016127f, u, 81.5925429f), u, -41.3416626f), u, 6.28318529f);
  const float cp = fmaf(fmaf(fmaf(fmaf(59.2201690f, u, -85.4428447f), u, 64.9393161f), u, -19.7392087f), u, 1.0f);
  const bool odd = quad & 1;
  const float sv = odd ? cp : sp, cv = odd ? sp : cp;
  *s = __uint_as_float(__float_as_uint(sv) ^ ((uint32_t)(quad & 2) << 30));
  *c = __uint_as_float(__float_as_uint(cv) ^ ((uint32_t)((quad + 1) & 2) << 30));
}

// Orders this wavefront's LDS accesses around it: its lanes read what other lanes of it
// wrote (LDS operations of one wavefront complete in order, so no wait is needed).
__device__ __forceinline__ void wavefront_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

constexpr float kFitTrigScale = 16.0f;  // scale of E in its fragments
// The largest scaled residual a tile is split at without rescaling: the halves stay finite
// (2^15 below FP16's largest) and the low halves' FP16 spacing, 2^-24, stays below 2^-24 of
// the largest.
constexpr float kFitResLow = 1.0f, kFitResHigh = 32768.0f;

// What the wavefronts of a workgroup leave of a part: per wavefront, chunk and lane two of
// the part's running sums of wave lane mod 16, and the loss.
template <int KMAX, int NW>
struct FitSums {
  float2 sums[NW][KMAX][64];
  float loss[NW];
};

constexpr int kRunFloats = 52;  // a run of 48 target floats, padded: rows of eight pairs on different banks

// The workgroup's LDS for up to KMAX chunks of 16 waves (`chunks` of them in use).
//  fwd, bwd: the column factors cos(kx delta), sin(kx delta) of the 32 column offsets
//    delta = (t + 1/2) spacing as matrix operands. Two chunks make the forward pass's inner
//    dimension of 32 (hi, then lo); a last odd chunk takes it as [hi | lo] of its 16 waves.
//    fwd [16 offsets][cos / sin][chunk][lane], bwd [chunk][cos / sin][plain / times
//    t + 1/2][hi / lo][lane].
//  time: exp(i omega s dt), [snapshot][wave] (cos, sin), then a row of zeros for the pairs
//    past the last; rows padded by 16 bytes to keep the 16-byte reads of eight neighbouring
//    rows on different banks.
//  row: per wavefront the factors exp(i (kx x + kz z_j + phase at t0)) at the strip's centre
//    of a tile's four rows, [row][wave] (cos, sin).
//  run: per wavefront one run of 16 columns' targets of 16 pairs, on the way to its lanes.
template <int KMAX, int NW, bool kTable>
struct FitShared {
  float4 coef[16 * KMAX];  // Q A Dx, A, Q A Dz, scaled by the problem's power of two
  float2 dir[16 * KMAX];   // Q Dx, Q Dz
  FitWaveLds wave[16 * KMAX];
  FitWaveGrad grad[16 * KMAX];
  uint32_t max;  // bits of the largest coefficient magnitude
  alignas(16) float row[NW][kTable ? 4 * 32 * KMAX : 4];
  alignas(16) float time[kTable ? (kFitMaxSnapshots + 1) * (32 * KMAX + 4) : 4];
  FitSums<KMAX, NW> end;
  alignas(16) float run[NW][kTable ? 16 * kRunFloats : 4];
  Half8 fwd[2 * 2 * KMAX * 64];
  Half8 bwd[KMAX * 2 * 2 * 2 * 64];
  __device__ __forceinline__ Half8* fwd_at(int chunks, int mt, int o, int k) { return fwd + ((mt * 2 + o) * chunks + k) * 64; }
  __device__ __forceinline__ Half8* bwd_at(int kc, int o, int m, int h) { return bwd + (((kc * 2 + o) * 2 + m) * 2 + h) * 64; }
};

constexpr int kStrip = 64, kHalf = 32;  // a strip's columns, and the offsets they pair up at

// The targets of one (row, snapshot) pair, twelve floats each of the columns 32 + t .. and
// 31 - t .. of the strip, t = 16 mt + 4 g + 0 .. 3 (up, dn). Columns past the grid and
// pairs past the last give zero. `whole` (the strip and the tile lie inside,
// wave-uniform): the four lanes of a pair together read each 192-byte run of 16 columns,
// 64 consecutive bytes per instruction, and unshuffle() hands every lane its own columns
// (a lane's 48 bytes read directly made every load instruction 64 cache accesses, 60% of
// the time of a tile of 32 waves).
__device__ __forceinline__ void load_targets(const FitDesc& P, bool whole, bool valid, uint32_t j, uint32_t sn,
                                             int col0, int g, float (&up)[2][12], float (&dn)[2][12]) {
  const float* tp = P.target + (size_t)sn * (3 * (size_t)P.n * (size_t)P.n) +
                    3 * ((size_t)j * (size_t)P.n + (size_t)(col0 + kHalf));
  if (whole) {
    const float* tl = tp + 4 * g;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const Target4 a = *reinterpret_cast<const Target4*>(tl + 48 * mt + 16 * k);
        const Target4 b = *reinterpret_cast<const Target4*>(tl - 48 * (mt + 1) + 16 * k);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          up[mt][4 * k + i] = a.v[i];
          dn[mt][4 * k + i] = b.v[i];
        }
      }
  } else {
    // columns clamped to the row, and what lies outside taken times zero (a select on a
    // loaded value would become a branch around every load)
    int last = P.n - 1 - (col0 + kHalf);  // the row's last column, from the strip's centre
    asm volatile("" : "+s"(last));  // keeps the clamped addresses out of the tile loop's live registers
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int iu = 16 * mt + 4 * g + r, id = -(16 * mt + 4 * g + 4) + r;
        const float mu = valid && iu <= last ? 1.0f : 0.0f, md = valid && id <= last ? 1.0f : 0.0f;
        const Target3 a = *reinterpret_cast<const Target3*>(tp + 3 * min(iu, last));
        const Target3 b = *reinterpret_cast<const Target3*>(tp + 3 * min(id, last));
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          up[mt][3 * r + c] = mu * a.v[c];
          dn[mt][3 * r + c] = md * b.v[c];
        }
      }
  }
}

// Reads one float of nearly every cache line of a tile's runs of 64 columns (16 runs of
// 768 bytes, eight reads 108 bytes apart each), which brings them to the L2 ahead of
// load_targets: issued before the set-up, whose tables need no memory, 512^2 x 16 x 32
// takes 21.1 us with its reduction where it took 22.7. For every tile ahead of its time it was slower.
__device__ __forceinline__ void touch_targets(const FitDesc& P, int strip, int tile, int lane, float& a, float& b) {
  const uint32_t pairs = (uint32_t)P.n * (uint32_t)P.S, q = min((uint32_t)tile * 16u + (uint32_t)(lane & 15), pairs - 1u);
  const uint32_t j = q / (uint32_t)P.S, sn = q - j * (uint32_t)P.S;
  const int col0 = max(0, min(strip * kStrip, P.n - kStrip)), last = 3 * (P.n - col0) - 1;
  const float* t = P.target + 3 * ((size_t)sn * (size_t)P.n * (size_t)P.n + (size_t)j * (size_t)P.n + (size_t)col0);
  a = t[min(27 * (lane >> 4), last)];
  b = t[min(27 * (lane >> 4) + 108, last)];
}

// One run through the wavefront's LDS buffer: from 64-byte pieces of every pair to lane
// g's twelve floats at 12 * column group `at`.
__device__ __forceinline__ void unshuffle(float* run, int n16, int g, int at, float (&v)[12]) {
  float4* w = reinterpret_cast<float4*>(run + n16 * kRunFloats);
#pragma unroll
  for (int k = 0; k < 3; ++k) w[4 * k + g] = make_float4(v[4 * k], v[4 * k + 1], v[4 * k + 2], v[4 * k + 3]);
  wavefront_lds_sync();
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const float4 t = w[3 * at + k];
    v[4 * k] = t.x;
    v[4 * k + 1] = t.y;
    v[4 * k + 2] = t.z;
    v[4 * k + 3] = t.w;
  }
  wavefront_lds_sync();
}

// The end of a round of parts: the wavefronts' sums in index order, then the parameter
// derivatives and the loss of every part. Returns the parts that ran side by side.
template <int KMAX, int NW>
__device__ __forceinline__ int finish_parts(const FitDesc& P, const FitSums<KMAX, NW>& of, const FitWaveGrad* grad,
                                            double x_mid, int part, int part_end, int end, int lane, int wid) {
  __syncthreads();
  const int waves_per = min(P.tiles_per_block, NW), side_by = NW >> __builtin_ctz(waves_per);
  const int wave_rows = (P.W + 63) >> 6;
#pragma unroll 1
  for (int it = wid; it < side_by * wave_rows; it += NW) {
    int wi = lane;
    asm volatile("" : "+v"(wi));  // keeps this block's addresses out of the tile loop's live registers
    const int mine = wave_rows > 1 ? it >> 1 : it;
    if (wave_rows > 1) wi += 64 * (it & 1);
    const int w0 = mine * waves_per;
    if (part_end - max(P.tiles_per_block, NW) + w0 >= end || wi >= P.W) continue;  // no such part
    double v[8];
    auto sum_waves = [&](auto whole) {  // the part's wavefronts, all loads in flight together
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float2* from = &of.sums[whole ? 0 : w0][wi >> 4][16 * r + (wi & 15)];
        float2 t = *from;
#pragma unroll
        for (int i = 1; i < (whole ? NW : NW / 2); ++i) {
          const float2 u = from[(whole || i < waves_per ? i : 0) * (KMAX * 64)];
          t.x += whole || i < waves_per ? u.x : 0.0f;
          t.y += whole || i < waves_per ? u.y : 0.0f;
        }
        const int k = ((r & 1) << 1) | (r >> 1);
        v[k] = (double)t.x;
        v[4 + k] = (double)t.y;
      }
    };
    if (waves_per == NW) sum_waves(std::true_type{});
    else sum_waves(std::false_type{});
    const FitWaveGrad w = grad[wi];
    // sums of r . dd/dtheta: plain, times t, times the world x and z
    const double A = w.A, Dx = w.Dx, Dz = w.Dz;
    const double g0 = A * v[3], gt = A * fma(P.t0, v[3], P.dt * v[4]);
    const double gx = A * fma(x_mid, v[3], P.spacing * v[6]);
    const double gz = A * fma(P.z0, v[3], P.spacing * v[5]);
    const double sec = fma(Dx, v[0], Dz * v[1]), sepc = fma(Dx, v[1], -(Dz * v[0]));
    const float out[5] = {(float)fma((double)w.Q, sec, v[2]),
                          (float)-fma((double)w.wL, fma(Dx, gx, Dz * gz), w.om2L * gt),
                          (float)fma((double)w.w, fma(Dx, gz, -(Dz * gx)), w.Q * A * sepc), (float)(A * sec), (float)g0};
    float* o = P.partials + (size_t)(part + mine) * (5 * P.W + 1);
#pragma unroll
    for (int k = 0; k < 5; ++k) o[5 * wi + k] = out[k];
    if (wi == 0) {
      float t = of.loss[w0];
      for (int i = w0 + 1; i < w0 + waves_per; ++i) t += of.loss[i];
      o[5 * P.W] = t;
    }
  }
  return side_by;
}

// A unit's tiles and the sums of its parts. Lane (n16, g) works in the forward pass on
// pair n16, the column offsets t = 16 mt + 4 g + r and the waves 4 g + u of a chunk; after the
// backward contraction on wave n16 of a chunk and the pairs 4 g + r. kTable: P from the
// time table and the tile's row factors, else a sine and cosine per pair and wave.
template <bool kByTable, int KMAX, int NW, bool kTable>
__device__ __forceinline__ void fit_tiles(const FitDesc& P, const FitUnit& unit, FitShared<KMAX, NW, kTable>& sh,
                                          int chunks, int coef_exp) {
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n16 = lane & 15, g = lane >> 4;
  const int time_row = 32 * chunks + 4;
  float* const s_row = sh.row[wid];
  // the last strip ends with the row (from 64 columns on), its columns that belong to the
  // strip before it left out
  const int lo_col = unit.strip * kStrip, col0 = max(0, min(lo_col, P.n - kStrip));
  const uint32_t pairs = (uint32_t)P.n * (uint32_t)P.S;  // n <= 8192, S <= 32
  // q / S by a multiply-high: exact for q < 2^18, S <= 32
  const uint32_t magic = 0xffffffffu / (uint32_t)P.S + 1u;
  const bool one = P.S == 1;
  auto row_of = [&](uint32_t q) { return one ? q : __umulhi(q, magic); };
  const int tiles = (int)((pairs + 15) >> 4);
  const int first = unit.part * P.tiles_per_block;
  const int end = min(tiles, first + unit.parts * P.tiles_per_block);
  const bool inside = P.n >= kStrip, full_strip = lo_col + kStrip <= P.n;
  const float fwd_scale = pow2f(coef_exp) * kFitTrigScale;
  const float inv_fwd = pow2f(-coef_exp) * (1.0f / kFitTrigScale), neg_half = -0.5f * fwd_scale;
  const double x_mid = P.x0 + ((double)col0 + 31.5) * P.spacing;  // the strip's centre

  for (int kc = 0; kc < chunks; ++kc) sh.end.sums[wid][kc][lane] = make_float2(0.0f, 0.0f);
  float sq = 0.0f;


  // a round of the parts of a workgroup: one part, or as many side by side as it has
  // wavefronts for (parts of fewer tiles than wavefronts, powers of two)
  int part = unit.strip * P.blocks_per_strip + unit.part, part_end = first + max(P.tiles_per_block, NW);
#pragma unroll 1
  for (int base = first; base < end; base += NW) {
    const int tile = base + wid;
    if (tile < end) {
      const uint32_t q = (uint32_t)tile * 16u + (uint32_t)n16;
      const bool valid = q < pairs;
      const uint32_t qc = valid ? q : pairs - 1u;
      const uint32_t j = row_of(qc), sn = qc - j * (uint32_t)P.S;
      const uint32_t j0 = row_of((uint32_t)tile * 16u);  // the tile's first row
      const bool whole = kTable && inside && (uint32_t)tile * 16u + 16u <= pairs;
      float up[2][12], dn[2][12];
      load_targets(P, whole, valid, j, sn, col0, g, up, dn);
      if constexpr (kByTable) {
#pragma unroll 1
        for (int kc = 0; kc < chunks; ++kc) {
          const FitWaveLds& w = sh.wave[16 * kc + n16];
          float cv, sv;
          sincos_turn(fma(w.kz, P.z0 + (double)(j0 + (uint32_t)g) * P.spacing, fma(w.kx, x_mid, w.c0)), &cv, &sv);
          *reinterpret_cast<float2*>(&s_row[(g * chunks + kc) * 32 + 2 * n16]) = make_float2(cv, sv);
        }
        wavefront_lds_sync();
      }

      if (whole) {
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) {
          unshuffle(sh.run[wid], n16, g, g, up[mt]);
          unshuffle(sh.run[wid], n16, g, 3 - g, dn[mt]);
        }
      }
      // forward, onto the negated folded targets in the contraction's units
      Float4 d[2][2][3];  // [16 offsets][even / odd][x, y, z]
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float a = up[mt][3 * r + c] * neg_half, b = dn[mt][3 * (3 - r) + c];
            d[mt][0][c][r] = fmaf(b, neg_half, a);
            d[mt][1][c][r] = fmaf(b, -neg_half, a);
          }
      // the pairs past the last take the table's zero row (or zeros) for P
      const float* trow = sh.time + (valid ? sn : (uint32_t)P.S) * (uint32_t)time_row + 8 * g;
      const float* rrow = s_row + (j - j0) * (uint32_t)(32 * chunks) + 8 * g;
      const double zj = P.z0 + (double)j * P.spacing, ts = (double)sn * P.dt;
      const float live = valid ? 1.0f : 0.0f;
      // P of a chunk times the coefficients, split: words [at, at + 2) of the operands
      auto coefficients = [&](int kc, int at, Frag(&bh)[2][3], Frag(&bl)[2][3]) {
        float pc[4], ps[4];
        if constexpr (kByTable) {
          const float4* rp = reinterpret_cast<const float4*>(rrow + 32 * kc);
          const float4* qp = reinterpret_cast<const float4*>(trow + 32 * kc);
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const float4 a = rp[h], t = qp[h];
            pc[2 * h] = fmaf(a.x, t.x, -(a.y * t.y));
            ps[2 * h] = fmaf(a.x, t.y, a.y * t.x);
            pc[2 * h + 1] = fmaf(a.z, t.z, -(a.w * t.w));
            ps[2 * h + 1] = fmaf(a.z, t.w, a.w * t.z);
          }
        } else {
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const FitWaveLds& w = sh.wave[16 * kc + 4 * g + u];
            sincos_turn(fma(w.om, ts, fma(w.kz, zj, fma(w.kx, x_mid, w.c0))), &pc[u], &ps[u]);
            pc[u] *= live;
            ps[u] *= live;
          }
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const float4 w0 = sh.coef[16 * kc + 4 * g + 2 * h], w1 = sh.coef[16 * kc + 4 * g + 2 * h + 1];
          const float c0 = pc[2 * h], s0 = ps[2 * h], c1 = pc[2 * h + 1], s1 = ps[2 * h + 1];
          split2(w0.x * c0, w1.x * c1, bh[0][0].w[at + h], bl[0][0].w[at + h]);
          split2(w0.y * s0, w1.y * s1, bh[0][1].w[at + h], bl[0][1].w[at + h]);
          split2(w0.z * c0, w1.z * c1, bh[0][2].w[at + h], bl[0][2].w[at + h]);
          split2(-w0.x * s0, -w1.x * s1, bh[1][0].w[at + h], bl[1][0].w[at + h]);
          split2(w0.y * c0, w1.y * c1, bh[1][1].w[at + h], bl[1][1].w[at + h]);
          split2(-w0.z * s0, -w1.z * s1, bh[1][2].w[at + h], bl[1][2].w[at + h]);
        }
      };
#pragma unroll 1
      for (int kp = 0; kp < chunks; kp += 2) {
        Frag bh[2][3], bl[2][3];  // [even / odd]
        const bool two = kp + 1 < chunks;
        coefficients(kp, 0, bh, bl);
        if (two) {
          coefficients(kp + 1, 2, bh, bl);
        } else {  // [hi | lo] x ([hi | hi] + [lo | 0])
#pragma unroll
          for (int o = 0; o < 2; ++o)
#pragma unroll
            for (int c = 0; c < 3; ++c) {
              bh[o][c].w[2] = bh[o][c].w[0];
              bh[o][c].w[3] = bh[o][c].w[1];
              bl[o][c].w[2] = bl[o][c].w[3] = 0u;
            }
        }
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
          for (int o = 0; o < 2; ++o) {
            const Half8 a = sh.fwd_at(chunks, mt, o, kp)[lane];
#pragma unroll
            for (int c = 0; c < 3; ++c) d[mt][o][c] = mma(a, bh[o][c].h, d[mt][o][c]);
#pragma unroll
            for (int c = 0; c < 3; ++c) d[mt][o][c] = mma(a, bl[o][c].h, d[mt][o][c]);
          }
        if (two) {
#pragma unroll
          for (int mt = 0; mt < 2; ++mt)
#pragma unroll
            for (int o = 0; o < 2; ++o) {
              const Half8 a = sh.fwd_at(chunks, mt, o, kp + 1)[lane];
#pragma unroll
              for (int c = 0; c < 3; ++c) d[mt][o][c] = mma(a, bh[o][c].h, d[mt][o][c]);
            }
        }
      }

      __builtin_amdgcn_sched_barrier(0);
      // d holds the folded residuals: r+ = even + odd, r- = even - odd. Columns outside the
      // strip's share are taken out of both (the last strip only).
      if (!full_strip) {
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int t = 16 * mt + 4 * g + r, cu = col0 + kHalf + t, cd = col0 + kHalf - 1 - t;
            const float mu = cu >= lo_col && cu < P.n ? 0.5f : 0.0f, md = cd >= lo_col && cd < P.n ? 0.5f : 0.0f;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
              const float u = mu * (d[mt][0][c][r] + d[mt][1][c][r]), v = md * (d[mt][0][c][r] - d[mt][1][c][r]);
              d[mt][0][c][r] = u + v;
              d[mt][1][c][r] = u - v;
            }
          }
      }
      float big = 0.0f;
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int o = 0; o < 2; ++o)
#pragma unroll
          for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int r = 0; r < 4; r += 2)
              big = fmaxf(fmaxf(fabsf(d[mt][o][c][r]), fabsf(d[mt][o][c][r + 1])), big);
      big = wave_max(big);
      // in these units a residual of the size of the largest coefficient is about 2^7: in
      // range as it is, unless the tile's largest is far from that
      int res_exp = 0;
      if (!(big >= kFitResLow && big <= kFitResHigh)) {
        res_exp = scale_exponent(big);
        const float res_scale = pow2f(res_exp);
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
          for (int o = 0; o < 2; ++o)
#pragma unroll
            for (int c = 0; c < 3; ++c) d[mt][o][c] *= res_scale;
      }
      const float inv_r = pow2f(-res_exp) * inv_fwd;  // a residual from its scaled value
      const float inv_g = 2.0f * inv_r * (1.0f / kFitTrigScale);  // r+ + r- is twice the even part
      Frag rh[2][3], rl[2][3];  // [even / odd]
      float sq_t = 0.0f;
#pragma unroll
      for (int o = 0; o < 2; ++o)
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const Float4& v = d[k >> 1][o][c];
            const float v0 = v[2 * (k & 1)], v1 = v[2 * (k & 1) + 1];
            sq_t = fmaf(v0, v0, sq_t);
            sq_t = fmaf(v1, v1, sq_t);
            split2(v0, v1, rh[o][c].w[k], rl[o][c].w[k]);
          }
      sq = fmaf(sq_t * inv_r, inv_r, sq);  // half the squares: r+^2 + r-^2 = 2 (even^2 + odd^2)

      // backward: per chunk the sums over the strip's columns of r cos and r sin of the
      // column factor, for 16 waves and 16 pairs; then P turns them into sums over theta
      float jf[4], sf[4];
      uint32_t r4[4], t4[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const uint32_t q4 = (uint32_t)tile * 16u + (uint32_t)(4 * g + r);
        const uint32_t j4 = row_of(q4), s4 = q4 - j4 * (uint32_t)P.S;
        jf[r] = (float)j4;
        sf[r] = (float)s4;
        r4[r] = (j4 - j0) * (uint32_t)(32 * chunks);
        t4[r] = s4 * (uint32_t)time_row;
      }
#pragma unroll 1
      for (int kc = 0; kc < chunks; ++kc) {
        const float2 dir = sh.dir[16 * kc + n16];
        const float qdx = dir.x, qdz = dir.y;
        float cp[4], sp[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if constexpr (kByTable) {
            const float2 a = *reinterpret_cast<const float2*>(&s_row[r4[r] + 32 * kc + 2 * n16]);
            const float2 b = *reinterpret_cast<const float2*>(&sh.time[t4[r] + 32 * kc + 2 * n16]);
            cp[r] = fmaf(a.x, b.x, -(a.y * b.y));
            sp[r] = fmaf(a.x, b.y, a.y * b.x);
          } else {
            const FitWaveLds& w = sh.wave[16 * kc + n16];
            sincos_turn(fma(w.om, (double)sf[r] * P.dt, fma(w.kz, P.z0 + (double)jf[r] * P.spacing, fma(w.kx, x_mid, w.c0))),
                        &cp[r], &sp[r]);
          }
        }
        // per wave of the lane, over its four pairs: sums of r_x cos, r_z cos, r_y sin, and
        // of h = the misfit's derivative by theta over A = sum r_y cos theta - Q (D . r) sin
        // theta (plain, times s, times j, times the column's offset). cos of the offset goes
        // with the even part and sin with the odd one; weighted the other way round.
        float t[7] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
        {
          Float4 gc[3], gn[3];  // [x, y, z] of the cos and the sin sums
#pragma unroll
          for (int c = 0; c < 3; ++c) gc[c] = gn[c] = Float4{0.0f, 0.0f, 0.0f, 0.0f};
          column_sums(sh.bwd_at(kc, 0, 0, 0)[lane], sh.bwd_at(kc, 0, 0, 1)[lane], rh[0], rl[0], gc);
          column_sums(sh.bwd_at(kc, 1, 0, 0)[lane], sh.bwd_at(kc, 1, 0, 1)[lane], rh[1], rl[1], gn);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            t[0] = fmaf(cp[r], gc[0][r], fmaf(-sp[r], gn[0][r], t[0]));
            t[1] = fmaf(cp[r], gc[2][r], fmaf(-sp[r], gn[2][r], t[1]));
            t[2] = fmaf(cp[r], gn[1][r], fmaf(sp[r], gc[1][r], t[2]));
            const float hc = fmaf(qdx, gc[0][r], qdz * gc[2][r]), hs = fmaf(qdx, gn[0][r], qdz * gn[2][r]);
            const float h = fmaf(cp[r], gc[1][r] - hs, -(sp[r] * (gn[1][r] + hc)));
            t[3] += h;
            t[4] = fmaf(sf[r], h, t[4]);
            t[5] = fmaf(jf[r], h, t[5]);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        {
          Float4 gc[3], gn[3];
#pragma unroll
          for (int c = 0; c < 3; ++c) gc[c] = gn[c] = Float4{0.0f, 0.0f, 0.0f, 0.0f};
          column_sums(sh.bwd_at(kc, 0, 1, 0)[lane], sh.bwd_at(kc, 0, 1, 1)[lane], rh[1], rl[1], gc);
          column_sums(sh.bwd_at(kc, 1, 1, 0)[lane], sh.bwd_at(kc, 1, 1, 1)[lane], rh[0], rl[0], gn);
          float wx = 0.0f, wy = 0.0f, wz = 0.0f;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            wy = fmaf(cp[r], gc[1][r], fmaf(-sp[r], gn[1][r], wy));
            wx = fmaf(cp[r], gn[0][r], fmaf(sp[r], gc[0][r], wx));
            wz = fmaf(cp[r], gn[2][r], fmaf(sp[r], gc[2][r], wz));
          }
          t[6] = fmaf(-qdx, wx, fmaf(-qdz, wz, wy));
        }
        // summed over the four groups of pairs by lane swaps: lane rows 0..3 then hold sums
        // 0, 2, 1, 3 and 4, 6, 5 and a zero
        const float lo = swap16_sum(swap32_sum(t[0], t[1]), swap32_sum(t[2], t[3]));
        const float hi = swap16_sum(swap32_sum(t[4], t[5]), swap32_sum(t[6], 0.0f));
        float2* o = &sh.end.sums[wid][kc][lane];
        const float2 old = *o;
        *o = make_float2(fmaf(lo, inv_g, old.x), fmaf(hi, inv_g, old.y));
      }
      if constexpr (kByTable) wavefront_lds_sync();  // the next tile rewrites the row factors
    }
    if (base + NW < part_end && base + NW < end) continue;

    // ---- the end of a part
    const float lsum = wave_sum63(sq);
    if (lane == 63) sh.end.loss[wid] = lsum;
    sq = 0.0f;
    const int side_by = finish_parts(P, sh.end, sh.grad, x_mid, part, part_end, end, lane, wid);
    __syncthreads();  // the sums have been read
    for (int kc = 0; kc < chunks; ++kc) sh.end.sums[wid][kc][lane] = make_float2(0.0f, 0.0f);
    part += side_by;
    part_end += max(P.tiles_per_block, NW);
  }
}

// ---- few waves
// A chunk of 16 waves would be mostly padding, and its tables and LDS leave two wavefronts
// on a SIMD, too few to keep the targets coming. Here the sums run on the VALU in FP32: a
// lane takes one column of the strip and steps through the pairs of the tile, theta's
// cosine and sine being a column factor (the lane's, in registers) times P (the pair's, a
// sine and cosine per lane for 64 of them, read back from LDS by the whole wavefront). The
// targets of a pair are one 768-byte run; a tile's are loaded while the one before it is
// summed, the first before the waves' constants are formed. Everything is a stated fused or
// single operation, so that the two kernels that hold it give the same bits.
// What bounds it: small problems the chain of loads, set-up, one tile and the part's end
// (64 x 64 x 4 snapshots, 1 wave: 4.7 us, and the reduction 1.8), large ones the targets'
// traffic (200 problems of 256 x 256 x 16, 1 wave: 5.7 TB/s) and, from 3 waves on, the sums.
// Four wavefronts to a workgroup, not eight (5.3 us for the small problem), tiles of 4 and 8
// pairs, not 16 (8.5 us with its reduction, where it takes 7.3), and a tile's rows formed by
// its lanes and read by lane, not stepped through in scalar registers (7.7).
template <int NW>
struct FitFewShared {
  FitWaveLds wave[8];
  FitWaveGrad grad[kFitFewWavesSmall];
  float4 coef[kFitFewWavesSmall];  // Q A Dx, A, Q A Dz
  float2 dir[kFitFewWavesSmall];   // Q Dx, Q Dz
  float2 column[kFitFewWavesSmall][kStrip];  // cos, sin of kx times the column's offset from the strip's centre
  alignas(16) float2 phase[NW][64];  // P, [pair][wave], 4 or 8 waves to a pair
  FitSums<1, NW> end[2];  // by turns: a part's sums are read while the next part's are formed
};

// The row of pair q = j S + s by a multiply-high: exact for q < 2^18, S <= 32.
struct RowOf {
  uint32_t magic;
  bool one;
  __device__ __forceinline__ explicit RowOf(int S) : magic(0xffffffffu / (uint32_t)S + 1u), one(S == 1) {}
  __device__ __forceinline__ uint32_t operator()(uint32_t q) const { return one ? q : __umulhi(q, magic); }
};

// The pairs of a tile, pair i in every lane l with l mod kPairs = i.
template <int kPairs>
struct PairLanes {
  int row;       // s n + j, the pair's row in the target; the last one's past the last pair
  float j, s;
  __device__ __forceinline__ PairLanes(const FitDesc& P, const RowOf& row_of, int tile, int lane) {
    const uint32_t q = (uint32_t)(tile * kPairs + (lane & (kPairs - 1)));
    const int jj = (int)row_of(q), ss = (int)q - jj * P.S;
    row = ss * P.n + min(jj, P.n - 1);
    j = (float)jj;
    s = (float)ss;
  }
};

// The lane's column of a strip's targets, clamped to the grid.
struct TargetColumn {
  const float* strip;  // the strip's first column in row 0, snapshot 0
  size_t row;          // floats of a row
  uint32_t lane_bytes;
  __device__ __forceinline__ TargetColumn(const FitDesc& P, int strip_index, int lane) {
    const int col0 = strip_index * kStrip;
    strip = P.target + 3 * (size_t)col0;
    row = 3 * (size_t)P.n;
    lane_bytes = 12u * (uint32_t)min(lane, P.n - 1 - col0);
  }
  __device__ __forceinline__ Target3 load(int row_index) const {  // the same for the wavefront
    const char* base = reinterpret_cast<const char*>(strip + (size_t)(uint32_t)row_index * row);
    return *reinterpret_cast<const Target3*>(base + lane_bytes);
  }
};

// v, the same in every lane, in a scalar register.
__device__ __forceinline__ float uniform(float v) {
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

template <int kPairs, int kW, int NW>
__device__ __forceinline__ void few_tiles(const FitDesc& P, const FitUnit& unit, const RowOf& row_of, FitFewShared<NW>& sh,
                                          TargetColumn targets, Target3 (&next)[8], int tid) {
  constexpr int kStride = kW <= 4 ? 4 : 8;
  const int lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t pairs = (uint32_t)P.n * (uint32_t)P.S;
  const int tiles = (int)((pairs + kPairs - 1) / kPairs);
  const int first = unit.part * P.tiles_per_block, end = min(tiles, first + unit.parts * P.tiles_per_block);
  const int col0 = unit.strip * kStrip;
  const bool in_grid = lane < P.n - col0;
  const float offset = (float)lane - 31.5f, half = in_grid ? 0.5f : 0.0f;
  const double x_mid = fma((double)col0 + 31.5, P.spacing, P.x0);
  // column factors (zero past the grid: such a lane's sums stay zero) and coefficients
  float ec[kW], es[kW], bx[kW], by[kW], bz[kW], qx[kW], qz[kW];
#pragma unroll
  for (int w = 0; w < kW; ++w) {
    const float2 e = sh.column[w][lane];
    ec[w] = in_grid ? e.x : 0.0f;
    es[w] = in_grid ? e.y : 0.0f;
    const float4 b = sh.coef[w];
    bx[w] = uniform(b.x);
    by[w] = uniform(b.y);
    bz[w] = uniform(b.z);
    qx[w] = uniform(sh.dir[w].x);
    qz[w] = uniform(sh.dir[w].y);
  }
  // per wave: sums of r_x cos, r_z cos, r_y sin, and of h = r_y cos - Q (D . r) sin plain,
  // times s and times j
  float t[kW][6];
#pragma unroll
  for (int w = 0; w < kW; ++w)
#pragma unroll
    for (int k = 0; k < 6; ++k) t[w][k] = 0.0f;
  float sq = 0.0f;

  int part = unit.strip * P.blocks_per_strip + unit.part, part_end = first + max(P.tiles_per_block, NW);
  int slot = 0, turn = 0;
  PairLanes<kPairs> ahead(P, row_of, first + wid, lane);
#pragma unroll 1
  for (int base = first; base < end; base += NW) {
    const int tile = base + wid;
    if (tile < end) {
      if (slot == 0) {  // P of this tile's pairs and of the wavefront's next tiles'
        int l = lane;
        asm volatile("" : "+v"(l));  // keeps the wave's constants out of the tile loop's live registers
        const uint32_t i = (uint32_t)(l / kStride);
        const uint32_t q = ((uint32_t)tile + i / kPairs * NW) * (uint32_t)kPairs + i % kPairs;
        const uint32_t j = row_of(q), sn = q - j * (uint32_t)P.S;
        const FitWaveLds& w = sh.wave[l & (kStride - 1)];
        const double z = fma((double)j, P.spacing, P.z0), ts = (double)sn * P.dt;
        float c, s;
        sincos_turn(fma(w.om, ts, fma(w.kz, z, fma(w.kx, x_mid, w.c0))), &c, &s);
        const float live = q < pairs ? 1.0f : 0.0f;
        wavefront_lds_sync();  // the last ones have been read
        sh.phase[wid][l] = make_float2(c * live, s * live);
        wavefront_lds_sync();
      }
      // the targets to load meanwhile are the next tile's or, after the last, one place over
      // and over
      const PairLanes<kPairs> now = ahead;
      if (tile + NW < end)
        ahead = PairLanes<kPairs>(P, row_of, tile + NW, lane);
      else
        targets.lane_bytes = 0u;
#pragma unroll
      for (int i = 0; i < kPairs; ++i) {
        const float2* phase = &sh.phase[wid][kStride * (slot + i)];
        float c[kW], s[kW], rx = -next[i].v[0], ry = -next[i].v[1], rz = -next[i].v[2];
#pragma unroll
        for (int w = 0; w < kW; ++w) {
          const float2 p = phase[w];
          c[w] = fmaf(-es[w], p.y, ec[w] * p.x);
          s[w] = fmaf(es[w], p.x, ec[w] * p.y);
          rx = fmaf(bx[w], c[w], rx);
          ry = fmaf(by[w], s[w], ry);
          rz = fmaf(bz[w], c[w], rz);
        }
        next[i] = targets.load(__builtin_amdgcn_readlane(ahead.row, i));
        const float r2 = fmaf(rz, rz, fmaf(ry, ry, rx * rx));
        sq = fmaf((uint32_t)(tile * kPairs + i) < pairs ? half : 0.0f, r2, sq);
        const float jf = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(now.j), i));
        const float sf = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(now.s), i));
#pragma unroll
        for (int w = 0; w < kW; ++w) {
          t[w][0] = fmaf(rx, c[w], t[w][0]);
          t[w][1] = fmaf(rz, c[w], t[w][1]);
          t[w][2] = fmaf(ry, s[w], t[w][2]);
          const float d = fmaf(qx[w], rx, qz[w] * rz);
          const float h = fmaf(-d, s[w], ry * c[w]);
          t[w][3] += h;
          t[w][4] = fmaf(sf, h, t[w][4]);
          t[w][5] = fmaf(jf, h, t[w][5]);
        }
        if ((i & 1) || kW > 4) __builtin_amdgcn_sched_barrier(0);  // every pair's P at once would not fit the registers
      }
      slot = (slot + kPairs) & (64 / kStride - 1);
    }
    if (base + NW < part_end && base + NW < end) continue;

    // ---- the end of a part: a wavefront's sums, row k of 16 lanes holding sums 0, 2, 1, 3
    // and 4, 6, 5 and a zero
    FitSums<1, NW>& of = sh.end[turn];
    const float lsum = wave_sum63(sq);
    if (lane == 63) of.loss[wid] = lsum;
    sq = 0.0f;
#pragma unroll
    for (int w = 0; w < kW; ++w) {
      const float lo = row_sum(swap16_sum(swap32_sum(t[w][0], t[w][1]), swap32_sum(t[w][2], t[w][3])));
      const float hi = row_sum(swap16_sum(swap32_sum(t[w][4], t[w][5]), swap32_sum(t[w][3] * offset, 0.0f)));
      if ((lane & 15) == w) of.sums[wid][0][lane] = make_float2(lo, hi);
#pragma unroll
      for (int k = 0; k < 6; ++k) t[w][k] = 0.0f;
    }
    part += finish_parts(P, of, sh.grad, x_mid, part, part_end, end, lane, wid);
    part_end += max(P.tiles_per_block, NW);
    turn ^= 1;
  }
}

// A unit of a problem of few waves, by NW wavefronts of a workgroup.
template <int NW>
__device__ __forceinline__ void fit_few(const FitDesc& P, const FitUnit& unit, const float (&params)[5],
                                        FitFewShared<NW>& sh, int tid) {
  const int lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  Target3 next[8];
  const RowOf row_of(P.S);
  const bool wide = P.tile_pairs == 8;
  const TargetColumn targets(P, unit.strip, lane);
  auto first_targets = [&](auto count) {
    const PairLanes<count> at(P, row_of, unit.part * P.tiles_per_block + wid, lane);
#pragma unroll
    for (int i = 0; i < count; ++i) next[i] = targets.load(__builtin_amdgcn_readlane(at.row, i));
  };
  if (wide) first_targets(std::integral_constant<int, 8>{});
  else first_targets(std::integral_constant<int, 4>{});
  if (tid < 8) {
    FitWave w{};
    if (tid < P.W) w = fit_wave(P, params);
    sh.wave[tid] = w.lds;
    if (tid < kFitFewWavesSmall) {
      sh.grad[tid] = w.grad;
      sh.coef[tid] = make_float4(w.bx, w.by, w.bz, 0.0f);
      sh.dir[tid] = w.dir;
    }
  }
  __syncthreads();
  static_assert(kStrip == 64, "a lane per column");
  for (int w = wid; w < kFitFewWavesSmall && w < ((P.W + 1) & ~1); w += NW) {
    float c, s;
    sincos_turn(sh.wave[w].kx * P.spacing * ((double)lane - 31.5), &c, &s);
    sh.column[w][lane] = make_float2(c, s);
  }
  __syncthreads();
  if (wide) {
    switch (P.W) {
      case 1: few_tiles<8, 1>(P, unit, row_of, sh, targets, next, tid); break;
      case 2: few_tiles<8, 2>(P, unit, row_of, sh, targets, next, tid); break;
      case 3: few_tiles<8, 3>(P, unit, row_of, sh, targets, next, tid); break;
      default: few_tiles<8, kFitFewWaves>(P, unit, row_of, sh, targets, next, tid); break;
    }
  } else {
    switch (P.W) {
      case 1: few_tiles<4, 1>(P, unit, row_of, sh, targets, next, tid); break;
      case 2: few_tiles<4, 2>(P, unit, row_of, sh, targets, next, tid); break;
      case 3: few_tiles<4, 3>(P, unit, row_of, sh, targets, next, tid); break;
      case 4: few_tiles<4, 4>(P, unit, row_of, sh, targets, next, tid); break;
      default: few_tiles<4, kFitFewWavesSmall>(P, unit, row_of, sh, targets, next, tid); break;
    }
  }
}

__global__ __launch_bounds__(64 * kFitFewWavefronts) __attribute__((amdgpu_waves_per_eu(4)))
void adjoint_few_kernel(const FitDesc* __restrict__ probs, const FitUnit* __restrict__ units, int bump_step) {
  __shared__ FitFewShared<kFitFewWavefronts> sh;
  const FitUnit unit = load_uniform(units, (long long)blockIdx.x);
  const FitDesc P = load_uniform(probs, unit.problem);
  if (bump_step && unit.strip == 0 && unit.part == 0 && threadIdx.x == 0) atomicAdd(P.step, 1);  // as in adjoint_kernel
  const float* pr = P.params + 5 * min((int)threadIdx.x, P.W - 1);
  const float params[5] = {pr[0], pr[1], pr[2], pr[3], pr[4]};
  fit_few(P, unit, params, sh, (int)threadIdx.x);
}

// One workgroup: a unit's strip and parts. KMAX bounds the problem's chunks of 16 waves.
// kFew: units of problems of few waves are among them.
template <int KMAX, int NW, bool kTable, bool kFew>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(NW / 4)))
void adjoint_kernel(const FitDesc* __restrict__ probs, const FitUnit* __restrict__ units, int bump_step) {
  __shared__ FitShared<KMAX, NW, kTable> sh;
  const int tid = threadIdx.x;
  // the problem and unit tables do not change during the launch: scalar loads, so the
  // descriptor sits in SGPRs rather than VGPRs
  const FitUnit unit = load_uniform(units, (long long)blockIdx.x);
  const FitDesc P = load_uniform(probs, unit.problem);
  // Adam step of this iteration, without a result to wait for: the load of `+= 1` held this
  // one workgroup up, and so the launch, by a round trip to memory
  if (bump_step && unit.strip == 0 && unit.part == 0 && tid == 0) atomicAdd(P.step, 1);
  const int chunks = (P.W + 15) >> 4, padded = 16 * chunks;

  // ---- the waves' constants, one thread per wave; the parameters' loads first, so that
  // they are not waited for behind the targets'
  const float* pr = P.params + 5 * min(kFew && P.tile_pairs < 16 ? tid & (64 * kFitFewWavefronts - 1) : tid, P.W - 1);
  const float params[5] = {pr[0], pr[1], pr[2], pr[3], pr[4]};
  if constexpr (kFew) {  // problems of few waves beside the others
    if (P.tile_pairs < 16) {
      // either half of the workgroup takes half of the parts. They pass the same barriers, and a
      // barrier waits for no wavefront that has ended
      static_assert(kFitWavefronts == 2 * kFitFewWavefronts && 2 * sizeof(FitFewShared<kFitFewWavefronts>) <= sizeof(sh));
      const int half = __builtin_amdgcn_readfirstlane(tid / (64 * kFitFewWavefronts)), lower = (unit.parts + 1) >> 1;
      FitUnit few{unit.problem, unit.strip, unit.part + half * lower, half ? unit.parts - lower : lower};
      asm volatile("" : "+s"(few.part));  // opaque, so that neither branch's work is hoisted above it
      if (few.parts == 0) return;
      fit_few(P, few, params, reinterpret_cast<FitFewShared<kFitFewWavefronts>*>(&sh)[half],
              tid & (64 * kFitFewWavefronts - 1));
      return;
    }
  }
  float touch_a, touch_b;
  const int tile = P.tiles_per_block * unit.part + min(tid >> 6, P.tiles_per_block * unit.parts - 1);
  touch_targets(P, unit.strip, min(tile, (P.n * P.S - 1) >> 4), tid & 63, touch_a, touch_b);
  if (tid == 0) sh.max = 0;
  __syncthreads();
  FitWaveLds wv{};
  float bx = 0.0f, by = 0.0f, bz = 0.0f;
  if (tid < P.W) {
    const FitWave w = fit_wave(P, params);
    wv = w.lds;
    bx = w.bx;
    by = w.by;
    bz = w.bz;
    sh.dir[tid] = w.dir;
    sh.grad[tid] = w.grad;
    atomicMax(&sh.max, __float_as_uint(fmaxf(fmaxf(fabsf(bx), fabsf(bz)), fabsf(by))));
  }
  __syncthreads();
  const int coef_exp = scale_exponent(__uint_as_float(__builtin_amdgcn_readfirstlane((int)sh.max)));
  if (tid < padded) {
    const float sc = pow2f(coef_exp);
    sh.coef[tid] = make_float4(bx * sc, by * sc, bz * sc, 0.0f);
    sh.wave[tid] = wv;
    if (tid >= P.W) sh.dir[tid] = make_float2(0.0f, 0.0f);
  }
  __syncthreads();

  // ---- the column factors, per thread and step one wave at two neighbouring offsets t,
  // t + 1: a word of a backward operand's lane slot (wave `slot mod 16` of a chunk, offsets
  // 16 (e / 4) + 4 (slot / 16) + e mod 4, the order in which the forward pass leaves them
  // in a lane), and the same values in the forward operand, whose lane (t mod 16, g) holds
  // waves 4 g .. 4 g + 3 of each chunk
  for (int it = tid; it < chunks * 256; it += 64 * NW) {
    const int slot = it & 63, k = (it >> 6) & 3, kc = it >> 8;
    const int wl = slot & 15;
    const int t = 16 * (k >> 1) + 4 * (slot >> 4) + 2 * (k & 1);
    const bool odd = (chunks & 1) && kc == chunks - 1;
    const double step = sh.wave[16 * kc + wl].kx * P.spacing;  // zero for the padding, whose coefficients are zero
#pragma unroll
    for (int o = 0; o < 2; ++o) {
      float c[2], s2[2];
      sincos_turn(step * ((double)t + 0.5), &c[0], &s2[0]);
      sincos_turn(step * ((double)t + 1.5), &c[1], &s2[1]);
      const float v0 = (o ? s2[0] : c[0]) * kFitTrigScale, v1 = (o ? s2[1] : c[1]) * kFitTrigScale;
      uint32_t hi, lo;
      split2(v0, v1, hi, lo);
      reinterpret_cast<uint32_t*>(&sh.bwd_at(kc, o, 0, 0)[slot])[k] = hi;
      reinterpret_cast<uint32_t*>(&sh.bwd_at(kc, o, 0, 1)[slot])[k] = lo;
      const int fs = (wl >> 2) * 16 + (t & 15);
      _Float16* fh = reinterpret_cast<_Float16*>(&sh.fwd_at(chunks, t >> 4, o, odd ? kc : kc & ~1)[fs]);
      _Float16* fl = reinterpret_cast<_Float16*>(&sh.fwd_at(chunks, t >> 4, o, odd ? kc : kc | 1)[fs]);
      const int eh = 4 * (kc & 1) + (wl & 3), el = odd ? 4 + (wl & 3) : eh;
      fh[eh] = __builtin_bit_cast(Half2, hi).x;
      fh[8 + eh] = __builtin_bit_cast(Half2, hi).y;  // the next lane's slot
      fl[el] = __builtin_bit_cast(Half2, lo).x;
      fl[8 + el] = __builtin_bit_cast(Half2, lo).y;
      split2(((float)t + 0.5f) * v0, ((float)t + 1.5f) * v1, hi, lo);
      reinterpret_cast<uint32_t*>(&sh.bwd_at(kc, o, 1, 0)[slot])[k] = hi;
      reinterpret_cast<uint32_t*>(&sh.bwd_at(kc, o, 1, 1)[slot])[k] = lo;
    }
  }
  // a tile's 16 pairs touch at most four rows from five snapshots on: P is then a row
  // factor times a time factor (4 FMAs per wave and pair, and one sine and cosine per wave
  // and row); below, each pair takes its own sine and cosine. The two ways are two copies
  // of the loop.
  if (kTable && P.S >= 5) {
    for (int it = tid; it < (P.S + 1) * padded; it += 64 * NW) {
      const int sn = it / padded, wi = it - sn * padded;
      float cv = 0.0f, sv = 0.0f;
      if (sn < P.S) sincos_turn(sh.wave[wi].om * ((double)sn * P.dt), &cv, &sv);
      *reinterpret_cast<float2*>(&sh.time[sn * (2 * padded + 4) + 2 * wi]) = make_float2(cv, sv);
    }
    __syncthreads();
    asm volatile("" ::"v"(touch_a), "v"(touch_b));  // the touches are over
    fit_tiles<true>(P, unit, sh, chunks, coef_exp);
  } else {
    __syncthreads();
    fit_tiles<false>(P, unit, sh, chunks, coef_exp);
  }
}

// Block `first` + its own index of the batch's reduce blocks.
__global__ __launch_bounds__(kReduceThreads) void reduce_adam_kernel(const FitDesc* __restrict__ probs,
                                                                  const int* __restrict__ reduce_prob, int first,
                                                                  FitAdam adam, int mode, float* __restrict__ grad_out,
                                                                  float* __restrict__ loss_out) {
  constexpr int kSide = kReduceThreads / kReduceRows;  // parts read side by side
  __shared__ double s[kReduceThreads / 64][kReduceRows];
  const int block = first + (int)blockIdx.x;
  const int prob = load_uniform(reduce_prob, (long long)block);
  const FitDesc P = load_uniform(probs, prob);
  const int r = threadIdx.x & (kReduceRows - 1), side = threadIdx.x / kReduceRows;
  const int row = (block - (int)P.reduce_offset) * kReduceRows + r;
  const int nparam = P.W * 5;
  // the row's Adam state, loaded while the partials are summed (a kernel this short is
  // bound by its chain of memory round trips)
  float m_old = 0.0f, v_old = 0.0f, p_old = 0.0f;
  int t = 0;
  if (side == 0 && mode != 0 && row < nparam) {
    m_old = P.adam_m[row];
    v_old = P.adam_v[row];
    p_old = P.params[row];
    t = P.step[0];
  }
  const float* src = P.partials + min(row, nparam);
  const size_t stride = (size_t)nparam + 1;
  double acc = 0.0;
  for (int b = side; b < P.nblocks; b += 4 * kSide) {
    float v[4];  // four loads in flight
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = src[(size_t)min(b + k * kSide, P.nblocks - 1) * stride];
#pragma unroll
    for (int k = 0; k < 4; ++k) acc += b + k * kSide < P.nblocks ? (double)v[k] : 0.0;
  }
  // fixed order: a wavefront's parts, then the wavefronts in index order
#pragma unroll
  for (int d = kReduceRows; d < 64; d *= 2) acc += __shfl_xor(acc, d);
  if ((threadIdx.x & 63) < kReduceRows) s[threadIdx.x >> 6][r] = acc;
  __syncthreads();
  if (side != 0 || row > nparam) return;
  double sum = s[0][r];
#pragma unroll
  for (int i = 1; i < kReduceThreads / 64; ++i) sum += s[i][r];
  const float total = (float)(sum * (1.0 / ((double)P.S * (double)P.n * (double)P.n)));
  if (row == nparam) {  // loss row
    if (loss_out) loss_out[prob] = total;
    P.loss[0] = total;
    return;
  }
  if (mode == 0) {  // gradient only
    grad_out[P.param_out_offset + row] = total;
    return;
  }
  // Adam (Kingma & Ba, 2015) with bias correction; step counter kept on the device
  const float g = total;
  float m = adam.beta1 * m_old + (1.0f - adam.beta1) * g;
  float v2 = adam.beta2 * v_old + (1.0f - adam.beta2) * g * g;
  P.adam_m[row] = m;
  P.adam_v[row] = v2;
  const float bc1 = 1.0f - powf(adam.beta1, (float)t), bc2 = 1.0f - powf(adam.beta2, (float)t);
  const float mhat = m / bc1, vhat = v2 / bc2;
  float p = p_old - adam.lr * mhat / (sqrtf(vhat) + adam.eps);
  if (row % 5 == 1 && p < 1e-3f) p = 1e-3f;  // wavelength stays positive
  P.params[row] = p;
}

// Synthetic target: displacement of the problem's wave set (read from params) at every
// grid point and snapshot, plus N(0, sigma) noise per component from a counter-based
// generator (SplitMix64 of seed and element index, Box-Muller), so the target does not
// depend on the launch shape. One thread per grid point, phases as in the adjoint.
__device__ __forceinline__ unsigned long long splitmix64(unsigned long long z) {
  z += 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

__device__ __forceinline__ double unit_double(unsigned long long z) { return (double)(z >> 11) * (1.0 / 9007199254740992.0); }

struct SynthWaveLds {
  double kx, kz, c0, om_rev;  // revolutions per metre along x / z, phase at t0 (fract), revolutions per second
  float qadx, qadz, A;
};

__device__ __forceinline__ void stage_synth_wave(const FitDesc& P, int i, SynthWaveLds* o) {
  const float* pr = P.params + 5 * i;
  const double A = pr[0], L = pr[1] > 1e-3f ? pr[1] : 1e-3f, al = pr[2], Q = pr[3], ph0 = pr[4];
  const double w = kTwoPi / L, om = sqrt(P.g * w);
  double sa, ca;
  sincos(al, &sa, &ca);
  o->kx = w * ca * kInvTwoPi;
  o->kz = w * sa * kInvTwoPi;
  const double ph = (om * P.t0 + ph0) * kInvTwoPi;
  o->c0 = ph - floor(ph);
  o->om_rev = om * kInvTwoPi;
  o->A = (float)A;
  o->qadx = (float)(Q * A * ca);
  o->qadz = (float)(Q * A * sa);
}

constexpr int kSynthThreads = 256;
__global__ __launch_bounds__(kSynthThreads) void synthesize_kernel(FitDesc P, float* __restrict__ out, float sigma,
                                                                 unsigned long long seed) {
  __shared__ SynthWaveLds s_wave[kFitMaxWaves];
  for (int i = threadIdx.x; i < P.W; i += blockDim.x) stage_synth_wave(P, i, &s_wave[i]);
  __syncthreads();
  const long long V = (long long)P.n * P.n;
  const long long v = (long long)blockIdx.x * kSynthThreads + threadIdx.x;
  if (v >= V) return;
  const double x = P.x0 + (double)(v % P.n) * P.spacing;
  const double z = P.z0 + (double)(v / P.n) * P.spacing;
  for (int s = 0; s < P.S; ++s) {
    float d0 = 0.0f, d1 = 0.0f, d2 = 0.0f;
    for (int i = 0; i < P.W; ++i) {
      const SynthWaveLds& wv = s_wave[i];
      // phase at snapshot s in FP64: phase at t0 plus omega s dt, reduced to one revolution
      const double ph = fma(wv.kx, x, fma(wv.kz, z, wv.c0)) + wv.om_rev * (P.dt * s);
      const float f = (float)__builtin_amdgcn_fract(ph);
      const float c = __builtin_amdgcn_cosf(f), sn = __builtin_amdgcn_sinf(f);
      d0 = fmaf(wv.qadx, c, d0);
      d1 = fmaf(wv.A, sn, d1);
      d2 = fmaf(wv.qadz, c, d2);
    }
    float* o = out + ((size_t)s * V + v) * 3;
    const float d[3] = {d0, d1, d2};
    for (int k = 0; k < 3; ++k) {
      float nz = 0.0f;
      if (sigma > 0.0f) {
        const unsigned long long idx = ((unsigned long long)s * V + v) * 3 + k;
        const double u1 = fmax(unit_double(splitmix64(seed ^ (2 * idx))), 1e-300);
        const double u2 = unit_double(splitmix64(seed ^ (2 * idx + 1)));
        nz = (float)(sqrt(-2.0 * log(u1)) * cos(kTwoPi * u2));
      }
      o[k] = fmaf(sigma, nz, d[k]);
    }
  }
}

hipError_t launch_synthesize(const FitDesc& P, float* out, float sigma, unsigned long long seed, hipStream_t st) {
  const long long V = (long long)P.n * P.n;
  const long long blocks = (V + kSynthThreads - 1) / kSynthThreads;
  hipLaunchKernelGGL(synthesize_kernel, dim3((unsigned)blocks), dim3(kSynthThreads), 0, st, P, out, sigma, seed);
  return hipGetLastError();
}

__global__ void zero_words_kernel(uint32_t* __restrict__ p, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = 0u;
}

hipError_t launch_zero_words(uint32_t* p, size_t n, hipStream_t st) {
  if (n == 0) return hipSuccess;
  size_t blocks = (n + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(zero_words_kernel, dim3((unsigned)blocks), dim3(256), 0, st, p, n);
  return hipGetLastError();
}

__global__ void fit_setup_single_kernel(FitDesc d, FitDesc* __restrict__ d_desc, FitUnit* __restrict__ d_units,
                                        size_t units, uint32_t* __restrict__ zero_begin, size_t zero_words) {
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  const size_t i0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i0 == 0) *d_desc = d;
  for (size_t i = i0; i < units; i += stride) {
    const int strip = (int)i / d.blocks_per_strip;
    d_units[i] = FitUnit{0, strip, (int)i - strip * d.blocks_per_strip, 1};
  }
  for (size_t i = i0; i < zero_words; i += stride) zero_begin[i] = 0u;
}

hipError_t launch_fit_setup_single(const FitDesc& d, FitDesc* d_desc, FitUnit* d_units, size_t units,
                                   uint32_t* zero_begin, size_t zero_words, hipStream_t st) {
  size_t n = units > zero_words ? units : zero_words;
  size_t blocks = (n + 255) / 256;
  if (blocks < 1) blocks = 1;
  if (blocks > 1024) blocks = 1024;
  hipLaunchKernelGGL(fit_setup_single_kernel, dim3((unsigned)blocks), dim3(256), 0, st, d, d_desc, d_units, units,
                     zero_begin, zero_words);
  return hipGetLastError();
}

// Calls launch(first, blocks) for the runs of `blocks` workgroups of `threads` that one launch
// may have: past 2^32 threads a launch reports no error and leaves workgroups out.
template <class Launch>
hipError_t in_launches(long long blocks, int threads, Launch launch) {
  const long long most = (1ll << 31) / threads;
  for (long long first = 0; first < blocks; first += most) {
    launch(first, dim3((unsigned)std::min(most, blocks - first)));
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// The adjoint launch of class c on stream st.
template <int C>
hipError_t launch_adjoint_class(const FitLaunch& L, int c, int bump, hipStream_t st) {
  if (c == C) {
    const int threads = 64 * (C == 0 ? kFitFewWavefronts : kFitWavefronts);
    return in_launches(L.class_blocks[C], threads, [&](long long first, dim3 grid) {
      const FitUnit* units = L.units + L.class_begin[C] + first;
      if constexpr (C == 0)
        hipLaunchKernelGGL(adjoint_few_kernel, grid, dim3(threads), 0, st, L.probs, units, bump);
      else
        hipLaunchKernelGGL((C == 1 && L.mixed ? adjoint_kernel<kFitClassChunks[C], kFitWavefronts, C == 1, C == 1>
                                              : adjoint_kernel<kFitClassChunks[C], kFitWavefronts, C == 1, false>),
                           grid, dim3(threads), 0, st, L.probs, units, bump);
    });
  }
  if constexpr (C + 1 < kFitClasses) return launch_adjoint_class<C + 1>(L, c, bump, st);
  return hipErrorInvalidValue;
}

hipError_t launch_fit_iteration(const FitLaunch& L, const FitAdam& adam, int mode, float* grad_out, float* loss_out,
                                hipStream_t st) {
  const int bump = mode == 1 ? 1 : 0;
  // the class with the most work (blocks x waves), and the other one if there are two
  auto work = [&](int c) { return (double)L.class_blocks[c] * kFitClassChunks[c]; };
  int big = 0, other = -1;
  for (int c = 1; c < kFitClasses; ++c)
    if (work(c) > work(big)) big = c;
  for (int c = 0; c < kFitClasses; ++c)
    if (c != big && L.class_blocks[c] > 0) other = c;
  hipError_t e = hipSuccess;
  if (other >= 0) {
    // on the side stream: the classes write disjoint partials and step counters, so they
    // may overlap
    if ((e = hipEventRecord(L.fork, st)) != hipSuccess) return e;
    if ((e = hipStreamWaitEvent(L.side, L.fork, 0)) != hipSuccess) return e;
  }
  if ((e = launch_adjoint_class<0>(L, big, bump, st)) != hipSuccess) return e;
  if (other >= 0) {
    if ((e = launch_adjoint_class<0>(L, other, bump, L.side)) != hipSuccess) return e;
    if ((e = hipEventRecord(L.join, L.side)) != hipSuccess) return e;
    if ((e = hipStreamWaitEvent(st, L.join, 0)) != hipSuccess) return e;
  }
  return in_launches(L.reduce_blocks, kReduceThreads, [&](long long first, dim3 grid) {
    hipLaunchKernelGGL(reduce_adam_kernel, grid, dim3(kReduceThreads), 0, st, L.probs, L.reduce_prob, (int)first, adam, mode,
                       grad_out, loss_out);
  });
}

}  // namespace wt
