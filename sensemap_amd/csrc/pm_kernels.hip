// pm_kernels.hip -- gfx950 kernels of the PatchMatch MVS engine.
//
// A 256-thread workgroup owns a 32x16 pixel tile (its 256 pixels of one
// checkerboard colour), or a 16x8 or 8x4 one in small launches.  The sweep and the
// local optimisation list the (hypothesis, pixel) pairs that need a cost and
// walk the windows of 64 pairs per wave; neighbouring pairs are neighbouring
// pixels, so the windows of a wave overlap and their source footprints hit
// the same cache lines.  Per workgroup the
// reference tile (+ window halo; one 32-bit word per texel holding the
// intensity and 3x the intensity, see ncc_eval) and the 256-entry bilateral colour
// table are staged in LDS; the spatial weight table and the per-source pose
// blocks are read with uniform (scalar) loads because the source loop and
// the window position are uniform across the wave.  Source images live in
// HBM in a zero-padded "quad" layout: texel (x, y) holds the 2x2 bilinear
// footprint {(x,y), (x+1,y), (x,y+1), (x+1,y+1)}, so one 32-bit (u8) or
// 64-bit (f16) load feeds one bilinear sample with no bounds checks.
//
// Per-pixel arithmetic follows the canonical FP32 order of the CPU
// transcription (oracle/pm_oracle.c): -ffp-contract=off, explicit fmaf,
// correctly rounded division and sqrt, project math from pm_math.h.  With
// PM_RCP_EXACT the maps are bitwise equal to the transcription's.
//
// Reference semantics (src/mvs/kernel_functions.cu):
//   k_ref_moments   <- FilterKernel (gpu_mat_ref_image.cu:16-56) + ComputeGradientMap (:1655-1675)
//   k_init          <- FillWithRandomNumbers/InitNormalMap/InitDepthMap (:689-737) + InitConfMapKernel (:1497-1601)
//   k_sweep         <- Black/RedPixelUpdateOpt -> SweepFromCheckerBoardOpt (:2136-2560, :2634-2734)
//   k_local_opt     <- Black/RedPixelLocalOptimization -> LocalOptimization (:2736-3017)
//   k_filter        <- FilterDepthMap (:3282-3354)
//   k_curvature     <- ComputeCurvatureMap (:1603-1651)
//   k_mask          <- MaskDepthMapKernel (:3080-3093)
//   k_geom_grad     <- ComputeGeomGradientMap (:3095-3120)
//   k_median        <- BlackPixelFilter / RedPixelFilter -> MedianFilter (:3122-3280)
//   ncc_eval        <- ComputeNCCCost<R,S> (:1245-1340) with ComposeHomography (:431-503)
//   geom_eval       <- ComputeGeomConsistencyCostShared (:505-568)
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <type_traits>

#include <map>
#include <mutex>
#include <utility>

#include "pm_device.h"
#include "pm_math.h"

namespace pm {
namespace {

// Pointers stored in ViewDev are generic; cast them to the global address
// space so loads and stores compile to global_* (or s_load for uniform
// addresses) instead of flat_*.
// A view descriptor as the colour-pass kernels read it: through the
// constant address space, so that the compiler may use scalar loads (the
// descriptor is written only by host copies between launches) and keeps
// its fields, the source texture bases among them, in scalar registers.
using VPtr = const __attribute__((address_space(4))) ViewDev*;
template <typename T>
using K4 = const __attribute__((address_space(4))) T;

template <typename T>
__device__ __forceinline__ __attribute__((address_space(1))) T* G(T* p) {
  return (__attribute__((address_space(1))) T*)p;
}

typedef float f4v __attribute__((ext_vector_type(4)));
typedef unsigned int u2v __attribute__((ext_vector_type(2)));

// 16-byte load of a float4 array element through the global address space.
__device__ __forceinline__ f4v ld_f4(const float4* p, int idx) {
  return *((const __attribute__((address_space(1))) f4v*)p + idx);
}

__constant__ int c_neighbor_offs[4][2] = {{0, -1}, {-1, 0}, {0, 1}, {1, 0}};
// Sample f of direction gi (dirSamples, kernel_functions.cu): for gi < 4 the
// wedge (-1, 2), (1, 2), (-2, 3), (2, 3) .. along its axis, for the others the
// odd distances 3, 5 .. 21; the axis is the columns for gi & 2 == 0, the rows
// otherwise, and points to smaller indices for even gi.  Computed, since the lanes of a wave
// may take different directions.
__device__ __forceinline__ void dir_sample(int gi, int sign, int f, int& dr, int& dc) {
  const int m = f / 2 + 1;
  const int along = sign * (gi < 4 ? m + 1 : 3 + 2 * f);
  const int across = gi < 4 ? ((f & 1) ? m : -m) : 0;
  dr = (gi & 2) ? along : across;
  dc = (gi & 2) ? across : along;
}
__constant__ float c_mweights[5] = {0.f, 1.f, 2.01f, 3.03f, 4.06f};

// ---------------------------------------------------------------------------
// per-lane pixel context

struct Pix {
  int row, col, lrow, lcol;
  int p;                 // row * W + col
  int c;                 // ref centre intensity (u8)
  float mu_r, var_r, inv_sw, err_r;
  float np0, np1;        // normalized point (x, y, 1)
  bool shifted;          // compensated moments for this pixel
};

// Workspace of one workgroup: a contiguous region of the launch's workspace
// holding, per pixel of a tile, hypotheses and costs ([field][pixel], so the
// pixels of a wave read consecutive words).  npx pixels per tile.
struct Ws {
  float* base;
  int npx, N;
  __device__ __attribute__((address_space(1))) f4v& hyp(int k, int px) const {
    return ((__attribute__((address_space(1))) f4v*)G(base))[k * npx + px];
  }
  __device__ __attribute__((address_space(1))) float& at(int row, int px) const {
    return G(base)[4 * (kMaxHyp + kNumRefine) * npx + row * npx + px];
  }
  __device__ __attribute__((address_space(1))) float& M(int k, int i, int px) const { return at(k * N + i, px); }
  __device__ __attribute__((address_space(1))) float& RM(int k, int i, int px) const { return at((kMaxHyp + k) * N + i, px); }
  __device__ __attribute__((address_space(1))) float& Wt(int i, int px) const {
    return at((kMaxHyp + kNumRefine) * N + i, px);
  }
};

// Per-thread counts of one pixel's phase, 32 bits: even the largest window
// (65x65) x 32 sources x 16 evaluations is 2.2e6 samples per pixel and
// phase (init: init_samples <= 64, checked by pm_options_check).
struct Counters {
  uint32_t ncc_eval = 0, ncc_samples = 0, geo_eval = 0;
};

// Counter slots: [0..2] all kernels, [3..5] the sweep kernel alone.
__device__ __forceinline__ void flush_counters(VPtr v, const Counters& c, bool sweep = false) {
  if (v->counters) {
    atomicAdd(&v->counters[0], (unsigned long long)c.ncc_eval);
    atomicAdd(&v->counters[1], (unsigned long long)c.ncc_samples);
    atomicAdd(&v->counters[2], (unsigned long long)c.geo_eval);
    if (sweep) {
      atomicAdd(&v->counters[3], (unsigned long long)c.ncc_eval);
      atomicAdd(&v->counters[4], (unsigned long long)c.ncc_samples);
      atomicAdd(&v->counters[5], (unsigned long long)c.geo_eval);
    }
  }
}

// 1/z of a window sample.
// PM_RCP_EXACT: v_rcp_f32 refined by two Newton steps with FMA.  On gfx950
//   v_rcp_f32 is within one ulp of the correctly rounded reciprocal for every
//   significand (and scales exactly with exponent and sign), and two Newton
//   steps from any seed within one ulp land on the correctly rounded value,
//   so this equals 1.0f / z for every normal z, bit for bit, at about half
//   the instructions of the IEEE division sequence.
// PM_RCP_FAST: one Newton step (within one ulp, not always correctly rounded).
template <int RCP>
__device__ __forceinline__ float rcp_z(float z) {
  float r = __builtin_amdgcn_rcpf(z);
  float e = fmaf(-z, r, 1.0f);
  r = fmaf(r, e, r);
  if constexpr (RCP == PM_RCP_EXACT) {
    e = fmaf(-z, r, 1.0f);
    r = fmaf(r, e, r);
  }
  return r;
}

// The 2x2 footprint of source texel (x0, y0) in the quad layout: one
// 4-byte (u8) or 8-byte (f16) load.  tex is uniform across the wave (the
// source loop is uniform) and off is the 32-bit texel index, so the load
// uses the scalar-base + 32-bit-offset form.
template <int STORE>
struct Quad {
  using type = uint32_t;
};
template <>
struct Quad<PM_STORAGE_F16> {
  using type = u2v;
};

template <int STORE>
__device__ __forceinline__ typename Quad<STORE>::type load_quad(const void* tex, uint32_t boff) {
  const __attribute__((address_space(1))) char* b = G((const char*)tex);
  if constexpr (STORE == PM_STORAGE_U8) {
    return *(const __attribute__((address_space(1))) uint32_t*)(b + boff);
  } else {
    return *(const __attribute__((address_space(1))) u2v*)(b + boff);
  }
}

// Bilinear value of a quad at fraction (fx, fy):
// top = t00 + fx (t01 - t00), bot = t10 + fx (t11 - t10), top + fy (bot - top).
// The f16 quad holds (t00, t01 - t00, t10, t11 - t10), all exact, so the
// two horizontal lerps read the halves directly (v_fma_mix_f32) and give the
// same bits as the u8 path.
template <int STORE>
__device__ __forceinline__ float bilerp(typename Quad<STORE>::type q, float fx, float fy) {
  float top, bot;
  if constexpr (STORE == PM_STORAGE_U8) {
    const float t0 = (float)(q & 0xffu);
    const float t1 = (float)((q >> 8) & 0xffu);
    const float t2 = (float)((q >> 16) & 0xffu);
    const float t3 = (float)(q >> 24);
    top = fmaf(fx, t1 - t0, t0);
    bot = fmaf(fx, t3 - t2, t2);
  } else {
    const float t0 = __half2float(__ushort_as_half((unsigned short)(q.x & 0xffffu)));
    const float d01 = __half2float(__ushort_as_half((unsigned short)(q.x >> 16)));
    const float t2 = __half2float(__ushort_as_half((unsigned short)(q.y & 0xffffu)));
    const float d23 = __half2float(__ushort_as_half((unsigned short)(q.y >> 16)));
    top = fmaf(fx, d01, t0);
    bot = fmaf(fx, d23, t2);
  }
  return fmaf(fy, bot - top, top);
}

// floor(x) as int in one instruction (v_cvt_flr_i32_f32); the compiler
// emits v_floor_f32 + v_cvt_i32_f32 for (int)floorf(x).  Exact for the
// clamped coordinate range [-3, W+2].
__device__ __forceinline__ int cvt_flr(float x) {
  int r;
  asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(r) : "v"(x));
  return r;
}

__device__ __forceinline__ void neumaier_add(float& s, float& c, float x) {
  const float t = s + x;
  c = c + ((fabsf(s) >= fabsf(x)) ? ((s - t) + x) : ((x - t) + s));
  s = t;
}

// Texel loads a window row keeps in flight (build knob).
#ifndef PM_PIPE_DEPTH
#define PM_PIPE_DEPTH 3
#endif

// ComputeNCCCost (kernel_functions.cu:1245-1340) for source i (uniform) and
// the lane's hypothesis.  tile points at the LDS ref tile entry of the
// window's top-left sample; tw is the tile row length.
template <int R_, int S_, int STORE, int RCP>
__device__ __forceinline__ float ncc_eval(VPtr v, int i, const Pix& px,
                                          const uint32_t* tile, int tw, const float* ct, const float* sp,
                                          float nx, float ny, float nz, float d, Counters& cnt) {
  const int R = R_ >= 0 ? R_ : v->radius;
  const int S = R_ >= 0 ? S_ : v->step;
  const int n = R_ >= 0 ? (2 * R_) / S_ + 1 : v->nwin;
  cnt.ncc_eval++;
  const __attribute__((address_space(1))) float* pose = G(v->poses) + i * PM_POSE_STRIDE;
  const float K0 = pose[0], K1 = pose[1], K2 = pose[2], K3 = pose[3];
  const __attribute__((address_space(1))) float* Rm = pose + 4;
  const __attribute__((address_space(1))) float* T = pose + 13;
  K4<float>* iK = v->refInvK;
  const float fcol = (float)px.col, frow = (float)px.row;
  const float ray0 = iK[0] * fcol + iK[1];
  const float ray1 = iK[2] * frow + iK[3];
  const float dist = d * (nx * ray0 + ny * ray1 + nz);
  const float inv_dist = 1.0f / dist;
  const float nd0 = inv_dist * nx, nd1 = inv_dist * ny, nd2 = inv_dist * nz;
  float A[9];
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    A[3 * r + 0] = Rm[3 * r + 0] + nd0 * T[r];
    A[3 * r + 1] = Rm[3 * r + 1] + nd1 * T[r];
    A[3 * r + 2] = Rm[3 * r + 2] + nd2 * T[r];
  }
  float B[9];
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    B[j] = K0 * A[j] + K1 * A[6 + j];
    B[3 + j] = K2 * A[3 + j] + K3 * A[6 + j];
    B[6 + j] = A[6 + j];
  }
  float H[9];
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    H[3 * r + 0] = B[3 * r + 0] * iK[0];
    H[3 * r + 1] = B[3 * r + 1] * iK[2];
    H[3 * r + 2] = B[3 * r + 0] * iK[1] + B[3 * r + 1] * iK[3] + B[3 * r + 2];
  }
  const float zc = H[6] * fcol + H[7] * frow + H[8];
  const float izc = 1.0f / zc;
  const float xf = (H[0] * fcol + H[1] * frow + H[2]) * izc;
  const float yf = (H[3] * fcol + H[4] * frow + H[5]) * izc;
  K4<SrcDev>& s = v->src[i];
  const float Wsf = (float)s.width, Hsf = (float)s.height;
  if (!(xf > -1.0f && xf < Wsf && yf > -1.0f && yf < Hsf)) return kMaxCost;
  if (px.var_r < kVarThreshold) return kMaxCost;
  const float c0 = (float)(px.col - R), r0 = (float)(px.row - R);
  float bx = H[0] * c0 + H[1] * r0 + H[2];
  float by = H[3] * c0 + H[4] * r0 + H[5];
  float bz = H[6] * c0 + H[7] * r0 + H[8];
  const float fs = (float)S;
  const float hxc = fs * H[0], hyc = fs * H[3], hzc = fs * H[6];
  const float hxr = fs * H[1], hyr = fs * H[4], hzr = fs * H[7];
  const float umax = Wsf + 2.0f, vmax = Hsf + 2.0f;
  const int pitch = s.pitch;
  const void* tex = s.tex;
  const uint32_t c4 = ((uint32_t)px.c << 16) | (3u * (uint32_t)px.c);
  float s1 = 0.0f, s2 = 0.0f, s3 = 0.0f;
  float e1 = 0.0f, e2 = 0.0f, e3 = 0.0f;
  const float mu_r = px.mu_r;
  const int ipitch = pitch;
  constexpr uint32_t kQuadShift = STORE == PM_STORAGE_U8 ? 2u : 3u;  // bytes per quad: 4 or 8
  const uint32_t pad_bytes = (uint32_t)(kQuadPad * pitch + kQuadPad) << kQuadShift;
  // One window walk; SHIFTED selects the compensated moment update.  A
  // sample is issued (projection, fraction, texel load) ahead of its use:
  // with compile-time window shapes each row keeps kDepth loads in flight,
  // so a wave waits for memory once per row instead of once per sample.
  // Issue order, arithmetic and accumulation order are those of a plain
  // sample-by-sample walk.
  struct Smp {
    float fx, fy;
    typename Quad<STORE>::type q;
  };
  auto issue = [&](float x, float y, float z, auto clamp_tag) __attribute__((always_inline)) {
    const float rz = rcp_z<RCP>(z);
    float u = x * rz, w_ = y * rz;
    if constexpr (decltype(clamp_tag)::value) {
      // clamp to [-3, W+2]: v_med3_f32 equals fminf(fmaxf(u, -3), umax) for
      // every input, NaN and infinities included (a NaN goes to -3)
      u = __builtin_amdgcn_fmed3f(u, -3.0f, umax);
      w_ = __builtin_amdgcn_fmed3f(w_, -3.0f, vmax);
    }
    Smp sm;
    // fraction = min(u - floor(u), 1 - 2^-24): v_fract_f32
    sm.fx = __builtin_amdgcn_fractf(u);
    sm.fy = __builtin_amdgcn_fractf(w_);
    const int x0 = cvt_flr(u), y0 = cvt_flr(w_);
    // texel (x0 + 4, y0 + 4) of the padded image, as a byte offset: the
    // signed y0 * pitch + x0 (>= -3 pitch - 3) plus the uniform padding offset
    const int t = __mul24(y0, ipitch) + x0;
    const uint32_t boff = ((uint32_t)t << kQuadShift) + pad_bytes;
    sm.q = load_quad<STORE>(tex, boff);
    // keep the load where it is issued: without this the scheduler sinks
    // the f16 loads next to their use and the row's loads no longer overlap
    __builtin_amdgcn_sched_barrier(0);
    return sm;
  };
  auto walk = [&](auto shifted_tag, auto clamp_tag) __attribute__((always_inline)) {
    constexpr bool kShifted = decltype(shifted_tag)::value;
    for (int ir = 0; ir < n; ++ir) {
      const uint32_t* trow = tile + ir * S * tw;
      const float* sprow = sp + ir * n;
      auto consume = [&](int j, const Smp& sm) __attribute__((always_inline)) {
        const float sv = bilerp<STORE>(sm.q, sm.fx, sm.fy);
        // tile word (ri << 16) | 3 ri: byte 2 is the intensity; v_sad_u16
        // adds the absolute differences of both 16-bit halves, so against
        // the centre's (c << 16) | 3 c it gives 3|ri - c| + |ri - c| =
        // 4|ri - c|, the colour weight's LDS byte offset
        const uint32_t tw4 = trow[j * S];
        const float r = (float)((tw4 >> 16) & 0xffu);  // v_cvt_f32_ubyte2
        const float w = sprow[j] * *(const float*)((const char*)ct + __builtin_amdgcn_sad_u16(tw4, c4, 0u));
        if constexpr (!kShifted) {
          const float ws = w * sv;
          s1 = s1 + ws;
          s2 = fmaf(ws, sv, s2);
          s3 = fmaf(ws, r, s3);
        } else {
          const float dd = sv - mu_r;
          const float rd = r - mu_r;
          const float wd = w * dd;
          neumaier_add(s1, e1, wd);
          neumaier_add(s2, e2, wd * dd);
          neumaier_add(s3, e3, wd * rd);
        }
      };
      float x = bx, y = by, z = bz;  // the next sample to issue
      if constexpr (R_ >= 0) {
        constexpr int kN = R_ >= 0 ? (2 * R_) / S_ + 1 : 1;
        constexpr int kDepth = kN < PM_PIPE_DEPTH ? kN : PM_PIPE_DEPTH;
        Smp ring[kDepth];
#pragma unroll
        for (int j = 0; j < kDepth; ++j) {
          ring[j] = issue(x, y, z, clamp_tag);
          x = x + hxc;
          y = y + hyc;
          z = z + hzc;
        }
#pragma unroll
        for (int j = 0; j < kN; ++j) {
          const Smp cur = ring[j % kDepth];
          if (j + kDepth < kN) {
            ring[j % kDepth] = issue(x, y, z, clamp_tag);
            x = x + hxc;
            y = y + hyc;
            z = z + hzc;
          }
          consume(j, cur);
        }
      } else {
        for (int j = 0; j < n; ++j) {
          const Smp cur = issue(x, y, z, clamp_tag);
          x = x + hxc;
          y = y + hyc;
          z = z + hzc;
          consume(j, cur);
        }
      }
      bx = bx + hxr;
      by = by + hyr;
      bz = bz + hzr;
    }
  };
  // The clamps are identities when every sample lands inside [-3, W+2] x
  // [-3, H+2].  Under the homography the window maps onto the convex
  // quadrilateral of its 4 corner samples when z > 0 at all of them (z is
  // affine over the window, so its minimum is at a corner).  Corners at
  // least kInsideMargin px inside the range with z varying by at most 4x
  // bound the incremental walk's rounding (<= ~30 ulp of the homogeneous
  // coordinates, < 0.2 px for images up to 2^14 px wide) well below the
  // margin, so such a window needs no clamp.  The choice is wave-uniform:
  // one lane near a border keeps the clamped walk for the wave.
  bool inside;
  {
    constexpr float kInsideMargin = 0.5f;
    const float span = (float)(n - 1);
    const float ex = span * hxc, ey = span * hyc, ez = span * hzc;
    const float fx_ = span * hxr, fy_ = span * hyr, fz_ = span * hzr;
    const float cx[4] = {bx, bx + ex, bx + fx_, (bx + ex) + fx_};
    const float cy[4] = {by, by + ey, by + fy_, (by + ey) + fy_};
    const float cz[4] = {bz, bz + ez, bz + fz_, (bz + ez) + fz_};
    float zmin = cz[0], zmax = cz[0];
    bool ok = true;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      zmin = fminf(zmin, cz[k]);
      zmax = fmaxf(zmax, cz[k]);
      const float iz = __builtin_amdgcn_rcpf(cz[k]);  // a test with a margin: the approximation serves
      const float u = cx[k] * iz, w_ = cy[k] * iz;
      ok = ok && u >= -3.0f + kInsideMargin && u <= umax - kInsideMargin && w_ >= -3.0f + kInsideMargin &&
           w_ <= vmax - kInsideMargin;
    }
    inside = __all(ok && zmin > 0.0f && zmax <= 4.0f * zmin);
  }
  if (!px.shifted) {
    if (inside)
      walk(std::false_type{}, std::false_type{});
    else
      walk(std::false_type{}, std::true_type{});
  } else {
    walk(std::true_type{}, std::true_type{});
  }
  cnt.ncc_samples += (uint32_t)(n * n);
  const float inv_sw = px.inv_sw;
  float var_s, cov;
  if (!px.shifted) {
    const float mu_s = s1 * inv_sw;
    const float m2_s = s2 * inv_sw;
    const float m_rs = s3 * inv_sw;
    var_s = m2_s - mu_s * mu_s;
    cov = m_rs - mu_r * mu_s;
  } else {
    const float m1 = (s1 + e1) * inv_sw;
    const float m2 = (s2 + e2) * inv_sw;
    const float m3 = (s3 + e3) * inv_sw;
    var_s = m2 - m1 * m1;
    cov = m3 - px.err_r * m1;
  }
  if (var_s < kVarThreshold) return kMaxCost;
  const float val = 1.0f - cov / sqrtf(px.var_r * var_s);
  return fmaxf(0.0f, fminf(kMaxCost, val));
}

// ComputeGeomConsistencyCostShared (kernel_functions.cu:505-568).
__device__ __forceinline__ float geom_eval(VPtr v, int i, const Pix& px, float depth,
                                           K4<float>* K, Counters& cnt) {
  cnt.geo_eval++;
  const __attribute__((address_space(1))) float* P = G(v->poses) + i * PM_POSE_STRIDE + 16;
  const __attribute__((address_space(1))) float* iP = G(v->poses) + i * PM_POSE_STRIDE + 28;
  const float fx = depth * px.np0, fy = depth * px.np1, fz = depth * 1.0f;
  const float inv_fz = 1.0f / (P[8] * fx + P[9] * fy + P[10] * fz + P[11]);
  float sc = inv_fz * (P[0] * fx + P[1] * fy + P[2] * fz + P[3]);
  float sr = inv_fz * (P[4] * fx + P[5] * fy + P[6] * fz + P[7]);
  K4<SrcDev>& s = v->src[i];
  float u = fminf(fmaxf(sc, -3.0f), (float)s.width + 2.0f);
  float w_ = fminf(fmaxf(sr, -3.0f), (float)s.height + 2.0f);
  const float x0f = floorf(u), y0f = floorf(w_);
  const float fxx = u - x0f, fyy = w_ - y0f;
  const f4v q = ld_f4(s.depth_q, ((int)y0f + kQuadPad) * s.pitch + ((int)x0f + kQuadPad));
  const float top = fmaf(fxx, q.y - q.x, q.x);
  const float bot = fmaf(fxx, q.w - q.z, q.z);
  const float sd = fmaf(fyy, bot - top, top);
  if (sd == 0.0f) return v->geom_max_cost;
  sc = sc * sd;
  sr = sr * sd;
  const float bx = iP[0] * sc + iP[1] * sr + iP[2] * sd + iP[3];
  const float by = iP[4] * sc + iP[5] * sr + iP[6] * sd + iP[7];
  const float bz = iP[8] * sc + iP[9] * sr + iP[10] * sd + iP[11];
  const float ibz = 1.0f / bz;
  const float bcol = ibz * K[0] * bx + K[1];
  const float brow = ibz * K[2] * by + K[3];
  const float dc = (float)px.col - bcol;
  const float dr = (float)px.row - brow;
  return fminf(v->geom_max_cost, sqrtf(dc * dc + dr * dr));
}

// ComputeMultiViewCostVector (kernel_functions.cu:1447-1495), priors off.
template <int R_, int S_, int STORE, int RCP>
__device__ __forceinline__ float mv_cost(VPtr v, int i, const Pix& px, const uint32_t* tile,
                                         int tw, const float* ct, const float* sp, float nx, float ny, float nz,
                                         float d, K4<float>* Kgeo, Counters& cnt) {
  float cost = ncc_eval<R_, S_, STORE, RCP>(v, i, px, tile, tw, ct, sp, nx, ny, nz, d, cnt);
  if (v->geom) cost = cost + v->geom_regularizer * geom_eval(v, i, px, d, Kgeo, cnt);
  return cost;
}

// ---------------------------------------------------------------------------
// random hypotheses (identical to the transcription)

__device__ __forceinline__ void random_normal(pm_rng* g, float r0, float r1, float n[3]) {
  float v1 = 0.0f, v2 = 0.0f, s = 2.0f;
  for (int t = 0; t < 64 && s >= 1.0f; ++t) {
    v1 = 2.0f * pm_rng_uniform(g) - 1.0f;
    v2 = 2.0f * pm_rng_uniform(g) - 1.0f;
    s = v1 * v1 + v2 * v2;
  }
  if (s >= 1.0f) {
    v1 = 0.0f;
    v2 = 0.0f;
    s = 0.0f;
  }
  const float s_norm = 2.0f * sqrtf(1.0f - s);
  n[0] = v1 * s_norm;
  n[1] = v2 * s_norm;
  n[2] = 1.0f - 2.0f * s;
  if (n[0] * r0 + n[1] * r1 + n[2] * 1.0f > 0.0f) {
    n[0] = -n[0];
    n[1] = -n[1];
    n[2] = -n[2];
  }
}

__device__ __forceinline__ float random_depth(pm_rng* g, float dmin, float dmax) {
  return pm_rng_uniform(g) * (dmax - dmin) + dmin;
}

__device__ __forceinline__ void perturb_normal(pm_rng* g, const float n[3], float a1, float a2, float out[3]) {
  const float y = pm_atan2f(sqrtf(n[0] * n[0] + n[1] * n[1]), n[2]);
  const float x = pm_atan2f(n[1], n[0]);
  const float nx = a1 * (2.0f * pm_rng_uniform(g) - 1.0f) + x;
  const float ny = a2 * (2.0f * pm_rng_uniform(g) - 1.0f) + y;
  const float siny = pm_sinf(ny);
  out[0] = pm_cosf(nx) * siny;
  out[1] = pm_sinf(nx) * siny;
  out[2] = pm_cosf(ny);
}

// CorrectNormal (kernel_functions.cu:227-306) with the reference's matrix.
__device__ __forceinline__ void correct_normal(float n[3], const float vd[3], float inv_view_len) {
  const float cosl = n[0] * vd[0] + n[1] * vd[1] + n[2] * vd[2];
  if (!(cosl >= 0.0f)) return;
  float c[3];
  c[0] = n[1] * vd[2] - n[2] * vd[1];
  c[1] = n[2] * vd[0] - n[0] * vd[2];
  c[2] = n[0] * vd[1] - n[1] * vd[0];
  const float a = cosl * inv_view_len;
  float phi;
  if (!(a <= 1.0f)) {
    phi = -0.001f;
  } else {
    phi = pm_acosf(a) - PM_HALF_PI_F;
    phi = fminf(phi * 1.01f, -0.001f);
  }
  const float inv_len = 1.0f / sqrtf(c[0] * c[0] + c[1] * c[1] + c[2] * c[2]);
  c[0] = c[0] * inv_len;
  c[1] = c[1] * inv_len;
  c[2] = c[2] * inv_len;
  const float o[9] = {0.0f, -c[2], c[1], c[2], 0.0f, -c[0], -c[1], c[0], 0.0f};
  const float sp = pm_sinf(phi);
  const float cp = 1.0f - pm_cosf(phi);
  float oo[9];
  oo[0] = cp * (o[0] * o[0] + o[1] * o[3] + o[2] * o[6]);
  oo[1] = cp * (o[0] * o[1] + o[1] * o[4] + o[2] * o[7]);
  oo[2] = cp * (o[0] * o[2] + o[1] * o[5] + o[2] * o[8]);
  oo[3] = cp * (o[3] * o[0] + o[4] * o[3] + o[5] * o[6]);
  oo[4] = oo[3];
  oo[5] = oo[3];
  oo[6] = cp * (o[6] * o[0] + o[7] * o[3] + o[8] * o[6]);
  oo[7] = oo[6];
  oo[8] = oo[6];
  float Rr[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    const float id = (k == 0 || k == 4 || k == 8) ? 1.0f : 0.0f;
    Rr[k] = id + o[k] * sp + oo[k];
  }
  const float r0 = Rr[0] * n[0] + Rr[1] * n[1] + Rr[2] * n[2];
  const float r1 = Rr[3] * n[0] + Rr[4] * n[1] + Rr[5] * n[2];
  const float r2 = Rr[6] * n[0] + Rr[7] * n[1] + Rr[8] * n[2];
  n[0] = r0;
  n[1] = r1;
  n[2] = r2;
}

__device__ __forceinline__ float propagate_depth(float d1, const float n1[3], K4<float>* iK, int row1, int col1,
                                                 float np0, float np1) {
  const float x1 = d1 * (iK[0] * (float)col1 + iK[1]);
  const float y1 = d1 * (iK[2] * (float)row1 + iK[3]);
  const float z1 = d1;
  const float dd = n1[0] * x1 + n1[1] * y1 + n1[2] * z1;
  const float t = dd / (n1[0] * np0 + n1[1] * np1 + n1[2] * 1.0f);
  if (fabsf(t) < 1e-5f) return d1;
  return t;
}

// ---------------------------------------------------------------------------
// workgroup set-up shared by the colour-pass kernels

// Sizes of the compiled windows (R_ >= 0); see WinLds.
template <int R_, int S_>
struct SpSize {
  static constexpr int kFloats = ((2 * R_) / S_ + 1) * ((2 * R_) / S_ + 1);
};

template <int R_>
struct TileSize {
  // The staged ref tile has one row pitch for every tile shape (the widest
  // tile plus the halo), so window offsets in LDS are compile-time
  // constants; rows: the tallest tile plus the halo.
  static constexpr int kPitch = (1 << kTileLog2WMax) + 2 * R_;
  static constexpr int kWords = ((kTilePixels >> kTileLog2WMin) + 2 * R_) * kPitch;
};

// Persistent colour-pass kernels: a launch runs at most as many workgroups
// as the chip holds at once, and each workgroup loops claiming tiles until
// the launch's tiles are exhausted.  The launch's tiles are split into
// 8 contiguous ranges, one per XCD (workgroups are dispatched round-robin
// over the XCDs, so block b starts on XCD b % 8); a workgroup takes tiles
// from its own XCD's range first, so the workgroups of one XCD cover compact
// bands of a view and share source footprints in that XCD's L2, and steals
// from the other ranges once its own is empty.
__device__ __forceinline__ int claim_tile(const LaunchTable* __restrict__ lt, int* next) {
  __syncthreads();  // the previous tile's LDS and *next are no longer read
  if (threadIdx.x == 0) {
    const __attribute__((address_space(1))) LaunchTable* g = G(lt);
    const int T = g->total_tiles;
    uint32_t* q = g->queue;
    const int xcd = blockIdx.x & 7;
    int tile = -1;
    for (int k = 0; k < 8 && tile < 0; ++k) {
      const int x = (xcd + k) & 7;
      const int lo = (int)(((long long)T * x) >> 3), hi = (int)(((long long)T * (x + 1)) >> 3);
      if (lo >= hi) continue;
      // a range already used up is skipped without an atomic: at the end of
      // a launch every workgroup scans all 8 ranges, and those atomics on 8
      // addresses serialise (counters only grow, so a stale read costs one
      // atomic, never a tile)
      if (__hip_atomic_load(q + x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= (uint32_t)(hi - lo)) continue;
      const uint32_t c = atomicAdd(q + x, 1u);
      if (c < (uint32_t)(hi - lo)) tile = lo + (int)c;
    }
    *next = tile;
  }
  __syncthreads();
  // the same value in every lane: keep it (and everything resolved from it,
  // the view's parameters and pointers) in scalar registers
  return __builtin_amdgcn_readfirstlane(*next);
}

// The launch entry (view, colour, pass) a tile belongs to.
struct Ctx {
  VPtr v;
  int color;
  uint32_t pass;
  float th_mc;
  int local_block;  // tile index within the view
  int lw;           // log2 of the tile width
  int lpx;          // log2 of the tile's pixels of one colour
  int group;        // sources a step of eval_selected takes
  float* ws;        // this workgroup's workspace
};

__device__ __forceinline__ Ctx resolve(const LaunchTable* __restrict__ lt, int t) {
  const __attribute__((address_space(1))) LaunchTable* g = G(lt);
  int lo = 0, hi = g->n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (g->e[mid].tile_start <= t) lo = mid;
    else hi = mid - 1;
  }
  Ctx c;
  c.v = (VPtr)g->e[lo].v;
  c.color = g->e[lo].color;
  c.pass = g->e[lo].pass;
  c.th_mc = g->e[lo].th_mc;
  c.local_block = t - g->e[lo].tile_start;
  c.lw = g->tile_lw;
  c.lpx = g->tile_lpx;
  // One source a step leaves out the most evaluations.  Small tiles have too
  // few pairs of one source for four waves: two sources (640x480: 6.07 ms a
  // run, against 6.25 with one and 6.21 with four), and four where every
  // workgroup has one tile at most, so that the chain of steps is what counts
  // (240x160: 2.33 ms, against 2.62 with two).
  c.group = c.lpx == kTileLog2Px ? 1 : g->total_tiles <= (int)gridDim.x ? 4 : 2;
  c.ws = g->ws + (size_t)blockIdx.x * g->ws_stride;
  return c;
}

// Where a tile lies, and its pixels of one colour.
struct Geo {
  int row0, col0, lw, color, pitch;
  // Pixel px of the tile: 2^(lw-1) pixels of the colour per row.
  __device__ __forceinline__ void pixel(int px, int& lrow, int& lcol) const {
    lrow = px >> (lw - 1);
    lcol = 2 * (px & ((1 << (lw - 1)) - 1)) + ((row0 + lrow + color) & 1);
  }
};

// Stage the colour table, the spatial weights and the ref tile (zero outside
// the image) into LDS.  The caller's barrier makes them visible.
__device__ __forceinline__ Geo stage_tile(const Ctx& cx, int R, int pitch, uint32_t* tile, float* ct, float* spl) {
  const VPtr v = cx.v;
  const int t = threadIdx.x;
  ct[t] = G(v->ct)[t];
  const int nsp = v->nwin * v->nwin;
  for (int e = t; e < nsp; e += kSweepThreads) spl[e] = G(v->sp)[e];
  const int W = v->W, H = v->H;
  const int lw = cx.lw;
  const int rows = (2 << cx.lpx) >> lw;
  const int tiles_x = (W + (1 << lw) - 1) >> lw;
  const int ty = cx.local_block / tiles_x;
  const int tx = cx.local_block - ty * tiles_x;
  const int row0 = ty * rows, col0 = tx << lw;
  const int tw = (1 << lw) + 2 * R;
  const int th = rows + 2 * R;
  for (int e = t; e < tw * th; e += kSweepThreads) {
    const int er = e / tw, ec = e - er * tw;
    const int rr = row0 - R + er, cc = col0 - R + ec;
    const uint32_t ri = (rr < 0 || rr >= H || cc < 0 || cc >= W) ? 0u : (uint32_t)G(v->ref)[rr * W + cc];
    tile[er * pitch + ec] = (ri << 16) | (3u * ri);
  }
  return Geo{row0, col0, lw, cx.color, pitch};
}

// The context of pixel (row, col) at tile position (lrow, lcol), with its
// moments m.
__device__ __forceinline__ Pix make_pix(VPtr v, const Geo& g, const uint32_t* tile, int R, int lrow, int lcol, f4v m) {
  Pix px;
  px.lrow = lrow;
  px.lcol = lcol;
  px.row = g.row0 + lrow;
  px.col = g.col0 + lcol;
  px.p = px.row * v->W + px.col;
  px.mu_r = m.x;
  px.var_r = m.y;
  px.inv_sw = m.z;
  px.err_r = m.w;
  px.c = (int)(tile[(lrow + R) * g.pitch + lcol + R] >> 16);
  px.shifted = (v->accum_mode == PM_ACCUM_COMPENSATED) && (px.var_r < kLowTexVar);
  px.np0 = v->refInvK[0] * (float)px.col + v->refInvK[1];
  px.np1 = v->refInvK[2] * (float)px.row + v->refInvK[3];
  return px;
}

// LDS of the windowed kernels.  The compiled windows have static arrays with
// one row pitch for every tile shape, so window offsets are immediates; any
// other window gets a launch-time block (window_lds_bytes) sized by its own
// radius, so a small one leaves room for more workgroups.
template <int R_, int S_>
struct WinLds {
  static constexpr int kTileWords = R_ >= 0 ? TileSize<R_>::kWords : 1;
  static constexpr int kSpWords = R_ >= 0 ? SpSize<R_, S_>::kFloats : 1;
  uint32_t tile[kTileWords];
  float spl[kSpWords];
  float ct[256];
};
extern __shared__ uint32_t win_dyn[];

template <int R_, int S_>
__device__ __forceinline__ uint32_t* lds_tile(WinLds<R_, S_>& l, VPtr v) {
  if constexpr (R_ >= 0) return l.tile;
  else return win_dyn + v->nwin * v->nwin;
}
template <int R_, int S_>
__device__ __forceinline__ float* lds_spl(WinLds<R_, S_>& l) {
  if constexpr (R_ >= 0) return l.spl;
  else return (float*)win_dyn;
}
template <int R_>
__device__ __forceinline__ int tile_pitch(int R, int lw) {
  if constexpr (R_ >= 0) return TileSize<R_>::kPitch;
  else return (1 << lw) + 2 * R;
}

// ---------------------------------------------------------------------------
// init: random (best of init_samples) or given depth/normal, then InitConf

template <int R_, int S_, int STORE, int RCP>
__device__ __forceinline__ void init_tile(const Ctx& cx, WinLds<R_, S_>& lds) {
  const VPtr v = cx.v;
  const uint32_t pass = cx.pass;
  const int R = R_ >= 0 ? R_ : v->radius;
  uint32_t* tile = lds_tile<R_, S_>(lds, v);
  float* spl = lds_spl<R_, S_>(lds);
  float* ct = lds.ct;
  const int tw = tile_pitch<R_>(R, cx.lw);
  const Geo geo = stage_tile(cx, R, tw, tile, ct, spl);
  __syncthreads();
  const int slot = threadIdx.x;
  int lrow, lcol;
  geo.pixel(slot, lrow, lcol);
  if (slot >= (1 << cx.lpx) || geo.row0 + lrow >= v->H || geo.col0 + lcol >= v->W) return;
  const Pix px = make_pix(v, geo, tile, R, lrow, lcol,
                          ld_f4(v->refm, (geo.row0 + lrow) * v->W + geo.col0 + lcol));
  const uint32_t* wt = tile + px.lrow * tw + px.lcol;
  const int N = v->N;
  const int plane = v->W * v->H;
  Ws ws{cx.ws, 1 << cx.lpx, N};
  Counters cnt;
  pm_rng g;
  pm_rng_init(&g, v->seed, (uint32_t)v->view_id, (uint32_t)px.p, pass);
  const int thk = v->thk < N ? v->thk : N;
  float hd, hn[3];
  float best_conf = 0.0f;
  uint32_t best_sel = 0;
  float bd = 0.0f, bn[3] = {0.0f, 0.0f, 0.0f};
  const int K = v->init_random ? (v->init_samples > 0 ? v->init_samples : 1) : 1;
  for (int smp = 0; smp < K; ++smp) {
    if (v->init_random) {
      hd = random_depth(&g, v->depth_min, v->depth_max);
      random_normal(&g, px.np0, px.np1, hn);
    } else {
      hd = G(v->depth)[px.p];
      hn[0] = G(v->normal)[px.p];
      hn[1] = G(v->normal)[plane + px.p];
      hn[2] = G(v->normal)[2 * plane + px.p];
      if (hd <= 0.0f) {
        hd = random_depth(&g, v->depth_min, v->depth_max);
        random_normal(&g, px.np0, px.np1, hn);
      }
      if (hn[0] * px.np0 + hn[1] * px.np1 + hn[2] * 1.0f >= 0.0f) random_normal(&g, px.np0, px.np1, hn);
    }
    for (int i = 0; i < N; ++i) {
      ws.M(0, i, slot) = mv_cost<R_, S_, STORE, RCP>(v, i, px, wt, tw, ct, spl, hn[0], hn[1], hn[2], hd, v->refK, cnt);
    }
    // thk smallest costs in stable ascending order (= the reference's
    // bubble sort, kernel_functions.cu:1588-1597)
    float conf = 0.0f;
    uint32_t taken = 0;
    for (int j = 0; j < thk; ++j) {
      int bi = -1;
      float bv = 0.0f;
      for (int i = 0; i < N; ++i) {
        if ((taken >> i) & 1u) continue;
        const float cv = ws.M(0, i, slot);
        if (bi < 0 || cv < bv) {
          bi = i;
          bv = cv;
        }
      }
      taken |= 1u << bi;
      conf = conf + bv;
    }
    conf = conf / c_mweights[thk];
    if (smp == 0 || conf < best_conf) {
      best_conf = conf;
      best_sel = taken;
      bd = hd;
      bn[0] = hn[0];
      bn[1] = hn[1];
      bn[2] = hn[2];
      for (int i = 0; i < N; ++i) ws.RM(0, i, slot) = ws.M(0, i, slot);
    }
  }
  G(v->depth)[px.p] = bd;
  G(v->normal)[px.p] = bn[0];
  G(v->normal)[plane + px.p] = bn[1];
  G(v->normal)[2 * plane + px.p] = bn[2];
  G(v->conf)[px.p] = best_conf;
  G(v->view_sel)[px.p] = best_sel;
  for (int i = 0; i < N; ++i) G(v->cost)[i * plane + px.p] = ws.RM(0, i, slot);
  flush_counters(v, cnt);
}

template <int R_, int S_, int STORE, int RCP>
__global__ __launch_bounds__(kSweepThreads) void k_init(const LaunchTable* __restrict__ lt) {
  __shared__ WinLds<R_, S_> lds;
  __shared__ int next;
  for (int t = claim_tile(lt, &next); t >= 0; t = claim_tile(lt, &next))
    init_tile<R_, S_, STORE, RCP>(resolve(lt, t), lds);
}

// ---------------------------------------------------------------------------
// evaluations shared by a workgroup
//
// What bounds the sweep is the VALU work of the window walks, so every walk
// should serve 64 lanes that need it.  The pixels of a tile need different
// evaluations (a candidate is missing, a source is not selected, a hypothesis
// can no longer win), and a wave that keeps to its own 64 pixels walks the
// union of what they need.  Here the (hypothesis, pixel) pairs that are needed
// are listed in LDS, in order of pixel within a hypothesis so that 64
// consecutive pairs still read neighbouring texels, and the four waves take
// the list in units of one source x 64 pairs.  The source is uniform across a
// unit: its pose and texture stay in scalar registers.  Listing also leaves
// nothing of a pixel live across a walk but what the walk reads (126 VGPRs,
// 4 waves per SIMD; one thread per pixel took 147 and 3).
// Run of a 1920x1080 view (10 sources, 15x15, 8 iterations): one thread per
// pixel 464 ms, here 342 ms.  160x120 (2 sources, 11x11 step 2, 5 iterations),
// where the four waves share 16 pixels (tile_shape): 2.33 against 1.02 ms.

// Per-workgroup LDS beside the window's: what the pairs need of a pixel.
struct PassLds {
  f4v refm[kSweepThreads];                    // {mu_r, var_r, 1/sum_w, err_r}
  uint16_t list[kMaxHyp * kSweepThreads];     // pairs: hypothesis << 8 | pixel
  float cost[kNumRefine * kSweepThreads];     // costs of a step, [source of the step][hypothesis][pixel]
  uint32_t sel[kSweepThreads];                // selected sources
  uint32_t bits[kSweepThreads];               // valid candidates
  float norm[kSweepThreads];                  // 1 / sum of the selected sources' weights
  uint32_t win[kSweepThreads];                // workspace slot of the winner, or kNone
  uint8_t own[4][kSweepThreads];              // per wave: pixels of a source
  int count[2][4];                            // pairs per source of a step
};
constexpr uint32_t kNone = 0xffffffffu;
constexpr int kLoTrials = 5;                    // trials of the local optimisation

__device__ __forceinline__ int lane_id() { return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)); }
__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); }
// Lanes below this one in the mask.
__device__ __forceinline__ int rank_in(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}
// LDS written by some lanes of a wave, read by others of the same wave.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Cost of hypothesis h of tile pixel q against source i.
template <int R_, int S_, int STORE, int RCP>
__device__ __forceinline__ float eval_pair(VPtr v, const Geo& geo, const PassLds& L, const uint32_t* tile,
                                           const float* ct, const float* spl, int R, int q, f4v h, int i,
                                           K4<float>* Kgeo, Counters& cnt) {
  int lrow, lcol;
  geo.pixel(q, lrow, lcol);
  const Pix px = make_pix(v, geo, tile, R, lrow, lcol, L.refm[q]);
  const int pitch = R_ >= 0 ? TileSize<R_>::kPitch : geo.pitch;
  return mv_cost<R_, S_, STORE, RCP>(v, i, px, tile + lrow * pitch + lcol, pitch, ct, spl, h.x, h.y, h.z, h.w, Kgeo, cnt);
}

// Hypotheses against the sources their pixels selected, source by source in
// ascending order, `group` sources a step.  Hypothesis k (0..nk-1) of a pixel
// is workspace slot slot0 + k; the running sums are those of the plain loop.
// A cost is >= 0 and a float sum of non-negative terms never decreases, so
// once dead(sum) holds the hypothesis cannot win and its further evaluations
// are left out (unless `all`: then every hypothesis meets every source).
// Owner threads (pixel px, hypotheses part, part + parts, ...) keep the sums;
// they return in sum[j] / alive bit j for hypothesis part + j * parts.
// Costs go to store(k, i, px, cost) and, summed, through weight(i).
template <int R_, int S_, int STORE, int RCP, int NK, typename Weight, typename Dead, typename Store>
__device__ __forceinline__ uint32_t eval_selected(VPtr v, const Geo& geo, PassLds& L, const Ws& ws, const uint32_t* tile,
                                                  const float* ct, const float* spl, int R, int px, int part, int parts,
                                                  int slot0, uint32_t sel, bool all, int group, float (&sum)[NK],
                                                  Weight weight, Dead dead, Store store, Counters& cnt) {
  const int N = v->N, npx = ws.npx;
  const int wave = wave_id(), lane = lane_id();
  uint32_t alive = 0;
#pragma unroll
  for (int j = 0; j < NK; ++j) {
    sum[j] = 0.0f;
    if (part + j * parts < NK) alive |= 1u << j;
  }
  if (!all && sel == 0) alive = 0;
  if (threadIdx.x < 8) (&L.count[0][0])[threadIdx.x] = 0;
  __syncthreads();
  const int cap = NK * npx;  // pairs of one source
  for (int i0 = 0, step = 0; i0 < N; i0 += group, step ^= 1) {
    for (int g = 0; g < group && i0 + g < N; ++g) {
      const bool want = all || ((sel >> (i0 + g)) & 1u);
      int total = 0;
#pragma unroll
      for (int j = 0; j < NK; ++j) total += __popcll(__ballot(want && ((alive >> j) & 1u)));
      if (total == 0) continue;
      int base = 0;
      if (lane == 0) base = atomicAdd(&L.count[step][g], total);
      base = g * cap + __builtin_amdgcn_readfirstlane(base);
#pragma unroll
      for (int j = 0; j < NK; ++j) {
        const bool on = want && ((alive >> j) & 1u);
        const uint64_t m = __ballot(on);
        if (on) L.list[base + rank_in(m)] = (uint16_t)(((part + j * parts) << 8) | px);
        base += __popcll(m);
      }
    }
    __syncthreads();
    if (threadIdx.x < 4) L.count[step ^ 1][threadIdx.x] = 0;
    int g = 0, n = __builtin_amdgcn_readfirstlane(L.count[step][0]), u0 = 0;
    for (int u = wave;; u += 4) {
      while (g < group && u >= u0 + ((n + 63) >> 6)) {
        u0 += (n + 63) >> 6;
        ++g;
        n = g < group ? __builtin_amdgcn_readfirstlane(L.count[step][g]) : 0;
      }
      if (g >= group) break;
      const int e = (u - u0) * 64 + lane;
      if (e < n) {
        const int code = L.list[g * cap + e];
        const int k = code >> 8, q = code & 0xff;
        const float m = eval_pair<R_, S_, STORE, RCP>(v, geo, L, tile, ct, spl, R, q, ws.hyp(slot0 + k, q), i0 + g,
                                                      v->refK, cnt);
        L.cost[(g * NK + k) * npx + q] = m;
        store(k, i0 + g, q, m);
      }
    }
    __syncthreads();
    for (int g2 = 0; g2 < group && i0 + g2 < N; ++g2) {
      const bool picked = (sel >> (i0 + g2)) & 1u;
      if (!picked && !all) continue;
      const float w = picked ? weight(i0 + g2) : 0.0f;
#pragma unroll
      for (int j = 0; j < NK; ++j) {
        if (!((alive >> j) & 1u)) continue;
        sum[j] = sum[j] + w * L.cost[(g2 * NK + part + j * parts) * npx + px];
        if (!all && dead(sum[j])) alive &= ~(1u << j);
      }
    }
  }
  return alive;
}

// Costs of the winners against the sources their pixels did not select, into
// the cost maps.  Each wave takes whole sources; no barrier inside.
template <int R_, int S_, int STORE, int RCP>
__device__ __forceinline__ void eval_unselected(VPtr v, const Geo& geo, PassLds& L, const Ws& ws, const uint32_t* tile,
                                                const float* ct, const float* spl, int R, K4<float>* Kgeo,
                                                Counters& cnt) {
  const int N = v->N, W = v->W, plane = v->W * v->H;
  const int wave = wave_id(), lane = lane_id();
  uint8_t* own = L.own[wave];
  for (int i = wave; i < N; i += 4) {
    int n = 0;
    for (int q0 = 0; q0 < ws.npx; q0 += 64) {
      const int q = q0 + lane;
      const bool on = q < ws.npx && L.win[q] != kNone && !((L.sel[q] >> i) & 1u);
      const uint64_t m = __ballot(on);
      if (on) own[n + rank_in(m)] = (uint8_t)q;
      n += __popcll(m);
    }
    wave_lds_sync();
    for (int e0 = 0; e0 < n; e0 += 64) {
      if (e0 + lane < n) {
        const int q = own[e0 + lane];
        const float m = eval_pair<R_, S_, STORE, RCP>(v, geo, L, tile, ct, spl, R, q, ws.hyp((int)L.win[q], q), i, Kgeo,
                                                      cnt);
        int lrow, lcol;
        geo.pixel(q, lrow, lcol);
        G(v->cost)[i * plane + (geo.row0 + lrow) * W + geo.col0 + lcol] = m;
      }
    }
    wave_lds_sync();
  }
}

// Whether every cost is a finite number >= 0 (NCC is in [0, 2]; the geometric
// term in [0, its maximum] times the regulariser): then a zero weight removes
// a source from a weighted sum exactly, and partial sums never decrease.
__device__ __forceinline__ bool costs_bounded(VPtr v) {
  return !v->geom || (v->geom_regularizer >= 0.0f && v->geom_max_cost >= 0.0f &&
                      v->geom_regularizer * v->geom_max_cost < 1e30f);
}

// ---------------------------------------------------------------------------
// checkerboard sweep

// Samples of the CDF held in registers at a time.
constexpr int kDraws = 16;

template <int R_, int S_, int STORE, int RCP>
__device__ __forceinline__ void sweep_tile(const Ctx& cx, WinLds<R_, S_>& lds, PassLds& L) {
  const VPtr v = cx.v;
  const int R = R_ >= 0 ? R_ : v->radius;
  uint32_t* tile = lds_tile<R_, S_>(lds, v);
  float* spl = lds_spl<R_, S_>(lds);
  const float* ct = lds.ct;
  const int W = v->W, H = v->H, N = v->N;
  const int plane = W * H;
  const int npx = 1 << cx.lpx, parts = kSweepThreads >> cx.lpx;
  const int px = threadIdx.x & (npx - 1), part = threadIdx.x >> cx.lpx;  // thread: a share of a pixel's bookkeeping
  const int wave = wave_id(), lane = lane_id();
  const Geo geo = stage_tile(cx, R, tile_pitch<R_>(R, cx.lw), tile, lds.ct, spl);
  const Ws ws{cx.ws, npx, N};
  Counters cnt;
  int lrow, lcol;
  geo.pixel(px, lrow, lcol);
  const int row = geo.row0 + lrow, col = geo.col0 + lcol;
  const bool in = row < H && col < W;
  const int p = row * W + col;
  if (part == 0) {
    if (in) L.refm[px] = ld_f4(v->refm, p);
    L.bits[px] = in ? 1u : 0u;
    L.sel[px] = 0u;
    L.win[px] = kNone;
  }
  if (threadIdx.x == 0) L.count[0][0] = 0;
  __syncthreads();

  K4<float>* iK = v->refInvK;
  const float vd[3] = {iK[0] * (float)col + iK[1], iK[2] * (float)row + iK[3], 1.0f};
  const float inv_view_len = 1.0f / sqrtf(vd[0] * vd[0] + vd[1] * vd[1] + vd[2] * vd[2]);
  const bool full = v->count_all != 0 || !costs_bounded(v);

  // candidates: slot 0 the current hypothesis, 1 and 2 the better of the
  // 4-neighbours, 3 + g the best of direction g
  if (in) {
    uint32_t valid = 0;
    for (int task = part; task < 9; task += parts) {
      if (task == 0) {
        ws.hyp(0, px) = f4v{G(v->normal)[p], G(v->normal)[plane + p], G(v->normal)[2 * plane + p], G(v->depth)[p]};
        if (!G(v->grad_ok)[p]) continue;
        float nconf[4];
        int order[4];
        int nvalid = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          order[k] = k;
          const int u = col + c_neighbor_offs[k][1], w = row + c_neighbor_offs[k][0];
          if (u < 0 || u >= W || w < 0 || w >= H) {
            nconf[k] = PM_FLT_MAX;
            continue;
          }
          nvalid++;
          nconf[k] = G(v->conf)[w * W + u];
        }
#pragma unroll
        for (int a = 0; a < 3; ++a) {
#pragma unroll
          for (int b = 0; b < 3 - a; ++b) {
            if (nconf[b] > nconf[b + 1]) {
              const float t = nconf[b];
              nconf[b] = nconf[b + 1];
              nconf[b + 1] = t;
              const int o = order[b];
              order[b] = order[b + 1];
              order[b + 1] = o;
            }
          }
        }
        if (nvalid > 2) nvalid = 2;
        for (int k = 0; k < nvalid; ++k) {
          const int idx = k == 0 ? order[0] : order[1];
          const int u = col + c_neighbor_offs[idx][1], w = row + c_neighbor_offs[idx][0];
          const int q = w * W + u;
          float nn[3] = {G(v->normal)[q], G(v->normal)[plane + q], G(v->normal)[2 * plane + q]};
          correct_normal(nn, vd, inv_view_len);
          const float dd = propagate_depth(G(v->depth)[q], nn, iK, w, u, vd[0], vd[1]);
          ws.hyp(1 + k, px) = f4v{nn[0], nn[1], nn[2], dd};
          valid |= 2u << k;
        }
      } else {
        const int gi = task - 1;
        float best_conf = PM_FLT_MAX;
        int br = 0, bc = 0;
        const int sign = (gi & 1) ? 1 : -1;
#pragma unroll
        for (int f = 0; f < 10; ++f) {
          int dr, dc;
          dir_sample(gi, sign, f, dr, dc);
          const int nr = row + dr, ncn = col + dc;
          if (nr < 0 || nr >= H || ncn < 0 || ncn >= W) continue;
          const float cv = G(v->conf)[nr * W + ncn];
          if (best_conf > cv) {
            best_conf = cv;
            br = nr;
            bc = ncn;
          }
        }
        if (best_conf < PM_FLT_MAX) {
          const int q = br * W + bc;
          float nn[3] = {G(v->normal)[q], G(v->normal)[plane + q], G(v->normal)[2 * plane + q]};
          correct_normal(nn, vd, inv_view_len);
          const float dd = propagate_depth(G(v->depth)[q], nn, iK, br, bc, vd[0], vd[1]);
          ws.hyp(3 + gi, px) = f4v{nn[0], nn[1], nn[2], dd};
          valid |= 8u << gi;
        }
      }
    }
    if (valid) atomicOr(&L.bits[px], valid);
  }
  __syncthreads();

  // the candidates' pairs; then the cost matrix, source by source
  if (wave * 64 < npx) {
    const uint32_t b = lane < npx ? L.bits[wave * 64 + lane] : 0u;
    int total = 0;
    for (int k = 1; k < kMaxHyp; ++k) total += __popcll(__ballot((b >> k) & 1u));
    int base = 0;
    if (lane == 0) base = atomicAdd(&L.count[0][0], total);
    base = __builtin_amdgcn_readfirstlane(base);
    for (int k = 1; k < kMaxHyp; ++k) {
      const uint64_t m = __ballot((b >> k) & 1u);
      if ((b >> k) & 1u) L.list[base + rank_in(m)] = (uint16_t)((k << 8) | (wave * 64 + lane));
      base += __popcll(m);
    }
  }
  __syncthreads();
  {
    const int n = __builtin_amdgcn_readfirstlane(L.count[0][0]);
    const int chunks = (n + 63) >> 6;
    int i = 0, c = wave;
    for (;;) {
      while (c >= chunks && i < N) {
        c -= chunks;
        ++i;
        if (chunks == 0) i = N;
      }
      if (i >= N) break;
      const int e = c * 64 + lane;
      if (e < n) {
        const int code = L.list[e];
        const int k = code >> 8, q = code & 0xff;
        ws.M(k, i, q) = eval_pair<R_, S_, STORE, RCP>(v, geo, L, tile, ct, spl, R, q, ws.hyp(k, q), i, v->refK, cnt);
      }
      c += 4;
    }
  }
  __syncthreads();

  // view selection (kernel_functions.cu:2364-2426)
  const uint32_t valid = L.bits[px];  // 0 outside the image
  if (in) {
    uint32_t flags = 0;
    for (int i = part; i < N; i += parts) {
      const float c0 = G(v->cost)[i * plane + p];
      ws.M(0, i, px) = c0;
      float pr = 0.0f;
      int n1 = 0, n2 = 0;
#pragma unroll
      for (int k = 0; k < kMaxHyp; ++k) {
        if (!((valid >> k) & 1u)) continue;
        const float cv = k == 0 ? c0 : ws.M(k, i, px);
        pr = pr + pm_expf(-(cv * cv) * v->inv_beta2);
        n1 += (cv < cx.th_mc);
        n2 += (cv > v->max_ncc_matching_cost);
      }
      ws.Wt(i, px) = pr;
      if (n1 >= v->num_good && n2 <= v->num_bad) flags |= 1u << i;
    }
    if (flags) atomicOr(&L.sel[px], flags);
  }
  __syncthreads();

  // the draws: a pixel's first thread picks the sources (L.sel: flags in,
  // selected sources out) and keeps the stream for the refinement
  const bool once = v->random_optimization != 0;  // a picked source weighs 1, or its number of picks
  uint32_t sel = L.sel[px];
  pm_rng g;
  float norm = 0.0f;  // 1 / sum of the weights
  if (part == 0 && sel != 0) {
    const uint32_t flags = sel;
    float psum = 0.0f;
    for (int i = 0; i < N; ++i) psum = psum + (((flags >> i) & 1u) ? ws.Wt(i, px) : 0.0f);
    const float inv_psum = 1.0f / psum;
    pm_rng_init(&g, v->seed, (uint32_t)v->view_id, (uint32_t)p, cx.pass);
    uint32_t picked = 0;
    int picks = 0;
    for (int s0 = 0; s0 < v->num_samples; s0 += kDraws) {
      float rp[kDraws];
      const int ns = v->num_samples - s0;
#pragma unroll
      for (int s = 0; s < kDraws; ++s) {
        rp[s] = INFINITY;
        if (s < ns) rp[s] = pm_rng_uniform(&g) - PM_FLT_EPSILON;
      }
      // each draw picks the first source whose CDF exceeds it
      float cum = 0.0f;
      for (int i = 0; i < N; ++i) {
        const float pr = ((flags >> i) & 1u) ? ws.Wt(i, px) : 0.0f;
        cum = cum + pr * inv_psum;
        int hits = 0;
#pragma unroll
        for (int s = 0; s < kDraws; ++s) {
          if (cum > rp[s]) {
            hits++;
            rp[s] = INFINITY;
          }
        }
        if (!once) ws.RM(0, i, px) = (s0 > 0 ? ws.RM(0, i, px) : 0.0f) + (float)hits;
        if (hits) picked |= 1u << i;
        picks += hits;
      }
    }
    const float wnorm = once ? (float)__popc(picked) : (float)picks;
    if (wnorm <= 1e-5f) picked = 0;
    else norm = 1.0f / wnorm;
    if (!once && picked) {
      for (int i = 0; i < N; ++i) ws.Wt(i, px) = ws.RM(0, i, px) * norm;
    }
    L.sel[px] = picked;
    L.norm[px] = norm;
  }
  __syncthreads();
  sel = L.sel[px];
  norm = L.norm[px];
  // weight of selected source i
  auto weight = [&](int i) __attribute__((always_inline)) { return once ? norm : ws.Wt(i, px); };
  int best = -1;
  float minc = PM_FLT_MAX;
  if (sel != 0) {
    for (int k = part; k < kMaxHyp; k += parts) {
      if (!((valid >> k) & 1u)) continue;
      float cc = 0.0f;
      for (int i = 0; i < N; ++i) {
        if (full || ((sel >> i) & 1u)) cc = cc + (((sel >> i) & 1u) ? weight(i) : 0.0f) * ws.M(k, i, px);
      }
      if (cc <= minc) {
        minc = cc;
        best = k;
      }
    }
  }
  if (parts > 1) {  // the last minimum wins: among equals the largest k
    float* pc = L.cost;
    int* pk = (int*)(L.cost + kSweepThreads);
    pc[threadIdx.x] = minc;
    pk[threadIdx.x] = best;
    __syncthreads();
    for (int o = 0; o < parts; ++o) {
      const float c2 = pc[o * npx + px];
      const int k2 = pk[o * npx + px];
      if (k2 >= 0 && (best < 0 || c2 < minc || (c2 == minc && k2 > best))) {
        minc = c2;
        best = k2;
      }
    }
  }
  float rc0 = minc;
  if (sel != 0 && best < 0) {  // no sum below FLT_MAX
    best = 0;
    rc0 = 0.0f;
    for (int i = 0; i < N; ++i) rc0 = rc0 + (((sel >> i) & 1u) ? weight(i) : 0.0f) * ws.M(0, i, px);
  }

  // refinement hypotheses (kernel_functions.cu:2449-2486): slots kMaxHyp + 1..4
  const int hb = kMaxHyp;
  if (part == 0 && sel != 0) {
    G(v->view_sel)[p] = sel;
    const f4v h = ws.hyp(best, px);
    const float depth = h.w;
    const float normal[3] = {h.x, h.y, h.z};
    const float dlo = (1.0f - v->random_depth_ratio) * depth;
    const float dhi = (1.0f + v->random_depth_ratio) * depth;
    const float nd = random_depth(&g, dlo, dhi);
    float nn[3];
    perturb_normal(&g, normal, v->angle1, v->angle2, nn);
    correct_normal(nn, vd, inv_view_len);
    const float rd = random_depth(&g, v->depth_min, v->depth_max_eff);
    float rn[3];
    random_normal(&g, vd[0], vd[1], rn);
    correct_normal(rn, vd, inv_view_len);
    ws.hyp(hb + 1, px) = f4v{nn[0], nn[1], nn[2], depth};
    ws.hyp(hb + 2, px) = f4v{normal[0], normal[1], normal[2], nd};
    ws.hyp(hb + 3, px) = f4v{rn[0], rn[1], rn[2], depth};
    ws.hyp(hb + 4, px) = f4v{normal[0], normal[1], normal[2], rd};
  }

  // A refined hypothesis replaces the best candidate if its weighted sum is
  // not above rc0; only the selected sources enter that sum.
  float sum[kNumRefine - 1];
  const uint32_t alive = eval_selected<R_, S_, STORE, RCP, kNumRefine - 1>(
      v, geo, L, ws, tile, ct, spl, R, px, part, parts, hb + 1, sel, full && sel != 0, full ? 1 : cx.group, sum, weight,
      [&](float s) __attribute__((always_inline)) { return s > rc0; },
      [&](int k, int i, int q, float m) __attribute__((always_inline)) { ws.RM(k + 1, i, q) = m; }, cnt);
  int b2 = -1;
  minc = PM_FLT_MAX;
  if (rc0 <= minc) {
    minc = rc0;
    b2 = 0;
  }
#pragma unroll
  for (int j = 0; j < kNumRefine - 1; ++j) {
    if (((alive >> j) & 1u) && sum[j] <= minc) {
      minc = sum[j];
      b2 = part + j * parts + 1;
    }
  }
  if (parts > 1) {
    float* pc = L.cost;
    int* pk = (int*)(L.cost + kSweepThreads);
    __syncthreads();  // the sums are no longer read
    pc[threadIdx.x] = minc;
    pk[threadIdx.x] = b2;
    __syncthreads();
    for (int o = 0; o < parts; ++o) {
      const float c2 = pc[o * npx + px];
      const int k2 = pk[o * npx + px];
      if (k2 >= 0 && (b2 < 0 || c2 < minc || (c2 == minc && k2 > b2))) {
        minc = c2;
        b2 = k2;
      }
    }
  }
  if (sel == 0) b2 = -1;  // b2 < 0 otherwise: every cost NaN, the pixel keeps its state
  if (part == 0) L.win[px] = b2 > 0 && !full ? (uint32_t)(hb + b2) : kNone;
  __syncthreads();
  if (b2 >= 0) {
    if (part == 0) {
      const f4v h = ws.hyp(b2 == 0 ? best : hb + b2, px);
      G(v->conf)[p] = minc;
      G(v->depth)[p] = h.w;
      G(v->normal)[p] = h.x;
      G(v->normal)[plane + p] = h.y;
      G(v->normal)[2 * plane + p] = h.z;
    }
    for (int i = part; i < N; i += parts) {
      if (b2 == 0) G(v->cost)[i * plane + p] = ws.M(best, i, px);
      else if (full || ((sel >> i) & 1u)) G(v->cost)[i * plane + p] = ws.RM(b2, i, px);
    }
  }
  eval_unselected<R_, S_, STORE, RCP>(v, geo, L, ws, tile, ct, spl, R, v->refK, cnt);
  flush_counters(v, cnt, true);
}

template <int R_, int S_, int STORE, int RCP>
__global__ __launch_bounds__(kSweepThreads) void k_sweep(const LaunchTable* __restrict__ lt) {
  __shared__ WinLds<R_, S_> lds;
  __shared__ PassLds pass;
  __shared__ int next;
  for (int t = claim_tile(lt, &next); t >= 0; t = claim_tile(lt, &next))
    sweep_tile<R_, S_, STORE, RCP>(resolve(lt, t), lds, pass);
}

// ---------------------------------------------------------------------------
// local optimisation

template <int R_, int S_, int STORE, int RCP>
__device__ __forceinline__ void local_opt_tile(const Ctx& cx, WinLds<R_, S_>& lds, PassLds& L) {
  const VPtr v = cx.v;
  const int R = R_ >= 0 ? R_ : v->radius;
  uint32_t* tile = lds_tile<R_, S_>(lds, v);
  float* spl = lds_spl<R_, S_>(lds);
  const float* ct = lds.ct;
  const int W = v->W, H = v->H, N = v->N;
  const int plane = W * H;
  const int npx = 1 << cx.lpx, parts = kSweepThreads >> cx.lpx;
  const int px = threadIdx.x & (npx - 1), part = threadIdx.x >> cx.lpx;
  const Geo geo = stage_tile(cx, R, tile_pitch<R_>(R, cx.lw), tile, lds.ct, spl);
  const Ws ws{cx.ws, npx, N};
  Counters cnt;
  int lrow, lcol;
  geo.pixel(px, lrow, lcol);
  const int row = geo.row0 + lrow, col = geo.col0 + lcol;
  const bool in = row < H && col < W;
  const int p = row * W + col;
  const uint32_t sel = in ? G(v->view_sel)[p] : 0u;
  const float conf0 = in ? G(v->conf)[p] : 0.0f;
  if (part == 0) {
    if (in) L.refm[px] = ld_f4(v->refm, p);
    L.sel[px] = sel;
    L.win[px] = kNone;
  }
  if (part == 0 && sel != 0) {
    const float depth = G(v->depth)[p];
    const float angle1 = (float)(4.0 * 0.0174532925199432);
    const float angle2 = (float)(2.0 * 0.0174532925199432);
    float low = depth, up = depth;
    float m0 = G(v->normal)[p], m1 = G(v->normal)[plane + p], m2 = G(v->normal)[2 * plane + p];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int u = col + c_neighbor_offs[k][1], w = row + c_neighbor_offs[k][0];
      if (u < 0 || u >= W || w < 0 || w >= H) continue;
      const int q = w * W + u;
      const float ndp = G(v->depth)[q];
      m0 = m0 + G(v->normal)[q];
      m1 = m1 + G(v->normal)[plane + q];
      m2 = m2 + G(v->normal)[2 * plane + q];
      if (ndp <= low) low = ndp;
      if (ndp > up) up = ndp;
    }
    float mn[3] = {m0, m1, m2};
    const float inv_norm = 1.0f / sqrtf(mn[0] * mn[0] + mn[1] * mn[1] + mn[2] * mn[2]);
    mn[0] = mn[0] * inv_norm;
    mn[1] = mn[1] * inv_norm;
    mn[2] = mn[2] * inv_norm;
    pm_rng g;
    pm_rng_init(&g, v->seed, (uint32_t)v->view_id, (uint32_t)p, cx.pass);
    for (int t = 0; t < kLoTrials; ++t) {
      float hn[3];
      const float hd = random_depth(&g, low, up);
      perturb_normal(&g, mn, angle1, angle2, hn);
      ws.hyp(t, px) = f4v{hn[0], hn[1], hn[2], hd};
    }
  }
  // A trial's mean over the selected sources is its running sum / mw.
  // Costs are >= 0 (NCC in [0, 2], the geometric term scaled by a
  // non-negative regulariser) and a float sum of non-negative terms never
  // decreases, so once sum / mw >= the pixel's conf the trial cannot be
  // taken: its remaining evaluations are skipped.  The maps are those of the
  // full evaluation; the transcription prunes the same evaluations (a run that
  // counts the algorithm's takes one source a step, as it does).
  const float mw = (float)__popc(sel);
  const bool prune = !v->geom || v->geom_regularizer >= 0.0f;
  float sum[kLoTrials];
  const uint32_t alive = eval_selected<R_, S_, STORE, RCP, kLoTrials>(
      v, geo, L, ws, tile, ct, spl, R, px, part, parts, 0, sel, false, v->count_all != 0 ? 1 : cx.group, sum,
      [](int) __attribute__((always_inline)) { return 1.0f; },
      [&](float s) __attribute__((always_inline)) { return prune && s / mw >= conf0; },
      [&](int k, int i, int q, float m) __attribute__((always_inline)) { ws.M(k, i, q) = m; }, cnt);
  // the first of the smallest means below the pixel's conf
  float conf = conf0;
  int best = -1;
#pragma unroll
  for (int j = 0; j < kLoTrials; ++j) {
    if (!((alive >> j) & 1u)) continue;
    const float mconf = sum[j] / mw;
    if (mconf < conf) {
      conf = mconf;
      best = part + j * parts;
    }
  }
  if (parts > 1) {
    float* pc = L.cost;
    int* pk = (int*)(L.cost + kSweepThreads);
    __syncthreads();  // the sums are no longer read
    pc[threadIdx.x] = conf;
    pk[threadIdx.x] = best;
    __syncthreads();
    for (int o = 0; o < parts; ++o) {
      const float c2 = pc[o * npx + px];
      const int k2 = pk[o * npx + px];
      if (k2 >= 0 && (best < 0 || c2 < conf || (c2 == conf && k2 < best))) {
        conf = c2;
        best = k2;
      }
    }
  }
  if (part == 0 && best >= 0) L.win[px] = (uint32_t)best;
  __syncthreads();
  if (best >= 0) {
    if (part == 0) {
      const f4v h = ws.hyp(best, px);
      G(v->conf)[p] = conf;
      G(v->depth)[p] = h.w;
      G(v->normal)[p] = h.x;
      G(v->normal)[plane + p] = h.y;
      G(v->normal)[2 * plane + p] = h.z;
    }
    for (int i = part; i < N; i += parts)
      if ((sel >> i) & 1u) G(v->cost)[i * plane + p] = ws.M(best, i, px);
  }
  eval_unselected<R_, S_, STORE, RCP>(v, geo, L, ws, tile, ct, spl, R, v->compat_lo_geo_bug ? v->refInvK : v->refK, cnt);
  flush_counters(v, cnt);
}

template <int R_, int S_, int STORE, int RCP>
__global__ __launch_bounds__(kSweepThreads) void k_local_opt(const LaunchTable* __restrict__ lt) {
  __shared__ WinLds<R_, S_> lds;
  __shared__ PassLds pass;
  __shared__ int next;
  for (int t = claim_tile(lt, &next); t >= 0; t = claim_tile(lt, &next))
    local_opt_tile<R_, S_, STORE, RCP>(resolve(lt, t), lds, pass);
}

// Tiles of a launch of an element-wise phase, assigned by workgroup index
// (no LDS, no barriers).  The work per tile is a few loads, so the tile
// queue's atomics (all on one cache line) would cost more than the tiles.
template <typename F>
__device__ __forceinline__ void for_each_tile(const LaunchTable* __restrict__ lt, F&& f) {
  const int T = __builtin_amdgcn_readfirstlane(G(lt)->total_tiles);
  for (int t = blockIdx.x; t < T; t += gridDim.x) f(t);
}

// ---------------------------------------------------------------------------
// FilterDepthMap (kernel_functions.cu:3282-3354)

__device__ __forceinline__ void filter_tile(const Ctx& cx) {
  const VPtr v = cx.v;
  const int t = threadIdx.x;
  const int W = v->W, H = v->H;
  const int lw = cx.lw;
  const int tiles_x = (W + (1 << lw) - 1) >> lw;
  const int ty = cx.local_block / tiles_x;
  const int tx = cx.local_block - ty * tiles_x;
  const int row = ty * (kTilePixels >> lw) + (t >> (lw - 1));
  const int col = (tx << lw) + 2 * (t & ((1 << (lw - 1)) - 1)) + ((row + cx.color) & 1);
  if (row >= H || col >= W) return;
  const int plane = W * H;
  const int p = row * W + col;
  K4<float>* iK = v->refInvK;
  const float depth = G(v->depth)[p];
  if (depth <= 0.0f) return;
  const float n[3] = {G(v->normal)[p], G(v->normal)[plane + p], G(v->normal)[2 * plane + p]};
  const float conf = G(v->conf)[p];
  const float pt[3] = {depth * (iK[0] * (float)col + iK[1]), depth * (iK[2] * (float)row + iK[3]), depth};
  int good = 0;
  for (int k = 0; k < 4; ++k) {
    const int u = col + c_neighbor_offs[k][1], w = row + c_neighbor_offs[k][0];
    if (u < 0 || u >= W || w < 0 || w >= H) continue;
    const int q = w * W + u;
    const float nd = G(v->depth)[q];
    const float nn[3] = {G(v->normal)[q], G(v->normal)[plane + q], G(v->normal)[2 * plane + q]};
    const float nc = G(v->conf)[q];
    const float npt[3] = {nd * (iK[0] * (float)u + iK[1]), nd * (iK[2] * (float)w + iK[3]), nd};
    const float e0 = pt[0] - npt[0], e1 = pt[1] - npt[1], e2 = pt[2] - npt[2];
    const float d1 = fabsf(e0 * n[0] + e1 * n[1] + e2 * n[2]);
    const float d2 = fabsf(e0 * nn[0] + e1 * nn[1] + e2 * nn[2]);
    if ((conf < v->conf_threshold && d1 / depth < v->depth_diff_threshold) ||
        (nc < v->conf_threshold && d2 / nd < v->depth_diff_threshold)) {
      good++;
    }
  }
  if (good < 2) {
    G(v->depth)[p] = 0.0f;
    G(v->normal)[p] = 0.0f;
    G(v->normal)[plane + p] = 0.0f;
    G(v->normal)[2 * plane + p] = 0.0f;
    G(v->conf)[p] = 0.0f;
  }
}

__global__ __launch_bounds__(kSweepThreads) void k_filter(const LaunchTable* __restrict__ lt) {
  for_each_tile(lt, [&](int t) { filter_tile(resolve(lt, t)); });
}

// Pixel of a colour-pass tile (the mapping of filter_tile); false outside the view.
__device__ __forceinline__ bool tile_pixel(const Ctx& cx, int& row, int& col) {
  const int W = cx.v->W;
  const int lw = cx.lw;
  const int t = threadIdx.x;
  const int tiles_x = (W + (1 << lw) - 1) >> lw;
  const int ty = cx.local_block / tiles_x;
  const int tx = cx.local_block - ty * tiles_x;
  row = ty * (kTilePixels >> lw) + (t >> (lw - 1));
  col = (tx << lw) + 2 * (t & ((1 << (lw - 1)) - 1)) + ((row + cx.color) & 1);
  return row < cx.v->H && col < W;
}

// Ascending bubble sort of the first n of K values (the reference's
// BubbleSort, utils.h:206-221), unrolled over K slots so the array stays in
// registers; the compare-swaps past n are switched off, which leaves the
// same sequence of swaps as the loop over n.
template <int K>
__device__ __forceinline__ void bubble_sort_regs(float (&a)[K], int n) {
#pragma unroll
  for (int i = 0; i < K - 1; ++i) {
#pragma unroll
    for (int j = 0; j < K - 1 - i; ++j) {
      if (j < n - 1 - i && a[j] > a[j + 1]) {
        const float t = a[j];
        a[j] = a[j + 1];
        a[j + 1] = t;
      }
    }
  }
}

template <int K>
__device__ __forceinline__ float pick_reg(const float (&a)[K], int k) {
  float r = 0.0f;
#pragma unroll
  for (int j = 0; j < K; ++j) r = j == k ? a[j] : r;
  return r;
}

// float -> unsigned short as the reference's stores convert: toward zero,
// NaN and negatives to 0, saturating at 65535.
__device__ __forceinline__ uint16_t sat_u16(float x) {
  if (!(x > 0.0f)) return 0;
  if (x >= 65535.0f) return 65535;
  return (uint16_t)(uint32_t)x;
}

// acos as the reference calls it: NaN outside [-1, 1] (a dot product of two
// unit normals can round above 1).
__device__ __forceinline__ float acos_or_nan(float x) { return fabsf(x) <= 1.0f ? pm_acosf(x) : __builtin_nanf(""); }

// ComputeCurvatureMap (kernel_functions.cu:1603-1651).  Slice 0: the Scharr
// gradient magnitude of the reference image (intensities / 255, zero
// outside the image, filter_kernel_x/y at :56-60) x 10000, capped at 32767.
// Slice 1: 10000 x the median of the angles between the pixel's normal and
// the normals of its 5x5 neighbourhood clipped to the image, taken as the
// reference does (angles in window order, bubble sort, element count / 2),
// so NaN angles keep their positions as they do there.  The compacted angle
// list and the sort are unrolled over the 24 slots with selects, so they
// stay in registers.
__device__ __forceinline__ void curvature_tile(const Ctx& cx) {
  int row, col;
  if (!tile_pixel(cx, row, col)) return;
  const VPtr v = cx.v;
  const int W = v->W, H = v->H;
  const int plane = W * H;
  const int p = row * W + col;
  constexpr float kx[3][3] = {{-3.0f, 0.0f, 3.0f}, {-10.0f, 0.0f, 10.0f}, {-3.0f, 0.0f, 3.0f}};
  constexpr float ky[3][3] = {{-3.0f, -10.0f, -3.0f}, {0.0f, 0.0f, 0.0f}, {3.0f, 10.0f, 3.0f}};
  float gx = 0.0f, gy = 0.0f;
#pragma unroll
  for (int dr = -1; dr <= 1; ++dr) {
#pragma unroll
    for (int dc = -1; dc <= 1; ++dc) {
      const int u = col + dc, w = row + dr;
      const float color = (u >= 0 && u < W && w >= 0 && w < H) ? (float)G(v->ref)[w * W + u] / 255.0f : 0.0f;
      gx = gx + color * kx[dr + 1][dc + 1];
      gy = gy + color * ky[dr + 1][dc + 1];
    }
  }
  const float grad = sqrtf(gx * gx + gy * gy);

  const float n0 = G(v->normal)[p], n1 = G(v->normal)[plane + p], n2 = G(v->normal)[2 * plane + p];
  float a[24];
#pragma unroll
  for (int k = 0; k < 24; ++k) a[k] = 0.0f;
  int cnt = 0;
#pragma unroll
  for (int dy = -2; dy <= 2; ++dy) {
#pragma unroll
    for (int dx = -2; dx <= 2; ++dx) {
      if (dy == 0 && dx == 0) continue;
      const int y = row + dy, x = col + dx;
      if (y < 0 || y >= H || x < 0 || x >= W) continue;
      const int q = y * W + x;
      const float d = n0 * G(v->normal)[q] + n1 * G(v->normal)[plane + q] + n2 * G(v->normal)[2 * plane + q];
      const float ang = acos_or_nan(d);
#pragma unroll
      for (int j = 0; j < 24; ++j) a[j] = j == cnt ? ang : a[j];
      ++cnt;
    }
  }
  bubble_sort_regs(a, cnt);
  const float med = pick_reg(a, cnt >> 1);
  G(v->curv)[p] = sat_u16(fminf(grad * 10000.0f, 32767.0f));
  G(v->curv)[plane + p] = cnt > 0 ? sat_u16(med * 10000.0f) : (uint16_t)31415;  // M_PI * 10000
}

__global__ __launch_bounds__(kSweepThreads) void k_curvature(const LaunchTable* __restrict__ lt) {
  for_each_tile(lt, [&](int t) { curvature_tile(resolve(lt, t)); });
}

// MaskDepthMapKernel (kernel_functions.cu:3080-3093): zero the depth where
// the mask is 0.  The reference leaves the last row and column as they are.
__device__ __forceinline__ void mask_tile(const Ctx& cx) {
  int row, col;
  if (!tile_pixel(cx, row, col)) return;
  const VPtr v = cx.v;
  if (row >= v->H - 1 || col >= v->W - 1) return;
  const int p = row * v->W + col;
  if (G(v->mask)[p] == 0) G(v->depth)[p] = 0.0f;
}

__global__ __launch_bounds__(kSweepThreads) void k_mask(const LaunchTable* __restrict__ lt) {
  for_each_tile(lt, [&](int t) { mask_tile(resolve(lt, t)); });
}

// ComputeGeomGradientMap (kernel_functions.cu:3095-3120): Scharr gradient of
// |d_q - d_p| / d_p over the in-image 3x3 neighbours (outside ones are
// skipped, not zero).  The reference leaves pixels with d_p <= 0 unwritten
// (uninitialised memory); here they read 0.
__device__ __forceinline__ void geom_grad_tile(const Ctx& cx) {
  int row, col;
  if (!tile_pixel(cx, row, col)) return;
  const VPtr v = cx.v;
  const int W = v->W, H = v->H;
  const int p = row * W + col;
  const float depth = G(v->depth)[p];
  if (depth <= 0.0f) {
    G(v->geom_grad)[p] = 0.0f;
    return;
  }
  constexpr float kx[3][3] = {{-3.0f, 0.0f, 3.0f}, {-10.0f, 0.0f, 10.0f}, {-3.0f, 0.0f, 3.0f}};
  constexpr float ky[3][3] = {{-3.0f, -10.0f, -3.0f}, {0.0f, 0.0f, 0.0f}, {3.0f, 10.0f, 3.0f}};
  float gx = 0.0f, gy = 0.0f;
#pragma unroll
  for (int dr = -1; dr <= 1; ++dr) {
#pragma unroll
    for (int dc = -1; dc <= 1; ++dc) {
      const int w = row + dr, u = col + dc;
      if (w < 0 || w >= H || u < 0 || u >= W) continue;
      const float diff = fabsf(G(v->depth)[w * W + u] - depth) / depth;
      gx = gx + diff * kx[dr + 1][dc + 1];
      gy = gy + diff * ky[dr + 1][dc + 1];
    }
  }
  G(v->geom_grad)[p] = sqrtf(gx * gx + gy * gy);
}

__global__ __launch_bounds__(kSweepThreads) void k_geom_grad(const LaunchTable* __restrict__ lt) {
  for_each_tile(lt, [&](int t) { geom_grad_tile(resolve(lt, t)); });
}

// MedianFilter (kernel_functions.cu:3122-3244) for the pixels of one colour
// (BlackPixelFilter: (row + col) even, then RedPixelFilter: odd).  Taps:
// the pixel, the cross at distances 1 and 3 (up, down, left, right), then
// the 8 knight moves, in the reference's order; a neighbour counts when the
// pixel's gradient is below 1.4 x depth_diff_threshold or its relative depth
// difference is below depth_diff_threshold.  Depth and each normal
// component take their own median (element count / 2 after the sort); the
// normal is then normalised.  Every tap of a colour-c pixel is of colour
// 1 - c, so a pass reads nothing it writes.
__device__ __forceinline__ void median_tile(const Ctx& cx) {
  int row, col;
  if (!tile_pixel(cx, row, col)) return;
  const VPtr v = cx.v;
  const int W = v->W, H = v->H;
  const int plane = W * H;
  const int p = row * W + col;
  const float thr = v->depth_diff_threshold;
  const float gthr = 1.4f * thr;
  const float grad = G(v->geom_grad)[p];
  const float cd = G(v->depth)[p];
  const float inv = 1.0f / cd;
  constexpr int kTaps = 17;
  constexpr int offs[kTaps - 1][2] = {{-1, 0}, {1, 0},  {0, -1}, {0, 1},  {-3, 0}, {3, 0},   {0, -3},  {0, 3},
                                      {-2, 1}, {-1, 2}, {1, 2},  {2, 1},  {2, -1}, {1, -2}, {-1, -2}, {-2, -1}};
  float dd[kTaps], nx[kTaps], ny[kTaps], nz[kTaps];
#pragma unroll
  for (int k = 0; k < kTaps; ++k) dd[k] = nx[k] = ny[k] = nz[k] = 0.0f;
  dd[0] = cd;
  nx[0] = G(v->normal)[p];
  ny[0] = G(v->normal)[plane + p];
  nz[0] = G(v->normal)[2 * plane + p];
  int cnt = 1;
#pragma unroll
  for (int k = 0; k < kTaps - 1; ++k) {
    const int w = row + offs[k][0], u = col + offs[k][1];
    if (w < 0 || w >= H || u < 0 || u >= W) continue;
    const int q = w * W + u;
    const float d = G(v->depth)[q];
    const float diff = fabsf(d - cd) * inv;
    if (grad < gthr || (grad >= gthr && diff < thr)) {
      const float a = G(v->normal)[q], b = G(v->normal)[plane + q], c = G(v->normal)[2 * plane + q];
#pragma unroll
      for (int j = 1; j < kTaps; ++j) {
        const bool at = j == cnt;
        dd[j] = at ? d : dd[j];
        nx[j] = at ? a : nx[j];
        ny[j] = at ? b : ny[j];
        nz[j] = at ? c : nz[j];
      }
      ++cnt;
    }
  }
  bubble_sort_regs(dd, cnt);
  bubble_sort_regs(nx, cnt);
  bubble_sort_regs(ny, cnt);
  bubble_sort_regs(nz, cnt);
  const int nth = cnt >> 1;
  const float mx = pick_reg(nx, nth), my = pick_reg(ny, nth), mz = pick_reg(nz, nth);
  const float inv_norm = 1.0f / sqrtf(mx * mx + my * my + mz * mz);
  G(v->depth)[p] = pick_reg(dd, nth);
  G(v->normal)[p] = mx * inv_norm;
  G(v->normal)[plane + p] = my * inv_norm;
  G(v->normal)[2 * plane + p] = mz * inv_norm;
}

__global__ __launch_bounds__(kSweepThreads) void k_median(const LaunchTable* __restrict__ lt) {
  for_each_tile(lt, [&](int t) { median_tile(resolve(lt, t)); });
}

// RunFilter (patch_match_cuda.cu:1074-1108): FilterDepthMapsKernel
// (kernel_functions.cu:3356-3450) or, with dedup, DeduplicDepthMapsKernel
// (:3452-3490).  The geometric-consistency cost is the sweep's geometric
// term (same bilinear source depth and back-projection).  One thread per
// pixel; each pixel reads and writes only its own depth.
__global__ __launch_bounds__(256) void k_run_filter(const ViewDev* vd, int dedup, float filter_max_cost,
                                                    int min_consistent) {
  const VPtr v = (VPtr)vd;
  const int col = blockIdx.x * 16 + (int)(threadIdx.x & 15u);
  const int row = blockIdx.y * 16 + (int)(threadIdx.x >> 4);
  if (col >= v->W || row >= v->H) return;
  const int p = row * v->W + col;
  __attribute__((address_space(1))) float* depth = G(v->depth);
  const float d = depth[p];
  if ((double)d < 1e-6) {
    depth[p] = 0.0f;
    return;
  }
  Pix px;
  px.row = row;
  px.col = col;
  px.np0 = v->refInvK[0] * (float)col + v->refInvK[1];
  px.np1 = v->refInvK[2] * (float)row + v->refInvK[3];
  Counters cnt;
  int good = 0;
  for (int i = 0; i < v->N; ++i) {
    if (geom_eval(v, i, px, d, v->refK, cnt) <= filter_max_cost) {
      if (dedup) {
        depth[p] = 0.0f;
        return;
      }
      good++;
    }
  }
  if (!dedup && good < min_consistent) depth[p] = 0.0f;
}

__global__ void k_zero_u32(uint32_t* __restrict__ p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0u;
}

// ---------------------------------------------------------------------------
// preprocessing

__global__ void k_quads_u8(const uint8_t* __restrict__ img, int W, int H, int stride, uint32_t* __restrict__ out) {
  const int pw = W + 2 * kQuadPad, ph = H + 2 * kQuadPad;
  const int px = blockIdx.x * blockDim.x + threadIdx.x;
  const int py = blockIdx.y * blockDim.y + threadIdx.y;
  if (px >= pw || py >= ph) return;
  const int x = px - kQuadPad, y = py - kQuadPad;
  uint32_t q = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int xx = x + (k & 1), yy = y + (k >> 1);
    const uint32_t t = (xx < 0 || xx >= W || yy < 0 || yy >= H) ? 0u : (uint32_t)img[yy * stride + xx];
    q |= t << (8 * k);
  }
  out[py * pw + px] = q;
}

__global__ void k_quads_f16(const uint8_t* __restrict__ img, int W, int H, int stride, uint2* __restrict__ out) {
  const int pw = W + 2 * kQuadPad, ph = H + 2 * kQuadPad;
  const int px = blockIdx.x * blockDim.x + threadIdx.x;
  const int py = blockIdx.y * blockDim.y + threadIdx.y;
  if (px >= pw || py >= ph) return;
  const int x = px - kQuadPad, y = py - kQuadPad;
  float t[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int xx = x + (k & 1), yy = y + (k >> 1);
    t[k] = (xx < 0 || xx >= W || yy < 0 || yy >= H) ? 0.0f : (float)img[yy * stride + xx];
  }
  // (t00, t01 - t00, t10, t11 - t10): integers of magnitude <= 255, exact in
  // f16, so each horizontal lerp is one mixed-precision FMA on the halves
  const unsigned short h0 = __half_as_ushort(__float2half(t[0]));
  const unsigned short h1 = __half_as_ushort(__float2half(t[1] - t[0]));
  const unsigned short h2 = __half_as_ushort(__float2half(t[2]));
  const unsigned short h3 = __half_as_ushort(__float2half(t[3] - t[2]));
  out[py * pw + px] = make_uint2((uint32_t)h0 | ((uint32_t)h1 << 16), (uint32_t)h2 | ((uint32_t)h3 << 16));
}

__global__ void k_depth_quads(const float* __restrict__ d, int W, int H, float4* __restrict__ out) {
  const int pw = W + 2 * kQuadPad, ph = H + 2 * kQuadPad;
  const int px = blockIdx.x * blockDim.x + threadIdx.x;
  const int py = blockIdx.y * blockDim.y + threadIdx.y;
  if (px >= pw || py >= ph) return;
  const int x = px - kQuadPad, y = py - kQuadPad;
  float t[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int xx = x + (k & 1), yy = y + (k >> 1);
    t[k] = (xx < 0 || xx >= W || yy < 0 || yy >= H) ? 0.0f : d[yy * W + xx];
  }
  out[py * pw + px] = make_float4(t[0], t[1], t[2], t[3]);
}

// FilterKernel + ComputeGradientMap
__global__ void k_ref_moments(const ViewDev* __restrict__ v, int accum_mode, float4* __restrict__ refm,
                              uint8_t* __restrict__ grad_ok) {
  const int col = blockIdx.x * blockDim.x + threadIdx.x;
  const int row = blockIdx.y * blockDim.y + threadIdx.y;
  const int W = v->W, H = v->H;
  if (col >= W || row >= H) return;
  const int R = v->radius, S = v->step;
  const uint8_t* ref = v->ref;
  auto px_at = [&](int r, int c) -> int { return (r < 0 || r >= H || c < 0 || c >= W) ? 0 : (int)ref[r * W + c]; };
  const int c = px_at(row, col);
  float sw = 0.0f, sr = 0.0f, srr = 0.0f;
  int k = 0;
  for (int dr = -R; dr <= R; dr += S) {
    for (int dc = -R; dc <= R; dc += S) {
      const int ri = px_at(row + dr, col + dc);
      const float r = (float)ri;
      const float w = G(v->sp)[k++] * G(v->ct)[abs(c - ri)];
      const float wr = w * r;
      sw = sw + w;
      sr = sr + wr;
      srr = fmaf(wr, r, srr);
    }
  }
  const float mu = sr / sw;
  const float m2 = srr / sw;
  float var = m2 - mu * mu;
  float err = 0.0f;
  if (accum_mode == PM_ACCUM_COMPENSATED) {
    float s1 = 0.0f, s2 = 0.0f;
    k = 0;
    for (int dr = -R; dr <= R; dr += S) {
      for (int dc = -R; dc <= R; dc += S) {
        const int ri = px_at(row + dr, col + dc);
        const float d = (float)ri - mu;
        const float w = G(v->sp)[k++] * G(v->ct)[abs(c - ri)];
        const float wd = w * d;
        s1 = s1 + wd;
        s2 = fmaf(wd, d, s2);
      }
    }
    err = s1 / sw;
    var = s2 / sw - err * err;
  }
  refm[row * W + col] = make_float4(mu, var, 1.0f / sw, err);
  const float kx[3][3] = {{-3, 0, 3}, {-10, 0, 10}, {-3, 0, 3}};
  const float ky[3][3] = {{-3, -10, -3}, {0, 0, 0}, {3, 10, 3}};
  float gx = 0.0f, gy = 0.0f;
#pragma unroll
  for (int dr = -1; dr <= 1; ++dr) {
#pragma unroll
    for (int dc = -1; dc <= 1; ++dc) {
      const float color = (float)px_at(row + dr, col + dc) / 255.0f;
      gx = gx + color * kx[dr + 1][dc + 1];
      gy = gy + color * ky[dr + 1][dc + 1];
    }
  }
  const float grad = sqrtf(gx * gx + gy * gy);
  grad_ok[row * W + col] = grad >= 1.0f ? 1 : 0;
}

// ---------------------------------------------------------------------------
// dispatch over the compiled (radius, step) shapes

template <int R, int S, int ST, int RC>
struct SweepK {
  static void* fn() { return (void*)&k_sweep<R, S, ST, RC>; }
};
template <int R, int S, int ST, int RC>
struct InitK {
  static void* fn() { return (void*)&k_init<R, S, ST, RC>; }
};
template <int R, int S, int ST, int RC>
struct LocalK {
  static void* fn() { return (void*)&k_local_opt<R, S, ST, RC>; }
};

template <template <int, int, int, int> class Kn, int R, int S>
void* pick_sr(int storage, int rcp) {
  if (storage == PM_STORAGE_U8) {
    return rcp == PM_RCP_EXACT ? Kn<R, S, PM_STORAGE_U8, PM_RCP_EXACT>::fn() : Kn<R, S, PM_STORAGE_U8, PM_RCP_FAST>::fn();
  }
  return rcp == PM_RCP_EXACT ? Kn<R, S, PM_STORAGE_F16, PM_RCP_EXACT>::fn() : Kn<R, S, PM_STORAGE_F16, PM_RCP_FAST>::fn();
}

template <template <int, int, int, int> class Kn>
void* pick_kernel(const LaunchCfg& cfg) {
  const int r = cfg.radius, st = cfg.step;
  if (r == 5 && st == 2) return pick_sr<Kn, 5, 2>(cfg.storage, cfg.rcp);
  if (r == 7 && st == 1) return pick_sr<Kn, 7, 1>(cfg.storage, cfg.rcp);
  if (r == 5 && st == 1) return pick_sr<Kn, 5, 1>(cfg.storage, cfg.rcp);
  if (r == 7 && st == 2) return pick_sr<Kn, 7, 2>(cfg.storage, cfg.rcp);
  return pick_sr<Kn, -1, -1>(cfg.storage, cfg.rcp);
}

bool compiled_window(const LaunchCfg& cfg) {
  return (cfg.radius == 5 || cfg.radius == 7) && (cfg.step == 1 || cfg.step == 2);
}

}  // namespace


hipError_t launch_build_quads_u8(const uint8_t* img, int W, int H, int stride, uint32_t* out, hipStream_t s) {
  if (W <= 0 || H <= 0 || stride < W) return hipErrorInvalidValue;
  const dim3 blk(32, 8), grd((W + 2 * kQuadPad + 31) / 32, (H + 2 * kQuadPad + 7) / 8);
  hipLaunchKernelGGL(k_quads_u8, grd, blk, 0, s, img, W, H, stride, out);
  return hipGetLastError();
}

hipError_t launch_build_quads_f16(const uint8_t* img, int W, int H, int stride, uint2* out, hipStream_t s) {
  if (W <= 0 || H <= 0 || stride < W) return hipErrorInvalidValue;
  const dim3 blk(32, 8), grd((W + 2 * kQuadPad + 31) / 32, (H + 2 * kQuadPad + 7) / 8);
  hipLaunchKernelGGL(k_quads_f16, grd, blk, 0, s, img, W, H, stride, out);
  return hipGetLastError();
}

hipError_t launch_build_depth_quads(const float* depth, int W, int H, float4* out, hipStream_t s) {
  if (W <= 0 || H <= 0) return hipErrorInvalidValue;
  const dim3 blk(32, 8), grd((W + 2 * kQuadPad + 31) / 32, (H + 2 * kQuadPad + 7) / 8);
  hipLaunchKernelGGL(k_depth_quads, grd, blk, 0, s, depth, W, H, out);
  return hipGetLastError();
}

hipError_t launch_ref_moments(const ViewDev* v, int W, int H, int accum_mode, float4* refm, uint8_t* grad_ok,
                              hipStream_t s) {
  if (W <= 0 || H <= 0) return hipErrorInvalidValue;
  const dim3 blk(32, 8), grd((W + 31) / 32, (H + 7) / 8);
  hipLaunchKernelGGL(k_ref_moments, grd, blk, 0, s, v, accum_mode, refm, grad_ok);
  return hipGetLastError();
}

namespace {

void* phase_kernel(PhaseKind kind, const LaunchCfg& cfg) {
  switch (kind) {
    case kPhaseInit: return pick_kernel<InitK>(cfg);
    case kPhaseSweep: return pick_kernel<SweepK>(cfg);
    case kPhaseLocal: return pick_kernel<LocalK>(cfg);
    case kPhaseFilter: return (void*)&k_filter;
    case kPhaseCurvature: return (void*)&k_curvature;
    case kPhaseMask: return (void*)&k_mask;
    case kPhaseGeomGrad: return (void*)&k_geom_grad;
    case kPhaseMedian: return (void*)&k_median;
  }
  return nullptr;
}

// Launch-time LDS of a windowed phase whose window has no compiled kernel:
// the spatial weights and the widest ref tile of the tile shapes.
size_t window_lds_bytes(PhaseKind kind, const LaunchCfg& cfg) {
  if (plain_phase(kind) || compiled_window(cfg)) return 0;
  const int n = (2 * cfg.radius) / cfg.step + 1;
  size_t words = 0;
  for (int lw = kTileLog2WMin; lw <= kTileLog2WMax; ++lw) {
    const size_t w = (size_t)((1 << lw) + 2 * cfg.radius) * ((kTilePixels >> lw) + 2 * cfg.radius);
    words = w > words ? w : words;
  }
  return ((size_t)n * n + words) * sizeof(uint32_t);
}

}  // namespace

namespace {
std::mutex g_occ_mu;
std::map<std::pair<void*, size_t>, int> g_occ;
std::map<int, int> g_cus;
}  // namespace

int phase_occupancy(PhaseKind kind, const LaunchCfg& cfg) {
  void* fn = phase_kernel(kind, cfg);
  if (!fn) return 1;
  const size_t dyn = window_lds_bytes(kind, cfg);
  std::lock_guard<std::mutex> lk(g_occ_mu);
  const std::pair<void*, size_t> key(fn, dyn);
  auto it = g_occ.find(key);
  if (it == g_occ.end()) {
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, fn, kSweepThreads, dyn) != hipSuccess || n <= 0) n = 1;
    it = g_occ.emplace(key, n).first;
  }
  return it->second;
}

int phase_grid(PhaseKind kind, const LaunchCfg& cfg, int tiles, int blocks_per_cu) {
  if (tiles <= 0) return 0;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  int per_cu = phase_occupancy(kind, cfg), n_cu = 0;
  {
    std::lock_guard<std::mutex> lk(g_occ_mu);
    std::map<int, int>& cus = g_cus;
    auto ic = cus.find(dev);
    if (ic == cus.end()) {
      int n = 0;
      if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 1;
      ic = cus.emplace(dev, n).first;
    }
    n_cu = ic->second;
  }
  if (per_cu > kMaxBlocksPerCU) per_cu = kMaxBlocksPerCU;
  if (blocks_per_cu > 0 && blocks_per_cu < per_cu) per_cu = blocks_per_cu;
  const long long g = (long long)n_cu * per_cu;
  return (int)(g < tiles ? g : tiles);
}

// Tiles of 64 pixels of a colour (four waves on each) where tiles of 256 would
// not give every workgroup slot of the chip one, and of 16 where those of 64
// would leave CUs idle (a quarter of the slots: 4 workgroups to a CU).  Above
// its line the larger tile wins: its lists of 64 pairs are fuller, and the
// work that a workgroup does once per tile is spread further.  Whole runs in
// ms, tiles of 256 / 64 / 16 pixels:
//   96x64     4.22 / 1.79 / 1.25     160x120 (2 sources)  2.26 / 1.27 / 1.15
//   240x160   4.50 / 2.33 / 2.87     640x480              6.58 / 6.25 / 12.9
//   1021x767  23.0 / 24.6            1920x1080 geometric  78.1 / 78.2
//
// What a tile costs once weighs the more the less its pixels' walks take, so
// the line between 256 and 64 pixels falls with the sources and the window
// samples of a pixel.  Thousands of pixels at which the two take the same time
// (1024 slots; 11x11 step 2 has 36 samples, 15x15 step 2 64, 11x11 121):
//   sources            1                2            4
//   samples       36   64  121    36   64  121    36   64
//   sweep        175  224  485   285  347  490   486 >520
//   local opt.   121  128  148   146  186  330   197  323
// Compensated moments weigh about three samples.  The lines are fitted to 756
// views (350x262 to 832x624, 1 to 9 sources, 16 to 225 samples; u8, f16,
// compensated, geometric), where a run takes at most 3% more than with 64
// pixels everywhere below 512 a slot, and 4% less on average.  Four iterations,
// 256 / 64 pixels: 640x480, 1 source, 36 samples 1.47 / 1.99 ms; 800x600, 1
// source, 9 samples 1.38 / 2.80.
double small_tile_line(PhaseKind kind, const LaunchCfg& cfg, int num_src, int accum_mode) {
  const int n = 2 * cfg.radius / cfg.step + 1;
  const double samples = (double)(n * n) * (accum_mode == PM_ACCUM_COMPENSATED ? 3.0 : 1.0);
  const double line = kind == kPhaseSweep ? 80.0 + 1.7 * num_src * (samples + 20.0) + 0.6 * samples
                                          : 110.0 + 0.8 * num_src * samples;
  return line < 512.0 ? line : 512.0;
}

TileShape tile_shape(PhaseKind kind, const LaunchCfg& cfg, int lw, long long pixels, double line, int blocks_per_cu) {
  if (kind == kPhaseSweep || kind == kPhaseLocal) {
    const long long slots = phase_grid(kind, cfg, INT32_MAX, blocks_per_cu);
    if (pixels < slots / 4 * 128) return TileShape{3, 4};
    if ((double)pixels < (double)slots * line) return TileShape{4, 6};
  }
  return TileShape{lw, kTileLog2Px};
}

hipError_t launch_phase(PhaseKind kind, const LaunchCfg& cfg, const LaunchTable* table, int grid, hipStream_t s) {
  if (grid <= 0 || !table) return hipErrorInvalidValue;
  void* fn = phase_kernel(kind, cfg);
  if (!fn) return hipErrorInvalidValue;
  void* args[] = {(void*)&table};
  return hipLaunchKernel(fn, dim3((unsigned)grid), dim3(kSweepThreads), args, window_lds_bytes(kind, cfg), s);
}

hipError_t launch_run_filter(const ViewDev* v, int W, int H, int dedup, float filter_max_cost, int min_consistent,
                             hipStream_t s) {
  if (W <= 0 || H <= 0 || !v) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_run_filter, dim3((unsigned)((W + 15) / 16), (unsigned)((H + 15) / 16)), dim3(256), 0, s, v, dedup,
                     filter_max_cost, min_consistent);
  return hipGetLastError();
}

hipError_t launch_zero_u32(uint32_t* p, int n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  if (!p) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_zero_u32, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p, n);
  return hipGetLastError();
}

}  // namespace pm
