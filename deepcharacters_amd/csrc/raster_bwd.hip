// Rasterizer backward (CudaRendererGradGpu) on gfx950.
//
// Gather form (with the workspace that dcx_render_bwd_workspace_size asks for):
// four lanes per (view, face), or a wavefront for the larger ones, find the
// pixels of the face's box whose stored face id is its own, form their contributions from the stored barycentrics
// (nothing per-pixel is kept from the forward pass besides the reference's
// face / barycentric buffers) and sum them in registers; eight lanes per
// vertex then add up the records of its faces in all views.  No atomics but
// the texture's and one flush of the SH gradients a workgroup, and the sums
// have a fixed order.
//
// Scatter form (the remaining pixels: faces over more than kGatherBox pixels,
// face buffers that were not rendered from these positions; and everything,
// for callers without that workspace): one lane per pixel, pixels in row-major
// order so a wavefront covers 64 consecutive pixels of a row; the wavefront
// combines runs of equal face ids with a segmented shuffle scan and only the
// last lane of each run issues the global atomics.  SH gradients (27 floats
// per camera, hit by every pixel of that camera) are reduced per block in LDS
// first.
//
// Shaded mode also differentiates the vertex normals (sums of the adjacent
// unnormalised face normals, CUDABasedRasterizationGrad.cu:441-493): both
// forms sum dL/d(vertex normal) per vertex into a [B,N,3] workspace, then the
// vertices' faces apply the face-normal Jacobians (RendererUtil.h:492-540) --
// a deterministic gather in place of the reference's per-pixel loop over the
// faces around each corner.
#include <type_traits>

#include "raster_common.hpp"
#include "raster_internal.hpp"

namespace dcx {
namespace {

constexpr int kB = 256;

struct BwdArgs {
  int B, C, N, F, H, W;
  int albedo, shaded, TH, TW, img_fs, tex_fs;
  const int* faces;
  const float* tc;
  const float* g_render;  // [B,C,H,W,3]
  const float* vpos;      // [B,N,3]
  const float* vcol;      // [B,N,3]
  const float* tex;       // [B,TH,TW,3]
  const float* sh;        // [B,C,27]
  const float* target;    // [B,C,H,W,3] or null
  const float* vnormal;   // [B,C,N,3]
  const float* bary;      // [B,C,H,W,2]
  const int* face;        // [B,C,H,W]
  const float* ext;
  const float* intr;
  float* g_vpos;
  float* g_vcol;
  float* g_tex;
  float* g_sh;
  float* g_vn;            // [B,N,3] shaded only
  // gather form
  float* rec;             // [B,C,F,rec_n] sums of a face's pixels in a view: position, colour, normal of 3 corners
  uint2* box;             // [B,C,F] a face's box: x0 | y0 << 16, nx | ny << 10 | (record written) << 20
  unsigned int* rest_n;   // pixel groups left to the scatter form, and
  unsigned int* rest;     // which ([pixels / kB] at most)
  unsigned int* wide_n;   // [B,C], kWideStride apart: faces left to a wavefront each, and
  unsigned int* wide;     // [B,C,F] which
  int rec_n, rec_col, rec_vn;
};

// Faces whose box holds more pixels are left to the scatter form, where a
// large triangle's pixels are spread over many wavefronts and its long runs
// combine well.  Below that, a face with a box of more than kLaneBox pixels or
// more than kLaneHits pixels a lane takes a wavefront: large faces lie together
// (the caps of a limb), so the wavefronts that hold them would be the last.
constexpr int kGatherBox = 1023;  // (nx and ny are stored in 10 bits)
constexpr int kLaneBox = 256;
constexpr int kLaneHits = 6;
constexpr int kWideStride = 32;   // counters that many workgroups add to, 128 bytes apart
constexpr int kFaceLanes = 4;

// Pixels that a face can cover: centres in the bounding box of its projection
// (and of its corners snapped to 1/256 pixel).  nx = 0: none, or not gathered.
struct FaceBox {
  int x0, y0, nx, ny;
  __device__ __forceinline__ bool has(int x, int y) const {
    return x >= x0 && x < x0 + nx && y >= y0 && y < y0 + ny;
  }
};
__device__ __forceinline__ FaceBox face_box(f4 p0, f4 p1, f4 p2, int W, int H) {
  FaceBox b{0, 0, 0, 0};
  if (!(p0.w > 0.f && p1.w > 0.f && p2.w > 0.f)) return b;
  constexpr float kMargin = 1.f / 256.f;
  const float x0 = fmaxf(ceilf(fminf(p0.x, fminf(p1.x, p2.x)) - 0.5f - kMargin), 0.f);
  const float y0 = fmaxf(ceilf(fminf(p0.y, fminf(p1.y, p2.y)) - 0.5f - kMargin), 0.f);
  const float x1 = fminf(floorf(fmaxf(p0.x, fmaxf(p1.x, p2.x)) - 0.5f + kMargin), (float)(W - 1));
  const float y1 = fminf(floorf(fmaxf(p0.y, fmaxf(p1.y, p2.y)) - 0.5f + kMargin), (float)(H - 1));
  if (!(x0 <= x1 && y0 <= y1 && (x1 - x0 + 1.f) * (y1 - y0 + 1.f) <= (float)kGatherBox)) return b;
  b.x0 = (int)x0; b.y0 = (int)y0; b.nx = (int)x1 - b.x0 + 1; b.ny = (int)y1 - b.y0 + 1;
  return b;
}
__device__ __forceinline__ FaceBox unpack_box(uint2 w) {
  return {(int)(w.x & 0xffff), (int)(w.x >> 16), (int)(w.y & 0x3ff), (int)((w.y >> 10) & 0x3ff)};
}

// imageGradient of RendererUtil.h:566-620 at a (possibly fractional) point:
// the sample index is formed as (int)((y + yy) * W + (x + xx)) in float.  kFs:
// the filter size where it is known, so that a row's loads are issued
// together (one tap after the other, a 5 x 5 filter was the longest part of a
// pixel); 0: any.
template <int kFs>
__device__ __forceinline__ void image_gradient_of(const float* img, float x, float y, int W, int H, int fs_, f3& du,
                                                  f3& dv) {
  const int fs = kFs ? kFs : fs_;
  du = mk3(0.f, 0.f, 0.f);
  dv = mk3(0.f, 0.f, 0.f);
  if (!(x >= (float)(fs + 1) && y >= (float)(fs + 1) && x < (float)(W - (fs + 1)) && y < (float)(H - (fs + 1))))
    return;
  float norm = 0.f;
  auto tap = [&](int xx, int yy, f3 I) {
    const float den = (float)(xx * xx + yy * yy);
    float gu = 0.f, gv = 0.f;
    if (den != 0.f) { gu = (float)xx / den; gv = (float)yy / den; }
    du = du + I * gu;
    dv = dv + I * gv;
    norm += fabsf(gu);
  };
  auto at = [&](int xx, int yy) {
    return ld3(img + (size_t)(int)((y + (float)yy) * (float)W + (x + (float)xx)) * 3);
  };
  if (kFs) {
#pragma unroll
    for (int yy = -kFs; yy <= kFs; ++yy) {
      f3 I[2 * kFs + 1];
#pragma unroll
      for (int xx = -kFs; xx <= kFs; ++xx) I[xx + kFs] = at(xx, yy);
#pragma unroll
      for (int xx = -kFs; xx <= kFs; ++xx) tap(xx, yy, I[xx + kFs]);
    }
  } else {
    for (int yy = -fs; yy <= fs; ++yy)
      for (int xx = -fs; xx <= fs; ++xx) tap(xx, yy, at(xx, yy));
  }
  du = mk3(du.x / norm, du.y / norm, du.z / norm);
  dv = mk3(dv.x / norm, dv.y / norm, dv.z / norm);
}
__device__ __forceinline__ void image_gradient(const float* img, float x, float y, int W, int H, int fs, f3& du, f3& dv) {
  if (fs == 1) image_gradient_of<1>(img, x, y, W, H, fs, du, dv);
  else if (fs == 2) image_gradient_of<2>(img, x, y, W, H, fs, du, dv);
  else image_gradient_of<0>(img, x, y, W, H, fs, du, dv);
}

// d(b0, b1, 1-b0-b1)/d(world vertex positions) contracted with gb = dL/d weights.
__device__ void bary_vjp(const float* E, const float* K, const f3 X[3], float px, float py, const float gb_in[3],
                         f3 out[3]) {
  float h0[3], h1[3], h2[3], u[3], v[3], iz[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const float xc = E[0] * X[i].x + E[1] * X[i].y + E[2] * X[i].z + E[3];
    const float yc = E[4] * X[i].x + E[5] * X[i].y + E[6] * X[i].z + E[7];
    const float zc = E[8] * X[i].x + E[9] * X[i].y + E[10] * X[i].z + E[11];
    h0[i] = K[0] * xc + K[1] * yc + K[2] * zc;
    h1[i] = K[3] * xc + K[4] * yc + K[5] * zc;
    h2[i] = K[6] * xc + K[7] * yc + K[8] * zc;
    u[i] = h0[i] / h2[i];
    v[i] = h1[i] / h2[i];
    iz[i] = 1.f / h2[i];
  }
  float e[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const int j = i == 2 ? 0 : i + 1, k = i == 0 ? 2 : i - 1;
    e[i] = (u[k] - u[j]) * (py - v[j]) - (v[k] - v[j]) * (px - u[j]);
  }
  const float q0 = e[0] * iz[0], q1 = e[1] * iz[1], q2 = e[2] * iz[2];
  const float Q = q0 + q1 + q2;
  const float b0 = q0 / Q, b1 = q1 / Q;
  const float g0 = gb_in[0] - gb_in[2], g1 = gb_in[1] - gb_in[2];
  const float s = g0 * b0 + g1 * b1;
  const float gq[3] = {(g0 - s) / Q, (g1 - s) / Q, (0.f - s) / Q};
  float gu[3] = {0.f, 0.f, 0.f}, gv[3] = {0.f, 0.f, 0.f}, giz[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    giz[i] = gq[i] * e[i];
    const float ge = gq[i] * iz[i];
    const int j = i == 2 ? 0 : i + 1, k = i == 0 ? 2 : i - 1;
    gu[j] += ge * (v[k] - py);
    gv[j] += ge * (px - u[k]);
    gu[k] += ge * (py - v[j]);
    gv[k] += ge * (u[j] - px);
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const float gh0 = gu[i] / h2[i], gh1 = gv[i] / h2[i];
    const float gh2 = -(gu[i] * u[i] + gv[i] * v[i]) / h2[i] - giz[i] * iz[i] * iz[i];
    const float gx = K[0] * gh0 + K[3] * gh1 + K[6] * gh2;
    const float gy = K[1] * gh0 + K[4] * gh1 + K[7] * gh2;
    const float gz = K[2] * gh0 + K[5] * gh1 + K[8] * gh2;
    out[i] = mk3(E[0] * gx + E[4] * gy + E[8] * gz, E[1] * gx + E[5] * gy + E[9] * gz,
                 E[2] * gx + E[6] * gy + E[10] * gz);
  }
}

// Segmented (by key) inclusive scan over a wavefront: afterwards the last lane
// of each run of equal keys holds the run's sum.  Every lane must call it.
template <int NV>
__device__ __forceinline__ bool seg_reduce(float* v, int key, int key2) {
  const int lane = threadIdx.x & 63;
  const int prev = __shfl_up(key, 1, 64), prev2 = __shfl_up(key2, 1, 64);
  const int next = __shfl_down(key, 1, 64), next2 = __shfl_down(key2, 1, 64);
  int start = (lane == 0 || prev != key || prev2 != key2) ? lane : 0;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int o = __shfl_up(start, d, 64);
    if (lane >= d) start = max(start, o);
  }
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const bool take = lane - d >= start;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const float o = __shfl_up(v[j], d, 64);
      if (take) v[j] += o;
    }
  }
  return lane == 63 || next != key || next2 != key2;
}

template <bool kRest>
__device__ __forceinline__ void bwd_group(const BwdArgs& a, unsigned int group) {
  __shared__ float s_sh[27];
  const long long HW = (long long)a.H * a.W;
  const long long i = (long long)group * kB + threadIdx.x;
  const bool valid = i < (long long)a.B * a.C * HW;
  const int view = valid ? (int)(i / HW) : 0;
  // SH accumulation is per camera; a block never straddles two views when HW % 256 == 0,
  // otherwise the per-lane atomics below handle the rest.
  const int view0 = (int)(((long long)group * kB) / HW);
  const bool block_one_view = ((long long)group * kB + kB - 1) / HW == view0;
  if (a.shaded && a.g_sh) {
    __syncthreads();  // the group before
    if (threadIdx.x < 27) s_sh[threadIdx.x] = 0.f;
    __syncthreads();
  }
  int f = valid ? a.face[i] : -1;
  if (kRest && f >= 0) {
    const int p = (int)(i - (long long)view * HW);
    if (unpack_box(a.box[(size_t)view * a.F + f]).has(p % a.W, p / a.W)) f = -1;
  }
  float acc[27];  // 0-8 position, 9-17 colour, 18-26 vertex-normal gradients of the 3 corners
#pragma unroll
  for (int k = 0; k < 27; ++k) acc[k] = 0.f;
  const int b = view / a.C;
  int i0 = 0, i1 = 0, i2 = 0;
  float shv[27];
  bool have_sh = false;
  if (f >= 0) {
    const int p = (int)(i - (long long)view * HW);
    const int x = p % a.W, y = p / a.W;
    const float px = (float)x + 0.5f, py = (float)y + 0.5f;
    const float* E = a.ext + (size_t)view * 12;
    const float* K = a.intr + (size_t)view * 9;
    i0 = a.faces[3 * f]; i1 = a.faces[3 * f + 1]; i2 = a.faces[3 * f + 2];
    const int idx[3] = {i0, i1, i2};
    const float wa = a.bary[2 * i], wb = a.bary[2 * i + 1];
    const float w[3] = {wa, wb, 1.f - wa - wb};
    const f3 g = ld3(a.g_render + 3 * i);
    const float* vp = a.vpos + (size_t)b * a.N * 3;
    // pixel normal (interpolated, normalised, flipped to face the camera)
    f3 n = mk3(0.f, 0.f, 0.f), pn = n;
    float pl = 1.f;
    bool flipped = false;
    const float* shc = a.sh ? a.sh + (size_t)view * 27 : nullptr;
    if (a.shaded || a.albedo == ALB_TEXTURED) {
      const float* vn = a.vnormal + (size_t)view * a.N * 3;
      const f3 n0 = ld3(vn + 3 * i0), n1 = ld3(vn + 3 * i1), n2 = ld3(vn + 3 * i2);
      pn = mk3(w[0] * n0.x + w[1] * n1.x + w[2] * n2.x, w[0] * n0.y + w[1] * n1.y + w[2] * n2.y,
               w[0] * n0.z + w[1] * n1.z + w[2] * n2.z);
      pl = sqrtf(dot(pn, pn));
      n = mk3(pn.x / pl, pn.y / pl, pn.z / pl);
      if (dot(n, world_ray_dir(E, K, px, py)) > 0.f) { n = -n; flipped = true; }
    }
    f3 light = mk3(1.f, 1.f, 1.f);
    if (a.shaded) light = sh_shade(mk3(1.f, 1.f, 1.f), n, shc);
    const f3 ga = mk3(g.x * light.x, g.y * light.y, g.z * light.z);
    f3 cols[3];
    f3 alb = mk3(0.f, 0.f, 0.f);
    float U0 = 0.f, V0 = 0.f;
    const float* t6 = a.tc ? a.tc + (size_t)f * 6 : nullptr;
    if (a.albedo == ALB_VERTEX_COLOR || a.albedo == ALB_FOREGROUND) {
      const float* vc = a.vcol + (size_t)b * a.N * 3;
#pragma unroll
      for (int k = 0; k < 3; ++k) cols[k] = ld3(vc + 3 * idx[k]);
      alb = cols[0] * w[0] + cols[1] * w[1] + cols[2] * w[2];
    } else if (a.albedo == ALB_TEXTURED) {
      U0 = (t6[0] * w[0] + t6[2] * w[1] + t6[4] * w[2]) * (float)a.TW;
      V0 = ((1.f - t6[1]) * w[0] + (1.f - t6[3]) * w[1] + (1.f - t6[5]) * w[2]) * (float)a.TH;
      U0 = fminf(fmaxf(U0, 0.f), (float)(a.TW - 1));
      V0 = fminf(fmaxf(V0, 0.f), (float)(a.TH - 1));
      const float LU = (float)(int)(U0 - 0.5f) + 0.5f, HU = LU + 1.f;
      const float LV = (float)(int)(V0 - 0.5f) + 0.5f, HV = LV + 1.f;
      const float* tx = a.tex + (size_t)b * a.TH * a.TW * 3;
      auto at = [&](float uu, float vv) { return ld3(tx + ((size_t)(int)vv * a.TW + (int)uu) * 3); };
      // the reference's swapped-weight "bilinear" albedo (CUDABasedRasterizationGrad.cu:242-243)
      alb = (at(LU, LV) * (U0 - LU) + at(HU, LV) * (HU - U0)) * (V0 - LV) +
            (at(LU, HV) * (U0 - LU) + at(HU, HV) * (HU - U0)) * (HV - V0);
      if (!flipped && a.g_tex) {
        float* gt = a.g_tex + (size_t)b * a.TH * a.TW * 3 + ((size_t)(int)(V0 - 0.5f) * a.TW + (int)(U0 - 0.5f)) * 3;
        atomicAdd(gt, ga.x); atomicAdd(gt + 1, ga.y); atomicAdd(gt + 2, ga.z);
      }
    }
    if (a.albedo == ALB_VERTEX_COLOR) {
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        acc[9 + 3 * k] = ga.x * w[k]; acc[10 + 3 * k] = ga.y * w[k]; acc[11 + 3 * k] = ga.z * w[k];
      }
    }
    if (a.shaded && a.g_sh) {
      const float basis[9] = {1.f, n.y, n.z, n.x, n.x * n.y, n.z * n.y, 3.f * n.z * n.z - 1.f, n.x * n.z, n.x * n.x - n.y * n.y};
      const float ca[3] = {g.x * alb.x, g.y * alb.y, g.z * alb.z};
#pragma unroll
      for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int k = 0; k < 9; ++k) shv[9 * d + k] = ca[d] * basis[k];
      have_sh = true;
    }
    float gw[3] = {0.f, 0.f, 0.f};
    if (a.albedo == ALB_VERTEX_COLOR || a.albedo == ALB_FOREGROUND) {
#pragma unroll
      for (int k = 0; k < 3; ++k) gw[k] = dot(ga, cols[k]);
    } else if (a.albedo == ALB_TEXTURED) {
      f3 du, dv;
      image_gradient(a.tex + (size_t)b * a.TH * a.TW * 3, U0, V0, a.TW, a.TH, a.tex_fs, du, dv);
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const float su = t6[2 * k] * (float)a.TW, sv = (1.f - t6[2 * k + 1]) * (float)a.TH;
        gw[k] = ga.x * (du.x * su + dv.x * sv) + ga.y * (du.y * su + dv.y * sv) + ga.z * (du.z * su + dv.z * sv);
      }
    }
    if (a.shaded) {
      f3 gn = mk3(0.f, 0.f, 0.f);
      const float gc[3] = {g.x * alb.x, g.y * alb.y, g.z * alb.z};
#pragma unroll
      for (int ch = 0; ch < 3; ++ch) {
        const float* s = shc + 9 * ch;
        const f3 Jn = mk3(s[3] + s[4] * n.y + s[7] * n.z + s[8] * 2.f * n.x,
                          s[1] + s[4] * n.x + s[5] * n.z + s[8] * -2.f * n.y,
                          s[2] + s[5] * n.y + s[6] * 6.f * n.z + s[7] * n.x);
        gn = gn + Jn * gc[ch];
      }
      const float sg = flipped ? -1.f : 1.f;
      const f3 nn = mk3(pn.x / pl, pn.y / pl, pn.z / pl);
      const float dg = sg * dot(gn, nn);
      const f3 gun = mk3((sg * gn.x - nn.x * dg) / pl, (sg * gn.y - nn.y * dg) / pl, (sg * gn.z - nn.z * dg) / pl);
      const float* vn = a.vnormal + (size_t)view * a.N * 3;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        gw[k] += dot(gun, ld3(vn + 3 * idx[k]));
        acc[18 + 3 * k] = w[k] * gun.x; acc[19 + 3 * k] = w[k] * gun.y; acc[20 + 3 * k] = w[k] * gun.z;
      }
    }
    f3 X[3] = {ld3(vp + 3 * i0), ld3(vp + 3 * i1), ld3(vp + 3 * i2)};
    f3 gx[3];
    bary_vjp(E, K, X, px, py, gw, gx);
    if (a.target) {
      f3 du, dv;
      image_gradient(a.target + (size_t)view * HW * 3, (float)x, (float)y, a.W, a.H, a.img_fs, du, dv);
      const float gu = -dot(g, du), gvv = -dot(g, dv);
      const f3 fp = X[0] * w[0] + X[1] * w[1] + X[2] * w[2];
      const float xc = E[0] * fp.x + E[1] * fp.y + E[2] * fp.z + E[3];
      const float yc = E[4] * fp.x + E[5] * fp.y + E[6] * fp.z + E[7];
      const float zc = E[8] * fp.x + E[9] * fp.y + E[10] * fp.z + E[11];
      const float hx = K[0] * xc + K[1] * yc + K[2] * zc;
      const float hy = K[3] * xc + K[4] * yc + K[5] * zc;
      const float hz = K[6] * xc + K[7] * yc + K[8] * zc;
      if (fabsf(hz) > 0.0001f) {
        const float gh0 = gu / hz, gh1 = gvv / hz, gh2 = -(gu * hx + gvv * hy) / (hz * hz);
        const float cx = K[0] * gh0 + K[3] * gh1 + K[6] * gh2;
        const float cy = K[1] * gh0 + K[4] * gh1 + K[7] * gh2;
        const float cz = K[2] * gh0 + K[5] * gh1 + K[8] * gh2;
        const f3 gX = mk3(E[0] * cx + E[4] * cy + E[8] * cz, E[1] * cx + E[5] * cy + E[9] * cz,
                          E[2] * cx + E[6] * cy + E[10] * cz);
#pragma unroll
        for (int k = 0; k < 3; ++k) gx[k] = gx[k] + gX * w[k];
      }
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) { acc[3 * k] = gx[k].x; acc[3 * k + 1] = gx[k].y; acc[3 * k + 2] = gx[k].z; }
  }
  // Combine runs of equal (view, face) within the wavefront.
  // (a wavefront without a covered pixel has nothing to combine)
  bool tail = false;
  if (__ballot(f >= 0)) tail = a.shaded ? seg_reduce<27>(acc, f, view) : seg_reduce<18>(acc, f, view);
  if (f >= 0 && tail) {
    float* gp = a.g_vpos + (size_t)b * a.N * 3;
    const int idx[3] = {i0, i1, i2};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      atomicAdd(gp + 3 * idx[k], acc[3 * k]);
      atomicAdd(gp + 3 * idx[k] + 1, acc[3 * k + 1]);
      atomicAdd(gp + 3 * idx[k] + 2, acc[3 * k + 2]);
    }
    if (a.albedo == ALB_VERTEX_COLOR) {
      float* gc = a.g_vcol + (size_t)b * a.N * 3;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        atomicAdd(gc + 3 * idx[k], acc[9 + 3 * k]);
        atomicAdd(gc + 3 * idx[k] + 1, acc[10 + 3 * k]);
        atomicAdd(gc + 3 * idx[k] + 2, acc[11 + 3 * k]);
      }
    }
    if (a.shaded) {
      float* gn = a.g_vn + (size_t)b * a.N * 3;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        atomicAdd(gn + 3 * idx[k], acc[18 + 3 * k]);
        atomicAdd(gn + 3 * idx[k] + 1, acc[19 + 3 * k]);
        atomicAdd(gn + 3 * idx[k] + 2, acc[20 + 3 * k]);
      }
    }
  }
  if (a.shaded && a.g_sh) {
    if (block_one_view) {
      for (int k = 0; k < 27 && __ballot(have_sh); ++k) {
        const float t = wave_sum(have_sh ? shv[k] : 0.f);
        if ((threadIdx.x & 63) == 0 && t != 0.f) atomicAdd(&s_sh[k], t);
      }
      __syncthreads();
      if (threadIdx.x < 27 && s_sh[threadIdx.x] != 0.f)
        atomicAdd(a.g_sh + (size_t)view0 * 27 + threadIdx.x, s_sh[threadIdx.x]);
    } else if (have_sh) {
      for (int k = 0; k < 27; ++k) atomicAdd(a.g_sh + (size_t)view * 27 + k, shv[k]);
    }
  }
}

// kRest: only the pixels that the gather form did not take, a.rest's groups of
// kB pixels in turn; otherwise the workgroup's own group.
template <bool kRest>
__global__ __launch_bounds__(kB) void render_bwd_kernel(BwdArgs a) {
  if (kRest) {
    const unsigned int n = *a.rest_n;
    for (unsigned int q = blockIdx.x; q < n; q += gridDim.x) bwd_group<true>(a, a.rest[q]);
  } else {
    bwd_group<false>(a, blockIdx.x);
  }
}

// Sums of one face's pixels in one view.
template <bool kTex, bool kShaded>
struct FaceSums {
  f3 gh[3];                // dL/d(the corners' homogeneous image points K [R | t] X)
  f3 gc[kTex ? 1 : 3];     // dL/d(vertex colour)
  f3 gn[kShaded ? 3 : 1];  // dL/d(vertex normal)
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int i = 0; i < 3; ++i) gh[i] = mk3(0.f, 0.f, 0.f);
#pragma unroll
    for (int i = 0; i < (kTex ? 1 : 3); ++i) gc[i] = mk3(0.f, 0.f, 0.f);
#pragma unroll
    for (int i = 0; i < (kShaded ? 3 : 1); ++i) gn[i] = mk3(0.f, 0.f, 0.f);
  }
};

// What a face's pixels share.
template <bool kTex, bool kShaded>
struct FaceInfo {
  f3 vn[kTex || kShaded ? 3 : 1], col[kTex ? 1 : 3];
  f4 p[3];
  float t6[kTex ? 6 : 1];
  FaceBox box;
  __device__ __forceinline__ void load(const BwdArgs& a, int view, int b, int f) {
    const float* E = a.ext + (size_t)view * 12;
    const float* K = a.intr + (size_t)view * 9;
    const float* vp = a.vpos + (size_t)b * a.N * 3;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int v = a.faces[3 * f + k];
      p[k] = project_vertex(E, K, vp + 3 * v);
      if (kTex || kShaded) vn[k] = ld3(a.vnormal + ((size_t)view * a.N + v) * 3);
      if (!kTex) col[k] = ld3(a.vcol + ((size_t)b * a.N + v) * 3);
    }
    if (kTex)
#pragma unroll
      for (int k = 0; k < 6; ++k) t6[k] = a.tc[(size_t)f * 6 + k];
    box = face_box(p[0], p[1], p[2], a.W, a.H);
  }
};

// Adds pixel (x, y) of the face to its sums; the same terms as in
// render_bwd_kernel, with what is linear in the pixels left to face_record.
// sh: the lane's 27 sums of the SH gradient, kB floats apart.
template <bool kTex, bool kShaded>
__device__ __forceinline__ void add_pixel(const BwdArgs& a, int view, int b, const FaceInfo<kTex, kShaded>& I, int x,
                                          int y, FaceSums<kTex, kShaded>& S, float* sh) {
  const long long HW = (long long)a.H * a.W, i = (long long)view * HW + (long long)y * a.W + x;
  const float px = (float)x + 0.5f, py = (float)y + 0.5f;
  const float* E = a.ext + (size_t)view * 12;
  const float* K = a.intr + (size_t)view * 9;
  const float wa = a.bary[2 * i], wb = a.bary[2 * i + 1];
  const float w[3] = {wa, wb, 1.f - wa - wb};
  const f3 g = ld3(a.g_render + 3 * i);
  f3 n = mk3(0.f, 0.f, 0.f), pn = n;
  float pl = 1.f;
  bool flipped = false;
  const float* shc = kShaded ? a.sh + (size_t)view * 27 : nullptr;
  if (kTex || kShaded) {
    pn = mk3(w[0] * I.vn[0].x + w[1] * I.vn[1].x + w[2] * I.vn[2].x, w[0] * I.vn[0].y + w[1] * I.vn[1].y + w[2] * I.vn[2].y,
             w[0] * I.vn[0].z + w[1] * I.vn[1].z + w[2] * I.vn[2].z);
    pl = sqrtf(dot(pn, pn));
    n = mk3(pn.x / pl, pn.y / pl, pn.z / pl);
    if (dot(n, world_ray_dir(E, K, px, py)) > 0.f) { n = -n; flipped = true; }
  }
  f3 light = mk3(1.f, 1.f, 1.f);
  if (kShaded) light = sh_shade(mk3(1.f, 1.f, 1.f), n, shc);
  const f3 ga = mk3(g.x * light.x, g.y * light.y, g.z * light.z);
  f3 alb = mk3(0.f, 0.f, 0.f);
  float gw[3];
  if (!kTex) {
    alb = I.col[0] * w[0] + I.col[1] * w[1] + I.col[2] * w[2];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      S.gc[k] = S.gc[k] + ga * w[k];
      gw[k] = dot(ga, I.col[k]);
    }
  } else {
    float U0 = (I.t6[0] * w[0] + I.t6[2] * w[1] + I.t6[4] * w[2]) * (float)a.TW;
    float V0 = ((1.f - I.t6[1]) * w[0] + (1.f - I.t6[3]) * w[1] + (1.f - I.t6[5]) * w[2]) * (float)a.TH;
    U0 = fminf(fmaxf(U0, 0.f), (float)(a.TW - 1));
    V0 = fminf(fmaxf(V0, 0.f), (float)(a.TH - 1));
    const float* tx = a.tex + (size_t)b * a.TH * a.TW * 3;
    if (kShaded) {
      const float LU = (float)(int)(U0 - 0.5f) + 0.5f, HU = LU + 1.f;
      const float LV = (float)(int)(V0 - 0.5f) + 0.5f, HV = LV + 1.f;
      auto at = [&](float uu, float vv) { return ld3(tx + ((size_t)(int)vv * a.TW + (int)uu) * 3); };
      alb = (at(LU, LV) * (U0 - LU) + at(HU, LV) * (HU - U0)) * (V0 - LV) +
            (at(LU, HV) * (U0 - LU) + at(HU, HV) * (HU - U0)) * (HV - V0);
    }
    if (!flipped && a.g_tex) {
      float* gt = a.g_tex + (size_t)b * a.TH * a.TW * 3 + ((size_t)(int)(V0 - 0.5f) * a.TW + (int)(U0 - 0.5f)) * 3;
      atomicAdd(gt, ga.x); atomicAdd(gt + 1, ga.y); atomicAdd(gt + 2, ga.z);
    }
    f3 du, dv;
    image_gradient(tx, U0, V0, a.TW, a.TH, a.tex_fs, du, dv);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const float su = I.t6[2 * k] * (float)a.TW, sv = (1.f - I.t6[2 * k + 1]) * (float)a.TH;
      gw[k] = ga.x * (du.x * su + dv.x * sv) + ga.y * (du.y * su + dv.y * sv) + ga.z * (du.z * su + dv.z * sv);
    }
  }
  if (kShaded) {
    const float basis[9] = {1.f, n.y, n.z, n.x, n.x * n.y, n.z * n.y, 3.f * n.z * n.z - 1.f, n.x * n.z, n.x * n.x - n.y * n.y};
    const float gc[3] = {g.x * alb.x, g.y * alb.y, g.z * alb.z};
    f3 gn = mk3(0.f, 0.f, 0.f);
#pragma unroll
    for (int ch = 0; ch < 3; ++ch) {
#pragma unroll
      for (int k = 0; k < 9; ++k) sh[(9 * ch + k) * kB] += gc[ch] * basis[k];
      const float* s = shc + 9 * ch;
      const f3 Jn = mk3(s[3] + s[4] * n.y + s[7] * n.z + s[8] * 2.f * n.x,
                        s[1] + s[4] * n.x + s[5] * n.z + s[8] * -2.f * n.y,
                        s[2] + s[5] * n.y + s[6] * 6.f * n.z + s[7] * n.x);
      gn = gn + Jn * gc[ch];
    }
    const float sg = flipped ? -1.f : 1.f;
    const f3 nn = mk3(pn.x / pl, pn.y / pl, pn.z / pl);
    const float dg = sg * dot(gn, nn);
    const f3 gun = mk3((sg * gn.x - nn.x * dg) / pl, (sg * gn.y - nn.y * dg) / pl, (sg * gn.z - nn.z * dg) / pl);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      gw[k] += dot(gun, I.vn[k]);
      S.gn[k] = S.gn[k] + gun * w[k];
    }
  }
  // through the barycentrics to the corners' image positions and 1/z
  // (bary_vjp), and from there to their homogeneous image points
  float e[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const f4 pj = I.p[k == 2 ? 0 : k + 1], pk = I.p[k == 0 ? 2 : k - 1];
    e[k] = (pk.x - pj.x) * (py - pj.y) - (pk.y - pj.y) * (px - pj.x);
  }
  const float q0 = e[0] * I.p[0].w, q1 = e[1] * I.p[1].w, q2 = e[2] * I.p[2].w;
  const float Q = q0 + q1 + q2;
  const float b0 = q0 / Q, b1 = q1 / Q;
  const float g0 = gw[0] - gw[2], g1 = gw[1] - gw[2];
  const float s = g0 * b0 + g1 * b1;
  const float gq[3] = {(g0 - s) / Q, (g1 - s) / Q, (0.f - s) / Q};
  float tu[3] = {0.f, 0.f, 0.f}, tv[3] = {0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const int jj = k == 2 ? 0 : k + 1, kk = k == 0 ? 2 : k - 1;
    const f4 pj = I.p[jj], pk = I.p[kk];
    const float ge = gq[k] * I.p[k].w;
    tu[jj] += ge * (pk.y - py);
    tv[jj] += ge * (px - pk.x);
    tu[kk] += ge * (py - pj.y);
    tv[kk] += ge * (pj.x - px);
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const f4 p = I.p[k];
    S.gh[k] = S.gh[k] + mk3(tu[k] * p.w, tv[k] * p.w, -((tu[k] * p.x + tv[k] * p.y) + gq[k] * e[k] * p.w) * p.w);
  }
  if (a.target) {
    f3 du, dv;
    image_gradient(a.target + (size_t)view * HW * 3, (float)x, (float)y, a.W, a.H, a.img_fs, du, dv);
    const float gu = -dot(g, du), gvv = -dot(g, dv);
    // the fragment's homogeneous image point: the projection is linear, so it
    // is the same blend of the corners' (a gathered face's corners are all in
    // front of the camera)
    const float z0 = I.p[0].z * w[0], z1 = I.p[1].z * w[1], z2 = I.p[2].z * w[2];
    const float hx = I.p[0].x * z0 + I.p[1].x * z1 + I.p[2].x * z2;
    const float hy = I.p[0].y * z0 + I.p[1].y * z1 + I.p[2].y * z2;
    const float hz = z0 + z1 + z2;
    if (fabsf(hz) > 0.0001f) {
      const f3 gf = mk3(gu / hz, gvv / hz, -(gu * hx + gvv * hy) / (hz * hz));
#pragma unroll
      for (int k = 0; k < 3; ++k) S.gh[k] = S.gh[k] + gf * w[k];
    }
  }
}

// The face's record: its corners' image-space sums taken to world space once.
template <bool kTex, bool kShaded>
__device__ __forceinline__ void face_record(const BwdArgs& a, int view, const FaceSums<kTex, kShaded>& S, float* r) {
  const float* E = a.ext + (size_t)view * 12;
  const float* K = a.intr + (size_t)view * 9;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const f3 h = S.gh[i];
    const float gx = K[0] * h.x + K[3] * h.y + K[6] * h.z;
    const float gy = K[1] * h.x + K[4] * h.y + K[7] * h.z;
    const float gz = K[2] * h.x + K[5] * h.y + K[8] * h.z;
    r[3 * i] = E[0] * gx + E[4] * gy + E[8] * gz;
    r[3 * i + 1] = E[1] * gx + E[5] * gy + E[9] * gz;
    r[3 * i + 2] = E[2] * gx + E[6] * gy + E[10] * gz;
    if (!kTex && a.rec_col) {
      float* c = r + a.rec_col + 3 * i;
      c[0] = S.gc[i].x; c[1] = S.gc[i].y; c[2] = S.gc[i].z;
    }
    if (kShaded) {
      float* c = r + a.rec_vn + 3 * i;
      c[0] = S.gn[i].x; c[1] = S.gn[i].y; c[2] = S.gn[i].z;
    }
  }
}

// Sums of every member over a face's lanes, or the wavefront's, in all of them.
template <bool kTex, bool kShaded>
__device__ __forceinline__ void lanes_total(FaceSums<kTex, kShaded>& S, bool wavefront) {
  static_assert(kFaceLanes == 4, "a quad");
  auto sum = [=](float& v) {
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, false));  // 1 apart
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xf, 0xf, false));  // 2 apart
    if (wavefront)
#pragma unroll
      for (int o = 4; o < 64; o <<= 1) v += __shfl_xor(v, o, 64);
  };
  auto f3sum = [&](f3& v) { sum(v.x); sum(v.y); sum(v.z); };
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    f3sum(S.gh[i]);
    if (!kTex) f3sum(S.gc[i]);
    if (kShaded) f3sum(S.gn[i]);
  }
}

// What one lane, four or a wavefront of them do for a face: pixel j of a lane is
// pixel first + stride * j of the face's box.  The box is searched first (its
// face ids, four loads at a time, into a bit a pixel), so that the wavefront
// runs the long part of the code as often as its lane with the most pixels of
// its own, not as often as the largest box.
template <bool kTex, bool kShaded>
struct FaceWalk {
  FaceInfo<kTex, kShaded> I;
  float inv_nx;
  __device__ __forceinline__ void load(const BwdArgs& a, int view, int b, int f) {
    I.load(a, view, b, f);
    inv_nx = __builtin_amdgcn_rcpf((float)I.box.nx);
  }
  // k / nx for k < kGatherBox: (k + 1/2) / nx is at least 1 / (2 nx) away from a whole number
  __device__ __forceinline__ int row_of(int k) const { return (int)(((float)k + 0.5f) * inv_nx); }
  // the lane's pixels among the box's first n that are the face's, a bit each
  template <int stride>
  __device__ __forceinline__ unsigned long long search(const BwdArgs& a, int view, int f, int n, int first) const {
    const int* ids = a.face + (size_t)view * a.H * a.W;
    unsigned long long mine = 0;
    for (int j0 = 0; j0 * stride + first < n; j0 += 4) {
      int id[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int k = min((j0 + j) * stride + first, n - 1), y = row_of(k);
        id[j] = ids[(size_t)(I.box.y0 + y) * a.W + I.box.x0 + k - y * I.box.nx];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
        mine |= (unsigned long long)(id[j] == f && (j0 + j) * stride + first < n) << (j0 + j);
    }
    return mine;
  }
  template <int stride>
  __device__ __forceinline__ void add(const BwdArgs& a, int view, int b, unsigned long long mine, int first,
                                      FaceSums<kTex, kShaded>& S, float* sh) const {
    while (mine) {
      const int k = (__ffsll(mine) - 1) * stride + first, y = row_of(k);
      mine &= mine - 1;
      add_pixel<kTex, kShaded>(a, view, b, I, I.box.x0 + k - y * I.box.nx, I.box.y0 + y, S, sh);
    }
  }
  __device__ __forceinline__ uint2 packed_box(bool any) const {
    return make_uint2((unsigned)I.box.x0 | (unsigned)I.box.y0 << 16,
                      (unsigned)I.box.nx | (unsigned)I.box.ny << 10 | (any ? 1u << 20 : 0u));
  }
};

// The workgroup's SH gradient: its lanes' sums (27, kB floats apart), then one
// atomic a value.
struct ShLds { float total[32], lane[27 * kB]; };
__device__ __forceinline__ void sh_clear(ShLds& L) {
  if (threadIdx.x < 32) L.total[threadIdx.x] = 0.f;
#pragma unroll
  for (int k = 0; k < 27; ++k) L.lane[k * kB + threadIdx.x] = 0.f;
  __syncthreads();
}
__device__ __forceinline__ void sh_flush(ShLds& L, const BwdArgs& a, int view, bool wave_has) {
  if (wave_has) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = 8 * r + k < 27 ? L.lane[min(8 * r + k, 26) * kB + threadIdx.x] : 0.f;
      const float t = wave_sum8(v);
      if ((threadIdx.x & 63) < 8) atomicAdd(&L.total[8 * r + (threadIdx.x & 63)], t);
    }
  }
  __syncthreads();
  if (threadIdx.x < 27 && L.total[threadIdx.x] != 0.f)
    atomicAdd(a.g_sh + (size_t)view * 27 + threadIdx.x, L.total[threadIdx.x]);
}

// kFaceLanes lanes per face, one view per workgroup row; the faces that this
// would take long for go onto their view's list.
// Pixel-parallel with segmented scans and up to 27 atomics a run, this part
// took 570 us for 25k vertices, 4 views of 1024 x 1024, shaded vertex colours
// (903 us textured, 50k vertices, 8 views of 1285 x 940).  With every box up
// to 256 pixels here, the lanes of the largest faces were the last of the
// launch (183 us, and 87 for the pixels left over; textured 413 and 140); now
// 97 here, 55 in face_wide_kernel, 31 in the vertex gather and 20 for the
// pixels left over (289, 93, 51 and 22; with at most 3 pixels a lane the two
// kernels take 81 + 102, with 12 118 + 53).  What bounds it is the latency of a pixel's loads at three
// wavefronts a SIMD; the sums of a shaded face are 27 registers, and the 27
// of the SH gradient are in LDS (with them in registers two wavefronts fit).
template <bool kTex, bool kShaded>
__global__ __launch_bounds__(kB) __attribute__((amdgpu_waves_per_eu(3))) void face_gather_kernel(BwdArgs a) {
  __shared__ std::conditional_t<kShaded, ShLds, char> s_sh;
  __shared__ unsigned int s_n, s_at;
  const int view = blockIdx.y, b = view / a.C, lane = threadIdx.x & 63, sub = threadIdx.x % kFaceLanes;
  const int f = (blockIdx.x * kB + threadIdx.x) / kFaceLanes;
  const bool in = f < a.F;
  if constexpr (kShaded) sh_clear(s_sh);
  if (threadIdx.x == 0) s_n = 0;
  FaceWalk<kTex, kShaded> w;
  w.load(a, view, b, in ? f : a.F - 1);
  const int n = in ? w.I.box.nx * w.I.box.ny : 0;
  static_assert(kLaneBox <= 64 * kFaceLanes, "a bit a pixel");
  unsigned long long mine = w.template search<kFaceLanes>(a, view, f, n > kLaneBox ? 0 : n, sub);
  auto of_face = [&](bool c) { return (__ballot(c) >> (lane - sub) & ((1u << kFaceLanes) - 1u)) != 0; };
  const bool wide = of_face(n > kLaneBox || __popcll(mine) > kLaneHits);
  if (wide) mine = 0;
  const bool any = of_face(mine != 0), wave_any = __ballot(mine != 0) != 0;
  const size_t at = (size_t)view * a.F + f;
  if (wave_any) {
    FaceSums<kTex, kShaded> S;
    S.clear();
    float* sh = nullptr;
    if constexpr (kShaded) sh = s_sh.lane + threadIdx.x;
    w.template add<kFaceLanes>(a, view, b, mine, sub, S, sh);
    lanes_total<kTex, kShaded>(S, false);
    if (sub == 0 && any) face_record<kTex, kShaded>(a, view, S, a.rec + at * a.rec_n);
  }
  if (sub == 0 && in) a.box[at] = w.packed_box(any);
  __syncthreads();
  unsigned int slot = 0;
  if (sub == 0 && wide) slot = atomicAdd(&s_n, 1u);
  __syncthreads();
  if (threadIdx.x == 0 && s_n) s_at = atomicAdd(a.wide_n + view * kWideStride, s_n);
  __syncthreads();
  if (sub == 0 && wide) a.wide[(size_t)view * a.F + s_at + slot] = (unsigned int)f;
  if constexpr (kShaded)
    if (a.g_sh) sh_flush(s_sh, a, view, wave_any);
}

// A wavefront per listed face of the view (a workgroup row).  (In the gather's
// own wavefronts, one large face after the other, this took 300 us: they lie
// together.)
template <bool kTex, bool kShaded>
__global__ __launch_bounds__(kB) __attribute__((amdgpu_waves_per_eu(kTex ? 3 : 2))) void face_wide_kernel(BwdArgs a) {
  __shared__ std::conditional_t<kShaded, ShLds, char> s_sh;
  static_assert(kGatherBox <= 64 * 64, "a bit a pixel");
  const int view = blockIdx.y, b = view / a.C, lane = threadIdx.x & 63;
  const unsigned int n = a.wide_n[view * kWideStride];
  if ((blockIdx.x * kB) >> 6 >= n) return;
  if constexpr (kShaded) sh_clear(s_sh);
  bool wave_any = false;
  for (unsigned int q = (blockIdx.x * kB + threadIdx.x) >> 6; q < n; q += gridDim.x * (kB / 64)) {
    const int f = __builtin_amdgcn_readfirstlane((int)a.wide[(size_t)view * a.F + q]);
    FaceWalk<kTex, kShaded> w;
    w.load(a, view, b, f);
    const unsigned long long mine = w.template search<64>(a, view, f, w.I.box.nx * w.I.box.ny, lane);
    if (!__ballot(mine != 0)) continue;  // its box says that there is no record
    wave_any = true;
    FaceSums<kTex, kShaded> S;
    S.clear();
    float* sh = nullptr;
    if constexpr (kShaded) sh = s_sh.lane + threadIdx.x;
    w.template add<64>(a, view, b, mine, lane, S, sh);
    lanes_total<kTex, kShaded>(S, true);
    const size_t at = (size_t)view * a.F + f;
    if (lane == 0) {
      face_record<kTex, kShaded>(a, view, S, a.rec + at * a.rec_n);
      a.box[at] = w.packed_box(true);
    }
  }
  if constexpr (kShaded)
    if (a.g_sh) sh_flush(s_sh, a, view, wave_any);
}

constexpr int kVertexLanes = 8;
constexpr int kManyFaces = 32;  // vertices with more faces are a whole wavefront's

// Sum over a group of 8 lanes, in all of them.
__device__ __forceinline__ float sum8(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, false));   // 1 apart
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xf, 0xf, false));   // 2 apart
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xf, 0xf, false));  // half mirror
  return v;
}

// Calls add(face id) for the vertex's faces, each once (a face that lists the
// vertex twice stands twice in its list, one after the other), and stores the
// sums: eight lanes a vertex, or the wavefront for vertices with many faces
// (the poles of a mesh; eight lanes walk 130 of them after the launch is done).
template <int kNV, class Add, class Store>
__device__ __forceinline__ void for_vertex_faces(const int* off, const int* lst, int N, int B, Add add, Store store) {
  const long long i = ((long long)blockIdx.x * kB + threadIdx.x) / kVertexLanes;
  const int sub = threadIdx.x % kVertexLanes, lane = threadIdx.x & 63;
  const bool in = i < (long long)B * N;
  const int b = in ? (int)(i / N) : 0, v = in ? (int)(i - (long long)b * N) : 0;
  const int k0 = in ? off[v] : 0, k1 = in ? off[v + 1] : 0;
  float s[kNV];
#pragma unroll
  for (int j = 0; j < kNV; ++j) s[j] = 0.f;
  const bool many = k1 - k0 > kManyFaces;
  if (!many)
    for (int k = k0 + sub; k < k1; k += kVertexLanes) {
      const int f = lst[k];
      if (k == k0 || lst[k - 1] != f) add(b, v, f, s);
    }
#pragma unroll
  for (int j = 0; j < kNV; ++j) s[j] = sum8(s[j]);
  if (in && !many && sub == 0) store(i, s);
  for (unsigned long long todo = __ballot(many && sub == 0); todo; todo &= todo - 1) {
    const int src = __ffsll(todo) - 1;
    const int c0 = __builtin_amdgcn_readlane(k0, src), c1 = __builtin_amdgcn_readlane(k1, src);
    const int cb = __builtin_amdgcn_readlane(b, src), cv = __builtin_amdgcn_readlane(v, src);
    float t[kNV];
#pragma unroll
    for (int j = 0; j < kNV; ++j) t[j] = 0.f;
    for (int k = c0 + lane; k < c1; k += 64) {
      const int f = lst[k];
      if (k == c0 || lst[k - 1] != f) add(cb, cv, f, t);
    }
#pragma unroll
    for (int j = 0; j < kNV; ++j) t[j] = wave_sum(t[j]);
    if (lane == src) store(i, t);
  }
}

// Pixels that no face's box took, four a lane: their groups into a.rest.
__device__ __forceinline__ void find_rest(const BwdArgs& a, unsigned int block) {
  __shared__ unsigned int s_any[4];  // of the workgroup's groups of kB pixels
  const long long HW = (long long)a.H * a.W, total = (long long)a.B * a.C * HW;
  if (threadIdx.x < 4) s_any[threadIdx.x] = 0;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const long long i = ((long long)block * 4 + j) * kB + threadIdx.x;
    const int f = i < total ? a.face[i] : -1;
    if (f < 0) continue;
    const int view = (int)(i / HW), p = (int)(i - (long long)view * HW), y = p / a.W;
    if (!unpack_box(a.box[(size_t)view * a.F + f]).has(p - y * a.W, y)) s_any[j] = 1;
  }
  __syncthreads();
  if (threadIdx.x < 4 && s_any[threadIdx.x]) a.rest[atomicAdd(a.rest_n, 1u)] = block * 4 + threadIdx.x;
}

// dL/d(position, colour, normal) of every vertex: the records of its faces in
// all views.  The launch's other workgroups look for what is left.
__global__ __launch_bounds__(kB) void vertex_gather_kernel(BwdArgs a, unsigned vertex_blocks, const int* __restrict__ off,
                                                           const int* __restrict__ lst) {
  if (blockIdx.x >= vertex_blocks) {
    find_rest(a, blockIdx.x - vertex_blocks);
    return;
  }
  for_vertex_faces<9>(
      off, lst, a.N, a.B,
      [&](int b, int v, int f, float* s) {
        const int i0 = a.faces[3 * f], i1 = a.faces[3 * f + 1], i2 = a.faces[3 * f + 2];
        for (int c = 0; c < a.C; ++c) {
          const size_t at = ((size_t)b * a.C + c) * a.F + f;
          if (!(a.box[at].y >> 20)) continue;
          const float* r = a.rec + at * a.rec_n;
          auto corner = [&](int q) {
#pragma unroll
            for (int j = 0; j < 3; ++j) {
              s[j] += r[3 * q + j];
              if (a.rec_col) s[3 + j] += r[a.rec_col + 3 * q + j];
              if (a.rec_vn) s[6 + j] += r[a.rec_vn + 3 * q + j];
            }
          };
          if (i0 == v) corner(0);
          if (i1 == v) corner(1);
          if (i2 == v) corner(2);
        }
      },
      [&](long long i, const float* s) {
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          a.g_vpos[3 * i + j] = s[j];
          a.g_vcol[3 * i + j] = s[3 + j];
          if (a.g_vn) a.g_vn[3 * i + j] = s[6 + j];
        }
      });
}

// n_v = sum over the faces around v (one entry per corner) of N_f =
// (v1 - v0) x (v2 - v0).  With G_f = sum of dL/dn over the three corners of f,
// dL/dv0 = (e1 - e2) x G_f, dL/dv1 = e2 x G_f, dL/dv2 = G_f x e1 (e1 = v1 - v0,
// e2 = v2 - v0); v takes the terms of the corners it occupies.  A lane per
// vertex took 67 us for 50k vertices (a chain of list, face and corner loads
// for each face); eight lanes 9.
__global__ __launch_bounds__(kB) void normal_grad_kernel(const float* __restrict__ vpos, const int* __restrict__ faces,
                                                         const int* __restrict__ off, const int* __restrict__ lst,
                                                         const float* __restrict__ g_vn, int N, int B,
                                                         float* __restrict__ g_vpos) {
  for_vertex_faces<3>(
      off, lst, N, B,
      [&](int b, int v, int f, float* s) {
        const float* vp = vpos + (size_t)b * N * 3;
        const float* gv = g_vn + (size_t)b * N * 3;
        const int i0 = faces[3 * f], i1 = faces[3 * f + 1], i2 = faces[3 * f + 2];
        const f3 G = ld3(gv + 3 * i0) + ld3(gv + 3 * i1) + ld3(gv + 3 * i2);
        const f3 p0 = ld3(vp + 3 * i0);
        const f3 e1 = ld3(vp + 3 * i1) - p0, e2 = ld3(vp + 3 * i2) - p0;
        f3 t = mk3(0.f, 0.f, 0.f);
        if (i0 == v) t = t + cross(e1 - e2, G);
        if (i1 == v) t = t + cross(e2, G);
        if (i2 == v) t = t + cross(G, e1);
        s[0] += t.x; s[1] += t.y; s[2] += t.z;
      },
      [&](long long i, const float* s) {
#pragma unroll
        for (int j = 0; j < 3; ++j) g_vpos[3 * i + j] += s[j];
      });
}

// Clears two arrays and some counters.
__global__ __launch_bounds__(kB) void clear2_kernel(float* __restrict__ p, long long n, float* __restrict__ q,
                                                    long long m, unsigned int* __restrict__ counters,
                                                    long long c) {
  const long long i = (long long)blockIdx.x * kB + threadIdx.x;
  if (i < n) p[i] = 0.f;
  else if (i < n + m) q[i - n] = 0.f;
  else if (i < n + m + c) counters[i - n - m] = 0u;
}

size_t vn_floats(const dcx_topo* topo, const dcx_raster_cfg* cfg, int B) {
  return cfg->shading_mode == DCX_SHADING_SHADED ? 3 * (size_t)B * topo->N : 0;
}
int record_floats(const dcx_raster_cfg* cfg) {
  return 9 + (cfg->albedo_mode == ALB_VERTEX_COLOR ? 9 : 0) + (cfg->shading_mode == DCX_SHADING_SHADED ? 9 : 0);
}

}  // namespace
}  // namespace dcx

using namespace dcx;

extern "C" size_t dcx_render_bwd_workspace_size(const dcx_topo* topo, const dcx_raster_cfg* cfg, int B) {
  if (!topo || !cfg || B <= 0) return 0;
  const size_t faces = (size_t)B * cfg->num_cameras * topo->F;
  const size_t pixels = (size_t)B * cfg->num_cameras * cfg->height * cfg->width;
  return sizeof(uint2) * faces + sizeof(float) * (vn_floats(topo, cfg, B) + faces * record_floats(cfg)) +
         sizeof(unsigned int) * ((pixels + kB - 1) / kB + 1 + kWideStride * (size_t)B * cfg->num_cameras + faces);
}

extern "C" dcx_status dcx_render_bwd(const dcx_topo* topo, const dcx_raster_cfg* cfg, int B,
                                     const float* render_grad, const float* vertex_pos,
                                     const float* vertex_color, const float* texture, int tex_h,
                                     int tex_w, const float* sh_coeff, const float* target_image,
                                     const float* vertex_normal, const float* barycentric,
                                     const int32_t* face, const float* extrinsics,
                                     const float* intrinsics, float* vertex_pos_grad,
                                     float* vertex_color_grad, float* texture_grad,
                                     float* sh_coeff_grad, void* workspace, size_t workspace_bytes,
                                     void* stream) {
  dcx_status st = validate_cfg(topo, cfg, B);
  if (st) return st;
  const int alb = cfg->albedo_mode;
  const bool shaded = cfg->shading_mode == DCX_SHADING_SHADED;
  DCX_REQUIRE(alb == ALB_VERTEX_COLOR || alb == ALB_TEXTURED || alb == ALB_FOREGROUND,
              "dcx_render_bwd: albedo mode %d has no gradient (the reference returns zeros)", alb);
  DCX_REQUIRE(render_grad && vertex_pos && barycentric && face && extrinsics && intrinsics &&
                  vertex_pos_grad && vertex_color_grad,
              "dcx_render_bwd: null input/output");
  DCX_REQUIRE(alb == ALB_TEXTURED || vertex_color, "dcx_render_bwd: vertex_color required");
  DCX_REQUIRE(alb != ALB_TEXTURED || (texture && topo->texcoords && tex_h > 0 && tex_w > 0),
              "dcx_render_bwd: textured mode needs texture + texcoords");
  DCX_REQUIRE(!(shaded || alb == ALB_TEXTURED) || vertex_normal, "dcx_render_bwd: vertex_normal required");
  DCX_REQUIRE(!shaded || sh_coeff, "dcx_render_bwd: shaded mode needs sh_coeff");
  const size_t vn = vn_floats(topo, cfg, B);
  DCX_REQUIRE(!shaded || (workspace && workspace_bytes >= sizeof(float) * vn),
              "dcx_render_bwd: shaded mode needs a workspace of at least %zu bytes", sizeof(float) * vn);
  hipStream_t s = as_stream(stream);
  const int N = topo->N, C = cfg->num_cameras;
  // the gather form wherever its records fit the workspace
  const bool gather = workspace && workspace_bytes >= dcx_render_bwd_workspace_size(topo, cfg, B) &&
                      ((uintptr_t)workspace & 7) == 0 && (long long)B * C <= 65535;  // (a grid row per view)
  const long long tex_n = texture_grad && tex_h > 0 && tex_w > 0 ? 3ll * B * tex_h * tex_w : 0;
  const long long sh_n = sh_coeff_grad ? 27ll * B * C : 0;
  BwdArgs a{};
  a.B = B; a.C = C; a.N = N; a.F = topo->F; a.H = cfg->height; a.W = cfg->width;
  a.albedo = alb; a.shaded = shaded ? 1 : 0; a.TH = tex_h; a.TW = tex_w;
  a.img_fs = cfg->image_filter_size; a.tex_fs = cfg->texture_filter_size;
  a.faces = topo->faces; a.tc = topo->texcoords;
  a.g_render = render_grad; a.vpos = vertex_pos; a.vcol = vertex_color; a.tex = texture; a.sh = sh_coeff;
  a.target = target_image; a.vnormal = vertex_normal; a.bary = barycentric; a.face = face;
  a.ext = extrinsics; a.intr = intrinsics;
  a.g_vpos = vertex_pos_grad; a.g_vcol = vertex_color_grad; a.g_tex = texture_grad;
  a.g_sh = shaded ? sh_coeff_grad : nullptr;
  // workspace: [boxes] normals [records, groups left over]
  const size_t faces = (size_t)B * C * topo->F;
  float* ws = (float*)workspace + (gather ? 2 * faces : 0);
  a.g_vn = shaded ? ws : nullptr;
  const unsigned pixels = ceil_div((long long)B * C * cfg->height * cfg->width, kB);
  auto clear = [&](float* p, long long n, float* q, long long m, unsigned int* counters, long long c) {
    if (n + m + c)
      hipLaunchKernelGGL(clear2_kernel, dim3(ceil_div(n + m + c, kB)), dim3(kB), 0, s, p, n, q, m, counters, c);
  };
  const unsigned vertices = ceil_div((long long)B * N * kVertexLanes, kB);
  if (gather) {
    a.box = (uint2*)workspace;
    a.rec = ws + vn;
    a.rec_n = record_floats(cfg);
    a.rec_col = alb == ALB_VERTEX_COLOR ? 9 : 0;
    a.rec_vn = shaded ? a.rec_n - 9 : 0;
    a.rest_n = (unsigned int*)(a.rec + faces * a.rec_n);
    a.wide_n = a.rest_n + 1;
    a.wide = a.wide_n + kWideStride * (size_t)B * C;
    a.rest = a.wide + faces;
    clear(texture_grad, tex_n, sh_coeff_grad, sh_n, a.rest_n, 1 + kWideStride * (long long)B * C);
    const unsigned views = (unsigned)(B * C);
    // as many workgroups as can be resident, and at least a few for each view's list
    const unsigned wide = views < 192 ? 768 / views : 4;
    auto launch = [&](auto kernel, auto wide_kernel) {
      hipLaunchKernelGGL(kernel, dim3(ceil_div(topo->F, kB / kFaceLanes), views), dim3(kB), 0, s, a);
      hipLaunchKernelGGL(wide_kernel, dim3(wide, views), dim3(kB), 0, s, a);
    };
    const bool tex = alb == ALB_TEXTURED;
    if (tex && shaded) launch(face_gather_kernel<true, true>, face_wide_kernel<true, true>);
    else if (tex) launch(face_gather_kernel<true, false>, face_wide_kernel<true, false>);
    else if (shaded) launch(face_gather_kernel<false, true>, face_wide_kernel<false, true>);
    else launch(face_gather_kernel<false, false>, face_wide_kernel<false, false>);
    hipLaunchKernelGGL(vertex_gather_kernel, dim3(vertices + ceil_div(pixels, 4)), dim3(kB), 0, s, a, vertices,
                       topo->vf_off, topo->vf_list);
    hipLaunchKernelGGL(render_bwd_kernel<true>, dim3(pixels < 1024 ? pixels : 1024), dim3(kB), 0, s, a);
  } else {
    clear(texture_grad, tex_n, sh_coeff_grad, sh_n, nullptr, 0);
    clear(vertex_pos_grad, 3ll * B * N, vertex_color_grad, 3ll * B * N, nullptr, 0);
    clear(ws, (long long)vn, nullptr, 0, nullptr, 0);
    hipLaunchKernelGGL(render_bwd_kernel<false>, dim3(pixels), dim3(kB), 0, s, a);
  }
  if (shaded)
    hipLaunchKernelGGL(normal_grad_kernel, dim3(vertices), dim3(kB), 0, s, vertex_pos, topo->faces, topo->vf_off,
                       topo->vf_list, ws, N, B, vertex_pos_grad);
  return check_launch("dcx_render_bwd");
}
