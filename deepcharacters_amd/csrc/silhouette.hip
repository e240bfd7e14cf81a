// Multi-view silhouette loss (MultiViewSilhouetteLossGpu / ...Grad), camera
// projection (CameraProjectionGpu / ...Grad) and projected-mesh boundary
// flags (ProjectedMeshBoundaryGpu) on gfx950.
//
// The data->model term searches, for each DT boundary pixel, the nearest
// boundary point within 30*scale.  DCX_SIL_BRUTE scans every point as the
// reference does (MultiViewSilhouetteLossGPUOp.cu:195-212).  DCX_SIL_BINNED
// first buckets the view's boundary points into a uniform grid of cells an
// eighth of the search radius wide.  A wavefront takes a boundary pixel and
// scans the 3x3 cells around it, then, only if something beyond them could
// still be nearer, all cells within the best distance so far; it evaluates
// the same float distance and keeps the lexicographic minimum of (distance,
// index), so both paths return the same ids as the reference's strict-< scan
// (lowest index among equal distances).
#include "raster_internal.hpp"

namespace dcx {

namespace {

constexpr int kB = 256;

__device__ __forceinline__ float remap(int v) { return v >= 127 ? (float)((v - 127) * 2) : (float)v; }

struct SilArgs {
  int B, C, N, U, V;
  const float* pts;      // [B,C,N,2]
  const float* nrm;      // [B,C,N,2]
  const unsigned char* isb;  // [B,C,N]
  const unsigned char* dt;   // [B,C,U*V]
  const float* crops;    // [B,C,7]
  float* res;            // [B,C,N]
  float* res1;           // [B,C,U,V,2]
  float* dtg;            // [B,C,N,2]
  float* cid;            // [B,C,U,V]
};

constexpr int kCellsPerRadius = 8;
constexpr int kListStride = 32;  // a counter per 128-byte line

struct GridArgs {
  int gx, gy, cells_per_view;
  unsigned int* cnt;     // [views, cells]; null: no grid (brute force)
  unsigned int* off;     // [views, cells + 1], from each view's first item
  f4* items;             // [views, N] (u, v, point id) by cell
  unsigned int* list_n;  // [views, kListStride] boundary pixels found so far
  unsigned int* list;    // [views, U * V] their indices in the view
};

struct GridGeom {
  float ox, oy, cell;
};

__device__ __forceinline__ GridGeom grid_geom(const float* cr) {
  const float sc = cr[2];
  const float R = 30.f * sc * (1.f + 1.f / 1024.f);
  GridGeom g;
  g.cell = R / (float)kCellsPerRadius;
  g.ox = (0.f - cr[0]) * sc + cr[3] - 2.f * R;
  g.oy = (0.f - cr[1]) * sc + cr[4] - 2.f * R;
  return g;
}

__device__ __forceinline__ int cell_of(const GridGeom& g, const GridArgs& ga, float x, float y) {
  const float fx = floorf((x - g.ox) / g.cell), fy = floorf((y - g.oy) / g.cell);
  if (!(fx >= 0.f && fy >= 0.f && fx < (float)ga.gx && fy < (float)ga.gy)) return -1;
  return (int)fy * ga.gx + (int)fx;
}

// Model->data residual per (batch, camera, point): MultiViewSilhouetteLossGPUOp.cu:11-138.
// Boundary points are also counted into their grid cells.
__global__ __launch_bounds__(kB) void sil_point_kernel(SilArgs a, GridArgs g) {
  const long long i = (long long)blockIdx.x * kB + threadIdx.x;
  if (i >= (long long)a.B * a.C * a.N) return;
  const int view = (int)(i / a.N);
  const float* cr = a.crops + (size_t)view * 7;
  const float pu = a.pts[2 * i], pv = a.pts[2 * i + 1];
  if (g.cnt && a.isb[i]) {
    const int c = cell_of(grid_geom(cr), g, pu, pv);
    if (c >= 0) atomicAdd(g.cnt + (size_t)view * g.cells_per_view + c, 1u);
  }
  const bool in_view = pu - 2 > cr[3] && pu + 2 < cr[5] && pv - 2 > cr[4] && pv + 2 < cr[6];
  const float fx = (pu - cr[3]) / cr[2] + cr[0], fy = (pv - cr[4]) / cr[2] + cr[1];
  const int x = (int)fx, y = (int)fy;
  const bool inside_img = x - 1 >= 0 && x + 1 < a.U && y - 1 >= 0 && y + 1 < a.V;
  if (!in_view || !inside_img) {
    a.dtg[2 * i] = 0.f; a.dtg[2 * i + 1] = 0.f; a.res[i] = 0.f;
    return;
  }
  const unsigned char* img = a.dt + (size_t)view * a.U * a.V;
  auto at = [&](int xx, int yy) { return (int)img[(size_t)yy * a.U + xx]; };
  float dv = remap(at(x, y));
  const float f00 = remap(at(x - 1, y - 1)), f01 = remap(at(x, y - 1)), f02 = remap(at(x + 1, y - 1));
  const float f10 = remap(at(x - 1, y)), f12 = remap(at(x + 1, y));
  const float f20 = remap(at(x - 1, y + 1)), f21 = remap(at(x, y + 1)), f22 = remap(at(x + 1, y + 1));
  const float du = (1.f / 8.f) * ((-1.f) * f00 + (+1.f) * f02 + (-2.f) * f10 + (+2.f) * f12 + (-1.f) * f20 + (+1.f) * f22);
  const float dvv = (1.f / 8.f) * ((-1.f) * f00 + (-2.f) * f01 + (-1.f) * f02 + (+1.f) * f20 + (+2.f) * f21 + (+1.f) * f22);
  float nx = du, ny = dvv, ux = du, uy = dvv;
  const bool inside_fg = at(x, y) <= 127;
  const float nonvan = (du != 0.f || dvv != 0.f) ? 1.f : 0.f;
  const float bnd = a.isb[i] ? 1.f : 0.f;
  if (inside_fg) { nx = -nx; ny = -ny; }
  const float dotn = nx * a.nrm[2 * i] + ny * a.nrm[2 * i + 1];
  if (!(dotn >= 0.f) && inside_fg) { ux = -ux; uy = -uy; }
  dv *= bnd;
  dv *= nonvan;
  ux *= bnd; uy *= bnd;
  ux *= nonvan; uy *= nonvan;
  a.dtg[2 * i] = ux * (1.f / (255.f));
  a.dtg[2 * i + 1] = uy * (1.f / (255.f));
  a.res[i] = dv * (1.f / (255.f));
}

// Value 127 and at least four 127s in the 5x5 window (pixels outside the image
// not counted).  The window's loads are issued together, clamped to the image.
__device__ __forceinline__ bool is_dt_boundary(const unsigned char* img, int U, int V, int ui, int vi) {
  if (img[(size_t)vi * U + ui] != 127) return false;
  int counter = 0;
#pragma unroll
  for (int j = -2; j <= 2; ++j) {
    const int yy = vi + j;
    const unsigned char* row = img + (size_t)min(max(yy, 0), V - 1) * U;
#pragma unroll
    for (int i = -2; i <= 2; ++i) {
      const int xx = ui + i;
      const bool in = yy >= 0 && yy < V && xx >= 0 && xx < U;
      counter += (row[min(max(xx, 0), U - 1)] == 127) & in;
    }
  }
  return counter >= 4;
}

__device__ __forceinline__ void write_d2m(const SilArgs& a, size_t o, int view, int best, float ix, float iy, float sc) {
  if (best >= 0) {
    const size_t pi = (size_t)view * a.N + best;
    a.res1[2 * o] = (a.pts[2 * pi] - ix) / (30.f * sc);
    a.res1[2 * o + 1] = (a.pts[2 * pi + 1] - iy) / (30.f * sc);
    a.cid[o] = (float)best;
  } else {
    a.res1[2 * o] = 0.f; a.res1[2 * o + 1] = 0.f;
    a.cid[o] = -1.f;
  }
}

// Data->model per DT pixel, brute force over all points.
__global__ __launch_bounds__(kB) void sil_pixel_brute_kernel(SilArgs a) {
  const long long o = (long long)blockIdx.x * kB + threadIdx.x;
  const long long UV = (long long)a.U * a.V;
  if (o >= (long long)a.B * a.C * UV) return;
  const int view = (int)(o / UV);
  const int p = (int)(o - (long long)view * UV);
  const int ui = p % a.U, vi = p / a.U;
  const unsigned char* img = a.dt + (size_t)view * UV;
  int best = -1;
  float ix = 0.f, iy = 0.f, sc = 1.f;
  if (is_dt_boundary(img, a.U, a.V, ui, vi)) {
    const float* cr = a.crops + (size_t)view * 7;
    sc = cr[2];
    ix = ((float)ui - cr[0]) * sc + cr[3];
    iy = ((float)vi - cr[1]) * sc + cr[4];
    float bd = 30.f * sc;
    const float* pv = a.pts + (size_t)view * a.N * 2;
    const unsigned char* bv = a.isb + (size_t)view * a.N;
    for (int v = 0; v < a.N; ++v) {
      if (!bv[v]) continue;
      const float dx = pv[2 * v] - ix, dy = pv[2 * v + 1] - iy;
      const float d = sqrtf(dx * dx + dy * dy);
      if (d < bd) { bd = d; best = v; }
    }
  }
  write_d2m(a, o, view, best, ix, iy, sc);
}

__global__ __launch_bounds__(kB) void clear_u32_kernel(unsigned int* __restrict__ p, long long n) {
  const long long i = (long long)blockIdx.x * kB + threadIdx.x;
  if (i < n) p[i] = 0u;
}

// Cell offsets of one view per workgroup: every view has its own N item slots,
// so no scan crosses views.
__global__ __launch_bounds__(1024) void sil_grid_scan_kernel(GridArgs g) {
  __shared__ unsigned int s_wave[16];
  const unsigned int* cnt = g.cnt + (size_t)blockIdx.x * g.cells_per_view;
  unsigned int* off = g.off + (size_t)blockIdx.x * (g.cells_per_view + 1);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  unsigned int base = 0;
  for (int c0 = 0; c0 < g.cells_per_view; c0 += 4096) {
    const int c = c0 + 4 * (int)threadIdx.x;
    unsigned int v[4], sum = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) { v[k] = c + k < g.cells_per_view ? cnt[c + k] : 0u; sum += v[k]; }
    unsigned int inc = sum;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const unsigned int o = __shfl_up(inc, d, 64);
      if (lane >= d) inc += o;
    }
    if (lane == 63) s_wave[wid] = inc;
    __syncthreads();
    unsigned int before = base, total = 0;
    for (int w = 0; w < 16; ++w) {
      before += w < wid ? s_wave[w] : 0u;
      total += s_wave[w];
    }
    before += inc - sum;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (c + k < g.cells_per_view) off[c + k] = before;
      before += v[k];
    }
    base += total;
    __syncthreads();
  }
  if (threadIdx.x == 0) off[g.cells_per_view] = base;
}

// The boundary points into their cells' slots, last slot first (the counts are
// used up; the order in a cell changes no result).
__global__ __launch_bounds__(kB) void sil_grid_scatter_kernel(SilArgs a, GridArgs g) {
  const long long i = (long long)blockIdx.x * kB + threadIdx.x;
  if (i >= (long long)a.B * a.C * a.N || !a.isb[i]) return;
  const int view = (int)(i / a.N);
  const float x = a.pts[2 * i], y = a.pts[2 * i + 1];
  const int c = cell_of(grid_geom(a.crops + (size_t)view * 7), g, x, y);
  if (c < 0) return;
  const unsigned int slot = g.off[(size_t)view * (g.cells_per_view + 1) + c] +
                            atomicSub(g.cnt + (size_t)view * g.cells_per_view + c, 1u) - 1u;
  g.items[(size_t)view * a.N + slot] = mk4(x, y, __int_as_float((int)(i - (long long)view * a.N)), 0.f);
}

// Nearest of the points in the cells within `ring` of (cx, cy), by a whole
// wavefront: four cell rows at a time, 16 lanes a row (a row's cells are one
// range of items).  Each lane updates its own (bd, best).
__device__ __forceinline__ void scan_ring(const GridArgs& g, const unsigned int* off, const f4* items, int cx, int cy,
                                          int ring, float ix, float iy, float& bd, int& best) {
  const int lane = threadIdx.x & 63;
  const int x0 = max(cx - ring, 0), x1 = min(cx + ring, g.gx - 1);
  const int y1 = min(cy + ring, g.gy - 1);
  if (x0 > x1) return;
  for (int yy = max(cy - ring, 0) + (lane >> 4); yy <= y1; yy += 4) {
    const unsigned int end = off[yy * g.gx + x1 + 1];
    // two items in flight; past the end the last one again, which changes nothing
    for (unsigned int k = off[yy * g.gx + x0] + (lane & 15); k < end; k += 32) {
      const f4 it[2] = {items[k], items[min(k + 16, end - 1)]};
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const float dx = it[j].x - ix, dy = it[j].y - iy;
        const float d = sqrtf(dx * dx + dy * dy);
        const int v = __float_as_int(it[j].z);
        if (d < bd || (d == bd && best >= 0 && v < best)) { bd = d; best = v; }
      }
    }
  }
}

// Smallest (distance, index) over the wavefront, the result in every lane.
__device__ __forceinline__ void nearest_of_wave(float& bd, int& best) {
  const unsigned d = best >= 0 ? __float_as_uint(bd) : 0xffffffffu;  // distances are not negative: bit order
  const unsigned m = group_min<64>(d);
  best = (int)group_min<64>(d == m ? (unsigned)best : 0xffffffffu);
  if (m != 0xffffffffu) bd = __uint_as_float(m);
}

// The views lie along the grid's second dimension, which ends at kMaxViewRows;
// a launch for more of them goes on with the next kMaxViewRows in its workgroups.
constexpr int kMaxViewRows = 65535;

// The boundary pixels' indices into their view's list, one reservation per
// workgroup; every other pixel gets its empty result.
__device__ __forceinline__ void sil_pixel_list_view(const SilArgs& a, const GridArgs& g, int view) {
  __shared__ unsigned int s_n, s_at;
  const int UV = a.U * a.V, p = blockIdx.x * kB + threadIdx.x;
  if (threadIdx.x == 0) s_n = 0;
  __syncthreads();
  unsigned int mine = 0;
  bool found = false;
  if (p < UV) {
    found = is_dt_boundary(a.dt + (size_t)view * UV, a.U, a.V, p % a.U, p / a.U);
    if (found) mine = atomicAdd(&s_n, 1u);
    else write_d2m(a, (size_t)view * UV + p, view, -1, 0.f, 0.f, 1.f);
  }
  __syncthreads();
  if (threadIdx.x == 0 && s_n) s_at = atomicAdd(g.list_n + view * kListStride, s_n);
  __syncthreads();
  if (found) g.list[(size_t)view * UV + s_at + mine] = (unsigned int)p;
}
__global__ __launch_bounds__(kB) void sil_pixel_list_kernel(SilArgs a, GridArgs g) {
  for (int view = blockIdx.y; view < a.B * a.C; view += gridDim.y) {
    sil_pixel_list_view(a, g, view);
    __syncthreads();  // the counters are the next view's
  }
}

// A wavefront per listed pixel.  (Contour pixels cluster: dealt out by the
// workgroup that finds them, a few workgroups searched for a whole horizontal
// edge while the rest of the chip was done.)  16 views of 256 x 256 with 50k
// points each, an eighth of them on the boundary: 3.49 ms with a lane per
// pixel over cells as wide as the radius, 0.06 with the list; what is left is
// the chain list -> cell offsets -> points of each search.
constexpr int kSearchBlocks = 256;  // per view
__device__ __forceinline__ void sil_search_view(const SilArgs& a, const GridArgs& g, int view) {
  const int UV = a.U * a.V;
  const unsigned int n = g.list_n[view * kListStride];
  for (unsigned int q = (blockIdx.x * kB + threadIdx.x) >> 6; q < n; q += kSearchBlocks * (kB / 64)) {
    const int p = __builtin_amdgcn_readfirstlane((int)g.list[(size_t)view * UV + q]);
    const int ui = p % a.U, vi = p / a.U;
    const float* cr = a.crops + (size_t)view * 7;
    const float sc = cr[2];
    const float ix = ((float)ui - cr[0]) * sc + cr[3], iy = ((float)vi - cr[1]) * sc + cr[4];
    const GridGeom gg = grid_geom(cr);
    const int cx = (int)floorf((ix - gg.ox) / gg.cell), cy = (int)floorf((iy - gg.oy) / gg.cell);
    const unsigned int* off = g.off + (size_t)view * (g.cells_per_view + 1);
    const f4* items = g.items + (size_t)view * a.N;
    float bd = 30.f * sc;
    int best = -1;
    scan_ring(g, off, items, cx, cy, 1, ix, iy, bd, best);
    nearest_of_wave(bd, best);
    // a point outside the cells within r of the pixel's is farther than
    // r * step (the margin covers the rounding of positions to cells)
    const float step = gg.cell * (1.f - 1.f / 256.f);
    if (!(bd < step)) {
      scan_ring(g, off, items, cx, cy, min((int)(bd / step) + 1, kCellsPerRadius + 1), ix, iy, bd, best);
      nearest_of_wave(bd, best);
    }
    if ((threadIdx.x & 63) == 0) write_d2m(a, (size_t)view * UV + p, view, best, ix, iy, sc);
  }
}
__global__ __launch_bounds__(kB) void sil_search_kernel(SilArgs a, GridArgs g) {
  for (int view = blockIdx.y; view < a.B * a.C; view += gridDim.y) sil_search_view(a, g, view);
}

__global__ __launch_bounds__(kB) void sil_bwd_point_kernel(const float* __restrict__ g, const float* __restrict__ dtg,
                                                            long long n, float* __restrict__ out) {
  const long long i = (long long)blockIdx.x * kB + threadIdx.x;
  if (i >= n) return;
  out[2 * i] = dtg[2 * i] * g[i];
  out[2 * i + 1] = dtg[2 * i + 1] * g[i];
}

__global__ __launch_bounds__(kB) void sil_bwd_pixel_kernel(const float* __restrict__ g1, const float* __restrict__ cid,
                                                            const float* __restrict__ crops, int N, long long UV,
                                                            long long n, float* __restrict__ out) {
  const long long o = (long long)blockIdx.x * kB + threadIdx.x;
  if (o >= n) return;
  const int k = (int)cid[o];
  if (k < 0) return;
  const int view = (int)(o / UV);
  const float sc = crops[(size_t)view * 7 + 2];
  const size_t pi = (size_t)view * N + k;
  atomicAdd(out + 2 * pi, g1[2 * o] / (30.f * sc));
  atomicAdd(out + 2 * pi + 1, g1[2 * o + 1] / (30.f * sc));
}

// CameraProjectionGPUOp.cu:12-86.
__global__ __launch_bounds__(kB) void camproj_kernel(const float* __restrict__ P, const float* __restrict__ D,
                                                      const float* __restrict__ ext, const float* __restrict__ intr,
                                                      int B, int C, int N, int is_point, float* __restrict__ out) {
  const long long i = (long long)blockIdx.x * kB + threadIdx.x;
  if (i >= (long long)B * C * N) return;
  const int view = (int)(i / N), v = (int)(i - (long long)view * N);
  const int b = view / C;
  const float* E = ext + (size_t)view * 12;
  const float* K = intr + (size_t)view * 9;
  const f3 p = ld3(P + ((size_t)b * N + v) * 3);
  const f3 xc = mk3(E[0] * p.x + E[1] * p.y + E[2] * p.z + E[3], E[4] * p.x + E[5] * p.y + E[6] * p.z + E[7],
                    E[8] * p.x + E[9] * p.y + E[10] * p.z + E[11]);
  auto proj = [&](f3 x) {
    const float h0 = K[0] * x.x + K[1] * x.y + K[2] * x.z;
    const float h1 = K[3] * x.x + K[4] * x.y + K[5] * x.z;
    float h2 = K[6] * x.x + K[7] * x.y + K[8] * x.z;
    if (!(h2 > 0.0000001f)) h2 = 0.00001f;
    return mk2(h0 / h2, h1 / h2);
  };
  const f2 uv = proj(xc);
  if (is_point) {
    out[2 * i] = uv.x; out[2 * i + 1] = uv.y;
  } else {
    const f3 d = ld3(D + ((size_t)b * N + v) * 3);
    const f3 x2 = mk3(xc.x + (E[0] * d.x + E[1] * d.y + E[2] * d.z), xc.y + (E[4] * d.x + E[5] * d.y + E[6] * d.z),
                      xc.z + (E[8] * d.x + E[9] * d.y + E[10] * d.z));
    const f2 uv2 = proj(x2);
    const float du = uv2.x - uv.x, dv = uv2.y - uv.y;
    const float l = sqrtf(du * du + dv * dv);
    out[2 * i] = du / l; out[2 * i + 1] = dv / l;
  }
}

// CameraProjectionGPUOpGrad.cu:12-79: sum over cameras of (dI/dxc R)^T g.
__global__ __launch_bounds__(kB) void camproj_bwd_kernel(const float* __restrict__ g, const float* __restrict__ P,
                                                          const float* __restrict__ ext, const float* __restrict__ intr,
                                                          int B, int C, int N, float* __restrict__ out) {
  const long long i = (long long)blockIdx.x * kB + threadIdx.x;
  if (i >= (long long)B * N) return;
  const int b = (int)(i / N), v = (int)(i - (long long)b * N);
  const f3 p = ld3(P + 3 * i);
  f3 acc = mk3(0.f, 0.f, 0.f);
  for (int c = 0; c < C; ++c) {
    const float* E = ext + ((size_t)b * C + c) * 12;
    const float* K = intr + ((size_t)b * C + c) * 9;
    const f3 xc = mk3(E[0] * p.x + E[1] * p.y + E[2] * p.z + E[3], E[4] * p.x + E[5] * p.y + E[6] * p.z + E[7],
                      E[8] * p.x + E[9] * p.y + E[10] * p.z + E[11]);
    const float ax = K[0], ay = K[4], gm = K[1];
    const float j00 = ax / xc.z, j01 = gm / xc.z, j02 = (-ax * xc.x - gm * xc.y) / (xc.z * xc.z);
    const float j11 = ay / xc.z, j12 = (-ay * xc.y) / (xc.z * xc.z);
    const float* gg = g + (((size_t)b * C + c) * N + v) * 2;
    for (int k = 0; k < 3; ++k) {
      const float dp0 = j00 * E[k] + j01 * E[4 + k] + j02 * E[8 + k];
      const float dp1 = j11 * E[4 + k] + j12 * E[8 + k];
      const float add = dp0 * gg[0] + dp1 * gg[1];
      if (k == 0) acc.x += add; else if (k == 1) acc.y += add; else acc.z += add;
    }
  }
  out[3 * i] = acc.x; out[3 * i + 1] = acc.y; out[3 * i + 2] = acc.z;
}

// ProjectedMeshBoundaryGpu semantics on a face buffer (face >= 0 = covered).
__global__ __launch_bounds__(kB) void boundary_kernel(const int* __restrict__ face, const float* __restrict__ uv, int B,
                                                       int C, int N, int H, int W, unsigned char* __restrict__ out) {
  const long long i = (long long)blockIdx.x * kB + threadIdx.x;
  if (i >= (long long)B * C * N) return;
  const int view = (int)(i / N);
  const float pu = uv[2 * i], pw = uv[2 * i + 1];
  unsigned char f = 0;
  // (int)p - 1 >= 0 && (int)p + 1 < W, tested in float so that huge or NaN
  // positions never reach the integer conversion
  if (pu >= 1.f && pu < (float)(W - 1) && pw >= 1.f && pw < (float)(H - 1)) {
    const int u = (int)pu, w = (int)pw;
    const int* fb = face + (size_t)view * H * W;
    for (int cc = u - 1; cc <= u + 1; ++cc)
      for (int r = w - 1; r <= w + 1; ++r)
        if (fb[(size_t)r * W + cc] < 0) f = 1;
  }
  out[i] = f;
}

// ProjectedMeshBoundaryGpu's own coverage raster (Skeletool/Mesh/
// CUDABasedRasterization.cu:64-140).  The vertices are projected as
// getCamSpacePoint / projectPointFloat3 do (project_vertex: z clamped to 1e-5
// when not in front); one lane per (view, face) walks the face's pixel box
// [min - 0.5, max + 0.5], clamped to the image and truncated, and marks every
// pixel centre whose 2D barycentrics (uv2barycentric) lie in [-0.001, 1.001].
// No depth test: the bitmap is the union of the faces' pixels, every writer
// stores the same byte.
__global__ __launch_bounds__(kB) void cov_project_kernel(const float* __restrict__ vpos, const float* __restrict__ ext,
                                                          const float* __restrict__ intr, int B, int C, int N,
                                                          float* __restrict__ uv) {
  const long long i = (long long)blockIdx.x * kB + threadIdx.x;
  if (i >= (long long)B * C * N) return;
  const int view = (int)(i / N), v = (int)(i - (long long)view * N);
  const int b = view / C;
  const f4 p = project_vertex(ext + (size_t)view * 12, intr + (size_t)view * 9, vpos + ((size_t)b * N + v) * 3);
  uv[2 * i] = p.x;
  uv[2 * i + 1] = p.y;
}

// uv2barycentric's weights of corners b and c are quotients num / den whose
// denominators are the triangle's; the first weight is 1 minus both.
struct EdgeQuotient {
  float dy, dx, pq, qp, den, r;
  // the line through p and q, with weight 1 at o; r is 1 / den to a few ulp
  __device__ __forceinline__ EdgeQuotient(f2 p, f2 q, f2 o)
      : dy(p.y - q.y), dx(q.x - p.x), pq(p.x * q.y), qp(q.x * p.y) {
    den = num(o.x, dx * o.y);
    r = __builtin_amdgcn_rcpf(den);
  }
  __device__ __forceinline__ float num(float u, float dxv) const { return dy * u + dxv + pq - qp; }
  // far from the ends of the exponent range: no overflow, no flushed reciprocal
  __device__ __forceinline__ bool plain() const {
    return fabsf(den) > 1e-30f && fabsf(den) < 1e30f && fabsf(pq) < 1e30f && fabsf(qp) < 1e30f;
  }
};

// Four lanes per (view, face), one row of its pixel box each.  A weight is
// compared with the limits as a product with the reciprocal, within 1e-6 of
// the quotient where it is near them, so the two divisions are made only for
// pixels within 1e-5 of a limit, and for triangles near the ends of the
// exponent range.  A lane per face walked boxes of 34 x 34 pixels (the long
// triangles of a cap, 64 of them in one wavefront) after the rest of the
// launch was done.  16 views of 1285 x 940, 100k faces: 294 -> 97 us (108 with
// eight lanes), which is the issue time of its vector instructions.
constexpr int kCovLanes = 4;
constexpr unsigned kMaxCovBlocks = 1u << 23;  // more faces: several a group of lanes
__global__ __launch_bounds__(kB) void cov_raster_kernel(const float* __restrict__ uv, const int* __restrict__ faces,
                                                         int B, int C, int N, int F, int H, int W,
                                                         unsigned char* __restrict__ cov) {
  const long long n = (long long)B * C * F;
  for (long long i = ((long long)blockIdx.x * kB + threadIdx.x) / kCovLanes; i < n;
       i += (long long)gridDim.x * (kB / kCovLanes)) {
    // (32-bit where it can be: a 64-bit division is some 100 instructions)
    const int view = n < 1ll << 32 ? (int)((unsigned)i / (unsigned)F) : (int)(i / F);
    const int f = (int)(i - (long long)view * F);
    const f2* P = (const f2*)uv + (size_t)view * N;
    const f2 p0 = P[faces[3 * f]], p1 = P[faces[3 * f + 1]], p2 = P[faces[3 * f + 2]];
    const float bx0 = fmaxf(fminf(p0.x, fminf(p1.x, p2.x)) - 0.5f, 0.f);
    const float by0 = fmaxf(fminf(p0.y, fminf(p1.y, p2.y)) - 0.5f, 0.f);
    const float bx1 = fminf(fmaxf(p0.x, fmaxf(p1.x, p2.x)) + 0.5f, (float)(W - 1));
    const float by1 = fminf(fmaxf(p0.y, fmaxf(p1.y, p2.y)) + 0.5f, (float)(H - 1));
    // first weights 1 at p1 and p2; e0 = 1 - e2 - e1
    const EdgeQuotient q1(p0, p2, p1), q2(p0, p1, p2);
    const bool plain = q1.plain() && q2.plain();
    constexpr float kLo = -0.001f, kHi = 1.001f, kMargin = 1e-5f;
    const int ue = bx1 >= 0.f ? (int)bx1 : -1, ve = by1 >= 0.f ? (int)by1 : -1;  // the last u, v with (float)u <= bx1
    for (int v = (int)by0 + (int)(threadIdx.x % kCovLanes); v <= ve; v += kCovLanes) {
      unsigned char* row = cov + (size_t)view * H * W + (size_t)v * W;
      const float py = (float)v + 0.5f, r1 = q1.dx * py, r2 = q2.dx * py;
      for (int u = (int)bx0; u <= ue; ++u) {
        const float n1 = q1.num((float)u + 0.5f, r1), n2 = q2.num((float)u + 0.5f, r2);
        const float a1 = n1 * q1.r, a2 = n2 * q2.r, a0 = 1.f - a2 - a1;
        const float lo = fminf(a0, fminf(a1, a2)), hi = fmaxf(a0, fmaxf(a1, a2));
        if (plain && (lo < kLo - kMargin || hi > kHi + kMargin)) continue;
        bool in = true;
        if (!(plain && lo > kLo + kMargin && hi < kHi - kMargin)) {
          const float e2 = n2 / q2.den, e1 = n1 / q1.den, e0 = 1.f - e2 - e1;
          in = e0 >= kLo && e1 >= kLo && e2 >= kLo && e0 <= kHi && e1 <= kHi && e2 <= kHi;
        }
        if (in) row[u] = 1;
      }
    }
  }
}

// The boundary test of boundary_kernel on the coverage bitmap (1 = covered).
__global__ __launch_bounds__(kB) void cov_boundary_kernel(const unsigned char* __restrict__ cov,
                                                           const float* __restrict__ uv, int B, int C, int N, int H,
                                                           int W, unsigned char* __restrict__ out) {
  const long long i = (long long)blockIdx.x * kB + threadIdx.x;
  if (i >= (long long)B * C * N) return;
  const int view = (int)(i / N);
  const float pu = uv[2 * i], pw = uv[2 * i + 1];
  unsigned char f = 0;
  if (pu >= 1.f && pu < (float)(W - 1) && pw >= 1.f && pw < (float)(H - 1)) {
    const int u = (int)pu, w = (int)pw;
    const unsigned char* cv = cov + (size_t)view * H * W;
    for (int cc = u - 1; cc <= u + 1; ++cc)
      for (int r = w - 1; r <= w + 1; ++r)
        if (!cv[(size_t)r * W + cc]) f = 1;
  }
  out[i] = f;
}

// 16 bytes a lane where the array starts on 16 bytes, the rest byte by byte.
__global__ __launch_bounds__(kB) void fill_u8_kernel(unsigned char* __restrict__ p, long long n) {
  const long long i = 16 * ((long long)blockIdx.x * kB + threadIdx.x);
  if (((uintptr_t)p & 15) == 0 && i + 16 <= n) {
    *reinterpret_cast<uint4*>(p + i) = make_uint4(0u, 0u, 0u, 0u);
  } else {
    for (int k = 0; k < 16 && i + k < n; ++k) p[i + k] = 0;
  }
}

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

struct SilWs {
  int gx, gy;
  size_t cnt, off, items, list, total;
};

// The grid reaches 2 radii beyond the DT image on every side.
SilWs sil_ws(int B, int C, int N, int U, int V) {
  SilWs w{};
  w.gx = kCellsPerRadius * (U / 30 + 6);
  w.gy = kCellsPerRadius * (V / 30 + 6);
  const size_t views = (size_t)B * C, cells = (size_t)w.gx * w.gy;
  size_t o = 0;
  w.cnt = o; o = align256(o + 4 * views * (cells + kListStride));  // the lists' lengths behind the counts
  w.off = o; o = align256(o + 4 * views * (cells + 1));
  w.items = o; o = align256(o + sizeof(f4) * views * N);
  w.list = o; o = align256(o + 4 * views * U * V);
  w.total = o;
  return w;
}

}  // namespace
}  // namespace dcx

using namespace dcx;

extern "C" size_t dcx_mvsil_workspace_size(int B, int C, int N, int U, int V) {
  if (B <= 0 || C <= 0 || N <= 0 || U <= 0 || V <= 0) return 0;
  return sil_ws(B, C, N, U, V).total;
}

extern "C" dcx_status dcx_mvsil_fwd(const float* points, const float* normals, const uint8_t* is_boundary,
                                    const uint8_t* dt_image, const float* crops, int B, int C, int N, int U, int V,
                                    int search, float* residual, float* residual1, float* dt_image_gradient,
                                    float* closest_vertex_id, void* workspace, size_t ws_bytes, void* stream) {
  DCX_REQUIRE(B > 0 && C > 0 && N > 0 && U > 0 && V > 0, "dcx_mvsil_fwd: bad sizes");
  DCX_REQUIRE(points && normals && is_boundary && dt_image && crops && residual && residual1 && dt_image_gradient &&
                  closest_vertex_id,
              "dcx_mvsil_fwd: null input/output");
  DCX_REQUIRE(search == DCX_SIL_BRUTE || search == DCX_SIL_BINNED, "dcx_mvsil_fwd: search mode %d", search);
  hipStream_t s = as_stream(stream);
  SilArgs a{B, C, N, U, V, points, normals, is_boundary, dt_image, crops, residual, residual1, dt_image_gradient,
            closest_vertex_id};
  const long long P = (long long)B * C * N, PIX = (long long)B * C * U * V;
  if (search == DCX_SIL_BRUTE) {
    hipLaunchKernelGGL(sil_point_kernel, dim3(ceil_div(P, kB)), dim3(kB), 0, s, a, GridArgs{});
    hipLaunchKernelGGL(sil_pixel_brute_kernel, dim3(ceil_div(PIX, kB)), dim3(kB), 0, s, a);
    return check_launch("dcx_mvsil_fwd(brute)");
  }
  const SilWs L = sil_ws(B, C, N, U, V);
  DCX_REQUIRE(workspace && ws_bytes >= L.total, "dcx_mvsil_fwd: workspace %zu < %zu", ws_bytes, L.total);
  const long long radii = (long long)B * C * (U / 30 + 6) * (V / 30 + 6);
  DCX_REQUIRE(radii <= 4096ll * 1024, "dcx_mvsil_fwd: a grid of %lld search radii exceeds 4M", radii);
  char* w = (char*)workspace;
  GridArgs g{L.gx, L.gy, L.gx * L.gy, (unsigned int*)(w + L.cnt), (unsigned int*)(w + L.off), (f4*)(w + L.items),
             nullptr, (unsigned int*)(w + L.list)};
  const long long cells = (long long)B * C * g.cells_per_view;
  g.list_n = g.cnt + cells;
  const long long clear = cells + (long long)B * C * kListStride;
  hipLaunchKernelGGL(clear_u32_kernel, dim3(ceil_div(clear, kB)), dim3(kB), 0, s, g.cnt, clear);
  const unsigned rows = (unsigned)(B * C < kMaxViewRows ? B * C : kMaxViewRows);
  hipLaunchKernelGGL(sil_pixel_list_kernel, dim3(ceil_div((long long)U * V, kB), rows), dim3(kB), 0, s, a, g);
  hipLaunchKernelGGL(sil_point_kernel, dim3(ceil_div(P, kB)), dim3(kB), 0, s, a, g);
  hipLaunchKernelGGL(sil_grid_scan_kernel, dim3((unsigned)(B * C)), dim3(1024), 0, s, g);
  hipLaunchKernelGGL(sil_grid_scatter_kernel, dim3(ceil_div(P, kB)), dim3(kB), 0, s, a, g);
  hipLaunchKernelGGL(sil_search_kernel, dim3(kSearchBlocks, rows), dim3(kB), 0, s, a, g);
  return check_launch("dcx_mvsil_fwd(binned)");
}

extern "C" dcx_status dcx_mvsil_bwd(const float* mv_dt_grad, const float* mv_dt_grad_1, const float* dt_image_grad,
                                    const float* closest_vertex_id, const float* crops, int B, int C, int N, int U,
                                    int V, float* points_grad, void* stream) {
  DCX_REQUIRE(B > 0 && C > 0 && N > 0 && U > 0 && V > 0, "dcx_mvsil_bwd: bad sizes");
  DCX_REQUIRE(mv_dt_grad && mv_dt_grad_1 && dt_image_grad && closest_vertex_id && crops && points_grad,
              "dcx_mvsil_bwd: null input/output");
  hipStream_t s = as_stream(stream);
  const long long P = (long long)B * C * N, PIX = (long long)B * C * U * V;
  hipLaunchKernelGGL(sil_bwd_point_kernel, dim3(ceil_div(P, kB)), dim3(kB), 0, s, mv_dt_grad, dt_image_grad, P,
                     points_grad);
  hipLaunchKernelGGL(sil_bwd_pixel_kernel, dim3(ceil_div(PIX, kB)), dim3(kB), 0, s, mv_dt_grad_1, closest_vertex_id,
                     crops, N, (long long)U * V, PIX, points_grad);
  return check_launch("dcx_mvsil_bwd");
}

extern "C" dcx_status dcx_camproj_fwd(const float* points, const float* vectors, const float* extrinsics,
                                      const float* intrinsics, int B, int C, int N, int is_point, float* out,
                                      void* stream) {
  DCX_REQUIRE(B > 0 && C > 0 && N > 0, "dcx_camproj_fwd: bad sizes");
  DCX_REQUIRE(points && extrinsics && intrinsics && out && (is_point || vectors), "dcx_camproj_fwd: null input");
  hipLaunchKernelGGL(camproj_kernel, dim3(ceil_div((long long)B * C * N, kB)), dim3(kB), 0, as_stream(stream), points,
                     vectors, extrinsics, intrinsics, B, C, N, is_point, out);
  return check_launch("dcx_camproj_fwd");
}

extern "C" dcx_status dcx_camproj_bwd(const float* points_image_grad, const float* points, const float* extrinsics,
                                      const float* intrinsics, int B, int C, int N, float* points_grad, void* stream) {
  DCX_REQUIRE(B > 0 && C > 0 && N > 0, "dcx_camproj_bwd: bad sizes");
  DCX_REQUIRE(points_image_grad && points && extrinsics && intrinsics && points_grad, "dcx_camproj_bwd: null input");
  hipLaunchKernelGGL(camproj_bwd_kernel, dim3(ceil_div((long long)B * N, kB)), dim3(kB), 0, as_stream(stream),
                     points_image_grad, points, extrinsics, intrinsics, B, C, N, points_grad);
  return check_launch("dcx_camproj_bwd");
}

extern "C" size_t dcx_projected_mesh_boundary_workspace_size(int B, int C, int N, int H, int W) {
  if (B <= 0 || C <= 0 || N <= 0 || H <= 0 || W <= 0) return 0;
  return align256(sizeof(float) * 2 * (size_t)B * C * N) + (size_t)B * C * H * W;
}

extern "C" dcx_status dcx_projected_mesh_boundary(const dcx_topo* topo, int B, int C, int H, int W,
                                                  const float* points, const float* extrinsics,
                                                  const float* intrinsics, uint8_t* is_boundary, uint8_t* coverage,
                                                  void* workspace, size_t workspace_bytes, void* stream) {
  DCX_REQUIRE(topo && B > 0 && C > 0 && H > 0 && W > 0, "dcx_projected_mesh_boundary: bad sizes");
  DCX_REQUIRE(points && extrinsics && intrinsics && is_boundary && workspace,
              "dcx_projected_mesh_boundary: null argument");
  const int N = topo->N, F = topo->F;
  DCX_REQUIRE(workspace_bytes >= dcx_projected_mesh_boundary_workspace_size(B, C, N, H, W),
              "dcx_projected_mesh_boundary: workspace too small");
  hipStream_t s = as_stream(stream);
  float* uv = (float*)workspace;
  unsigned char* cov = coverage ? coverage : (unsigned char*)workspace + align256(sizeof(float) * 2 * (size_t)B * C * N);
  const long long npix = (long long)B * C * H * W;
  const unsigned cov_blocks = ceil_div((long long)B * C * F, kB / kCovLanes);
  hipLaunchKernelGGL(fill_u8_kernel, dim3(ceil_div(npix, 16 * kB)), dim3(kB), 0, s, cov, npix);
  hipLaunchKernelGGL(cov_project_kernel, dim3(ceil_div((long long)B * C * N, kB)), dim3(kB), 0, s, points, extrinsics,
                     intrinsics, B, C, N, uv);
  hipLaunchKernelGGL(cov_raster_kernel, dim3(cov_blocks < kMaxCovBlocks ? cov_blocks : kMaxCovBlocks), dim3(kB), 0, s, uv,
                     topo->faces, B, C, N, F, H, W, cov);
  hipLaunchKernelGGL(cov_boundary_kernel, dim3(ceil_div((long long)B * C * N, kB)), dim3(kB), 0, s, cov, uv, B, C, N,
                     H, W, is_boundary);
  return check_launch("dcx_projected_mesh_boundary");
}

extern "C" dcx_status dcx_mesh_boundary(const int32_t* face, const float* points_image, int B, int C, int N, int H,
                                        int W, uint8_t* is_boundary, void* stream) {
  DCX_REQUIRE(B > 0 && C > 0 && N > 0 && H > 0 && W > 0, "dcx_mesh_boundary: bad sizes");
  DCX_REQUIRE(face && points_image && is_boundary, "dcx_mesh_boundary: null input");
  hipLaunchKernelGGL(boundary_kernel, dim3(ceil_div((long long)B * C * N, kB)), dim3(kB), 0, as_stream(stream), face,
                     points_image, B, C, N, H, W, is_boundary);
  return check_launch("dcx_mesh_boundary");
}
