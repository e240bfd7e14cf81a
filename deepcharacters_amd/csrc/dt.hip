// Distance transforms of silhouette masks and the native DT silhouette loss
// on gfx950.  The reference ships DT images computed offline
// (CreateTFRecordDataset.py:65-67 only loads them); here they are built on
// the GPU from the target masks, exactly:
//
//   edt: squared distance from every pixel centre to the nearest foreground
//        pixel centre, as integers: a column pass (vertical distance g to the
//        nearest foreground pixel of the column) and a row pass (min over
//        columns x' of (x - x')^2 + g(x')^2).  Output sqrt of it as float
//        (+inf when the view has no foreground).
//   dt_encode: the uint8 encoding the silhouette op reads (value 127 on the
//        contour band, the inside distance below 127, 127 + half the
//        outside distance above), from the inside and outside transforms.
//   dtloss: L_view = sum over boundary points of D(q)^2 with D the bilinear
//        interpolation of the distance image at the point's DT-grid position
//        q = (p - crop_min) / scale + border_offset; dL/dp = 2 D grad D / scale.
#include "dcx_common.hpp"

namespace dcx {
namespace {

constexpr int kB = 256;
constexpr int kInfDist = 0x3fffffff;

// ---------------------------------------------------------------------------
// Images of up to kMaxSide pixels a side
//
// Column pass: the mask is packed into one 32-row word per column, with the
// last set row before and the first set row after the word, so the row pass
// finds a pixel's vertical distance with one bit scan.  The packed form is a
// twelfth (with one class) of the distances themselves.
//
// Row pass, one workgroup per row: the column index of the minimum never
// decreases along a row ((x - x')^2 has a strictly negative mixed difference,
// so a minimiser further left at a larger x would already win at the smaller
// x).  The minimisers of every 256th column are found by full scans, then
// those of every 64th, 16th and 4th column, and at last the row's values, each
// between the minimisers of its neighbours on the level above.  That is about
// 20 candidates a pixel and independent of the distances, where scanning
// outward until the distance is reached takes as many as the distance in
// pixels.  Integers throughout, so the values are the same.
//
// 16 views of 1024 x 1024 with a body in each: edt 3.68 -> 0.16 ms (14 us of it
// the packing), dt_encode 4.64 -> 0.27 ms.  What bounds it now is instruction
// issue: about 1,300 a wavefront and row, a quarter of them group minima.
// ---------------------------------------------------------------------------
constexpr int kMaxSide = 4096;             // a row's squared distances and values fit 40 KB of LDS
constexpr int kNone = 0x40000000;          // > 2 * kMaxSide^2, and kNone + 2 * kMaxSide^2 stays in range
constexpr int kFar = 0x7fffffff;
constexpr int kColumns = 64;               // columns per workgroup of the packing pass
constexpr int kPackBlock = 512;

// Last set row before and first set row after a word (0xffff: none).
__device__ __forceinline__ unsigned pack_ud(int up, int dn) {
  return ((unsigned)(up & 0xffff) << 16) | (unsigned)(dn & 0xffff);
}

// words[v][k][x]: bit r = row 32 k + r of column x is set; ud_fg / ud_bg: the
// nearest rows outside the word that are set / clear (ud_bg may be null).
__global__ __launch_bounds__(kPackBlock) void edt_pack_kernel(const unsigned char* __restrict__ mask, int H, int W,
                                                              int HB, unsigned* __restrict__ words,
                                                              unsigned* __restrict__ ud_fg,
                                                              unsigned* __restrict__ ud_bg) {
  extern __shared__ unsigned s_words[];  // [HB][kColumns]
  const int strips = (W + kColumns - 1) / kColumns;
  const int v = blockIdx.x / strips, strip = (blockIdx.x - v * strips) * kColumns;
  // packing: four columns a lane, one 4-byte load a row where rows start on
  // 4-byte boundaries
  const int quad = threadIdx.x % (kColumns / 4) * 4;
  const unsigned char* m = mask + (size_t)v * H * W + strip + quad;
  const bool whole = (W & 3) == 0 && ((uintptr_t)mask & 3) == 0 && strip + quad + 4 <= W;
  for (int k = threadIdx.x / (kColumns / 4); k < HB; k += kPackBlock / (kColumns / 4)) {
    unsigned w[4] = {0u, 0u, 0u, 0u};
    const int rows = min(32, H - 32 * k);
    const unsigned char* mk = m + (size_t)32 * k * W;
    if (whole && rows == 32) {
#pragma unroll
      for (int r = 0; r < 32; ++r) {
        const unsigned b = *(const unsigned*)(mk + (size_t)r * W);
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] |= (unsigned)(((b >> (8 * j)) & 0xffu) != 0) << r;
      }
    } else {
      for (int j = 0; j < 4 && strip + quad + j < W; ++j)
        for (int r = 0; r < rows; ++r) w[j] |= (unsigned)(mk[(size_t)r * W + j] != 0) << r;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      s_words[k * kColumns + quad + j] = w[j];
      if (strip + quad + j < W) words[((size_t)v * HB + k) * W + strip + quad + j] = w[j];
    }
  }
  const int col = threadIdx.x % kColumns, x = strip + col;
  const size_t base = (size_t)v * HB * W + x;
  __syncthreads();
  // one lane per (column, class): sweep down with the row above, then up with
  // the row below
  const int cls = threadIdx.x / kColumns;
  if (cls > 1 || x >= W || (cls == 1 && !ud_bg)) return;
  unsigned* ud = cls ? ud_bg : ud_fg;
  auto word = [&](int k) {
    const unsigned w = s_words[k * kColumns + col];
    if (!cls) return w;
    const int rows = H - 32 * k;
    return ~w & (rows >= 32 ? 0xffffffffu : (1u << rows) - 1u);
  };
  int up = 0xffff;
  for (int k = 0; k < HB; ++k) {
    ud[base + (size_t)k * W] = (unsigned)up << 16;
    const unsigned w = word(k);
    if (w) up = 32 * k + 31 - __clz((int)w);
  }
  int dn = 0xffff;
  for (int k = HB - 1; k >= 0; --k) {
    ud[base + (size_t)k * W] |= (unsigned)dn;
    const unsigned w = word(k);
    if (w) dn = 32 * k + __ffs(w) - 1;
  }
}

// Squared vertical distance from row y (bit r of word w) to the nearest set
// row of the column, kNone if there is none.
__device__ __forceinline__ unsigned column_d2(unsigned w, unsigned ud, int y, int r) {
  const unsigned above = w & (0xffffffffu >> (31 - r)), below = w & (0xffffffffu << r);
  const int up = (int)(ud >> 16), dn = (int)(ud & 0xffffu);
  int g = 0xffff;
  if (above) g = r - (31 - __clz((int)above));
  else if (up != 0xffff) g = y - up;
  if (below) g = min(g, __ffs(below) - 1 - r);
  else if (dn != 0xffff) g = min(g, dn - y);
  return g == 0xffff ? kNone : __mul24(g, g);
}

// The row pass compares (x - c)^2 + g(c)^2 at one x for many c, so LDS holds
// h(c) = g(c)^2 + c^2 and a candidate costs one multiply-add, h(c) - 2 x c (24
// bits a factor), and x^2 is added to the row's values at the end.
__device__ __forceinline__ int at_column(int d2, int c) { return d2 + __mul24(c, c); }
__device__ __forceinline__ int candidate(int h, int c, int minus_2x) { return __mul24(c, minus_2x) + h; }
// sign flipped: the order of signed values for an unsigned minimum
__device__ __forceinline__ unsigned ordered(int v) { return (unsigned)v ^ 0x80000000u; }

// Positions (columns p0 .. p0 + n - 1) and candidates (columns c0 .. c1) of a
// row's transform.
struct RowSpan { int p0, n, c0, c1; };

// The smallest of a group's values and the column of one that has it.
template <int kLanes>
__device__ __forceinline__ int group_argmin(int best, int at) {
  const unsigned m = group_min<kLanes>(ordered(best));
  const unsigned long long have = __ballot(ordered(best) == m);
  if (kLanes == 64) return __builtin_amdgcn_readlane(at, __ffsll(have) - 1);
  const int first = (threadIdx.x & 63) & ~(kLanes - 1);
  return __shfl(at, first + __ffs((unsigned)(have >> first) & ((1u << (kLanes & 31)) - 1u)) - 1, 64);
}

// Minimisers at left + S, left + 2 S and left + 3 S of the intervals of 4 S
// positions, kLanes lanes an interval, between the minimisers at its ends.
template <int S, int kLanes>
__device__ __forceinline__ void refine_row(const int* h, unsigned short* arg, int last, RowSpan sp) {
  const int lane = threadIdx.x % kLanes;
  for (int left = (threadIdx.x / kLanes) * 4 * S; left < sp.n; left += kB / kLanes * 4 * S) {
    const int lo = arg[left >> 2], hi = left + 4 * S < sp.n ? arg[(left + 4 * S) >> 2] : last;
    const int m2x = -2 * (sp.p0 + left);
    int best[3] = {kFar, kFar, kFar}, at[3] = {lo, lo, lo};
    for (int c = lo + lane; c <= hi; c += kLanes) {
      const int hc = h[c];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const int val = candidate(hc, c, m2x - 2 * (k + 1) * S);
        if (val < best[k]) { best[k] = val; at[k] = c; }
      }
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int a = group_argmin<kLanes>(best[k], at[k]);
      const int p = left + (k + 1) * S;
      if (lane == 0 && p < sp.n) arg[p >> 2] = (unsigned short)a;
    }
  }
  __syncthreads();
}

// val[x] = min over the candidates c of (x - c)^2 + g(c)^2 for the positions
// with want(x), by all lanes of the workgroup.  arg: (W + 3) / 4 + 1 entries.
template <class Want>
__device__ __forceinline__ void row_transform(const int* h, unsigned short* arg, RowSpan sp, int* val,
                                              Want want) {
  const int wlane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int quads = (sp.n + 3) / 4, coarse = (sp.n + 255) / 256;
  // full scans, two positions a wavefront: every 256th position and, in the
  // last slot, the last one
  for (int i = wave; i <= coarse; i += 2 * (kB / 64)) {
    const int j = i + kB / 64;
    const int x = sp.p0 + (i < coarse ? i * 256 : sp.n - 1), x2 = sp.p0 + (j < coarse ? j * 256 : sp.n - 1);
    int best = kFar, best2 = kFar, at = sp.c0, at2 = sp.c0;
    for (int c = sp.c0 + wlane; c <= sp.c1; c += 64) {
      const int hc = h[c], v = candidate(hc, c, -2 * x);
      if (v < best) { best = v; at = c; }
      if (j <= coarse) {
        const int v2 = candidate(hc, c, -2 * x2);
        if (v2 < best2) { best2 = v2; at2 = c; }
      }
    }
    at = group_argmin<64>(best, at);
    if (wlane == 0) arg[i < coarse ? i * 64 : quads] = (unsigned short)at;
    if (j <= coarse) {
      at2 = group_argmin<64>(best2, at2);
      if (wlane == 0) arg[j < coarse ? j * 64 : quads] = (unsigned short)at2;
    }
  }
  __syncthreads();
  const int last = arg[quads];
  refine_row<64, 64>(h, arg, last, sp);
  refine_row<16, 16>(h, arg, last, sp);
  refine_row<4, 4>(h, arg, last, sp);
  // the row's values, one lane per four positions; where the minimiser jumps
  // (between two far parts of the shape) the wavefront shares the scan
  for (int q0 = 0; q0 < quads; q0 += kB) {
    const int q = q0 + (int)threadIdx.x, left = sp.p0 + 4 * q;
    const bool in = q < quads;
    const int lo = in ? arg[q] : 0, hi = in ? (4 * q + 4 < sp.n ? arg[q + 1] : last) : 0;
    const bool far = in && hi - lo > 24;
    int best[4] = {kFar, kFar, kFar, kFar};
    if (in && !far)
      for (int c = lo; c <= hi; ++c) {
        const int hc = h[c];
#pragma unroll
        for (int k = 0; k < 4; ++k) best[k] = min(best[k], candidate(hc, c, -2 * (left + k)));
      }
    unsigned long long todo = __ballot(far);
    while (todo) {
      const int src = __ffsll(todo) - 1;
      todo &= todo - 1;
      const int l0 = __builtin_amdgcn_readlane(lo, src), h0 = __builtin_amdgcn_readlane(hi, src);
      const int x0 = __builtin_amdgcn_readlane(left, src);
      int b[4] = {kFar, kFar, kFar, kFar};
      for (int c = l0 + wlane; c <= h0; c += 64) {
        const int hc = h[c];
#pragma unroll
        for (int k = 0; k < 4; ++k) b[k] = min(b[k], candidate(hc, c, -2 * (x0 + k)));
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int m = (int)(group_min<64>(ordered(b[k])) ^ 0x80000000u);
        if (wlane == src) best[k] = m;
      }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (in && 4 * q + k < sp.n && want(left + k)) val[left + k] = best[k] + __mul24(left + k, left + k);
  }
  __syncthreads();
}

// First and last column with f, over a row that all lanes of the workgroup
// walk (s_span: two words, unsigned).  Returns {W, -1} if there is none.
struct ColumnSpan {
  unsigned lo = 0x7fffffffu, hi_inv = 0x7fffffffu;
  __device__ __forceinline__ void add(int x) { lo = min(lo, (unsigned)x); hi_inv = min(hi_inv, 0x7fffffffu - (unsigned)x); }
  __device__ __forceinline__ void gather(unsigned* s_span) const {
    const unsigned a = group_min<64>(lo), b = group_min<64>(hi_inv);
    if ((threadIdx.x & 63) == 0) { atomicMin(&s_span[0], a); atomicMin(&s_span[1], b); }
  }
};

__global__ __launch_bounds__(kB) void edt_rows_kernel(const unsigned* __restrict__ words,
                                                      const unsigned* __restrict__ ud_fg, int H, int W, int HB,
                                                      float* __restrict__ dist) {
  extern __shared__ int s_row[];  // h [W], values [W], minimisers
  __shared__ unsigned s_span[2];  // columns with any foreground: the only candidates
  int* h = s_row;
  int* val = s_row + W;
  unsigned short* arg = (unsigned short*)(s_row + 2 * W);
  const int v = blockIdx.x / H, y = blockIdx.x - v * H;
  const size_t base = ((size_t)v * HB + (y >> 5)) * W;
  float* out = dist + (size_t)blockIdx.x * W;
  if (threadIdx.x < 2) s_span[threadIdx.x] = 0x7fffffffu;
  __syncthreads();
  ColumnSpan cs;
  for (int x = threadIdx.x; x < W; x += kB) {
    const int d2 = column_d2(words[base + x], ud_fg[base + x], y, y & 31);
    h[x] = at_column(d2, x);
    if (d2 != kNone) cs.add(x);
  }
  cs.gather(s_span);
  __syncthreads();
  if (s_span[0] == 0x7fffffffu) {  // a view without foreground
    for (int x = threadIdx.x; x < W; x += kB) out[x] = __int_as_float(0x7f800000);
    return;
  }
  row_transform(h, arg, {0, W, (int)s_span[0], (int)(0x7fffffffu - s_span[1])}, val, [](int) { return true; });
  for (int x = threadIdx.x; x < W; x += kB) out[x] = sqrtf((float)val[x]);
}

// ---------------------------------------------------------------------------
// Larger images, and images of one row: distances kept whole, scanned outward
// ---------------------------------------------------------------------------

// Column pass: g[v][y][x] = |y - y*| to the nearest pixel of class `fg` in
// column x (kInfDist if none).
__global__ __launch_bounds__(kB) void edt_col_kernel(const unsigned char* mask, int V, int H, int W, int fg,
                                                     int* g) {
  const long long i = (long long)blockIdx.x * kB + threadIdx.x;
  if (i >= (long long)V * W) return;
  const int v = (int)(i / W), x = (int)(i - (long long)v * W);
  const unsigned char* m = mask + (size_t)v * H * W;
  int* gv = g + (size_t)v * H * W;
  int last = -1;
  for (int y = 0; y < H; ++y) {
    if ((m[(size_t)y * W + x] != 0) == (fg != 0)) last = y;
    gv[(size_t)y * W + x] = last >= 0 ? y - last : kInfDist;
  }
  last = -1;
  for (int y = H - 1; y >= 0; --y) {
    if ((m[(size_t)y * W + x] != 0) == (fg != 0)) last = y;
    if (last >= 0 && last - y < gv[(size_t)y * W + x]) gv[(size_t)y * W + x] = last - y;
  }
}

// Row pass: exact squared distance, as a 64-bit integer (kInfDist^2 marks none).
__device__ __forceinline__ long long edt_row(const int* gr, int W, int x) {
  long long best = 0x7fffffffffffffffll;
  for (int d = 0; d < W; ++d) {
    const long long dd = (long long)d * d;
    if (dd >= best) break;
    if (x - d >= 0 && gr[x - d] != kInfDist) best = min(best, dd + (long long)gr[x - d] * gr[x - d]);
    if (d > 0 && x + d < W && gr[x + d] != kInfDist) best = min(best, dd + (long long)gr[x + d] * gr[x + d]);
  }
  return best;
}

__global__ __launch_bounds__(kB) void edt_row_kernel(const int* g, int V, int H, int W, float* dist) {
  const long long i = (long long)blockIdx.x * kB + threadIdx.x;
  if (i >= (long long)V * H * W) return;
  const long long row = i / W;
  const int x = (int)(i - row * W);
  const long long d2 = edt_row(g + row * W, W, x);
  dist[i] = d2 == 0x7fffffffffffffffll ? __int_as_float(0x7f800000) : sqrtf((float)d2);
}

// The encoded value of a pixel of class f that is not on the contour band, d2
// its squared distance to the other class (dd = 1e30 where there is none).
__device__ __forceinline__ int dt_value(bool f, float dd) {
  return f ? (int)fminf(fmaxf(rintf(dd) - 1.f, 0.f), 126.f) : 127 + (int)fminf(fmaxf(rintf(dd / 2.f), 1.f), 128.f);
}

// The DT image encoding: contour band (foreground pixels with a background
// or out-of-image 4-neighbour and background pixels with a foreground
// 4-neighbour) = 127;
// other foreground: clamp(rint(d_in) - 1, 0, 126); other background:
// 127 + clamp(rint(d_out / 2), 1, 128).  d_in is the distance to the
// nearest background pixel, d_out to the nearest foreground pixel.
__global__ __launch_bounds__(kB) void dt_encode_kernel(const unsigned char* mask, const int* g_fg, const int* g_bg,
                                                       int V, int H, int W, unsigned char* out) {
  const long long i = (long long)blockIdx.x * kB + threadIdx.x;
  if (i >= (long long)V * H * W) return;
  const long long row = i / W;
  const int x = (int)(i - row * W);
  const int y = (int)(row % H);
  const unsigned char* m = mask + (i - (long long)y * W - x);
  const bool f = m[(size_t)y * W + x] != 0;
  // outside the image counts as background (a foreground pixel on the image
  // border is on the contour; a background one is not made so by the border)
  bool edge = false;
  const int nx[4] = {x - 1, x + 1, x, x}, ny[4] = {y, y, y - 1, y + 1};
  for (int k = 0; k < 4; ++k) {
    const bool in = nx[k] >= 0 && nx[k] < W && ny[k] >= 0 && ny[k] < H;
    const bool nf = in && m[(size_t)ny[k] * W + nx[k]] != 0;
    if (nf != f) edge = true;
  }
  int val;
  if (edge) {
    val = 127;
  } else if (f) {
    const long long d2 = edt_row(g_bg + row * W, W, x);
    const float dd = d2 == 0x7fffffffffffffffll ? 1e30f : sqrtf((float)d2);
    val = dt_value(true, dd);
  } else {
    const long long d2 = edt_row(g_fg + row * W, W, x);
    const float dd = d2 == 0x7fffffffffffffffll ? 1e30f : sqrtf((float)d2);
    val = dt_value(false, dd);
  }
  out[i] = (unsigned char)val;
}

// dt_encode_kernel's image from the packed mask: one workgroup per row, the
// transform of each class evaluated at the other class's pixels only.
__global__ __launch_bounds__(kB) void dt_encode_rows_kernel(const unsigned* __restrict__ words,
                                                            const unsigned* __restrict__ ud_fg,
                                                            const unsigned* __restrict__ ud_bg, int H, int W, int HB,
                                                            unsigned char* __restrict__ out) {
  extern __shared__ int s_row[];
  __shared__ unsigned s_span[4];  // columns with any foreground; foreground columns of this row
  int* h = s_row;
  int* val = s_row + W;
  unsigned short* arg = (unsigned short*)(s_row + 2 * W);
  unsigned char* cls = (unsigned char*)(arg + (W + 3) / 4 + 1);  // bits: this row, the row above, the row below
  const int v = blockIdx.x / H, y = blockIdx.x - v * H, k = y >> 5, r = y & 31;
  const size_t base = ((size_t)v * HB + k) * W;
  if (threadIdx.x < 4) s_span[threadIdx.x] = 0x7fffffffu;
  __syncthreads();
  ColumnSpan sites, fg;
  int any_bg = 0;
  for (int x = threadIdx.x; x < W; x += kB) {
    const unsigned w = words[base + x];
    const unsigned here = (w >> r) & 1u;
    const unsigned up = r > 0 ? (w >> (r - 1)) & 1u : (k > 0 ? words[base - W + x] >> 31 : 0u);
    const unsigned dn = r < 31 ? (w >> (r + 1)) & 1u : (k + 1 < HB ? words[base + W + x] & 1u : 0u);
    cls[x] = (unsigned char)(here | (up << 1) | (dn << 2));
    if (here) fg.add(x); else any_bg = 1;
    const int d2 = column_d2(w, ud_fg[base + x], y, r);
    h[x] = at_column(d2, x);
    val[x] = kNone;
    if (d2 != kNone) sites.add(x);
  }
  sites.gather(s_span);
  fg.gather(s_span + 2);
  any_bg = __syncthreads_or(any_bg);
  const bool have = s_span[0] != 0x7fffffffu, any_fg = s_span[2] != 0x7fffffffu;
  if (any_bg && have)
    row_transform(h, arg, {0, W, (int)s_span[0], (int)(0x7fffffffu - s_span[1])}, val,
                  [&](int x) { return (cls[x] & 1) == 0; });
  if (any_fg) {
    // the background columns next to the row's foreground are nearer than
    // anything beyond them
    const int x0 = max((int)s_span[2] - 1, 0), x1 = min((int)(0x7fffffffu - s_span[3]) + 1, W - 1);
    const int rows = H - 32 * k;
    const unsigned valid = rows >= 32 ? 0xffffffffu : (1u << rows) - 1u;
    for (int x = x0 + threadIdx.x; x <= x1; x += kB)
      h[x] = at_column(column_d2(~words[base + x] & valid, ud_bg[base + x], y, r), x);
    __syncthreads();
    row_transform(h, arg, {x0, x1 - x0 + 1, x0, x1}, val, [&](int x) { return (cls[x] & 1) != 0; });
  }
  unsigned char* o = out + (size_t)blockIdx.x * W;
  for (int x = threadIdx.x; x < W; x += kB) {
    const unsigned c = cls[x], f = c & 1u;
    const unsigned lf = x > 0 ? cls[x - 1] & 1u : 0u, rt = x + 1 < W ? cls[x + 1] & 1u : 0u;
    const bool edge = lf != f || rt != f || ((c >> 1) & 1u) != f || ((c >> 2) & 1u) != f;
    o[x] = (unsigned char)(edge ? 127 : dt_value(f != 0, val[x] >= kNone ? 1e30f : sqrtf((float)val[x])));
  }
}

struct DtSample { float d, gx, gy; bool ok; };

// Bilinear sample of the distance image at DT-grid position (qx, qy) (pixel
// i's centre at i + 0.5) and its gradient; ok = false when the footprint
// leaves the image or touches an infinite value.
__device__ __forceinline__ DtSample dt_sample(const float* D, int H, int W, float qx, float qy) {
  DtSample s{0.f, 0.f, 0.f, false};
  const float fx = qx - 0.5f, fy = qy - 0.5f;
  if (!(fx >= 0.f && fy >= 0.f && fx < (float)(W - 1) && fy < (float)(H - 1))) return s;
  const int x0 = (int)fx, y0 = (int)fy;
  const float tx = fx - (float)x0, ty = fy - (float)y0;
  const float d00 = D[(size_t)y0 * W + x0], d10 = D[(size_t)y0 * W + x0 + 1];
  const float d01 = D[(size_t)(y0 + 1) * W + x0], d11 = D[(size_t)(y0 + 1) * W + x0 + 1];
  if (!(isfinite(d00) && isfinite(d10) && isfinite(d01) && isfinite(d11))) return s;
  s.d = (1.f - ty) * ((1.f - tx) * d00 + tx * d10) + ty * ((1.f - tx) * d01 + tx * d11);
  s.gx = (1.f - ty) * (d10 - d00) + ty * (d11 - d01);
  s.gy = (1.f - tx) * (d01 - d00) + tx * (d11 - d10);
  s.ok = true;
  return s;
}

// One workgroup per (view, block of points): residuals D(q), the block's sum
// of D^2 into a partial, and (bwd) dL/dp.
__global__ __launch_bounds__(kB) void dtloss_kernel(const float* points, const unsigned char* isb, const float* dist,
                                                    const float* crops, int N, int H, int W, float* residual,
                                                    float* partial, const float* g_loss, float* g_points) {
  __shared__ float s_red[kB / 64];
  const int view = blockIdx.y;
  const int v = blockIdx.x * kB + threadIdx.x;
  float l = 0.f;
  if (v < N) {
    const size_t i = (size_t)view * N + v;
    const float* cr = crops + (size_t)view * 7;
    const float sc = cr[2];
    const float qx = (points[2 * i] - cr[3]) / sc + cr[0], qy = (points[2 * i + 1] - cr[4]) / sc + cr[1];
    DtSample s = dt_sample(dist + (size_t)view * H * W, H, W, qx, qy);
    if (isb && !isb[i]) s.ok = false;
    const float r = s.ok ? s.d : 0.f;
    if (residual) residual[i] = r;
    l = r * r;
    if (g_points) {
      const float gl = g_loss[view];
      g_points[2 * i] = s.ok ? gl * 2.f * r * s.gx / sc : 0.f;
      g_points[2 * i + 1] = s.ok ? gl * 2.f * r * s.gy / sc : 0.f;
    }
  }
  if (!partial) return;
  l = wave_sum(l);
  if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = l;
  __syncthreads();
  if (threadIdx.x == 0) {
    float t = 0.f;
    for (int k = 0; k < kB / 64; ++k) t += s_red[k];
    partial[(size_t)view * gridDim.x + blockIdx.x] = t;
  }
}

// One wavefront per view (a lane per view walks its partials one load after
// the other: 13 us for 98 partials, against 4).
__global__ __launch_bounds__(64) void dtloss_sum_kernel(const float* partial, int nblk, float* loss) {
  float t = 0.f;
  for (int k = threadIdx.x; k < nblk; k += 64) t += partial[(size_t)blockIdx.x * nblk + k];
  t = wave_sum(t);
  if (threadIdx.x == 0) loss[blockIdx.x] = t;
}

// The packed form's words and row pairs fit the workspace where at least two
// rows share a word; its row pass holds a row in LDS and launches a workgroup
// per row, whose threads a grid has to count in 32 bits.
bool packed_form(int V, int H, int W) {
  return H >= 2 && H <= kMaxSide && W <= kMaxSide && (long long)V * H <= 1 << 23;
}

size_t row_lds(int W) { return 2 * sizeof(unsigned) * (size_t)W + 2 * (size_t)((W + 3) / 4 + 1) + W; }

}  // namespace
}  // namespace dcx

using namespace dcx;

extern "C" size_t dcx_edt_workspace_size(int V, int H, int W) {
  if (V <= 0 || H <= 0 || W <= 0) return 0;
  return 2 * sizeof(int) * (size_t)V * H * W;
}

extern "C" dcx_status dcx_edt(const uint8_t* mask, int V, int H, int W, float* dist, void* workspace,
                              size_t workspace_bytes, void* stream) {
  DCX_REQUIRE(mask && dist && V > 0 && H > 0 && W > 0, "dcx_edt: bad arguments");
  DCX_REQUIRE(workspace && workspace_bytes >= sizeof(int) * (size_t)V * H * W, "dcx_edt: workspace too small");
  hipStream_t s = as_stream(stream);
  if (packed_form(V, H, W)) {
    const int HB = (H + 31) / 32;
    unsigned* words = (unsigned*)workspace;
    unsigned* ud = words + (size_t)V * HB * W;
    hipLaunchKernelGGL(edt_pack_kernel, dim3(ceil_div(W, kColumns) * (unsigned)V), dim3(kPackBlock), sizeof(unsigned) * kColumns * HB, s,
                       mask, H, W, HB, words, ud, (unsigned*)nullptr);
    hipLaunchKernelGGL(edt_rows_kernel, dim3((unsigned)V * H), dim3(kB), row_lds(W), s, words, ud, H, W, HB, dist);
    return check_launch("dcx_edt");
  }
  int* g = (int*)workspace;
  hipLaunchKernelGGL(edt_col_kernel, dim3(ceil_div((long long)V * W, kB)), dim3(kB), 0, s, mask, V, H, W, 1, g);
  hipLaunchKernelGGL(edt_row_kernel, dim3(ceil_div((long long)V * H * W, kB)), dim3(kB), 0, s, g, V, H, W, dist);
  return check_launch("dcx_edt");
}

extern "C" dcx_status dcx_dt_encode(const uint8_t* mask, int V, int H, int W, uint8_t* dt_out, void* workspace,
                                    size_t workspace_bytes, void* stream) {
  DCX_REQUIRE(mask && dt_out && V > 0 && H > 0 && W > 0, "dcx_dt_encode: bad arguments");
  DCX_REQUIRE(workspace && workspace_bytes >= dcx_edt_workspace_size(V, H, W), "dcx_dt_encode: workspace too small");
  hipStream_t s = as_stream(stream);
  if (packed_form(V, H, W)) {
    const int HB = (H + 31) / 32;
    const size_t n = (size_t)V * HB * W;
    unsigned* words = (unsigned*)workspace;
    hipLaunchKernelGGL(edt_pack_kernel, dim3(ceil_div(W, kColumns) * (unsigned)V), dim3(kPackBlock), sizeof(unsigned) * kColumns * HB, s,
                       mask, H, W, HB, words, words + n, words + 2 * n);
    hipLaunchKernelGGL(dt_encode_rows_kernel, dim3((unsigned)V * H), dim3(kB), row_lds(W), s, words, words + n,
                       words + 2 * n, H, W, HB, dt_out);
    return check_launch("dcx_dt_encode");
  }
  int* g_fg = (int*)workspace;
  int* g_bg = g_fg + (size_t)V * H * W;
  hipLaunchKernelGGL(edt_col_kernel, dim3(ceil_div((long long)V * W, kB)), dim3(kB), 0, s, mask, V, H, W, 1, g_fg);
  hipLaunchKernelGGL(edt_col_kernel, dim3(ceil_div((long long)V * W, kB)), dim3(kB), 0, s, mask, V, H, W, 0, g_bg);
  hipLaunchKernelGGL(dt_encode_kernel, dim3(ceil_div((long long)V * H * W, kB)), dim3(kB), 0, s, mask, g_fg, g_bg, V,
                     H, W, dt_out);
  return check_launch("dcx_dt_encode");
}

extern "C" size_t dcx_dtloss_workspace_size(int V, int N) {
  if (V <= 0 || N <= 0) return 0;
  return sizeof(float) * (size_t)V * ceil_div(N, kB);
}

extern "C" dcx_status dcx_dtloss_fwd(const float* points, const uint8_t* is_boundary, const float* dist,
                                     const float* crops, int V, int N, int H, int W, float* residual, float* loss,
                                     void* workspace, size_t workspace_bytes, void* stream) {
  DCX_REQUIRE(points && dist && crops && loss && V > 0 && N > 0 && H > 1 && W > 1, "dcx_dtloss_fwd: bad arguments");
  DCX_REQUIRE(workspace && workspace_bytes >= dcx_dtloss_workspace_size(V, N), "dcx_dtloss_fwd: workspace too small");
  hipStream_t s = as_stream(stream);
  const unsigned nblk = ceil_div(N, kB);
  float* partial = (float*)workspace;
  hipLaunchKernelGGL(dtloss_kernel, dim3(nblk, V), dim3(kB), 0, s, points, is_boundary, dist, crops, N, H, W, residual,
                     partial, nullptr, nullptr);
  hipLaunchKernelGGL(dtloss_sum_kernel, dim3(V), dim3(64), 0, s, partial, (int)nblk, loss);
  return check_launch("dcx_dtloss_fwd");
}

extern "C" dcx_status dcx_dtloss_bwd(const float* points, const uint8_t* is_boundary, const float* dist,
                                     const float* crops, int V, int N, int H, int W, const float* g_loss,
                                     float* points_grad, void* stream) {
  DCX_REQUIRE(points && dist && crops && g_loss && points_grad && V > 0 && N > 0 && H > 1 && W > 1,
              "dcx_dtloss_bwd: bad arguments");
  hipLaunchKernelGGL(dtloss_kernel, dim3(ceil_div(N, kB), V), dim3(kB), 0, as_stream(stream), points, is_boundary,
                     dist, crops, N, H, W, nullptr, nullptr, g_loss, points_grad);
  return check_launch("dcx_dtloss_bwd");
}
