// Dual-quaternion and linear-blend skinning on gfx950, forward and backward.
//
// One lane per (batch, vertex).  A block covers 256 consecutive vertices of a
// single batch element (grid.y = batch), so the batch's joint table is staged
// once into LDS and every per-vertex gather of a joint transform is an LDS
// read.  Per-vertex records (positions [N,3], weights [N,K], joint indices
// [N,K]) are read as contiguous 12/16-byte vectors: a wavefront touches one
// contiguous 768-1024 byte span per array, which is fully coalesced.
//
// Joint-level gradients (d/d joint DQ, d/d joint transform) are summed per
// wavefront and joint in registers, per workgroup in LDS, and then issued as
// one global atomic per (workgroup, joint, component).
#include <type_traits>

#include "dcx_common.hpp"
#include "skin_common.hpp"

namespace dcx {
namespace {

constexpr int kBlock = 256;
constexpr int kMaxLdsJoints = 256;   // joint table staged in LDS up to this size

// A vertex's skin weights and joint ids.  kK = 4: one 16-byte load each (the
// caller has checked the alignment) and loops of a known length, so the
// arrays stay in registers; kK = 0: any K.
template <int kK>
__device__ __forceinline__ void load_skin(const float* wv, const int* jv, int K, int* idx, float* w) {
  if (kK == 4) {
    const int4 j = *reinterpret_cast<const int4*>(jv);
    const float4 x = *reinterpret_cast<const float4*>(wv);
    idx[0] = j.x; idx[1] = j.y; idx[2] = j.z; idx[3] = j.w;
    w[0] = x.x; w[1] = x.y; w[2] = x.z; w[3] = x.w;
  } else {
    for (int k = 0; k < K; ++k) { idx[k] = jv[k]; w[k] = wv[k]; }
  }
}

// The op's copies of its inputs (dual quaternions / transforms, weights) are
// written by the same launch: table entries by the first block of a pose.
template <int kRow>
__device__ __forceinline__ void copy_table(const float* src, float* dst, int b, int J) {
  if (!dst || blockIdx.x != 0) return;
  for (int i = threadIdx.x; i < J * kRow; i += kBlock) dst[(size_t)b * J * kRow + i] = src[(size_t)b * J * kRow + i];
}

template <bool kLds, int kK>
__global__ __launch_bounds__(kBlock) void dqs_fwd_kernel(
    const float* __restrict__ dq, const float* __restrict__ weights,
    const int* __restrict__ jidx, const float* __restrict__ rest_pos,
    const float* __restrict__ rest_nrm, int N, int K_, int J, float* __restrict__ pos,
    float* __restrict__ nrm, float* __restrict__ dq_out, float* __restrict__ w_out) {
  __shared__ float s_tab[kLds ? kMaxLdsJoints * 8 : 1];
  const int K = kK ? kK : K_;
  const int b = blockIdx.y;
  const float* tab = dq + (size_t)b * J * 8;
  copy_table<8>(dq, dq_out, b, J);
  if (kLds) {
    for (int i = threadIdx.x; i < J * 8; i += kBlock) s_tab[i] = tab[i];
    __syncthreads();
    tab = s_tab;
  }
  const int v = blockIdx.x * kBlock + threadIdx.x;
  if (v >= N) return;
  int idx[kMaxK];
  float w[kMaxK];
  const size_t at = ((size_t)b * N + v) * K;
  load_skin<kK>(weights + at, jidx + (size_t)v * K, K, idx, w);
  if (w_out) {
    if (kK == 4)
      *reinterpret_cast<float4*>(w_out + at) = make_float4(w[0], w[1], w[2], w[3]);
    else
      for (int k = 0; k < K; ++k) w_out[at + k] = w[k];
  }
  DqBlend bl = dq_blend(tab, idx, w, K);
  m3 R = quat_to_mat(bl.r);
  f3 p = mk3(rest_pos[3 * v], rest_pos[3 * v + 1], rest_pos[3 * v + 2]);
  f3 out = mul(R, p) + dq_translation(bl.r, bl.d);
  float* po = pos + ((size_t)b * N + v) * 3;
  po[0] = out.x; po[1] = out.y; po[2] = out.z;
  if (nrm) {
    f3 n = mk3(rest_nrm[3 * v], rest_nrm[3 * v + 1], rest_nrm[3 * v + 2]);
    f3 m = mul(R, n);
    float inv = 1.f / len(m);
    float* no = nrm + ((size_t)b * N + v) * 3;
    no[0] = m.x * inv; no[1] = m.y * inv; no[2] = m.z * inv;
  }
}

// Reference-compatible skin-weight gradient (DQSkinningGPUOpGrad.cu:64-138):
// derivative of the normalised blend w.r.t. weight k, pushed through the
// point-rotation Jacobian of DQHelper.h:93-179 whose entries add vert.z
// instead of multiplying by it, plus the translation Jacobians (:184-235).
__device__ float ref_weight_grad(const DqBlend& bl, f4 qr, f4 qd, float sgn, f3 p, f3 g) {
  const float L = bl.small ? 1.f : len(bl.br);
  f4 dsc1 = bl.br * (1.f / (2.f * L) * 2.f);
  float dS = bl.small ? 0.f : dot(dsc1, qr * sgn);
  f4 dR = (qr * sgn * L - bl.br * dS) * (1.f / (L * L));
  f4 dT = (qd * sgn * L - bl.bd * dS) * (1.f / (L * L));
  const f4 r = bl.r, d = bl.d;
  const float x = r.x, y = r.y, z = r.z, w = r.w;
  // Rows of the (defective) rotated-point Jacobian: sum_c dRi0/dc*p.x + dRi1/dc*p.y + dRi2/dc + p.z
  float J0[4] = {0.f * p.x + 2.f * y * p.y + 2.f * z + p.z, -4.f * y * p.x + 2.f * x * p.y + 2.f * w + p.z,
                 -4.f * z * p.x + -2.f * w * p.y + 2.f * x + p.z, 0.f * p.x + -2.f * z * p.y + 2.f * y + p.z};
  float J1[4] = {2.f * y * p.x + -4.f * x * p.y + -2.f * w + p.z, 2.f * x * p.x + 0.f * p.y + 2.f * z + p.z,
                 2.f * w * p.x + -4.f * z * p.y + 2.f * y + p.z, 2.f * z * p.x + 0.f * p.y + -2.f * x + p.z};
  float J2[4] = {2.f * z * p.x + 2.f * w * p.y + -4.f * x + p.z, -2.f * w * p.x + 2.f * z * p.y + -4.f * y + p.z,
                 2.f * x * p.x + 2.f * y * p.y + 0.f + p.z, -2.f * y * p.x + 2.f * x * p.y + 0.f + p.z};
  float TR0[4] = {2.f * -d.w, 2.f * d.z, 2.f * -d.y, 2.f * d.x};
  float TR1[4] = {2.f * -d.z, 2.f * -d.w, 2.f * d.x, 2.f * d.y};
  float TR2[4] = {2.f * d.y, 2.f * -d.x, 2.f * -d.w, 2.f * d.z};
  float TT0[4] = {2.f * w, 2.f * -z, 2.f * y, 2.f * -x};
  float TT1[4] = {2.f * z, 2.f * w, 2.f * -x, 2.f * -y};
  float TT2[4] = {2.f * -y, 2.f * x, 2.f * w, 2.f * -z};
  float dr[4] = {dR.x, dR.y, dR.z, dR.w}, dt[4] = {dT.x, dT.y, dT.z, dT.w};
  f3 gs = mk3(0.f, 0.f, 0.f);
  for (int c = 0; c < 4; ++c) {
    gs.x += J0[c] * dr[c] + TR0[c] * dr[c] + TT0[c] * dt[c];
    gs.y += J1[c] * dr[c] + TR1[c] * dr[c] + TT1[c] * dt[c];
    gs.z += J2[c] * dr[c] + TR2[c] * dr[c] + TT2[c] * dt[c];
  }
  return dot(gs, g);
}

// Adds a wavefront's joint gradients to LDS: lane's slot k adds coef[k] *
// grad[e] to word e of joint idx[k].  An LDS float add takes the crossbar
// about four cycles a lane, conflicts or not (32 adds a lane were 76 us of
// the 106 us backward of 16 poses of 25k vertices), and neighbouring vertices
// share joints, so the wavefront goes through its distinct joints, sums over
// its lanes in registers and adds each word once: 21 us.  Lanes whose
// joints are still left after kJointRounds (a skinning without order) add
// their words themselves.  All lanes call it; those without a vertex with
// active = false.
constexpr int kJointRounds = 24;
template <int kRow, int kK>
__device__ __forceinline__ void add_joint_grads(float* s_acc, bool active, const int* idx, const float* coef,
                                                const float* grad, int K) {
  static_assert(kRow == 8 || kRow == 12, "dual quaternions or transforms");
  const int lane = threadIdx.x & 63;
  unsigned todo = active ? (1u << K) - 1u : 0u;
  for (int r = 0; r < kJointRounds; ++r) {
    const unsigned long long left = __ballot(todo != 0);
    if (!left) return;
    // the first such lane's first joint
    int mine = 0;
#pragma unroll
    for (int k = (kK ? kK : kMaxK) - 1; k >= 0; --k)
      if ((todo >> k) & 1u) mine = idx[k];
    const int j = __builtin_amdgcn_readlane(mine, __ffsll(left) - 1);
    float c = 0.f;
    bool has = false;  // (an infinite gradient must not reach joints that are not the lane's)
#pragma unroll
    for (int k = 0; k < (kK ? kK : kMaxK); ++k)
      if (((todo >> k) & 1u) && idx[k] == j) {
        c += coef[k];
        has = true;
        todo &= ~(1u << k);
      }
    float v[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) v[e] = e < kRow && has ? grad[e] * c : 0.f;
    const float t = wave_sum8(v);
    if (lane < 8) atomicAdd(&s_acc[j * kRow + lane], t);
    if (kRow > 8) {
      const float t2 = wave_sum8(v + 8);
      if (lane < kRow - 8) atomicAdd(&s_acc[j * kRow + 8 + lane], t2);
    }
  }
#pragma unroll
  for (int k = 0; k < (kK ? kK : kMaxK); ++k)
    if ((todo >> k) & 1u)
      for (int e = 0; e < kRow; ++e) atomicAdd(&s_acc[idx[k] * kRow + e], grad[e] * coef[k]);
}
__device__ __forceinline__ void acc_flush(const float* s_acc, int words, float* dst) {
  for (int i = threadIdx.x; i < words; i += kBlock)
    if (s_acc[i] != 0.f) atomicAdd(dst + i, s_acc[i]);
}

// `per` blocks of vertices per workgroup (one joint flush for all of them).
template <bool kLds, int kK>
__global__ __launch_bounds__(kBlock) void dqs_bwd_kernel(
    const float* __restrict__ g_pos, const float* __restrict__ g_nrm,
    const float* __restrict__ dq, const float* __restrict__ weights,
    const int* __restrict__ jidx, const float* __restrict__ rest_pos,
    const float* __restrict__ rest_nrm, int N, int K_, int J, float* __restrict__ g_dq,
    float* __restrict__ g_w, float* __restrict__ g_rest, int flags, int per) {
  __shared__ float s_tab[kLds ? kMaxLdsJoints * 8 : 1];
  __shared__ float s_acc[kLds ? kMaxLdsJoints * 8 : 1];
  const int K = kK ? kK : K_;
  const int b = blockIdx.y;
  const float* tab = dq + (size_t)b * J * 8;
  if (kLds) {
    for (int i = threadIdx.x; i < J * 8; i += kBlock) { s_tab[i] = tab[i]; s_acc[i] = 0.f; }
    __syncthreads();
    tab = s_tab;
  }
  for (int c = 0; c < per; ++c) {
    // (lanes past the last vertex repeat it and store nothing)
    const int v0 = (blockIdx.x * per + c) * kBlock + threadIdx.x;
    const bool in = v0 < N;
    const int v = in ? v0 : N - 1;
    int idx[kMaxK];
    float w[kMaxK];
    const size_t at = ((size_t)b * N + v) * K;
    load_skin<kK>(weights + at, jidx + (size_t)v * K, K, idx, w);
    DqBlend bl = dq_blend(tab, idx, w, K);
    m3 R = quat_to_mat(bl.r);
    f3 p = mk3(rest_pos[3 * v], rest_pos[3 * v + 1], rest_pos[3 * v + 2]);
    const float* gp = g_pos + ((size_t)b * N + v) * 3;
    f3 g = mk3(gp[0], gp[1], gp[2]);
    // dL/dR = g p^T (+ normal term)
    float G[9] = {g.x * p.x, g.x * p.y, g.x * p.z, g.y * p.x, g.y * p.y, g.y * p.z,
                  g.z * p.x, g.z * p.y, g.z * p.z};
    if (g_nrm) {
      const float* gn = g_nrm + ((size_t)b * N + v) * 3;
      f3 n = mk3(rest_nrm[3 * v], rest_nrm[3 * v + 1], rest_nrm[3 * v + 2]);
      f3 m = mul(R, n);
      float il = 1.f / len(m);
      f3 nn = m * il;
      f3 gnv = mk3(gn[0], gn[1], gn[2]);
      f3 gm = (gnv - nn * dot(nn, gnv)) * il;
      G[0] += gm.x * n.x; G[1] += gm.x * n.y; G[2] += gm.x * n.z;
      G[3] += gm.y * n.x; G[4] += gm.y * n.y; G[5] += gm.y * n.z;
      G[6] += gm.z * n.x; G[7] += gm.z * n.y; G[8] += gm.z * n.z;
    }
    const f4 r = bl.r, d = bl.d;
    f4 gr = dR_dq_contract(r, G);
    gr.x += 2.f * (-d.w * g.x - d.z * g.y + d.y * g.z);
    gr.y += 2.f * (d.z * g.x - d.w * g.y - d.x * g.z);
    gr.z += 2.f * (-d.y * g.x + d.x * g.y - d.w * g.z);
    gr.w += 2.f * (d.x * g.x + d.y * g.y + d.z * g.z);
    f4 gd = mk4(2.f * (r.w * g.x + r.z * g.y - r.y * g.z), 2.f * (-r.z * g.x + r.w * g.y + r.x * g.z),
                2.f * (r.y * g.x - r.x * g.y + r.w * g.z), 2.f * (-r.x * g.x - r.y * g.y - r.z * g.z));
    // Through the normalisation r = br/|br|, d = bd/|br|.
    f4 gbr, gbd;
    if (bl.small) {
      gbr = gr; gbd = gd;
    } else {
      float proj = dot(gr, r) + dot(gd, d);
      gbr = (gr - r * proj) * bl.scale;
      gbd = gd * bl.scale;
    }
    if (g_rest && in) {
      f3 gq = mulT(R, g);
      float* o = g_rest + ((size_t)b * N + v) * 3;
      o[0] = gq.x; o[1] = gq.y; o[2] = gq.z;
    }
    if (g_w && in) {
      float gw[kMaxK];
#pragma unroll
      for (int k = 0; k < (kK ? kK : kMaxK); ++k) {
        if (k >= K) break;
        const float* q = tab + idx[k] * 8;
        f4 qr = ld4(q), qd = ld4(q + 4);
        const float s = bl.sgn[k];
        gw[k] = flags & DCX_FLAG_REF_COMPAT ? ref_weight_grad(bl, qr, qd, s, p, g)
                                            : s * (dot(gbr, qr) + dot(gbd, qd));
        if (kK != 4) g_w[at + k] = gw[k];
      }
      if (kK == 4) *reinterpret_cast<float4*>(g_w + at) = make_float4(gw[0], gw[1], gw[2], gw[3]);
    }
    if (g_dq) {
      const float gb[8] = {gbr.x, gbr.y, gbr.z, gbr.w, gbd.x, gbd.y, gbd.z, gbd.w};
      float coef[kMaxK];
#pragma unroll
      for (int k = 0; k < (kK ? kK : kMaxK); ++k) coef[k] = k < K ? w[k] * bl.sgn[k] : 0.f;
      if (kLds) {
        add_joint_grads<8, kK>(s_acc, in, idx, coef, gb, K);
      } else if (in) {
        for (int k = 0; k < K; ++k)
          for (int e = 0; e < 8; ++e) atomicAdd(g_dq + ((size_t)b * J + idx[k]) * 8 + e, gb[e] * coef[k]);
      }
    }
  }
  if (kLds && g_dq) {
    __syncthreads();
    acc_flush(s_acc, J * 8, g_dq + (size_t)b * J * 8);
  }
}

// One workgroup per (batch, dof) over the DOF's influence row, which ends at
// the first entry whose vertex field is -1, with a deterministic sum
// (reference: one serial thread per DOF).  The row is taken in tiles of 4,096
// entries, the next tile's entries loading while this one's vertices are
// gathered; a tile looks for the end itself, so a row is read once and not
// past its tile (a pass over the whole padded row came first, and 256 lanes
// took an entry at a time: the root's rows hold every vertex, 100k entries
// for a 25k-vertex body).  16 poses, 57 DOFs: 1,202 -> 124 us.
constexpr int kDofBlock = 1024;
constexpr int kDofPer = 4;
template <bool kVec>
__global__ __launch_bounds__(kDofBlock) void dof_grad_kernel(
    const float* __restrict__ g_pos, const float* __restrict__ skinned,
    const float* __restrict__ jpos, const float* __restrict__ jaxis,
    const float* __restrict__ infl, int N, int Jall, int D, int maxE,
    float* __restrict__ g_dofs) {
  const int dof = blockIdx.x, b = blockIdx.y;
  __shared__ float s_part[kDofBlock / 64];
  __shared__ int s_end;
  if (threadIdx.x == 0) s_end = maxE;
  const float* row = infl + (size_t)dof * maxE * 4;
  const float* gb = g_pos + (size_t)b * N * 3;
  const float* sb = skinned + (size_t)b * N * 3;
  float4 cur[kDofPer], next[kDofPer];
  auto load = [&](float4* to, int base) {
#pragma unroll
    for (int k = 0; k < kDofPer; ++k) {
      const int e = base + k * kDofBlock + (int)threadIdx.x;
      if (e >= maxE) { to[k] = make_float4(-1.f, 0.f, 0.f, 0.f); continue; }
      if (kVec)
        to[k] = *reinterpret_cast<const float4*>(row + 4 * (size_t)e);
      else
        to[k] = make_float4(row[4 * (size_t)e], row[4 * (size_t)e + 1], row[4 * (size_t)e + 2], row[4 * (size_t)e + 3]);
    }
  };
  float acc = 0.f;
  load(cur, 0);
  for (int base = 0; base < maxE; base += kDofPer * kDofBlock) {
    int first = maxE;
#pragma unroll
    for (int k = kDofPer - 1; k >= 0; --k)
      if (cur[k].x == -1.f) first = base + k * kDofBlock + (int)threadIdx.x;
    const bool last = __syncthreads_or(first < maxE);
    int end = maxE;
    if (last) {
      if (first < maxE) atomicMin(&s_end, first);
      __syncthreads();
      end = s_end;
    } else {
      load(next, base + kDofPer * kDofBlock);
    }
#pragma unroll
    for (int k = 0; k < kDofPer; ++k) {
      if (base + k * kDofBlock + (int)threadIdx.x >= end) continue;
      const int vtx = (int)cur[k].x, type = (int)cur[k].y, j = (int)cur[k].z;
      const f3 gv = mk3(gb[3 * (size_t)vtx], gb[3 * (size_t)vtx + 1], gb[3 * (size_t)vtx + 2]);
      const float* a = jaxis + ((size_t)b * Jall + j) * 3;
      f3 rd = mk3(a[0], a[1], a[2]);
      if (type == 0) {
        const float* c = jpos + ((size_t)b * Jall + j) * 3;
        const float* vp = sb + 3 * (size_t)vtx;
        rd = cross(rd, mk3(vp[0] - c[0], vp[1] - c[1], vp[2] - c[2]));
      }
      acc += dot(rd * cur[k].w, gv);
    }
    if (last) break;
#pragma unroll
    for (int k = 0; k < kDofPer; ++k) cur[k] = next[k];
  }
  acc = wave_sum(acc);
  if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    float t = 0.f;
    for (int i = 0; i < kDofBlock / 64; ++i) t += s_part[i];
    g_dofs[(size_t)b * D + dof] = t;
  }
}

// The same with the row split over workgroups and kDofPoses poses taken
// together, for callers with a workspace: one workgroup's row of 100k entries
// is the launch's critical path above, and every pose reads the table again
// (24 MB for 57 DOFs of a 25k-vertex body, more than an XCD's L2).  Each
// workgroup leaves its partial sums and the place of the first -1 in its
// part; parts after a row's end are computed (with indices checked, whatever
// they hold) and dropped by the second launch, which adds the others in
// order.  16 poses, 57 DOFs, 25k vertices: 72 us against the 124 of the
// kernel above.
//
// Poses per workgroup: 8 (a table entry serves all of them), but single ones
// below 4 poses, where the other places would repeat the last pose.
constexpr int kDofPoses = 8;
constexpr int kDofPart = 2048;  // entries per workgroup
constexpr int kDofLdsJoints = 128;  // joints staged in LDS (24 KB) up to this many
template <int kP, bool kVec, bool kLds>
__global__ __launch_bounds__(kBlock) void dof_part_kernel(
    const float* __restrict__ g_pos, const float* __restrict__ skinned,
    const float* __restrict__ jpos, const float* __restrict__ jaxis,
    const float* __restrict__ infl, int B, int N, int Jall, int D, int maxE, int parts,
    float* __restrict__ partial, int* __restrict__ ends) {
  const int dof = blockIdx.x / parts, part = blockIdx.x - dof * parts, b0 = blockIdx.y * kP;
  const int nb = min(kP, B - b0), base = part * kDofPart, stop = min(maxE, base + kDofPart);
  __shared__ float s_part[kBlock / 64][kP];
  __shared__ int s_end;
  __shared__ float s_joint[kLds ? kP * kDofLdsJoints * 6 : 1];  // axis, position
  const float* row = infl + (size_t)dof * maxE * 4;
  constexpr int kPer = kDofPart / kBlock;
  float4 ent[kPer];
  int first = stop;
#pragma unroll
  for (int k = kPer - 1; k >= 0; --k) {
    const int e = base + k * kBlock + (int)threadIdx.x;
    ent[k] = make_float4(-1.f, 0.f, 0.f, 0.f);
    if (e >= stop) continue;
    if (kVec)
      ent[k] = *reinterpret_cast<const float4*>(row + 4 * (size_t)e);
    else
      ent[k] = make_float4(row[4 * (size_t)e], row[4 * (size_t)e + 1], row[4 * (size_t)e + 2], row[4 * (size_t)e + 3]);
    if (ent[k].x == -1.f) first = e;
  }
  if (threadIdx.x == 0) s_end = stop;
  __syncthreads();
  if (first < stop) atomicMin(&s_end, first);
  __syncthreads();
  const int end = s_end;
  if (threadIdx.x == 0 && blockIdx.y == 0) ends[blockIdx.x] = end;
  float* out = partial + ((size_t)blockIdx.x * gridDim.y + blockIdx.y) * kP;
  if (end == base) {  // a part behind the row's end
    if (threadIdx.x < kP) out[threadIdx.x] = 0.f;
    return;
  }
  if (kLds) {
    for (int i = threadIdx.x; i < nb * Jall * 3; i += kBlock) {
      const int r = i / 3, c = i - 3 * r;
      s_joint[6 * r + c] = jaxis[(size_t)b0 * Jall * 3 + i];
      s_joint[6 * r + 3 + c] = jpos[(size_t)b0 * Jall * 3 + i];
    }
    __syncthreads();
  }
  float acc[kP];
#pragma unroll
  for (int q = 0; q < kP; ++q) acc[q] = 0.f;
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int vtx = (int)ent[k].x, type = (int)ent[k].y, j = (int)ent[k].z;
    if (base + k * kBlock + (int)threadIdx.x >= end || vtx < 0 || vtx >= N || j < 0 || j >= Jall) continue;
    // all poses' vertices first (past the batch the last pose's again), so the
    // loads overlap
    f3 gv[kP], vp[kP];
#pragma unroll
    for (int q = 0; q < kP; ++q) {
      const size_t at = ((size_t)(b0 + min(q, nb - 1)) * N + vtx) * 3;
      gv[q] = mk3(g_pos[at], g_pos[at + 1], g_pos[at + 2]);
      vp[q] = mk3(skinned[at], skinned[at + 1], skinned[at + 2]);
    }
#pragma unroll
    for (int q = 0; q < kP; ++q) {
      const int r = min(q, nb - 1) * Jall + j;
      const float* ax = kLds ? s_joint + 6 * r : jaxis + ((size_t)b0 * Jall + r) * 3;
      const float* ce = kLds ? ax + 3 : jpos + ((size_t)b0 * Jall + r) * 3;
      f3 rd = mk3(ax[0], ax[1], ax[2]);
      if (type == 0) rd = cross(rd, mk3(vp[q].x - ce[0], vp[q].y - ce[1], vp[q].z - ce[2]));
      acc[q] += dot(rd * ent[k].w, gv[q]);
    }
  }
  static_assert(kP == 8 || kP == 1, "wave_sum8 or wave_sum");
  const float t = kP == 8 ? wave_sum8(acc) : wave_sum(acc[0]);
  if ((threadIdx.x & 63) < kP) s_part[threadIdx.x >> 6][threadIdx.x & 63] = t;
  __syncthreads();
  if (threadIdx.x < kP) {
    float sum = 0.f;
#pragma unroll
    for (int w = 0; w < kBlock / 64; ++w) sum += s_part[w][threadIdx.x];
    out[threadIdx.x] = sum;
  }
}

// One wavefront per (dof, group of poses): the parts up to the row's end, in
// part order for every pose (lane q: pose q).
template <int kP>
__global__ __launch_bounds__(64) void dof_sum_kernel(const float* __restrict__ partial, const int* __restrict__ ends,
                                                     int B, int D, int maxE, int parts, float* __restrict__ g_dofs) {
  const int dof = blockIdx.x, q = threadIdx.x % kP, b = blockIdx.y * kP + q;
  constexpr int kStep = 64 / kP;
  // the first part that holds the row's end
  int last = parts - 1;
  for (int p0 = 0; p0 < parts; p0 += 64) {
    const int p = p0 + (int)threadIdx.x;
    const bool ended = p < parts && ends[(size_t)dof * parts + p] < min(maxE, (p + 1) * kDofPart);
    const unsigned long long m = __ballot(ended);
    if (m) { last = p0 + __ffsll(m) - 1; break; }
  }
  float t = 0.f;
  for (int p = (int)threadIdx.x / kP; p <= last; p += kStep)
    t += partial[(((size_t)dof * parts + p) * gridDim.y + blockIdx.y) * kP + q];
#pragma unroll
  for (int o = kP; o < 64; o <<= 1) t += __shfl_xor(t, o, 64);
  if (threadIdx.x < kP && b < B) g_dofs[(size_t)b * D + dof] = t;
}

template <bool kLds>
__global__ __launch_bounds__(kBlock) void lbs_fwd_kernel(
    const float* __restrict__ trans, const float* __restrict__ weights,
    const int* __restrict__ jidx, const float* __restrict__ rest_pos,
    const float* __restrict__ rest_nrm, const float* __restrict__ disp, int N, int K, int J,
    float* __restrict__ pos, float* __restrict__ nrm, float* __restrict__ trans_out, float* __restrict__ w_out) {
  __shared__ float s_tab[kLds ? kMaxLdsJoints * 12 : 1];
  const int b = blockIdx.y;
  copy_table<12>(trans, trans_out, b, J);
  const float* tab = trans + (size_t)b * J * 12;
  if (kLds) {
    for (int i = threadIdx.x; i < J * 12; i += kBlock) s_tab[i] = tab[i];
    __syncthreads();
    tab = s_tab;
  }
  const int v = blockIdx.x * kBlock + threadIdx.x;
  if (v >= N) return;
  m3 Rb = m3_zero();
  f3 tb = mk3(0.f, 0.f, 0.f);
  const float* wv = weights + ((size_t)b * N + v) * K;
  for (int k = 0; k < K; ++k) {
    const float* T = tab + jidx[(size_t)v * K + k] * 12;
    const float wk = wv[k];
    if (w_out) w_out[((size_t)b * N + v) * K + k] = wk;
    for (int i = 0; i < 9; ++i) Rb.m[i] = Rb.m[i] + T[i] * wk;
    tb = tb + mk3(T[9], T[10], T[11]) * wk;
  }
  const float* dp = disp + ((size_t)b * N + v) * 3;
  f3 p = mk3(rest_pos[3 * v] + dp[0], rest_pos[3 * v + 1] + dp[1], rest_pos[3 * v + 2] + dp[2]);
  f3 o = mul(Rb, p) + tb;
  float* po = pos + ((size_t)b * N + v) * 3;
  po[0] = o.x; po[1] = o.y; po[2] = o.z;
  if (nrm) {
    f3 n = mul(Rb, mk3(rest_nrm[3 * v], rest_nrm[3 * v + 1], rest_nrm[3 * v + 2]));
    float* no = nrm + ((size_t)b * N + v) * 3;
    no[0] = n.x; no[1] = n.y; no[2] = n.z;
  }
}

template <bool kLds>
__global__ __launch_bounds__(kBlock) void lbs_bwd_kernel(
    const float* __restrict__ g_pos, const float* __restrict__ trans,
    const float* __restrict__ weights, const int* __restrict__ jidx,
    const float* __restrict__ rest_pos, const float* __restrict__ disp, int N, int K, int J,
    float* __restrict__ g_w, float* __restrict__ g_disp, float* __restrict__ g_trans,
    int flags, int per) {
  __shared__ float s_tab[kLds ? kMaxLdsJoints * 12 : 1];
  __shared__ float s_acc[kLds ? kMaxLdsJoints * 12 : 1];
  const int b = blockIdx.y;
  const float* tab = trans + (size_t)b * J * 12;
  if (kLds) {
    for (int i = threadIdx.x; i < J * 12; i += kBlock) { s_tab[i] = tab[i]; s_acc[i] = 0.f; }
    __syncthreads();
    tab = s_tab;
  }
  const bool ref = (flags & DCX_FLAG_REF_COMPAT) != 0;
  for (int c = 0; c < per; ++c) {
    const int v0 = (blockIdx.x * per + c) * kBlock + threadIdx.x;
    const bool in = v0 < N;
    const int v = in ? v0 : N - 1;
    const float* gp = g_pos + ((size_t)b * N + v) * 3;
    f3 g = mk3(gp[0], gp[1], gp[2]);
    const float* dp = disp + ((size_t)b * N + v) * 3;
    f3 base = mk3(rest_pos[3 * v], rest_pos[3 * v + 1], rest_pos[3 * v + 2]);
    f3 p = mk3(base.x + dp[0], base.y + dp[1], base.z + dp[2]);
    const float* wv = weights + ((size_t)b * N + v) * K;
    m3 Rb = m3_zero();
    for (int k = 0; k < K; ++k) {
      const int j = jidx[(size_t)v * K + k];
      if (g_w && in) {
        // Reference: joint index = slot index, rest position without displacement.
        const float* T = ref ? trans + ((size_t)b * J + k) * 12 : tab + j * 12;
        f3 pp = ref ? base : p;
        m3 R; for (int i = 0; i < 9; ++i) R.m[i] = T[i];
        g_w[((size_t)b * N + v) * K + k] = dot(mul(R, pp) + mk3(T[9], T[10], T[11]), g);
      }
      if (g_disp) {
        if (ref) {
          const float wr = weights[(size_t)v * K + k];  // batch-0 weights
          if (!(wr < 1e-4f)) {
            const float* T = trans + ((size_t)b * J + k) * 12;
            for (int i = 0; i < 9; ++i) Rb.m[i] += T[i] * wr;
          }
        } else {
          const float* T = tab + j * 12;
          for (int i = 0; i < 9; ++i) Rb.m[i] += T[i] * wv[k];
        }
      }
    }
    if (g_trans) {
      const float gt[12] = {g.x * p.x, g.x * p.y, g.x * p.z, g.y * p.x, g.y * p.y, g.y * p.z,
                            g.z * p.x, g.z * p.y, g.z * p.z, g.x, g.y, g.z};
      // kMaxK slots at a time (the op takes any number)
      for (int k0 = 0; k0 < K; k0 += kMaxK) {
        const int n = min(K - k0, kMaxK);
        int idx[kMaxK];
        float coef[kMaxK];
#pragma unroll
        for (int k = 0; k < kMaxK; ++k) {
          idx[k] = k < n ? jidx[(size_t)v * K + k0 + k] : 0;
          coef[k] = k < n ? wv[k0 + k] : 0.f;
        }
        if (kLds) {
          add_joint_grads<12, 0>(s_acc, in, idx, coef, gt, n);
        } else if (in) {
          for (int k = 0; k < n; ++k)
            for (int e = 0; e < 12; ++e) atomicAdd(g_trans + ((size_t)b * J + idx[k]) * 12 + e, gt[e] * coef[k]);
        }
      }
    }
    if (g_disp && in) {
      f3 gd = mulT(Rb, g);
      float* o = g_disp + ((size_t)b * N + v) * 3;
      o[0] = gd.x; o[1] = gd.y; o[2] = gd.z;
    }
  }
  if (kLds && g_trans) {
    __syncthreads();
    acc_flush(s_acc, J * 12, g_trans + (size_t)b * J * 12);
  }
}

__global__ __launch_bounds__(kBlock) void clear_f_kernel(float* __restrict__ p, long long n) {
  const long long i = (long long)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) p[i] = 0.f;
}
dcx_status clear_f(float* p, long long n, hipStream_t s) {
  hipLaunchKernelGGL(clear_f_kernel, dim3(ceil_div(n, kBlock)), dim3(kBlock), 0, s, p, n);
  return check_launch("clear");
}

bool vec16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// Vertex blocks per workgroup of the backward passes: where there are several
// workgroups a CU anyway, four blocks share one flush of the joint gradients.
int blocks_per_group(int B, int N) { return (long long)ceil_div(N, kBlock) * B >= 1024 ? 4 : 1; }

}  // namespace
}  // namespace dcx

using namespace dcx;

extern "C" dcx_status dcx_dqs_fwd(const float* dq, const float* weights, const int32_t* joint_idx,
                                  const float* rest_pos, const float* rest_nrm, int B, int N,
                                  int K, int J, float* pos, float* nrm, float* dq_out,
                                  float* w_out, void* stream) {
  DCX_REQUIRE(B > 0 && N > 0 && J > 0, "dcx_dqs_fwd: bad sizes B=%d N=%d J=%d", B, N, J);
  DCX_REQUIRE(K >= 1 && K <= kMaxK, "dcx_dqs_fwd: K=%d outside [1,%d]", K, kMaxK);
  DCX_REQUIRE(dq && weights && joint_idx && rest_pos && pos, "dcx_dqs_fwd: null input");
  DCX_REQUIRE(!nrm || rest_nrm, "dcx_dqs_fwd: normals requested without rest normals");
  hipStream_t s = as_stream(stream);
  dim3 grid(ceil_div(N, kBlock), B);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(kBlock), 0, s, dq, weights, joint_idx, rest_pos, rest_nrm, N, K, J, pos, nrm,
                       dq_out, w_out);
  };
  if (J > kMaxLdsJoints) launch(dqs_fwd_kernel<false, 0>);
  else if (K == 4 && vec16(weights) && vec16(joint_idx) && vec16(w_out)) launch(dqs_fwd_kernel<true, 4>);
  else launch(dqs_fwd_kernel<true, 0>);
  return check_launch("dcx_dqs_fwd");
}

extern "C" dcx_status dcx_dqs_bwd(const float* g_pos, const float* g_nrm, const float* dq,
                                  const float* weights, const int32_t* joint_idx,
                                  const float* rest_pos, const float* rest_nrm, int B, int N,
                                  int K, int J, float* g_dq, float* g_w, float* g_rest,
                                  int flags, void* stream) {
  DCX_REQUIRE(B > 0 && N > 0 && J > 0, "dcx_dqs_bwd: bad sizes B=%d N=%d J=%d", B, N, J);
  DCX_REQUIRE(K >= 1 && K <= kMaxK, "dcx_dqs_bwd: K=%d outside [1,%d]", K, kMaxK);
  DCX_REQUIRE(g_pos && dq && weights && joint_idx && rest_pos, "dcx_dqs_bwd: null input");
  DCX_REQUIRE(!g_nrm || rest_nrm, "dcx_dqs_bwd: normal gradient without rest normals");
  hipStream_t s = as_stream(stream);
  if (g_dq)
    if (dcx_status e = clear_f(g_dq, 8ll * J * B, s)) return e;
  const int per = blocks_per_group(B, N);
  dim3 grid(ceil_div(N, kBlock * per), B);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(kBlock), 0, s, g_pos, g_nrm, dq, weights, joint_idx, rest_pos, rest_nrm, N, K,
                       J, g_dq, g_w, g_rest, flags, per);
  };
  if (J > kMaxLdsJoints) launch(dqs_bwd_kernel<false, 0>);
  else if (K == 4 && vec16(weights) && vec16(joint_idx) && vec16(g_w)) launch(dqs_bwd_kernel<true, 4>);
  else launch(dqs_bwd_kernel<true, 0>);
  return check_launch("dcx_dqs_bwd");
}

extern "C" dcx_status dcx_dof_grad(const float* g_pos, const float* skinned_pos,
                                   const float* joint_pos, const float* joint_axis,
                                   const float* influence, int B, int N, int Jall, int D,
                                   int max_entries, float* g_dofs, void* stream) {
  DCX_REQUIRE(B > 0 && N > 0 && Jall > 0 && D > 0 && max_entries > 0,
              "dcx_dof_grad: bad sizes B=%d N=%d Jall=%d D=%d E=%d", B, N, Jall, D, max_entries);
  DCX_REQUIRE(g_pos && skinned_pos && joint_pos && joint_axis && influence && g_dofs,
              "dcx_dof_grad: null pointer");
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(D, B), dim3(kDofBlock), 0, as_stream(stream), g_pos, skinned_pos, joint_pos,
                       joint_axis, influence, N, Jall, D, max_entries, g_dofs);
  };
  if (vec16(influence)) launch(dof_grad_kernel<true>);
  else launch(dof_grad_kernel<false>);
  return check_launch("dcx_dof_grad");
}

static int dof_poses(int B) { return B >= 4 ? kDofPoses : 1; }
static int dof_parts(int max_entries) { return (max_entries + kDofPart - 1) / kDofPart; }

extern "C" size_t dcx_dof_grad_workspace_size(int B, int D, int max_entries) {
  if (B <= 0 || D <= 0 || max_entries <= 0) return 0;
  const size_t parts = (size_t)D * dof_parts(max_entries);
  return parts * (sizeof(int) + sizeof(float) * dof_poses(B) * ceil_div(B, dof_poses(B)));
}

extern "C" dcx_status dcx_dof_grad_split(const float* g_pos, const float* skinned_pos, const float* joint_pos,
                                         const float* joint_axis, const float* influence, int B, int N, int Jall, int D,
                                         int max_entries, float* g_dofs, void* workspace, size_t workspace_bytes,
                                         void* stream) {
  DCX_REQUIRE(B > 0 && N > 0 && Jall > 0 && D > 0 && max_entries > 0,
              "dcx_dof_grad_split: bad sizes B=%d N=%d Jall=%d D=%d E=%d", B, N, Jall, D, max_entries);
  DCX_REQUIRE(g_pos && skinned_pos && joint_pos && joint_axis && influence && g_dofs, "dcx_dof_grad_split: null pointer");
  DCX_REQUIRE(workspace && workspace_bytes >= dcx_dof_grad_workspace_size(B, D, max_entries),
              "dcx_dof_grad_split: workspace too small");
  const int parts = dof_parts(max_entries);
  const unsigned groups = ceil_div(B, dof_poses(B));
  int* ends = (int*)workspace;
  float* partial = (float*)(ends + (size_t)D * parts);
  hipStream_t s = as_stream(stream);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)D * parts, groups), dim3(kBlock), 0, s, g_pos, skinned_pos, joint_pos,
                       joint_axis, influence, B, N, Jall, D, max_entries, parts, partial, ends);
  };
  const bool vec = vec16(influence), lds = Jall <= kDofLdsJoints;
  auto pick = [&](auto poses) {
    constexpr int kP = decltype(poses)::value;
    if (vec && lds) launch(dof_part_kernel<kP, true, true>);
    else if (vec) launch(dof_part_kernel<kP, true, false>);
    else if (lds) launch(dof_part_kernel<kP, false, true>);
    else launch(dof_part_kernel<kP, false, false>);
    hipLaunchKernelGGL(dof_sum_kernel<kP>, dim3(D, groups), dim3(64), 0, s, partial, ends, B, D, max_entries, parts,
                       g_dofs);
  };
  if (dof_poses(B) == kDofPoses) pick(std::integral_constant<int, kDofPoses>{});
  else pick(std::integral_constant<int, 1>{});
  return check_launch("dcx_dof_grad_split");
}

extern "C" dcx_status dcx_lbs_fwd(const float* transforms, const float* weights,
                                  const int32_t* joint_idx, const float* rest_pos,
                                  const float* rest_nrm, const float* disp, int B, int N, int K,
                                  int J, float* pos, float* nrm, float* trans_out, float* w_out,
                                  void* stream) {
  DCX_REQUIRE(B > 0 && N > 0 && J > 0 && K >= 1, "dcx_lbs_fwd: bad sizes");
  DCX_REQUIRE(transforms && weights && joint_idx && rest_pos && disp && pos,
              "dcx_lbs_fwd: null input");
  DCX_REQUIRE(!nrm || rest_nrm, "dcx_lbs_fwd: normals requested without rest normals");
  hipStream_t s = as_stream(stream);
  dim3 grid(ceil_div(N, kBlock), B);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(kBlock), 0, s, transforms, weights, joint_idx, rest_pos, rest_nrm, disp, N, K,
                       J, pos, nrm, trans_out, w_out);
  };
  if (J <= kMaxLdsJoints) launch(lbs_fwd_kernel<true>);
  else launch(lbs_fwd_kernel<false>);
  return check_launch("dcx_lbs_fwd");
}

extern "C" dcx_status dcx_lbs_bwd(const float* g_pos, const float* transforms,
                                  const float* weights, const int32_t* joint_idx,
                                  const float* rest_pos, const float* disp, int B, int N, int K,
                                  int J, float* g_w, float* g_disp, float* g_trans, int flags,
                                  void* stream) {
  DCX_REQUIRE(B > 0 && N > 0 && J > 0 && K >= 1, "dcx_lbs_bwd: bad sizes");
  DCX_REQUIRE(g_pos && transforms && weights && joint_idx && rest_pos && disp,
              "dcx_lbs_bwd: null input");
  DCX_REQUIRE(!(flags & DCX_FLAG_REF_COMPAT) || K <= J,
              "dcx_lbs_bwd: reference mode indexes joints by slot and needs K <= J");
  hipStream_t s = as_stream(stream);
  if (g_trans)
    if (dcx_status e = clear_f(g_trans, 12ll * J * B, s)) return e;
  const int per = blocks_per_group(B, N);
  dim3 grid(ceil_div(N, kBlock * per), B);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(kBlock), 0, s, g_pos, transforms, weights, joint_idx, rest_pos, disp, N, K, J,
                       g_w, g_disp, g_trans, flags, per);
  };
  if (J <= kMaxLdsJoints) launch(lbs_bwd_kernel<true>);
  else launch(lbs_bwd_kernel<false>);
  return check_launch("dcx_lbs_bwd");
}
