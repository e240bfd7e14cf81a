"""GPU parity of the skinning kernels against the oracle (called through the C ABI)."""
import numpy as np
import pytest
import torch

from deepcharacters_amd import scenes, skinning
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

RTOL = 1e-5  # float outputs vs FP64 oracle, relative to the output's scale


def _t(a, dtype=torch.float32):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=dtype, device="cuda")


def _rel(a, b):
    a = np.asarray(a, np.float64)
    b = np.asarray(b, np.float64)
    return float(np.abs(a - b).max() / max(np.abs(b).max(), 1e-30))


def rig(seed, N=3000, J=24, K=4, B=3):
    ch = scenes.ellipsoid_character(3, seed=seed, n_joints=J, K=K)
    rng = np.random.default_rng(seed)
    dq = scenes.random_joint_dqs(rng, ch.joint_centres, B)
    w = np.broadcast_to(ch.joint_w, (B, ch.N, K)).copy()
    w *= rng.uniform(0.5, 1.5, size=w.shape)  # per-batch weights differ
    return ch, dq, w


@pytest.mark.parametrize("seed", [0, 1])
def test_dqs_forward_matches_oracle(seed):
    ch, dq, w = rig(seed)
    pos, nrm, dq_out, w_out = skinning.dq_skinning_gpu(_t(dq), _t(w), _t(ch.joint_idx, torch.int32),
                                                        _t(ch.verts), _t(ch.normals))
    rp, rn = orc.dqs_fwd(dq, w, ch.joint_idx, ch.verts, ch.normals)
    assert _rel(pos.cpu(), rp) < RTOL
    assert _rel(nrm.cpu(), rn) < RTOL
    assert torch.equal(dq_out.cpu(), torch.as_tensor(dq, dtype=torch.float32))
    assert torch.equal(w_out.cpu(), torch.as_tensor(w, dtype=torch.float32))


@pytest.mark.parametrize("ref_compat", [False, True])
def test_dqs_backward_matches_oracle(ref_compat):
    ch, dq, w = rig(3)
    rng = np.random.default_rng(9)
    gp = rng.normal(size=(dq.shape[0], ch.N, 3))
    gn = rng.normal(size=(dq.shape[0], ch.N, 3))
    g_dq, g_w, g_r = skinning.dq_skinning_backward(
        _t(gp), _t(dq), _t(w), _t(ch.joint_idx, torch.int32), _t(ch.verts), _t(ch.normals),
        g_nrm=None if ref_compat else _t(gn), ref_compat=ref_compat, need_rest=True)
    o_dq, o_w, o_r = orc.dqs_bwd(gp, dq, w, ch.joint_idx, ch.verts, ch.normals,
                                 g_nrm=None if ref_compat else gn, ref_compat=ref_compat)
    assert _rel(g_w.cpu(), o_w) < 1e-5
    assert _rel(g_r.cpu(), o_r) < 1e-5
    # joint reduction over ~N*K/J terms: fp32 accumulation tolerance
    assert _rel(g_dq.cpu(), o_dq) < 1e-4


def test_dqs_edge_cases():
    # K=1, J=1, zero weights (|b_r| below the normalisation threshold), N not a multiple of 256
    N = 257
    rng = np.random.default_rng(1)
    v = rng.normal(size=(N, 3))
    n = scenes.random_unit(rng, (N,))
    ji = np.zeros((N, 1), np.int32)
    w = np.zeros((1, N, 1))
    w[0, ::2, 0] = 1.0
    dq = scenes.random_joint_dqs(rng, np.zeros((1, 3)), 1)
    pos, nrm, _, _ = skinning.dq_skinning_gpu(_t(dq), _t(w), _t(ji, torch.int32), _t(v), _t(n))
    rp, rn = orc.dqs_fwd(dq, w, ji, v, n)
    assert _rel(pos.cpu(), rp) < 1e-5
    assert np.isfinite(nrm.cpu().numpy()).all()


def test_lbs_forward_backward_match_oracle():
    rng = np.random.default_rng(5)
    N, J, K, B = 2000, 20, 4, 2
    v = rng.normal(size=(N, 3))
    n = scenes.random_unit(rng, (N,))
    ji = np.stack([rng.permutation(J)[:K] for _ in range(N)]).astype(np.int32)
    w = rng.uniform(0.0, 1.0, size=(B, N, K))
    tr = rng.normal(size=(B, J, 12))
    disp = rng.normal(size=(B, N, 3)) * 0.01
    pos, nrm, tr_out, w_out = skinning.lb_skinning_gpu(_t(tr), _t(w), _t(ji, torch.int32), _t(v),
                                                       _t(n), _t(disp))
    rp, rn = orc.lbs_fwd(tr, w, ji, v, n, disp)
    assert _rel(pos.cpu(), rp) < 1e-5 and _rel(nrm.cpu(), rn) < 1e-5
    gp = rng.normal(size=(B, N, 3))
    for ref in (False, True):
        g_w, g_d, g_t = skinning.lb_skinning_backward(_t(gp), _t(tr), _t(w), _t(ji, torch.int32),
                                                      _t(v), _t(disp), ref_compat=ref)
        o_w, o_d, o_t = orc.lbs_bwd(gp, tr, w, ji, v, disp, ref_compat=ref)
        assert _rel(g_w.cpu(), o_w) < 1e-5
        assert _rel(g_d.cpu(), o_d) < 1e-5
        assert _rel(g_t.cpu(), o_t) < 1e-4


def test_dof_grad_matches_oracle():
    rng = np.random.default_rng(6)
    B, N, Jall, D, E = 2, 500, 6, 7, 900
    gp = rng.normal(size=(B, N, 3))
    sp = rng.normal(size=(B, N, 3))
    jp = rng.normal(size=(B, Jall, 3))
    ja = scenes.random_unit(rng, (B, Jall))
    infl = np.full((D, E, 4), -1.0)
    for d in range(D):
        m = rng.integers(0, E + 1) if d else E  # one row completely full (no terminator)
        infl[d, :m, 0] = rng.integers(0, N, m)
        infl[d, :m, 1] = rng.integers(0, 3, m)
        infl[d, :m, 2] = rng.integers(0, Jall, m)
        infl[d, :m, 3] = rng.uniform(0, 1, m)
    out = skinning.dof_grad(_t(gp), _t(sp), _t(jp), _t(ja), _t(infl))
    ref = orc.dof_grad(gp, sp, jp, ja, infl)
    assert _rel(out.cpu(), ref) < 1e-5


def test_autograd_matches_finite_differences_fp64_oracle():
    ch, dq, w = rig(4, B=1)
    t_dq = _t(dq).requires_grad_(True)
    t_w = _t(w).requires_grad_(True)
    pos = skinning.DQSkinFn.apply(t_dq, t_w, _t(ch.verts), _t(ch.joint_idx, torch.int32))
    gp = torch.randn_like(pos)
    (pos * gp).sum().backward()
    gpn = gp.cpu().double().numpy()
    h = 1e-6
    flat = dq.reshape(-1)
    idxs = np.random.default_rng(0).choice(flat.size, 24, replace=False)
    for i in idxs:
        old = flat[i]
        flat[i] = old + h
        lp = np.sum(orc.dqs_fwd(dq, w, ch.joint_idx, ch.verts)[0] * gpn)
        flat[i] = old - h
        lm = np.sum(orc.dqs_fwd(dq, w, ch.joint_idx, ch.verts)[0] * gpn)
        flat[i] = old
        fd = (lp - lm) / (2 * h)
        got = float(t_dq.grad.reshape(-1)[i])
        assert abs(got - fd) <= 1e-4 * max(1.0, abs(fd)), (i, got, fd)


@pytest.mark.parametrize("B,E,Jall", [(1, 1, 1), (8, 2048, 3), (9, 2049, 128), (3, 4500, 129), (17, 70, 5)])
def test_split_dof_grad_at_the_edges_of_parts_poses_and_joints(B, E, Jall):
    """Rows that end before, at and after the end of a part, with entries after
    the end that name no vertex; the one-workgroup-a-row entry as well.  Sums
    of up to E products of order 1 in 32 bits: within E * 2^-24 of their size."""
    rng = np.random.default_rng(B * 1000 + E)
    N, D = 300, 6
    gp, sp = rng.normal(size=(B, N, 3)), rng.normal(size=(B, N, 3))
    jp, ja = rng.normal(size=(B, Jall, 3)), scenes.random_unit(rng, (B, Jall))
    infl = np.full((D, E, 4), 1e9)  # nothing behind a row's end may be read as a vertex
    for d, m in enumerate([E, 0, min(E, 2048), min(E, 2047), E // 2, max(E - 1, 0)]):
        infl[d, :m, 0] = rng.integers(0, N, m)
        infl[d, :m, 1] = rng.integers(0, 2, m)
        infl[d, :m, 2] = rng.integers(0, Jall, m)
        infl[d, :m, 3] = rng.uniform(0, 1, m)
        if m < E:
            infl[d, m, 0] = -1
    args = [_t(a) for a in (gp, sp, jp, ja, infl)]
    out = skinning.dof_grad(*args)
    ref = orc.dof_grad(*[a.cpu().numpy() for a in args])
    one = torch.empty_like(out)
    from deepcharacters_amd import _lib
    _lib.call("dcx_dof_grad", *[a.data_ptr() for a in args], B, N, Jall, D, E, one.data_ptr(),
              torch.cuda.current_stream().cuda_stream)
    for got in (out, one):
        assert np.abs(got.cpu().numpy() - ref).max() <= 4e-6 * max(1.0, np.sqrt(E))


@pytest.mark.parametrize("N,J,K,order", [(1, 1, 4, "one"), (64, 5, 4, "few"), (257, 256, 4, "random"),
                                         (300, 257, 4, "random"), (1000, 40, 3, "random"), (513, 30, 8, "random")])
def test_joint_gradients_of_ordered_and_unordered_skinnings(N, J, K, order):
    """Few joints a wavefront (summed in registers), more than it goes through
    (the rest added one by one), more than LDS holds; sums of about N K / J
    products in 32 bits."""
    rng = np.random.default_rng(N + J)
    B = 2
    ji = {"one": np.zeros((N, K)), "few": np.arange(N)[:, None] // 40 + np.arange(K) % 3,
          "random": rng.integers(0, J, (N, K))}[order].astype(np.int32) % J
    dq = scenes.random_joint_dqs(rng, rng.normal(size=(J, 3)), B, 0.4)
    w, v, g = rng.uniform(0.1, 1, (B, N, K)), rng.normal(size=(N, 3)), rng.normal(size=(B, N, 3))
    g_dq, g_w, g_r = skinning.dq_skinning_backward(_t(g), _t(dq), _t(w), _t(ji, torch.int32), _t(v), need_rest=True)
    o_dq, o_w, o_r = orc.dqs_bwd(g, dq, w, ji, v)
    assert _rel(g_dq.cpu(), o_dq) < 1e-4 and _rel(g_r.cpu(), o_r) < 1e-5
    # a weight's gradient is a dot product with the joint's gradient, exactly 0
    # where one joint has all the weight: its rounding is relative to the factors
    assert np.abs(g_w.cpu().numpy() - o_w).max() < 1e-5 * max(np.abs(o_w).max(), np.abs(o_dq).max())
    tr, disp = rng.normal(size=(B, J, 12)), 0.01 * rng.normal(size=(B, N, 3))
    g_w, g_d, g_t = skinning.lb_skinning_backward(_t(g), _t(tr), _t(w), _t(ji, torch.int32), _t(v), _t(disp))
    o_w, o_d, o_t = orc.lbs_bwd(g, tr, w, ji, v, disp)
    assert _rel(g_t.cpu(), o_t) < 1e-4 and _rel(g_w.cpu(), o_w) < 1e-5 and _rel(g_d.cpu(), o_d) < 1e-5
    # an infinite gradient of one vertex reaches its own joints only
    g[0, 0] = np.inf
    got = skinning.dq_skinning_backward(_t(g), _t(dq), _t(w), _t(ji, torch.int32), _t(v))[0].cpu().numpy()
    mine = np.isin(np.arange(J), ji[0])
    assert np.isfinite(got[1]).all() and np.isfinite(got[0][~mine]).all() and not np.isfinite(got[0][mine]).all()
