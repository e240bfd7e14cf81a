"""GPU embedded-graph op parity against the oracle (through the C ABI)."""
import numpy as np
import pytest
import torch

from deepcharacters_amd import embedded_graph as edm
from deepcharacters_amd import renderer, scenes
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _t(a, dtype=torch.float32):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=dtype, device="cuda")


def _rel(a, b):
    return float(np.abs(np.asarray(a, np.float64) - b).max() / max(np.abs(b).max(), 1e-30))


def setup(seed=0, subdiv=4, M=300, B=3, markers=True):
    ch = scenes.ellipsoid_character(subdiv, seed=seed)
    g = scenes.embedded_graph(ch.verts, M, 4, 0.06)
    rng = np.random.default_rng(seed)
    dT = rng.normal(size=(B, M, 3)) * 0.01
    dA = rng.uniform(-0.2, 0.2, size=(B, M, 3))
    sT = rng.normal(size=(B, M, 3)) * 0.05
    sA = rng.uniform(-0.5, 0.5, size=(B, M, 3))
    disp = rng.normal(size=(B, ch.N, 3)) * 0.002
    mk_node = (np.array([1, 10, 50, 120]) % M).astype(np.int32) if markers else None
    bm = ch.verts[g.node_vertex[mk_node]] + 0.01 if markers else None
    topo = renderer.Topology(ch.faces, ch.N)
    gd = edm.GraphData(ch.verts, g, bm, mk_node, topo)
    return ch, g, gd, (dT, dA, sT, sA, disp), mk_node, bm, rng


@pytest.mark.parametrize("seed", [0, 1])
def test_ed_forward_matches_oracle(seed):
    ch, g, gd, (dT, dA, sT, sA, disp), mk_node, bm, _ = setup(seed)
    verts, nrms, mk, graph, a_out, s_out = edm.embedded_graph_gpu(gd, _t(dT), _t(dA), _t(sT), _t(sA), _t(disp))
    ov, on, omk, og = orc.ed_fwd(g, ch.verts, dT, dA, sT, sA, disp, faces=ch.faces, base_markers=bm,
                                 marker_node=mk_node)
    assert _rel(verts.cpu(), ov) < 1e-5
    assert _rel(mk.cpu(), omk) < 1e-5
    assert _rel(graph.cpu(), og) < 1e-5
    assert np.abs(nrms.cpu().numpy() - on).max() < 2e-4  # unit vectors from float face sums
    assert torch.equal(a_out.cpu(), torch.as_tensor(dA, dtype=torch.float32))
    assert torch.equal(s_out.cpu(), torch.as_tensor(sA, dtype=torch.float32))


def test_ed_backward_matches_oracle():
    ch, g, gd, (dT, dA, sT, sA, disp), mk_node, bm, rng = setup(2)
    B = dT.shape[0]
    gv = rng.normal(size=(B, ch.N, 3))
    gm = rng.normal(size=(B, 4, 3))
    gT, gR, gsT, gsR, gdp = edm.embedded_graph_gpu_grad(gd, _t(gv), _t(gm), _t(dA), _t(sA))
    node_marker = np.full(g.num_nodes, -1, np.int32)
    node_marker[mk_node] = np.arange(4)
    o = orc.ed_bwd(g, ch.verts, gv, dA, sA, g_markers=gm, base_markers=bm, node_marker=node_marker)
    for got, ref in zip((gT, gR, gsT, gsR, gdp), o):
        if not ref.any():
            assert not got.cpu().numpy().any()
        else:
            assert _rel(got.cpu(), ref) < 1e-5


def test_ed_autograd_wrapper_and_finite_differences():
    ch, g, gd, (dT, dA, sT, sA, disp), mk_node, bm, rng = setup(3, subdiv=3, M=60, B=1)
    tdT, tdA = _t(dT).requires_grad_(True), _t(dA).requires_grad_(True)
    tsT, tsA, tdisp = _t(sT).requires_grad_(True), _t(sA).requires_grad_(True), _t(disp).requires_grad_(True)
    op = edm.EmbeddedGraphGpu(gd, 1, tdT, tdA, tsT, tsA, tdisp, refinement=False, nodeName="eg")
    v, n, mk, graph = op.getNode()
    gv = torch.randn_like(v)
    (v * gv).sum().backward()
    assert tsT.grad is not None and torch.count_nonzero(tsT.grad) == 0  # reference: zero skinned grads
    gvn = gv.cpu().double().numpy()
    h = 1e-6
    for arr, grad in ((dT, tdT.grad), (dA, tdA.grad)):
        flat = arr.reshape(-1)
        for i in np.random.default_rng(0).choice(flat.size, 12, replace=False):
            old = flat[i]
            flat[i] = old + h
            lp = np.sum(orc.ed_fwd(g, ch.verts, dT, dA, sT, sA, disp)[0] * gvn)
            flat[i] = old - h
            lm = np.sum(orc.ed_fwd(g, ch.verts, dT, dA, sT, sA, disp)[0] * gvn)
            flat[i] = old
            fd = (lp - lm) / (2 * h)
            got = float(grad.reshape(-1)[i])
            assert abs(got - fd) <= 1e-4 * max(1.0, abs(fd)), (i, got, fd)


def test_ed_edge_cases():
    """Vertices with a single node, a node with no vertices, no markers."""
    rng = np.random.default_rng(4)
    N, M = 37, 9
    base = rng.normal(size=(N, 3))
    node_vertex = rng.choice(N, M, replace=False).astype(np.int32)
    counts = rng.integers(1, 4, N)
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    nodes = np.concatenate([rng.choice(M - 1, c, replace=False) for c in counts]).astype(np.int32)  # node M-1 unused
    w = rng.uniform(0.1, 1, offsets[-1])
    g = scenes.EmbeddedGraph(node_vertex, offsets, nodes, w)
    gd = edm.GraphData(base, g)
    B = 2
    dT, dA = rng.normal(size=(B, M, 3)) * 0.1, rng.normal(size=(B, M, 3)) * 0.3
    sT, sA = rng.normal(size=(B, M, 3)) * 0.1, rng.normal(size=(B, M, 3)) * 0.3
    disp = rng.normal(size=(B, N, 3)) * 0.01
    v, _, _, gr, _, _ = edm.embedded_graph_gpu(gd, _t(dT), _t(dA), _t(sT), _t(sA), _t(disp))
    ov, _, _, og = orc.ed_fwd(g, base, dT, dA, sT, sA, disp)
    assert _rel(v.cpu(), ov) < 1e-5 and _rel(gr.cpu(), og) < 1e-5
    gv = rng.normal(size=(B, N, 3))
    out = edm.embedded_graph_gpu_grad(gd, _t(gv), None, _t(dA), _t(sA))
    ref = orc.ed_bwd(g, base, gv, dA, sA)
    assert _rel(out[0].cpu(), ref[0]) < 1e-5 and _rel(out[1].cpu(), ref[1]) < 1e-5
    assert float(out[0][:, M - 1].abs().max()) == 0.0


def _arap_graph(seed, M=120, k=6):
    ch = scenes.capsule_body(3000, seed=seed, ed_nodes=M)
    nv = ch.graph.node_vertex.astype(np.int32)
    off, size, idx = scenes.node_neighbours(ch.verts, nv, k=k)
    rig = np.random.default_rng(seed).uniform(0.5, 2.0, len(nv))
    return ch.verts, nv, off, size, idx, rig


def test_arap_forward_backward_and_autograd_match_oracle():
    base, nv, off, size, idx, rig = _arap_graph(3)
    g = edm.ArapGraph(base, nv, off, size, idx, rig)
    M, C = len(nv), g.max_conn
    rng = np.random.default_rng(5)
    dT = rng.normal(0, 0.03, (2, M, 3)).astype(np.float32)
    dA = rng.normal(0, 0.3, (2, M, 3)).astype(np.float32)
    res, cw, rot = edm.embedded_graph_arap_gpu(g, torch.as_tensor(dT, device="cuda"),
                                                          torch.as_tensor(dA, device="cuda"))
    rres, rcw = orc.arap_fwd(base, nv, off, size, idx, rig, dT, dA, C)
    assert float(np.abs(res.cpu().numpy() - rres).max()) < 1e-6
    assert np.allclose(cw.cpu().numpy(), rcw, rtol=1e-6, atol=0)
    assert torch.equal(rot.cpu(), torch.as_tensor(dA))
    G = rng.normal(size=(2, M, C, 3)).astype(np.float32)
    for j in range(M):
        G[:, j, size[j]:] = 0.0
    gT, gA = edm.embedded_graph_arap_gpu_grad(g, torch.as_tensor(G, device="cuda"), rot)
    rT, rA = orc.arap_bwd(base, nv, off, size, idx, G, dA)
    rel = lambda a, b: float(np.abs(a.cpu().numpy() - b).max() / np.abs(b).max())
    assert rel(gT, rT) < 1e-5 and rel(gA, rA) < 1e-5
    # autograd: L = sum(w * |r|^2) through ArapFn
    t = torch.as_tensor(dT, device="cuda").requires_grad_(True)
    a = torch.as_tensor(dA, device="cuda").requires_grad_(True)
    r, w = edm.ArapFn.apply(t, a, g)
    (w[..., None] * r * r).sum().backward()
    Gw = (2 * rcw[..., None] * rres)
    rT2, rA2 = orc.arap_bwd(base, nv, off, size, idx, Gw, dA)
    assert float(np.abs(t.grad.cpu().numpy() - rT2).max() / np.abs(rT2).max()) < 1e-5
    assert float(np.abs(a.grad.cpu().numpy() - rA2).max() / np.abs(rA2).max()) < 1e-5


def test_arap_truncates_neighbour_lists_at_max_connections():
    base, nv, off, size, idx, rig = _arap_graph(4, M=80)
    C = int(size.max()) - 2
    g = edm.ArapGraph(base, nv, off, size, idx, rig, max_conn=C)
    rng = np.random.default_rng(6)
    dT = rng.normal(0, 0.03, (1, len(nv), 3)).astype(np.float32)
    dA = rng.normal(0, 0.3, (1, len(nv), 3)).astype(np.float32)
    res, cw, rot = edm.embedded_graph_arap_gpu(g, torch.as_tensor(dT, device="cuda"),
                                                          torch.as_tensor(dA, device="cuda"))
    rres, rcw = orc.arap_fwd(base, nv, off, size, idx, rig, dT, dA, C)
    assert float(np.abs(res.cpu().numpy() - rres).max()) < 1e-6
    G = rng.normal(size=(1, len(nv), C, 3)).astype(np.float32)
    gT, gA = edm.embedded_graph_arap_gpu_grad(g, torch.as_tensor(G, device="cuda"), rot)
    assert torch.isfinite(gT).all() and torch.isfinite(gA).all()


def test_normals_of_vertices_with_many_faces():
    """Fans of 1 to 130 faces round a hub: lists at the edges of the batched and
    of the whole-wavefront sums.  A sum of k terms in 32 bits is within
    (k - 1) eps of the sum of their lengths; the face normals add a few eps each."""
    degrees = [1, 3, 4, 5, 15, 16, 17, 63, 64, 65, 128, 130] * 3
    rng = np.random.default_rng(8)
    verts, faces = [], []
    for k in degrees:
        a = 2 * np.pi * np.arange(k + 1) / (k + 1)
        hub = len(verts)
        verts += [[0, 0, 0.4]] + [[np.cos(x), np.sin(x), rng.uniform(-0.2, 0.2)] for x in a]
        faces += [[hub, hub + 1 + j, hub + 2 + j] for j in range(k)]
    verts, faces = np.array(verts, np.float32), np.array(faces, np.int32)
    N, B = len(verts), 3
    g = scenes.EmbeddedGraph(np.zeros(1, np.int32), np.arange(N + 1, dtype=np.int32), np.zeros(N, np.int32),
                             np.ones(N, np.float32))
    gd = edm.GraphData(verts, g, topology=renderer.Topology(faces, N))
    z = torch.zeros((B, 1, 3), device="cuda")
    v, n, *_ = edm.embedded_graph_gpu(gd, z, z, z, _t(rng.uniform(-1, 1, (B, 1, 3))),
                                      _t(rng.normal(0, 0.05, (B, N, 3))))
    v, n = v.cpu().numpy().astype(np.float64), n.cpu().numpy()
    for b in range(B):
        p = v[b][faces]
        fn = np.cross(p[:, 1] - p[:, 0], p[:, 2] - p[:, 0])
        s, scale = np.zeros((N, 3)), np.zeros(N)
        np.add.at(s, faces.reshape(-1), np.repeat(fn, 3, 0))
        size = (np.linalg.norm(p[:, 1] - p[:, 0], axis=1) * np.linalg.norm(p[:, 2] - p[:, 0], axis=1))
        np.add.at(scale, faces.reshape(-1), np.repeat(size, 3))
        count = np.bincount(faces.reshape(-1), minlength=N)
        length = np.linalg.norm(s, axis=1)
        bound = np.finfo(np.float32).eps * ((count + 8) * scale / length + 4)
        assert (np.abs(n[b] - s / length[:, None]).max(1) <= bound).all()


@pytest.mark.parametrize("degree", [1, 15, 16, 17, 33])
def test_arap_gradient_at_neighbour_counts_around_the_lane_group(degree):
    M = 36
    near = [d for h in range(1, degree // 2 + 1) for d in (h, -h)] + ([M // 2] if degree % 2 else [])
    idx = np.array([[(i + d) % M for d in near] for i in range(M)], np.int32).reshape(-1)  # symmetric
    off, size = np.arange(M, dtype=np.int32) * degree, np.full(M, degree, np.int32)
    rng = np.random.default_rng(degree)
    base = rng.normal(size=(M, 3)).astype(np.float32)
    nv = np.arange(M, dtype=np.int32)
    g = edm.ArapGraph(base, nv, off, size, idx, np.ones(M))
    G = rng.normal(size=(3, M, degree, 3)).astype(np.float32)
    dA = rng.normal(0, 0.3, (3, M, 3)).astype(np.float32)
    for got, ref in zip(edm.embedded_graph_arap_gpu_grad(g, _t(G), _t(dA)),
                        orc.arap_bwd(base, nv, off, size, idx, G, dA)):
        assert _rel(got.cpu(), ref) < 1e-5


def test_gradients_when_no_output_but_one_carries_any():
    """Outputs without a gradient reach the backward as None."""
    ch, g, gd, (dT, dA, sT, sA, disp), mk_node, bm, _ = setup(3)
    args = [_t(x).requires_grad_(True) for x in (dT, dA, sT, sA, disp)]
    edm.EmbeddedGraphGpu(gd, dT.shape[0], *args, False, "g").getNode()[2].sum().backward()  # markers alone
    node_marker = np.full(g.num_nodes, -1, np.int32)
    node_marker[mk_node] = np.arange(4)
    gv, gm = np.zeros((dT.shape[0], ch.N, 3)), np.ones((dT.shape[0], 4, 3))
    for a, ref in zip(args, orc.ed_bwd(g, ch.verts, gv, dA, sA, g_markers=gm, base_markers=bm,
                                       node_marker=node_marker)):
        assert float(np.abs(a.grad.cpu().numpy() - ref).max()) <= 1e-5 * max(float(np.abs(ref).max()), 1.0)
