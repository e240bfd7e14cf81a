"""GPU rasterizer parity against the oracle (through the C ABI).

Forward: tri-id, barycentrics, render and vertex normals are compared bit for
bit with the FP32 oracle (same rule, same operation order); the FP64 oracle
bounds the FP32 error of the barycentrics.  Backward: gradients against the
FP64 oracle evaluated on the GPU's own forward buffers."""
import numpy as np
import pytest
import torch

from deepcharacters_amd import renderer, scenes
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _t(a, dtype=torch.float32):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=dtype, device="cuda")


def make_scene(seed=0, B=2, C=3, W=200, H=150, subdiv=3, f=None):
    rng = np.random.default_rng(seed)
    ch = scenes.ellipsoid_character(subdiv, seed=seed)
    V = np.stack([ch.verts + rng.normal(0, 0.005, ch.verts.shape) for _ in range(B)])
    col = rng.uniform(0, 1, (B, ch.N, 3))
    exts, intrs = [], []
    for b in range(B):
        e, k = scenes.ring_cameras(C, 2.6, f or 0.45 * W * 2.6, W, H, rng=rng, phase=0.3 * b + 0.1)
        exts.append(e.reshape(-1))
        intrs.append(k.reshape(-1))
    tex = rng.uniform(0, 1, (B, 32, 48, 3))
    sh = rng.normal(0, 0.3, (B, C, 27))
    sh[..., [0, 9, 18]] += 1.0
    return ch, V, col, np.array(exts), np.array(intrs), tex, sh


def gpu_forward(ch, V, col, ext, intr, tex, sh, W, H, albedo="vertexColor", shading="shadeless", path="binned",
                ws_extra=None, topo=None):
    C = ext.shape[1] // 12
    topo = topo or renderer.Topology(ch.faces, ch.N, ch.texcoords)
    cfg = renderer.make_cfg(C, W, H, albedo, shading, path=path)
    ws = None
    if ws_extra is not None:
        import ctypes
        from deepcharacters_amd import _lib
        full = _lib.load().dcx_render_workspace_size(topo.handle, ctypes.byref(cfg), V.shape[0])
        ws = torch.empty(full + ws_extra, dtype=torch.uint8, device="cuda")
    out = renderer.render_forward(topo, cfg, _t(V), _t(col), _t(tex), _t(sh), _t(ext), _t(intr), ws=ws)
    torch.cuda.synchronize()
    return [o.cpu().numpy() for o in out]


@pytest.mark.parametrize("path", ["binned", "plain"])
@pytest.mark.parametrize("albedo,shading", [("vertexColor", "shadeless"), ("vertexColor", "shaded"),
                                            ("textured", "shadeless"), ("normal", "shadeless"),
                                            ("lighting", "shadeless"), ("position", "shadeless"),
                                            ("depth", "shadeless"), ("uv", "shadeless"),
                                            ("foregroundMask", "shadeless")])
def test_forward_bit_exact_vs_fp32_oracle(path, albedo, shading):
    W, H = 200, 150
    ch, V, col, ext, intr, tex, sh = make_scene(1, W=W, H=H)
    bary, face, render, vn = gpu_forward(ch, V, col, ext, intr, tex, sh, W, H, albedo, shading, path)
    of, ob, orr, ovn = orc.raster_fwd(ch.faces, V, ext, intr, H, W, vcol=col, albedo=albedo, shading=shading,
                                      tex=tex, sh=sh, texcoords=ch.texcoords.reshape(-1, 6), dtype=np.float32)
    assert (face >= 0).mean() > 0.1
    assert np.array_equal(face, of), (face != of).sum()
    assert np.array_equal(bary, ob), np.abs(bary - ob).max()
    assert np.array_equal(vn, ovn), np.abs(vn - ovn).max()
    assert np.abs(render - orr).max() <= 1e-6 * max(1.0, np.abs(orr).max())


def test_fp32_barycentrics_vs_fp64_oracle():
    """FP32 conditioning of metre-scale geometry: barycentrics from float32
    projections vs the same algorithm in FP64 (same tri-ids)."""
    W, H = 256, 256
    ch, V, col, ext, intr, tex, sh = make_scene(2, B=1, C=2, W=W, H=H, subdiv=4)
    bary, face, _, _ = gpu_forward(ch, V, col, ext, intr, tex, sh, W, H)
    of, ob, _, _ = orc.raster_fwd(ch.faces, V, ext, intr, H, W, vcol=col, dtype=np.float64)
    m = (face == of) & (face >= 0)
    assert m.mean() > 0.2 and (face == of).mean() > 0.999
    err = np.abs(bary - ob)[m]
    assert np.median(err) < 1e-5 and err.max() < 5e-3, (np.median(err), err.max())


def test_binned_equals_plain_and_is_deterministic():
    W, H = 320, 240
    ch, V, col, ext, intr, tex, sh = make_scene(3, W=W, H=H, subdiv=4)
    topo = renderer.Topology(ch.faces, ch.N, ch.texcoords)
    a = gpu_forward(ch, V, col, ext, intr, tex, sh, W, H, path="binned", topo=topo)
    b = gpu_forward(ch, V, col, ext, intr, tex, sh, W, H, path="binned", topo=topo)
    c = gpu_forward(ch, V, col, ext, intr, tex, sh, W, H, path="plain", topo=topo)
    for x, y, z in zip(a, b, c):
        assert np.array_equal(x, y) and np.array_equal(x, z)


def test_bin_overflow_falls_back_exactly():
    """A workspace with (almost) no tile-list capacity forces every tile onto the
    per-view scan path; results must not change."""
    W, H = 96, 64
    ch, V, col, ext, intr, tex, sh = make_scene(4, W=W, H=H)
    import ctypes
    from deepcharacters_amd import _lib
    topo = renderer.Topology(ch.faces, ch.N, ch.texcoords)
    C = ext.shape[1] // 12
    cfg = renderer.make_cfg(C, W, H)
    full = _lib.load().dcx_render_workspace_size(topo.handle, ctypes.byref(cfg), V.shape[0])
    cap_bytes = 4 * max(4 * ch.F * V.shape[0] * C, 65536)  # default tile-list capacity
    small = torch.empty(full - cap_bytes + 64, dtype=torch.uint8, device="cuda")  # 16 entries
    out_small = renderer.render_forward(topo, cfg, _t(V), _t(col), _t(tex), _t(sh), _t(ext), _t(intr), ws=small)
    out_full = renderer.render_forward(topo, cfg, _t(V), _t(col), _t(tex), _t(sh), _t(ext), _t(intr))
    for x, y in zip(out_small, out_full):
        assert torch.equal(x, y)


@pytest.mark.parametrize("W,H", [(1, 1), (33, 9), (7, 300)])
def test_odd_resolutions(W, H):
    ch, V, col, ext, intr, tex, sh = make_scene(5, B=1, C=2, W=W, H=H, f=0.45 * 64 * 2.6)
    for path in ("binned", "plain"):
        bary, face, render, _ = gpu_forward(ch, V, col, ext, intr, tex, sh, W, H, path=path)
        of, ob, orr, _ = orc.raster_fwd(ch.faces, V, ext, intr, H, W, vcol=col)
        assert np.array_equal(face, of) and np.array_equal(bary, ob)


def test_empty_degenerate_and_full_screen():
    ext = np.array([[1.0, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, 2.0]])
    intr = np.array([[40.0, 0, 24, 0, 40, 16, 0, 0, 1]])
    V = np.array([[[-0.5, -0.5, 0.2], [0.0, 0.0, 0.2], [0.5, 0.5, 0.2],        # collinear
                   [-0.5, -0.5, -2.5], [0.5, -0.5, -2.5], [0.0, 0.5, -2.5],     # behind
                   [-50, -50, 1.0], [50, -50, 1.0], [50, 50, 1.0], [-50, 50, 1.0]]])  # full screen quad
    faces = np.array([[0, 1, 2], [3, 4, 5], [6, 7, 8], [6, 8, 9]], np.int32)
    col = np.ones((1, 10, 3))

    class Ch:
        pass
    ch = Ch()
    ch.faces, ch.N, ch.texcoords = faces, 10, None
    for path in ("binned", "plain"):
        bary, face, render, _ = gpu_forward(ch, V, col, ext, intr, np.zeros((1, 1, 1, 3)), np.zeros((1, 1, 27)),
                                            48, 32, path=path)
        of, ob, orr, _ = orc.raster_fwd(faces, V, ext, intr, 32, 48, vcol=col)
        assert np.array_equal(face, of)
        assert set(np.unique(face).tolist()) <= {2, 3}
        assert np.isfinite(bary).all() and np.isfinite(render).all()


@pytest.mark.parametrize("albedo,shading,target", [("vertexColor", "shadeless", False),
                                                   ("vertexColor", "shadeless", True),
                                                   ("vertexColor", "shaded", True),
                                                   ("textured", "shadeless", False),
                                                   ("textured", "shaded", True)])
def test_backward_matches_oracle(albedo, shading, target):
    W, H = 160, 120
    ch, V, col, ext, intr, tex, sh = make_scene(6, W=W, H=H)
    C = ext.shape[1] // 12
    topo = renderer.Topology(ch.faces, ch.N, ch.texcoords)
    cfg = renderer.make_cfg(C, W, H, albedo, shading)
    bary, face, render, vn = renderer.render_forward(topo, cfg, _t(V), _t(col), _t(tex), _t(sh), _t(ext), _t(intr))
    rng = np.random.default_rng(7)
    g = rng.normal(size=render.shape)
    tgt = rng.uniform(0, 1, render.shape) if target else None
    gvp, gvc, gtx, gsh = renderer.render_backward(topo, cfg, _t(g), _t(V), _t(col),
                                                  _t(tex) if albedo == "textured" else None, _t(sh),
                                                  _t(tgt) if target else None, vn, bary, face, _t(ext), _t(intr))
    o = orc.raster_bwd(ch.faces, g, V.astype(np.float32), ext.astype(np.float32), intr.astype(np.float32),
                       face.cpu().numpy(), bary.cpu().numpy(), vn.cpu().numpy(), vcol=col.astype(np.float32),
                       albedo=albedo, shading=shading, tex=tex.astype(np.float32), sh=sh.astype(np.float32),
                       target=tgt, texcoords=ch.texcoords.reshape(-1, 6), dtype=np.float64)
    names = ["vertex_pos_grad", "vertex_color_grad", "texture_grad", "sh_coeff_grad"]
    for name, got, ref in zip(names, (gvp, gvc, gtx, gsh), o):
        if name == "texture_grad" and albedo != "textured":
            continue
        if name == "sh_coeff_grad" and shading != "shaded":
            continue
        got = got.cpu().numpy()
        scale = max(np.abs(ref).max(), 1e-12)
        # per-pixel float32 evaluation vs FP64, summed with atomics
        assert np.abs(got - ref).max() / scale < 2e-4, (name, np.abs(got - ref).max() / scale)


def test_cuda_renderer_gpu_wrapper_and_gradient_wiring():
    W, H = 96, 72
    ch, V, col, ext, intr, tex, sh = make_scene(8, B=1, C=2, W=W, H=H)
    vp = _t(V).requires_grad_(True)
    vc = _t(col).requires_grad_(True)
    r = renderer.CudaRendererGpu(faces_attr=ch.faces.reshape(-1).tolist(), texCoords_attr=ch.texcoords.reshape(-1).tolist(),
                                 numberOfVertices_attr=ch.N, numberOfCameras_attr=2, renderResolutionU_attr=W,
                                 renderResolutionV_attr=H, albedoMode_attr="vertexColor", shadingMode_attr="shadeless",
                                 image_filter_size_attr=2, texture_filter_size_attr=2, vertexPos_input=vp,
                                 vertexColor_input=vc, texture_input=_t(tex), shCoeff_input=_t(sh),
                                 targetImage_input=torch.zeros((1, 2, H, W, 3), device="cuda"),
                                 extrinsics_input=ext, intrinsics_input=intr)
    img = r.getRenderBufferTF()
    mask = r.getModelMaskTF()
    assert mask.shape == (1, 2, H, W, 3)
    assert torch.equal(mask[..., 0] > 0, r.getFaceBufferTF() >= 0)
    loss = (img * img).sum()
    loss.backward()
    assert vp.grad is not None and vc.grad is not None and vp.grad.abs().sum() > 0
    # normal mode: zero gradients, as the reference registers
    vp2 = _t(V).requires_grad_(True)
    r2 = renderer.CudaRendererGpu(faces_attr=ch.faces.reshape(-1).tolist(), numberOfVertices_attr=ch.N,
                                  numberOfCameras_attr=2, renderResolutionU_attr=W, renderResolutionV_attr=H,
                                  albedoMode_attr="normal", vertexPos_input=vp2, vertexColor_input=_t(col),
                                  extrinsics_input=ext, intrinsics_input=intr)
    r2.getRenderBufferTF().sum().backward()
    assert torch.count_nonzero(vp2.grad) == 0


@pytest.mark.parametrize("W,H,order", [(200, 90, "mixed"), (1100, 40, "mixed"), (65, 700, "shuffled"), (300, 300, "fan")])
def test_binning_of_small_large_and_scattered_triangles(W, H, order):
    """Bit-exact against the oracle: triangles of a pixel, around 64 pixels
    wide (where the walk changes to 64 bits), over more than 16 tiles and over
    the whole image, in one wavefront; faces without any order; a vertex with
    300 faces."""
    rng = np.random.default_rng(W)
    ext = np.array([[1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, 0]], np.float32)
    intr = np.array([[1, 0, 0, 0, 1, 0, 0, 0, 1]], np.float32)  # (x z, y z, z) is seen at (x, y)
    if order == "fan":
        a = np.linspace(0, 2 * np.pi, 301)[:-1]
        xy = np.concatenate([[[150.2, 149.7]], np.stack([150 + 140 * np.cos(a), 150 + 140 * np.sin(a)], 1)])
        z = np.concatenate([[1.0], rng.uniform(1, 2, 300)])
        i = np.arange(300)
        faces = np.stack([0 * i, 1 + i, 1 + (i + 1) % 300], 1).astype(np.int32)
    else:
        sizes = np.concatenate([rng.uniform(0.3, 3, 400), rng.choice([31.9, 32.0, 32.1], 60), rng.uniform(60, 200, 20), [2000.0]])
        xy = np.concatenate([rng.uniform(0, [W, H]) + s * rng.uniform(-1, 1, (3, 2)) for s in sizes])
        # corners exactly 64 pixels (and one 256th more) apart
        xy[-63:-60] = np.array([[8.5, 4.5], [72.5, 4.5], [8.5, 30.5]])
        xy[-66:-63] = np.array([[8.5, 4.5], [72.5 + 1 / 256, 4.5], [8.5, 30.5]])
        z = rng.uniform(1, 5, len(xy))
        faces = np.arange(len(xy), dtype=np.int32).reshape(-1, 3)
        faces = rng.permutation(faces, axis=0) if order == "shuffled" else faces
    V = np.concatenate([xy * z[:, None], z[:, None]], 1)[None].astype(np.float32)
    col = rng.uniform(0, 1, V.shape).astype(np.float32)
    topo = renderer.Topology(faces, V.shape[1])
    cfg = renderer.make_cfg(1, W, H)
    bary, face, render, vn = renderer.render_forward(topo, cfg, _t(V), _t(col), None, None, _t(ext), _t(intr))
    of, ob, orr, ovn = orc.raster_fwd(faces, V, ext, intr, H, W, vcol=col)
    for got, ref in ((face, of), (bary, ob), (render, orr), (vn, ovn)):
        assert np.array_equal(got.cpu().numpy().reshape(np.shape(ref)), ref)
    assert (of >= 0).mean() > 0.3


def _backward_with(ws_bytes, topo, cfg, g, V, col, tex, sh, tgt, vn, bary, face, ext, intr):
    """dcx_render_bwd with a workspace of that many bytes (None: as many as it asks for)."""
    import ctypes
    from deepcharacters_amd import _lib
    B, N = V.shape[:2]
    full = _lib.load().dcx_render_bwd_workspace_size(topo.handle, ctypes.byref(cfg), B)
    ws = torch.full((max(full if ws_bytes is None else ws_bytes, 1),), 0xff, dtype=torch.uint8, device="cuda")  # NaNs
    out = [torch.full_like(V, float("nan")), torch.full_like(V, float("nan")),
           None if tex is None else torch.full_like(tex, float("nan")), torch.full((B, cfg.num_cameras, 27), float("nan"), device="cuda")]
    p = lambda x: None if x is None else x.data_ptr()
    th, tw = (0, 0) if tex is None else tex.shape[1:3]
    _lib.call("dcx_render_bwd", topo.handle, ctypes.byref(cfg), B, p(g), p(V), p(col), p(tex), th, tw, p(sh), p(tgt),
              p(vn), p(bary), p(face), p(ext), p(intr), *[p(o) for o in out], p(ws) if ws_bytes != 0 else None,
              ws.numel() if ws_bytes != 0 else 0, torch.cuda.current_stream().cuda_stream)
    return [o for o in out if o is not None]


@pytest.mark.parametrize("albedo,shading", [("vertexColor", "shadeless"), ("vertexColor", "shaded"),
                                            ("textured", "shadeless"), ("textured", "shaded"), ("foregroundMask", "shadeless")])
@pytest.mark.parametrize("buffers", ["rendered", "shifted", "random"])
@pytest.mark.parametrize("W,H,subdiv", [(160, 120, 3), (61, 47, 4), (300, 200, 1)])
def test_gathered_gradients_equal_the_scattered_ones(albedo, shading, buffers, W, H, subdiv):
    """The two forms of the backward on the same buffers: faces of a pixel and
    of thousands (left to the scatter form), and face buffers that were not
    rendered from these positions, whose pixels lie outside their faces' boxes.
    Sums of the same terms in another order, and the corners' image-space sums
    transformed once: 32-bit rounding of terms up to the largest of the sums."""
    ch, V, col, ext, intr, tex, sh = make_scene(8, W=W, H=H)
    ch = scenes.ellipsoid_character(subdiv, scale=(0.6, 0.45, 0.35), seed=3)
    rng = np.random.default_rng(11)
    B, C = V.shape[0], ext.shape[1] // 12
    V = np.stack([ch.verts + rng.normal(scale=0.005, size=ch.verts.shape) for _ in range(B)])
    Vt, colt, extt, intrt, sht = _t(V), _t(np.stack([ch.colors] * B)), _t(ext), _t(intr), _t(sh)
    text = _t(tex) if albedo == "textured" else None
    topo = renderer.Topology(ch.faces, ch.N, ch.texcoords)
    cfg = renderer.make_cfg(C, W, H, albedo, shading)
    bary, face, render, vn = renderer.render_forward(topo, cfg, Vt, colt, text, sht, extt, intrt)
    if buffers == "shifted":
        face, bary = face.roll((2, 3), (2, 3)).contiguous(), bary.roll((2, 3), (2, 3)).contiguous()
    elif buffers == "random":
        face = torch.where(torch.rand(face.shape, device="cuda") < 0.2, torch.randint(0, ch.F, face.shape, device="cuda"), -1).int()
        bary = torch.rand(bary.shape, device="cuda") * 0.5
    g, tgt = _t(rng.normal(size=render.shape)), _t(rng.uniform(0, 1, render.shape))
    args = (topo, cfg, g, Vt, colt, text, sht, tgt, vn, bary, face, extt, intrt)
    small = 12 * B * ch.N if shading == "shaded" else 0
    gathered, scattered = _backward_with(None, *args), _backward_with(small, *args)
    assert int((face >= 0).sum()) > 100
    for a, b in zip(gathered, scattered):
        assert torch.isfinite(b).all() or buffers != "rendered"
        ok = torch.isfinite(b)
        assert torch.equal(ok, torch.isfinite(a))
        assert float((a - b)[ok].abs().max()) <= 2e-4 * max(float(b[ok].abs().max()), 1e-12)
    if albedo != "textured":  # no atomics but the SH gradients': the same bits again
        again = _backward_with(None, *args)
        if buffers == "rendered" and subdiv >= 3:
            assert all(torch.equal(a, b) for a, b in zip(gathered[:2], again[:2]))


@pytest.mark.parametrize("albedo,shading", [("vertexColor", "shaded"), ("textured", "shaded"), ("textured", "shadeless"),
                                            ("foregroundMask", "shadeless")])
def test_gathered_gradients_at_the_edges_of_the_face_sizes(albedo, shading):
    """Triangles whose boxes and pixel counts lie around the limits between a
    face's own lanes, a wavefront and the scatter form: boxes of up to 16 x 16,
    31 x 33 and 32 x 32 pixels, single rows and columns of up to 1024, a few
    pixels (24, 28) and a single one, several views' lists of different lengths.
    32-bit sums of the same terms, as above."""
    W, H = 1100, 1090
    sizes = [(1, 1), (2, 2), (7, 7), (7, 8), (8, 8), (15, 17), (16, 16), (16, 17), (17, 17), (31, 33), (32, 32), (33, 33),
             (64, 4), (64, 5), (256, 1), (257, 1), (1, 257), (1022, 1), (1023, 1), (1024, 1), (1, 1023), (1, 1024), (40, 60)]
    rng = np.random.default_rng(12)
    tris, x, y, row = [], 4, 4, 0
    for w, h in [s for s in sizes for _ in range(6)]:
        if x + w + 2 > W - 6:
            x, y, row = 4, y + row + 2, 0
        if y + h + 2 < H - 6:
            # corners on the box's outer pixels' centres, off by under half a pixel
            c = np.array([[x, y], [x + w - 1, y + (h - 1) * rng.integers(0, 2)], [x + (w - 1) // 2, y + h - 1]])
            tris.append(c + 0.5 + rng.uniform(-0.45, 0.45, (3, 2)))
            x, row = x + w + 2, max(row, h)
    xy = np.concatenate(tris)
    z = rng.uniform(1, 1.5, len(xy))
    V = np.concatenate([xy * z[:, None], z[:, None]], 1)[None].astype(np.float32)
    faces = np.arange(len(xy), dtype=np.int32).reshape(-1, 3)
    intr = np.tile(np.array([1, 0, 0, 0, 1, 0, 0, 0, 1], np.float32), 3)[None]  # (x z, y z, z) is seen at (x, y)
    ext = np.array([[1, 0, 0, t, 0, 1, 0, 0, 0, 0, 1, 0] for t in (0, 700, -700)], np.float32).reshape(1, 36)
    topo = renderer.Topology(faces, len(xy), rng.uniform(0.1, 0.9, (len(faces), 6)).astype(np.float32))
    cfg = renderer.make_cfg(3, W, H, albedo, shading)
    Vt, colt, extt, intrt = _t(V), _t(rng.uniform(0, 1, V.shape)), _t(ext), _t(intr)
    text = _t(rng.uniform(0, 1, (1, 64, 64, 3))) if albedo == "textured" else None
    sht = _t(rng.uniform(0.1, 0.5, (1, 3, 27)))
    bary, face, render, vn = renderer.render_forward(topo, cfg, Vt, colt, text, sht, extt, intrt)
    g, tgt = _t(rng.normal(size=render.shape)), _t(rng.uniform(0, 1, render.shape))
    args = (topo, cfg, g, Vt, colt, text, sht, tgt, vn, bary, face, extt, intrt)
    seen = torch.bincount(face[0, 0].flatten()[face[0, 0].flatten() >= 0].long(), minlength=len(faces))
    assert int((seen > 0).sum()) > len(faces) // 2 and int(seen.max()) > 500 and int((seen == 1).sum()) > 0
    small = 12 * V.shape[1] if shading == "shaded" else 0
    gathered, scattered = _backward_with(None, *args), _backward_with(small, *args)
    assert bool(scattered[0].any())
    for a, b in zip(gathered, scattered):
        assert torch.isfinite(b).all()
        assert float((a - b).abs().max()) <= 2e-4 * max(float(b.abs().max()), 1e-12)
