"""The renderer's, the fit harness's and the proposal network's work as a user's program has it done.

Kinds of case:
  render    one mesh (capped cylinder or icosphere, batch x views at width x height) rendered through
            `Rasterizer` ("direct": forward, then backward with a given upstream gradient, as a serving or
            training loop with its own loss does; "autograd": `Rasterizer.render` under torch.autograd; or
            "dropin": the `CudaRenderer.CudaRendererGpu` class with a squared loss, as the demo scripts use it);
            `backward` off is a forward alone; `target_term` adds the model-to-data term (an upstream gradient
            of the target image)
  multi     a batch of uneven meshes, forward and backward, through `MultiRenderer`
  fit       value and gradient of one analysis-by-synthesis step: shape model, render, masked loss, backward
  shape     the fit's shape model alone: posed vertices and the gradients of coefficients and pose
  train     the proposal network's forward and backward, and the refresh of its bf16 weight copies
  propose   the proposal network on new renders: mosaic packing and forward

Inputs follow gvv_amd.scenes: millimetre meshes of about 1 m radius seen from 3 to 3.5 m, seeded smooth
textures, SH lighting around a DC of 0.8.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "gvv-differentiable-cuda-renderer_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import CudaRenderer  # noqa: E402
from gvv_amd import Rasterizer, fit, multi, proposal, scenes  # noqa: E402

MAX_EXACT_CANDIDATES = 24_000_000     # (face, pixel) tests of a scene that exact() still renders (some seconds)
NET = ((256, 8, 32), (128, 32, 64), (64, 64, 128), (32, 128, 128), (16, 128, 256), (8, 256, 256))   # H, Cin, Cout


# ---------------------------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------------------------
def _render_case(name, mesh, detail, batch, views, width, height, albedo, shading="shaded", tex=(1, 1), backward=True,
                 target_term=False, entry="direct"):
    return dict(name=name, kind="render", mesh=mesh, detail_a=detail[0], detail_b=detail[1], batch=batch, views=views,
                width=width, height=height, albedo=albedo, shading=shading, tex_h=tex[0], tex_w=tex[1],
                backward=backward, target_term=target_term, entry=entry)


def listed():
    return [
        # the smallest training step: a 5,120-face sphere in four 256^2 views under autograd, where launches count
        _render_case("sphere_4x256", "sphere", (4, 0), 1, 4, 256, 256, "vertexColor", entry="autograd"),
        # a demo script's iteration: the drop-in class, one camera, a 4,000-face textured mesh, squared loss
        _render_case("demo_textured_640x480", "cylinder", (50, 40), 1, 1, 640, 480, "textured", tex=(512, 512),
                     entry="dropin"),
        # a capture studio's step: 100,000 textured faces in eight 1024^2 views
        _render_case("studio_textured_8x1024", "cylinder", (250, 200), 1, 8, 1024, 1024, "textured", tex=(1024, 1024)),
        # silhouettes of a small batch at an odd size, forward alone
        _render_case("silhouette_12x517x389", "sphere", (5, 0), 4, 3, 517, 389, "foregroundMask", backward=False),
        # textured, with the model-to-data term, ragged image and texture
        _render_case("m2d_textured_6x333x477", "cylinder", (100, 80), 2, 3, 333, 477, "textured", tex=(300, 211),
                     target_term=True),
        # a low-polygon proxy whose faces cover thousands of pixels each, unlit
        _render_case("lowpoly_4x1024", "sphere", (2, 0), 1, 4, 1024, 1024, "vertexColor", shading="shadeless"),
        # the largest: two subjects of 200,000 faces in eight 1024^2 views each
        _render_case("subjects_vertexcolor_16x1024", "cylinder", (354, 283), 2, 8, 1024, 1024, "vertexColor"),
        # an uneven batch of meshes of different topology
        dict(name="multi_uneven_8", kind="multi", topology=0, meshes=8, faces_min=2000, faces_max=60000, views_max=6),
        # one step of the fit: 16 subjects x 4 views at 512^2, 70,000-face template, 80 coefficients
        dict(name="fit_16x4x512", kind="fit", batch=16, views=4, resolution=512, cols=175, rows=200, basis=80),
        # its shape model alone
        dict(name="shape_16x35002x80", kind="shape", batch=16, vertices=35002, basis=80),
        # the proposal network: a training batch, and one new subject
        dict(name="proposal_train_16", kind="train", batch=16),
        dict(name="propose_1", kind="propose", batch=1, views=4, resolution=512),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["render"] * 6 + ["multi", "fit", "shape", "train", "propose", "render"])
    if kind == "render":
        if rng.random() < 0.5:
            mesh, a, b = "sphere", rng.randint(2, 5), 0
        else:
            mesh = "cylinder"
            a = _log_int(rng, 12, 300)
            b = max(4, int(a * rng.uniform(0.6, 1.0)))
        while True:
            width, height = _log_int(rng, 64, 1100), _log_int(rng, 64, 1100)
            batch, views = rng.choice([1, 1, 2, 3, 4]), rng.randint(1, 8)
            if width * height * batch * views <= 12_000_000:
                break
        backward = rng.random() < 0.75
        albedo = rng.choice(["vertexColor", "textured", "foregroundMask"] if backward else
                            ["vertexColor", "textured", "foregroundMask", "normal", "lighting"])
        tex = (_log_int(rng, 16, 1100), _log_int(rng, 16, 1100)) if albedo == "textured" else (1, 1)
        target = backward and rng.random() < 0.25
        entry = "direct" if target or not backward else rng.choice(["direct", "autograd", "dropin"])
        c = _render_case("", mesh, (a, b), batch, views, width, height, albedo,
                         rng.choice(["shaded", "shaded", "shadeless"]), tex, backward, target, entry)
    elif kind == "multi":
        c = dict(kind="multi", topology=rng.randint(1, 1000), meshes=rng.randint(2, 8), faces_min=2000,
                 faces_max=_log_int(rng, 6000, 60000), views_max=rng.randint(1, 6))
    elif kind == "fit":
        c = dict(kind="fit", batch=_log_int(rng, 1, 16), views=rng.randint(1, 4), resolution=rng.choice([128, 256, 400, 512]),
                 cols=_log_int(rng, 40, 175), rows=_log_int(rng, 40, 200), basis=rng.choice([10, 33, 64, 80]))
    elif kind == "shape":
        c = dict(kind="shape", batch=_log_int(rng, 1, 40), vertices=_log_int(rng, 500, 60000), basis=_log_int(rng, 4, 128))
    elif kind == "train":
        c = dict(kind="train", batch=_log_int(rng, 1, 24))
    else:
        c = dict(kind="propose", batch=_log_int(rng, 1, 24), views=rng.choice([1, 2, 4]), resolution=rng.choice([128, 256, 512]))
    c.pop("name", None)
    return c


# ---------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------
def _scene(case, seed):
    """The numpy inputs of a render case."""
    rng = np.random.Generator(np.random.PCG64(seed))
    if case["mesh"] == "sphere":
        v, f = scenes.icosphere(case["detail_a"])
        v = v + rng.normal(0.0, 0.01, size=v.shape)
        uv = rng.uniform(0.0, 1.0, size=(f.shape[0], 3, 2)).astype(np.float32)
    else:
        v, f, uv = scenes.capped_cylinder(case["detail_a"], case["detail_b"], 1.0, 2.0, rng, 0.05)
    B, C, W, H = case["batch"], case["views"], case["width"], case["height"]
    scale = rng.uniform(0.95, 1.05, size=(B, 1, 1))
    vpos = (v[None] * scale * scenes.MM).astype(np.float32)
    if case["mesh"] == "sphere":
        E, K = scenes.sphere_cameras(C, 3.0, W, H, rng)
    else:
        E, K = scenes.ring_cameras(C, 3.5, W, H)
    if case["albedo"] == "textured":
        tex = np.stack([scenes.smooth_texture(rng, case["tex_h"], case["tex_w"]) for _ in range(B)])
    else:
        tex = np.full((B, case["tex_h"], case["tex_w"], 3), 0.5, np.float32)
    return dict(faces=f, uv=uv, vpos=vpos, vcol=rng.uniform(0.0, 1.0, size=vpos.shape).astype(np.float32), tex=tex,
                sh=np.stack([scenes.sh_coefficients(C, rng) for _ in range(B)]),
                extr=np.tile(E.reshape(1, C, 12), (B, 1, 1)), intr=np.tile(K.reshape(1, C, 9), (B, 1, 1)))


def _images(case, seed):
    """Seeded upstream gradient, target image and target gradient of a render case (host float32)."""
    g = torch.Generator().manual_seed(seed + 100)
    shape = (case["batch"], case["views"], case["height"], case["width"], 3)
    return torch.randn(shape, generator=g), torch.rand(shape, generator=g), \
        torch.randn(shape, generator=g) if case["target_term"] else None


def _dev(a):
    return torch.as_tensor(np.ascontiguousarray(a) if isinstance(a, np.ndarray) else a).cuda()


def _shape_inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    B, N, K = case["batch"], case["vertices"], case["basis"]
    r = lambda *s: torch.randn(s, generator=g, device="cuda")
    return dict(alpha=0.5 * r(B, K), pose=0.2 * r(B, 6), template=700.0 * r(N, 3), basis=20.0 * r(K, 3 * N),
                centre=10.0 * r(3), g=r(B, N, 3))


def _net_weights(seed):
    """Seeded He-initialised weights of the proposal network, with biases off zero."""
    g = torch.Generator().manual_seed(seed + 7)
    sd = dict(features=torch.tensor(0))
    for i, (_, cin, cout) in enumerate(NET):
        w = torch.randn((cout, 3, 3, cin), generator=g) * math.sqrt(2.0 / (9 * (3 if i == 0 else cin)))
        if i == 0:
            w[..., 3:] = 0.0
        sd["w%d" % i], sd["b%d" % i] = w, 0.05 * torch.randn(cout, generator=g)
    w, b = torch.randn((128, 1, 1, 4096), generator=g) / 64.0, 0.05 * torch.randn(128, generator=g)
    w[113:], b[113:] = 0.0, 0.0
    sd["w6"], sd["b6"] = w, b
    return sd


def _blobs(n, res, seed):
    """Renders of about the statistics of the fit's: a shaded shape before the renderer's (0, 1, 0) background."""
    g = torch.Generator().manual_seed(seed + 3)
    y, x = torch.meshgrid(torch.linspace(-1, 1, res), torch.linspace(-1, 1, res), indexing="ij")
    p = torch.rand((n, 8, 1, 1), generator=g)
    inside = (((x - 0.2 * (p[:, 0] - 0.5)) / (0.5 + 0.2 * p[:, 1])).abs() < 1) & \
             (((y - 0.2 * (p[:, 2] - 0.5)) / (0.7 + 0.2 * p[:, 3])).abs() < 1)
    shade = 0.5 + 0.3 * torch.sin(9.0 * p[:, 4] * x + 6.0 * p[:, 5] * y)
    col = torch.stack([shade, shade * (0.5 + p[:, 6]), shade * (0.5 + p[:, 7])], -1)
    col = (col + 0.1 * torch.randn(col.shape, generator=g)).clamp(0.0, 1.2)
    return torch.where(inside[..., None], col, torch.tensor([0.0, 1.0, 0.0]))


def _train_inputs(case, seed):
    B = case["batch"]
    x = torch.zeros((B, 256, 256, 8), dtype=torch.bfloat16)
    x[..., :3] = _blobs(B, 256, seed).to(torch.bfloat16)
    return x, torch.randn((B, 113), generator=torch.Generator().manual_seed(seed + 5))


def _propose_inputs(case, seed):
    B, V, R = case["batch"], case["views"], case["resolution"]
    return _blobs(B * V, R, seed).view(B, V, R, R, 3)


def _net(seed):
    net = proposal.ProposalNet(torch.device("cuda", torch.cuda.current_device()))
    net.load_state_dict(_net_weights(seed))
    return net


def _fit_state(case, seed):
    cfg = fit.FitConfig(n_basis=case["basis"], cols=case["cols"], rows=case["rows"], views=case["views"],
                        resolution=case["resolution"], batch=case["batch"], seed=seed, basis_smoothing=0)
    model = fit.ShapeModel(cfg)
    # smooth low-frequency fields in the place of the (slow to make) smoothed noise, 2 cm of spread each
    g = torch.Generator(device="cuda").manual_seed(seed)
    k = torch.randn((case["basis"], 3, 3), generator=g, device="cuda") * 0.003
    ph = torch.rand((case["basis"], 3, 1), generator=g, device="cuda") * 2 * math.pi
    model.basis = (28.0 * torch.sin(k @ model.template.T + ph)).transpose(1, 2).reshape(case["basis"], -1).contiguous()
    rng = np.random.Generator(np.random.PCG64(seed))
    truth = fit.sample_params(rng, case["batch"], case["basis"], model.device)
    target, mask = fit.make_targets(model, truth)
    start = fit.plain_init(case["batch"], case["basis"], model.device).flat()
    x = (0.5 * (start + truth.flat())).requires_grad_(True)
    return dict(kind="fit", model=model, target=target, mask=mask, weight=1.0 / mask.sum(), x=x, basis=case["basis"])


def _multi_scenes(case, seed):
    """The batch of one topology seed (mesh sizes, views, resolutions), with positions and colours of this seed."""
    out = scenes.config2(seed=case["topology"], n_meshes=case["meshes"],
                         tri_range=(case["faces_min"], case["faces_max"]), max_views=case["views_max"])
    rng = np.random.Generator(np.random.PCG64(seed))
    for s in out:
        s.vpos = (s.vpos * rng.uniform(0.95, 1.05) + rng.normal(0.0, 0.2, size=s.vpos.shape)).astype(np.float32)
        s.vcol = rng.uniform(0.0, 1.0, size=s.vcol.shape).astype(np.float32)
    return out


def prepare(case, seed):
    kind = case["kind"]
    if kind == "render":
        s = _scene(case, seed)
        g, target, g_target = _images(case, seed)
        grad = case["entry"] != "direct"
        st = dict(case, target=_dev(target), g=_dev(g), g_target=_dev(g_target) if g_target is not None else None)
        for k in ("vpos", "vcol", "tex", "sh", "extr", "intr"):
            st[k] = _dev(s[k]).requires_grad_(grad and k in ("vpos", "vcol", "tex", "sh"))
        B = case["batch"]
        st["extr"], st["intr"] = st["extr"].reshape(B, -1), st["intr"].reshape(B, -1)
        st["faces"], st["uv"] = s["faces"].reshape(-1), s["uv"].reshape(-1)
        st["N"] = s["vpos"].shape[1]
        if case["entry"] != "dropin":
            st["rast"] = Rasterizer(st["faces"], st["uv"], st["N"], case["views"], case["width"], case["height"],
                                    albedo_mode=case["albedo"], shading_mode=case["shading"])
        return st
    if kind == "multi":
        mr = multi.MultiRenderer(_multi_scenes(case, seed))
        g = torch.Generator(device="cuda").manual_seed(seed)
        for b in mr.bufs:
            b["g_render"].normal_(generator=g)
        return dict(kind=kind, mr=mr)
    if kind == "fit":
        return _fit_state(case, seed)
    if kind == "shape":
        st = _shape_inputs(case, seed)
        st["alpha"].requires_grad_(True)
        st["pose"].requires_grad_(True)
        return dict(st, kind=kind)
    if kind == "train":
        x, y = _train_inputs(case, seed)
        return dict(kind=kind, net=_net(seed), x=_dev(x), y=_dev(y))
    return dict(kind=kind, net=_net(seed), render=_dev(_propose_inputs(case, seed)))


# ---------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------
def _run_render(s):
    leaves = [s["vpos"], s["vcol"], s["tex"], s["sh"]]
    if s["entry"] == "dropin":
        r = CudaRenderer.CudaRendererGpu(
            faces_attr=s["faces"], texCoords_attr=s["uv"], numberOfVertices_attr=s["N"],
            numberOfCameras_attr=s["views"], renderResolutionU_attr=s["width"], renderResolutionV_attr=s["height"],
            albedoMode_attr=s["albedo"], shadingMode_attr=s["shading"], vertexPos_input=s["vpos"],
            vertexColor_input=s["vcol"], texture_input=s["tex"], shCoeff_input=s["sh"], targetImage_input=s["target"],
            extrinsics_input=s["extr"], intrinsics_input=s["intr"])
        render = r.getRenderBufferTF()
        loss = ((render - s["target"]) ** 2).sum()
        grads = torch.autograd.grad(loss, leaves)
        return dict(bary=r.getBaryCentricBufferTF(), face=r.getFaceBufferTF(), render=render, grads=list(grads))
    if s["entry"] == "autograd":
        bary, face, render, vnormal, _, _ = s["rast"].render(*leaves, s["target"], s["extr"], s["intr"])
        grads = torch.autograd.grad(render, leaves, grad_outputs=s["g"])
        return dict(bary=bary, face=face, render=render, vnormal=vnormal, grads=list(grads))
    bary, face, render, vnormal, _ = s["rast"].forward(*leaves, s["extr"], s["intr"])
    out = dict(bary=bary, face=face, render=render, vnormal=vnormal)
    if s["backward"]:
        out["grads"] = list(s["rast"].backward(s["g"], s["g_target"], s["target"] if s["target_term"] else None, *leaves,
                                               vnormal, face, s["extr"], s["intr"]))
    return out


def run(state):
    kind = state["kind"]
    if kind == "render":
        return _run_render(state)
    if kind == "multi":
        state["mr"].run(backward=True)
        keys = ("face", "bary", "render", "vnormal", "g_pos", "g_col", "g_sh")
        return [{k: b[k] for k in keys} for b in state["mr"].bufs]
    if kind == "fit":
        render, face = state["model"].render(fit.Params.from_flat(state["x"], state["basis"]))
        sq = fit.masked_sq_error(render, state["target"], state["mask"])
        grad, = torch.autograd.grad(sq.sum() * state["weight"], state["x"])
        return dict(render=render, face=face, sq=sq, grad=grad)
    if kind == "shape":
        v = fit.ShapeVertices.apply(state["alpha"], state["pose"], state["template"], state["basis"], state["centre"])
        ga, gp = torch.autograd.grad(v, [state["alpha"], state["pose"]], grad_outputs=state["g"])
        return dict(v=v, alpha=ga, pose=gp)
    net = state["net"]
    if kind == "train":
        out = net.forward(state["x"])
        net.backward((out - state["y"]) * (2.0 / out.numel()))
        net.refresh()
        return dict(out=out, gw=list(net.gw), gb=list(net.gb))
    x = proposal.pack_mosaic(state["render"])
    return dict(x=x, out=net.forward(x))


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------
def _mesh_counts(case):
    if case["mesh"] == "sphere":
        return 10 * 4 ** case["detail_a"] + 2, 20 * 4 ** case["detail_a"]
    return case["detail_a"] * case["detail_b"] + 2, 2 * case["detail_a"] * case["detail_b"]


def _render_work(B, C, N, F, P, T, backward, target_term, shaded):
    """Every input and output byte once; about 60% of the pixels covered, 100 operations of projection, ray,
    barycentrics and shading each (and 200 of gradient)."""
    b = 36 * F + 24 * B * N + 12 * B * T + 192 * B * C + 24 * P + 12 * B * C * N
    fl = 100 * 0.6 * P + 60 * B * C * N
    if backward:
        b += 12 * P + 24 * B * N + 12 * B * T + 108 * B * C + (24 * P if target_term else 0)
        fl += (200 if shaded else 60) * 0.6 * P
    return b, fl


def work(case):
    kind = case["kind"]
    if kind == "render":
        B, C = case["batch"], case["views"]
        N, F = _mesh_counts(case)
        b, fl = _render_work(B, C, N, F, B * C * case["width"] * case["height"], case["tex_h"] * case["tex_w"],
                             case["backward"], case["target_term"],
                             case["shading"] == "shaded" and case["albedo"] != "foregroundMask")
        if case["entry"] == "dropin":
            b += 24 * B * C * case["width"] * case["height"]
    elif kind == "multi":
        # the expectation over the drawn meshes: log-uniform face counts, uniform views and resolutions
        lo, hi = case["faces_min"], case["faces_max"]
        F = (hi - lo) / math.log(hi / lo)
        C, px = (1 + case["views_max"]) / 2.0, (256 ** 2 + 512 ** 2 + 1024 ** 2) / 3.0
        b, fl = (case["meshes"] * x for x in _render_work(1, C, F / 2, F, C * px, 1, True, False, True))
    elif kind == "fit":
        B, C, K = case["batch"], case["views"], case["basis"]
        N, F = case["cols"] * case["rows"] + 2, 2 * case["cols"] * case["rows"]
        P = B * C * case["resolution"] ** 2
        b, fl = _render_work(B, C, N, F, P, 1, True, False, True)
        b += 28 * P + 12 * K * N
        fl += 15 * P + 12 * B * K * N
    elif kind == "shape":
        B, N, K = case["batch"], case["vertices"], case["basis"]
        b, fl = 12 * K * N + 24 * B * N + 12 * N, 12 * B * K * N
    else:
        B = case["batch"]
        macs = sum((h // 2) ** 2 * cout * 9 * (3 if h == 256 else cin) for h, cin, cout in NET) + 4096 * 113
        params = sum(9 * cin * cout + cout for _, cin, cout in NET) + 4096 * 113 + 113
        if kind == "train":
            b, fl = 2 * B * 256 * 256 * 3 + 8 * params + 4 * B * 113 * 2, 6 * B * macs
        else:
            b = 12 * B * case["views"] * case["resolution"] ** 2 + 16 * B * 256 * 256 + 2 * params + 4 * B * 113
            fl = 2 * B * macs
    return dict(bytes=int(b), flops=int(fl))


# ---------------------------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------------------------
# The renderer's decisions (which face a pixel shows, its nearest texel, whether its normal is turned) are fixed as
# binary32 arithmetic in a given order; everything computed from them is a number with a value in 64 bits.  So the
# decisions are taken in numpy float32 below and the values in float64.
_COFACTORS = (   # signed triples of each entry of a 4x4 inverse, in order
    "+5,10,15 -5,11,14 -9,6,15 +9,7,14 +13,6,11 -13,7,10|-1,10,15 +1,11,14 +9,2,15 -9,3,14 -13,2,11 +13,3,10|"
    "+1,6,15 -1,7,14 -5,2,15 +5,3,14 +13,2,7 -13,3,6|-1,6,11 +1,7,10 +5,2,11 -5,3,10 -9,2,7 +9,3,6|"
    "-4,10,15 +4,11,14 +8,6,15 -8,7,14 -12,6,11 +12,7,10|+0,10,15 -0,11,14 -8,2,15 +8,3,14 +12,2,11 -12,3,10|"
    "-0,6,15 +0,7,14 +4,2,15 -4,3,14 -12,2,7 +12,3,6|+0,6,11 -0,7,10 -4,2,11 +4,3,10 +8,2,7 -8,3,6|"
    "+4,9,15 -4,11,13 -8,5,15 +8,7,13 +12,5,11 -12,7,9|-0,9,15 +0,11,13 +8,1,15 -8,3,13 -12,1,11 +12,3,9|"
    "+0,5,15 -0,7,13 -4,1,15 +4,3,13 +12,1,7 -12,3,5|-0,5,11 +0,7,9 +4,1,11 -4,3,9 -8,1,7 +8,3,5|"
    "-4,9,14 +4,10,13 +8,5,14 -8,6,13 -12,5,10 +12,6,9|+0,9,14 -0,10,13 -8,1,14 +8,2,13 +12,1,10 -12,2,9|"
    "-0,5,14 +0,6,13 +4,1,14 -4,2,13 -12,1,6 +12,2,5|+0,5,10 -0,6,9 -4,1,10 +4,2,9 +8,1,6 -8,2,5").split("|")


def _inverse32(e):
    e = e.reshape(-1)
    inv = np.zeros(16, np.float32)
    for k, terms in enumerate(_COFACTORS):
        for j, t in enumerate(terms.split()):
            a, b, c = (int(x) for x in t[1:].split(","))
            p = (e[a] * e[b]) * e[c]
            inv[k] = (p if t[0] == "+" else -p) if j == 0 else (inv[k] + p if t[0] == "+" else inv[k] - p)
    det = e[0] * inv[0] + e[1] * inv[4] + e[2] * inv[8] + e[3] * inv[12]
    return (inv * (np.float32(1) / det)).reshape(4, 4)


def _dot(a, b):
    return (a[..., 0] * b[..., 0] + a[..., 1] * b[..., 1]) + a[..., 2] * b[..., 2]


def _cross(a, b):
    return np.stack([a[..., 1] * b[..., 2] - a[..., 2] * b[..., 1], a[..., 2] * b[..., 0] - a[..., 0] * b[..., 2],
                     a[..., 0] * b[..., 1] - a[..., 1] * b[..., 0]], -1)


def _sat(z):
    z = np.where(np.isnan(z), 0, z).astype(np.float64)
    return np.clip(z, -2147483648, 2147483647).astype(np.int64)      # float32 values: the truncation is exact


class _View32:
    """Camera, projected vertices and pixel rays of one view in binary32."""

    def __init__(self, E, K, v, W, H):
        E4, K4 = np.eye(4, dtype=np.float32), np.eye(4, dtype=np.float32)
        E4[:3], K4[:3, :3] = E.reshape(3, 4), K.reshape(3, 3)
        M = np.zeros((4, 4), np.float32)
        for r in range(4):
            for c in range(4):
                M[r, c] = ((K4[r, 0] * E4[0, c] + K4[r, 1] * E4[1, c]) + K4[r, 2] * E4[2, c]) + K4[r, 3] * E4[3, c]
        self.E, self.K = E4, K4
        P, Ei = _inverse32(M), _inverse32(E4)
        self.o = Ei[:3, 3] / Ei[3, 3]
        self.os = self.o / np.float32(1000)
        e, k = E4, K4
        cam = np.stack([((e[r, 0] * v[:, 0] + e[r, 1] * v[:, 1]) + e[r, 2] * v[:, 2]) + e[r, 3] for r in range(3)], -1)
        x, y, z = (((cam[:, 0] * k[r, 0] + cam[:, 1] * k[r, 1]) + cam[:, 2] * k[r, 2]) for r in range(3))
        z = np.where(z > np.float32(1e-7), z, np.float32(1e-5))
        self.p = np.stack([x / z, y / z, z], -1)
        px, py = np.meshgrid(np.arange(W, dtype=np.float32) + np.float32(0.5),
                             np.arange(H, dtype=np.float32) + np.float32(0.5))
        tx, ty, tz = px * np.float32(1000), py * np.float32(1000), np.float32(1000)
        d = np.stack([((P[r, 0] * tx + P[r, 1] * ty) + P[r, 2] * tz) + P[r, 3] for r in range(3)], -1) - self.o
        self.d = (d * (np.float32(1) / np.sqrt(_dot(d, d)))[..., None]).reshape(-1, 3)

    def boxes(self, faces, W, H):
        q, h = self.p[faces], np.float32(0.5)
        lo = [_sat(np.maximum(q[..., a].min(1) - h, 0)) for a in (0, 1)]
        hi = [_sat(np.minimum(q[..., a].max(1) + h, np.float32(n - 1))) for a, n in ((0, W), (1, H))]
        w, h = np.maximum(hi[0] - lo[0] + 1, 0), np.maximum(hi[1] - lo[1] + 1, 0)
        return lo[0], lo[1], w, np.where(w > 0, h, 0)


def _bary32(v0, v1, v2, N, os_, d):
    """Barycentrics of unit rays d from os_ (scaled by 1/1000) on scaled triangles; -1 on a miss."""
    ndr = _dot(d, N)
    t = (_dot(v0, N) - _dot(np.broadcast_to(os_, N.shape), N)) / ndr
    P = os_ + t[:, None] * d
    a, b, c = _dot(N, _cross(v2 - v1, P - v1)), _dot(N, _cross(v0 - v2, P - v2)), _dot(N, _cross(v1 - v0, P - v0))
    miss = (np.abs(ndr) < np.float32(1e-7)) | (t < 0) | (c < 0) | (a < 0) | (b < 0)
    den = _dot(N, N)
    a, b = a / den, b / den
    abc = np.stack([a, b, (np.float32(1) - a) - b], -1)
    abc[miss] = -1
    return abc


def _visible(view, vs, faces, W, H):
    """The face that each pixel of a view shows (-1: none) and its binary32 barycentrics."""
    keys = np.full(W * H, ~np.uint64(0), np.uint64)
    x0, y0, w, h = view.boxes(faces, W, H)
    area = w * h
    ids = np.nonzero(area)[0]
    step = 2_000_000
    starts = np.concatenate([[0], np.cumsum(area[ids])])
    at = 0
    while at < len(ids):
        end = max(at + 1, int(np.searchsorted(starts, starts[at] + step, side="right")) - 1)
        f = np.repeat(ids[at:end], area[ids[at:end]])
        k = np.arange(starts[at], starts[end]) - np.repeat(starts[at:end], area[ids[at:end]])
        pix = (y0[f] + k // w[f]) * W + x0[f] + k % w[f]
        v0, v1, v2 = (vs[faces[f, i]] for i in range(3))
        N = _cross(v1 - v0, v2 - v0)
        abc = _bary32(v0, v1, v2, N, view.os, view.d[pix])
        ok = np.all((abc >= np.float32(-0.001)) & (abc <= np.float32(1.001)), -1)
        abc, f, pix = abc[ok], f[ok], pix[ok]
        z = [view.p[faces[f, i], 2] for i in range(3)]
        zq = _sat((np.float32(1) / ((abc[:, 0] / z[0] + abc[:, 1] / z[1]) + abc[:, 2] / z[2])) * np.float32(10000))
        key = ((zq + 2147483648).astype(np.uint64) << np.uint64(32)) | f.astype(np.uint64)
        np.minimum.at(keys, pix, key)
        at = end
    face = np.where(keys == ~np.uint64(0), -1, (keys & np.uint64(0xffffffff)).astype(np.int64))
    on = np.nonzero(face >= 0)[0]
    v0, v1, v2 = (vs[faces[face[on], i]] for i in range(3))
    return face, on, _bary32(v0, v1, v2, _cross(v1 - v0, v2 - v0), view.os, view.d[on])


def _normals64(v, faces):
    """Unnormalised vertex normals: the sum of the incident faces' cross products, each face once per vertex."""
    n = torch.linalg.cross(v[faces[:, 1]] - v[faces[:, 0]], v[faces[:, 2]] - v[faces[:, 0]])
    out = torch.zeros_like(v)
    for i in range(3):
        once = torch.ones(len(faces), dtype=torch.bool)
        for j in range(i):
            once &= faces[:, i] != faces[:, j]
        out = out.index_add(0, faces[:, i], n * once[:, None])
    return out


def _light64(n, sh):
    x, y, z = n.unbind(-1)
    Y = torch.stack([torch.ones_like(x), y, z, x, x * y, z * y, 3 * z * z - 1, x * z, x * x - y * y], -1)
    return Y @ sh.view(3, 9).T


def _view64(case, s, b, c, faces, img):
    """One view's outputs in 64 bits and, with a backward, the scalar whose gradient its backward is."""
    W, H, ft = case["width"], case["height"], torch.from_numpy(faces).long()
    f32 = np.float32
    v32 = s["vpos"][b].detach().numpy().astype(f32)
    view = _View32(s["extr"][b, c], s["intr"][b, c], v32, W, H)
    face, on, abc32 = _visible(view, v32 / f32(1000), faces, W, H)
    fc = face[on]
    tri = ft[fc]
    # values: ray, barycentrics, normal
    T = lambda a: torch.from_numpy(np.asarray(a, np.float64))
    E, K = T(view.E), T(view.K)
    px, py = T(on % W) + 0.5, T(on // W) + 0.5
    o, d = T(view.o), T(view.d[on])                  # the ray is the binary32 one
    v = s["vpos"][b]
    v0, v1, v2 = v[tri[:, 0]], v[tri[:, 1]], v[tri[:, 2]]

    def bary(v0, v1, v2):
        N = torch.linalg.cross(v1 - v0, v2 - v0)
        P = o + (((v0 - o) * N).sum(-1) / (d * N).sum(-1))[:, None] * d
        den = (N * N).sum(-1)
        a = (N * torch.linalg.cross(v2 - v1, P - v1)).sum(-1) / den
        bb = (N * torch.linalg.cross(v0 - v2, P - v2)).sum(-1) / den
        cos = ((d * N).sum(-1) / den.sqrt()).abs().detach()
        dead = (cos < 0.001) | ((den * den).detach() < 0.001)        # no gradient through a grazing hit
        abc = torch.stack([a, bb, 1 - a - bb], -1)
        return torch.where(dead[:, None], abc.detach(), abc)

    # the barycentrics are part of the binary32 contract too: what follows them takes their binary32 values, and its
    # derivatives at them
    abc = bary(v0, v1, v2)
    exact_abc, hit = abc.detach(), T(abc32)
    abc = hit + (abc - exact_abc)
    vn = _normals64(v, ft)
    vn32 = vn.detach().numpy().astype(f32)
    un = (vn[tri] * abc[..., None]).sum(1)
    n = un / un.norm(dim=-1, keepdim=True)
    u32 = (vn32[tri.numpy()] * abc32[..., None]).astype(f32)
    u32 = (u32[:, 0] + u32[:, 1]) + u32[:, 2]
    turned = torch.from_numpy(_dot(u32 / np.sqrt(_dot(u32, u32))[:, None], view.d[on]) > 0)
    n = n + torch.where(turned[:, None], -2 * n.detach(), torch.zeros(()).double())      # the turn takes no gradient
    lit = (case["shading"] == "shaded" and case["albedo"] not in ("foregroundMask", "normal")) or case["albedo"] == "lighting"
    L = _light64(n, s["sh"][b, c]) if lit else torch.ones_like(n)
    blend = texel = None
    if case["albedo"] == "vertexColor":
        alb = (s["vcol"][b][tri] * hit[..., None]).sum(1)
    elif case["albedo"] == "textured":
        tw, th = case["tex_w"], case["tex_h"]
        uv = s["uv"][fc].astype(f32)
        one = f32(1)
        fx = (uv[:, 0, 0] * abc32[:, 0] + uv[:, 1, 0] * abc32[:, 1]) + uv[:, 2, 0] * abc32[:, 2]
        fy = ((one - uv[:, 0, 1]) * abc32[:, 0] + (one - uv[:, 1, 1]) * abc32[:, 1]) + (one - uv[:, 2, 1]) * abc32[:, 2]
        fx = np.minimum(np.maximum(fx * f32(tw), f32(0)), f32(tw - 1))
        fy = np.minimum(np.maximum(fy * f32(th), f32(0)), f32(th - 1))
        lu, lv = _sat(fx - f32(0.5)), _sat(fy - f32(0.5))
        flat = s["tex"][b].reshape(-1, 3)
        cell = lambda u, w_: flat[np.clip(w_, 0, th - 1) * tw + np.clip(u, 0, tw - 1)]
        alb = texel = cell(lu, lv)
        U, V = T(fx) - T(lu), T(fy) - T(lv)
        su, sv, tu, tv = (x[:, None] for x in (U - 0.5, V - 0.5, 1.5 - U, 1.5 - V))
        blend = sv * (su * cell(lu, lv) + tu * cell(lu + 1, lv)) + tv * (su * cell(lu, lv + 1) + tu * cell(lu + 1, lv + 1))
    elif case["albedo"] == "normal":
        alb = (1 + n) / 2
    else:
        alb = torch.ones_like(n)
    render = torch.zeros((W * H, 3), dtype=torch.float64)
    render[:, 1] = 1.0
    render[on] = (L * alb).detach()
    bout = torch.zeros((W * H, 2), dtype=torch.float64)
    bout[on] = exact_abc[:, :2]
    out = dict(bary=bout.view(H, W, 2), render=render.view(H, W, 3), vnormal=vn.detach())
    if img is None:
        return out, None
    g, target, g_target = (x[b, c].double() if x is not None else None for x in img)
    g = 2 * (out["render"] - target) if case["entry"] == "dropin" else g
    gp = g.reshape(-1, 3)[on]
    if case["albedo"] == "textured":
        energy = (gp * L * blend.detach()).sum() + (gp * L.detach() * texel * (~turned)[:, None]).sum()
    else:
        energy = (gp * L * alb).sum()
    if g_target is not None:
        du, dv = torch.zeros((H, W, 3)).double(), torch.zeros((H, W, 3)).double()
        for y in (-1, 0, 1):
            for x in (-1, 0, 1):
                if x or y:
                    I = torch.roll(target, (-y, -x), (0, 1)) / (x * x + y * y)
                    du, dv = du + x * I, dv + y * I
        inner = (px >= 2.5) & (py >= 2.5) & (px < W - 1.5) & (py < H - 1.5)
        q = [((g_target * t).sum(-1).reshape(-1)[on] / 4.0) * inner for t in (du, dv)]
        X = (torch.stack([v0, v1, v2], 1) * hit[..., None]).sum(1)
        p = X @ (K @ E)[:3, :3].T + (K @ E)[:3, 3]
        energy = energy + (q[0] * p[:, 0] / p[:, 2] + q[1] * p[:, 1] / p[:, 2]).sum()
    return out, energy


def _exact_render(case, seed):
    s = _scene(case, seed)
    faces = s["faces"]
    B, C, W, H = case["batch"], case["views"], case["width"], case["height"]
    tests = sum(int(np.prod(_View32(s["extr"][b, c], s["intr"][b, c], s["vpos"][b], 1, 1).boxes(faces, W, H)[2:], 0).sum())
                for b in range(B) for c in range(C))
    leaves = {k: torch.from_numpy(s[k].astype(np.float64)).requires_grad_(True) for k in ("vpos", "vcol", "tex", "sh")}
    if tests > MAX_EXACT_CANDIDATES:
        if case["entry"] == "dropin":
            return None
        vn = [_normals64(leaves["vpos"][b].detach(), torch.from_numpy(faces).long()) for b in range(B)]
        return dict(bary=None, face=None, render=None, vnormal=torch.stack(vn)[:, None].repeat(1, C, 1, 1),
                    grads=[None] * 4)
    s = dict(s, **leaves)
    img = _images(case, seed) if case["backward"] else None
    outs, grads = [], {k: torch.zeros_like(t) for k, t in leaves.items()}
    for b in range(B):
        for c in range(C):
            out, energy = _view64(case, s, b, c, faces, img)
            outs.append(out)
            if energy is not None and energy.requires_grad:
                for (k, t), gr in zip(leaves.items(), torch.autograd.grad(energy, list(leaves.values()), allow_unused=True)):
                    if gr is not None:
                        grads[k] += gr
    res = {k: torch.stack([o[k] for o in outs]).view(B, C, *outs[0][k].shape) for k in outs[0]}
    res["face"] = None
    if case["entry"] == "dropin":
        del res["vnormal"]
    if case["backward"]:
        res["grads"] = [grads[k] for k in ("vpos", "vcol", "tex", "sh")]
    return res


def _rodrigues64(w):
    K = torch.zeros(w.shape[0], 3, 3, dtype=torch.float64)
    for i, j, k, sign in ((2, 1, 0, 1), (1, 2, 0, -1), (0, 2, 1, 1), (2, 0, 1, -1), (1, 0, 2, 1), (0, 1, 2, -1)):
        K = K + sign * torch.nn.functional.one_hot(torch.tensor(3 * i + j), 9).view(3, 3).double() * w[:, k, None, None]
    return torch.linalg.matrix_exp(K)


def _exact_shape(case, seed):
    s = {k: t.double().cpu() for k, t in _shape_inputs(case, seed).items()}
    a, p = s["alpha"].requires_grad_(True), s["pose"].requires_grad_(True)
    X = s["template"] - s["centre"] + (a @ s["basis"]).view(a.shape[0], -1, 3)
    v = X @ _rodrigues64(p[:, :3]).transpose(1, 2) + s["centre"] + 100.0 * p[:, None, 3:]
    ga, gp = torch.autograd.grad(v, [a, p], grad_outputs=s["g"])
    return dict(v=v.detach(), alpha=ga, pose=gp)


def _net64(sd, x):
    for i in range(len(NET)):
        w = sd["w%d" % i].permute(0, 3, 1, 2)
        x = torch.relu(torch.nn.functional.conv2d(x, w, sd["b%d" % i], stride=2, padding=1))
    x = x.permute(0, 2, 3, 1).reshape(x.shape[0], -1)
    return (x @ sd["w6"].view(128, -1).T + sd["b6"])[:, :113]


def exact(case, seed):
    kind = case["kind"]
    if kind == "render":
        return _exact_render(case, seed)
    if kind == "multi":
        res = []
        for s in _multi_scenes(case, seed):
            vn = _normals64(torch.from_numpy(s.vpos[0]).double(), torch.from_numpy(s.faces).long())
            res.append(dict(face=None, bary=None, render=None, vnormal=vn[None, None].repeat(1, s.C, 1, 1), g_pos=None,
                            g_col=None, g_sh=None))
        return res
    if kind == "fit":
        return None       # its rendered vertices are themselves computed in binary32, and decide what is seen
    if kind == "shape":
        return _exact_shape(case, seed)
    sd = {k: w.double().requires_grad_(True) for k, w in _net_weights(seed).items() if k != "features"}
    if kind == "train":
        x, y = _train_inputs(case, seed)
        out = _net64(sd, x.double().permute(0, 3, 1, 2))
        names = ["w%d" % i for i in range(7)] + ["b%d" % i for i in range(7)]
        gr = torch.autograd.grad(((out - y.double()) ** 2).mean(), [sd[k] for k in names])
        gr[0][..., 3:] = 0.0
        return dict(out=out.detach(), gw=list(gr[:7]), gb=list(gr[7:]))
    r = _propose_inputs(case, seed).double()
    B, V, R = r.shape[:3]
    cols = int(math.ceil(math.sqrt(V)))
    r = r.view(B, V, 128, R // 128, 128, R // 128, 3).mean((3, 5))
    x = torch.zeros((B, 256, 256, 8), dtype=torch.float64)
    for i in range(V):
        y0, x0 = 128 * (i // cols), 128 * (i % cols)
        x[:, y0:y0 + 128, x0:x0 + 128, :3] = r[:, i]
    with torch.no_grad():
        return dict(x=x, out=_net64(sd, x.permute(0, 3, 1, 2)))
