"""The measured work of this framework: frames, stages, sorts and training passes through its public entry points.

A case is a dict of plain values.  Its "kind" names the path:

  frame   one frame of a loaded renderer (pipeline.Renderer.render): the viewer's loop
  stages  the reference's stage order, one entry point per stage (pipeline.reference_frame)
  sort    the stable key/value sort (pipeline.sort_kv) on a program's own pairs
  train   forward + backward of one or many views (diff.render, diff.render_batch_flat)
  graph   the same captured once and replayed (diff.GraphedStep)

Scenes are synthetic with the distributions of vkgs_amd.scene, made on the GPU from the seed alone:

  cloud   positions N(0, 2) around the origin, orbit radius 6: splats from near the camera to far
  town    64 anisotropic clusters in a 40 x 10 x 40 box and a ground plane, radius 15: a captured place,
          about a third of it in view
  city    256 clusters in an 80 x 20 x 80 box, radius 60: a large scene seen from afar, nearly all in view
"""
import math

import numpy as np
import torch

from vkgs_amd import diff as D
from vkgs_amd import pipeline as P
from vkgs_amd import scene as S

RADIUS = {"cloud": 6.0, "town": 15.0, "city": 60.0}


def listed():
    return [
        # the smallest frame: a thumbnail of a small object, where launches and latency are all there is
        {"name": "frame_thumbnail", "kind": "frame", "scene": "cloud", "n": 5000, "w": 320, "h": 240, "triangles": False},
        # a single scanned object in a viewer window
        {"name": "frame_100k", "kind": "frame", "scene": "cloud", "n": 100_000, "w": 1600, "h": 900, "triangles": False},
        # a captured place, the camera among its splats
        {"name": "frame_1m", "kind": "frame", "scene": "town", "n": 1_000_000, "w": 1600, "h": 900, "triangles": False},
        # the frame rate that the reference is quoted on: 6M splats at 1600x900
        {"name": "frame_6m", "kind": "frame", "scene": "city", "n": 6_000_000, "w": 1600, "h": 900, "triangles": False},
        # an odd size near 4K, whose tile rectangles need more than 32 bits
        {"name": "frame_4k_ragged", "kind": "frame", "scene": "town", "n": 2_345_677, "w": 3839, "h": 2159,
         "triangles": False},
        # the reference's exact triangle coverage, the renderer's parity option
        {"name": "frame_triangles", "kind": "frame", "scene": "town", "n": 400_003, "w": 1279, "h": 719, "triangles": True},
        # a program that keeps the reference's stages apart and replaces them one by one
        {"name": "stages_300k", "kind": "stages", "scene": "town", "n": 300_001, "w": 1279, "h": 719},
        # a depth sort of a program's own keys, all 32 bits
        {"name": "sort_4m", "kind": "sort", "n": 4_000_037, "bits": 32},
        # the smallest training step: one small view of a small object
        {"name": "train_small", "kind": "train", "scene": "cloud", "n": 20_000, "views": 1, "w": 320, "h": 240},
        # one optimizer step's view of a mid-sized scene
        {"name": "train_500k", "kind": "train", "scene": "cloud", "n": 500_000, "views": 1, "w": 1024, "h": 1024},
        # a batch of views of one scene in one call, at several sizes
        {"name": "train_batch", "kind": "train", "scene": "town", "n": 1_500_000, "views": 12, "w": 1000, "h": 750},
        # a short training loop captured into a graph, spatial processing order on
        {"name": "train_graph", "kind": "graph", "scene": "cloud", "n": 60_000, "views": 6, "w": 480, "h": 360},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "stages", "sort", "train", "train", "graph"])
    if kind == "sort":
        return {"kind": kind, "n": _log_int(rng, 5_000, 8_000_000), "bits": rng.choice([13, 24, 30, 32])}
    w = _log_int(rng, 200, 1920)
    h = max(64, int(w * rng.uniform(0.5, 1.0)))
    scene = rng.choice(["cloud", "town", "city"])
    # near, dense clouds cover many tiles per splat: fewer of them
    top = 500_000 if scene == "cloud" else 4_000_000
    if kind == "frame":
        return {"kind": kind, "scene": scene, "n": _log_int(rng, 3_000, top), "w": w, "h": h,
                "triangles": rng.random() < 0.15}
    if kind == "stages":
        # reference_frame() gives the draw four tile pairs a splat and a million: near clouds need more
        top = 40_000 if scene == "cloud" else 2_000_000
        return {"kind": kind, "scene": scene, "n": _log_int(rng, 3_000, top), "w": w, "h": h}
    if kind == "graph":
        return {"kind": kind, "scene": scene, "n": _log_int(rng, 3_000, 200_000), "views": rng.randint(2, 8),
                "w": min(w, 640), "h": min(h, 480)}
    views = rng.choice([1, 1, 2, 5])
    return {"kind": kind, "scene": scene, "n": _log_int(rng, 3_000, top // (2 * views)), "views": views,
            "w": min(w, 1200), "h": min(h, 1000)}


# ------------------------------------------------------------------ inputs ---


def _rows(kind, n, seed):
    """(n, 62) float32 PLY rows of a scene on the GPU, with the distributions of vkgs_amd.scene."""
    g = torch.Generator(device="cuda").manual_seed(seed * 1009 + 17)
    randn = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    rand = lambda *s: torch.rand(*s, generator=g, device="cuda")  # noqa: E731
    c = S.COL
    rows = torch.zeros((n, S.STRIDE), device="cuda")
    if kind == "cloud":
        rows[:, 0:3] = 2.0 * randn(n, 3)
        logscale, logit = (-4.0, 0.5), (0.0, 1.5)
    else:
        clusters, box = (64, (40.0, 10.0, 40.0)) if kind == "town" else (256, (80.0, 20.0, 80.0))
        size = torch.tensor(box, device="cuda")
        centers = rand(clusters, 3) * size - torch.tensor([box[0] / 2, 0.0, box[2] / 2], device="cuda")
        stds = 0.2 + rand(clusters, 3) * (0.1 * max(box) - 0.2)
        rot = torch.linalg.qr(randn(clusters, 3, 3).cpu())[0].cuda()
        which = torch.randint(clusters, (n,), generator=g, device="cuda")
        local = randn(n, 3) * stds[which]
        pos = centers[which] + (rot[which] * local[:, None, :]).sum(-1)
        ground = rand(n) < 0.2
        flat = (rand(n, 3) - 0.5) * size
        flat[:, 1] = 0.02 * randn(n)
        rows[:, 0:3] = torch.where(ground[:, None], flat, pos)
        logscale, logit = (-4.5, 0.8), (0.5, 2.0)
    rows[:, c["scale_0"]:c["scale_0"] + 3] = logscale[0] + logscale[1] * randn(n, 3)
    rows[:, c["rot_0"]:c["rot_0"] + 4] = torch.nn.functional.normalize(randn(n, 4), dim=1)
    rows[:, c["opacity"]] = logit[0] + logit[1] * randn(n)
    rows[:, c["f_dc_0"]:c["f_dc_0"] + 3] = 0.5 * randn(n, 3)
    rows[:, c["f_rest_0"]:c["f_rest_0"] + 45] = 0.05 * randn(n, 45)
    return rows


def _ply_buffer(rows):
    buf = np.empty(60 + rows.numel(), np.uint32)
    buf[:60] = S.standard_offsets()
    buf[60:] = rows.reshape(-1).cpu().numpy().view(np.uint32)
    return buf


def _params(rows, requires_grad=True):
    """The five parameter tensors of vkgs_amd.diff from PLY rows."""
    c = S.COL
    sh = torch.from_numpy(S.standard_offsets()[10:58].astype(np.int64)).cuda()
    p = {"means": rows[:, 0:3], "log_scales": rows[:, c["scale_0"]:c["scale_0"] + 3],
         "quats": rows[:, c["rot_0"]:c["rot_0"] + 4], "opacity_logits": rows[:, c["opacity"]], "sh": rows[:, sh]}
    return {k: v.clone().contiguous().requires_grad_(requires_grad) for k, v in p.items()}


def _cameras(case, seed):
    """One orbit camera per view: the first at the scene's own radius, the others around and nearer or
    farther, at the case's size and at three quarters and half of it."""
    rng = np.random.default_rng([seed, 7])
    cams = []
    for i in range(case.get("views", 1)):
        part = (4, 3, 2)[i % 3]
        w, h = max(16, case["w"] * part // 4), max(16, case["h"] * part // 4)
        r = RADIUS[case["scene"]] * (1.0 if i == 0 else rng.uniform(0.8, 1.4))
        cams.append(S.orbit_camera(w, h, r, phi=rng.uniform(0.6, 1.0), theta=rng.uniform(0.0, 2 * math.pi)))
    return cams


def _target(cams, seed):
    """dL/dimage of every pixel, flat (P, 4): what a mean loss over each view sends back."""
    g = torch.Generator(device="cuda").manual_seed(seed * 1009 + 23)
    parts = [(0.5 + torch.rand((c.screen_size[0] * c.screen_size[1], 4), generator=g, device="cuda"))
             / (c.screen_size[0] * c.screen_size[1]) for c in cams]
    return torch.cat(parts)


def _sort_pairs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed * 1009 + 29)
    hi = 1 << case["bits"]
    key = torch.randint(0, hi, (case["n"],), generator=g, device="cuda", dtype=torch.int64)
    key = torch.where(key >= 1 << 31, key - (1 << 32), key).to(torch.int32)
    return key, torch.arange(case["n"], device="cuda", dtype=torch.int32)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "sort":
        key, value = _sort_pairs(case, seed)
        count = torch.full((1,), case["n"], dtype=torch.int32, device="cuda")
        return {"case": case, "key": key, "value": value, "count": count}
    rows = _rows(case["scene"], case["n"], seed)
    cams = _cameras(case, seed)
    if kind == "frame":
        r = P.Renderer(case["n"])
        r.load_buffer(_ply_buffer(rows), case["n"])
        if case["triangles"]:
            r.set_config(tile_w=8, tile_h=8, triangles=True)
        out = torch.empty((case["h"], case["w"], 4), dtype=torch.float32, device="cuda")
        # the first frame sizes the tile lists, and is drawn again where they were too short, as pygs does
        for _ in range(3):
            r.render(cams[0], out=out)
            if r.frame_info()[0] == 0:
                break
        return {"case": case, "renderer": r, "cam": cams[0], "out": out}
    if kind == "stages":
        return {"case": case, "storage": P.parse_ply(_ply_buffer(rows), case["n"]), "cam": cams[0]}
    params = _params(rows)
    grad = _target(cams, seed)
    state = {"case": case, "params": params, "cams": cams, "grad": grad}
    if kind == "graph":
        views = [(0, c) for c in cams]
        state["step"] = D.GraphedStep([params], views, lambda flat: grad * (0.5 + flat), spatial_order=True)
    return state


# -------------------------------------------------------------------- runs ---


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "frame":
        return state["renderer"].render(state["cam"], out=state["out"])
    if kind == "stages":
        f = P.reference_frame(state["cam"], state["storage"], case["w"], case["h"])
        return {k: f[k] for k in ("image", "instances", "draw_indirect", "count", "inverse")}
    if kind == "sort":
        key, value = state["key"].clone(), state["value"].clone()
        P.sort_kv(state["count"], key, value, case["bits"])
        return {"key": key, "value": value}
    params = state["params"]
    if kind == "graph":
        flat = state["step"].step()
    else:
        for t in params.values():
            t.grad = None
        if case["views"] == 1:
            img = D.render(**params, camera=state["cams"][0])
            img.backward(state["grad"].view_as(img))
            flat = img.detach().view(-1, 4)
        else:
            flat, _ = D.render_batch_flat([params], [(0, c) for c in state["cams"]])
            flat.backward(state["grad"])
            flat = flat.detach()
    return {"image": flat, "grads": {k: params[k].grad for k in D.PARAM_NAMES}}


def work(case):
    """Each splat's storage read once and each pixel written once (136 B as the renderer keeps a splat, 236 B
    of raw parameters); in training the output's gradient read and the parameters' gradients written.  The
    operations are those of the projection alone (about 500 per splat and view, three times that with its
    backward): the blend's follow from the scene.  A sort reads and writes its pairs once."""
    if case["kind"] == "sort":
        return {"bytes": 16 * case["n"], "flops": 0}
    n = case["n"]
    pixels = 0
    for i in range(case.get("views", 1)):
        part = (4, 3, 2)[i % 3]
        pixels += max(16, case["w"] * part // 4) * max(16, case["h"] * part // 4)
    if case["kind"] == "frame":
        return {"bytes": 136 * n + 16 * pixels, "flops": 500 * n}
    if case["kind"] == "stages":
        return {"bytes": 136 * n + 16 * pixels + 52 * n, "flops": 500 * n}
    return {"bytes": 2 * 236 * n + 32 * pixels, "flops": 2000 * n * case["views"]}


# ------------------------------------------------------- the same in 64 bits ---

SH0, SH1 = 0.28209479177387814, 0.4886025119029199
SH2 = (1.0925484305920792, 0.31539156525252005, 0.5462742152960396)
SH3 = (0.5900435899266435, 2.890611442640554, 0.4570457994644658, 0.3731763325901154, 1.445305721320277)


def _sh_basis(d):
    x, y, z = d.unbind(-1)
    xx, yy, zz = x * x, y * y, z * z
    return torch.stack([
        torch.full_like(x, SH0), -SH1 * y, SH1 * z, -SH1 * x,
        SH2[0] * x * y, -SH2[0] * y * z, SH2[1] * (2 * zz - xx - yy), -SH2[0] * x * z, SH2[2] * (xx - yy),
        -SH3[0] * y * (3 * xx - yy), SH3[1] * x * y * z, -SH3[2] * y * (4 * zz - xx - yy),
        SH3[3] * z * (2 * zz - 3 * xx - 3 * yy), -SH3[2] * x * (4 * zz - xx - yy), SH3[4] * z * (xx - yy),
        -SH3[0] * x * (xx - 3 * yy)], -1)


def _depth_order(means, cam):
    """The visible splats, nearest first.  The order is part of the format and not a computed number: the key
    is fl(1 - z) of single-precision arithmetic, equal keys go by id."""
    f = np.float32
    proj = np.frombuffer(bytes(cam.projection), f).reshape(4, 4)
    view = np.frombuffer(bytes(cam.view), f).reshape(4, 4)  # [column][row]
    pv = np.zeros((4, 4), f)
    for col in range(4):
        for row in range(4):
            s = proj[0][row] * view[col][0]
            for k in range(1, 4):
                s = f(s + proj[k][row] * view[col][k])
            pv[col][row] = s
    x, y, z = means.float().unbind(-1)
    clip = []
    for row in range(4):
        s = float(pv[0][row]) * x
        s = s + float(pv[1][row]) * y
        s = s + float(pv[2][row]) * z
        clip.append(s + float(pv[3][row]))
    nx, ny, nz = (clip[i] / clip[3] for i in range(3))
    key = 1.0 - nz
    vis = (nx.abs() <= 1) & (ny.abs() <= 1) & (nz >= 0) & (nz <= 1)
    ids = vis.nonzero()[:, 0]
    return ids[torch.sort(key[ids], stable=True).indices].flip(0)


def _project64(p, cam, ids, half_sh):
    """Per visible splat: pixel centre (2), pixel covariance's inverse (3), inverse rot_scale (4, detached),
    colour (3), opacity, all in 64 bits."""
    m = lambda a: torch.tensor(np.frombuffer(bytes(a), np.float32).reshape(4, 4).T.astype(np.float64), device="cuda")  # noqa: E731
    proj, view = m(cam.projection), m(cam.view)
    eye = torch.tensor(list(cam.camera_position), dtype=torch.float64, device="cuda")
    w, h = cam.screen_size[0], cam.screen_size[1]
    pos = p["means"][ids]
    q = torch.nn.functional.normalize(p["quats"][ids], dim=1)
    qw, qx, qy, qz = q.unbind(-1)
    R = torch.stack([1 - 2 * (qy * qy + qz * qz), 2 * (qx * qy - qw * qz), 2 * (qx * qz + qw * qy),
                     2 * (qx * qy + qw * qz), 1 - 2 * (qx * qx + qz * qz), 2 * (qy * qz - qw * qx),
                     2 * (qx * qz - qw * qy), 2 * (qy * qz + qw * qx), 1 - 2 * (qx * qx + qy * qy)], -1).view(-1, 3, 3)
    L = R * p["log_scales"][ids].exp()[:, None, :]
    pv = pos @ view[:3, :3].T + view[:3, 3]
    x, y, z = pv.unbind(-1)
    zero = torch.zeros_like(z)
    J = torch.stack([-1 / z, zero, x / z ** 2, zero, -1 / z, y / z ** 2], -1).view(-1, 2, 3)
    G = proj[:2, :2] @ J @ view[:3, :3] @ L  # cov2 = G G^T
    cov = G @ G.transpose(1, 2)
    a, b, c = cov[:, 0, 0] + 1.0 / w / w, cov[:, 1, 1] + 1.0 / h / h, cov[:, 0, 1]
    clip = torch.cat([pv, torch.ones_like(pv[:, :1])], 1) @ proj.T
    ndc = clip[:, :3] / clip[:, 3:]
    hw, hh = 0.5 * w, 0.5 * h
    centre = torch.stack([(ndc[:, 0] + 1) * hw, (ndc[:, 1] + 1) * hh], -1)
    det = a * b - c * c
    conic = torch.stack([b / det / hw ** 2, -c / det / (hw * hh), a / det / hh ** 2], -1)
    with torch.no_grad():
        d = torch.sqrt((a - b) ** 2 + 4 * c * c)
        s0, s1 = torch.sqrt(0.5 * (a + b + d)), torch.sqrt(0.5 * (a + b - d))
        cos2, sin2 = (a - b) / d, 2 * c / d
        ct = torch.sqrt(((1 + cos2) / 2).clamp_min(0))
        st = torch.copysign(torch.sqrt(((1 - cos2) / 2).clamp_min(0)), sin2)
        rs = torch.stack([hw * s0 * ct, -hw * s1 * st, hh * s0 * st, hh * s1 * ct], -1).view(-1, 2, 2)
        inv = torch.linalg.inv(rs)
        ext = 3 * rs.abs().sum(2)
    dirs = torch.nn.functional.normalize(pos - eye, dim=1)
    sh = p["sh"][ids]
    sh = sh.half().double() if half_sh else sh
    colour = torch.clamp_min((sh.view(-1, 3, 16) * _sh_basis(dirs)[:, None, :]).sum(-1) + 0.5, 0)
    opacity = torch.sigmoid(p["opacity_logits"][ids])
    return torch.cat([centre, conic, colour, opacity[:, None]], 1), inv, ext, (ndc[:, 2] >= 0) & (ndc[:, 2] < 1)


def _tile_pairs(centre, ext, ok, w, h):
    """(tile, visible index) pairs over 8x8 tiles, nearest first within a tile, and the tile grid's width."""
    lo = torch.floor((centre - ext - 1) / 8).long().clamp_min(0)
    top = torch.tensor([(w - 1) // 8, (h - 1) // 8], device="cuda")
    hi = torch.minimum(torch.floor((centre + ext + 1) / 8).long(), top)
    span = (hi - lo + 1).clamp_min(0) * ok[:, None]
    cnt = span[:, 0] * span[:, 1]
    idx = torch.repeat_interleave(torch.arange(len(cnt), device="cuda"), cnt)
    k = torch.arange(len(idx), device="cuda") - (torch.cumsum(cnt, 0) - cnt)[idx]
    tile = (lo[idx, 1] + k // span[idx, 0]) * (top[0] + 1) + lo[idx, 0] + k % span[idx, 0]
    tile, perm = torch.sort(tile, stable=True)
    return tile, idx[perm], int(top[0]) + 1, int(top[0] + 1) * int(top[1] + 1)


def _view64(p, cam, clamp, half_sh, grad=None):
    """(H * W, 4) image in 64 bits; with grad (H * W, 4), adds the gradients to p's .grad."""
    w, h = cam.screen_size[0], cam.screen_size[1]
    ids = _depth_order(p["means"].detach(), cam)
    with torch.set_grad_enabled(grad is not None):
        rec, inv, ext, ok = _project64(p, cam, ids, half_sh)
    leaf = rec.detach().requires_grad_(grad is not None)
    tile, idx, tiles_x, tiles = _tile_pairs(leaf.detach()[:, :2], ext, ok, w, h)
    image = torch.zeros((w * h, 4), dtype=torch.float64, device="cuda")
    image[:, 3] = 1.0
    length = torch.bincount(tile, minlength=tiles)
    first = torch.cumsum(length, 0) - length
    order = torch.argsort(length, descending=True)
    lengths = length[order].tolist()
    at, px = 0, torch.arange(64, device="cuda")
    while at < tiles and lengths[at] > 0:
        n = max(1, min(tiles - at, (1 << 24) // (64 * lengths[at])))
        t = order[at:at + n]
        at += n
        e = torch.arange(lengths[at - n], device="cuda")
        valid = e[None, :] < length[t][:, None]
        pick = idx[torch.where(valid, first[t][:, None] + e[None, :], 0)]
        X = (t % tiles_x)[:, None] * 8 + px % 8
        Y = torch.div(t, tiles_x, rounding_mode="floor")[:, None] * 8 + px // 8
        with torch.set_grad_enabled(grad is not None):
            r = leaf[pick]  # (tiles, entries, 9)
            dx = X[:, None, :] + 0.5 - r[..., 0:1]
            dy = Y[:, None, :] + 0.5 - r[..., 1:2]
            with torch.no_grad():
                i = inv[pick]
                cover = (i[..., 0, 0:1] * dx + i[..., 0, 1:2] * dy).abs() <= 3
                cover &= (i[..., 1, 0:1] * dx + i[..., 1, 1:2] * dy).abs() <= 3
                cover &= valid[..., None]
            power = r[..., 2:3] * dx * dx + 2 * r[..., 3:4] * dx * dy + r[..., 4:5] * dy * dy
            alpha = torch.where(cover, r[..., 8:9] * torch.exp(-0.5 * power), 0.0)
            if clamp:
                alpha = alpha.clamp_max(0.999)
            T = torch.cumprod(1 - alpha, 1)
            ta = alpha * torch.cat([torch.ones_like(T[:, :1]), T[:, :-1]], 1)
            rgb = (ta[..., None] * r[:, :, None, 5:8]).sum(1)
            out = torch.cat([rgb, ((alpha * ta).sum(1) + T[:, -1])[..., None]], -1)
        inside = (X < w) & (Y < h)
        pix = (Y * w + X)[inside]
        image[pix] = out.detach()[inside]
        if grad is not None:
            out[inside].backward(grad[pix])
    if grad is not None and leaf.grad is not None:
        rec.backward(leaf.grad)
    return image


def exact(case, seed):
    """The image (and, of a training pass, the gradients) by plain torch in 64 bits: every splat composited,
    none left out below a transmittance.  None for whole numbers, for the triangle coverage, whose vertices are
    snapped to 1/256 pixel by definition, and for the graphed step, whose blend order at equal depth keys is
    the spatial one."""
    kind = case["kind"]
    if kind in ("sort", "graph") or case.get("triangles"):
        return None
    rows = _rows(case["scene"], case["n"], seed)
    cams = _cameras(case, seed)
    if kind in ("frame", "stages"):
        p = {k: v.double() for k, v in _params(rows, False).items()}
        image = _view64(p, cams[0], False, True).view(case["h"], case["w"], 4)
        if kind == "frame":
            return image
        return {"image": image, "instances": None, "draw_indirect": None, "count": None, "inverse": None}
    p = {k: v.double().requires_grad_() for k, v in _params(rows, False).items()}
    grad = _target(cams, seed).double()
    images, at = [], 0
    for c in cams:
        n = c.screen_size[0] * c.screen_size[1]
        images.append(_view64(p, c, True, False, grad[at:at + n]))
        at += n
    grads = {k: v.grad if v.grad is not None else torch.zeros_like(v) for k, v in p.items()}
    return {"image": torch.cat(images), "grads": {k: grads[k] for k in D.PARAM_NAMES}}
