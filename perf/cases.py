"""Workloads of the splatting framework, through its public entry points.

Each case is one call sequence that a program using the framework repeats: a
training frame of the drop-in renderer in one of its shading modes, a frame of
the Poisson-rate renderer over one or many views, or the per-pixel operators
and the rate network on their own.  The sizes run from the 256-splat, 64x64
scene to 1M splats at 512x512 and the 2M-surfel room seen by 16 cameras.

  listed()            the named cases
  draw(rng)           another case of the same ranges
  prepare(case, seed) the inputs and objects a program holds before the call
  run(state)          one pass; returns the outputs
  work(case)          the bytes and operations a pass cannot do without
  exact(case, seed)   float64 values of the outputs, in plain torch, where a
                      pass is a closed formula of its inputs
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "unbiased-differentiable-splatting_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

MODES = ("None", "forward", "deferred", "sphericalHarmonics", "forwardHarmonics", "silhouette")


def _dev():
    return torch.device("cuda:0")


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # a toy or preview optimisation with the renderer's default shading: launch latency counts
        {"name": "frame_small", "kind": "frame", "scene": "sphere", "splats": 4096, "views": 1, "width": 128,
         "height": 128, "samples": 40, "mode": "forward", "lamps": 2, "host_indices": False},
        # the full training frame, 1M surfels at 512x512
        {"name": "frame_large", "kind": "frame", "scene": "ellipsoids", "splats": 1_000_000, "views": 1,
         "width": 512, "height": 512, "samples": 40, "mode": "None", "lamps": 1, "host_indices": False},
        # a mini-batch of views with deferred Lambert shading, odd sizes, the renderer's
        # default of keeping the sampled indices on the host
        {"name": "frame_views", "kind": "frame", "scene": "ellipsoids", "splats": 60_003, "views": 4, "width": 301,
         "height": 203, "samples": 40, "mode": "deferred", "lamps": 4, "host_indices": True},
        # a mid-size frame under spherical-harmonics lighting with fewer samples per pixel
        {"name": "frame_harmonics", "kind": "frame", "scene": "ellipsoids", "splats": 250_000, "views": 1,
         "width": 640, "height": 480, "samples": 24, "mode": "sphericalHarmonics", "lamps": 1,
         "host_indices": False},
        # the smallest scene of the Poisson-rate renderer through autograd (the backward redraws its samples)
        {"name": "poisson_small", "kind": "render", "scene": "sphere", "splats": 256, "views": 1, "width": 64,
         "height": 64, "samples": 24, "rate": 6.0, "composite": False},
        # the Poisson-rate training frame at full size
        {"name": "poisson_large", "kind": "poisson", "scene": "ellipsoids", "splats": 1_000_000, "views": 1,
         "width": 512, "height": 512, "samples": 40, "rate": 10.0, "proposal": "bands"},
        # a batch of views inside a room, every stage over all views at once
        {"name": "poisson_room", "kind": "poisson", "scene": "room", "splats": 2_000_000, "views": 16, "width": 640,
         "height": 480, "samples": 40, "rate": 10.0, "proposal": "bands"},
        # the composited Poisson-rate estimate on an ordinary small scene
        {"name": "poisson_composite", "kind": "render", "scene": "sphere", "splats": 20_011, "views": 2,
         "width": 200, "height": 150, "samples": 40, "rate": 8.0, "composite": True},
        # z-sort and compositing with more samples per pixel than a wavefront has lanes
        {"name": "compositing_wide", "kind": "compositing", "splats": 100_000, "views": 1, "width": 256,
         "height": 192, "samples": 100},
        # the float64 operator chain of a gradient check or a double-precision optimisation
        {"name": "operators_double", "kind": "double", "splats": 20_011, "views": 1, "width": 151, "height": 97,
         "samples": 40},
        # the operators behind the normal and surface regularisers: rows per sampled slot, their
        # adjoint, and every splat's nearest co-sampled splats
        {"name": "neighbours", "kind": "neighbours", "splats": 100_000, "views": 2, "width": 256, "height": 256,
         "samples": 16, "channels": 3, "nearest": 10},
        # one training evaluation of the per-tile rate network and its use on one image's tiles
        {"name": "rate_network", "kind": "network", "tiles": 20_480, "image_tiles": 1024},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "render", "poisson", "poisson", "compositing", "double",
                       "neighbours", "network"])
    if kind == "network":
        return {"kind": kind, "tiles": _log_int(rng, 256, 20_480), "image_tiles": _log_int(rng, 16, 1200)}
    W, H = _log_int(rng, 64, 640), _log_int(rng, 64, 480)
    if kind == "frame":
        views = rng.choice([1, 1, 2, 4])
        N = _log_int(rng, 4096, 1_000_000 // views)
        if W * H * views > 512 * 512:
            W, H = 200 + rng.randrange(56), 200 + rng.randrange(56)
        mode = rng.choice([m for m in MODES if views == 1 or m != "forwardHarmonics"])
        return {"kind": kind, "scene": rng.choice(["sphere", "ellipsoids"]),
                "splats": min(N, 400_000) if mode == "forwardHarmonics" else N, "views": views, "width": W,
                "height": H, "samples": rng.choice([16, 24, 33, 40]), "mode": mode, "lamps": rng.randrange(1, 5),
                "host_indices": rng.random() < 0.3}
    if kind == "render":
        W, H = _log_int(rng, 64, 300), _log_int(rng, 64, 300)
        rate = rng.choice([4.0, 6.0, 8.0])
        return {"kind": kind, "scene": "sphere", "splats": _log_int(rng, 256, 40_000), "views": rng.choice([1, 2]),
                "width": W, "height": H, "samples": int(4 * rate) + 8, "rate": rate,
                "composite": rng.random() < 0.5}
    if kind == "poisson":
        room = rng.random() < 0.4
        views = rng.randrange(2, 13) if room else 1
        return {"kind": kind, "scene": "room" if room else "ellipsoids", "splats": _log_int(rng, 20_000, 1_000_000),
                "views": views, "width": W, "height": H, "samples": 40, "rate": rng.choice([6.0, 10.0]),
                "proposal": rng.choice(["bands", "bands", "footprint"])}
    if kind == "compositing":
        k = rng.choice([72, 100, 128, 200, 256])
        W, H = _log_int(rng, 64, 256), _log_int(rng, 64, 192)
        return {"kind": kind, "splats": _log_int(rng, 20_000, 400_000), "views": rng.choice([1, 2]), "width": W,
                "height": H, "samples": k}
    if kind == "double":
        W, H = _log_int(rng, 32, 200), _log_int(rng, 32, 150)
        return {"kind": kind, "splats": _log_int(rng, 2000, 60_000), "views": rng.choice([1, 2]), "width": W,
                "height": H, "samples": rng.choice([12, 24, 40, 64])}
    return {"kind": kind, "splats": _log_int(rng, 10_000, 400_000), "views": rng.choice([1, 2]),
            "width": _log_int(rng, 64, 300), "height": _log_int(rng, 64, 300),
            "samples": rng.choice([16, 24, 40]), "channels": rng.choice([1, 3, 6]),
            "nearest": rng.choice([4, 8, 10])}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _cameras(case, rng):
    """World-to-camera matrices: the standard camera, turned about the vertical axis per view."""
    from splatting_amd import scenes
    M = np.stack([scenes.camera_matrix()] * case["views"])
    for v in range(case["views"]):
        a = rng.uniform(-0.7, 0.7) if v else 0.0
        R = np.eye(4, dtype=np.float32)
        R[0, 0], R[0, 2], R[2, 0], R[2, 2] = math.cos(a), math.sin(a), -math.sin(a), math.cos(a)
        M[v] = M[v] @ R
    return M.astype(np.float32)


def _scene(case, seed):
    """The surfels of a scene and its cameras."""
    from splatting_amd import scenes
    n, W, H = case["splats"], case["width"], case["height"]
    rng = np.random.default_rng([seed, 17])
    if case["scene"] == "room":
        p, nrm, s, a = scenes.box_room(n, seed=1000 + seed)
        M = scenes.room_cameras(case["views"], seed=2000 + seed, boxes=scenes.room_boxes(seed=1000 + seed))
        return scenes.Scene(p, nrm, s, a, W, H, 400.0 * W / 640.0, M)
    if case["scene"] == "sphere":
        p, nrm, s, a = scenes.unit_sphere(n, seed)
    else:
        p, nrm, s, a = (x[:n] for x in scenes.ellipsoids(64, (n + 63) // 64, seed))
    return scenes.Scene(p, nrm, s, a, W, H, 1.2 * max(W, H), _cameras(case, rng))


def _gpu(x):
    return torch.from_numpy(np.ascontiguousarray(x, np.float32)).to(_dev())


def _image(case, seed, scale=1.0):
    """A target image: colours in [0, scale)."""
    g = torch.Generator(device=_dev()).manual_seed(seed + 77)
    return torch.rand((case["views"], case["width"], case["height"], 3), generator=g, device=_dev()) * scale


def _slot_inputs(case, seed, dtype):
    """Camera-space surfels in front of the camera and the indices of the splats sampled at each
    pixel, drawn from the splats of the pixel's 16x16 cell; one pixel in 16 has a shorter list
    (-1 padded), as pixels at the rim of an object do."""
    g = torch.Generator(device=_dev()).manual_seed(seed)
    N, V, W, H, k = (case[x] for x in ("splats", "views", "width", "height", "samples"))
    f = 1.2 * max(W, H)
    rnd = lambda *s: torch.rand(s, generator=g, device=_dev(), dtype=torch.float64)  # noqa: E731
    cw, ch = (W + 15) // 16, (H + 15) // 16
    i = torch.arange(W, device=_dev()).view(W, 1, 1)
    j = torch.arange(H, device=_dev()).view(1, H, 1)
    pts, ids = [], []
    for _ in range(V):
        sx, sy = rnd(N) * W, rnd(N) * H
        cell = (sx.long() // 16) * ch + sy.long() // 16
        order = torch.argsort(cell, stable=True)
        sx, sy, cell = sx[order], sy[order], cell[order]
        z = -(2.0 + rnd(N))
        pts.append(torch.stack([-(sx - 0.5 * W) * z / f, (sy - 0.5 * H) * z / f, z], -1))
        first = torch.searchsorted(cell, torch.arange(cw * ch + 1, device=_dev()))
        c = (i // 16) * ch + j // 16
        lo, cnt = first[c], first[c + 1] - first[c]
        pick = lo + (rnd(W, H, k) * cnt).long()
        length = torch.where(rnd(W, H, 1) < 1.0 / 16, (rnd(W, H, 1) * (k + 1)).long(), torch.full_like(lo, k))
        slot = torch.arange(k, device=_dev()).view(1, 1, k)
        ids.append(torch.where((slot < length) & (cnt > 0), pick, torch.full_like(pick, -1)))
    P = torch.stack(pts)
    tilt = (rnd(V, N, 2) - 0.5) * 1.2
    nrm = torch.cat([tilt, -torch.ones(V, N, 1, device=_dev(), dtype=torch.float64)], -1)
    nrm = nrm / nrm.norm(dim=-1, keepdim=True)
    sd = (0.5 + 1.5 * rnd(V, N, 2)) * -P[..., 2:3] / f
    out = {"f": f, "W": W, "H": H, "P": P, "N": nrm, "S": sd, "A": rnd(V, N, 3), "idx":
           torch.stack(ids).to(torch.int32).contiguous()}
    w = rnd(*out["idx"].shape) ** 2
    out["w"] = torch.where(out["idx"] >= 0, w, torch.zeros_like(w))
    out["g"] = torch.randn(w.shape, generator=g, device=_dev(), dtype=torch.float64)
    out["gi"] = torch.randn(w.shape[:3] + (3,), generator=g, device=_dev(), dtype=torch.float64)
    return {q: x.to(dtype).contiguous() if isinstance(x, torch.Tensor) and x.is_floating_point() else x
            for q, x in out.items()}


def _network_inputs(case, seed):
    g = torch.Generator(device=_dev()).manual_seed(seed)
    n = lambda *s: torch.randn(s, generator=g, device=_dev())  # noqa: E731
    T, I = case["tiles"], case["image_tiles"]
    # He-initialised weights and small biases: W1, b1, W2, b2, W3, b3 in one block
    params = torch.cat([n(2048) * (2.0 / 32) ** 0.5, 0.1 * n(64), n(4096) * (2.0 / 64) ** 0.5, 0.1 * n(64),
                        n(64) * (2.0 / 64) ** 0.5, 0.1 * n(1)]).contiguous()
    return {"X": n(T, 32), "y": 0.5 * n(T), "w": n(T).abs() * 200.0, "F": n(I, 32), "c": n(I).abs() * 2000.0 + 1.0,
            "params": params}


def prepare(case, seed):
    kind = case["kind"]
    st = {"kind": kind, "case": case, "seed": seed}
    if kind == "frame":
        from splatting_amd.render import Options, Splatting
        sc = _scene(case, seed)
        r = Splatting(Options(numSamples=case["samples"], precision=0.01, shadingMode=case["mode"], device=_dev()),
                      None, sc.width, sc.height, sc.focal, 0.1, 50.0, 0.0)
        for m in (r.sphericalHarmonics, r.forwardHarmonics):
            g = torch.Generator().manual_seed(seed)
            with torch.no_grad():
                c = torch.rand(m.coefficients.shape, generator=g) * 0.2 - 0.1
                c[..., 0] = 0.5
                m.coefficients.copy_(c)
        r.to(_dev())
        r.keepIndicesOnHost = case["host_indices"]
        r.seed = seed
        rng = np.random.default_rng([seed, 5])
        lamp = rng.normal(size=(1, case["lamps"], 3))
        lamp[..., 2] = np.abs(lamp[..., 2]) + 0.5
        lamp /= np.linalg.norm(lamp, axis=-1, keepdims=True)
        st.update(r=r, M=_gpu(sc.view), leaves=[_gpu(x)[None].requires_grad_(True) for x in
                                                (sc.positions, sc.normals, sc.stddevs, sc.albedo)],
                  amb=_gpu(np.full((1, 3), 0.1)), lamp=_gpu(lamp),
                  ints=_gpu(rng.uniform(0.5, 1.5, size=(1, case["lamps"], 3))),
                  target=_image(case, seed)[..., :1 if case["mode"] == "silhouette" else 3].contiguous())
    elif kind == "render":
        sc = _scene(case, seed)
        st.update(M=_gpu(sc.view), f=sc.focal, target=_image(case, seed),
                  P=_gpu(sc.positions)[None].requires_grad_(True), N=_gpu(sc.normals)[None].requires_grad_(True),
                  S=_gpu(sc.stddevs)[None].requires_grad_(True), A=_gpu(sc.albedo)[None].requires_grad_(True))
    elif kind == "poisson":
        from splatting_amd.learned import PoissonFrame
        st["frame"] = PoissonFrame(_scene(case, seed), _dev(), rate=case["rate"], kcap=case["samples"],
                                   target=_image(case, seed, 300.0), proposal=case["proposal"])
    elif kind == "network":
        from splatting_amd.learned import RateNet
        st.update(_network_inputs(case, seed))
        st["net"] = RateNet(st["params"], torch.zeros(32, device=_dev()), torch.ones(32, device=_dev()))
    elif kind == "double":
        st.update(_slot_inputs(case, seed, torch.float64))
    else:
        st.update(_slot_inputs(case, seed, torch.float32))
        if kind == "neighbours":
            g = torch.Generator(device=_dev()).manual_seed(seed + 1)
            V, N, C = case["views"], case["splats"], case["channels"]
            st["values"] = torch.randn((V, N, C), generator=g, device=_dev())
            st["rows"] = torch.randn(st["idx"].shape + (C,), generator=g, device=_dev())
    return st


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(st):
    return _RUN[st["kind"]](st)


def _run_frame(st):
    leaves = st["leaves"]
    params = [*leaves, st["r"].sphericalHarmonics.coefficients, st["r"].forwardHarmonics.coefficients]
    for t in params:
        t.grad = None
    image, indices, depth = st["r"](None, None, *leaves, st["amb"], st["lamp"], st["ints"], transformMatrix=st["M"])
    ((image - st["target"]) ** 2).sum().backward()
    out = {"image": image.detach(), "indices": indices, "depth": depth.detach()}
    if st["case"]["host_indices"]:
        out["host"] = st["r"].indices
    for name, t in zip(("gP", "gN", "gS", "gA", "gSh", "gFh"), params):
        if t.grad is not None:
            out[name] = t.grad
    return out


def _run_render(st):
    from splatting_amd import poisson
    c = st["case"]
    leaves = [st[q] for q in "PNSA"]
    for t in leaves:
        t.grad = None
    V = c["views"]
    S = leaves[2] if V == 1 else leaves[2].expand(V, -1, -1)
    A = leaves[3] if V == 1 else leaves[3].expand(V, -1, -1)
    image = poisson.render(st["M"], leaves[0], leaves[1], S, A, c["width"], c["height"], st["f"],
                           numSamples=c["samples"], precision=0.01, rate=c["rate"], seed=st["seed"],
                           composite=c["composite"])
    ((image - st["target"]) ** 2).sum().backward()
    return [image.detach(), *(t.grad for t in leaves)]


def _run_poisson(st):
    loss, image, grads, g = st["frame"].step(st["seed"])
    return {"loss": loss, "image": image, "grads": list(grads), "indices": st["frame"].last_ids}


def _run_network(st):
    loss, grad = st["net"].loss_grad(st["X"], st["y"], st["w"])
    return [loss, grad, st["net"].tile_scale(st["F"], st["c"])]


def _run_compositing(st):
    from cudaExtensions import filtering
    a = (st["W"], st["H"], st["f"], st["P"], st["N"])
    return [filtering.forward(st["idx"], st["w"], *a), filtering.backward(st["idx"], st["w"], st["g"], *a)]


def _run_double(st):
    from cudaExtensions import filtering, interpolation, splatting
    W, H, f, idx, P, N, S, A = (st[q] for q in ("W", "H", "f", "idx", "P", "N", "S", "A"))
    w = splatting.forward(W, H, f, idx, P, N, S, 0.0)
    d = filtering.forward(idx, w, W, H, f, P, N)
    image = interpolation.forward(idx, d, A)
    gD, gA = interpolation.backward(st["gi"], idx, d, A)
    gW = filtering.backward(idx, w, gD, W, H, f, P, N, exact=True)
    return [w, d, image, gA, gW, *splatting.backward(W, H, f, gW, idx, P, N, S, 0.0)]


def _run_neighbours(st):
    from cudaExtensions import nearestsamples, pixelgather
    c = st["case"]
    return [pixelgather.scatter(st["idx"], st["values"]), pixelgather.gather(st["idx"], st["rows"], c["splats"]),
            nearestsamples.nearest(st["idx"], st["w"], st["P"][:1].contiguous(), c["nearest"])]


_RUN = {"frame": _run_frame, "render": _run_render, "poisson": _run_poisson, "network": _run_network,
        "compositing": _run_compositing, "double": _run_double, "neighbours": _run_neighbours}


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    if case["kind"] == "network":
        T, I = case["tiles"], case["image_tiles"]
        params = 6337
        return {"bytes": 4.0 * (34 * T + 34 * I + 2 * params), "flops": 6.0 * 6208 * T + 2.0 * 6208 * I}
    N, V, k = case["splats"], case["views"], case["samples"]
    P = case["width"] * case["height"] * V
    if case["kind"] == "frame":
        # splats and their gradients (11 values each way), the target and the image, the indices
        # and the compositing weights; per slot about 150 operations forward and backward
        return {"bytes": 88.0 * N + 24.0 * P + 8.0 * P * k * (1.5 if case["host_indices"] else 1.0),
                "flops": 150.0 * P * k + 400.0 * N * V}
    if case["kind"] in ("render", "poisson"):
        return {"bytes": 88.0 * N + 24.0 * P + (4.0 * P * k if case["kind"] == "poisson" else 0.0),
                "flops": 150.0 * P * case["rate"] + 400.0 * N * V}
    if case["kind"] == "compositing":
        # indices, weights and the upstream gradient in, two slot tensors out
        return {"bytes": 24.0 * N * V + 20.0 * P * k, "flops": (60.0 + 2.0 * math.log2(k)) * P * k}
    if case["kind"] == "double":
        return {"bytes": 176.0 * N * V + 48.0 * P + 28.0 * P * k, "flops": 150.0 * P * k + 600.0 * N * V}
    C, K = case["channels"], case["nearest"]
    return {"bytes": 8.0 * N * V * C + P * k * (8.0 + 8.0 * C) + 12.0 * N + 4.0 * N * K, "flops": 12.0 * P * k}


# ---------------------------------------------------------------------------
# Float64 values in plain torch
# ---------------------------------------------------------------------------
def _ray_depth(W, H, f, P, N, idx):
    """Distance along each pixel's ray to the plane of every sampled surfel (10000 behind the eye
    and for empty slots), in float64."""
    V = idx.shape[0]
    dev = idx.device
    bx = (W - 2.0 * torch.arange(W, device=dev, dtype=torch.float64)) / (2.0 * f)
    by = -(H - 2.0 * torch.arange(H, device=dev, dtype=torch.float64)) / (2.0 * f)
    d = torch.stack([bx[:, None].expand(W, H), by[None, :].expand(W, H), torch.ones(W, H, device=dev).double()], -1)
    d = -d / d.norm(dim=-1, keepdim=True)
    out = []
    for v in range(V):
        i = idx[v].long().clamp(min=0)
        plane = (P[v] * N[v]).sum(-1)
        den = (d[:, :, None, :] * N[v][i]).sum(-1)
        t = plane[i] / den
        out.append(torch.where((t > 0) & (idx[v] >= 0), t, torch.full_like(t, 10000.0)))
    return torch.stack(out)


def _composite(w, order):
    """w times the product of 1 - w over the slots in front."""
    ws = w.gather(-1, order)
    front = torch.cat([torch.ones_like(ws[..., :1]), torch.cumprod(1.0 - ws, -1)[..., :-1]], -1)
    return torch.zeros_like(w).scatter(-1, order, ws * front), front


def _exact_compositing(case, seed):
    s = _slot_inputs(case, seed, torch.float32)
    P, N, w, g = (s[q].double() for q in ("P", "N", "w", "g"))
    order = torch.argsort(_ray_depth(s["W"], s["H"], s["f"], P, N, s["idx"]), dim=-1, stable=True)
    out, front = _composite(w, order)
    # the reference's adjoint: own term unless |w| <= 1e-4, occlusion term unless |1 - w| <= 1e-4
    a, b = (g * w).gather(-1, order), 1.0 - w.gather(-1, order)
    behind = torch.zeros_like(a)
    acc = torch.zeros_like(a[..., 0])
    for q in range(a.shape[-1] - 1, -1, -1):
        behind[..., q] = acc
        acc = a[..., q] + b[..., q] * acc
    own = front * g.gather(-1, order) * (w.gather(-1, order).abs() > 1e-4)
    gs = own - front * behind * (b.abs() > 1e-4)
    return [out, torch.zeros_like(w).scatter(-1, order, gs)]


def _ewa(W, H, f, P, N, S, idx):
    """min(weight, 1) of every slot: the screen-space Gaussian of each surfel, normalised by the
    area it covers, at the pixel."""
    x, y, z = P.unbind(-1)
    sx, sy = -(x * f) / z + 0.5 * W, (y * f) / z + 0.5 * H
    one = torch.ones_like(sx)
    ray = lambda u, v: torch.stack([(W - 2.0 * u) / (2.0 * f), -(H - 2.0 * v) / (2.0 * f), one], -1)  # noqa: E731
    plane = (P * N).sum(-1, keepdim=True)
    hit = lambda r: r * plane / (r * N).sum(-1, keepdim=True) - P  # noqa: E731
    t0, t1 = hit(ray(sx + 1.0, sy)), hit(ray(sx, sy + 1.0))
    a00 = t0.norm(dim=-1)
    u0 = t0 / a00[..., None]
    u1 = torch.linalg.cross(u0, N)
    a01, a11 = (t1 * u0).sum(-1), (t1 * u1).sum(-1)
    det = a00 * a11
    j00, j01, j11 = a11 / det, -a01 / det, a00 / det
    s0, s1 = S[..., 0] ** 2, S[..., 1] ** 2
    v00, v01, v11 = j00 * j00 * s0 + j01 * j01 * s1, j01 * j11 * s1, j11 * j11 * s1
    dv = v00 * v11 - v01 * v01
    norm = 1.0 / (2.0 * math.pi * dv.sqrt() * det.abs())
    dev = P.device
    px = torch.arange(W, device=dev, dtype=torch.float64).view(W, 1, 1)
    py = torch.arange(H, device=dev, dtype=torch.float64).view(1, H, 1)
    out = []
    for v in range(idx.shape[0]):
        i = idx[v].long().clamp(min=0)
        dx, dy = px - sx[v][i], py - sy[v][i]
        e = (v11[v][i] * dx * dx - 2.0 * v01[v][i] * dx * dy + v00[v][i] * dy * dy) / dv[v][i]
        w = (norm[v][i] * torch.exp(-0.5 * e)).clamp(max=1.0)
        out.append(torch.where(idx[v] >= 0, w, torch.zeros_like(w)))
    return torch.stack(out)


def _exact_double(case, seed):
    s = _slot_inputs(case, seed, torch.float64)
    P, N, S, A = (s[q].requires_grad_(True) for q in ("P", "N", "S", "A"))
    w = _ewa(s["W"], s["H"], s["f"], P, N, S, s["idx"])
    with torch.no_grad():
        order = torch.argsort(_ray_depth(s["W"], s["H"], s["f"], P, N, s["idx"]), dim=-1, stable=True)
    w.retain_grad()
    d, _ = _composite(w, order)
    i = s["idx"].long().clamp(min=0)
    rows = torch.stack([A[v][i[v]] for v in range(i.shape[0])])
    image = (torch.where(s["idx"] >= 0, d, torch.zeros_like(d))[..., None] * rows).sum(-2)
    gP, gN, gS, gA, gW = torch.autograd.grad((image * s["gi"]).sum(), [P, N, S, A, w])
    return [w.detach(), d.detach(), image.detach(), gA, gW, gP, gN, gS]


def _exact_neighbours(case, seed):
    st = prepare(case, seed)
    idx, C = st["idx"], case["channels"]
    i = idx.long().clamp(min=0)
    on = (idx >= 0)[..., None]
    sc = torch.stack([st["values"][v][i[v]] for v in range(idx.shape[0])]).double() * on
    ga = torch.zeros((idx.shape[0], case["splats"], C), dtype=torch.float64, device=idx.device)
    for v in range(idx.shape[0]):
        ga[v].index_add_(0, i[v].reshape(-1), (st["rows"][v].double() * on[v]).reshape(-1, C))
    return [sc, ga, None]


def _exact_network(case, seed):
    """The network in float64 with its operands (features, weights, hidden activations and their
    gradients) rounded to bfloat16, the precision it is defined in; the tile multipliers follow
    from the forward pass."""
    s = _network_inputs(case, seed)
    p = s["params"].double()
    b = lambda x: x.float().bfloat16().double()  # noqa: E731
    W1, b1, W2, b2, W3, b3 = (x.view(*q) for x, q in zip(
        p.split([2048, 64, 4096, 64, 64, 1]), ((32, 64), (64,), (64, 64), (64,), (64,), (1,))))
    W1, W2, W3 = b(W1), b(W2), b(W3)

    def forward(x):
        h1 = b((b(x) @ W1 + b1).clamp(min=0.0))
        h2 = b((h1 @ W2 + b2).clamp(min=0.0))
        return h1, h2, h2 @ W3 + b3
    h1, h2, y = forward(s["X"])
    w, t = s["w"].double(), s["y"].double()
    dy = 2.0 * w * (y - t) / w.sum()
    d2 = torch.where(h2 > 0, dy[:, None] * W3, torch.zeros_like(h2))
    d1 = torch.where(h1 > 0, b(d2) @ W2.T, torch.zeros_like(h1))
    grad = torch.cat([(b(s["X"]).T @ b(d1)).reshape(-1), d1.sum(0), (h1.T @ b(d2)).reshape(-1), d2.sum(0),
                      h2.T @ dy, dy.sum().view(1)])
    c = s["c"].double()
    tot = c.sum()
    v = forward(s["F"])[2]
    v = torch.exp((v - (v * c).sum() / tot).clamp(-20.0, 20.0))
    for _ in range(3):
        v = (v * (tot / (v * c).sum())).clamp(0.75, 4.0)
    return [((w * (y - t) ** 2).sum() / w.sum()).view(1), grad, v]


def exact(case, seed):
    fn = {"network": _exact_network, "compositing": _exact_compositing, "double": _exact_double, "neighbours": _exact_neighbours}
    if case["kind"] not in fn:
        return None          # the sampled sets have no plain float64 value
    return fn[case["kind"]](case, seed)
