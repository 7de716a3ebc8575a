"""GPU parity of the per-slot operators against the FP64 oracle.

Tolerance (FP32 kernels vs FP64 oracle), per element:
|gpu - oracle| <= 1e-4 |oracle| + 64 * 2^-24 * mag (+ 1e-30), where mag is the
sum of |terms| the output accumulates (the oracle's abs-terms mode): the
relative bound holds wherever the terms do not cancel, and the floor is what a
float32 sum of the same terms can lose where they do.  Inputs are seeded sphere
scenes with std-devs scaled up so each splat covers several pixels, and slot
tensors mixing nearby splats, random splats and empty (-1) slots.
"""
import numpy as np
import pytest
import torch

from helpers import scene_inputs, near_slots, random_slots, assert_close, magnitude
from oracle import oracle as O

pytestmark = pytest.mark.gpu

RTOL = 1e-4


@pytest.fixture(scope="module")
def case():
    sc, p, n, nb, sd = scene_inputs(2, sd_scale=8.0)
    rng = np.random.default_rng(7)
    idx = near_slots(rng, p, sc.width, sc.height, sc.focal, 12)
    return sc, p, n, nb, sd, idx


def t(x, dev):
    return torch.from_numpy(np.ascontiguousarray(x)).to(dev)


def test_splat_forward(dev, case):
    from cudaExtensions import splatting
    sc, p, n, nb, sd, idx = case
    w = splatting.forward(sc.width, sc.height, sc.focal, t(idx, dev), t(p[None], dev), t(n[None], dev),
                          t(sd[None], dev), 0.0)
    ref = O.splat_forward(sc.width, sc.height, sc.focal, idx, p[None], n[None], sd[None])
    mag = magnitude(O.splat_forward, sc.width, sc.height, sc.focal, idx, p[None], n[None], sd[None])
    assert (ref > 0).mean() > 0.05
    assert_close(w.cpu().numpy(), ref, RTOL, "splat forward", mag=mag)
    assert np.all(w.cpu().numpy()[idx < 0] == 0)


@pytest.mark.parametrize("smoothing", [0.0, 0.5])
def test_splat_backward(dev, case, smoothing):
    from cudaExtensions import splatting
    sc, p, n, nb, sd, idx = case
    rng = np.random.default_rng(11)
    g = rng.normal(size=idx.shape).astype(np.float32)
    gp, gn, gs = splatting.backward(sc.width, sc.height, sc.focal, t(g, dev), t(idx, dev), t(p[None], dev),
                                    t(n[None], dev), t(sd[None], dev), smoothing)
    args = (sc.width, sc.height, sc.focal, g, idx, p[None], n[None], sd[None], smoothing)
    rp, rn, rs = O.splat_backward(*args)
    mp, mn, ms = magnitude(O.splat_backward, *args)
    assert_close(gp.cpu().numpy(), rp, RTOL, "grad points", mag=mp)
    assert_close(gn.cpu().numpy(), rn, RTOL, "grad normals", mag=mn)
    assert_close(gs.cpu().numpy(), rs, RTOL, "grad stddevs", mag=ms)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_splat_backward_normalized(dev, dtype):
    """splatting.backward(normalized=True) equals the raw backward followed by the
    reference's torch post-processing (conditionalNormalization, NaN -> 0) of the
    point and std-dev gradients; the normal gradient stays raw."""
    import torch
    from cudaExtensions import splatting
    from splatting_amd.utils import conditionalNormalization
    sc, p, n, nb, sd = scene_inputs(2, sd_scale=8.0)[:5]
    rng = np.random.default_rng(21)
    idx = near_slots(rng, p, sc.width, sc.height, sc.focal, 6)
    g = (rng.normal(size=idx.shape) * 30.0).astype(dtype)
    args = (sc.width, sc.height, sc.focal, t(g, dev), t(idx, dev), t(p[None].astype(dtype), dev),
            t(n[None].astype(dtype), dev), t(sd[None].astype(dtype), dev), 0.0)
    rp, rn, rs = splatting.backward(*args)
    gp, gn, gs = splatting.backward(*args, normalized=True)
    ep = torch.nan_to_num(conditionalNormalization(rp), nan=0.0, posinf=float("inf"), neginf=float("-inf"))
    es = torch.nan_to_num(conditionalNormalization(rs), nan=0.0, posinf=float("inf"), neginf=float("-inf"))
    # the two calls sum their slot moments with atomics in different orders
    tol = 1e-5 if dtype == np.float32 else 1e-12
    assert torch.allclose(gp, ep, rtol=tol, atol=tol * float(ep.abs().max()))
    assert torch.allclose(gs, es, rtol=tol, atol=tol * float(es.abs().max()))
    assert torch.allclose(gn, rn, rtol=tol, atol=tol * float(rn.abs().max()))
    norms = rp.norm(dim=-1)
    assert bool((norms > 1.5).any()) and bool(((norms > 0) & (norms < 0.5)).any())   # both branches taken
    # two views sharing one std-dev row: the post-processing would have to follow the sum over views
    p2, n2 = np.stack([p, p]).astype(dtype), np.stack([n, n]).astype(dtype)
    idx2, g2 = np.concatenate([idx, idx]), np.concatenate([g, g])
    with pytest.raises(ValueError):
        splatting.backward(sc.width, sc.height, sc.focal, t(g2, dev), t(idx2, dev), t(p2, dev), t(n2, dev),
                           t(sd[None].astype(dtype), dev), 0.0, normalized=True)


def test_splat_batched_views_and_broadcast_sd(dev):
    """bn = 2 views with shared (1, N, 2) std-devs: gradients of the std-devs sum over views."""
    from cudaExtensions import splatting
    sc, p, n, nb, sd = scene_inputs(2, sd_scale=8.0)[:5]
    rng = np.random.default_rng(3)
    p2 = np.stack([p, p + np.float32(0.01)])
    n2 = np.stack([n, n])
    idx = np.concatenate([near_slots(rng, p, sc.width, sc.height, sc.focal, 6)] * 2)
    g = rng.normal(size=idx.shape).astype(np.float32)
    w = splatting.forward(sc.width, sc.height, sc.focal, t(idx, dev), t(p2, dev), t(n2, dev), t(sd[None], dev), 0.0)
    ref = O.splat_forward(sc.width, sc.height, sc.focal, idx, p2, n2, sd[None])
    mag = magnitude(O.splat_forward, sc.width, sc.height, sc.focal, idx, p2, n2, sd[None])
    assert_close(w.cpu().numpy(), ref, RTOL, "batched forward", mag=mag)
    gp, gn, gs = splatting.backward(sc.width, sc.height, sc.focal, t(g, dev), t(idx, dev), t(p2, dev), t(n2, dev),
                                    t(sd[None], dev), 0.0)
    rp, rn, rs = O.splat_backward(sc.width, sc.height, sc.focal, g, idx, p2, n2, sd[None])
    mp, mn, ms = magnitude(O.splat_backward, sc.width, sc.height, sc.focal, g, idx, p2, n2, sd[None])
    assert_close(gp.cpu().numpy(), rp, RTOL, "batched grad points", mag=mp)
    assert_close(gn.cpu().numpy(), rn, RTOL, "batched grad normals", mag=mn)
    assert_close(gs.cpu().numpy(), rs, RTOL, "batched grad stddevs", mag=ms)


def test_covariance(dev, case):
    from cudaExtensions import sampling
    sc, p, n, nb, sd, idx = case
    c = sampling.covariance(sc.width, sc.height, sc.focal, t(p[None], dev), t(n[None], dev), t(sd[None], dev), 0.1)
    ref = O.covariance(sc.width, sc.height, sc.focal, p[None], n[None], sd[None], 0.1)
    assert_close(c.cpu().numpy(), ref, RTOL, "covariance")


@pytest.mark.parametrize("k", [12, 40, 64, 100])
def test_filter_forward_backward(dev, k):
    from cudaExtensions import filtering
    sc, p, n, nb, sd = scene_inputs(2, sd_scale=8.0)[:5]
    rng = np.random.default_rng(5 + k)
    idx = random_slots(rng, 1, sc.width, sc.height, k, p.shape[0])
    w = rng.uniform(0.0, 1.0, size=idx.shape).astype(np.float32)
    w[idx < 0] = 0.0
    g = rng.normal(size=idx.shape).astype(np.float32)
    out = filtering.forward(t(idx, dev), t(w, dev), sc.width, sc.height, sc.focal, t(p[None], dev), t(n[None], dev))
    ref = O.filter_forward(idx, w, sc.width, sc.height, sc.focal, p[None], n[None])
    assert_close(out.cpu().numpy(), ref, RTOL, "filter forward")
    gw = filtering.backward(t(idx, dev), t(w, dev), t(g, dev), sc.width, sc.height, sc.focal, t(p[None], dev),
                            t(n[None], dev))
    rg = O.filter_backward(idx, w, g, sc.width, sc.height, sc.focal, p[None], n[None])
    mg = magnitude(O.filter_backward, idx, w, g, sc.width, sc.height, sc.focal, p[None], n[None])
    assert_close(gw.cpu().numpy(), rg, RTOL, "filter backward", mag=mg)
    # the exact adjoint, on weights that put slots inside the reference's gates
    # (|w| <= 1e-4, |1 - w| <= 1e-4) where the two differ
    w2 = w.copy()
    gated = rng.uniform(size=idx.shape)
    w2[gated < 0.1] = 5e-5
    w2[gated > 0.9] = np.float32(1.0 - 5e-5)
    w2[idx < 0] = 0.0
    ge = filtering.backward(t(idx, dev), t(w2, dev), t(g, dev), sc.width, sc.height, sc.focal, t(p[None], dev),
                            t(n[None], dev), exact=True)
    re = O.filter_backward(idx, w2, g, sc.width, sc.height, sc.focal, p[None], n[None], exact=True)
    me = magnitude(O.filter_backward, idx, w2, g, sc.width, sc.height, sc.focal, p[None], n[None], exact=True)
    assert_close(ge.cpu().numpy(), re, RTOL, "exact filter backward", mag=me)
    assert np.abs(re - O.filter_backward(idx, w2, g, sc.width, sc.height, sc.focal, p[None], n[None])).max() > 1e-2


@pytest.mark.parametrize("k", [40, 64])
def test_filter_equal_depths(dev, k):
    """Slots drawn from three splats, so most pixels hold runs of equal depths with
    different weights: the compositing order among equal depths is the slot order
    (the reference's stable insertion sort), forward and backward."""
    from cudaExtensions import filtering
    sc, p, n, nb, sd = scene_inputs(2, sd_scale=8.0)[:5]
    rng = np.random.default_rng(77 + k)
    idx = random_slots(rng, 1, sc.width, sc.height, k, 3, p_empty=0.3)
    w = rng.uniform(0.0, 1.0, size=idx.shape).astype(np.float32)
    w[idx < 0] = rng.uniform(0.0, 1.0, size=int((idx < 0).sum())).astype(np.float32)   # ties at depth 10000 too
    g = rng.normal(size=idx.shape).astype(np.float32)
    out = filtering.forward(t(idx, dev), t(w, dev), sc.width, sc.height, sc.focal, t(p[None], dev), t(n[None], dev))
    ref = O.filter_forward(idx, w, sc.width, sc.height, sc.focal, p[None], n[None])
    assert_close(out.cpu().numpy(), ref, RTOL, "filter forward, equal depths")
    gw = filtering.backward(t(idx, dev), t(w, dev), t(g, dev), sc.width, sc.height, sc.focal, t(p[None], dev),
                            t(n[None], dev))
    rg = O.filter_backward(idx, w, g, sc.width, sc.height, sc.focal, p[None], n[None])
    mg = magnitude(O.filter_backward, idx, w, g, sc.width, sc.height, sc.focal, p[None], n[None])
    assert_close(gw.cpu().numpy(), rg, RTOL, "filter backward, equal depths", mag=mg)
    # a wrong order among equal depths changes the forward output by far more than the tolerance
    wrong = O.filter_forward(idx[..., ::-1].copy(), w[..., ::-1].copy(), sc.width, sc.height, sc.focal, p[None],
                             n[None])[..., ::-1]
    assert np.abs(wrong - ref).max() > 1e-2


@pytest.mark.parametrize("W,H,bn", [(5, 3, 2), (256, 86, 3), (181, 121, 3), (219, 200, 3)])
@pytest.mark.parametrize("k", [1, 16, 31, 32, 33, 64])
def test_filter_pixels_per_wave(dev, k, W, H, bn):
    """One pixel per wavefront, several, and two at a time in halves, around their slot
    counts: partial groups, groups that run into the next view, points per view, many equal
    depths.  Bounds as for the wider kernels."""
    from cudaExtensions import filtering
    sc, p, n, nb, sd = scene_inputs(2, sd_scale=8.0)[:5]
    rng = np.random.default_rng(277 + k)
    P = np.stack([p * np.float32(1 + 0.1 * b) for b in range(bn)])
    Nn = np.stack([n] * bn)
    idx = rng.integers(0, 40, size=(bn, W, H, k)).astype(np.int32)
    idx[rng.uniform(size=idx.shape) < 0.3] = -1
    w = rng.uniform(0.0, 1.0, size=idx.shape).astype(np.float32)
    g = rng.normal(size=idx.shape).astype(np.float32)
    a = (W, H, sc.focal)
    out = filtering.forward(t(idx, dev), t(w, dev), *a, t(P, dev), t(Nn, dev))
    assert_close(out.cpu().numpy(), O.filter_forward(idx, w, *a, P, Nn), max(RTOL, 2 * k * 2.0 ** -24), "filter forward")
    gw = filtering.backward(t(idx, dev), t(w, dev), t(g, dev), *a, t(P, dev), t(Nn, dev))
    rg = O.filter_backward(idx, w, g, *a, P, Nn)
    mg = magnitude(O.filter_backward, idx, w, g, *a, P, Nn)
    assert_close(gw.cpu().numpy(), rg, RTOL, "filter backward", mag=mg, ops=max(64, 4 * k))


@pytest.mark.parametrize("splats", [3, 400])
@pytest.mark.parametrize("k", [65, 127, 128, 129, 250, 256, 257, 319, 1024])
def test_filter_wide(dev, k, splats):
    """More than 64 slots: around the lane-row, wavefront and workgroup sizes, with many
    equal depths (three splats) and few (400); both batch entries, every slot filled in some
    pixels and none in others.  A product of k factors 1 - w carries up to 2 k float32
    roundings (2^-24 each), a suffix sum over it twice as many."""
    from cudaExtensions import filtering
    sc, p, n, nb, sd = scene_inputs(2, sd_scale=8.0)[:5]
    W, H = 5, 3                                         # 15 pixels: a partial group of wavefronts
    rng = np.random.default_rng(177 + k)
    idx = rng.integers(0, min(splats, p.shape[0]), size=(2, W, H, k)).astype(np.int32)
    idx[rng.uniform(size=idx.shape) < 0.3] = -1
    idx[0, 0, 0] = 1
    idx[1, 2, 1] = -1
    w = (rng.uniform(0.0, 1.0, size=idx.shape) * min(1.0, 24.0 / k)).astype(np.float32)
    g = rng.normal(size=idx.shape).astype(np.float32)
    a = (W, H, sc.focal)
    dv = (t(idx, dev), t(w, dev))
    out = filtering.forward(*dv, *a, t(p[None], dev), t(n[None], dev))
    rtol = max(RTOL, 2 * k * 2.0 ** -24)
    assert_close(out.cpu().numpy(), O.filter_forward(idx, w, *a, p[None], n[None]), rtol, "wide filter forward")
    for exact in (False, True):
        gw = filtering.backward(*dv, t(g, dev), *a, t(p[None], dev), t(n[None], dev), exact=exact)
        rg = O.filter_backward(idx, w, g, *a, p[None], n[None], exact=exact)
        mg = magnitude(O.filter_backward, idx, w, g, *a, p[None], n[None], exact=exact)
        assert_close(gw.cpu().numpy(), rg, RTOL, "wide filter backward", mag=mg, ops=max(64, 4 * k))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("bn,N", [(2, 1), (2, 4095), (3, 4097), (65, 1030), (130, 64)])
def test_transform_backward_shared_vectors(dev, bn, N, dtype):
    """One vector set under all views, around the workgroup's points and its views in LDS;
    each sum has N or bn terms, so its bound takes that many roundoffs."""
    from cudaExtensions import transform
    rng = np.random.default_rng(bn + N)
    M, v, g = rng.normal(size=(bn, 4, 4)), rng.normal(size=(1, N, 3)), rng.normal(size=(bn, N, 3))
    if dtype == torch.float32:
        M, v, g = (x.astype(np.float32) for x in (M, v, g))
    eps = float(np.finfo(M.dtype).eps) / 2
    for affine in (True, False):
        bw = transform.affineBackward if affine else transform.linearBackward
        got = bw(t(g, dev), t(M, dev), t(v, dev))
        ref = O.transform_backward(affine, g, M, v)
        mag = magnitude(O.transform_backward, affine, g, M, v)
        for a, r, m in zip(got, ref, mag):
            assert_close(a.cpu().numpy(), r, 8 * eps, "shared transform backward", mag=m, ops=max(64, bn), eps=eps)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("bn,N", [(2, 99_999), (2, 100_000), (3, 102_401), (65, 100_003), (200, 300)])
def test_transform_backward_of_many_and_few_points(dev, bn, N, dtype):
    """Both sides of the point count from which the views share their points' registers,
    partial workgroups and more views than its sums hold; each sum has N or bn terms."""
    from cudaExtensions import transform
    rng = np.random.default_rng(bn + N)
    M, v, g = rng.normal(size=(bn, 4, 4)), rng.normal(size=(1, N, 3)), rng.normal(size=(bn, N, 3))
    if dtype == torch.float32:
        M, v, g = (x.astype(np.float32) for x in (M, v, g))
    eps = float(np.finfo(M.dtype).eps) / 2
    got = transform.affineBackward(t(g, dev), t(M, dev), t(v, dev))
    ref = O.transform_backward(True, g, M, v)
    mag = magnitude(O.transform_backward, True, g, M, v)
    for a, r, m in zip(got, ref, mag):
        assert_close(a.cpu().numpy(), r, 8 * eps, "transform backward", mag=m, ops=max(64, bn), eps=eps)


@pytest.mark.parametrize("affine", [True, False])
@pytest.mark.parametrize("bn,vb", [(1, 1), (3, 1), (3, 3)])
def test_transform(dev, affine, bn, vb):
    """Forward and adjoint against the oracle; the vector gradient is written
    without a prior fill when every element gets one value (stale NaN memory is
    handed to the allocation first to show it)."""
    from cudaExtensions import transform
    rng = np.random.default_rng(1)
    N = 5000
    M = rng.normal(size=(bn, 4, 4)).astype(np.float32)
    v = rng.normal(size=(vb, N, 3)).astype(np.float32)
    g = rng.normal(size=(bn, N, 3)).astype(np.float32)
    fw = transform.affineForward if affine else transform.linearForward
    bw = transform.affineBackward if affine else transform.linearBackward
    out = fw(t(M, dev), t(v, dev))
    assert_close(out.cpu().numpy(), O.transform_forward(affine, M, v), RTOL, "transform forward",
                 mag=magnitude(O.transform_forward, affine, M, v))
    if not affine:      # the fused camera-facing copy equals the renderer's torch.where, bit for bit
        same, facing = transform.linearForwardFacing(t(M, dev), t(v, dev))
        assert torch.equal(same, out)
        assert torch.equal(facing, torch.where(out[..., 2:3] > 0, -out, out))
    gd, Md, vd = t(g, dev), t(M, dev), t(v, dev)
    junk = torch.full((vb, N, 3), float("nan"), device=dev)
    del junk
    gM, gV = bw(gd, Md, vd)
    rM, rV = O.transform_backward(affine, g, M, v)
    mM, mV = magnitude(O.transform_backward, affine, g, M, v)
    assert_close(gM.cpu().numpy(), rM, RTOL, "transform grad M", mag=mM)
    assert_close(gV.cpu().numpy(), rV, RTOL, "transform grad v", mag=mV)


@pytest.mark.parametrize("C,ab", [(3, 1), (16, 2)])
def test_interpolation(dev, C, ab):
    from cudaExtensions import interpolation
    rng = np.random.default_rng(C)
    bn, W, H, k, N = 2, 24, 20, 9, 300
    idx = random_slots(rng, bn, W, H, k, N)
    w = rng.uniform(size=idx.shape).astype(np.float32)
    a = rng.normal(size=(ab, N, C)).astype(np.float32)
    g = rng.normal(size=(bn, W, H, C)).astype(np.float32)
    out = interpolation.forward(t(idx, dev), t(w, dev), t(a, dev))
    assert_close(out.cpu().numpy(), O.interp_forward(idx, w, a), RTOL, "interp forward",
                 mag=magnitude(O.interp_forward, idx, w, a))
    gW, gA = interpolation.backward(t(g, dev), t(idx, dev), t(w, dev), t(a, dev))
    rW, rA = O.interp_backward(g, idx, w, a)
    mW, mA = magnitude(O.interp_backward, g, idx, w, a)
    assert_close(gW.cpu().numpy(), rW, RTOL, "interp grad w", mag=mW)
    assert_close(gA.cpu().numpy(), rA, RTOL, "interp grad attr", mag=mA)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("W,H,k,N,ab", [(8, 8, 1, 2, 1), (9, 7, 40, 30, 2), (3, 50, 130, 5000, 1), (300, 190, 9, 100_000, 2),
                                        (257, 241, 16, 700, 1)])
def test_interpolation_tiles(dev, W, H, k, N, ab, dtype):
    """Three channels around the tiles of both sizes: partial tiles, slots that share their
    rows and slots that share none, more rows in a tile than its table holds, zero weights.
    An attribute row sums as many terms as slots name it."""
    from cudaExtensions import interpolation
    rng = np.random.default_rng(W + k)
    idx = random_slots(rng, 2, W, H, k, N)
    w = rng.uniform(size=idx.shape).astype(dtype)
    w[rng.uniform(size=idx.shape) < 0.1] = 0.0
    a = rng.normal(size=(ab, N, 3)).astype(dtype)
    g = rng.normal(size=(2, W, H, 3)).astype(dtype)
    eps = float(np.finfo(dtype).eps) / 2
    most = int(np.bincount(idx[idx >= 0].ravel()).max())
    out = interpolation.forward(t(idx, dev), t(w, dev), t(a, dev))
    assert_close(out.cpu().numpy(), O.interp_forward(idx, w, a), 8 * eps, "interp forward",
                 mag=magnitude(O.interp_forward, idx, w, a), ops=max(64, k), eps=eps)
    gW, gA = interpolation.backward(t(g, dev), t(idx, dev), t(w, dev), t(a, dev))
    rW, rA = O.interp_backward(g, idx, w, a)
    mW, mA = magnitude(O.interp_backward, g, idx, w, a)
    assert_close(gW.cpu().numpy(), rW, 8 * eps, "interp grad w", mag=mW, eps=eps)
    assert_close(gA.cpu().numpy(), rA, 8 * eps, "interp grad attr", mag=mA, ops=max(64, most), eps=eps)


@pytest.mark.parametrize("k", [1, 2, 7, 8, 9])
def test_interpolation_double_few_slots(dev, k):
    """Both sides of the slot count from which a pixel has several lanes; sums of k terms."""
    from cudaExtensions import interpolation
    rng = np.random.default_rng(k)
    idx = random_slots(rng, 2, 37, 21, k, 90)
    w, a = rng.uniform(size=idx.shape), rng.normal(size=(2, 90, 3))
    eps = float(np.finfo(np.float64).eps) / 2
    out = interpolation.forward(t(idx, dev), t(w, dev), t(a, dev))
    assert_close(out.cpu().numpy(), O.interp_forward(idx, w, a), 8 * eps, "interp forward",
                 mag=magnitude(O.interp_forward, idx, w, a), eps=eps)


@pytest.mark.parametrize("cb", [1, 2])
def test_sh_shading(dev, cb):
    from cudaExtensions import shading
    rng = np.random.default_rng(20 + cb)
    bn, W, H = 2, 16, 20
    coef = rng.normal(size=(cb, 3, 9)).astype(np.float32)
    nrm = rng.normal(size=(bn, W, H, 3)).astype(np.float32)
    nrm[0, 0, 0] = 0.0
    diff = rng.uniform(size=(bn, W, H, 3)).astype(np.float32)
    g = rng.normal(size=(bn, W, H, 3)).astype(np.float32)
    out = shading.forwardSh(t(coef, dev), t(nrm, dev), t(diff, dev))
    assert_close(out.cpu().numpy(), O.sh_forward(coef, nrm, diff), RTOL, "sh forward",
                 mag=magnitude(O.sh_forward, coef, nrm, diff))
    gc, gn, gd = shading.backwardSh(t(g, dev), t(coef, dev), t(nrm, dev), t(diff, dev))
    rc, rn, rd = O.sh_backward(g, coef, nrm, diff)
    mc, mn, md = magnitude(O.sh_backward, g, coef, nrm, diff)
    assert_close(gc.cpu().numpy(), rc, RTOL, "sh grad coef", mag=mc)
    assert_close(gn.cpu().numpy(), rn, RTOL, "sh grad normals", mag=mn)
    assert_close(gd.cpu().numpy(), rd, RTOL, "sh grad diffuse", mag=md)


@pytest.mark.parametrize("ib", [1, 2])
def test_lambert_shading(dev, ib):
    from cudaExtensions import shading
    rng = np.random.default_rng(30 + ib)
    bn, W, H, L = 2, 16, 12, 3
    dirs = rng.normal(size=(bn, L, 3)).astype(np.float32)
    ints = rng.uniform(size=(ib, L, 3)).astype(np.float32)
    nrm = rng.normal(size=(bn, W, H, 3)).astype(np.float32)
    diff = rng.uniform(size=(bn, W, H, 3)).astype(np.float32)
    g = rng.normal(size=(bn, W, H, 3)).astype(np.float32)
    out = shading.forward(t(dirs, dev), t(ints, dev), t(nrm, dev), t(diff, dev))
    assert_close(out.cpu().numpy(), O.lambert_forward(dirs, ints, nrm, diff), RTOL, "lambert forward",
                 mag=magnitude(O.lambert_forward, dirs, ints, nrm, diff))
    gdir, gint, gn, gd = shading.backward(t(g, dev), t(dirs, dev), t(ints, dev), t(nrm, dev), t(diff, dev))
    r = O.lambert_backward(g, dirs, ints, nrm, diff)
    m = magnitude(O.lambert_backward, g, dirs, ints, nrm, diff)
    for a, b, mm, nm in zip((gdir, gint, gn, gd), r, m, ("dir", "int", "normal", "diffuse")):
        assert_close(a.cpu().numpy(), b, RTOL, "lambert grad " + nm, mag=mm)


@pytest.mark.parametrize("W,H,L", [(1, 1, 1), (7, 37, 4), (300, 230, 5), (33, 16, 9)])
def test_shading_backward_sums(dev, W, H, L):
    """The light gradients are register sums of a grid-stride loop over a view's
    pixels, lamps four at a time: one pixel, less than a workgroup, more pixels
    than the grid has threads, and lamp counts at and past a multiple of four."""
    from cudaExtensions import shading
    rng = np.random.default_rng(W + L)
    bn = 2
    draw = lambda *s: rng.normal(size=s).astype(np.float32)
    nrm, g, diff = draw(bn, W, H, 3), draw(bn, W, H, 3), rng.uniform(size=(bn, W, H, 3)).astype(np.float32)
    dirs, ints, coef = draw(bn, L, 3), rng.uniform(size=(1, L, 3)).astype(np.float32), draw(bn, 3, 9)
    for dt, rtol, eps, ops in ((np.float32, RTOL, 2.0 ** -24, 64), (np.float64, 1e-10, 2.0 ** -53, 1024)):
        x = [t(a.astype(dt), dev) for a in (g, dirs, ints, nrm, diff, coef)]
        got = [*shading.backward(*x[:5]), *shading.backwardSh(x[0], x[5], x[3], x[4])]
        ref = [*O.lambert_backward(g, dirs, ints, nrm, diff), *O.sh_backward(g, coef, nrm, diff)]
        mag = [*magnitude(O.lambert_backward, g, dirs, ints, nrm, diff), *magnitude(O.sh_backward, g, coef, nrm, diff)]
        for q, (a, b, m) in enumerate(zip(got, ref, mag)):
            assert_close(a.cpu().numpy(), b, rtol, "shading grad %d %s" % (q, dt.__name__), mag=m, eps=eps, ops=ops)
