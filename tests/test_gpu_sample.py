"""GPU parity of sampling.sample: sampled index sets must equal the oracle's
bit for bit given the same Philox seed (LBVH, Hermite FGT and the sequential
Poisson descent all reproduce the oracle's FP32 operation order)."""
import numpy as np
import pytest
import torch

from helpers import scene_inputs
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def t(x, dev):
    return torch.from_numpy(np.ascontiguousarray(x)).to(dev)


def run_gpu(dev, sc, p, nb, sd, k, precision=0.01, smoothing=0.0, seed=0):
    from cudaExtensions import sampling
    out = sampling.sample(sc.width, sc.height, sc.focal, t(p[None], dev), t(nb[None], dev), t(sd[None], dev),
                          t(sd[None], dev), k, smoothing, precision, seed=seed)
    sampling.check_errors()
    return out[0].cpu().numpy()


@pytest.mark.parametrize("cfg,sd_scale,k", [(2, 8.0, 8), (2, 8.0, 40), (0, 1.0, 40), (0, 4.0, 40), (0, 4.0, 16),
                                            (0, 4.0, 100)])
def test_sample_bit_exact(dev, cfg, sd_scale, k):
    sc, p, n, nb, sd = scene_inputs(cfg, sd_scale=sd_scale)
    got = run_gpu(dev, sc, p, nb, sd, k, seed=1234)
    ref = O.sample_view(sc.width, sc.height, sc.focal, p, nb, sd, k, 0.0, 0.01, seed=1234)
    assert (ref >= 0).sum() > 0
    mism = np.argwhere((got != ref).any(-1))
    assert mism.shape[0] == 0, "%d / %d pixels differ, first %s: gpu %s oracle %s" % (
        mism.shape[0], got.shape[0] * got.shape[1], mism[0], got[tuple(mism[0])], ref[tuple(mism[0])])


def test_sample_equal_keys(dev):
    """Equal keys, where the reference's insertion (a strict < that carries each
    displaced entry down the list, sequentialPoissonRadixTree.cuh:15-41) orders
    and drops entries unlike a sort by (key, draw number): 256 copies of a splat
    at every pixel centre of a 48x48 image, so the leaves there weigh exactly 1
    and their keys are the 24-bit uniforms themselves; k = 256.  The oracle's
    lists meet equal keys at about 30 pixels; the GPU's indices must equal it
    bit for bit everywhere."""
    from cudaExtensions import sampling
    W = H = 48
    f = 64.0
    ii, jj = np.meshgrid(np.arange(W), np.arange(H), indexing="ij")
    x = (ii - W / 2).ravel().astype(np.float32)
    y = (H / 2 - jj).ravel().astype(np.float32)
    P = np.repeat(np.stack([x, y, np.full_like(x, -f)], 1), 256, 0).astype(np.float32)
    N = np.tile(np.float32([0.0, 0.0, 1.0]), (P.shape[0], 1))
    S = np.full((P.shape[0], 2), 1.0, np.float32)
    ref = O.sample_view(W, H, f, P, N, S, 256, 0.0, 0.01, seed=4)
    assert O.tie_pixels() >= 10
    got = sampling.sample(W, H, f, t(P[None], dev), t(N[None], dev), t(S[None], dev), t(S[None], dev), 256, 0.0,
                          0.01, seed=4)
    sampling.check_errors()
    got = got[0].cpu().numpy()
    mism = np.argwhere((got != ref).any(-1))
    assert mism.shape[0] == 0, "%d / %d pixels differ, first %s" % (mism.shape[0], W * H, mism[0])


@pytest.mark.parametrize("precision,smoothing", [(0.001, 0.0), (0.05, 0.25)])
def test_sample_precision_smoothing(dev, precision, smoothing):
    sc, p, n, nb, sd = scene_inputs(0, sd_scale=2.0)
    got = run_gpu(dev, sc, p, nb, sd, 24, precision, smoothing, seed=5)
    ref = O.sample_view(sc.width, sc.height, sc.focal, p, nb, sd, 24, smoothing, precision, seed=5)
    assert np.array_equal(got, ref)


def test_sample_batched_views(dev):
    """Two views in one call: view b uses Philox view index b."""
    from cudaExtensions import sampling
    sc, p, n, nb, sd = scene_inputs(0, sd_scale=2.0)
    rot = np.array([[0.0, 0.0, 1.0], [0.0, 1.0, 0.0], [-1.0, 0.0, 0.0]], np.float32)
    p1 = (p + np.float32([0, 0, 2.5])) @ rot.T - np.float32([0, 0, 2.5])
    n1 = n @ rot.T
    nb1 = np.where(n1[:, 2:3] > 0, -n1, n1).astype(np.float32)
    P = np.stack([p, p1.astype(np.float32)])
    NB = np.stack([nb, nb1])
    out = sampling.sample(sc.width, sc.height, sc.focal, t(P, dev), t(NB, dev), t(sd[None], dev), t(sd[None], dev),
                          20, 0.0, 0.01, seed=9).cpu().numpy()
    ref = O.sample(sc.width, sc.height, sc.focal, P, NB, sd[None], 20, 0.0, 0.01, seed=9)
    assert np.array_equal(out, ref)


def test_sample_edge_cases(dev):
    from cudaExtensions import sampling
    sc, p, n, nb, sd = scene_inputs(2, sd_scale=8.0)
    # everything behind the camera: nothing survives the cull
    out = run_gpu(dev, sc, -p, nb, sd, 8)
    assert np.all(out == -1)
    # a single visible splat
    p1 = p[:1].copy()
    p1[0] = [0.0, 0.0, -2.0]
    out = run_gpu(dev, sc, p1, nb[:1], sd[:1], 8, seed=3)
    ref = O.sample_view(sc.width, sc.height, sc.focal, p1, nb[:1], sd[:1], 8, 0.0, 0.01, seed=3)
    assert np.array_equal(out, ref)
    # no splats at all
    z = np.zeros((1, 0, 3), np.float32)
    out = sampling.sample(8, 8, 9.6, t(z, dev), t(z, dev), None, t(np.zeros((1, 0, 2), np.float32), dev), 4, 0.0,
                          0.01, seed=0)
    assert out.shape == (1, 8, 8, 4) and bool((out == -1).all())


def test_sample_duplicate_positions(dev):
    """Many splats at identical screen positions (duplicate Morton keys)."""
    sc, p, n, nb, sd = scene_inputs(2, sd_scale=8.0)
    pd = np.repeat(p[:16], 16, axis=0)
    nd = np.repeat(nb[:16], 16, axis=0)
    sdd = np.repeat(sd[:16], 16, axis=0)
    got = run_gpu(dev, sc, pd, nd, sdd, 12, seed=77)
    ref = O.sample_view(sc.width, sc.height, sc.focal, pd, nd, sdd, 12, 0.0, 0.01, seed=77)
    assert np.array_equal(got, ref)


def test_sample_large_strip_and_properties(dev):
    """1M splats on 64 ellipsoids at 512x512, k = 40 (the sampler of the reference
    method at scale).  The oracle builds the whole tree and samples the 64 pixel
    rows 224 <= x < 288 (a 64 x 512 strip through the scene's centre, 32,768
    pixels): the GPU's indices there must equal it bit for bit.  The full image is
    checked by size-independent properties: indices in range, every sampled
    splat in front of the camera, determinism per seed, a new seed draws anew."""
    sc, p, n, nb, sd = scene_inputs(1)
    k = 40
    a = run_gpu(dev, sc, p, nb, sd, k, seed=21)
    ref, _ = O.sample_view_rows(sc.width, sc.height, sc.focal, p, nb, sd, k, 224, 288, 0.0, 0.01, seed=21)
    strip, rstrip = a[224:288], ref[224:288]
    assert (rstrip >= 0).sum() > 500_000
    mism = np.argwhere((strip != rstrip).any(-1))
    assert mism.shape[0] == 0, "%d / %d strip pixels differ, first %s: gpu %s oracle %s" % (
        mism.shape[0], 64 * sc.height, mism[0], strip[tuple(mism[0])], rstrip[tuple(mism[0])])
    b = run_gpu(dev, sc, p, nb, sd, k, seed=21)
    assert np.array_equal(a, b)
    v = a[a >= 0]
    assert v.size > 0 and v.max() < p.shape[0]
    assert np.all(p[np.unique(v), 2] <= 0)
    c = run_gpu(dev, sc, p, nb, sd, k, seed=22)
    assert not np.array_equal(a, c)


def test_sample_golden_fixture(dev):
    """Sampled indices equal the committed oracle fixture (256 splats, 64x64, k = 8)."""
    import os
    from cudaExtensions import sampling
    g = np.load(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "golden_cfg2.npz"))
    W, H, k, seed = (int(v) for v in g["dims"])
    out = sampling.sample(W, H, float(g["focal"]), t(g["pts"][None], dev), t(g["nrm"][None], dev), None,
                          t(g["sd"][None], dev), k, 0.0, float(g["precision"]), seed=seed)
    sampling.check_errors()
    assert np.array_equal(out[0].cpu().numpy(), g["idx"])


@pytest.mark.parametrize("k", [1, 5, 63, 64, 65, 128, 129, 256])
def test_sample_counts_at_row_edges(dev, k):
    """The drawing kernel holds a pixel's selected keys in 1, 2 or 4 rows of 64
    (k <= 64, 128, 256): the smallest count and both sides of every row edge, on
    an image whose sides are no multiples of the 8x8 tile, 4,096 splats dense
    enough that most pixels have more candidates than a row holds."""
    from cudaExtensions import sampling
    sc, p, n, nb, sd = scene_inputs(0, sd_scale=4.0)
    W, H, f = 45, 31, 1.2 * 45
    got = sampling.sample(W, H, f, t(p[None], dev), t(nb[None], dev), t(sd[None], dev), t(sd[None], dev), k, 0.0,
                          0.01, seed=k)
    sampling.check_errors()
    ref = O.sample_view(W, H, f, p, nb, sd, k, 0.0, 0.01, seed=k)
    assert (ref >= 0).mean() > 0.2
    assert np.array_equal(got[0].cpu().numpy(), ref)


@pytest.mark.parametrize("W,H,precision,k", [(24, 24, 1e-7, 40), (20, 13, 1e-6, 16), (16, 16, 1e-8, 3)])
def test_sample_walk_beyond_the_tile_lists(dev, W, H, precision, k):
    """A tile's walk keeps up to 448 walked and 448 evaluated nodes in LDS; tiles
    with more go to the depth-first form.  8,192 small splats over a few tiles at a
    small precision: 300 to 960 evaluated nodes per tile (so both forms run, on
    ragged tiles too), with a count of samples whose trie rows are the fewest."""
    from cudaExtensions import sampling
    sc, p, n, nb, sd = scene_inputs(0, 8192, sd_scale=4.0 if W == 16 else 2.0)
    f = 1.2 * W
    got = sampling.sample(W, H, f, t(p[None], dev), t(nb[None], dev), t(sd[None], dev), t(sd[None], dev), k, 0.0,
                          precision, seed=k)
    sampling.check_errors()
    ref = O.sample_view(W, H, f, p, nb, sd, k, 0.0, precision, seed=k)
    assert (ref >= 0).mean() > 0.5
    assert np.array_equal(got[0].cpu().numpy(), ref)


@pytest.mark.parametrize("perViewSd", [False, True])
def test_sample_views_in_groups(dev, monkeypatch, perViewSd):
    """Five views with different counts of visible splats (one sees none): in one group, in
    groups of two with a last one of one, one by one, and where the memory for a group is
    not there: the same indices bit for bit (the batch above is equal to the oracle's)."""
    from cudaExtensions import _lib, sampling
    sc, p, n, nb, sd = scene_inputs(2, sd_scale=8.0)
    W, H, f = 52, 36, sc.focal * 52 / sc.width
    shift = np.float32([[0, 0, 0], [1.5, 0, 0], [0, 0, 2000.0], [0, -2.0, 0], [0, 0, -3.0]])
    P = t(np.stack([p + s for s in shift]), dev)
    NB = t(np.stack([nb] * 5), dev)
    SD = t(np.stack([sd * (1 + 0.2 * b) for b in range(5)]) if perViewSd else sd[None], dev)
    run = lambda: sampling.sample(W, H, f, P, NB, None, SD, 16, 0.0, 0.01, seed=9).cpu().numpy()  # noqa: E731
    ref = run()
    for views in (1, 2, 5):
        monkeypatch.setattr(sampling, "_views_at_once", lambda *a, v=views: v)
        assert np.array_equal(run(), ref), views
    full = _lib.workspace

    def small(nbytes, device):
        if nbytes > _lib.lib().ude_sample_workspace_bytes(P.shape[1], W, H, 16):
            raise torch.OutOfMemoryError("not for several trees")
        return full(nbytes, device)
    monkeypatch.setattr(_lib, "workspace", small)
    assert np.array_equal(run(), ref)
    assert (ref[0] >= 0).any() and (ref[2] == -1).all()


@pytest.mark.parametrize("N,k", [(2, 12), (3, 40), (5, 5), (11, 12), (12, 12), (13, 12), (40, 40)])
def test_sample_fewer_splats_than_slots(dev, N, k):
    """At most k visible splats, spread so far that many pixels see one or none: the root is
    one subtree for every launch's descent, so a pixel draws each splat once per launch."""
    from cudaExtensions import sampling
    rng = np.random.default_rng(N)
    W, H, f = 33, 26, 40.0
    p = rng.uniform([-1.2, -1.0, -4.0], [1.2, 1.0, -2.0], size=(N, 3)).astype(np.float32)
    nb = np.tile(np.float32([0.0, 0.0, -1.0]), (N, 1))
    sd = rng.uniform(0.02, 0.2, size=(N, 2)).astype(np.float32)
    got = sampling.sample(W, H, f, t(p[None], dev), t(nb[None], dev), None, t(sd[None], dev), k, 0.0, 0.01, seed=3)
    assert np.array_equal(got[0].cpu().numpy(), O.sample_view(W, H, f, p, nb, sd, k, 0.0, 0.01, seed=3))


@pytest.mark.parametrize("case", [28, 70, 145, 216])
def test_sample_keys_near_the_largest(dev, case):
    """Random scenes in which a pixel has fewer than k draws of ordinary keys and more others
    than its wavefront keeps, with keys near the largest float: the search for the pixel's
    threshold ends there too."""
    from cudaExtensions import sampling
    rng = np.random.default_rng([1, case])
    N = int(np.exp(rng.uniform(0, np.log(20000))))
    bn, W, H = int(rng.integers(1, 4)), int(rng.integers(1, 90)), int(rng.integers(1, 90))
    k = int(rng.choice([1, 2, 3, 5, 8, 12, 16, 24, 40, 64, 65, 100, 128, 200, 256]))
    precision = float(10 ** rng.uniform(-3.5, -0.5))
    f = float(max(W, H)) * rng.uniform(0.6, 2.5)
    ext = rng.uniform(0.05, 1.5)
    p = rng.uniform([-ext, -ext, -4], [ext, ext, -1.5], size=(bn, N, 3)).astype(np.float32)
    if rng.uniform() < 0.3:
        p[..., :2] = np.round(p[..., :2] * 8) / 8
    if rng.uniform() < 0.3:
        p[rng.uniform(size=(bn, N)) < 0.3, 2] *= -1
    if rng.uniform() < 0.2:
        p[:, :N // 2] = p[:, :1]
    n = rng.normal(size=(bn, N, 3)).astype(np.float32)
    n[..., 2] = -np.abs(n[..., 2]) - 0.2
    n /= np.linalg.norm(n, axis=-1, keepdims=True)
    sd = (10 ** rng.uniform(-3.5, -0.3) * rng.uniform(0.5, 2, size=(1 if rng.uniform() < .5 else bn, N, 2))).astype(np.float32)
    smoothing = 0.0 if rng.uniform() < 0.6 else float(rng.uniform(0, 0.5))
    got = sampling.sample(W, H, f, t(p, dev), t(n, dev), None, t(sd, dev), k, smoothing, precision, seed=case)
    ref = O.sample(W, H, f, p, n, sd, k, smoothing, precision, seed=case)
    assert np.array_equal(got.cpu().numpy(), ref)


@pytest.mark.parametrize("N", [1, 2, 3, 64, 65, 129, 1023, 1025, 4095, 4096, 4097])
def test_sizes_around_one_workgroup(dev, N):
    """The tree's front in one workgroup up to 4096 splats: counts around its wavefronts, its
    rounds and its sorting network, with splats behind the camera among them, splats at the
    same place (equal keys keep their order) and out of the frame; sampler and Poisson-rate
    draws equal to the oracle bit for bit."""
    from cudaExtensions import sampling
    rng = np.random.default_rng(N)
    W, H, f = 33, 26, 40.0
    p = rng.uniform([-1.2, -1.0, -4.0], [1.2, 1.0, -2.0], size=(N, 3)).astype(np.float32)
    if N > 3:
        p[rng.uniform(size=N) < 0.1, 2] *= -1.0
        p[N // 2:N // 2 + N // 8] = p[0]
    nb = np.tile(np.float32([0.0, 0.0, -1.0]), (N, 1))
    sd = rng.uniform(0.02, 0.2, size=(N, 2)).astype(np.float32)
    got = sampling.sample(W, H, f, t(p[None], dev), t(nb[None], dev), None, t(sd[None], dev), 12, 0.0, 0.01, seed=3)
    assert np.array_equal(got[0].cpu().numpy(), O.sample_view(W, H, f, p, nb, sd, 12, 0.0, 0.01, seed=3))
    ids, ipi = sampling.samplePoisson(W, H, f, t(p[None], dev), t(nb[None], dev), None, t(sd[None], dev), 40, 0.0, 0.01,
                                      seed=3, rate=3.0)
    rid, ripi, _, over = O.poisson_view(W, H, f, p, nb, sd, 40, 3.0, 0.0, 0.01, seed=3)
    assert not over and np.array_equal(ids[0].cpu().numpy(), rid) and np.array_equal(ipi[0].cpu().numpy(), ripi)


@pytest.mark.parametrize("N", [4097, 5121, 65536, 131_071, 131_073, 262_144, 262_145, 300_000])
def test_sort_and_cull_sizes(dev, N):
    """Around the line between the sort's tiles, the counts that the cull's workgroups add up
    themselves, and partial tiles, with most splats out of the frame in one view and all in
    the other; a low precision keeps the trees shallow.  Density images equal to the
    oracle's, which any splat lost or out of order changes."""
    from cudaExtensions import sampling
    rng = np.random.default_rng(N)
    W, H, f = 24, 17, 30.0
    p = rng.uniform([-1.0, -0.7, -4.0], [1.0, 0.7, -3.0], size=(2, N, 3)).astype(np.float32)
    p[1, :, :2] *= 3.0
    p[1, N // 3:N // 2, 2] *= -1.0
    nb = np.tile(np.float32([0.0, 0.0, -1.0]), (2, N, 1))
    sd = np.full((1, N, 2), 0.05, np.float32)
    got = sampling.approximateFMMWeights(W, H, f, t(p, dev), t(nb, dev), None, t(sd, dev), 0.0, 0.05).cpu().numpy()
    for b in range(2):
        ref = O.fmm_weights_view(W, H, f, p[b], nb[b], sd[0], 0.0, 0.05)
        assert np.array_equal(got[b], ref), b


@pytest.mark.parametrize("k", [2, 9, 16, 23, 24, 25])
def test_sample_draws_in_halves(dev, k):
    """Two pixels per wavefront up to k = 24: on an image whose sides are no multiples of the
    tile, with more candidates than a half holds at most pixels and none at others."""
    from cudaExtensions import sampling
    sc, p, n, nb, sd = scene_inputs(0, sd_scale=4.0)
    W, H, f = 45, 31, 0.5 * 45
    got = sampling.sample(W, H, f, t(p[None], dev), t(nb[None], dev), t(sd[None], dev), t(sd[None], dev), k, 0.0,
                          0.01, seed=k)
    sampling.check_errors()
    ref = O.sample_view(W, H, f, p, nb, sd, k, 0.0, 0.01, seed=k)
    assert (ref >= 0).any() and (ref < 0).any()
    assert np.array_equal(got[0].cpu().numpy(), ref)


@pytest.mark.parametrize("seed,ties", [(1, 2), (2, 1), (0, 0)])
def test_sample_equal_keys_in_halves(dev, seed, ties):
    """Equal keys among a half's 24 slots: 24 copies of a splat at every pixel centre, whose
    keys are the 24-bit uniforms themselves."""
    from cudaExtensions import sampling
    W = H = 96
    f = 128.0
    ii, jj = np.meshgrid(np.arange(W), np.arange(H), indexing="ij")
    x = (ii - W / 2).ravel().astype(np.float32)
    y = (H / 2 - jj).ravel().astype(np.float32)
    P = np.repeat(np.stack([x, y, np.full_like(x, -f)], 1), 24, 0).astype(np.float32)
    N = np.tile(np.float32([0.0, 0.0, 1.0]), (P.shape[0], 1))
    S = np.full((P.shape[0], 2), 1.0, np.float32)
    ref = O.sample_view(W, H, f, P, N, S, 24, 0.0, 0.01, seed=seed)
    assert O.tie_pixels() == ties
    got = sampling.sample(W, H, f, t(P[None], dev), t(N[None], dev), None, t(S[None], dev), 24, 0.0, 0.01, seed=seed)
    assert np.array_equal(got[0].cpu().numpy(), ref)


def test_sample_most_tiles_beyond_the_lists(dev):
    """Two views of 10x9 tiles of which about 80 each have up to 950 walked and 870
    evaluated nodes, most of them more than a tile's lists hold."""
    from cudaExtensions import sampling
    sc, p, n, nb, sd = scene_inputs(0, 100_000, sd_scale=0.7)
    W, H, f, k = 80, 72, 1.2 * 80, 16
    P = np.stack([p, p * np.float32([-1.0, 1.0, 1.0])])
    NB = np.stack([nb, nb * np.float32([-1.0, 1.0, 1.0])])
    got = sampling.sample(W, H, f, t(P, dev), t(NB, dev), None, t(sd[None], dev), k, 0.0, 1e-7, seed=8)
    sampling.check_errors()
    for b in range(2):
        ref = O.sample_view(W, H, f, P[b], NB[b], sd, k, 0.0, 1e-7, seed=8, view=b)
        assert (ref >= 0).mean() > 0.5
        assert np.array_equal(got[b].cpu().numpy(), ref)


@pytest.mark.parametrize("k", [1, 9, 24, 25, 64, 128, 129])
@pytest.mark.parametrize("W,H", [(725, 724), (1025, 516)])
def test_sample_large_images(dev, W, H, k):
    """Images of more than 8192 tiles, on which a wavefront draws for 16 pixels: tiles without
    splats, with a few pixels that have some, and dense ones, partial tiles at both edges."""
    from cudaExtensions import sampling
    rng = np.random.default_rng(k)
    N, f = 700, 700.0
    p = rng.uniform([-1.0, -0.8, -3.0], [1.0, 0.8, -2.0], size=(N, 3)).astype(np.float32)
    p[: N // 2, :2] = p[: N // 2, :2] * 0.05 + 0.2
    p[0, :2] = (W / 2 - 1) / f * -p[0, 2], (H / 2 - 1) / f * p[0, 2]
    nb = np.tile(np.float32([0.0, 0.0, -1.0]), (N, 1))
    sd = rng.uniform(0.002, 0.02, size=(N, 2)).astype(np.float32)
    got = sampling.sample(W, H, f, t(p[None], dev), t(nb[None], dev), None, t(sd[None], dev), k, 0.0, 0.01, seed=k)
    sampling.check_errors()
    ref = O.sample_view(W, H, f, p, nb, sd, k, 0.0, 0.01, seed=k)
    assert 0.01 < (ref[..., 0] >= 0).mean() < 0.9
    assert np.array_equal(got[0].cpu().numpy(), ref)
