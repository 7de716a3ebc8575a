"""nearestsamples.nearest through the C ABI (FMMKdTreeSampling/nearestSamples.cpp:30-75,
nearestSamplesCuda.cu:290-564) on the regularizer's inputs -- indices of the
reference sampler (k = 16) and the compositing weights of the 4,096-splat
sphere at 128x128, two views -- equal to the oracle bit for bit (float32 and
float64), independent of the order the pixels are inserted in (a permuted
pixel order gives the same rows), and empty inputs."""
import numpy as np
import pytest
import torch

from helpers import scene_inputs
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def t(x, dev):
    return torch.from_numpy(np.ascontiguousarray(x)).to(dev)


def inputs(dev):
    from cudaExtensions import filtering, sampling, splatting
    sc, p, n, nb, sd = scene_inputs(0, sd_scale=2.0)
    W, H, f = sc.width, sc.height, sc.focal
    rot = np.array([[0.0, 0.0, 1.0], [0.0, 1.0, 0.0], [-1.0, 0.0, 0.0]], np.float32)
    p1 = ((p + np.float32([0, 0, 2.5])) @ rot.T - np.float32([0, 0, 2.5])).astype(np.float32)
    n1 = (n @ rot.T).astype(np.float32)
    P, Nn = t(np.stack([p, p1]), dev), t(np.stack([n, n1]), dev)
    NB = torch.where(Nn[..., 2:3] > 0, -Nn, Nn).contiguous()
    S = t(sd[None], dev)
    idx = sampling.sample(W, H, f, P, NB, None, S, 16, 0.0, 0.01, seed=2)
    w = filtering.forward(idx, splatting.forward(W, H, f, idx, P, Nn, S, 0.0), W, H, f, P, Nn)
    return sc, p, idx, w


@pytest.mark.parametrize("K", [1, 10])
def test_nearest_equals_oracle(dev, K):
    from cudaExtensions import nearestsamples
    sc, p, idx, w = inputs(dev)
    got = nearestsamples.nearest(idx, w, t(p[None], dev), K)
    ref = O.nearest_samples(idx.cpu().numpy(), w.cpu().numpy(), p[None], K)
    assert (ref >= 0).sum() > 1000
    assert np.array_equal(got.cpu().numpy(), ref)
    got64 = nearestsamples.nearest(idx, w.double(), t(p[None], dev).double(), K)
    assert np.array_equal(got64.cpu().numpy(), ref)


def test_nearest_independent_of_pixel_order(dev):
    from cudaExtensions import nearestsamples
    sc, p, idx, w = inputs(dev)
    perm = torch.randperm(idx.shape[1] * idx.shape[2], generator=torch.Generator().manual_seed(0)).to(dev)
    pi = idx.reshape(2, -1, 16)[:, perm].reshape(idx.shape).contiguous()
    pw = w.reshape(2, -1, 16)[:, perm].reshape(w.shape).contiguous()
    a = nearestsamples.nearest(idx, w, t(p[None], dev), 8)
    b = nearestsamples.nearest(pi, pw, t(p[None], dev), 8)
    assert torch.equal(a, b)


@pytest.mark.parametrize("k,K,N", [(1, 3, 9), (2, 2, 9), (5, 40, 30), (16, 10, 60), (17, 3, 200), (64, 12, 90),
                                   (65, 7, 2000), (130, 64, 150)])
def test_nearest_of_shared_rows(dev, k, K, N):
    """Few splats under many pixels: rows that many wavefronts enter at once, splats drawn
    twice at a pixel, equal points (ties by index), equal and NaN weights, empty slots, and
    slot counts around the lane groups.  The rows are whole numbers and equal the oracle's."""
    from cudaExtensions import nearestsamples
    rng = np.random.default_rng(100 * k + K)
    idx = rng.integers(-1, N, size=(2, 37, 11, k)).astype(np.int32)
    idx[0, 0, 0] = -1
    w = (rng.integers(0, 6, size=idx.shape) / 4).astype(np.float32)
    w[rng.uniform(size=idx.shape) < 0.05] = np.nan
    p = (rng.integers(0, 8, size=(1, N, 3)) / 8).astype(np.float32)
    # slots are compared in order by w > largest: a NaN in slot 0 stays, one elsewhere never
    # wins (the oracle's argmax orders NaN first wherever it stands)
    wo = np.where(np.isnan(w), np.float32(-1.0), w)
    wo[..., 0] = np.where(np.isnan(w[..., 0]), np.float32(9.0), w[..., 0])
    ref = O.nearest_samples(idx, wo, p, K)
    for dt in (torch.float32, torch.float64):
        got = nearestsamples.nearest(t(idx, dev), t(w, dev).to(dt), t(p, dev).to(dt), K)
        assert np.array_equal(got.cpu().numpy(), ref), dt


def test_nearest_empty(dev):
    from cudaExtensions import nearestsamples
    idx = torch.full((1, 4, 4, 5), -1, dtype=torch.int32, device=dev)
    out = nearestsamples.nearest(idx, torch.zeros(1, 4, 4, 5, device=dev), torch.zeros(1, 7, 3, device=dev), 3)
    assert out.shape == (1, 7, 3) and bool((out == -1).all())
    with pytest.raises(ValueError):
        nearestsamples.nearest(idx, torch.zeros(1, 4, 4, 5, device=dev), torch.zeros(2, 7, 3, device=dev), 3)
