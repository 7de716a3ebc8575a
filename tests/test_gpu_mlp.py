"""GPU rate network (bfloat16 matrix cores, FP32 accumulation) against the FP64
oracle with the same bfloat16 rounding points: forward, loss gradient, Adam,
and a training run that fits a known network."""
import numpy as np
import pytest
import torch

from oracle import mlp as M

pytestmark = pytest.mark.gpu


def t(x, dev):
    return torch.from_numpy(np.ascontiguousarray(x, np.float32)).to(dev)


def rel(a, b):
    return np.abs(np.asarray(a, np.float64) - b).max() / max(np.abs(b).max(), 1e-30)


@pytest.mark.parametrize("T", [1, 17, 1024, 5000])
def test_mlp_forward_and_grad_match_oracle(dev, T):
    from splatting_amd.learned import RateNet
    rng = np.random.default_rng(T)
    X = rng.normal(size=(T, M.N_IN)).astype(np.float32)
    P = (rng.normal(size=M.N_PARAMS) * 0.2).astype(np.float32)
    tgt = rng.normal(size=T).astype(np.float32)
    w = rng.uniform(0.5, 2.0, size=T).astype(np.float32)
    net = RateNet(t(P, dev), t(np.zeros(M.N_IN), dev), t(np.ones(M.N_IN), dev))
    y = net.forward(t(X, dev)).cpu().numpy()
    yr, _ = M.forward(X, P, quant=True)
    # FP32 accumulation vs FP64, then occasional one-ulp bfloat16 flips of hidden units
    assert rel(y, yr) < 5e-3
    loss, g = net.loss_grad(t(X, dev), t(tgt, dev), t(w, dev))
    lr, gr = M.loss_grad(X, P, tgt, w, quant=True)
    assert abs(float(loss.item()) - lr) <= 1e-2 * lr
    g = g.cpu().numpy()
    for a, b in ((M.OFF_W1, M.OFF_B1), (M.OFF_B1, M.OFF_W2), (M.OFF_W2, M.OFF_B2), (M.OFF_B2, M.OFF_W3),
                 (M.OFF_W3, M.OFF_B3), (M.OFF_B3, M.N_PARAMS)):
        assert rel(g[a:b], gr[a:b]) < 2e-2, (a, b, rel(g[a:b], gr[a:b]))


def test_adam_step_matches_oracle(dev):
    from cudaExtensions import _lib
    rng = np.random.default_rng(3)
    n = 6337
    P, g, m, v = (rng.normal(size=n).astype(np.float32) for _ in range(4))
    v = np.abs(v)
    Pt, gt, mt, vt = t(P, dev), t(g, dev), t(m, dev), t(v, dev)
    rc = _lib.lib().ude_adam_step(n, _lib.ptr(Pt), _lib.ptr(gt), _lib.ptr(mt), _lib.ptr(vt), 1e-3, 0.9, 0.999, 1e-8,
                                  5, _lib.stream(dev))
    assert rc == 0
    Pr, mr, vr = M.adam_step(P.astype(np.float64), g, m, v, 1e-3, 0.9, 0.999, 1e-8, 5)
    assert rel(Pt.cpu().numpy(), Pr) < 1e-6 and rel(mt.cpu().numpy(), mr) < 1e-6 and rel(vt.cpu().numpy(), vr) < 1e-6


def test_training_fits_a_known_network(dev):
    from splatting_amd.learned import RateNet
    rng = np.random.default_rng(4)
    T = 4096
    X = rng.normal(size=(T, M.N_IN)).astype(np.float32)
    true = (rng.normal(size=M.N_PARAMS) * 0.15).astype(np.float32)
    y, _ = M.forward(X, true, quant=False)
    net = RateNet.init(dev, seed=1)
    hist = net.fit(t(X, dev), t(y, dev), steps=1500, lr=3e-3, log_every=500)
    assert hist[-1][1] < 0.05 * hist[0][1], hist


@pytest.mark.parametrize("T,weighted", [(16, True), (64, False), (65, True), (8193, False), (20011, True)])
def test_mlp_grad_over_row_blocks(dev, T, weighted):
    """16 rows per wavefront, 64 per workgroup, 8,192 per pass of the grid: both sides
    of each, against the FP64 oracle with the same rounding points (bounds as above:
    occasional one-ulp bfloat16 flips of hidden units)."""
    from splatting_amd.learned import RateNet
    rng = np.random.default_rng(T)
    X = rng.normal(size=(T, M.N_IN)).astype(np.float32)
    P = (rng.normal(size=M.N_PARAMS) * 0.2).astype(np.float32)
    tgt = rng.normal(size=T).astype(np.float32)
    w = rng.uniform(0.5, 2.0, size=T).astype(np.float32) if weighted else None
    net = RateNet(t(P, dev), t(np.zeros(M.N_IN), dev), t(np.ones(M.N_IN), dev))
    loss, g = net.loss_grad(t(X, dev), t(tgt, dev), None if w is None else t(w, dev))
    lr, gr = M.loss_grad(X, P, tgt, w, quant=True)
    assert abs(float(loss.item()) - lr) <= 1e-2 * lr
    assert rel(g.cpu().numpy(), gr) < 2e-2
    assert rel(net.forward(t(X, dev)).cpu().numpy(), M.forward(X, P, quant=True)[0]) < 5e-3


@pytest.mark.parametrize("shape", [(1,), (2, 5, 7), (1, 1500)])
def test_tile_scale_formula(dev, shape):
    """RateNet.tile_scale equals its formula in float64 on the network's own
    predictions (non-finite ones included) to float32 rounding."""
    from splatting_amd.learned import RateNet
    rng = np.random.default_rng(len(shape))
    T = int(np.prod(shape))
    F = t(rng.normal(size=shape + (M.N_IN,)), dev)
    if T > 1:
        F.view(-1, M.N_IN)[1, 3] = float("nan")
    c = t(rng.uniform(0.0, 3000.0, size=shape), dev)
    net = RateNet(t(rng.normal(size=M.N_PARAMS) * 0.3, dev), t(rng.normal(size=M.N_IN), dev),
                  t(rng.uniform(0.5, 2.0, size=M.N_IN), dev))
    y = torch.nan_to_num(net.forward(F.reshape(-1, M.N_IN)).double(), nan=0.0, posinf=20.0, neginf=-20.0)
    cd = c.reshape(-1).double()
    tot = cd.sum().clamp(min=1e-30)
    s = torch.exp((y - (y * cd).sum() / tot).clamp(-20.0, 20.0))
    for _ in range(3):
        s = (s * (tot / (s * cd).sum().clamp(min=1e-30))).clamp(0.75, 4.0)
    got = net.tile_scale(F, c)
    assert got.shape == c.shape
    assert rel(got.reshape(-1).cpu().numpy(), s.cpu().numpy()) < 2.0 ** -23


def scale_case(dev, T, seed=5):
    from splatting_amd.learned import RateNet
    rng = np.random.default_rng(seed)
    net = RateNet(t(rng.normal(size=M.N_PARAMS) * 0.3, dev), t(rng.normal(size=M.N_IN), dev),
                  t(rng.uniform(0.5, 2.0, size=M.N_IN), dev))
    return net, t(rng.normal(size=(T, M.N_IN)), dev), t(rng.uniform(0.0, 3000.0, size=T), dev)


def scale_formula(net, F, c, lo, hi):
    y = net.forward(F).double()
    cd = c.double()
    tot = cd.sum()
    s = torch.exp((y - (y * cd).sum() / tot).clamp(-20.0, 20.0))
    for _ in range(3):
        s = (s * (tot / (s * cd).sum())).clamp(lo, hi)
    return s


@pytest.mark.parametrize("T", [65535, 65536, 65537, 300_000])
def test_tile_scale_of_many_tiles(dev, T):
    """Around the count from which the sums over the tiles leave their one workgroup, to
    float32 rounding of the formula in float64."""
    net, F, c = scale_case(dev, T)
    assert rel(net.tile_scale(F, c).cpu().numpy(), scale_formula(net, F, c, 0.75, 4.0).cpu().numpy()) < 2.0 ** -23


@pytest.mark.parametrize("lo,hi", [(None, 4.0), (0.75, None), (torch.tensor(0.5), torch.tensor(2.0))])
def test_tile_scale_open_and_tensor_bounds(dev, lo, hi):
    """Bounds as torch.clamp takes them."""
    lo, hi = (x.to(dev) if isinstance(x, torch.Tensor) else x for x in (lo, hi))
    net, F, c = scale_case(dev, 40)
    assert rel(net.tile_scale(F, c, lo, hi).cpu().numpy(), scale_formula(net, F, c, lo, hi).cpu().numpy()) < 2.0 ** -23


def test_tile_scale_gradient_of_counts(dev):
    """The multipliers are differentiable in the counts, in reverse and in forward mode."""
    net, F, c = scale_case(dev, 60)
    g = t(np.random.default_rng(2).normal(size=60), dev)
    v = t(np.random.default_rng(3).normal(size=60), dev)
    a, b = (c.double().requires_grad_(True) for _ in range(2))
    ga, = torch.autograd.grad(net.tile_scale(F, a), a, g)
    gb, = torch.autograd.grad(scale_formula(net, F, b, 0.75, 4.0), b, g.double())
    assert torch.allclose(ga, gb, rtol=1e-6, atol=1e-9 * float(gb.abs().max()))
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(c.double(), v.double())
        tangent = torch.autograd.forward_ad.unpack_dual(net.tile_scale(F, dual)).tangent
    assert abs(float((tangent.double() * g).sum()) - float((gb * v).sum())) < 1e-5 * float((gb * v).abs().sum())
    with torch.no_grad():
        assert not net.tile_scale(F, a).requires_grad


def ordered_case(T, seed):
    """Hidden units that are exact: H1 = relu of the features and of their negatives, H2 = H1."""
    rng = np.random.default_rng(seed)
    X = M.bf16(rng.normal(size=(T, M.N_IN))).astype(np.float32)
    P = np.zeros(M.N_PARAMS, np.float32)
    P[:M.OFF_B1] = np.hstack([np.eye(M.N_IN), -np.eye(M.N_IN)]).ravel()
    P[M.OFF_W2:M.OFF_B2] = np.eye(M.N_HID).ravel()
    P[M.OFF_W3:M.OFF_B3] = M.bf16(rng.normal(size=M.N_HID))
    P[M.OFF_B3] = rng.normal()
    tgt, w = rng.normal(size=T).astype(np.float32), rng.uniform(0.5, 2.0, size=T).astype(np.float32)
    H = np.maximum(np.hstack([X, -X]), 0.0).astype(np.float32)
    y = np.zeros(T, np.float32)
    for k in range(M.N_HID):                    # exact products (16 bits), float32 sums in order
        y = y + H[:, k] * P[M.OFF_W3 + k]
    return X, P, tgt, w, H, y + P[M.OFF_B3]


@pytest.mark.parametrize("T", [1, 15, 64, 333, 20011])
def test_output_layer_sums_in_order(dev, T):
    from splatting_amd.learned import RateNet
    X, P, _, _, _, y = ordered_case(T, T)
    net = RateNet(t(P, dev), t(np.zeros(M.N_IN), dev), t(np.ones(M.N_IN), dev))
    assert np.array_equal(net.forward(t(X, dev)).cpu().numpy(), y)


@pytest.mark.parametrize("T", [1, 33, 320, 1025])
def test_output_gradient_rounds_the_ordered_sums(dev, T):
    """dZ2 = bf16(dy W3) of dy in float32 from the sums in order.  dW2 sums at most T exact
    products per element in float32, within T 2^-23 of their magnitudes; a term rounded the
    other way is 2^-8 of itself off."""
    from splatting_amd.learned import RateNet
    f = np.float32
    for seed in range(12):
        X, P, tgt, w, H, y = ordered_case(T, 1000 * T + seed)
        s = np.zeros(1024, f)
        for a in range(0, T, 1024):
            s[:min(1024, T - a)] += w[a:a + 1024]
        while len(s) > 1:
            s = s[:len(s) // 2] + s[len(s) // 2:]
        dy = (f(2.0) * w) * (y - tgt) * (f(1.0) / s[0])
        z = M.bf16(dy[:, None] * P[M.OFF_W3:M.OFF_B3]) * (H > 0)
        ref, mag = H.T.astype(np.float64) @ z, H.T.astype(np.float64) @ np.abs(z)
        net = RateNet(t(P, dev), t(np.zeros(M.N_IN), dev), t(np.ones(M.N_IN), dev))
        g = net.loss_grad(t(X, dev), t(tgt, dev), t(w, dev))[1].cpu().numpy()
        assert np.all(np.abs(g[M.OFF_W2:M.OFF_B2].reshape(ref.shape) - ref) <= T * 2.0 ** -23 * mag)
