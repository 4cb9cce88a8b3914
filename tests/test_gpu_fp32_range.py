"""FP32 products of the 8x256 net over FP32's range: nets whose neurons are rescaled by powers of
two are the same functions and have to give the same bits, and values pass through unchanged."""
import importlib

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
M = 777


@pytest.fixture(scope="module")
def nerf():
    return importlib.import_module("nerf-tf2_amd")


def _weights(nerf, seed=3):
    mlp = nerf.NerfMLP("fine", seed=seed, device=DEV)
    rng = np.random.default_rng(seed)
    w = [a if a.ndim == 2 else rng.normal(0.0, 0.05, a.shape).astype(np.float32) for a in mlp.get_weights()]
    w[-1] = w[-1] + np.float32(0.3)
    return mlp, w


def _points(m=M, seed=5):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = 1.2 * (2 * torch.rand((m, 3), generator=g, device=DEV) - 1)
    d = torch.randn((m, 3), generator=g, device=DEV)
    return x, d / d.norm(dim=1, keepdim=True)


def _forward(mlp, w, m=M):
    mlp.set_weights(w)
    x, d = _points(m)
    rgb, sigma, stash = torch.empty((m, 3), device=DEV), torch.empty((m, 1), device=DEV), mlp._alloc_stash(m)
    mlp._launch_forward(m, x, d, None, None, None, rgb, sigma, stash)
    with torch.no_grad():
        assert all(torch.equal(a, b) for a, b in zip((rgb, sigma), mlp((x, d))))
    return rgb, sigma, stash


# layer -> (its weights, the next layer's): the next layer's first 256 rows are the hidden input
# (below the encoding's rows in the skip layer and the rgb branch)
LAYERS = {"plain": (4, 6), "skip": (8, 10), "rgb branch": (16, 18)}


def rescale(w, layer, k, features):
    """`features` of the layer's outputs times 2^k, their rows of the next kernel times 2^-k."""
    a, b = LAYERS[layer]
    w = [v.copy() for v in w]
    w[a][:, features] = np.ldexp(w[a][:, features], k)
    w[a + 1][features] = np.ldexp(w[a + 1][features], k)
    rows = np.arange(256)[features]
    w[b][rows] = np.ldexp(w[b][rows], -k)
    return w


FEATURES = {"some": np.arange(5, 256, 32), "one": np.array([77]), "all": np.arange(256)}


@pytest.mark.parametrize("layer", list(LAYERS))
@pytest.mark.parametrize("features", list(FEATURES))
@pytest.mark.parametrize("k", [-100, -40, -30, -24, 20, 24, 40, 100])
def test_rescaled_neurons_forward(nerf, layer, features, k):
    mlp, w = _weights(nerf)
    rgb, sigma, _ = _forward(mlp, w)
    rgb_k, sigma_k, _ = _forward(mlp, rescale(w, layer, k, FEATURES[features]))
    assert torch.equal(rgb, rgb_k) and torch.equal(sigma, sigma_k)


@pytest.mark.parametrize("k", [-100, -20, 0, 20, 120])
def test_values_pass_through_a_permutation(nerf, k):
    """A layer whose kernel is 2^k times a permutation, without a bias: its outputs are the layer's
    inputs times 2^k, bit for bit, also where they differ by many powers of two."""
    mlp, w = _weights(nerf)
    perm = np.random.default_rng(0).permutation(256)
    spread = np.random.default_rng(1).integers(-18, 1, 256) if k > 0 else np.random.default_rng(1).integers(0, 19, 256)
    w[4], w[5] = np.ldexp(w[4], spread), np.ldexp(w[5], spread)
    w[6] = np.zeros_like(w[6])
    w[6][perm, np.arange(256)] = np.float32(2.0 ** k)
    w[7] = np.zeros_like(w[7])
    _, _, stash = _forward(mlp, w)
    h2, h3 = stash[:, 64 + 512:64 + 768], stash[:, 64 + 768:64 + 1024]
    assert bool((h2 > 0).any()) and torch.equal(h3, h2[:, torch.from_numpy(perm).to(DEV)] * 2.0 ** k)


def _dz_rows(nerf, mlp, w, shift=0, m=M):
    """dz rows of the net for cotangents of ordinary size times 2^shift."""
    import ctypes
    L = nerf._lib
    rgb, sigma, stash = _forward(mlp, w, m)
    g = torch.Generator(device=DEV).manual_seed(11)
    g_rgb = torch.randn((m, 3), generator=g, device=DEV) * 2.0 ** shift
    g_sigma = torch.randn((m, 1), generator=g, device=DEV) * 2.0 ** shift
    dz = torch.full((m, mlp.dz_per_sample), float("nan"), device=DEV)
    L.call("nerf_mlp_backward", ctypes.byref(mlp._desc), mlp.prec, L.ptr(mlp.packed), m, L.ptr(g_rgb), L.ptr(g_sigma),
           L.ptr(rgb), L.ptr(sigma), L.ptr(stash), L.ptr(dz), L.stream())
    return dz[:, :9 * 256 + 128]


DZ = {"plain": 2, "skip": 4, "rgb branch": 8}     # the layer's block of 256 dz columns


@pytest.mark.parametrize("layer", list(LAYERS))
@pytest.mark.parametrize("features", list(FEATURES))
@pytest.mark.parametrize("k", [-60, -40, -24, 24, 40, 60])
def test_rescaled_neurons_backward(nerf, layer, features, k):
    mlp, w = _weights(nerf)
    want = _dz_rows(nerf, mlp, w).clone()
    cols = torch.from_numpy(256 * DZ[layer] + np.arange(256)[FEATURES[features]]).to(DEV)
    want[:, cols] *= 2.0 ** -k
    assert torch.equal(_dz_rows(nerf, mlp, rescale(w, layer, k, FEATURES[features])), want)


@pytest.mark.parametrize("m", [33, 8211])      # one and two sample blocks a workgroup
@pytest.mark.parametrize("k", [-115, -105, -95, -60, 60, 110])
def test_backward_is_linear_in_its_cotangents(nerf, k, m):
    """The same bits for cotangents times 2^k while no value leaves FP32's normal range; where small
    ones do (k <= -95), rounded at 2^-149 as in FP32, each sample's rows to within a few 2^-24 of
    their norm (values of 2^-115 to 2^-122: 2^-149 is at most 2^-27 of them)."""
    mlp, w = _weights(nerf)
    want = _dz_rows(nerf, mlp, w, 0, m).double()
    got = _dz_rows(nerf, mlp, w, k, m).double() * 2.0 ** -k
    if abs(k) <= 60 or k > 0:
        assert torch.equal(got, want)
    else:
        err = (got - want).norm(dim=1)
        assert bool((err <= 1e-6 * want.norm(dim=1)).all()), float((err / want.norm(dim=1)).max())


# a chunk of 32 samples is summed in FP32, chunks and splits after it: 2^-24 of the sum of |x| |z| each
# time, a few of them; the six products leave out 2^-24 of a term at most
TOL_SUM = 1e-6


@pytest.mark.parametrize("width", [32, 128, 256])
@pytest.mark.parametrize("m", [33, 4099])
@pytest.mark.parametrize("spread", [40, 60, 120])
def test_weight_grads_of_samples_of_unlike_size(nerf, width, m, spread):
    """dz of every second sample is 2^-spread of the others', and half of the features are zero in
    the large samples: their gradients are sums of small terms only, each as good as in FP32."""
    import ctypes
    L = nerf._lib
    cfg = nerf.MLPConfig(depth=3, width=width, skip=-1)
    mlp = nerf.NerfMLP("fine", cfg, "fp32", seed=1, device=DEV)
    d = ctypes.byref(mlp._desc)
    g = torch.Generator(device=DEV).manual_seed(m)
    stash = torch.randn((m, mlp.stash_per_sample), generator=g, device=DEV).relu()
    dz = torch.randn((m, mlp.dz_per_sample), generator=g, device=DEV)
    odd = torch.arange(m, device=DEV)[:, None] % 2
    dz *= 2.0 ** (spread // 2 - spread * odd)
    stash[:, ::2] *= odd
    work = torch.empty(int(L.load().nerf_mlp_wgrad_workspace_bytes(d, m)), dtype=torch.uint8, device=DEV)
    grad = torch.full((mlp.n_params,), float("nan"), device=DEV)
    L.call("nerf_mlp_weight_grads", d, 0, m, L.ptr(stash), L.ptr(dz), L.ptr(grad), 0, L.ptr(work), work.numel(),
           L.stream())
    enc, off = 2 * ((2 + 3 * cfg.l_xyz + 7) // 8 * 8), 0
    for j, (name, fi, fo) in enumerate(cfg.layer_shapes()[:3]):
        k = grad[off:off + fi * fo].view(fi, fo).cpu().double()
        off += fi * fo + fo
        if j == 0:
            continue
        x = stash[:, enc + (j - 1) * width:enc + j * width].cpu().double()
        z = dz[:, j * width:(j + 1) * width].cpu().double()
        err, most = (k - x.T @ z).abs(), x.T @ z.abs()
        assert bool((err <= TOL_SUM * most).all()), (name, float((err / most).nan_to_num().max()))


@pytest.mark.parametrize("m", [33, 8211])      # one and two sample blocks a workgroup
@pytest.mark.parametrize("layer", [1, 4, 6])   # (4: the skip layer's input)
def test_infinite_hidden_values(nerf, m, layer):
    """A feature that passes FP32's range is infinite and stays so: the next layer's outputs are
    infinite or zero by the sign of its weights, as the FP32 product of each of them is."""
    mlp, w = _weights(nerf)
    f = 77
    w[2 * layer][:, f], w[2 * layer + 1][f] = 2.0 ** 127, 3.3e38   # infinite for any input above 0.1
    w[22] = np.abs(w[22])
    x, _ = _points(m)
    _, sigma, stash = _forward(mlp, w, m)
    h = lambda i: stash[:, 64 + 256 * i:64 + 256 * (i + 1)]
    assert bool((h(layer)[:, f] == float("inf")).all())
    sign = torch.from_numpy(np.sign(w[2 * layer + 2][f])).to(DEV)
    assert bool((h(layer + 1)[:, sign > 0] == float("inf")).all()) and bool((h(layer + 1)[:, sign < 0] == 0).all())
    if layer == 6:
        assert bool((sigma == float("inf")).all())


@pytest.mark.parametrize("top", [3.3e38, 3.4e38])   # within and above the largest bf16, 3.39e38
def test_largest_finite_values_forward(nerf, top):
    """Hidden values up to FP32's largest are finite inputs: the next layer's kernel takes them back."""
    mlp, w = _weights(nerf)
    f = 77
    w[4][:, f], w[5][f] = 0.0, top                       # h2[f] = top for every sample
    w[6][f] = np.sign(w[6][f]) * np.float32(2.0 ** -127)
    _, _, stash = _forward(mlp, w)
    h = lambda i: stash[:, 64 + 256 * i:64 + 256 * (i + 1)].cpu().double()
    assert bool((h(2)[:, f] == float(np.float32(top))).all())
    want = torch.relu(h(2) @ torch.from_numpy(w[6]).double() + torch.from_numpy(w[7]).double())
    assert float((h(3) - want).norm()) <= 1e-6 * float(want.norm())
