"""FP32 forward of the 8x256 net on split FP16 products: batch sizes around the workgroup and
dispatch edges against 64 bits, and power-of-two scales that leave the result's bits alone."""
import importlib

import numpy as np
import pytest
import torch

oracle = importlib.import_module("oracle.restatement")
pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def nerf():
    return importlib.import_module("nerf-tf2_amd")


def _net(nerf, seed=3, scale=None):
    mlp = nerf.NerfMLP("fine", seed=seed, device=DEV)
    w = mlp.get_weights()
    rng = np.random.default_rng(seed)
    w = [a if a.ndim == 2 else rng.normal(0.0, 0.05, a.shape).astype(np.float32) for a in w]
    w[-1] = w[-1] + np.float32(0.3)
    if scale is not None:
        w = scale(w)
    mlp.set_weights(w)
    return mlp, w


def _points(m, seed, size=1.2):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = size * (2 * torch.rand((m, 3), generator=g, device=DEV) - 1)
    d = torch.randn((m, 3), generator=g, device=DEV)
    return x, d / d.norm(dim=1, keepdim=True)


def _encode64(x, L):
    """Arguments in float32, as the encoding defines them; sines and cosines in 64 bits."""
    mult = 2.0 ** torch.arange(L, dtype=torch.float32) * torch.tensor(np.float32(np.pi))
    a = (x.cpu()[..., None] * mult).double()
    return torch.cat([x.cpu().double(), torch.stack([a.sin(), a.cos()], -1).reshape(x.shape[0], -1)], -1)


def _forward64(w, x, d):
    w = [torch.from_numpy(a).double() for a in w]
    e = _encode64(x, 10)
    h = e
    for i in range(8):
        h = torch.relu(h @ w[2 * i] + w[2 * i + 1])
        if i == 4:
            h = torch.cat([h, e], -1)
    r = torch.relu(torch.cat([h @ w[16] + w[17], _encode64(d, 4)], -1) @ w[18] + w[19])
    return torch.sigmoid(r @ w[20] + w[21]), torch.relu(h @ w[22] + w[23])


# One FP32 rounding per term of a K-term sum is off by about sqrt(K) 2^-25 of the sum's norm, 5e-7 at
# K = 256, and ReLU layers pass a relative error on as it is: 1e-6 holds for FP32 sums.
TOL = 1e-6


@pytest.mark.parametrize("m", [1, 31, 33, 65, 8191, 8193, 16411])
@pytest.mark.parametrize("size", [1.2, 300.0])
def test_forward_against_64_bits(nerf, m, size):
    mlp, w = _net(nerf)
    x, d = _points(m, m, size)
    with torch.no_grad():
        rgb, sigma = mlp((x, d))
    stash = mlp._alloc_stash(m)
    rgb2, sigma2 = torch.empty_like(rgb), torch.empty_like(sigma)
    mlp._launch_forward(m, x, d, None, None, None, rgb2, sigma2, stash)
    assert torch.equal(rgb, rgb2) and torch.equal(sigma, sigma2)
    pick = torch.unique(torch.cat([torch.arange(min(m, 300)), torch.arange(max(0, m - 300), m)]))
    rgb64, sigma64 = _forward64(w, x[pick], d[pick])
    for got, want in ((rgb, rgb64), (sigma, sigma64)):
        err = (got[pick].cpu().double() - want).norm()
        assert float(err) <= TOL * float(want.norm()), float(err)     # (0 <= 0 where a single density is 0)


@pytest.mark.parametrize("e", [40, -40])
def test_power_of_two_scales(nerf, e):
    """Layer 2 times 2^e (its ReLU output with it) and layer 3's kernel times 2^-e: the same bits."""
    def scale(w):
        w = list(w)
        w[4], w[5] = np.ldexp(w[4], e), np.ldexp(w[5], e)
        w[6] = np.ldexp(w[6], -e)
        return w
    x, d = _points(777, 5)
    a, _ = _net(nerf)
    b, _ = _net(nerf, scale=scale)
    with torch.no_grad():
        ra, sa = a((x, d))
        rb, sb = b((x, d))
    assert torch.equal(ra, rb) and torch.equal(sa, sb)


NETS = {"nerf": dict(), "proposal": dict(depth=4, width=64, skip=-1, l_xyz=8, l_dir=0),
        "narrow": dict(depth=4, width=32, skip=1)}


@pytest.mark.parametrize("m", [1, 31, 33, 257, 8209, 30011])
@pytest.mark.parametrize("net", list(NETS))
@pytest.mark.parametrize("least", [False, True])
def test_weight_grads_against_64_bits(nerf, net, m, least):
    """FP32 weight gradients of the hidden layers and the density head from a random stash and dz
    whose rows differ by powers of two, against 64 bits: chunk and split edges, every tile shape,
    with the workspace that is asked for and with the least that is taken (least)."""
    import ctypes
    L = nerf._lib
    cfg = nerf.MLPConfig(**NETS[net])
    mlp = nerf.NerfMLP("fine", cfg, "fp32", seed=1, device=DEV)
    d = ctypes.byref(mlp._desc)
    g = torch.Generator(device=DEV).manual_seed(m)
    stash = torch.randn((m, mlp.stash_per_sample), generator=g, device=DEV).relu()
    dz = torch.randn((m, mlp.dz_per_sample), generator=g, device=DEV)
    dz *= 2.0 ** torch.randint(-12, 13, (m, 1), generator=g, device=DEV)
    ws = int(L.load().nerf_mlp_wgrad_workspace_bytes(d, m))
    if least:
        rc = L.load().nerf_mlp_weight_grads(d, 0, m, stash.data_ptr(), dz.data_ptr(), dz.data_ptr(), 0,
                                            stash.data_ptr(), 0, L.stream())
        assert rc == L.NERF_ERR_INVALID_ARG
        ws = int(L.load().nerf_last_error().decode().split("needs ")[1].split()[0])
    work = torch.empty(ws, dtype=torch.uint8, device=DEV)
    grad = torch.full((mlp.n_params,), float("nan"), device=DEV)
    L.call("nerf_mlp_weight_grads", d, 0, m, L.ptr(stash), L.ptr(dz), L.ptr(grad), 0, L.ptr(work), ws, L.stream())
    assert bool(torch.isfinite(grad).all())
    W, D = cfg.width, cfg.depth
    enc = 2 * ((2 + 3 * cfg.l_xyz + 7) // 8 * 8)
    z_sigma = D * W + (W + (W // 2 + 31) // 32 * 32 if cfg.l_dir else 0)
    off = 0
    for i, (name, fi, fo) in enumerate(cfg.layer_shapes()):
        k, b = grad[off:off + fi * fo].view(fi, fo), grad[off + fi * fo:off + fi * fo + fo]
        off += fi * fo + fo
        if name == "sigma":
            x0, z0 = enc + (D - 1) * W, z_sigma
        elif 1 <= i < D:
            x0, z0 = enc + (i - 1) * W, i * W
        else:
            continue
        x, z = stash[:, x0:x0 + W].cpu().double(), dz[:, z0:z0 + fo].cpu().double()
        for got, want in ((k[:W], x.T @ z), (b, z.sum(0))):
            err = (got.cpu().double() - want).norm()
            assert float(err) <= TOL * float(want.norm()), (name, float(err / want.norm()))


@pytest.mark.parametrize("m", [129, 4099])
@pytest.mark.parametrize("width", [32, 64, 128, 160, 256])
@pytest.mark.parametrize("shift", [0, 1])
def test_weight_grads_of_growing_rows(nerf, width, m, shift):
    """dz grows by 2^30 over every 128 rows, and every second feature is zero in the larger half of
    them: its gradients are sums of small terms only.  Rows on 16 bytes and 4 bytes off them
    (shift); every tile shape, whole and in part."""
    import ctypes
    L = nerf._lib
    cfg = nerf.MLPConfig(depth=3, width=width, skip=1)
    mlp = nerf.NerfMLP("fine", cfg, "fp32", seed=1, device=DEV)
    d = ctypes.byref(mlp._desc)
    g = torch.Generator(device=DEV).manual_seed(m)
    stash = torch.randn(m * mlp.stash_per_sample + shift, generator=g, device=DEV)[shift:].view(m, -1).relu_()
    dz = torch.randn(m * mlp.dz_per_sample + shift, generator=g, device=DEV)[shift:].view(m, -1)
    i = torch.arange(m, device=DEV)[:, None] % 128
    dz *= 2.0 ** (i * 30 // 128)
    stash[:, ::2] *= i < 64
    work = torch.empty(int(L.load().nerf_mlp_wgrad_workspace_bytes(d, m)), dtype=torch.uint8, device=DEV)
    grad = torch.full((mlp.n_params,), float("nan"), device=DEV)
    L.call("nerf_mlp_weight_grads", d, 0, m, stash.data_ptr(), dz.data_ptr(), L.ptr(grad), 0, L.ptr(work), work.numel(),
           L.stream())
    enc, off = 2 * ((2 + 3 * cfg.l_xyz + 7) // 8 * 8), 0
    for j, (name, fi, fo) in enumerate(cfg.layer_shapes()[:3]):
        k = grad[off:off + fi * fo].view(fi, fo)[:width].cpu().double()
        off += fi * fo + fo
        if j == 0:
            continue
        x = stash[:, enc + (j - 1) * width:enc + j * width].cpu().double()
        want = x.T @ dz[:, j * width:(j + 1) * width].cpu().double()
        for half in (0, 1):
            err = (k[half::2] - want[half::2]).norm()
            assert float(err) <= TOL * float(want[half::2].norm()), (name, half, float(err / want[half::2].norm()))


@pytest.mark.parametrize("m", [1, 33, 8191, 8193])
def test_dx_rows_against_64_bits(nerf, m):
    """Every sample's dz rows of the 8x256 net against 64 bits on the GPU's ReLU branches, sample
    by sample, with cotangents from 2^-40 to 2^40 (each sample has its own scale) and some zero."""
    import ctypes
    L = nerf._lib
    mlp, w = _net(nerf)
    x, d = _points(m, m)
    rgb, sigma, stash = torch.empty((m, 3), device=DEV), torch.empty((m, 1), device=DEV), mlp._alloc_stash(m)
    mlp._launch_forward(m, x, d, None, None, None, rgb, sigma, stash)
    g = torch.Generator(device=DEV).manual_seed(m)
    scale = 2.0 ** torch.randint(-40, 41, (m, 1), generator=g, device=DEV)
    scale[torch.rand((m, 1), generator=g, device=DEV) < 0.1] = 0.0
    g_rgb = scale * torch.randn((m, 3), generator=g, device=DEV)
    g_sigma = scale * torch.randn((m, 1), generator=g, device=DEV)
    dz = torch.full((m, mlp.dz_per_sample), float("nan"), device=DEV)
    L.call("nerf_mlp_backward", ctypes.byref(mlp._desc), mlp.prec, L.ptr(mlp.packed), m, L.ptr(g_rgb), L.ptr(g_sigma),
           L.ptr(rgb), L.ptr(sigma), L.ptr(stash), L.ptr(dz), L.stream())
    pick = torch.unique(torch.cat([torch.arange(min(m, 200)), torch.arange(max(0, m - 200), m)]))
    st, z = stash[pick].cpu().double(), dz[pick].cpu().double()
    w = [torch.from_numpy(a).double() for a in w]
    y = rgb[pick].cpu().double()
    d_rgb = g_rgb[pick].cpu().double() * y * (1 - y)
    d_sig = g_sigma[pick].cpu().double() * (sigma[pick].cpu() > 0)
    h = lambda i: st[:, 64 + 256 * i:64 + 256 * (i + 1)]
    dr = (d_rgb @ w[20].T) * (st[:, 64 + 9 * 256:64 + 9 * 256 + 128] > 0)
    db = dr @ w[18][:256].T
    want = {"rbr": (9 * 256, dr), "bottleneck": (8 * 256, db)}
    cur = (db @ w[16].T + d_sig @ w[22].T) * (h(7) > 0)
    want["h7"] = (7 * 256, cur)
    for i in range(7, 0, -1):
        cur = (cur @ w[2 * i][:256].T) * (h(i - 1) > 0)
        want[f"h{i - 1}"] = ((i - 1) * 256, cur)
    for name, (z0, v) in want.items():
        err = (z[:, z0:z0 + v.shape[1]] - v).norm(dim=1)
        assert bool((err <= TOL * v.norm(dim=1)).all()), (name, float((err / v.norm(dim=1)).nan_to_num().max()))
