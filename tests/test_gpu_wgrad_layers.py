"""FP32 weight gradients of every layer, encoding rows, branches and heads among them, against 64 bits."""
import ctypes
import importlib

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"

NETS = {"nerf": dict(), "proposal": dict(depth=4, width=64, skip=-1, l_xyz=8, l_dir=0),
        "narrow": dict(depth=4, width=32, skip=1)}


@pytest.fixture(scope="module")
def nerf():
    return importlib.import_module("nerf-tf2_amd")


def encoding_features(L, slots):
    """Feature of each of the 2 x slots columns of an encoding in the stash; -1 for padding."""
    first = (3 * L - 2) // 2
    out = []
    for half in (0, 1):
        for e in range(slots):
            if half == 0 and e < 4:
                out.append(e if e < 3 else -1)
                continue
            pair = (e - 4) // 2 if half == 0 else first + e // 2
            last = first if half == 0 else 3 * L
            out.append(3 + pair // L * 2 * L + 2 * (pair % L) + e % 2 if pair < last else -1)
    assert sorted(f for f in out if f >= 0) == list(range(3 + 6 * L))
    return out


def layers(cfg):
    """name -> ([(stash column of each input or -1 columns dropped, input rows)], dz column)."""
    W, D = cfg.width, cfg.depth
    pad = lambda L: (2 + 3 * L + 7) // 8 * 8
    wr = (W // 2 + 31) // 32 * 32
    kx, kd = pad(cfg.l_xyz), pad(cfg.l_dir) if cfg.l_dir else 0
    h0 = 2 * kx
    bott = h0 + D * W
    rbr = bott + W
    encd = rbr + wr
    hidden = lambda at, n: (list(range(at, at + n)), list(range(n)))

    def enc(at, L, slots, base):
        f = encoding_features(L, slots)
        return [at + i for i, v in enumerate(f) if v >= 0], [base + v for v in f if v >= 0]

    out = []
    for i in range(D):
        parts = [enc(0, cfg.l_xyz, kx, 0)] if i == 0 else [hidden(h0 + (i - 1) * W, W)]
        if i > 0 and i - 1 == cfg.skip:
            parts.append(enc(0, cfg.l_xyz, kx, W))
        out.append((parts, i * W))
    if cfg.l_dir:
        out.append(([hidden(h0 + (D - 1) * W, W)], D * W))
        out.append(([hidden(bott, W), enc(encd, cfg.l_dir, kd, W)], (D + 1) * W))
        sigma = (D + 1) * W + wr
        out.append(([hidden(rbr, W // 2)], sigma + 8))
        out.append(([hidden(h0 + (D - 1) * W, W)], sigma))
    else:
        out.append(([hidden(h0 + (D - 1) * W, W)], D * W))
    return out


# FP32 sums of 32 samples, of chunks and of splits, of the norm (as in test_gpu_split_products.py)
TOL = 1e-6


@pytest.mark.parametrize("m", [1, 31, 33, 257, 8209, 30011])
@pytest.mark.parametrize("net", list(NETS))
@pytest.mark.parametrize("least", [False, True])
def test_every_layer_against_64_bits(nerf, net, m, least):
    L = nerf._lib
    cfg = nerf.MLPConfig(**NETS[net])
    mlp = nerf.NerfMLP("fine", cfg, "fp32", seed=1, device=DEV)
    d = ctypes.byref(mlp._desc)
    g = torch.Generator(device=DEV).manual_seed(m + 1)
    stash = torch.randn((m, mlp.stash_per_sample), generator=g, device=DEV)
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
    s64, z64, grad = stash.cpu().double(), dz.cpu().double(), grad.cpu().double()
    off = 0
    for (name, fi, fo), (parts, z0) in zip(cfg.layer_shapes(), layers(cfg)):
        k, b = grad[off:off + fi * fo].view(fi, fo), grad[off + fi * fo:off + fi * fo + fo]
        off += fi * fo + fo
        z = z64[:, z0:z0 + fo]
        want = torch.full((fi, fo), float("nan"), dtype=torch.float64)
        for cols, rows in parts:
            want[rows] = s64[:, cols].T @ z
        assert not bool(want.isnan().any())
        # (a head's bias is a single sum, which may cancel: held to the sum of its magnitudes)
        checks = [(f"rows {rows[0]}..", k[rows], want[rows], want[rows]) for _, rows in parts]
        checks.append(("bias", b, z.sum(0), z.abs().sum(0)))
        for what, got, ref, size in checks:
            err = float((got - ref).norm() / size.norm())
            assert err <= TOL, (name, what, err)
    assert off == mlp.n_params
