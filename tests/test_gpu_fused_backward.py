"""nerf_mlp_backward_grads (dX chain and weight gradients of the proposal net in one
kernel) against nerf_mlp_backward + nerf_mlp_weight_grads, whose dz it shares bit for bit
(the products are the same, only their order of summation differs).  The reference is
the float64 product of the stash and dz that the separate call writes.

Tolerance, from FP32 sums of M terms: each element is a sum of M products x z, exact in
FP32 (8-bit significands), added in some order in FP32: |error| <= d u sum |x z|, u = 2^-24,
d the longest chain of additions.  A workgroup's half chunk is at most ceil(M / (256 groups
x 256)) x 128 samples in chains, the rest is a tree: d <= 128 ceil(M / 65536) + 256."""
import ctypes

import pytest
import torch

from test_gpu_parity import DEV

pytestmark = pytest.mark.gpu


def _slots(g, e, L):
    """Reference feature of encoding slot e on half g, -1 for padding."""
    H, P0 = 2 + 3 * L, (3 * L - 2) // 2
    if e >= H:
        return -1
    if g == 0:
        if e < 3:
            return e
        if e == 3:
            return -1
        p, sc = (e - 4) // 2, (e - 4) % 2
    else:
        p, sc = P0 + e // 2, e % 2
    return 3 + (p // L) * 2 * L + 2 * (p % L) + sc


def _rows(buf, M):
    """A buffer blocked by 32 samples as plain (M, elements) float64 rows."""
    S = buf.shape[1]
    flat, out = buf.reshape(-1), []
    for b in range(0, M, 32):
        n = min(32, M - b)
        out.append(flat[b * S:(b + n) * S].view(S // 8, n, 8).permute(1, 0, 2).reshape(n, S))
    return torch.cat(out).double()


@pytest.mark.parametrize("M", [1, 31, 32, 255, 257, 4099, 65536 + 33, 150001])
def test_fused_backward(nerf, M):
    L = nerf._lib
    net = nerf.NerfMLP("fine", nerf.MLPConfig(4, 64, -1, 8, 0), "bf16", seed=3, device=DEV)
    g = torch.Generator(device=DEV).manual_seed(M)
    net.params.add_(0.05 * torch.randn(net.params.shape, generator=g, device=DEV))
    net.repack()
    d = ctypes.byref(net._desc)
    assert L.load().nerf_mlp_has_backward_grads(d, net.prec) == 1
    xyz = 2.4 * torch.rand((M, 3), generator=g, device=DEV) - 1.2
    sigma, stash = torch.empty((M, 1), device=DEV), net._alloc_stash(M)
    net._launch_forward(M, xyz, None, None, None, None, None, sigma, stash)
    g_sigma = torch.randn((M, 1), generator=g, device=DEV) * 10.0 ** (-3.0 * torch.rand((M, 1), generator=g, device=DEV))
    dz = torch.empty((M, net.dz_per_sample), dtype=torch.bfloat16, device=DEV)
    L.call("nerf_mlp_backward", d, net.prec, L.ptr(net.packed), M, None, L.ptr(g_sigma), None, L.ptr(sigma),
           L.ptr(stash), L.ptr(dz), L.stream())
    ws = torch.empty(int(L.load().nerf_mlp_wgrad_workspace_bytes(d, M)), dtype=torch.uint8, device=DEV)
    out = torch.full((net.n_params,), float("nan"), device=DEV)

    def grads(accumulate):
        L.call("nerf_mlp_backward_grads", d, net.prec, L.ptr(net.packed), M, L.ptr(g_sigma), L.ptr(sigma),
               L.ptr(stash), L.ptr(out), accumulate, L.ptr(ws), ws.numel(), L.stream())
    grads(0)
    X, Z = _rows(stash, M), _rows(dz, M)
    feats = [_slots(e // 32, e % 32, 8) for e in range(64)]
    keep = torch.tensor([e for e in range(64) if feats[e] >= 0], device=DEV)
    order = torch.argsort(torch.tensor([feats[e] for e in keep.tolist()], device=DEV))
    want, size = [], []
    for l in range(5):
        x = X[:, :64][:, keep[order]] if l == 0 else X[:, 64 * l:64 * l + 64]
        z = Z[:, 64 * l:64 * l + 64] if l < 4 else Z[:, 256:257]
        want += [(x.T @ z).reshape(-1), z.sum(0)]
        size += [(x.abs().T @ z.abs()).reshape(-1), z.abs().sum(0)]
    want, size = torch.cat(want), torch.cat(size)
    tol = (128 * ((M + 65535) // 65536) + 256) * 2.0 ** -24 * size
    assert bool(((out.double() - want).abs() <= tol).all())
    once = out.clone()
    grads(1)
    assert torch.equal(out, once + once)          # deterministic, and added to
    with pytest.raises(ValueError):
        L.call("nerf_mlp_backward_grads", d, 0, L.ptr(net.packed), M, L.ptr(g_sigma), L.ptr(sigma), L.ptr(stash),
               L.ptr(out), 0, L.ptr(ws), ws.numel(), L.stream())
    with pytest.raises(ValueError):
        L.call("nerf_mlp_backward_grads", d, net.prec, L.ptr(net.packed), M, L.ptr(g_sigma), L.ptr(sigma),
               L.ptr(stash), L.ptr(out), 0, L.ptr(ws), 1024, L.stream())
