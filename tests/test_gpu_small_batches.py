"""The BF16 8x256 forward with one, two and four sample blocks per workgroup (chosen by the
batch's size): every sample's value is computed in the same order whatever the batch, so a
batch's outputs equal, bit for bit, those of the same samples inside a batch large enough
for the four-block form.  Sizes at the edges of blocks, workgroups and of the dispatch (32 and
64 samples per compute unit)."""
import pytest
import torch

from test_gpu_parity import DEV

pytestmark = pytest.mark.gpu


def test_small_batches(nerf):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    net = nerf.NerfMLP("fine", nerf.MLPConfig(), "bf16", seed=5, device=DEV)
    g = torch.Generator(device=DEV).manual_seed(7)
    most = 64 * cus + 129
    xyz = 2.4 * torch.rand((most, 3), generator=g, device=DEV) - 1.2
    dirs = torch.nn.functional.normalize(torch.randn((most, 3), generator=g, device=DEV), dim=1)
    with torch.no_grad():
        rgb, sigma = net((xyz, dirs))
        for n in (1, 31, 32, 33, 63, 64, 65, 1000, 32 * cus - 1, 32 * cus, 32 * cus + 1, 64 * cus - 31, 64 * cus,
                  64 * cus + 1):
            r, s = net((xyz[:n], dirs[:n]))
            assert torch.equal(r, rgb[:n]) and torch.equal(s, sigma[:n]), n
        # rays: 3 samples a ray, so that rays straddle blocks
        for n in (1, 11, 400, 3000):
            o, d = xyz[:n].contiguous(), dirs[:n].contiguous()
            t = torch.sort(torch.rand((n, 3), generator=g, device=DEV), dim=1).values
            r, s = net.forward_rays(o, d, t)
            pts = (o[:, None] + t[..., None] * d[:, None]).reshape(-1, 3)
            rp, sp = net((pts, d[:, None].expand(n, 3, 3).reshape(-1, 3)))
            assert torch.equal(r, rp) and torch.equal(s, sp), n


def test_proposal_batches(nerf):
    """The 64-wide density net's forward at the edges of blocks, workgroups and of the grid (four
    workgroups of 128 samples a compute unit): a prefix of a batch has the batch's values bit
    for bit, and so have the outputs and whole blocks of the stash of a training forward."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    net = nerf.NerfMLP("fine", nerf.MLPConfig(4, 64, -1, 8, 0), "bf16", seed=6, device=DEV)
    g = torch.Generator(device=DEV).manual_seed(8)
    most = 4 * cus * 128 + 205
    xyz = 2.4 * torch.rand((most, 3), generator=g, device=DEV) - 1.2

    def forward(n, stash=None):
        sigma = torch.full((n, 1), float("nan"), device=DEV)
        net._launch_forward(n, xyz[:n], None, None, None, None, None, sigma, stash)
        return sigma
    full_stash = net._alloc_stash(most)
    full = forward(most, full_stash)
    assert bool(torch.isfinite(full).all()) and torch.equal(forward(most), full)
    S = 5 * 64                                    # written elements of a stash row
    for n in (1, 31, 32, 33, 127, 128, 129, 4 * cus * 128 - 1, 4 * cus * 128 + 1):
        stash = net._alloc_stash(n)
        assert torch.equal(forward(n, stash), full[:n]) and torch.equal(forward(n), full[:n]), n
        k = n // 32 * 32                          # whole blocks: the same layout in both
        a, b = stash.reshape(-1)[:k * stash.shape[1]], full_stash.reshape(-1)[:k * stash.shape[1]]
        chunks = lambda t: t.view(-1, stash.shape[1] // 8, 32, 8)[:, :S // 8].view(torch.int16)
        assert torch.equal(chunks(a), chunks(b)), n
