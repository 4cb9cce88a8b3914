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
