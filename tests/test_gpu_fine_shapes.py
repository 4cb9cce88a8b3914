"""The wave-per-ray resampler at every compiled shape (32, 48, 64 coarse bins x 64, 128
fine samples), both cdf modes: bin indices, draws and the merged row against the
oracle bit for bit (TF order), and the merged row as the sorted union of the coarse
and fine values with ties, empty and one-hot weights, and draws on the inner edges
(both modes).  The oracle's float operations are the kernel's, so no tolerance."""
import pytest
import torch

from test_gpu_parity import DEV, _oracle_coarse_weights, _rays_batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 6, 261])
@pytest.mark.parametrize("compensated", [False, True])
@pytest.mark.parametrize("Nf", [64, 128])
@pytest.mark.parametrize("Nc", [32, 48, 64])
def test_fine_shapes(nerf, oracle, Nc, Nf, compensated, n):
    P, Po = nerf.Params(N_coarse=Nc, N_fine=Nf), oracle.make_params(N_coarse=Nc, N_fine=Nf)
    ro, rd, near, far = _rays_batch(nerf, n, seed=3)
    u_c = torch.rand((n, Nc), device=DEV, generator=torch.Generator(device=DEV).manual_seed(1))
    u_c[0, ::2] = 1.0                        # a coarse value on its bin's right edge
    if n > 1:
        u_c[1] = 0.0                         # coarse values on the left edges: ties with draws of 0
    dc = nerf.ray_utils.create_input_batch_coarse_model(P, ro, rd, near, far, u_vals=u_c, materialize=False)
    rc = oracle.create_input_batch_coarse_model(Po, ro.cpu(), rd.cpu(), near.cpu(), far.cpu(), u_vals=u_c.cpu())
    assert torch.equal(dc["t_vals"].cpu(), rc["t_vals"]) and \
        torch.equal(dc["bin_data"]["bin_edges"].cpu(), rc["bin_data"]["bin_edges"])
    w = _oracle_coarse_weights(oracle, max(n, 3), Nc, seed=5)[:n]
    u_f = torch.rand((n, Nf), generator=torch.Generator().manual_seed(2))
    agg = oracle.sample_pdf(w, rc["bin_data"]["left_edges"], rc["bin_data"]["bin_widths"], u_f)[3]
    if n > 5:
        u_f[1, : Nc - 1] = agg[1, 1:Nc]      # exactly on every inner edge
        u_f[3] = 0.0
        u_f[4] = 1.0 - 2.0 ** -24
        u_f[5] = agg[5, 2:3].expand(Nf)
    df = nerf.ray_utils.create_input_batch_fine_model(P, ro, rd, w.to(DEV), dc["bin_data"], dc["t_vals"],
                                                      u_vals=u_f.to(DEV), return_indices=True,
                                                      compensated=compensated, return_cdf=True)
    if not compensated:
        rf = oracle.create_input_batch_fine_model(Po, ro.cpu(), rd.cpu(), w, rc["bin_data"], rc["t_vals"], u_vals=u_f)
        for k in ("piece_idxs", "t_vals_fine", "t_vals", "xyz_inputs", "dir_inputs"):
            assert torch.equal(df[k].cpu(), rf[k]), k
    want = torch.searchsorted(df["cdf"][:, 1:-1].contiguous(), u_f.to(DEV), right=True)
    assert torch.equal(df["piece_idxs"].long(), want)
    union = torch.sort(torch.cat([dc["t_vals"], df["t_vals_fine"]], dim=1), dim=1).values
    assert torch.equal(df["t_vals"], union)
