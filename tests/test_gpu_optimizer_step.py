"""nerf_optimizer_step (one call for the check, Adam, packing and step state of all models)
against the separate entry points: the same bits in every buffer, with and without the check,
clean and overflowing, 1 to 9 models of two topologies, aligned and unaligned buffers."""
import ctypes
import importlib

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _setup(nerf, prec, count, shift):
    """Models (every third one the proposal net) whose buffers start `shift` floats into theirs."""
    out = []
    for i in range(count):
        cfg = nerf.proposal.PROPOSAL_CONFIG if i % 3 == 2 else nerf.MLPConfig()
        mlp = nerf.NerfMLP("fine", cfg, prec, seed=i, device=DEV)
        g = torch.Generator(device=DEV).manual_seed(i)
        buf = lambda t: torch.cat([torch.zeros(shift, device=DEV), t])[shift:]
        n = mlp.n_params
        out.append(dict(mlp=mlp, var=buf(mlp.params), m=buf(1e-3 * torch.randn(n, generator=g, device=DEV)),
                        v=buf(1e-6 * torch.rand(n, generator=g, device=DEV)),
                        grad=buf(32768.0 * torch.randn(n, generator=g, device=DEV)), packed=torch.zeros_like(mlp.packed)))
    return out


@pytest.mark.parametrize("prec,count,shift", [("fp32", 1, 0), ("bf16", 3, 0), ("bf16", 2, 1), ("fp32", 9, 3)])
@pytest.mark.parametrize("check,bad", [(0, None), (1, None), (1, float("inf")), (1, float("nan"))])
def test_matches_separate_calls(nerf, prec, count, shift, check, bad):
    L = nerf._lib
    st0 = torch.zeros(16, dtype=torch.int32, device=DEV)
    st0.view(torch.float32)[0] = 32768.0 if check else 1.0
    st0[4], st0[3] = 7, 1                                   # iterations, good steps (interval 2: the scale moves)
    ends = (2, 2.0, 1.0)
    results = []
    for fused in (False, True):
        ms, st = _setup(nerf, prec, count, shift), st0.clone()
        if bad is not None:
            ms[-1]["grad"][-1] = bad
        s = L.stream()
        if fused:
            arr = (L.NerfOptModel * count)()
            for o, q in zip(arr, ms):
                o.desc, o.precision = ctypes.pointer(q["mlp"]._desc), q["mlp"].prec
                o.params, o.m, o.v, o.grad = (q[k].data_ptr() for k in ("var", "m", "v", "grad"))
                o.grad_n, o.packed = q["grad"].numel(), q["packed"].data_ptr()
            L.call("nerf_optimizer_step", count, arr, 5e-4, 500000, 0.1, 0.9, 0.999, 1e-7, st.data_ptr(), check, *ends, s)
        else:
            L.call("nerf_step_begin", st.data_ptr(), 5e-4, 500000, 0.1, 0.9, 0.999, s)
            for q in ms:
                if check:
                    L.call("nerf_check_finite", q["grad"].numel(), q["grad"].data_ptr(), st.data_ptr() + 8, s)
            for q in ms:
                L.call("nerf_adam_tf_state", q["mlp"].n_params, q["var"].data_ptr(), q["m"].data_ptr(), q["v"].data_ptr(),
                       q["grad"].data_ptr(), 1e-7, st.data_ptr(), s)
                L.call("nerf_mlp_pack", ctypes.byref(q["mlp"]._desc), q["mlp"].prec, q["var"].data_ptr(),
                       q["packed"].data_ptr(), s)
            L.call("nerf_step_end", st.data_ptr(), *ends, s)
        results.append((ms, st))
    (a, sa), (b, sb) = results
    assert torch.equal(sa, sb)
    for qa, qb in zip(a, b):
        for k in ("var", "m", "v", "packed"):
            assert torch.equal(qa[k], qb[k]), k
