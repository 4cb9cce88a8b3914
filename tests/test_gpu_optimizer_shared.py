"""Optimizer steps over a list that names one net more than once, and over more gradients than nets."""
import importlib

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def nerf():
    return importlib.import_module("nerf-tf2_amd")


@pytest.mark.parametrize("order", [[0, 0], [0, 1, 0], [0, 1, 1, 0, 0]])
@pytest.mark.parametrize("scaled", [False, True])
def test_a_net_listed_twice_is_updated_twice(nerf, order, scaled):
    """The same bits as one Adam update (of its own moments) after the other."""
    L = nerf._lib
    nets = [nerf.NerfMLP("fine", nerf.MLPConfig(), "bf16", seed=i, device=DEV) for i in (1, 2)]
    models = [nets[i] for i in order]
    grads = [torch.randn(m.n_params, generator=torch.Generator(device=DEV).manual_seed(i), device=DEV)
             for i, m in enumerate(models)]
    want = [net.params.clone() for net in nets]
    ms, vs = [torch.zeros_like(g) for g in grads], [torch.zeros_like(g) for g in grads]
    opt = nerf.AdamTF(models)
    scaler = nerf.DynamicLossScaler(opt) if scaled else None
    st, s = opt.state.clone(), L.stream()
    L.call("nerf_step_begin", st.data_ptr(), 5e-4, 500000, 0.1, 0.9, 0.999, s)
    for i, m, v, g in zip(order, ms, vs, grads):
        L.call("nerf_adam_tf_state", g.numel(), want[i].data_ptr(), m.data_ptr(), v.data_ptr(), g.data_ptr(), 1e-7,
               st.data_ptr(), s)
    opt.apply_gradients(grads, scaler)
    for net, w in zip(nets, want):
        assert torch.equal(net.params, w)
        packed = net.packed.clone()
        net.repack()
        assert torch.equal(net.packed, packed)
    assert all(torch.equal(a, b) for a, b in zip(opt.m + opt.v, ms + vs))


@pytest.mark.parametrize("bad", [None, float("inf"), float("nan")])
def test_gradients_past_the_models_are_checked(nerf, bad):
    """With a scaler every gradient that is given is checked, those of no model too."""
    net = nerf.NerfMLP("fine", nerf.MLPConfig(), "bf16", seed=1, device=DEV)
    opt = nerf.AdamTF([net])
    scaler = nerf.DynamicLossScaler(opt)
    extra = torch.ones(1000, device=DEV)
    if bad is not None:
        extra[999] = bad
    before = net.params.clone()
    for step in (1, 2):
        opt.apply_gradients([torch.ones(net.n_params, device=DEV), extra], scaler)
        assert (opt.iterations, scaler.skipped) == ((step, 0) if bad is None else (0, step))
    assert torch.equal(net.params, before) == (bad is not None)
    opt.apply_gradients([torch.ones(net.n_params, device=DEV)], scaler)
    assert opt.iterations == (3 if bad is None else 1)
