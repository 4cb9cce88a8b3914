"""Operand packing of descriptions that have no compiled forward: every weight is in the operands."""
import importlib

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def nerf():
    return importlib.import_module("nerf-tf2_amd")


@pytest.mark.parametrize("desc", [(8, 256, 4, 12, 4), (8, 256, 4, 16, 16), (8, 256, 4, 10, 12), (6, 256, 2, 10, 4),
                                  (8, 256, -1, 16, 4), (8, 224, 4, 16, 16)])
def test_every_weight_is_packed(nerf, desc):
    """FP32 operands hold every kernel and bias value (all different and nonzero) as they are, up
    to the widest layers that a description can have (256 + 99 inputs)."""
    depth, width, skip, lx, ld = desc
    cfg = nerf.MLPConfig(depth=depth, width=width, skip=skip, l_xyz=lx, l_dir=ld)
    mlp = nerf.NerfMLP("fine", cfg, "fp32", seed=1, device=DEV)
    values = torch.arange(1, mlp.n_params + 1, dtype=torch.float32, device=DEV)
    mlp.params.copy_(values)
    mlp.packed.fill_(0)
    mlp.repack()
    torch.cuda.synchronize()
    packed = mlp.packed.cpu().numpy().view(np.uint8)
    packed = packed[:packed.size // 4 * 4].view(np.float32)
    assert np.isin(values.cpu().numpy(), packed).all()
