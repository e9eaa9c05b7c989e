"""The training step's loss at the edges of its sum over workgroups (16 reads at a time,
chunks of 1024): a batch that repeats one group of 64 samples has that group's loss, up to
the FP32 rounding of a sum of nblk equal terms, nblk * 2^-24, and of one more operation."""
from __future__ import annotations

import sys

import numpy as np
import pytest

from tests.test_gpu_mlp import _data, _dev, _params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nblk", [2, 15, 16, 17, 1024, 1025, 2050])
def test_loss_of_repeated_blocks(nblk):
    import torch
    from sailfish_amd.closure import ClosureMLP
    print(f"[case] mlp loss nblk={nblk}", file=sys.stderr, flush=True)
    Xb, Yd = _dev(*_data(64))
    mlp = ClosureMLP(max_blocks=nblk, params=_params())
    loss = []
    for n in (1, nblk):
        mlp.train_step(Xb, Yd, torch.arange(64, dtype=torch.int32).repeat(n).cuda(), adam=False, ntile=1)
        loss.append(float(mlp.get_grad()[1]))
    mlp.close()
    assert np.isfinite(loss[0]) and loss[0] > 0
    assert abs(loss[1] - loss[0]) <= (nblk + 2) * 2.0 ** -24 * loss[0]
