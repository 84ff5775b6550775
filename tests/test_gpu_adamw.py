"""``HFFNTrainRuntime.adamw`` over all four arrays: tensors a caller puts into the dictionaries that ``gradients`` and
``moments`` hand out are the ones the update reads and writes, the same bits as the same values in the runtime's own
tensors."""
from __future__ import annotations

import pytest
import torch

from hffn_amd import synth
from hffn_amd.ffn import hip_layer
from hffn_amd.runtime import HFFNRuntime
from hffn_amd.train_runtime import PARAMETERS, HFFNTrainRuntime

pytestmark = pytest.mark.gpu


def _trainer(device):
    layer = hip_layer(synth.make_layer(synth.CASES["irreg_512_2048"]))
    return HFFNTrainRuntime(HFFNRuntime([layer], device), max_tokens=1)


def test_update_reads_replaced_tensors(device):
    own, other = _trainer(device), _trainer(device)
    drawn = torch.Generator(device=device).manual_seed(5)
    for name in PARAMETERS:
        count = own.gradients(0)[name].numel()
        g, m, v = (torch.randn(count, generator=drawn, device=device) for _ in range(3))
        for target, source in zip((own.gradients(0)[name], *own.moments(0)[name]), (g, m, v.abs())):
            target.copy_(source)
        other.gradients(0)[name], other.moments(0)[name] = g, (m, v.abs())
    for trainer in (own, other):
        trainer.adamw(0)
    for name in PARAMETERS:
        assert torch.equal(own.parameters(0)[name], other.parameters(0)[name])
        for a, b in zip(own.moments(0)[name], other.moments(0)[name]):
            assert torch.equal(a, b)
