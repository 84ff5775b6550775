"""The choice of planes of the call (``HFFNRuntime.transient``) as a function of N and the layers only: whatever was reserved
and allocated before, on layers whose estimates cross more than once between 65 and 2100 tokens."""
from __future__ import annotations

import pytest

from hffn_amd import _lib
from hffn_amd.runtime import HFFNRuntime, StoreShape

LAYERS = [(512, 2048, 0.05, False), (768, 3072, 0.05, False), (768, 3072, 0.1, False), (1024, 4096, 0.05, False), (2048, 8192, 0.05, True)]


def _runtime(d, h, density, bf16):
    """A runtime's policy without its device buffers."""
    slots = int(2 * d * h * density)
    runtime = HFFNRuntime.__new__(HFFNRuntime)
    runtime.__dict__.update(d_model=d, d_ff=h, density=density, forced_up=None, forced_down=None, _planes=None, _tiles=[], _tokens=0,
                            _transient={}, _transient_allowed=True, _prefill_work=None, _longest=int(density * (d + h)),
                            _store=StoreShape(slots, slots * (4 if bf16 else 6), h),
                            _args=[(_lib.VALUE_BF16 if bf16 else _lib.VALUE_F32,)])
    return runtime


@pytest.mark.parametrize("d,h,density,bf16", LAYERS)
def test_the_path_depends_on_n_and_the_layers_only(d, h, density, bf16):
    counts = (65, 128, 129, 256, 257, 300, 512, 700, 1023, 1024, 1273, 1280, 1281, 1540, 1792, 2000, 2048)
    first = _runtime(d, h, density, bf16)
    chosen = {n: first.transient(n) for n in counts}
    for reserved in (1, 64, 128, 1280, 1281, 1540, 2048):
        for work in (None, object()):
            runtime = _runtime(d, h, density, bf16)
            runtime._tokens, runtime._prefill_work = reserved, work
            assert {n: runtime.transient(n) for n in reversed(counts)} == dict(reversed(chosen.items())), reserved


def test_these_estimates_cross():
    """(What the test above needs to see a choice that follows the reserves: some counts on either path.)"""
    mixed = 0
    for layer in LAYERS:
        runtime = _runtime(*layer)
        mixed += len({runtime.transient(n) for n in range(65, 2100)}) == 2
    assert mixed >= 3
