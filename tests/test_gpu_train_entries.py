"""The training step's entry points where one path stands in for another: both stores of gx."""
from __future__ import annotations

import pytest
import torch

from hffn_amd import _lib
from hffn_amd.runtime import leading_dim

pytestmark = pytest.mark.gpu


def _support(rows, width, slots, device, seed=0):
    """(offsets, sorted distinct indices, values) of ``rows`` rows of ``slots`` slots."""
    drawn = torch.Generator(device=device).manual_seed(seed)
    index = torch.rand(rows, width, generator=drawn, device=device).argsort(dim=1)[:, :slots].sort(dim=1).values
    offsets = torch.arange(0, (rows + 1) * slots, slots, dtype=torch.int32, device=device)
    return offsets, index.to(torch.int16).flatten().contiguous(), torch.randn(rows * slots, generator=drawn, device=device)


def _stream():
    return torch.cuda.current_stream().cuda_stream


@pytest.mark.parametrize("d,h,n", [(512, 2048, 1535), (512, 2048, 1536), (512, 2048, 1541), (784, 1600, 1003), (784, 1600, 1004)])
def test_grad_x_on_both_sides_of_its_rule(d, h, n, device):
    """gx token-major (below 3 << 18 entries) and through gx_t (from there on): float32 sums of 48 products in stored order,
    within 48 roundings of the float64 result; buffers of NaNs, so that every entry is written."""
    lib, ld, slots = _lib.load(), leading_dim(n), 48
    offsets, hidden, value = _support(d, h, slots, device)
    gz = torch.randn(h * ld, generator=torch.Generator(device=device).manual_seed(1), device=device)
    gx_t, gx = torch.full((d * ld,), float("nan"), device=device), torch.full((n + 1, d), float("nan"), device=device)
    _lib.check(lib.hffn_grad_x(gz.data_ptr(), offsets.data_ptr(), hidden.data_ptr(), value.data_ptr(), gx_t.data_ptr(), gx.data_ptr(), d, h,
                               d * slots, n, ld, _stream()), "gx")
    dense = torch.zeros(d, h, dtype=torch.float64, device=device)
    dense.scatter_(1, hidden.long().view(d, slots), value.double().view(d, slots))
    rows = gz.view(h, ld)[:, :n].double()
    expected, size = (dense @ rows).T, (dense.abs() @ rows.abs()).T
    assert bool(((gx[:n].double() - expected).abs() <= slots * 2.0 ** -24 * size + 1e-30).all()) and bool(gx[n].isnan().all())
    assert bool(gx_t.isnan().all()) == (n * d < 3 << 18)
