"""The training step's entry points where one stands in for another: both stores of gx and both tile heights of the dense
sampled products."""
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


@pytest.mark.parametrize("rows,cols,n", [(1024, 4096, 512), (4096, 1024, 515), (1024, 4096, 2048), (512, 2048, 300)])
def test_dense_sampled_products_on_either_tile_height(rows, cols, n, device):
    """hffn_grad_dense and hffn_grad_dense_planes: the same bits, and the sampled product within the split operands' error
    (2^-21 of the sum of the products' magnitudes)."""
    lib, ld, slots = _lib.load(), leading_dim(n), 40
    offsets, index, _ = _support(rows, cols, slots, device)
    drawn = torch.Generator(device=device).manual_seed(2)
    row, mat = (torch.randn(count * ld, generator=drawn, device=device) for count in (rows, cols))
    need = _lib.query_bytes(lib.hffn_grad_dense_workspace, rows, cols, n)
    results = []
    for entry in (lib.hffn_grad_dense, lib.hffn_grad_dense_planes):
        work = torch.empty(need, dtype=torch.uint8, device=device)
        g, gb = torch.full((rows * slots,), float("nan"), device=device), torch.full((rows,), float("nan"), device=device)
        _lib.check(entry(row.data_ptr(), mat.data_ptr(), offsets.data_ptr(), index.data_ptr(), g.data_ptr(), gb.data_ptr(), rows, cols, n,
                         ld, work.data_ptr(), need, _stream()), "sampled product")
        results.append((g, gb))
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])
    a, b = row.view(rows, ld)[:, :n].double(), mat.view(cols, ld)[:, :n].double()
    owner, column = torch.arange(rows, device=device).repeat_interleave(slots), index.long()
    expected, size = (a @ b.T)[owner, column], (a.abs() @ b.abs().T)[owner, column]
    assert bool(((results[0][0].double() - expected).abs() <= 2.0 ** -21 * size).all())
    assert bool(((results[0][1].double() - a.sum(1)).abs() <= n * 2.0 ** -24 * a.abs().sum(1)).all())
