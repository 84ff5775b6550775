"""The training step's entry points where one stands in for another: both stores of gx, both tile heights of the dense
sampled products, the forward that rebuilds its planes, the backward on planes of its own, AdamW over one array and over
all, gathered values."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from hffn_amd import _lib, synth
from hffn_amd.ffn import hip_layer
from hffn_amd.runtime import HFFNRuntime, leading_dim
from hffn_amd.train_runtime import HFFNTrainRuntime

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


def _trainer(d, h, degrees, device):
    """A trainer with planes over a layer of ``degrees`` slots per neuron on both sides."""
    rng = np.random.default_rng([d, h, int(degrees.sum())])
    offsets = np.zeros(h + 1, np.int32)
    offsets[1:] = np.cumsum(degrees)

    def side():
        index = np.concatenate([np.sort(rng.choice(d, k, replace=False)) for k in degrees]).astype(np.int16)
        return offsets, index, (rng.standard_normal(index.size) * 0.02).astype(np.float32)
    up, down = side(), side()
    b_up, b_down = ((rng.standard_normal(k) * 0.01).astype(np.float32) for k in (h, d))
    layer = synth.CompactLayer(d, h, synth._groups(h), *up, b_up, *down, b_down)
    return HFFNTrainRuntime(HFFNRuntime([hip_layer(layer)], device, dense=True), max_tokens=1)


def _mixed(h, low, high):
    """Alternating numbers of slots, one neuron with ``high`` and one without any."""
    degrees = np.where(np.arange(h) % 2 == 0, low, 1024 - low)
    degrees[5], degrees[6] = high, 0
    return degrees


PLANES = [(512, 2048, np.full(2048, 52), 96),           # both sides read by position, two column chunks of W_up^T
          (1024, 4096, _mixed(4096, 400, 1024), 515),   # W_up^T gathered first; rows of W_down^T beyond a wave's 504 slots
          (1024, 4096, np.full(4096, 103), 300)]        # W_up^T gathered first (four chunks of 418 k slots)
IDS = ["in_place", "long_rows", "gathered"]


def _planes(offsets, index, value, rows, k, device):
    lib = _lib.load()
    plane = torch.full((_lib.query_bytes(lib.hffn_dense_planes_bytes, rows, k) // 2,), float("nan"), dtype=torch.float16, device=device)
    binades = torch.full((rows,), 77, dtype=torch.int32, device=device)
    _lib.check(lib.hffn_densify(_lib.VALUE_F32, offsets.data_ptr(), index.data_ptr(), value.data_ptr(), rows, k, plane.data_ptr(),
                                binades.data_ptr(), _stream()), "densify")
    return plane, binades


def _nan(count, device):
    return torch.full((count,), float("nan"), device=device)


@pytest.mark.parametrize("d,h,degrees,n", PLANES, ids=IDS)
def test_forward_that_rebuilds_its_planes(d, h, degrees, n, device):
    """hffn_forward_mfma_z_refresh on planes of NaNs: planes, z, act, x_t and y bit for bit those of hffn_densify and
    hffn_forward_mfma_z."""
    lib, ld = _lib.load(), leading_dim(n)
    trainer = _trainer(d, h, degrees, device)
    arrays, (_, *model) = trainer.runtime._tensors[0], trainer.runtime._args[0]
    x = torch.randn(n, d, generator=torch.Generator(device=device).manual_seed(3), device=device)
    need = _lib.query_bytes(lib.hffn_train_mfma_workspace, n, d, h)

    def run(refresh):
        up = _planes(arrays["up_offsets"], arrays["up_idx"], arrays["up_val"], h, d, device)
        down = _planes(arrays["out_offsets"], arrays["out_hidden"], arrays["out_val"], d, h, device)
        x_t, act, z, y = _nan(d * ld, device), _nan(h * ld, device), _nan(h * ld, device), _nan(n * d, device)
        work = torch.zeros(need, dtype=torch.uint8, device=device)
        tail = (work.data_ptr(), need, x_t.data_ptr(), act.data_ptr(), z.data_ptr(), y.data_ptr(), d, h, n, ld, _stream())
        held = [t.data_ptr() for t in (*up, *down)]
        if refresh:
            for plane, binades in (up, down):
                plane.fill_(float("nan"))
                binades.fill_(77)
            _lib.check(lib.hffn_forward_mfma_z_refresh(x.data_ptr(), *model, *held, *tail), "refresh")
        else:
            _lib.check(lib.hffn_forward_mfma_z(x.data_ptr(), *held[:2], arrays["b_up"].data_ptr(), *held[2:], arrays["b_down"].data_ptr(),
                                               *tail), "forward with z")
        tokens = [t.view(-1, ld)[:, :n] for t in (x_t, act, z)]
        return [*up, *down, *tokens, y]
    for kept, rebuilt in zip(run(False), run(True)):
        assert not bool(kept.isnan().any()) and torch.equal(kept, rebuilt)


def test_step_after_an_update_reads_the_new_values(device):
    """forward with z after the values changed (invalidate_planes): the bits of a runtime built on the new values, and the
    planes no longer stale; without the change the first values' bits."""
    d, h, n = 512, 2048, 96
    trainer, ld = _trainer(d, h, np.full(2048, 52), device), leading_dim(96)
    x = torch.randn(n, d, generator=torch.Generator(device=device).manual_seed(4), device=device)
    z = torch.empty(h * ld, device=device)
    trainer.forced_train = "mfma"
    before = trainer.forward(0, x, z).clone()
    for name in ("up_val", "out_val"):
        trainer.runtime._tensors[0][name].mul_(-1.5)
    trainer.runtime.invalidate_planes(0)
    after, z_after = trainer.forward(0, x, z).clone(), z.clone()
    assert not trainer.runtime._stale and not torch.equal(before, after)
    fresh = HFFNTrainRuntime(HFFNRuntime(trainer.runtime.layers, device, dense=True), max_tokens=1)
    fresh.forced_train = "mfma"
    assert torch.equal(fresh.forward(0, x, z), after)
    assert torch.equal(z.view(h, ld)[:, :n], z_after.view(h, ld)[:, :n])


@pytest.mark.parametrize("d,h,degrees,n", PLANES, ids=IDS)
def test_backward_on_planes_of_its_own(d, h, degrees, n, device):
    """hffn_backward_planes: gz, gx and gy_t bit for bit those of hffn_densify over gathered values and hffn_backward_mfma,
    from a workspace of any content; both against float64."""
    lib, ld = _lib.load(), leading_dim(n)
    trainer = _trainer(d, h, degrees, device)
    arrays, s = trainer.runtime._tensors[0], trainer.supports(0)
    drawn = torch.Generator(device=device).manual_seed(6)
    gy, z = torch.randn(n, d, generator=drawn, device=device), torch.randn(h * ld, generator=drawn, device=device)
    nnz = arrays["up_val"].numel(), arrays["out_val"].numel()
    hid, into = (torch.empty(count, device=device) for count in reversed(nnz))
    for source, position, target in (("out_val", "hid_pos", hid), ("up_val", "in_pos", into)):
        _lib.check(lib.hffn_gather_values(arrays[source].data_ptr(), s[position].data_ptr(), target.data_ptr(), target.numel(), _stream()), "gather")
        assert torch.equal(target, arrays[source][s[position].long()])
    down_t = _planes(s["hid_offsets"], s["hid_output"], hid, h, d, device)
    up_t = _planes(s["in_offsets"], s["in_hidden"], into, d, h, device)
    need = _lib.query_bytes(lib.hffn_train_mfma_workspace, n, d, h)
    work = torch.zeros(need, dtype=torch.uint8, device=device)
    gz, gx = _nan(h * ld, device), _nan(n * d, device)
    _lib.check(lib.hffn_backward_mfma(gy.data_ptr(), z.data_ptr(), *(t.data_ptr() for t in (*down_t, *up_t)), work.data_ptr(), need,
                                      gz.data_ptr(), gx.data_ptr(), d, h, n, ld, _stream()), "backward")
    need = _lib.query_bytes(lib.hffn_train_planes_workspace, n, d, h)
    work = torch.full((need + 256,), 0x7f, dtype=torch.uint8, device=device)  # (halves and floats of it are NaN)
    own_gz, own_gx, gy_t = _nan(h * ld, device), _nan(n * d, device), _nan(d * ld, device)
    hid.fill_(float("nan"))
    into.fill_(float("nan"))
    _lib.check(lib.hffn_backward_planes(gy.data_ptr(), z.data_ptr(), s["hid_offsets"].data_ptr(), s["hid_output"].data_ptr(),
                                        s["hid_pos"].data_ptr(), arrays["out_val"].data_ptr(), s["in_offsets"].data_ptr(),
                                        s["in_hidden"].data_ptr(), s["in_pos"].data_ptr(), arrays["up_val"].data_ptr(), hid.data_ptr(),
                                        into.data_ptr(), work.data_ptr(), need, gy_t.data_ptr(), own_gz.data_ptr(), own_gx.data_ptr(), d, h,
                                        *nnz, n, ld, _stream()), "backward on its planes")
    assert bool((work[need:] == 0x7f).all()) and torch.equal(gy_t.view(d, ld)[:, :n], gy.T)
    assert torch.equal(own_gz.view(h, ld)[:, :n], gz.view(h, ld)[:, :n]) and torch.equal(own_gx, gx)
    owner = torch.repeat_interleave(torch.arange(h, device=device), s["hid_offsets"].diff().long())
    w_down = torch.zeros(h, d, dtype=torch.float64, device=device)
    w_down[owner, s["hid_output"].long()] = arrays["out_val"][s["hid_pos"].long()].double()
    w_up = torch.zeros(h, d, dtype=torch.float64, device=device)
    w_up[torch.repeat_interleave(torch.arange(h, device=device), arrays["up_offsets"].diff().long()), arrays["up_idx"].long()] = arrays["up_val"].double()
    v = z.view(h, ld)[:, :n].T.double()
    slope = 0.5 * (1 + torch.special.erf(v / 2 ** 0.5)) + v * torch.exp(-0.5 * v * v) / (2 * torch.pi) ** 0.5
    expected = (gy.double() @ w_down.T) * slope
    assert float((gz.view(h, ld)[:, :n].T - expected).norm() / expected.norm()) <= 2e-6
    assert float((gx.view(n, d) - expected @ w_up).norm() / (expected @ w_up).norm()) <= 2e-6


def test_adamw_over_one_array_and_over_all(device):
    """hffn_adamw on each array and hffn_adamw_arrays on all: the same bits (misaligned, empty and odd-sized arrays among
    them), and the update in float64 within float32's roundings."""
    lib, counts = _lib.load(), (1027, 0, 4096, 13)
    drawn = torch.Generator(device=device).manual_seed(8)
    drawn = [[torch.randn(count + 1, generator=drawn, device=device).abs() for _ in range(4)] for count in counts]
    # the last array misaligned in both calls: its entries go one by one, which the compiler contracts in its own way
    arrays, single = ([[t.clone()[k == 3:][:count] for t in drawn[k]] for k, count in enumerate(counts)] for _ in range(2))
    scalars = (1e-5, 0.9, 0.1, 0.999, 0.001, 2e-3, 0.8, 1e-8)
    pointers = [(_lib.ctypes.c_void_p * 4)(*(four[i].data_ptr() for four in arrays)) for i in range(4)]
    start = [[t.double() for t in four] for four in arrays]
    _lib.check(lib.hffn_adamw_arrays(4, *pointers, (_lib.ctypes.c_uint32 * 4)(*counts), *scalars, _stream()), "adamw")
    for four, count in zip(single, counts):
        _lib.check(lib.hffn_adamw(*(t.data_ptr() for t in four), count, *scalars, _stream()), "adamw of one")
    for all_four, own, (p, g, m, v) in zip(arrays, single, start):
        for a, b in zip(all_four, own):
            assert torch.equal(a, b)
        m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
        p = p - 1e-5 * p
        p = p - 2e-3 * m / (v.sqrt() / 0.8 + 1e-8)
        for a, b in zip(all_four, (p, g, m, v)):
            torch.testing.assert_close(a.double(), b, rtol=1e-6, atol=1e-6)
