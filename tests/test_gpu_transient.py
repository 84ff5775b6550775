"""Calls on planes densified for the call (``hffn_forward_prefill``, the policy's ``transient`` calls above 64 tokens)
against the float64 oracle: widths that are and are not multiples of 256, both value types, neurons without slots,
rows longer than the densify kernel holds in registers, the edges of its token tiles (64, 128, 256), a call of several
pieces, arrays off their 16-byte boundaries, and the planned and captured forms of the call.

Tolerance: a relative error (2-norm) of 6e-7. Every operand is hi + lo in fp16 (2^-23 of the entry at most), the sums run
in chains of at most 24 products and at most 32 chains, each rounded to float32: about sqrt(24 + 32) 2^-24 = 4.5e-7
per projection at worst, 2e-7 measured for both."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from hffn_amd import _lib, synth
from hffn_amd.ffn import hip_layer
from hffn_amd.prepared_runtime import PreparedRuntime
from hffn_amd.runtime import HFFNLayer, HFFNRuntime
from hffn_amd.train_runtime import HFFNTrainRuntime
from oracle import reference

pytestmark = pytest.mark.gpu
RELATIVE = 6e-7


def _side(rng, h, d, density, full):
    degrees = rng.integers(0, max(2, int(2 * density * d)), h)
    degrees[::11] = 0
    degrees[full] = d  # neurons of every slot: one output (down) or neuron (up) row of full length
    offsets = np.zeros(h + 1, np.int32)
    offsets[1:] = np.cumsum(degrees)
    index = np.concatenate([np.sort(rng.choice(d, k, replace=False)) for k in degrees] or [[]]).astype(np.int16)
    return offsets, index, (rng.standard_normal(index.size) * 0.02).astype(np.float32)


def _layer(d, h, density, bf16, seed=3):
    rng = np.random.default_rng([seed, d, h])
    up, down = _side(rng, h, d, density, [1]), _side(rng, h, d, density, [2, h - 1])
    if bf16:  # values the bfloat16 store holds exactly
        up, down = ((o, i, torch.from_numpy(v).bfloat16().float().numpy()) for o, i, v in (up, down))
    b_up, b_down = ((rng.standard_normal(k) * 0.01).astype(np.float32) for k in (h, d))
    return synth.CompactLayer(d, h, synth._groups(h), *up, b_up, *down, b_down)


def _device_layer(layer, bf16, device):
    t = lambda a: torch.from_numpy(a).to(device)  # noqa: E731
    value = lambda a: t(a).bfloat16() if bf16 else t(a)  # noqa: E731
    return HFFNLayer.from_hidden_major(layer.d_model, layer.d_ff, t(layer.b_up), t(layer.up_offsets), t(layer.up_idx),
                                       value(layer.up_val), t(layer.b_down), t(layer.down_offsets), t(layer.down_idx),
                                       value(layer.down_val))


def _prefill(runtime, x, shift=0):
    """hffn_forward_prefill on a workspace of NaNs, guard words behind y and the workspace; ``shift``: slots by which
    copies of the index and value arrays start off their boundaries."""
    lib, n = _lib.load(), x.shape[0]
    tensors, keep = runtime._tensors[0], []

    def at(name):
        tensor = tensors[name]
        if shift and name in ("up_idx", "up_val", "out_hidden", "out_val"):
            moved = torch.zeros(tensor.numel() + shift, dtype=tensor.dtype, device=x.device)
            moved[shift:] = tensor
            keep.append(moved)
            tensor = moved[shift:]
        return tensor.data_ptr()

    need = _lib.query_bytes(lib.hffn_prefill_workspace, runtime._args[0][0], n, runtime.d_model, runtime.d_ff)
    work = torch.full((need // 4 + 64,), float("nan"), device=x.device)
    y = torch.full((n + 1, runtime.d_model), -7.0, device=x.device)
    arrays = [at(name) for name in ("up_offsets", "up_idx", "up_val", "b_up", "out_offsets", "out_hidden", "out_val", "b_down")]
    _lib.check(lib.hffn_forward_prefill(runtime._args[0][0], x.data_ptr(), *arrays, work.data_ptr(), need, y.data_ptr(),
                                        runtime.d_model, runtime.d_ff, n, torch.cuda.current_stream().cuda_stream), "prefill")
    torch.cuda.synchronize()
    assert bool((y[n] == -7.0).all()) and bool(torch.isnan(work[need // 4:]).all())
    return y[:n]


def _relative(y, expected):
    return float(np.linalg.norm(y.double().cpu().numpy() - expected) / np.linalg.norm(expected))


@pytest.mark.parametrize("d,h,density,bf16,tokens", [
    (16, 8, 0.5, False, (1, 65)), (256, 1024, 0.2, False, (65, 129, 16384 + 70)), (400, 1608, 0.3, False, (64, 128, 257)),
    (400, 1608, 0.3, True, (65, 300)), (768, 3072, 0.05, False, (128, 512)), (1104, 4424, 0.2, True, (70, 256, 513)),
    (272, 9000, 0.1, False, (100,)), (2048, 8192, 0.1, True, (1030,))])
def test_prefill_matches_the_oracle(d, h, density, bf16, tokens, device):
    layer = _layer(d, h, density, bf16)
    runtime = HFFNRuntime([_device_layer(layer, bf16, device)], device, dense=False)
    weights = reference.dense_weights(layer)
    for n in tokens:
        x = np.random.default_rng([5, n]).standard_normal((n, d)).astype(np.float32)
        x[n // 2] *= 1e-3  # tokens of other scales, and one of zeros
        x[-1] = 0.0
        expected = reference.forward_dense(layer, x, weights)
        xd = torch.from_numpy(x).to(device)
        y = _prefill(runtime, xd)
        assert _relative(y, expected) <= RELATIVE, n
        if n <= 300:
            assert torch.equal(_prefill(runtime, xd, shift=3), y), n  # off the boundaries: the same planes, the same bits


def test_policy_plans_and_capture(device):
    """An unforced call above 64 tokens takes the planes of the call where estimated faster, eager, prepared and
    captured with the same bits; forced pairs, dense=False and unsorted rows keep the compact store's kernels."""
    d, h, n = 400, 1608, 300
    layer = _layer(d, h, 0.3, False)
    compact = hip_layer(layer)
    runtime, prepared = HFFNRuntime([compact], device), PreparedRuntime([compact], device)
    x = torch.from_numpy(np.random.default_rng(9).standard_normal((n, d)).astype(np.float32)).to(device)
    y = runtime.forward(0, x).clone()
    assert runtime.transient(n) and not runtime.transient(64) and sum(runtime.calls.values()) == 1
    assert torch.equal(y, _prefill(runtime, x)) and torch.equal(prepared.forward(0, x), y) and torch.equal(prepared.forward(0, x), y)
    assert _relative(y, reference.forward(layer, x.cpu().numpy())) <= RELATIVE
    graph, out = torch.cuda.CUDAGraph(), torch.empty_like(y)
    with torch.cuda.graph(graph):
        out.copy_(runtime.forward(0, x))
    for k in range(3):
        x.mul_(0.5)
        expected = prepared.forward(0, x).clone()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, expected), k
    small = x[:70].contiguous()
    runtime.force("rows", "rows")
    assert not runtime.transient(n)
    rows = runtime.forward(0, small).clone()
    runtime.force(None, None)
    assert float((runtime.forward(0, small) - rows).abs().max()) <= 1e-5
    never = HFFNRuntime([compact], device, dense=False)
    never.forward(0, x)
    assert not never.transient(n) and never._prefill_work is None


@pytest.mark.parametrize("d,h,density,tokens", [(256, 1024, 0.2, 600), (768, 3072, 0.1, 100), (2048, 8192, 0.1, 1100)])
@pytest.mark.parametrize("first", [False, True], ids=["float32_first", "bf16_first"])
def test_layers_of_both_value_types(d, h, density, tokens, first, device):
    """A runtime of a bfloat16 and a float32 layer: the workspaces hold either layer's calls (above and below 64 tokens),
    whichever comes first."""
    compact = {bf16: _layer(d, h, density, bf16) for bf16 in (False, True)}
    order = [first, not first]
    runtime = HFFNRuntime([_device_layer(compact[bf16], bf16, device) for bf16 in order], device)
    for n in (tokens, 48):
        x = np.random.default_rng(n).standard_normal((n, d)).astype(np.float32)
        for index, bf16 in enumerate(order):
            expected = reference.forward_dense(compact[bf16], x, reference.dense_weights(compact[bf16]))
            assert _relative(runtime.forward(index, torch.from_numpy(x).to(device)), expected) <= 1e-6, (n, bf16)


def _even_layer(d, h, slots):
    rng = np.random.default_rng([slots, d, h])
    offsets = np.arange(0, (h + 1) * slots, slots, dtype=np.int32)
    sides = [(offsets, np.concatenate([np.sort(rng.choice(d, slots, replace=False)) for _ in range(h)]).astype(np.int16),
              (rng.standard_normal(h * slots) * 0.02).astype(np.float32)) for _ in range(2)]
    b_up, b_down = ((rng.standard_normal(k) * 0.01).astype(np.float32) for k in (h, d))
    return synth.CompactLayer(d, h, synth._groups(h), *sides[0], b_up, *sides[1], b_down)


def test_results_do_not_depend_on_earlier_calls(device):
    """The same input gives the same bits whatever larger call came before (counts on either side of a step of the
    estimates), with HFFNRuntime and PreparedRuntime; a training runtime holds no prefill workspace until a call needs it."""
    layer = hip_layer(_even_layer(512, 2048, 26))
    policy = HFFNRuntime([layer], device)
    below = next(n for n in range(700, 2100) if policy.transient(n) and not policy.transient(n + 1))
    counts = (100, below, below + 1)
    inputs = {n: torch.from_numpy(np.random.default_rng(n).standard_normal((n, 512)).astype(np.float32)).to(device) for n in counts}
    alone = {n: HFFNRuntime([layer], device).forward(0, inputs[n]).clone() for n in counts}
    for kind in (HFFNRuntime, PreparedRuntime):
        runtime = kind([layer], device)
        for n in (*counts, below, 100):
            assert torch.equal(runtime.forward(0, inputs[n]), alone[n]), (kind, n)
    runtime = HFFNRuntime([layer], device)
    HFFNTrainRuntime(runtime, max_tokens=below).reserve(below)
    assert runtime._prefill_work is None
    assert torch.equal(runtime.forward(0, inputs[below]), alone[below]) and runtime._prefill_work is not None


def test_path_and_calls_name_what_runs(device):
    """``path`` and ``calls`` name the planes of the call where they run, ``modes`` otherwise: the small and the large
    workload layers, forced pairs, prepared calls."""
    for name, counts in (("pythia70m_d20", (64, 65, 128, 2048)), ("pythia1p4b_d20_bf16", (64, 65, 300, 2048))):
        layer = hip_layer(synth.make_workload_layer(name))
        for kind in (HFFNRuntime, PreparedRuntime):
            runtime = kind([layer], device)
            for n in counts:
                x = torch.randn(n, runtime.d_model, device=device)
                expected = ("prefill", "prefill") if runtime.transient(n) else runtime.modes(n)
                runtime.calls.clear()
                runtime.forward(0, x)
                assert runtime.path(n) == expected and dict(runtime.calls) == {expected: 1}, (name, n)
            assert runtime.path(counts[-1]) == ("prefill", "prefill") and runtime.path(64) == ("tiles", "tiles")
            runtime.force("rows", "rows")
            runtime.calls.clear()
            runtime.forward(0, x)
            assert runtime.path(counts[-1]) == ("rows", "rows") and dict(runtime.calls) == {("rows", "rows"): 1}


def test_bench_times_the_path_that_runs(device):
    """bench.py's kernel record of a call on planes of the call is that call, not the compact store's kernels."""
    import bench
    runtime = HFFNRuntime([hip_layer(_layer(400, 1608, 0.3, False))], device)
    x = torch.randn(300, 400, device=device)
    runtime.forward(0, x)
    runtime.calls.clear()
    assert runtime.transient(300) and list(bench.time_kernels(runtime, x, 3, 1)) == ["prefill"]


def test_prefill_refusals(device):
    lib, size = _lib.load(), ctypes.c_uint64(0)
    p, odd = 256, 264  # never dereferenced: the calls are refused before any launch
    assert lib.hffn_prefill_workspace(0, 100, 400, 1608, ctypes.byref(size)) == _lib.OK
    for arguments, message in (((0, odd, *[p] * 9, size.value, p, 400, 1608, 100), "aligned"),
                               ((0, *[p] * 9, odd, size.value, p, 400, 1608, 100), "aligned"),
                               ((0, *[p] * 10, size.value - 1, p, 400, 1608, 100), "workspace"),
                               ((0, *[p] * 10, size.value, p, 400, 1604, 100), "multiple of 8"),
                               ((0, *[p] * 10, size.value, p, 408, 1608, 100), "multiple of 16"),
                               ((7, *[p] * 10, size.value, p, 400, 1608, 100), "value type"),
                               ((0, *[p] * 5, None, *[p] * 4, size.value, p, 400, 1608, 100), "null")):
        assert lib.hffn_forward_prefill(*arguments, None) == -1 and message in lib.hffn_last_error().decode(), message
