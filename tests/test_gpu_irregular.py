"""Tokens and weights that the fp16 planes of a call cannot hold (infinities, NaN, magnitudes beyond the clamp of a plane's
power of two, tokens of only tiny entries) on calls of the policy that densify planes: they are the lane-per-token kernels'
results (the same bits, float32 in stored slot order), and the other tokens keep theirs. Inputs with outlier columns are
held to the float64 oracle."""
from __future__ import annotations

import functools
import math

import numpy as np
import pytest
import torch

from hffn_amd import synth
from hffn_amd.ffn import hip_layer
from hffn_amd.runtime import HFFNRuntime
from oracle import reference

pytestmark = pytest.mark.gpu
WIDE = {w.name: w for w in (synth.Workload("wide", 2048, 1024, 205, 7), synth.Workload("wide_bf16", 2048, 1024, 205, 7, value_dtype="bf16"))}
# a split down GEMM and its reduction; one split on row tiles of 64, 128 and 256 (y written by the GEMM); bfloat16
SHAPES = [("pythia70m_d20", 128), ("pythia70m_d20", 300), ("pythia70m_d20", 3000), ("pythia70m_d20", 6000), ("pythia1p4b_d20_bf16", 300),
          ("wide", 2560), ("wide_bf16", 2560)]
IDS = [f"{name}_{n}" for name, n in SHAPES]


@functools.lru_cache(maxsize=None)
def _compact(name):
    return synth.make_workload_layer(WIDE.get(name, name))


def _pair(name, device):
    """A runtime whose policy densifies planes for the call, and one forced to the lane-per-token kernels, on the same
    arrays (a store of its own per test: some change it)."""
    layer = hip_layer(_compact(name))
    policy, rows = HFFNRuntime([layer], device), HFFNRuntime([layer], device)
    rows.force("rows", "rows")
    return policy, rows


def _input(n, d, device):
    return torch.randn((n, d), generator=torch.Generator(device=device).manual_seed(n), device=device)


def _same(a, b):
    return torch.equal(a.isnan(), b.isnan()) and torch.equal(torch.nan_to_num(a, nan=0.0), torch.nan_to_num(b, nan=0.0))


@pytest.mark.parametrize("name,n", SHAPES, ids=IDS)
def test_irregular_tokens(name, n, device):
    policy, rows = _pair(name, device)
    x = _input(n, policy.d_model, device)
    clean = policy.forward(0, x).clone()
    assert policy.transient(n)
    x[1, 3] = float("inf")
    x[2, 5], x[2, 9] = float("-inf"), float("inf")
    x[n // 2, 7] = float("nan")
    x[n - 2, 1] = 3e38     # finite: 2^127.8
    x[n - 3, 0] = -2.0 ** 105
    x[n - 1] *= 2.0 ** -120
    odd = [1, 2, n // 2, n - 3, n - 2, n - 1]
    y, expected = policy.forward(0, x).clone(), rows.forward(0, x).clone()
    assert _same(y[odd], expected[odd])
    others = torch.ones(n, dtype=torch.bool, device=device)
    others[odd] = False
    assert torch.equal(y[others], clean[others])


@pytest.mark.parametrize("name,n", SHAPES, ids=IDS)
@pytest.mark.parametrize("side", ["up_val", "out_val"])
@pytest.mark.parametrize("value", [float("inf"), float("nan"), 2.0 ** 110], ids=["inf", "nan", "large"])
def test_irregular_weights(name, n, side, value, device):
    policy, rows = _pair(name, device)
    x = _input(n, policy.d_model, device)
    values = policy._tensors[0][side]
    assert values.data_ptr() == rows._tensors[0][side].data_ptr()
    values[values.numel() // 2] = value
    y, expected = policy.forward(0, x), rows.forward(0, x)
    assert policy.transient(n)
    if side == "up_val" or not math.isfinite(value):  # a whole token; or the outputs of that weight
        odd = ~expected.isfinite() if side == "out_val" else torch.ones_like(expected, dtype=torch.bool)
        assert int(odd.sum()) and _same(y[odd], expected[odd])
    regular = expected.isfinite()
    assert torch.equal(y.isfinite(), regular)
    torch.testing.assert_close(y[regular], expected[regular], rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("name,n", [("pythia70m_d20", 128), ("pythia70m_d20", 3000), ("pythia1p4b_d20_bf16", 300)])
def test_irregular_tokens_of_a_call_on_its_own_output(name, n, device):
    """x may be (a part of) the output of the call before, which the call overwrites: the results of a call on a copy."""
    policy, rows = _pair(name, device)
    x = _input(n + 7, policy.d_model, device)
    for skip in (0, 7):
        policy.forward(0, x)
        own = policy._y[skip:skip + n]
        own[1, 3], own[n // 2, 7], own[n - 2, 1] = float("inf"), float("nan"), 3e38
        copy = own.clone()
        y = policy.forward(0, own).clone()
        assert policy.transient(n) and own.data_ptr() == policy._y.data_ptr() + 4 * skip * policy.d_model
        assert _same(y, policy.forward(0, copy))
        odd = [1, n // 2, n - 2]
        assert _same(y[odd], rows.forward(0, copy)[odd])


def test_activations_beyond_the_planes(device):
    """A pre-activation whose GELU is not finite from finite operands: only the outputs that read that neuron are lost."""
    policy, rows = _pair("pythia70m_d20", device)
    n = 128
    x = _input(n, policy.d_model, device)
    tensors = policy._tensors[0]
    tensors["up_val"][0] = 2.0 ** 20
    x[5] = 0.0
    x[5, int(tensors["up_idx"][0])] = 2.0 ** 60
    y, expected = policy.forward(0, x).clone(), rows.forward(0, x).clone()
    finite = int(expected[5].isfinite().sum())
    assert 0 < finite < policy.d_model and _same(y[5], expected[5]), finite
    assert bool(y[6:].isfinite().all())


@pytest.mark.parametrize("name,n", [("pythia70m_d20", 128), ("pythia1p4b_d20_bf16", 300)], ids=["70m", "1p4b"])
@pytest.mark.parametrize("scale", [1e2, 1e4])
def test_outlier_columns(name, n, scale, device):
    """A few input columns of large magnitude in every token, as deep transformer layers have them. Every operand of the
    planes is hi + lo of at least 21 bits down to 2^-15 of its row's largest, so the relative error keeps its bound of 6e-7
    (2-norm; sums in chains of at most 24 products and at most 32 chains), and is no worse than the lane-per-token kernels'."""
    policy, rows = _pair(name, device)
    layer = _compact(name)
    x = _input(n, policy.d_model, device)
    x[:, [3, 101]] *= scale
    weights = reference.dense_weights(layer)
    expected = reference.forward_dense(layer, x.cpu().numpy(), weights)
    error = {label: np.abs(runtime.forward(0, x).double().cpu().numpy() - expected) for label, runtime in (("planes", policy), ("rows", rows))}
    assert policy.transient(n)
    print(name, scale, {label: (float(np.linalg.norm(e) / np.linalg.norm(expected)), float(e.max() / expected.std())) for label, e in error.items()})
    assert np.linalg.norm(error["planes"]) <= 6e-7 * np.linalg.norm(expected)
    assert np.linalg.norm(error["planes"]) <= np.linalg.norm(error["rows"])
