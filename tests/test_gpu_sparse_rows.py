# SPDX-License-Identifier: MIT
"""Rows with few finite entries (logits masked by a grammar, or a top-k or top-p
filter; vocabularies shorter than a shortlist) in the row passes that keep
shortlists: the CPU oracle's bits, and no row read in full by the select pass.
Every finite entry is listed, so nothing is left out that a bound would have
to cover."""

import ctypes as C

import numpy as np
import pytest

from tests.cases import first_difference, to_bits

pytestmark = pytest.mark.gpu

STREAM, SHORT, ONE_READ, AUTO = 7, 8, 3, -1


def _rescans(hip, oracle, x, dtype, kind, overlap=-1, offset=0, **kw):
    """Checks a decode against the oracle; returns the rows it read in full."""
    xin = to_bits(x, dtype)
    want = oracle.decode(xin, dtype=dtype, **kw)
    prev = hip.lib.dbs_hip_set_row_pass(kind), hip.lib.dbs_hip_set_decode_overlap(overlap)
    try:
        hip.lib.dbs_hip_profile_enable(1)  # clears the counters
        got = hip.decode(xin, dtype, x_offset=offset, **kw)
        ms, n = C.c_double(), C.c_int64()
        assert hip.lib.dbs_hip_profile_read(5, C.byref(ms), C.byref(n)) == 0
    finally:
        hip.lib.dbs_hip_profile_enable(0)
        hip.lib.dbs_hip_set_row_pass(prev[0])
        hip.lib.dbs_hip_set_decode_overlap(prev[1])
    assert first_difference(got, want) is None, first_difference(got, want)
    return n.value


def _sparse(seed, shape, finite):
    """Rows with `finite` entries each, the others -inf."""
    rng = np.random.default_rng(seed)
    x = np.full(shape, -np.inf, np.float32)
    flat = x.reshape(-1, shape[-1])
    for row in flat:
        at = rng.choice(shape[-1], size=finite, replace=False)
        row[at] = rng.normal(-3.0, 2.0, size=finite)
    return x


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("logits", [False, True])
@pytest.mark.parametrize("kind,V", [(STREAM, 12301), (STREAM, 4097), (SHORT, 2001), (SHORT, 6144), (ONE_READ, 2048),
                                    (ONE_READ, 40957), (AUTO, 50257)])
def test_few_finite_entries(hip, oracle, kind, V, logits, dtype):
    if kind == ONE_READ and logits:
        pytest.skip("the one-read pass takes log-probs")
    for finite in (0, 1, 3, 10, 20):
        x = _sparse(finite, (3, 5, 4, V), finite)
        kw = dict(from_logits=logits, eos_token=7, min_length=2, alpha=0.6, steps=[5, 1, 3])
        assert _rescans(hip, oracle, x, dtype, kind, offset=finite % 3, **kw) == 0, finite
        assert _rescans(hip, oracle, x, dtype, kind, overlap=1, **kw) == 0, finite


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("K", [1, 8, 20, 70])
def test_around_the_list_length(hip, oracle, K, dtype):
    """As many finite entries as a list holds, one less and one more, the type's
    lowest value among them."""
    M = (K + 16 + 7) // 8 * 8 if K <= 64 else 80
    lowest = {"f32": np.finfo(np.float32).min, "f16": -65504.0, "bf16": np.float32(-3.3895314e38)}[dtype]
    for logits in (False, True):
        for finite in (M - 1, M, M + 1):
            x = _sparse(K + finite, (2, 3, K, 5003), finite)
            flat = x.reshape(-1, x.shape[-1])
            for row in flat[::2]:
                row[np.flatnonzero(row > -np.inf)[finite // 2]] = lowest
            _rescans(hip, oracle, x, dtype, STREAM, from_logits=logits, alpha=0.6)
            _rescans(hip, oracle, x, dtype, SHORT, from_logits=logits, alpha=0.6)
            if not logits:
                _rescans(hip, oracle, x, dtype, ONE_READ, alpha=0.6)


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("logits", [False, True])
@pytest.mark.parametrize("V", [1, 2, 9, 23])
def test_vocabularies_shorter_than_a_list(hip, oracle, V, logits, dtype):
    rng = np.random.default_rng(V)
    x = rng.normal(0.0, 2.0, size=(4, 6, 3, V)).astype(np.float32)
    for kind in (AUTO, STREAM, SHORT):
        assert _rescans(hip, oracle, x, dtype, kind, from_logits=logits, eos_token=V - 1, alpha=0.6) == 0


def test_rows_filled_with_the_lowest_value(hip, oracle):
    """Masked by the type's lowest finite value, as many libraries do: such
    rows hold more entries at the threshold than a list, and are read in full."""
    for dtype, lowest in (("f32", np.finfo(np.float32).min), ("f16", -65504.0), ("bf16", np.float32(-3.3895314e38))):
        for logits in (False, True):
            x = _sparse(5, (2, 4, 3, 3001), 10)
            x[np.isinf(x)] = lowest
            for kind in (AUTO, STREAM, SHORT):
                _rescans(hip, oracle, x, dtype, kind, from_logits=logits, alpha=0.6)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("K", [3, 12, 17, 64, 80, 257])
def test_sums_that_overflow(hip, oracle, K, dtype):
    """Fewer candidates than beams, some of them sums below the lowest value:
    such a sum is no candidate."""
    lowest = np.finfo(np.float32).min if dtype == "f32" else np.float32(-3.3895314e38)
    rng = np.random.default_rng(K)
    for V in (5, 23):
        x = rng.normal(0.0, 1.0, size=(2, 5, K, V)).astype(np.float32)
        x[rng.random(x.shape) < 0.7] = lowest
        for logits in (False, True):
            for overlap in (0, 1):
                _rescans(hip, oracle, x, dtype, AUTO, overlap=overlap, from_logits=logits, alpha=0.6, steps=[5, 2])


@pytest.mark.parametrize("alpha", [0.0, 0.6])
@pytest.mark.parametrize("K", [8, 20, 64, 70])
def test_full_reads_at_the_threshold(hip, oracle, monkeypatch, K, alpha):
    """Every row read in full, with very many entries of the threshold's score:
    rows of one value, of a few, masked with the lowest value; thresholds from
    rows before and after the row read, and from finished beams."""
    monkeypatch.setenv("DBS_HIP_SHORTLIST", "0")
    rng = np.random.default_rng(K)
    V = 4001
    for rows in ("constant", "coarse", "lowest"):
        x = np.zeros((2, 4, K, V), np.float32)
        if rows == "coarse":
            x = np.round(rng.normal(0.0, 1.0, size=x.shape)).astype(np.float32)
        if rows == "lowest":
            x = _sparse(K, x.shape, 12)
            x[np.isinf(x)] = np.finfo(np.float32).min
        x[..., 9] += 3.0  # beams finish
        for kw in (dict(eos_token=-1), dict(eos_token=9, min_length=2), dict(eos_token=9, repetition_penalty=1.3)):
            for logits in (False, True):
                _rescans(hip, oracle, x, "f32", AUTO, from_logits=logits, alpha=alpha, **kw)
