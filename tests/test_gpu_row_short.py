# SPDX-License-Identifier: MIT
"""The row pass of short rows (one wavefront a row, row-pass kind 8) against the
CPU oracle bit for bit: lengths around each register count and the last it
takes, every type, logits and log-probs, unaligned starts, masks, rows with
NaN, +inf or nothing finite, and more survivors than its list holds."""

import numpy as np
import pytest

from tests.cases import first_difference, to_bits

pytestmark = pytest.mark.gpu


def _check(hip, oracle, x, dtype, kind=8, overlap=-1, offset=0, **kw):
    want = oracle.decode(x, dtype=dtype, **kw)
    hip.lib.dbs_hip_set_row_pass(kind)
    hip.lib.dbs_hip_set_decode_overlap(overlap)
    try:
        got = hip.decode(x, dtype, x_offset=offset, **kw)
    finally:
        hip.lib.dbs_hip_set_row_pass(-1)
        hip.lib.dbs_hip_set_decode_overlap(-1)
    assert first_difference(got, want) is None, first_difference(got, want)


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("logits", [False, True])
@pytest.mark.parametrize("V", [1, 63, 64, 65, 257, 512, 513, 1023, 1025, 2047, 2049, 3073, 4095, 4096, 4097, 6144, 6145])
def test_lengths(hip, oracle, dtype, logits, V):
    rng = np.random.default_rng(V)
    x = to_bits(rng.normal(0.0, 3.0, size=(3, 5, 4, V)).astype(np.float32), dtype)
    kw = dict(from_logits=logits, eos_token=V // 2, min_length=2, alpha=0.6, steps=[5, 1, 4])
    for offset in (0, 1):
        _check(hip, oracle, x, dtype, offset=offset, **kw)
    _check(hip, oracle, x, dtype, overlap=1, **kw)


@pytest.mark.parametrize("logits", [False, True])
def test_values(hip, oracle, logits):
    rng = np.random.default_rng(3)
    x = rng.normal(0.0, 2.0, size=(6, 4, 5, 700)).astype(np.float32)
    x[1, 1, 2, 5] = np.nan
    x[2, 0, 0, 699] = np.inf
    x[3, 2] = -np.inf
    x[4] = np.float32(0.25)  # every entry ties: no list holds them
    x[5][rng.random(x[5].shape) < 0.97] = -np.inf
    banned = (rng.random((700,)) < 0.3).astype(np.uint8)
    for dtype in ("f32", "bf16"):
        _check(hip, oracle, to_bits(x, dtype), dtype, from_logits=logits, eos_token=9, min_length=3, alpha=0.6,
               banned=banned)


@pytest.mark.parametrize("K", [1, 8, 33, 64, 70])
def test_beams(hip, oracle, K):
    """Lists of 24 to 80 entries out of 256 lane maxima, the automatic choice."""
    rng = np.random.default_rng(K)
    x = to_bits(rng.normal(0.0, 1.0, size=(2, 4, K, 1500)).astype(np.float32), "f16")
    for logits in (False, True):
        _check(hip, oracle, x, "f16", kind=-1, from_logits=logits, eos_token=2, alpha=1.0)
