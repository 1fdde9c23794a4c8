# SPDX-License-Identifier: MIT
"""The one-wavefront select pass of up to eight beams (candidates in a grid of
lanes) against the CPU oracle bit for bit: every beam count to the first one
past the grid, step counts around the distance its words are loaded ahead,
beams that finish (ranked by score across lengths) until all have, dead beams
(fewer candidates than beams), ties, steps whose rows are read in full (short
shortlists), per-example beams, and the decode beside its row pass."""

import numpy as np
import pytest

from tests.cases import first_difference, log_softmax, to_bits

pytestmark = pytest.mark.gpu


def _check(hip, oracle, x, dtype, overlap=-1, **kw):
    xin = to_bits(x, dtype)
    beams = kw.pop("beams", None)
    want = (oracle.decode(xin, dtype=dtype, **kw) if beams is None
            else oracle.decode_per_example(xin, dtype=dtype, beams=beams, **kw))
    hip.lib.dbs_hip_set_decode_overlap(overlap)
    try:
        got = hip.decode(xin, dtype, beams=beams, **kw)
    finally:
        hip.lib.dbs_hip_set_decode_overlap(-1)
    assert first_difference(got, want) is None, first_difference(got, want)


@pytest.mark.parametrize("overlap", [0, 1])
@pytest.mark.parametrize("K", range(1, 10))
def test_grid_beams(hip, oracle, K, overlap):
    rng = np.random.default_rng(K)
    B, T, V = 6, 13, 600
    x = rng.normal(0.0, 2.0, size=(B, T, K, V)).astype(np.float32)
    x[..., 5] += 5.0  # beams finish at every step
    _check(hip, oracle, log_softmax(x), "f32", overlap, eos_token=5, extra_eos=[9], min_length=2, alpha=0.6,
           steps=[13, 1, 4, 5, 8, 12])
    _check(hip, oracle, x, "bf16", overlap, from_logits=True, eos_token=-1, alpha=1.0)


@pytest.mark.parametrize("K", [1, 3, 8])
@pytest.mark.parametrize("V", [1, 2, 3, 9])
def test_grid_dead_beams(hip, oracle, K, V):
    rng = np.random.default_rng(10 * K + V)
    x = log_softmax(rng.normal(0.0, 1.0, size=(3, 6, K, V)).astype(np.float32))
    x[rng.random(x.shape) < 0.2] = -np.inf
    _check(hip, oracle, x, "f32", eos_token=V - 1, alpha=0.6)
    _check(hip, oracle, x, "f32", eos_token=-1, alpha=0.0)


@pytest.mark.parametrize("K", [2, 5, 8])
@pytest.mark.parametrize("shortlist", ["0", "1", "3", "8", "9"])
def test_grid_full_reads(hip, oracle, monkeypatch, K, shortlist):
    """Lists shorter than the beams take the general step, lists just longer
    fail the exactness check now and then."""
    monkeypatch.setenv("DBS_HIP_SHORTLIST", shortlist)
    rng = np.random.default_rng(100 + K)
    x = rng.normal(0.0, 1.0, size=(4, 7, K, 300)).astype(np.float32)
    x[..., 3] += 2.5
    x = log_softmax(x)
    x[rng.random(x.shape) < 0.4] = np.float32(-6.0)  # ties at the lists' ends
    for overlap in (0, 1):
        _check(hip, oracle, x, "f32", overlap, eos_token=3, alpha=0.6)


def test_grid_per_example_beams(hip, oracle):
    rng = np.random.default_rng(7)
    x = log_softmax(rng.normal(0.0, 2.0, size=(5, 9, 7, 257)).astype(np.float32))
    _check(hip, oracle, x, "f32", eos_token=8, alpha=0.6, beams=[7, 1, 3, 6, 2])
