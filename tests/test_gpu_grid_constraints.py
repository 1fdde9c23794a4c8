# SPDX-License-Identifier: MIT
"""Constrained decodes of up to eight beams through the one-wavefront select
pass's grid of candidates, against the CPU oracle bit for bit: every beam
count to the first past the grid, n-grams of every length its hash treats
apart, prefixes around one wavefront's lookup (64 tokens), rows whose beams
repeat and block most tokens, rows whose best candidates lie past the entries
held, beams that finish, and short lists."""

import numpy as np
import pytest

from tests.cases import first_difference, log_softmax, to_bits

pytestmark = pytest.mark.gpu


def _check(hip, oracle, x, dtype, overlap=-1, **kw):
    xin = to_bits(x, dtype)
    want = oracle.decode(xin, dtype=dtype, **kw)
    hip.lib.dbs_hip_set_decode_overlap(overlap)
    try:
        got = hip.decode(xin, dtype, **kw)
    finally:
        hip.lib.dbs_hip_set_decode_overlap(-1)
    assert first_difference(got, want) is None, first_difference(got, want)


@pytest.mark.parametrize("overlap", [0, 1])
@pytest.mark.parametrize("ngram,rep", [(0, 1.3), (2, 1.0), (3, 1.2), (6, 1.05)])
@pytest.mark.parametrize("K", range(1, 10))
def test_constrained_beams(hip, oracle, K, ngram, rep, overlap):
    rng = np.random.default_rng(10 * K + ngram)
    B, T, V = 4, 21, 40
    x = log_softmax(rng.normal(0.0, 1.5, size=(B, T, K, V)).astype(np.float32))
    kw = dict(no_repeat_ngram_size=ngram, repetition_penalty=rep, min_length=2, alpha=0.6)
    _check(hip, oracle, x, "f32", overlap, eos_token=5, extra_eos=[9], steps=[21, 1, 2, 20], **kw)
    _check(hip, oracle, x * 3, "bf16", overlap, from_logits=True, eos_token=-1, **kw)


@pytest.mark.parametrize("T", [63, 64, 65, 66, 130])
@pytest.mark.parametrize("ngram,rep", [(2, 1.5), (4, 1.1)])
def test_constrained_long_prefixes(hip, oracle, T, ngram, rep):
    rng = np.random.default_rng(T)
    x = rng.normal(0.0, 0.4, size=(2, T, 5, 30)).astype(np.float32)
    x += rng.normal(0.0, 2.0, size=(1, 1, 1, 30)).astype(np.float32)  # the same tokens at every step
    _check(hip, oracle, log_softmax(x), "f32", no_repeat_ngram_size=ngram, repetition_penalty=rep, eos_token=3,
           alpha=1.0)


@pytest.mark.parametrize("V", [2, 7, 25, 300])
@pytest.mark.parametrize("K", [1, 4, 8])
def test_constrained_past_the_held_entries(hip, oracle, K, V):
    """A penalty larger than the differences within a row: its best candidates
    lie anywhere; rows of two tokens block every one."""
    rng = np.random.default_rng(V + K)
    x = log_softmax(rng.normal(0.0, 0.02, size=(3, 30, K, V)).astype(np.float32))
    x[rng.random(x.shape) < 0.1] = -np.inf
    _check(hip, oracle, x, "f32", no_repeat_ngram_size=2, repetition_penalty=20.0, eos_token=-1, alpha=0.6)
    _check(hip, oracle, x, "f16", no_repeat_ngram_size=0, repetition_penalty=3.0, eos_token=V - 1, alpha=0.0)


@pytest.mark.parametrize("shortlist", ["0", "1", "5", "8", "13"])
def test_constrained_full_reads(hip, oracle, monkeypatch, shortlist):
    monkeypatch.setenv("DBS_HIP_SHORTLIST", shortlist)
    rng = np.random.default_rng(5)
    x = log_softmax(rng.normal(0.0, 1.0, size=(4, 12, 5, 300)).astype(np.float32))
    x[rng.random(x.shape) < 0.4] = np.float32(-6.0)  # ties at the lists' ends
    for overlap in (0, 1):
        _check(hip, oracle, x, "f32", overlap, no_repeat_ngram_size=2, repetition_penalty=1.2, eos_token=3, alpha=0.6)
