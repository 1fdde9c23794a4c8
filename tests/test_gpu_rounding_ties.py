# SPDX-License-Identifier: MIT
"""Log-probs that differ and give one raw score, against the CPU oracle bit for
bit. Shortlists are ordered by log-prob, candidates by (score, raw, parent,
token): where fl(p + lp), or fl(x - lse) from logits, maps several entries to
one raw score, the lowest token comes first wherever its entry stands in the
list. One beam to past the grid of lanes, the first step and later ones, ties
that end at, straddle and begin past the entries a step holds."""

import numpy as np
import pytest

from tests.cases import first_difference, to_bits

pytestmark = pytest.mark.gpu


def _check(hip, oracle, x, dtype, overlap, **kw):
    xin = to_bits(x, dtype)
    want = oracle.decode(xin, dtype=dtype, **kw)
    prev = hip.lib.dbs_hip_set_decode_overlap(overlap)
    try:
        got = hip.decode(xin, dtype, **kw)
    finally:
        hip.lib.dbs_hip_set_decode_overlap(prev)
    assert first_difference(got, want) is None, first_difference(got, want)


def _ladder(top: float, n: int, step: int = 1) -> np.ndarray:
    """n float32 values from `top` down, `step` ulps apart."""
    a = np.full(n, np.float32(top))
    for i in range(1, n):
        a[i] = a[i - 1]
        for _ in range(step):
            a[i] = np.nextafter(a[i], np.float32(-np.inf))
    return a


@pytest.mark.parametrize("overlap", [0, 1])
@pytest.mark.parametrize("alpha", [0.0, 0.6])
@pytest.mark.parametrize("K", range(1, 10))
def test_log_prob_ties(hip, oracle, K, alpha, overlap):
    """After a first step at -300, log-probs a few ulps apart, best token last."""
    B, T, V = 6, 5, 600
    rng = np.random.default_rng(K)
    x = rng.uniform(-90.0, -50.0, size=(B, T, K, V)).astype(np.float32)
    for b in range(B):
        n = [1, K, K + 1, K + 2, 2 * K + 3, 22][b]  # tied entries (a list holds 24 or 32)
        for t in range(T):
            for k in range(K):
                tokens = np.sort(rng.choice(V, size=n, replace=False))[::-1]
                top = -300.0 if t == 0 else -1.5 - (0.25 * k if b % 2 else 0.0)
                x[b, t, k, tokens] = _ladder(top, n)
    _check(hip, oracle, x, "f32", overlap, eos_token=-1, alpha=alpha)
    _check(hip, oracle, x, "f32", overlap, eos_token=7, alpha=alpha)


@pytest.mark.parametrize("K", range(1, 10))
def test_greedy_and_long(hip, oracle, K):
    """Random log-probs, 128 steps: ties by rounding as they come."""
    rng = np.random.default_rng(40 + K)
    x = rng.normal(0.0, 2.0, size=(16, 128, K, 1000)).astype(np.float32)
    x = x - np.log(np.exp(x).sum(-1, keepdims=True))
    _check(hip, oracle, x, "f32", -1, eos_token=-1, alpha=0.6)


@pytest.mark.parametrize("overlap", [0, 1])
@pytest.mark.parametrize("K", range(1, 10))
def test_logits_ties(hip, oracle, K, overlap):
    """Logits a few ulps apart far below one large one: one log-prob at every
    step, the first among them."""
    B, T, V = 4, 4, 600
    rng = np.random.default_rng(80 + K)
    x = rng.uniform(-90.0, -50.0, size=(B, T, K, V)).astype(np.float32)
    banned = np.zeros(V, np.uint8)
    banned[11] = 1
    x[..., 11] = 30.0  # lse 30: x - lse near -30 has ulps of 2^-19
    for b in range(B):
        n = [K + 1, K + 2, 2 * K + 3, 22][b]
        for t in range(T):
            for k in range(K):
                tokens = np.sort(rng.choice(np.arange(12, V), size=n, replace=False))[::-1]
                x[b, t, k, tokens] = _ladder(0.125, n)
    _check(hip, oracle, x, "f32", overlap, from_logits=True, eos_token=-1, alpha=0.6, banned=banned)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("K", [1, 4, 8])
def test_equal_log_probs(hip, oracle, K, dtype):
    """16-bit log-probs that are equal, and ones that round to one raw."""
    rng = np.random.default_rng(K)
    x = -rng.integers(1, 9, size=(8, 9, K, 700)).astype(np.float32) / 2
    x[:, 0] -= 4000.0
    x[4:, 1:] *= np.float32(2.0 ** -13)  # far below the raw's ulp
    _check(hip, oracle, x, dtype, -1, eos_token=-1, alpha=0.6)


def _wide_rows():
    """72 beams: after a first step near -30000, 71 rows give one good entry
    each, and 80 entries of the last row share the raw of the 72nd place. Its
    lowest token stands past one that ranks after the eleven before it."""
    B, T, K, V, R = 2, 3, 72, 700, -30005.0
    rng = np.random.default_rng(5)
    x = rng.uniform(-20000.0, -19000.0, size=(B, T, K, V)).astype(np.float32)
    first = (-30000.0 + np.arange(K)[::-1] * 2.0 ** -7).astype(np.float32)
    x[:, 0, 0] -= 30000.0
    x[:, 0, 0, 100:100 + K] = first
    for k in range(K - 1):
        x[:, 1, k, 650] = np.float32(R + 1.0) - first[k]
    tokens = np.concatenate([np.arange(600, 611), [680], np.arange(300, 368)[::-1]])
    lp = (np.float64(R) - np.float64(first[K - 1]) + 4e-4 - 1e-5 * np.arange(80)).astype(np.float32)
    assert len(np.unique(lp)) == 80 and np.all(first[K - 1] + lp == np.float32(R))
    x[:, 1, K - 1, tokens] = lp
    return x


@pytest.mark.parametrize("overlap", [0, 1])
def test_wide_lists_in_rounds(hip, oracle, overlap):
    _check(hip, oracle, _wide_rows(), "f32", overlap, eos_token=-1, alpha=0.6, repetition_penalty=1.2)


def test_wide_lists_step_api(hip, oracle):
    x = _wide_rows()
    want = oracle.decode(x, dtype="f32", eos_token=-1, alpha=0.6)
    got = hip.steps(x, "f32", eos_token=-1, alpha=0.6)
    for name in got:
        a, b = np.asarray(got[name]), np.asarray(want[name])
        assert np.array_equal(a.view(np.uint32) if a.dtype == np.float32 else a,
                              b.view(np.uint32) if b.dtype == np.float32 else b), name


@pytest.mark.parametrize("K", [12, 24, 64, 65, 130, 300])
@pytest.mark.parametrize("constrained", [False, True])
def test_more_beams(hip, oracle, K, constrained):
    """Past the grid, where every entry that reaches tau is a candidate."""
    rng = np.random.default_rng(K)
    x = rng.uniform(-90.0, -50.0, size=(2, 4, K, 900)).astype(np.float32)
    x[:, 0] -= 300.0
    for b in range(2):
        for t in range(4):
            for k in range(K):
                n = int(rng.integers(1, 100))
                tokens = np.sort(rng.choice(900, size=n, replace=False))[::-1]
                top = (-300.0 if t == 0 else -1.5) - 0.25 * float(rng.integers(0, 3))
                x[b, t, k, tokens] = _ladder(top, n)
    kw = dict(no_repeat_ngram_size=2, repetition_penalty=1.3) if constrained else {}
    _check(hip, oracle, x, "f32", -1, eos_token=-1, alpha=0.6, **kw)
