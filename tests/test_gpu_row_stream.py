# SPDX-License-Identifier: MIT
"""The row pass that reads logits rows twice (dbs_hip_set_row_pass(7)) against
the CPU oracle bit for bit: every input type, vocabularies around its group of
4096 entries and its 16-byte blocks, rows at any element offset, rows with NaN,
+inf, -inf and entries far below the maximum, maxima around the bounds of the
bfloat16 term table, long shortlists, and the decode beside its select pass."""

import numpy as np
import pytest

from tests.cases import first_difference, make_case, to_bits

pytestmark = pytest.mark.gpu

VOCABS = [1, 2, 7, 255, 256, 257, 2047, 4095, 4096, 4097, 8191, 8192, 8193, 12001, 12288, 20483]


@pytest.fixture
def stream(hip):
    prev = hip.lib.dbs_hip_set_row_pass(7)
    yield
    hip.lib.dbs_hip_set_row_pass(prev)


def _check(hip, oracle, xin, dtype, **kw):
    offset = kw.pop("x_offset", 0)
    want = oracle.decode(xin, dtype=dtype, **kw)
    got = hip.decode(xin, dtype, x_offset=offset, **kw)
    assert first_difference(got, want) is None, first_difference(got, want)


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("V", VOCABS)
def test_stream_vocabularies(hip, oracle, stream, dtype, V):
    rng = np.random.default_rng(V)
    K = min(4, V)
    x = rng.normal(0.0, 3.0, size=(3, 4, K, V)).astype(np.float32)
    x[rng.random(x.shape) < 0.05] = -np.inf
    for offset in (0, 1, 3):
        _check(hip, oracle, to_bits(x, dtype), dtype, from_logits=True, eos_token=min(1, V - 1), min_length=2,
               alpha=0.6, x_offset=offset)


@pytest.mark.parametrize("seed", range(24))
def test_stream_random(hip, oracle, stream, seed):
    case = make_case(7300 + seed, big=True, logits=True)  # ties, NaN, +inf, constraints, banned masks
    _check(hip, oracle, case["xin"], case["dtype"], **case["kw"])


@pytest.mark.parametrize("overlap", [0, 1])
@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
def test_stream_beside_the_select_pass(hip, oracle, stream, dtype, overlap):
    rng = np.random.default_rng(5)
    x = rng.normal(0.0, 3.0, size=(4, 9, 5, 12345)).astype(np.float32)
    x[..., 77] += 8.0
    hip.lib.dbs_hip_set_decode_overlap(overlap)
    try:
        _check(hip, oracle, to_bits(x, dtype), dtype, from_logits=True, eos_token=77, alpha=1.0, steps=[9, 1, 4, 7])
    finally:
        hip.lib.dbs_hip_set_decode_overlap(-1)


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
def test_stream_row_values(hip, oracle, stream, dtype):
    """One row per kind of value the terms and the table turn on."""
    rng = np.random.default_rng(17)
    V = 12601
    rows = []
    for top in (0.0, -3.0, 0.99, 1.0, 1.5, 64.0, 126.5, 127.0, 127.5, 300.0):
        r = rng.normal(0.0, 2.0, size=V).astype(np.float32)
        r = np.minimum(r, top - 0.25)
        r[V // 3] = top
        rows.append(r)
    far = rows[3].copy()
    far[::7] = np.float32(1.0) - rng.uniform(86.0, 89.0, size=far[::7].shape).astype(np.float32)  # terms around 0
    rows.append(far)
    tiny = (rng.normal(0.0, 1.0, size=V) * 2.0 ** rng.integers(-40, 3, size=V)).astype(np.float32)  # slots of the table
    rows.append(tiny)
    for value in (np.nan, np.inf, -np.inf):
        r = rows[4].copy()
        r[[5, 4096, V - 1]] = value
        rows.append(r)
    negative_nan = rows[4].copy()
    negative_nan[9] = np.copysign(np.float32(np.nan), np.float32(-1.0))
    rows.append(negative_nan)
    rows.append(np.full(V, -np.inf, np.float32))
    rows.append(np.full(V, -7.0, np.float32))  # constant: more survivors than are kept
    masked = np.full(V, -np.inf, np.float32)
    masked[[3, V - 1]] = [2.0, 1.0]
    rows.append(masked)
    x = np.stack(rows)[:, None, None, :]
    _check(hip, oracle, to_bits(x, dtype), dtype, from_logits=True, alpha=0.6)
    x = np.repeat(np.stack(rows)[:, None, None, :], 3, axis=1)
    _check(hip, oracle, to_bits(x, dtype), dtype, from_logits=True, alpha=0.6)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_stream_long_shortlists(hip, oracle, stream, dtype):
    rng = np.random.default_rng(23)
    x = rng.normal(0.0, 1.0, size=(2, 3, 64, 5003)).astype(np.float32)
    banned = (rng.random(5003) < 0.3).astype(np.uint8)
    _check(hip, oracle, to_bits(x, dtype), dtype, from_logits=True, alpha=0.6, banned=banned)


@pytest.mark.parametrize("dtype,V", [("f32", 1), ("f32", 4097), ("f32", 20483), ("f16", 8191), ("bf16", 12289)])
def test_stream_log_probs(hip, oracle, stream, dtype, V):
    rng = np.random.default_rng(V)
    x = rng.normal(-9.0, 2.0, size=(2, 4, 3, V)).astype(np.float32)
    x[rng.random(x.shape) < 0.05] = -np.inf
    x[1, 2, 0, V // 2] = np.nan  # read: the row is flagged and read in full
    for offset in (0, 1):
        _check(hip, oracle, to_bits(x, dtype), dtype, eos_token=-1, alpha=0.6, x_offset=offset)


# around the log-prob row pass's blocks per thread: 40, 46 and 52 of 256
# threads, 32, 40 and 52 of 512, and past them (the stream pass)
@pytest.mark.parametrize("dtype,V", [("f32", 40957), ("f32", 47100), ("f32", 53233), ("f32", 65533), ("f32", 81918),
                                     ("f32", 106480), ("f32", 106489), ("f16", 81913), ("bf16", 106481),
                                     ("f16", 131069), ("bf16", 151936), ("f16", 212960), ("bf16", 212977)])
def test_long_log_prob_rows(hip, oracle, dtype, V):
    rng = np.random.default_rng(V)
    x = rng.normal(-12.0, 2.0, size=(2, 3, 3, V)).astype(np.float32)
    x[1, 1, 1, 5] = np.inf  # flagged where read
    x[0, :, :, V - 1] = -3.0  # the last element is selected
    for offset in (0, 3):
        _check(hip, oracle, to_bits(x, dtype), dtype, eos_token=-1, alpha=0.6, x_offset=offset)
