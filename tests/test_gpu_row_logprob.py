# SPDX-License-Identifier: MIT
"""The one-read row pass for log-prob rows against the CPU oracle bit for bit
where its block test by pattern takes each of its forms: thresholds below, at
and above zero, zeros of both signs, rows of one value, and rows that end at
and beside a block and a 256-block edge, at unaligned starts."""

import numpy as np
import pytest

from tests.cases import first_difference, to_bits

pytestmark = pytest.mark.gpu

VALUES = {
    "negative": lambda r, s: -np.abs(r.normal(0.0, 3.0, size=s)),
    "positive": lambda r, s: np.abs(r.normal(0.0, 3.0, size=s)),
    "around zero": lambda r, s: r.normal(0.0, 1e-3, size=s),
    "zero threshold": lambda r, s: np.where(r.random(s) < 0.05, 1.0, np.where(r.random(s) < 0.5, 0.0, -0.0)),
    "negative zeros": lambda r, s: np.where(r.random(s) < 0.3, -0.0, -1.0),
    "denormals": lambda r, s: -np.abs(r.normal(0.0, 1e-7, size=s)),
    "infinite": lambda r, s: np.where(r.random(s) < 0.8, -np.inf, -r.random(s)),
}


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("values", list(VALUES))
@pytest.mark.parametrize("V", [9, 1024, 2047, 2049, 12301])
def test_block_test(hip, oracle, dtype, values, V):
    rng = np.random.default_rng(V)
    x = to_bits(VALUES[values](rng, (2, 4, 5, V)).astype(np.float32), dtype)
    kw = dict(eos_token=3, min_length=2, alpha=0.6)
    want = oracle.decode(x, dtype=dtype, **kw)
    hip.lib.dbs_hip_set_row_pass(3)
    try:
        for offset in (0, 1):
            got = hip.decode(x, dtype, x_offset=offset, **kw)
            assert first_difference(got, want) is None, first_difference(got, want)
    finally:
        hip.lib.dbs_hip_set_row_pass(-1)
