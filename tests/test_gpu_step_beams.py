# SPDX-License-Identifier: MIT
"""beamgrad::step_beams (one step and the beams it leaves, in one operator)
against decode_step followed by the same in torch operations, step by step:
one beam to more beams than the kernel's block, finished beams until all have,
dead beams, and rows flagged by validation."""

import pytest
import torch

import beamgrad_amd as bg
from beamgrad_amd._search import _Beams, _ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,K,V", [(1, 1, 5), (3, 5, 40), (70, 8, 33), (2, 3, 2), (2, 200, 7), (5, 64, 1)])
@pytest.mark.parametrize("constrained", [False, True])
def test_step_beams(B, K, V, constrained):
    gen = torch.Generator().manual_seed(B * K)
    opts = bg.BeamOptions(beam_size=K, eos_token=0, length_penalty_alpha=0.6,
                          no_repeat_ngram_size=2 if constrained else 0,
                          repetition_penalty=1.3 if constrained else 1.0)
    fast, slow = _Beams(B, K, torch.device("cuda")), _Beams(B, K, torch.device("cuda"))
    for t in range(6):
        rows = torch.randn(B, K, V, generator=gen).log_softmax(-1)
        rows[..., 0] += 1.0 if t < 4 else 20.0  # at the end every beam finishes
        rows = rows.cuda()
        out, any_active = fast.step(rows, t, 0, [], opts, None)
        want = _ops.decode_step(rows, slow.raw, slow.lengths, slow.finished, slow.sequences.int(), 0, 0, 0.6, None,
                                opts.no_repeat_ngram_size, opts.repetition_penalty, True, [])
        slow.advance(want, t)
        for a, b in zip(out, want, strict=True):
            assert a.dtype == b.dtype and torch.equal(a, b)
        state = fast.state
        active = slow.active()
        assert any_active == bool(active.any())
        for a, b in zip(state, slow.entering(t + 1, active), strict=True):
            assert (a == b) if isinstance(a, int) else (a.dtype == b.dtype and torch.equal(a, b))
        assert torch.equal(fast.prefixes, slow.sequences.int())
    if K <= 8:  # (more beams than candidates before the last steps keep a few unfinished)
        assert not any_active


def test_step_beams_flags():
    beams = _Beams(2, 2, torch.device("cuda"))
    rows = torch.zeros(2, 2, 4).log_softmax(-1)
    rows[1, 0, 3] = float("nan")
    with pytest.raises(ValueError, match="example 1: log_probs contains NaN"):
        beams.step(rows.cuda(), 0, -1, [], bg.BeamOptions(beam_size=2), None)
    beams.step(rows.cuda(), 0, -1, [], bg.BeamOptions(beam_size=2, validate_inputs=False), None)
