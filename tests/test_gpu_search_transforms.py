# SPDX-License-Identifier: MIT
"""beam_search where its rows or its state carry more than values: rows that are
forward-mode dual tensors, rows of the caller's under a functorch transform,
and a last step that nothing has to be read back from."""

import pytest
import torch
import torch.autograd.forward_ad as forward_ad

import beamgrad_amd as bg

pytestmark = pytest.mark.gpu

OPTS = bg.BeamOptions(beam_size=3, eos_token=2, length_penalty_alpha=0.6)


def _rows(T=3, B=2, V=11):
    gen = torch.Generator().manual_seed(11)
    return torch.randn(T, B, 3, V, generator=gen).log_softmax(-1).cuda()


@pytest.mark.parametrize("enabled", [True, False])
@pytest.mark.parametrize("dual_step", [0, 2])
def test_dual_rows_are_refused(enabled, dual_step):
    """There is no forward-mode rule: an error, never scores without a tangent."""
    rows = _rows()
    with forward_ad.dual_level(), torch.set_grad_enabled(enabled):
        dual = forward_ad.make_dual(rows[dual_step], torch.ones_like(rows[dual_step]))
        with pytest.raises((NotImplementedError, RuntimeError), match="jvp"):
            bg.beam_search(lambda s: dual if s.step == dual_step else rows[s.step], OPTS, 3, batch_size=2, device="cuda")
        # rows without a tangent inside a level are plain rows
        scores = bg.beam_search(lambda s: rows[s.step], OPTS, 3, batch_size=2, device="cuda").scores
        assert forward_ad.unpack_dual(scores).tangent is None


@pytest.mark.parametrize("max_steps", [1, 3])
def test_last_step_is_not_waited_for(max_steps):
    """Without validation, nothing follows from the last step's outcome."""
    rows = _rows()
    options = bg.BeamOptions(beam_size=3, eos_token=2, length_penalty_alpha=0.6, validate_inputs=False)
    busy = torch.randn(8192, 8192, device="cuda")
    queued = torch.cuda.Event()

    def step(state):
        if state.step + 1 == max_steps:
            for _ in range(20):
                busy @ busy  # tens of milliseconds ahead of the last step
            queued.record()
        return rows[state.step]

    bg.beam_search(lambda s: rows[s.step], options, max_steps, batch_size=2, device="cuda")
    busy @ busy
    torch.cuda.synchronize()
    bg.beam_search(step, options, max_steps, batch_size=2, device="cuda")
    assert not queued.query()


def test_outer_rows_under_transforms():
    """The caller's own rows inside torch.func transforms, whose beams are wrapped."""
    rows = _rows()

    def weighted(w):
        return (bg.beam_search(lambda s: rows[s.step], OPTS, 3, batch_size=2, device="cuda").scores * w).sum()

    def first_step(x):
        return bg.beam_search(lambda s: x if s.step == 0 else rows[s.step], OPTS, 3, batch_size=2,
                              device="cuda").scores.sum()

    scores = bg.beam_search(lambda s: rows[s.step], OPTS, 3, batch_size=2, device="cuda").scores
    w = torch.arange(6.0, device="cuda").reshape(2, 3)
    assert torch.equal(torch.func.grad(weighted)(w), scores)
    value, tangent = torch.func.jvp(weighted, (w,), (w,))
    assert torch.equal(value, (scores * w).sum()) and torch.equal(tangent, value)
    x = rows[0].clone().requires_grad_(True)
    first_step(x).backward()
    assert torch.equal(torch.func.grad(first_step)(rows[0]), x.grad)
