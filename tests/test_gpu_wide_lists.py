# SPDX-License-Identifier: MIT
"""More than 64 beams over rows longer than their shortlists (80 entries), on
the GPU against the CPU oracle bit for bit: beams past which the lists stay in
global memory (65), one and two candidates per thread of the rank compaction
(K to 512) and the sort past it, rows with many ties (the collector overflows,
every list is offered in turn) and constant rows (every row is read in full,
with more candidates at the threshold than the rescan buffer holds);
constraints, per-example beams, finished beams, the step API and the decode
beside its row pass."""

import numpy as np
import pytest

from tests.cases import first_difference, log_softmax, to_bits

pytestmark = pytest.mark.gpu

CASES = [
    # K, V, dtype, logits, rows, options
    (65, 1200, "f32", False, "plain", dict(eos_token=2, min_length=2, alpha=0.6)),
    (100, 4003, "f16", False, "ties", dict(eos_token=7, extra_eos=[11], alpha=1.0)),
    (128, 2048, "bf16", True, "plain", dict(eos_token=5, alpha=0.6)),
    (256, 5000, "f32", False, "plain", dict(alpha=0.6)),
    (256, 900, "f32", True, "ties", dict(eos_token=3, alpha=0.0)),
    (257, 1500, "f32", False, "plain", dict(no_repeat_ngram_size=2, repetition_penalty=1.3)),
    (520, 1031, "bf16", False, "ties", dict(eos_token=1, alpha=0.6)),
    (1024, 1100, "f32", False, "plain", dict(alpha=1.0)),
    (80, 700, "f32", False, "constant", dict(alpha=0.6)),
    (300, 640, "f32", False, "constant", dict(repetition_penalty=1.5)),
]


def _case(i):
    K, V, dtype, logits, rows, opts = CASES[i]
    B, T = 2, 4
    rng = np.random.default_rng(4100 + i)
    x = rng.normal(0.0, 2.0, size=(B, T, K, V)).astype(np.float32)
    if rows == "constant":
        x[:] = 0.0
    if opts.get("eos_token", -1) >= 0:
        x[..., opts["eos_token"]] += 6.0  # beams finish
    if not logits:
        x = log_softmax(x)
    if rows == "ties":
        pool = np.quantile(x, [0.9, 0.99, 0.999]).astype(np.float32)
        mask = rng.random(x.shape) < 0.2
        x[mask] = rng.choice(pool, size=int(mask.sum()))
    x[rng.random(x.shape) < 0.01] = -np.inf
    kw = dict(from_logits=logits, eos_token=-1, alpha=0.0)
    kw.update(opts)
    return x, to_bits(x, dtype), dtype, kw


@pytest.mark.parametrize("overlap", [0, 1])
@pytest.mark.parametrize("i", range(len(CASES)))
def test_wide_lists_decode(hip, oracle, i, overlap):
    x, xin, dtype, kw = _case(i)
    if i % 2 == 0:
        kw["steps"] = [4, 3]
    want = oracle.decode(xin, dtype=dtype, **kw)
    hip.lib.dbs_hip_set_decode_overlap(overlap)
    try:
        got = hip.decode(xin, dtype, **kw)
    finally:
        hip.lib.dbs_hip_set_decode_overlap(-1)
    assert first_difference(got, want) is None, first_difference(got, want)


@pytest.mark.parametrize("i", [0, 3, 4, 6, 8])
def test_wide_lists_step_api(hip, oracle, i):
    x, xin, dtype, kw = _case(i)
    want = oracle.decode(xin, dtype=dtype, **kw)
    got = hip.steps(xin, dtype, **kw)
    for name in got:
        a, b = np.asarray(got[name]), np.asarray(want[name])
        assert np.array_equal(a.view(np.uint32) if a.dtype == np.float32 else a,
                              b.view(np.uint32) if b.dtype == np.float32 else b), name


def test_wide_lists_per_example_beams(hip, oracle):
    x, xin, dtype, kw = _case(3)
    beams = [70, 9]
    want = oracle.decode_per_example(xin, dtype=dtype, beams=beams, **kw)
    got = hip.decode(xin, dtype, beams=beams, **kw)
    assert first_difference(got, want) is None, first_difference(got, want)


def test_wide_without_room_for_lists(hip, oracle):
    """A workspace with no room for the lists (and the static scratch past
    its limit with them) reads every row in full, as before; less than that is
    refused."""
    import ctypes as C

    import torch

    from beamgrad_amd import _abi

    x, xin, dtype, kw = _case(0)
    want = oracle.decode(xin, dtype=dtype, **kw)
    full = hip.lib.dbs_cuda_decode_workspace_size

    def smaller(args):
        return full(args) - 80 * 8 * x.shape[0] * x.shape[1] * x.shape[2]

    hip.lib.dbs_cuda_decode_workspace_size = smaller
    try:
        got = hip.decode(xin, dtype, **kw)
    finally:
        hip.lib.dbs_cuda_decode_workspace_size = full
    assert first_difference(got, want) is None
    # rows whose lists alone pass the static scratch: 16 bytes a row fit it
    B, T, K, V = 16, 64, 128, 96
    args = _abi.DecodeArgs()
    args.batch_size, args.steps, args.beam_size, args.vocab_size = B, T, K, V
    args.eos_token, args.repetition_penalty = -1, 1.0
    assert full(C.byref(args)) > _abi.NOALLOC_SCRATCH_BYTES
    rows = torch.randn(B, T, K, V, generator=torch.Generator().manual_seed(5)).log_softmax(-1).numpy()
    got = hip.decode(rows, "f32", noalloc=True)
    assert first_difference(got, hip.decode(rows, "f32")) is None


def test_wide_lists_without_memory_for_them():
    """Where the device has no room for the lists (656 bytes a row against 16),
    a decode through torch goes without them, as one with a smaller workspace
    does: the same results, every row read in full."""
    import torch

    import beamgrad_amd as bg

    B, T, K, V = 16, 128, 128, 4
    x = torch.randn(B, T, K, V, generator=torch.Generator().manual_seed(3)).log_softmax(-1).cuda()
    options = bg.BeamOptions(beam_size=K, eos_token=-1, length_penalty_alpha=0.6)
    want = [t.clone() for t in bg.decode(x, options)]
    lists = 80 * 8 * B * T * K  # 168 MB
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.empty_cache()
    room = torch.cuda.memory_reserved() + lists // 2
    torch.cuda.set_per_process_memory_fraction(room / total)
    try:
        got = bg.decode(x, options)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    for a, b in zip(got, want, strict=True):
        assert torch.equal(a, b)
