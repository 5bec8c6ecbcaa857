"""Prefill of prompts of unequal length packed in whole 16-row tiles (the layered body, lengths given on the host): prompts
at the edges of the tiles, prompts longer than the sessions' window, no attention, head widths of no whole tile, both ring
formats, and more prompts than the packing kernel has threads; then steps that read the exported state."""
import numpy as np
import pytest

from helpers import assert_close, oracle_model, tiny_spec, uniform_model_bytes
from mignon_ai_amd import Model, engine_option, synth

pytestmark = pytest.mark.gpu

V = 131
# D, H, heads, window, blocks
SHAPES = [
    (160, 288, 5, 48, [(2, 2, 1), (2, 2, 2)]),
    (132, 100, 3, 7, [(0, 2, 1), (1, 2, 32)]),
    (256, 320, 4, 64, [(1, 2, 1)] * 2),
    (136, 64, 0, 0, [(3, 2, 1), (1, 2, 16)]),
]
LENS = [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 1, 3, 5, 64, 65, 8, 9, 100]


@pytest.fixture(autouse=True)
def restore():
    prev = engine_option("kv_rings")
    yield
    engine_option("kv_rings", prev)


def _build(shape):
    D, H, heads, window, blocks = shape
    spec = tiny_spec(blocks, V=V, D=D, H=H, heads=heads, window=window, context=128, tied=False)
    return uniform_model_bytes(spec, seed=9, scale=0.25), sum(b[0] for b in blocks)


def _prefill(m, s, prompts, lens, steps):
    m.profile(True)
    lg = s.prefill(prompts, lens)[0]
    prof = m.profile_read()
    m.profile(False)
    # the packed prefill scans each rule step in one launch, where as few sequences as these otherwise take two
    assert prof["latch_scan"][0] == steps, prof
    return lg


@pytest.mark.parametrize("rings", ["fp32", "packed"])
@pytest.mark.parametrize("window", [128, 40])
@pytest.mark.parametrize("shape", SHAPES)
def test_unequal_prompts(shape, window, rings):
    data, rule_steps = _build(shape)
    engine_option("kv_rings", rings)
    m, om = Model(data), oracle_model(data)
    lens = np.array((LENS if window == 128 else [min(n, 16) for n in LENS[:-1]] + [100]) * 8, np.int32)
    S, T = len(lens), int(lens.max())
    prompts = synth.token_ids(81, f"pk{shape}", (S, T), V)
    nexts = synth.token_ids(82, f"pn{shape}", (4, S), V)
    s = m.sessions(S, window)
    out = [_prefill(m, s, prompts, lens, rule_steps)] + [s.step(n)[0] for n in nexts]
    for i in range(0, S, 8):  # every length once
        if window < 128 and lens[i] > window:  # the state is that of the last `window` tokens, later steps follow on
            seq = prompts[i, lens[i] - window:lens[i]]
        else:
            seq = prompts[i, :lens[i]]
        assert_close(out[0][i], om.call(seq), what=f"{shape} {window} {rings} session {i} prefill")
        if window == 128:
            for k in range(1, len(out)):
                assert_close(out[k][i], om.call(np.concatenate([seq, nexts[:k, i]])),
                             what=f"{shape} {rings} session {i} step {k}")


def test_many_prompts():
    """More prompts than threads of the packing kernel; every one also alone in a set of its own kind."""
    data, _ = _build(SHAPES[0])
    m, om = Model(data), oracle_model(data)
    S, T = 2500, 40
    lens = 1 + (np.arange(S) * 7919 % 20).astype(np.int32)
    lens[-1] = T
    prompts = synth.token_ids(83, "many", (S, T), V)
    lg, am, _ = m.sessions(S, 128).prefill(prompts, lens)
    for i in (0, 1, 2, 3, 1023, 1024, 1025, 2047, 2048, 2498, 2499):
        assert_close(lg[i], om.call(prompts[i, :lens[i]]), what=f"session {i}")
    assert np.array_equal(am, lg.argmax(-1))
    for n in (1, 13, 20):  # prompts of one length are not packed
        at = np.flatnonzero(lens == n)
        want = m.sessions(len(at), 128).prefill(np.ascontiguousarray(prompts[at, :n]))[0]
        assert_close(lg[at], want, rtol=2e-5, what=f"prompts of {n}")
