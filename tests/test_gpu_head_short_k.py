"""The weight-stationary head GEMM over one or two K steps of 64 (whole tiles of activations in flight): row counts
at the edges of a 16-row tile and of a workgroup's eight tiles, runs of one and of two groups of eight with a partial last
one, vocabularies with partial channel tiles and unaligned rows, bit-identical to the streaming kernel (the same exact
digit sums, the same epilogue)."""
import numpy as np
import pytest

from helpers import assert_close, oracle_model, tiny_spec, uniform_model_bytes
from mignon_ai_amd import Model, engine_option, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def restore():
    prev = {k: engine_option(k) for k in ("gemm", "operands")}
    engine_option("operands", "limbs")
    yield
    for k, v in prev.items():
        engine_option(k, v)


def _compare(D, V, shapes, seed=3):
    data = uniform_model_bytes(tiny_spec([(1, 2, 1)], V=V, D=D, H=40), seed=seed, scale=0.3)
    m, om = Model(data), oracle_model(data)
    for B, T in shapes:
        ids = synth.token_ids(81, f"head{D}{V}{T}", (B, T), V)
        out = {}
        for mode in ("stream", "slab"):
            engine_option("gemm", mode)
            out[mode] = m.forward_batch(ids, logits=True, probs=True, logprob=True)
            out[mode].update({k + "2": v for k, v in m.forward_batch(ids, logits=False, logprob=True, bits=True).items()})
        for k in out["stream"]:
            assert np.array_equal(out["stream"][k].view(np.uint32), out["slab"][k].view(np.uint32)), (D, V, B, T, k)
        assert_close(out["slab"]["logits"][-1:], om.forward_all(ids[-1:]), what=f"D{D} V{V} {B}x{T}")


@pytest.mark.parametrize("D", [32, 64, 100, 128])
@pytest.mark.parametrize("V", [16, 131, 300])
def test_slab_equals_stream(D, V):
    _compare(D, V, [(1, 1), (1, 15), (1, 17), (3, 43), (8, 16), (1, 129), (9, 128), (70, 31)])


@pytest.mark.parametrize("D", [40, 64, 128])
def test_runs_of_several_groups(D):
    """Eight channel tiles: from 16384 rows on a workgroup's run is two groups of eight tiles, so that the tiles in flight
    carry over from one to the next; 16500 rows leave the last run half full and its last tile with four rows, 16404 one
    group with two tiles in its run."""
    _compare(D, 1000, [(132, 125), (1367, 12)])
