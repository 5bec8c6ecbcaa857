"""The one-kernel body (csrc/seq.hip) against the oracle and the layered kernels: every compiled variant (state of one
or two 64-channel groups, hidden sizes of one to four, with and without attention), sequences at the edges of the
16-token tiles and of the eight tiles of a workgroup, several sequences per workgroup, rows the head does not read,
and the session state it exports in both ring formats."""
import numpy as np
import pytest

from helpers import assert_close, model_bytes, oracle_model, rel_err, tiny_spec, uniform_model_bytes
from mignon_ai_amd import Model, engine_option, synth
from mignon_ai_amd.evaluate import score_sequences

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

# D, H, heads, window, blocks: one entry per compiled variant, among them head widths of no whole groups of four or
# below 16, several rule steps with dilations up to 32, blocks without steps (the last one too), windows of one key, of a
# whole tile and of the longest span
SHAPES = [
    (32, 64, 0, 0, [(2, 2, 1)]),
    (64, 100, 0, 0, [(3, 3, 2), (1, 2, 1)]),
    (100, 128, 0, 0, [(1, 2, 1)] * 3),
    (128, 180, 0, 0, [(1, 2, 32)]),
    (72, 256, 0, 0, [(2, 2, 1), (1, 2, 16)]),
    (48, 60, 2, 64, [(1, 2, 1)] * 2),
    (60, 128, 2, 7, [(0, 2, 1), (2, 2, 1)]),
    (96, 128, 4, 64, [(1, 2, 1)] * 2),
    (100, 160, 4, 1, [(1, 2, 1)] * 2),
    (128, 256, 4, 17, [(2, 2, 1), (0, 2, 1), (1, 2, 2)]),
    (24, 60, 2, 16, [(1, 2, 1), (0, 2, 1)]),
    (128, 160, 4, 65, [(1, 2, 1), (2, 2, 1)]),
]


@pytest.fixture(autouse=True)
def restore():
    prev = {k: engine_option(k) for k in ("gemm", "scan", "attention", "operands", "kv_rings")}
    yield
    for k, v in prev.items():
        engine_option(k, v)


def _build(shape, seed=5):
    D, H, heads, window, blocks = shape
    spec = tiny_spec(blocks, V=131, D=D, H=H, heads=heads, window=window, context=128, tied=False)
    return uniform_model_bytes(spec, seed=seed, scale=0.3)


def _classes(m, fn):
    m.profile(True)
    out = fn()
    prof = m.profile_read()
    m.profile(False)
    return out, prof


@pytest.mark.parametrize("shape", SHAPES)
def test_forward_lengths(shape):
    data = _build(shape)
    m, om = Model(data), oracle_model(data)
    for B, T in [(1, 1), (9, 15), (17, 16), (5, 17), (3, 63), (5, 64), (3, 65), (2, 127), (3, 128)]:
        ids = synth.token_ids(71, f"seq{shape}{T}", (B, T), 131)
        ids[0, 0] = -3  # out of range: token 0
        got, prof = _classes(m, lambda: m.forward_batch(ids, logits=True, logprob=True, bits=True))
        assert "sequence_body" in prof and "gemm_glu" not in prof, (T, prof)
        assert_close(got["logits"], om.forward_all(ids), what=f"{shape} T={T}")
        engine_option("operands", "limbs")  # the layered body
        want = Model(data).forward_batch(ids, logits=True, logprob=True, bits=True)
        engine_option("operands", "auto")
        for k in ("logits", "bits"):
            assert_close(got[k], want[k], rtol=2e-5, what=f"{shape} T={T} {k} vs layered")
    # longer sequences and any option that names a layered kernel take the layered body
    ids = synth.token_ids(72, f"seq{shape}", (2, 129), 131)
    got, prof = _classes(m, lambda: m.forward_batch(ids)["logits"])
    assert "sequence_body" not in prof
    assert_close(got, om.forward_all(ids), what=f"{shape} T=129")


@pytest.mark.parametrize("shape", SHAPES)
def test_call_and_score(shape):
    """Rows the head does not read: the last position only, and windows scored at one or at all positions."""
    data = _build(shape)
    m, om = Model(data), oracle_model(data)
    ids = synth.token_ids(73, f"call{shape}", (150,), 131)
    for n in (1, 2, 16, 17, 64, 65, 80, 113, 128, 150):
        assert_close(m.call(ids[:n]), om.call(ids[max(0, n - 128):n]), what=f"{shape} call {n}")
    docs = [synth.token_ids(74, f"doc{n}", (n,), 131) for n in (2, 17, 40, 129, 140)]
    for ctx in (128, 20):
        for d, lp in zip(docs, score_sequences(m, docs, ctx)):
            for t in range(1, len(d), 7):
                lg = om.call(d[max(0, t - ctx):t]).astype(np.float64)
                want = lg[d[t]] - lg.max() - np.log(np.exp(lg - lg.max()).sum())
                assert abs(lp[t - 1] - want) <= 1e-4 * max(1.0, abs(want)), (shape, ctx, len(d), t)


@pytest.mark.parametrize("rings", ["fp32", "packed"])
@pytest.mark.parametrize("shape", SHAPES)
def test_prefill_exports_the_state(shape, rings):
    """Prefill of unequal lengths, then steps that read every part of the exported state, rings wrapping."""
    data = _build(shape)
    engine_option("kv_rings", rings)
    m, om = Model(data), oracle_model(data)
    S, T = 19, 100
    prompts = synth.token_ids(75, f"pre{shape}", (S, T), 131)
    lens = np.array([1, 2, 15, 16, 17, 31, 33, 48, 63, 64, 65, 66, 79, 80, 81, 96, 97, 99, 100], np.int32)
    steps = synth.token_ids(76, f"pst{shape}", (6, S), 131)
    s = m.sessions(S, 128)
    (lg, am, _), prof = _classes(m, lambda: s.prefill(prompts, lens))
    assert "sequence_body" in prof
    out = [lg] + [s.step(steps[k])[0] for k in range(len(steps))]
    for i in range(S):
        for k in range(len(out)):
            seq = np.concatenate([prompts[i, :lens[i]], steps[:k, i]])
            assert_close(out[k][i], om.call(seq), what=f"{shape} {rings} session {i} step {k}")


def test_forward_many_sequences():
    """More workgroups than compute units, the benchmark's D128 model: both ends against the oracle, and against the
    layered body everywhere."""
    data = model_bytes("c3")
    ids = synth.token_ids(77, "seq:c3", (600, 100), 2048)
    got = Model(data).forward_batch(ids, logits=False, logprob=True)["logprob"]
    engine_option("operands", "limbs")
    want = Model(data).forward_batch(ids, logits=False, logprob=True)["logprob"]
    engine_option("operands", "auto")
    assert rel_err(got[:, :-1], want[:, :-1]).max() < 2e-5
    sub = [0, 599]
    assert_close(Model(data).forward_batch(ids[sub])["logits"], oracle_model(data).forward_all(ids[sub]), what="c3")


def test_many_steps():
    """A block's rule steps share one copy of the kernel's weights: a file of many steps loads in the memory of its
    weights, and repeated steps, waves without work among them, equal the layered body."""
    spec = tiny_spec([(20000, 2, 1)], V=131, D=32, H=64, context=128)
    data = uniform_model_bytes(spec, seed=6, scale=0.3)
    free = torch.cuda.mem_get_info()[0]
    m = Model(data)
    used = free - torch.cuda.mem_get_info()[0]
    assert used < 64 << 20, used  # its 20000 copies would be 20000 steps x 7 units x 6 KiB = 820 MiB
    del m
    ids = synth.token_ids(78, "steps", (11, 70), 131)
    lens = np.array([1, 70, 17, 33, 40, 16, 69, 2, 50, 64, 65], np.int32)
    for D, H, heads, blocks in ((32, 64, 0, [(7, 2, 1), (5, 2, 1)]), (128, 256, 4, [(3, 2, 1), (9, 2, 2), (6, 2, 1)])):
        spec = tiny_spec(blocks, V=131, D=D, H=H, heads=heads, window=64 if heads else 0, context=128, tied=False)
        m = Model(uniform_model_bytes(spec, seed=7, scale=0.25))
        out = {}
        for mode in ("auto", "limbs"):
            engine_option("operands", mode)
            s = m.sessions(len(ids), 128)
            out[mode] = m.forward_batch(ids)["logits"], s.prefill(ids, lens)[0], s.step(ids[:, 0])[0]
        for a, b in zip(out["auto"], out["limbs"]):
            assert_close(a, b, rtol=2e-5, what=f"{blocks}")


# D, H, heads, blocks, T, sequences, whether the one-kernel body is the faster one there: both sides of the line
FILL = [
    (128, 256, 0, [(1, 2, 1)] * 2, 1, 2048, True),
    (128, 256, 0, [(1, 2, 1)] * 2, 1, 8192, False),
    (128, 128, 0, [(1, 2, 1)] * 2, 4, 65536, False),
    (128, 128, 0, [(1, 2, 1)] * 2, 6, 65536, True),
    (32, 64, 0, [(2, 2, 1)], 1, 8192, True),
    (32, 64, 0, [(2, 2, 1)], 1, 32768, False),
    (96, 160, 4, [(1, 2, 1)] * 2, 1, 8192, True),
    (96, 160, 4, [(1, 2, 1)] * 2, 1, 32768, False),
    (96, 160, 4, [(1, 2, 1)] * 2, 3, 32768, True),
]


@pytest.mark.parametrize("D,H,heads,blocks,T,B,one", FILL)
def test_short_sequences_take_the_faster_body(D, H, heads, blocks, T, B, one):
    """Many sequences of a few tokens leave the kernel's tiles mostly empty and take the layered body (forward, prefill
    and scoring with a short context), a few of them or longer ones the kernel; the same outputs either way."""
    spec = tiny_spec(blocks, V=131, D=D, H=H, heads=heads, window=64 if heads else 0, context=128, tied=False)
    data = uniform_model_bytes(spec, seed=8, scale=0.3)
    m, om = Model(data), oracle_model(data)
    ids = synth.token_ids(79, f"fill{D}{T}", (B, T), 131)
    got, prof = _classes(m, lambda: m.forward_batch(ids)["logits"])
    assert ("sequence_body" in prof) == one and ("gemm_glu" in prof) != one, prof
    for b in (0, 1, 15, 16, B // 2, B - 1):
        assert_close(got[b], om.forward_all(ids[b:b + 1])[0], what=f"sequence {b}")
    if B <= 8192:
        s = m.sessions(B, 128)
        (lg, _, _), prof = _classes(m, lambda: s.prefill(ids))
        assert ("sequence_body" in prof) == one, prof
        assert_close(lg, got[:, -1], rtol=2e-5, what="prefill")
        nexts = ids[::-1, 0].copy()
        after = s.step(nexts)[0]
        for b in (0, 17, B - 1):
            assert_close(after[b], om.call(np.append(ids[b], nexts[b])), what=f"step of session {b}")
    doc = ids.ravel()[:B + T - 1]  # about B windows of T tokens
    (lp,), prof = _classes(m, lambda: score_sequences(m, [doc], T))
    assert ("sequence_body" in prof) == one, prof
    for t in (1, 2, len(doc) // 2, len(doc) - 1):
        want = om.call(doc[max(0, t - T):t]).astype(np.float64)
        want = want[doc[t]] - want.max() - np.log(np.exp(want - want.max()).sum())
        assert abs(lp[t - 1] - want) <= 1e-4 * max(1.0, abs(want)), t


@pytest.mark.parametrize("shape", [SHAPES[0], SHAPES[6], SHAPES[8], SHAPES[9], (128, 160, 4, 64, [(1, 2, 1)] * 2)])
def test_profile_counts_what_runs(shape):
    """The profiler's work of the kernel, wave by wave as it runs: a 16-token tile past a sequence's end does nothing, and
    the last block's products run only where a row the head reads depends on them."""
    D, H, heads, window, blocks = shape
    m = Model(_build(shape))
    Dp = -(-D // 64) * 64

    def want(seqs):
        ops = out = 0
        for n, first, count in seqs:
            for t in range(-(-n // 16)):
                tokens = min(16, n - 16 * t)
                read = 16 * t < first + count and 16 * t + 15 >= first
                key = 16 * t < first + count and 16 * t + 15 >= first - window + 1
                for i, (steps, _, _) in enumerate(blocks):
                    last = i + 1 == len(blocks)
                    for st in range(steps):
                        ops += 2 * tokens * D * D
                        if not last or st + 1 < steps or (key if heads else read):
                            ops += 2 * tokens * 8 * D * H
                    if heads:
                        ops += 2 * tokens * D * D * (3 * (not last or key) + (not last or read))
            out += 4 * n + count * (4 + 3 * Dp)
        return out, ops

    def check(fn, seqs):
        prof = _classes(m, fn)[1]["sequence_body"]
        assert prof[2:] == want(seqs), (shape, seqs[:3])

    ids = synth.token_ids(80, "prof", (9, 128), 131)
    check(lambda: m.forward_batch(ids), [(128, 0, 128)] * 9)
    check(lambda: m.forward_batch(ids[:, :33].copy()), [(33, 0, 33)] * 9)
    for n in (1, 16, 17, 45, 128):
        check(lambda: m.call(ids[0, :n]), [(n, n - 1, 1)])
    lens = np.array([1, 16, 17, 33, 64, 65, 80, 127, 128], np.int32)
    check(lambda: m.sessions(9, 128).prefill(ids, lens), [(n, n - 1, 1) for n in lens.tolist()])
    # a first window of the context's length, scored at all its targets, then one of that length per later target
    check(lambda: score_sequences(m, [ids[0]], 40), [(40, 0, 40)] + [(40, 39, 1)] * 87)
