"""Timed cases of the batched INT8 engine: what a program that holds a model has it do, through the public entry
points of mignon_ai_amd, at the smallest sizes (one streaming token, one prefix, one row of a product), ordinary
ones and the largest, with aligned and ragged lengths.

kinds
  append    Session.append: one streaming session's next-token logits on the host (an interactive reply)
  call      Model.call: the next-token logits of one prefix, nothing kept between calls (an infer.LogitsFn)
  forward   Model.forward_batch_device: teacher-forced scoring of B sequences of T tokens (logits, log-probabilities,
            probabilities, bits per token)
  prefill   Sessions.prefill: prompts of unequal length taken in by a set of sessions, the logits after each
  step      Sessions.step_device: one token for every session of a set whose windows are full
  decode    Sessions.decode_greedy_device: prompts in, greedy replies and their probabilities out
  score     score_sequences: held-out scoring of documents of unequal length, each target from its own window
  gemm      gemm_i8_device: the standalone INT8 product with per-channel scales

A model is a file of seeded weights (every matrix normal, quantised per tensor as quant.NewTensorF32 does), loaded once
and kept, as a program keeps it; the inputs come from the seed.
"""
import math

import numpy as np
import torch

from mignon_ai_amd import Model, gemm_i8_device, mgnn, synth
from mignon_ai_amd.evaluate import score_sequences

# name: (V, D, H, blocks as (steps, dilation base, initial dilation), heads, window). tiny, medium, wide and large are
# the benchmark's configurations, base the shape of the trained order-search model, deep an odd-sized one whose blocks
# take several rule steps.
MODELS = {
    "tiny": (512, 32, 64, ((2, 2, 1),), 0, 0),
    "base": (2048, 96, 160, ((1, 2, 1),) * 2, 4, 64),
    "medium": (2048, 128, 256, ((1, 2, 1),) * 2, 4, 64),
    "deep": (1000, 160, 288, ((2, 2, 1), (2, 2, 2)), 5, 48),
    "wide": (4096, 256, 512, ((1, 2, 1),) * 3, 8, 64),
    "large": (8192, 384, 1024, ((1, 2, 1),) * 4, 6, 64),
}
CONTEXT = 128
PLAIN = ("tiny", "base", "medium", "deep", "wide", "large")


def listed():
    return [
        # one interactive session: each token waits for the one before it
        {"name": "append", "kind": "append", "model": "medium", "prompt": 64},
        # a caller without a session asks for the token after a short prefix
        {"name": "call", "kind": "call", "model": "base", "n": 45},
        # a small model over a small batch: latency and launches
        {"name": "forward_tiny", "kind": "forward", "model": "tiny", "B": 64, "T": 128, "out": "logits"},
        # sequences as long as the texts happen to be
        {"name": "forward_ragged", "kind": "forward", "model": "base", "B": 300, "T": 100, "out": "logits"},
        # the ordinary scoring batch
        {"name": "forward_medium", "kind": "forward", "model": "medium", "B": 1024, "T": 128, "out": "logits"},
        # full distributions of the largest model
        {"name": "forward_large", "kind": "forward", "model": "large", "B": 2048, "T": 128, "out": "probs"},
        # a serving set takes in prompts of 1 to 90 tokens
        {"name": "prefill", "kind": "prefill", "model": "wide", "S": 400, "T": 90},
        # a step of a few sessions at once, and of a busy server's
        {"name": "step_few", "kind": "step", "model": "wide", "S": 24},
        {"name": "step_many", "kind": "step", "model": "base", "S": 1500},
        # a batch of whole greedy replies
        {"name": "decode", "kind": "decode", "model": "wide", "S": 4096, "T": 32, "G": 64},
        # held-out scoring of documents, most shorter than the window, some longer
        {"name": "score", "kind": "score", "model": "medium", "docs": 60, "longest": 400},
        # the standalone product at the benchmark's size
        {"name": "gemm", "kind": "gemm", "M": 262144, "K": 384, "N": 512},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("append", "call", "forward", "forward", "forward", "prefill", "step", "step", "decode", "score",
                       "gemm", "gemm"))
    c = {"kind": kind}
    if kind == "gemm":
        c.update(M=_log(rng, 1, 262144), K=_log(rng, 16, 1536), N=_log(rng, 16, 4096))
        while c["M"] * c["N"] > 1 << 27:
            c["M"] = max(1, c["M"] // 2)
        return c
    name = c["model"] = rng.choice(PLAIN)
    if kind == "append":
        c["prompt"] = _log(rng, 1, CONTEXT)
    elif kind == "call":
        c["n"] = _log(rng, 1, CONTEXT)
    elif kind == "forward":
        c["T"] = rng.choice((128, _log(rng, 8, 128), _log(rng, 8, 128)))
        most = {"tiny": 1 << 20, "base": 1 << 18, "medium": 1 << 18, "deep": 1 << 18, "wide": 1 << 17,
                "large": 1 << 17}[name]
        c["B"] = max(1, _log(rng, 16, most) // c["T"])
        c["out"] = rng.choice(("logits", "probs", "bits"))
    elif kind == "prefill":
        c.update(S=_log(rng, 1, 1000), T=_log(rng, 4, CONTEXT))
    elif kind == "step":
        c["S"] = _log(rng, 1, 4096)
    elif kind == "decode":
        c.update(S=_log(rng, 1, 700 if name == "large" else 2048), T=_log(rng, 4, 64), G=_log(rng, 8, 64))
    else:
        c.update(docs=_log(rng, 1, 20 if name == "large" else 100), longest=_log(rng, 16, 300))
    return c


# ---- models ------------------------------------------------------------------------------------------------------
def _spec(name):
    V, D, H, blocks, heads, window = MODELS[name]
    return synth.ModelSpec(V=V, D=D, H=H, blocks=[synth.BlockSpec(*b) for b in blocks], heads=heads, window=window,
                           context=CONTEXT)


def _weights(name):
    """Checkpoint arrays: int8 matrices with their scales, fp32 vectors."""
    V, D, H, blocks, heads, _ = MODELS[name]
    rng = np.random.default_rng(20240 + PLAIN.index(name))

    def matrix(rows, cols, gain=1.0):
        w = rng.standard_normal(rows * cols, np.float32) * np.float32(gain / math.sqrt(cols))
        s = np.float32(np.abs(w).max() / np.float32(127))
        return np.clip(np.rint(w / s), -127, 127).astype(np.int8), s

    def vector(n, mean, std):
        return (mean + std * rng.standard_normal(n)).astype(np.float32)

    q = {}
    q["embed"], q["embed.scale"] = matrix(V, D, 2.0)
    for b in range(len(blocks)):
        p = "b%d." % b
        q[p + "w1"], q[p + "w1.scale"] = matrix(2 * H, 3 * D)
        q[p + "w2"], q[p + "w2.scale"] = matrix(2 * D, H)
        q[p + "wsel"], q[p + "wsel.scale"] = matrix(D, D)
        q[p + "b1"] = vector(2 * H, 0, 0.1)
        q[p + "b2"] = np.concatenate([vector(D, 0, 0.1), vector(D, -1.386, 0.1)])
        q[p + "gamma"] = vector(D, 1, 0.1)
        if heads:
            q[p + "attn_norm"] = vector(D, 1, 0.1)
            q[p + "qkv"], q[p + "qkv.scale"] = matrix(3 * D, D)
            q[p + "out"], q[p + "out.scale"] = matrix(D, D, 0.5)
    q["final_norm"] = vector(D, 1, 0.1)
    q["head_b"] = vector(V, 0, 0.1)
    return q


_models = {}


def _model(name):
    if name not in _models:
        _models[name] = Model(mgnn.encode(_spec(name), _weights(name)))
    return _models[name]


def _ids(rng, shape, V):
    """Token ids with the skew of text: rank r about as often as 1 / r."""
    u = rng.random(shape)
    return np.minimum((np.power(float(V + 1), u) - 1).astype(np.int64), V - 1).astype(np.int32)


def _outputs(c):
    return {"logits": ("logits", "logprob"), "probs": ("probs", "bits"), "bits": ("logprob", "bits")}[c["out"]]


def _lengths(c):
    """Document lengths: most short, the longest last."""
    rng = np.random.default_rng([c["docs"], c["longest"]])
    return [max(2, int(c["longest"] * rng.random() ** 2)) for _ in range(c["docs"] - 1)] + [c["longest"]]


def _inputs(c, seed):
    """What the seed decides, on the host."""
    rng = np.random.default_rng([int(seed), 7])
    kind = c["kind"]
    if kind == "gemm":
        return {"A": rng.integers(-127, 128, (c["M"], c["K"]), np.int8),
                "W": rng.integers(-127, 128, (c["N"], c["K"]), np.int8),
                "scale": (1e-3 + 9e-3 * rng.random(c["N"])).astype(np.float32)}
    V = MODELS[c["model"]][0]
    if kind == "append":
        return {"prompt": _ids(rng, c["prompt"], V), "next": _ids(rng, 64, V)}
    if kind == "call":
        return {"ids": _ids(rng, c["n"], V)}
    if kind == "forward":
        return {"ids": _ids(rng, (c["B"], c["T"]), V)}
    if kind == "score":
        return {"docs": [_ids(rng, n, V) for n in _lengths(c)]}
    if kind == "step":
        return {"ids": _ids(rng, (c["S"], CONTEXT // 2), V), "lens": np.full(c["S"], CONTEXT // 2, np.int32),
                "next": _ids(rng, c["S"], V)}
    lens = rng.integers(1, c["T"] + 1, c["S"]).astype(np.int32)  # prefill, decode
    if kind == "decode":
        lens[:] = c["T"]
    lens[0] = c["T"]
    return {"ids": _ids(rng, (c["S"], c["T"]), V), "lens": lens}


def prepare(case, seed):
    c, x = case, _inputs(case, seed)
    kind, s = c["kind"], {"kind": case["kind"]}
    if kind == "gemm":
        s.update({k: torch.from_numpy(v).cuda() for k, v in x.items()})
        s["C"] = torch.empty((c["M"], c["N"]), dtype=torch.float32, device="cuda")
        s["stream"] = torch.cuda.current_stream().cuda_stream
        return s
    m = s["model"] = _model(c["model"])
    V = m.vocab_size()
    if kind == "append":
        s["session"] = m.new_session(CONTEXT)
        s["session"].prefill(x["prompt"])
        s["next"], s["at"] = x["next"].tolist(), 0
    elif kind == "call":
        s["ids"] = x["ids"]
    elif kind == "forward":
        s["ids"] = torch.from_numpy(x["ids"]).cuda()
        B, T = s["ids"].shape
        shape = {"logits": (B, T, V), "probs": (B, T, V), "logprob": (B, T), "bits": (B,)}
        s["out"] = {k: torch.empty(shape[k], dtype=torch.float32, device="cuda") for k in _outputs(c)}
    elif kind == "prefill":
        s["sessions"], s["ids"], s["lens"] = m.sessions(c["S"], CONTEXT), x["ids"], x["lens"]
    elif kind == "step":
        s["sessions"] = m.sessions(c["S"], CONTEXT)
        s["sessions"].prefill(x["ids"], x["lens"], logits=False)
        s["next"] = torch.from_numpy(x["next"]).cuda()
        s["out"] = {"logits": torch.empty((c["S"], V), dtype=torch.float32, device="cuda"),
                    "argmax": torch.empty(c["S"], dtype=torch.int32, device="cuda"),
                    "prob": torch.empty(c["S"], dtype=torch.float64, device="cuda")}
    elif kind == "decode":
        s["sessions"] = m.sessions(c["S"], CONTEXT)
        s["ids"], s["lens"] = torch.from_numpy(x["ids"]).cuda(), torch.from_numpy(x["lens"]).cuda()
        s["out"] = {"ids": torch.empty((c["S"], c["G"]), dtype=torch.int32, device="cuda"),
                    "probs": torch.empty((c["S"], c["G"]), dtype=torch.float64, device="cuda")}
        s["G"] = c["G"]
    else:
        s["docs"] = x["docs"]
    torch.cuda.synchronize()  # the model works on a stream of its own
    return s


def run(s):
    kind = s["kind"]
    if kind == "gemm":
        gemm_i8_device(s["A"], s["W"], s["scale"], s["C"], None, s["stream"])
        return s["C"]
    if kind == "append":
        token = s["next"][s["at"] % len(s["next"])]
        s["at"] += 1
        return s["session"].append(token)
    if kind == "call":
        return s["model"].call(s["ids"])
    if kind == "forward":
        s["model"].forward_batch_device(s["ids"], **s["out"])
        return s["out"]
    if kind == "prefill":
        logits, argmax, prob = s["sessions"].prefill(s["ids"], s["lens"])
        return {"logits": logits, "argmax": argmax, "prob": prob}
    if kind == "step":
        s["sessions"].step_device(s["next"], s["out"]["logits"], s["out"]["argmax"], s["out"]["prob"])
        return s["out"]
    if kind == "decode":
        s["sessions"].decode_greedy_device(s["ids"], s["lens"], s["G"], s["out"]["ids"], s["out"]["probs"])
        return s["out"]
    return np.concatenate(score_sequences(s["model"], s["docs"], CONTEXT))


# ---- what a pass cannot do without -------------------------------------------------------------------------------
def _per_token(name):
    """(multiply-adds of one position's body, of its head, attention's per attended key, weight bytes)"""
    V, D, H, blocks, heads, _ = MODELS[name]
    steps = sum(b[0] for b in blocks)
    body = steps * (D * D + 6 * D * H + 2 * D * H) + (len(blocks) * 4 * D * D if heads else 0)
    return body, D * V, (2 * D * len(blocks) if heads else 0), body + D * V


def work(case):
    c, kind = case, case["kind"]
    if kind == "gemm":
        M, K, N = c["M"], c["K"], c["N"]
        return {"bytes": M * K + N * K + 4 * N + 4 * M * N, "flops": 2 * M * K * N}
    V, D, _, blocks, heads, window = MODELS[c["model"]]
    body, head, per_key, weights = _per_token(c["model"])
    span = min(window or CONTEXT, CONTEXT)
    ring = 2 * 4 * D * span * len(blocks) if heads else 0  # one session's keys and values

    def pair(positions, heads_run, keys, extra):
        return {"bytes": weights + 4 * positions + extra, "flops": 2 * (positions * body + heads_run * head + keys * per_key)}

    def keys_of(n):  # keys attended by the positions 0 .. n - 1
        return sum(min(t + 1, span) for t in range(n))

    if kind == "append":
        return pair(1, 1, span, ring + 4 * V)
    if kind == "call":
        return pair(c["n"], 1, keys_of(c["n"]), 4 * V)
    if kind == "forward":
        B, T = c["B"], c["T"]
        out = {"logits": 4 * B * T * (V + 1), "probs": 4 * B * T * V + 4 * B, "bits": 4 * B * T + 4 * B}[c["out"]]
        return pair(B * T, B * T, B * keys_of(T), out)
    if kind == "step":
        return pair(c["S"], c["S"], c["S"] * span, c["S"] * (ring + 4 * V + 12))
    if kind == "prefill":
        n = c["S"] * (c["T"] + 1) // 2
        return pair(n, c["S"], n * keys_of(c["T"]) / c["T"], c["S"] * (4 * V + 12))
    if kind == "decode":
        n = c["S"] * (c["T"] + c["G"] - 1)
        keys = c["S"] * keys_of(c["T"] + c["G"] - 1)
        seen = c["S"] * sum(min(c["T"] + k, span) for k in range(c["G"] - 1))
        return pair(n, c["S"] * c["G"], keys, (seen * 8 * D * len(blocks) if heads else 0) + 12 * c["S"] * c["G"])
    lens = _lengths(c)
    n = sum(min(L - 1, CONTEXT) + max(0, L - 1 - CONTEXT) * CONTEXT for L in lens)
    return pair(n, sum(lens) - len(lens), n * keys_of(CONTEXT) / CONTEXT, 4 * sum(lens))


def tolerance(case):
    # Whole-number products of at most 1536 terms below 2^24 are exact, and each is scaled once.
    if case["kind"] == "gemm":
        return "exact"
    # Two kernel selections of the engine (and 32-bit sums in another order) differ by about 1e-6 in the logits of these
    # models; "differ" is for greedy choices between tokens whose logits agree to that many digits. A reply that takes
    # another token there is another reply from that token on.
    if case["kind"] == "decode":
        return {"rel": 1e-2, "max": 0.99, "differ": 4e-3}
    return {"rel": 1e-5, "max": 1e-3, "differ": 1e-3}


# ---- the same in 64 bits -----------------------------------------------------------------------------------------
class _Exact:
    """The model in float64 torch: whole sequences, one rule step at a time."""

    def __init__(self, name):
        self.V, self.D, self.H, self.blocks, self.heads, self.window = MODELS[name]
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        q = _weights(name)
        shape = {"embed": (self.V, self.D), "w1": (2 * self.H, 3 * self.D), "w2": (2 * self.D, self.H),
                 "wsel": (self.D, self.D), "qkv": (3 * self.D, self.D), "out": (self.D, self.D)}
        self.w = {}
        for k, v in q.items():
            if k.endswith(".scale"):
                continue
            t = torch.from_numpy(np.asarray(v)).to(self.dev).double()
            kind = k.split(".")[-1]
            if k + ".scale" in q:
                t = t.reshape(shape[kind]) * float(q[k + ".scale"])
            self.w[k] = t
        # ca.ComputeSelectiveLatchBaseLogits: decay 2^(-1/T_d), T_d geometric from 1.5 to 64 tokens, in float32
        d = np.arange(self.D, dtype=np.float64)
        td = 1.5 * (64 / 1.5) ** (d / max(self.D - 1, 1))
        lam = np.float32(2.0 ** (-1.0 / td)).astype(np.float64)
        self.base = torch.from_numpy(np.log(lam / (1 - lam)).astype(np.float32)).to(self.dev).double()

    @staticmethod
    def sig(x):
        y = torch.sigmoid(x)
        return torch.where(x > 15, torch.ones_like(y), torch.where(x < -15, torch.zeros_like(y), y))

    @staticmethod
    def norm(x, g):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * g

    def body(self, ids):
        B, T = ids.shape
        D, H = self.D, self.H
        cur = self.w["embed"][ids]
        block_in = cur
        for b, (steps, dil_base, dil0) in enumerate(self.blocks):
            p = "b%d." % b
            if b:
                block_in = block_in + cur
                cur = block_in
            for st in range(steps):
                dil = min(dil0 * dil_base ** st, 32)
                n = self.norm(cur, self.w[p + "gamma"])
                lam = self.sig(n @ self.w[p + "wsel"].T + self.base)
                g, G = torch.zeros((B, D), dtype=torch.float64, device=self.dev), torch.empty_like(n)
                for t in range(T):
                    g = lam[:, t] * g + (1 - lam[:, t]) * n[:, t]
                    G[:, t] = g
                left = torch.zeros_like(n)
                if dil < T:
                    left[:, dil:] = n[:, :T - dil]
                hid = torch.cat([n, left, G], -1) @ self.w[p + "w1"].T + self.w[p + "b1"]
                h = hid[..., :H] * self.sig(hid[..., H:])
                o = h @ self.w[p + "w2"].T + self.w[p + "b2"]
                gate = self.sig(o[..., D:])
                cur = (1 - gate) * cur + gate * o[..., :D]
            if self.heads:
                dh = D // self.heads
                qkv = self.norm(cur, self.w[p + "attn_norm"]) @ self.w[p + "qkv"].T
                qkv = qkv.view(B, T, 3, self.heads, dh).permute(2, 0, 3, 1, 4).contiguous()
                s = qkv[0] @ qkv[1].transpose(-1, -2).contiguous() / math.sqrt(dh)
                i = torch.arange(T, device=self.dev)
                far = self.window or CONTEXT
                seen = (i[None, :] <= i[:, None]) & (i[None, :] > i[:, None] - far)
                a = torch.softmax(s.masked_fill(~seen, -math.inf), -1) @ qkv[2]
                cur = cur + a.permute(0, 2, 1, 3).reshape(B, T, D) @ self.w[p + "out"].T
        return self.norm(cur, self.w["final_norm"])

    def logits(self, rows):
        return rows @ self.w["embed"].T + self.w["head_b"]

    def rows(self, ids, at=None):
        """Normalised final rows of [B, T] ids, in pieces; with `at`, of position at[b] only."""
        ids = torch.from_numpy(np.ascontiguousarray(ids)).to(self.dev).long()
        piece = max(1, (1 << 15) // ids.shape[1])
        for i in range(0, len(ids), piece):
            r = self.body(ids[i:i + piece])
            if at is not None:
                a = torch.from_numpy(np.asarray(at[i:i + piece])).to(self.dev).long()
                r = r[torch.arange(len(r), device=self.dev), a]
            yield i, r


def exact(case, seed):
    c, x = case, _inputs(case, seed)
    kind = c["kind"]
    if kind == "gemm":
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        A, W, s = (torch.from_numpy(x[k]).to(dev).double() for k in ("A", "W", "scale"))
        return A @ W.T * s
    if kind == "decode":
        return None  # the greedy choices are the engine's own
    e = _Exact(c["model"])
    if kind in ("append", "call"):
        ids = x["ids"] if kind == "call" else np.concatenate([x["prompt"], x["next"][:1]])
        r = torch.cat([r for _, r in e.rows(ids[None, :], [len(ids) - 1])])
        return e.logits(r)[0].cpu().numpy()
    if kind in ("prefill", "step"):
        ids, at = x["ids"], x["lens"] - 1
        if kind == "step":
            ids, at = np.concatenate([ids, x["next"][:, None]], 1), x["lens"]
        lg = e.logits(torch.cat([r for _, r in e.rows(ids, at)]))
        return {"logits": lg, "argmax": None, "prob": torch.softmax(lg, -1).max(-1).values}
    if kind == "forward":
        ids = torch.from_numpy(x["ids"]).to(e.dev).long()
        B, T = ids.shape
        out = {k: torch.empty((B, T, e.V) if k in ("logits", "probs") else (B, T), dtype=torch.float64, device=e.dev)
               for k in _outputs(c) if k != "bits"}
        lp = torch.full((B, T), math.nan, dtype=torch.float64, device=e.dev)
        for i, r in e.rows(x["ids"]):
            lg = e.logits(r)
            lse = torch.logsumexp(lg, -1)
            n = len(r)
            if T > 1:
                lp[i:i + n, :-1] = lg[:, :-1].gather(-1, ids[i:i + n, 1:, None])[..., 0] - lse[:, :-1]
            if "logits" in out:
                out["logits"][i:i + n] = lg
            if "probs" in out:
                out["probs"][i:i + n] = torch.exp(lg - lse[..., None])
        if "logprob" in out:
            out["logprob"] = lp
        if "bits" in _outputs(c):
            out["bits"] = -lp[:, :-1].mean(-1) / math.log(2) if T > 1 else torch.zeros(B, dtype=torch.float64, device=e.dev)
        return out
    # score: target t of a document from the (at most) CONTEXT tokens before it
    got = [np.empty(len(d) - 1) for d in x["docs"]]
    rows = []
    for k, d in enumerate(x["docs"]):
        n = min(len(d) - 1, CONTEXT)
        rows.append((d[:n], [(k, j, j) for j in range(n)], d))
        rows += [(d[t - CONTEXT:t], [(k, t - 1, CONTEXT - 1)], d) for t in range(CONTEXT + 1, len(d))]
    ids = np.zeros((len(rows), CONTEXT), np.int32)
    for i, (r, _, _) in enumerate(rows):
        ids[i, :len(r)] = r
    for i, r in e.rows(ids):
        pick = [(a, pos, d[j + 1], k, j) for a in range(len(r)) for k, j, pos in rows[i + a][1] for d in (rows[i + a][2],)]
        a, pos, tgt = (torch.tensor([p[n] for p in pick], device=e.dev).long() for n in range(3))
        lg = e.logits(r[a, pos])
        lp = (lg.gather(-1, tgt[:, None])[:, 0] - torch.logsumexp(lg, -1)).cpu().numpy()
        for p, v in zip(pick, lp):
            got[p[3]][p[4]] = v
    return np.concatenate(got)
