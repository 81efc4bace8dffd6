"""Timed cases of the decode-path ops: inputs, one call, its work and its result in 64 bits.

``listed()`` is a fixed set over the ops a decoder-serving program calls
(Qwen3 0.6B / VL-2B / 8B layer shapes, the per-op configurations of
``ezops.workloads``); ``draw(rng)`` makes one more case of the same ops with
sizes drawn over the whole range.  Every case is a dict of plain values with
an ``op`` key.  ``prepare`` builds the tensors and the op object, ``run`` is
one forward call of the op.

Values are synthetic: activations and caches ~ N(0, 1), weights ~ N(0, 0.02),
norm weights ~ N(1, 0.1), RoPE theta 1e6.  Ragged lengths are seeded by the
case's ``lens_seed``, so they are part of the case, not of the inputs.
"""

from __future__ import annotations

import random
import sys
from pathlib import Path

import torch

_PKG = str(Path(__file__).resolve().parent.parent / "ez-ops_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import ezops  # noqa: E402
from ezops.ops.fused_qk_norm_rope import rope_tables  # noqa: E402

BF = torch.bfloat16
F64 = torch.float64
EPS = 1e-6
THETA = 1e6
VOCAB = 151936

MODELS = {
    "0.6b": dict(hidden_size=1024, intermediate_size=3072, num_heads=16, head_dim=128, num_kv_heads=8),
    "vl-2b": dict(hidden_size=2048, intermediate_size=6144, num_heads=16, head_dim=128, num_kv_heads=8),
    "8b": dict(hidden_size=4096, intermediate_size=12288, num_heads=32, head_dim=128, num_kv_heads=8),
}


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest call: the final norm of a 64-sequence decode step (latency)
        dict(name="rmsnorm_64x4096", op="rmsnorm", rows=64, dim=4096, dtype="bf16"),
        # probabilities over the vocabulary for sampling, one row per sequence
        dict(name="softmax_64xvocab", op="softmax", rows=64, dim=VOCAB),
        # a whole-tensor reduction of odd length
        dict(name="sum_100000007", op="sum", n=100000007),
        # one projection of a single sequence
        dict(name="gemv_4096x4096", op="gemv", N=4096, K=4096),
        # decode attention of a full batch over long contexts, contiguous cache
        dict(name="attn_b32_s8192", op="attn", batch=32, heads=32, kv_heads=8, head_dim=128, seq=8192, min_len=8192,
             lens_seed=0, page=0),
        # one decode layer: a single long conversation
        dict(name="layer_8b_b1", op="layer", model="8b", batch=1, seq=16384, min_len=9291, max_len=9291, lens_seed=0,
             page=0),
        # one decode layer of a small server: ragged batch over a paged cache
        dict(name="layer_8b_b16_paged", op="layer", model="8b", batch=16, seq=16384, min_len=1024, max_len=16384,
             lens_seed=4, page=64),
        # one decode layer at high concurrency: many shorter conversations
        dict(name="layer_8b_b64_paged", op="layer", model="8b", batch=64, seq=4096, min_len=256, max_len=4096,
             lens_seed=5, page=128),
        # a whole decode step of the small model, from hidden state to logits
        dict(name="step_0.6b_b4", op="step", model="0.6b", batch=4, layers=28, seq=2048, min_len=200, max_len=2048,
             lens_seed=6, page=0),
        # prefill: one fresh long prompt
        dict(name="prefill_8b_4096", op="prefill", model="8b", seqs=1, seq=4096, min_new=4096, max_new=4096,
             max_past=0, lens_seed=0, page=0),
        # prefill: short ragged prompts, some on top of cached prefixes, paged cache
        dict(name="prefill_8b_ragged", op="prefill", model="8b", seqs=6, seq=4096, min_new=17, max_new=260,
             max_past=2000, lens_seed=7, page=64),
        # prefill attention of a very long prompt
        dict(name="prefill_attn_16384", op="prefill_attn", heads=32, kv_heads=8, seqs=1, seq=16384, min_new=16384,
             max_new=16384, max_past=0, lens_seed=0, page=0),
    ]


def _log(rng, lo, hi):
    """An integer in [lo, hi], uniform in its logarithm."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    op = rng.choice(["rmsnorm", "softmax", "sum", "gemv", "qk_rope", "attn", "attn", "ffn", "layer", "layer", "layer",
                     "step", "prefill", "prefill", "prefill", "prefill_attn"])
    seed = rng.randrange(1 << 20)
    if op == "rmsnorm":
        dim = _log(rng, 64, 16384)
        return dict(op=op, rows=_log(rng, 1, min(8192, (1 << 26) // dim)), dim=dim if rng.random() < 0.3 else -(-dim // 64) * 64,
                    dtype=rng.choice(["bf16", "f32"]))
    if op == "softmax":
        dim = _log(rng, 100, VOCAB)
        return dict(op=op, rows=_log(rng, 1, min(4096, (1 << 27) // dim)), dim=dim if rng.random() < 0.5 else -(-dim // 8) * 8)
    if op == "sum":
        return dict(op=op, n=_log(rng, 1000, 1 << 28))
    if op == "gemv":
        K = _log(rng, 256, 32768)
        return dict(op=op, N=_log(rng, 256, min(VOCAB, (1 << 28) // K)), K=K if rng.random() < 0.2 else -(-K // 64) * 64)
    if op == "qk_rope":
        return dict(op=op, batch=_log(rng, 1, 64), heads=rng.choice([16, 32]), kv_heads=8, head_dim=128,
                    seq=_log(rng, 128, 8192), lens_seed=seed)
    if op == "attn":
        kv, g = rng.choice([1, 2, 8]), rng.choice([1, 2, 4, 8, 16])
        page = rng.choice([0, 32, 64, 128])
        seq = _log(rng, 100, 32768)
        seq = -(-seq // page) * page if page else seq
        batch = _log(rng, 1, max(1, min(64, (1 << 18) * 8 // (kv * seq))))
        return dict(op=op, batch=batch, heads=kv * g, kv_heads=kv, head_dim=rng.choice([64, 128, 128]), seq=seq,
                    min_len=rng.choice([max(1, seq // 8), seq]), lens_seed=seed, page=page)
    if op == "ffn":
        return dict(op=op, model=rng.choice(list(MODELS)), batch=_log(rng, 1, 64))
    if op in ("layer", "step"):
        page = rng.choice([0, 32, 64, 256])
        seq = -(-_log(rng, 256, 16384) // 256) * 256
        batch = _log(rng, 1, min(64, (1 << 18) // seq))
        hi = rng.randint(seq // 2, seq)
        c = dict(op=op, model=rng.choice(list(MODELS)), batch=batch, seq=seq, min_len=rng.choice([max(1, hi // 8), hi]),
                 max_len=hi, lens_seed=seed, page=page)
        if op == "step":  # a few layers and the LM head
            c.update(model=rng.choice(["0.6b", "vl-2b"]), layers=rng.randint(2, 4), batch=min(batch, (1 << 16) // seq))
        return c
    # prefill of a chunk of new tokens: 1 to 8 sequences, about 40 to 4000 tokens in all
    seqs = rng.choice([1, 1, 2, 4, 8])
    hi = _log(rng, 40, 4000) // seqs + 1
    past = rng.choice([0, 0, 1000])
    page = rng.choice([0, 64, 256])
    c = dict(op=op, seqs=seqs, seq=-(-(hi + past) // 256) * 256, min_new=rng.choice([max(1, hi // 3), hi]), max_new=hi,
             max_past=past, lens_seed=seed, page=page)
    if op == "prefill":
        c["model"] = rng.choice(list(MODELS))
    else:
        c.update(heads=8 * rng.choice([1, 2, 4, 8]), kv_heads=8)
    return c


def _lens(c):
    """Per-sequence live lengths of a decode case."""
    r = random.Random(c["lens_seed"])
    return [r.randint(c["min_len"], c.get("max_len", c["seq"])) for _ in range(c["batch"])]


def _chunks(c):
    """(new tokens, cached tokens) per sequence of a prefill case."""
    r = random.Random(c["lens_seed"])
    new = [r.randint(c["min_new"], c["max_new"]) for _ in range(c["seqs"])]
    past = [min(r.randint(0, c["max_past"]), c["seq"] - n) if c["max_past"] and r.random() < 0.7 else 0 for n in new]
    return new, past


# ------------------------------------------------------------------- inputs
class _Gen:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, std=1.0, mean=0.0, dtype=BF):
        return torch.empty(*shape, dtype=dtype, device="cuda").normal_(mean, std, generator=self.g)

    def uniform(self, *shape):
        return torch.rand(*shape, generator=self.g, device="cuda")

    def pages(self, n_pages, shape):
        ids = torch.randperm(n_pages, generator=self.g, device="cuda")[: shape[0] * shape[1]]
        return ids.reshape(*shape).to(torch.int32)

    def cache(self, batch, kv, seq, D, page):
        shape = (batch * (seq // page), kv, page, D) if page else (batch, kv, seq, D)
        return self.normal(*shape), self.normal(*shape)

    def weights(self, m):
        HS, IS, D = m["hidden_size"], m["intermediate_size"], m["head_dim"]
        QR, KVR = m["num_heads"] * D, m["num_kv_heads"] * D
        w = [self.normal(QR + 2 * KVR, HS, std=0.02), self.normal(HS, QR, std=0.02),
             self.normal(2 * IS, HS, std=0.02), self.normal(HS, IS, std=0.02)]
        return w, [self.normal(n, std=0.1, mean=1.0) for n in (HS, D, D, HS)]


def _inputs(c, seed):
    """The case's tensors (a dict), in the order one generator draws them."""
    r, op = _Gen(seed), c["op"]
    if op == "rmsnorm":
        dt = BF if c["dtype"] == "bf16" else torch.float32
        d = dict(X=r.normal(c["rows"], c["dim"], dtype=dt), Out=torch.empty(c["rows"], c["dim"], dtype=dt, device="cuda"))
        if dt == BF:
            d["W"] = r.normal(c["dim"], std=0.1, mean=1.0)
        return d
    if op == "softmax":  # logits
        X = r.normal(c["rows"], c["dim"], std=3.0, dtype=torch.float32)
        return dict(X=X, Out=torch.empty_like(X))
    if op == "sum":  # non-negative terms (losses, probabilities): a well-conditioned sum
        return dict(A=r.uniform(c["n"]), Out=torch.empty(1, device="cuda"))
    if op == "gemv":
        return dict(A=r.normal(c["K"]), B=r.normal(c["N"], c["K"], std=0.02), C=torch.empty(c["N"], dtype=BF, device="cuda"))
    if op == "qk_rope":
        B, H, Hk, D, S = c["batch"], c["heads"], c["kv_heads"], c["head_dim"], c["seq"]
        d = dict(q=r.normal(B, H, D), k=r.normal(B, Hk, D), v=r.normal(B, Hk, D), qw=r.normal(D, std=0.1, mean=1.0),
                 kw=r.normal(D, std=0.1, mean=1.0))
        d["cos"], d["sin"] = rope_tables(S, D, THETA, "cuda")
        d["K"], d["V"] = r.cache(B, Hk, S, D, 0)
        return d
    if op == "attn":
        d = dict(Q=r.normal(c["batch"], c["heads"], 1, c["head_dim"]))
        d["K"], d["V"] = r.cache(c["batch"], c["kv_heads"], c["seq"], c["head_dim"], c["page"])
        if c["page"]:
            d["bt"] = r.pages(d["K"].shape[0], (c["batch"], c["seq"] // c["page"]))
        d["lens"] = torch.tensor(_lens(c), dtype=torch.int32, device="cuda")
        return d
    if op == "prefill_attn":
        new, past = _chunks(c)
        d = dict(Q=r.normal(sum(new), c["heads"], 128))
        d["K"], d["V"] = r.cache(c["seqs"], c["kv_heads"], c["seq"], 128, c["page"])
        if c["page"]:
            d["bt"] = r.pages(d["K"].shape[0], (c["seqs"], c["seq"] // c["page"]))
        return d
    m = MODELS[c["model"]]
    HS = m["hidden_size"]
    if op == "ffn":
        (_, Wo, Wgu, Wd), (_, _, _, pw) = r.weights(m)
        IS = m["intermediate_size"]
        return dict(attn=r.normal(c["batch"], Wo.shape[1]), residual=r.normal(c["batch"], HS), Wo=Wo, pw=pw,
                    Wg=Wgu[:IS].clone(), Wu=Wgu[IS:].clone(), Wd=Wd)
    seqs = c["seqs"] if op == "prefill" else c["batch"]
    T = sum(_chunks(c)[0]) if op == "prefill" else c["batch"]
    n_layers = c.get("layers", 1)
    d = dict(hidden=r.normal(T, HS), layers=[])
    page, seq = c["page"], c["seq"]
    shape = (seqs * (seq // page), m["num_kv_heads"], page, 128) if page else (seqs, m["num_kv_heads"], seq, 128)
    d["kv"] = r.normal(n_layers, 2, *shape)  # every layer's K and V cache in one allocation
    for i in range(n_layers):
        w, nw = r.weights(m)
        d["layers"].append((d["kv"][i, 0], d["kv"][i, 1], *w, *nw))
    d["cos"], d["sin"] = rope_tables(seq, 128, THETA, "cuda")
    d["bt"] = r.pages(shape[0], (seqs, seq // page)) if page else None
    if op == "step":
        d["final_w"] = r.normal(HS, std=0.1, mean=1.0)
        d["lm_head"] = r.normal(VOCAB, HS, std=0.02)
    return d


def _op(c):
    op = c["op"]
    if op == "rmsnorm":
        bf = c["dtype"] == "bf16"
        return ezops.RmsNormOp(c["rows"], c["dim"], "hip", dtype=BF if bf else torch.float32, weighted=bf)
    if op == "softmax":
        return ezops.SoftmaxOp(c["rows"], c["dim"], "hip")
    if op == "sum":
        return ezops.ReduceOp(c["n"], "hip")
    if op == "gemv":
        return ezops.GemvOp(c["N"], c["K"], "hip")
    if op == "qk_rope":
        r = random.Random(c["lens_seed"])
        pos = [r.randrange(c["seq"]) for _ in range(c["batch"])]
        return ezops.FusedQkNormRopeOp(c["batch"], c["heads"], c["head_dim"], c["seq"], pos, "hip", c["kv_heads"])
    if op == "attn":
        if c["page"]:
            return ezops.PagedAttnDecodeOp(c["batch"], c["heads"], c["kv_heads"], c["head_dim"], c["page"],
                                           c["seq"] // c["page"], backend="hip")
        return ezops.AttnDecodeOp(c["batch"], c["heads"], c["seq"], c["head_dim"], "hip", c["kv_heads"])
    if op == "prefill_attn":
        new, past = _chunks(c)
        return ezops.PrefillAttnOp(c["seqs"], c["heads"], c["kv_heads"], 128, c["seq"], new, past, "hip",
                                   page_size=c["page"] or None)
    m = MODELS[c["model"]]
    shape = (m["hidden_size"], m["intermediate_size"], m["num_heads"], m["head_dim"])
    if op == "ffn":
        return ezops.FusedOProjFfnOp(c["batch"], *shape, backend="hip")
    kw = dict(norm_weights=True, rope_theta=THETA, page_size=c["page"] or None)
    if op == "layer":
        return ezops.Qwen3DenseDecodeOp(c["batch"], c["seq"], *shape, "hip", m["num_kv_heads"], kv_lens=_lens(c), **kw)
    if op == "step":
        return ezops.Qwen3DecodeStepOp(c["batch"], c["seq"], *shape, c["layers"], "hip", m["num_kv_heads"],
                                       vocab_size=VOCAB, kv_lens=_lens(c), **kw)
    new, past = _chunks(c)
    return ezops.Qwen3PrefillOp(c["seqs"], c["seq"], *shape, new, past, "hip", m["num_kv_heads"], **kw)


def prepare(case, seed):
    d = _inputs(case, seed)
    d["op"], d["case"] = _op(case), case
    if case["op"] == "attn":
        d["max_len"] = max(_lens(case))
    return d


def run(s):
    c, op = s["case"], s["op"]
    kind = c["op"]
    if kind == "rmsnorm":
        op(s["X"], s["W"], s["Out"]) if "W" in s else op(s["X"], s["Out"])
        return s["Out"]
    if kind == "softmax":
        op(s["X"], s["Out"])
        return s["Out"]
    if kind == "sum":
        op(s["A"], s["Out"])
        return s["Out"]
    if kind == "gemv":
        op(s["A"], s["B"], s["C"])
        return s["C"]
    if kind == "qk_rope":
        q, k = op(s["q"], s["k"], s["v"], s["qw"], s["kw"], s["cos"], s["sin"], s["K"], s["V"])
        return q, k, s["K"], s["V"]
    if kind == "attn":
        if c["page"]:
            return op(s["Q"], s["K"], s["V"], s["bt"], s["lens"], s["max_len"])
        return op(s["Q"], s["K"], s["V"]) if c["min_len"] == c["seq"] else op(s["Q"], s["K"], s["V"], s["lens"])
    if kind == "prefill_attn":
        return op(s["Q"], s["K"], s["V"], *([s["bt"]] if c["page"] else []))
    if kind == "ffn":
        return op(s["attn"], s["residual"], s["Wo"], s["pw"], s["Wg"], s["Wu"], s["Wd"])
    if kind == "step":
        h, logits = op(s["hidden"], s["layers"], s["cos"], s["sin"], s["final_w"], s["lm_head"], s["bt"])
        return h, logits, s["kv"]
    out = op(s["hidden"], *s["layers"][0], s["cos"], s["sin"], *([s["bt"]] if c["page"] else []))
    return out, s["kv"]


# --------------------------------------------------------------------- work
def work(case):
    c, op = case, case["op"]
    if op == "rmsnorm":
        n, e = c["rows"] * c["dim"], 2 if c["dtype"] == "bf16" else 4
        return dict(bytes=2 * n * e + (c["dim"] * 2 if e == 2 else 0), flops=4 * n)
    if op == "softmax":
        return dict(bytes=8 * c["rows"] * c["dim"], flops=5 * c["rows"] * c["dim"])
    if op == "sum":
        return dict(bytes=4 * c["n"] + 4, flops=c["n"])
    if op == "gemv":
        return dict(bytes=2 * (c["N"] * c["K"] + c["N"] + c["K"]), flops=2 * c["N"] * c["K"])
    if op == "qk_rope":
        q, k = c["batch"] * c["heads"] * 128, c["batch"] * c["kv_heads"] * 128
        return dict(bytes=2 * (2 * q + 5 * k) + 4 * 128 * c["batch"], flops=10 * (q + k))
    if op == "attn":
        n = sum(_lens(c))
        return dict(bytes=2 * (2 * c["kv_heads"] * c["head_dim"] * n + 2 * c["batch"] * c["heads"] * c["head_dim"]),
                    flops=4 * c["heads"] * c["head_dim"] * n)
    if op in ("prefill", "prefill_attn"):
        new, past = _chunks(c)
        T = sum(new)
        pairs = sum(n * p + n * (n + 1) // 2 for n, p in zip(new, past))
        if op == "prefill_attn":
            return dict(bytes=2 * 128 * (2 * T * c["heads"] + 2 * c["kv_heads"] * (T + sum(past))),
                        flops=4 * 128 * c["heads"] * pairs)
    m = MODELS[c["model"]]
    HS, IS, QR, KVR = m["hidden_size"], m["intermediate_size"], m["num_heads"] * 128, m["num_kv_heads"] * 128
    ffn = HS * QR + 3 * IS * HS
    if op == "ffn":
        B = c["batch"]
        return dict(bytes=2 * (ffn + B * (QR + 2 * HS)), flops=2 * B * ffn)
    wts = ffn + HS * (QR + 2 * KVR)
    if op == "prefill":
        return dict(bytes=2 * (wts + 2 * T * HS + 2 * T * KVR + 2 * KVR * (T + sum(past))),
                    flops=2 * T * wts + 4 * QR * pairs)
    B, n, L = c["batch"], sum(_lens(c)), c.get("layers", 1)
    head = HS * VOCAB if op == "step" else 0
    return dict(bytes=2 * (L * (wts + 2 * KVR * n + 2 * B * KVR) + 2 * B * HS + head + (B * VOCAB if head else 0)),
                flops=2 * B * (L * wts + head) + 4 * L * QR * n)


def tolerance(case):
    """rel: 2-norm of the difference over the 2-norm of the result; max: the
    largest difference over the larger of the value and the result's RMS."""
    op = case["op"]
    if op == "sum":
        return dict(rel=1e-6, max=1e-6)  # fp32 sums in another order
    if op == "softmax" or (op == "rmsnorm" and case["dtype"] == "f32"):
        return dict(rel=2e-6, max=1e-5)  # fp32 statistics in another order
    if op in ("rmsnorm", "qk_rope", "gemv", "attn", "prefill_attn"):
        # one bf16 rounding of an fp32 result: a tie that flips moves a value by one ulp (2^-7 at most); prefill
        # attention also rounds its probabilities
        return dict(rel=1e-2 if op == "prefill_attn" else 4e-3, max=0.1 if op == "prefill_attn" else 0.02)
    # chains of bf16-rounded stages: a flipped rounding in one travels through those that follow
    return dict(rel=2e-2 if op == "step" else 1e-2, max=0.25)


# ------------------------------------------------------- the result in fp64
def _rms(x, w=None):
    y = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS)
    return y if w is None else y * w.double()


def _rope(x, cos, sin):
    """Half-split RoPE of x [T, heads, D] at the rows cos / sin [T, D]."""
    h = x.shape[-1] // 2
    rot = torch.cat((-x[..., h:], x[..., :h]), -1)
    return x * cos.double()[:, None] + rot * sin.double()[:, None]


def _rows(cache, bt, b, n):
    """Rows [0, n) of sequence b of one cache: [kv heads, n, D] in fp64."""
    if bt is None:
        return cache[b, :, :n].double()
    P = cache.shape[2]
    g = cache[bt[b, : -(-n // P)].long()]
    return g.permute(1, 0, 2, 3).reshape(cache.shape[1], -1, cache.shape[3])[:, :n].double()


def _attend(q, K, V, past):
    """Causal attention of q [n, H, D] (token i sees rows [0, past + i]) over K, V [Hkv, L, D]."""
    n, H, D = q.shape
    G = H // K.shape[0]
    out = torch.empty(n, H, D, dtype=F64, device=q.device)
    step = max(1, (1 << 25) // (G * K.shape[1]))
    for i in range(0, n, step):
        j = min(n, i + step)
        L = past + j
        seen = torch.arange(L, device=q.device)[None] <= (past + torch.arange(i, j, device=q.device))[:, None]
        for h in range(K.shape[0]):
            qh = q[i:j, h * G:(h + 1) * G].transpose(0, 1).reshape(-1, D)
            s = (qh @ K[h, :L].T.contiguous() * D ** -0.5).reshape(G, j - i, L).masked_fill_(~seen, float("-inf"))
            o = torch.softmax(s, -1).reshape(-1, L) @ V[h, :L]
            out[i:j, h * G:(h + 1) * G] = o.reshape(G, j - i, D).transpose(0, 1)
    return out


def _ffn(attn, residual, Wo, pw, Wg, Wu, Wd):
    x2 = residual + attn @ Wo.double().T
    xn = _rms(x2, pw)
    g = xn @ Wg.double().T
    return x2 + (g * torch.sigmoid(g) * (xn @ Wu.double().T)) @ Wd.double().T


def _layer(m, hidden, layer, cos, sin, bt, new, past, kv):
    """One decoder layer over the chunk; kv [2, ...] (fp64) receives the new rows.  Returns the hidden state."""
    K, V, Wqkv, Wo, Wgu, Wd, inw, qw, kw, pw = layer
    H, Hk, IS = m["num_heads"], m["num_kv_heads"], m["intermediate_size"]
    T = hidden.shape[0]
    pos = torch.cat([torch.arange(p, p + n, device=hidden.device) for n, p in zip(new, past)])
    qkv = (_rms(hidden, inw) @ Wqkv.double().T).reshape(T, H + 2 * Hk, 128)
    c, s = cos[pos], sin[pos]
    q, k, v = _rope(_rms(qkv[:, :H], qw), c, s), _rope(_rms(qkv[:, H:H + Hk], kw), c, s), qkv[:, H + Hk:]
    attn, t = torch.empty_like(q), 0
    for b, (n, p) in enumerate(zip(new, past)):
        for cache, x in ((kv[0], k), (kv[1], v)):
            r = torch.arange(p, p + n, device=hidden.device)
            if bt is None:
                cache[b, :, p:p + n] = x[t:t + n].transpose(0, 1)
            else:
                P = cache.shape[2]
                cache[bt[b].long()[r // P], :, r % P] = x[t:t + n]
        attn[t:t + n] = _attend(q[t:t + n], _rows(kv[0], bt, b, p + n), _rows(kv[1], bt, b, p + n), p)
        t += n
    return _ffn(attn.reshape(T, -1), hidden, Wo, pw, Wgu[:IS], Wgu[IS:], Wd)


def exact(case, seed):
    c, op, d = case, case["op"], _inputs(case, seed)
    if op == "rmsnorm":
        return _rms(d["X"].double(), d.get("W"))
    if op == "softmax":
        return torch.softmax(d["X"].double(), -1)
    if op == "sum":
        return d["A"].double().sum().reshape(1)
    if op == "gemv":
        return torch.cat([b.double() @ d["A"].double() for b in d["B"].split(8192)])
    if op == "qk_rope":
        r = random.Random(c["lens_seed"])
        pos = torch.tensor([r.randrange(c["seq"]) for _ in range(c["batch"])], device="cuda")
        q, k = (_rope(_rms(d[x].double(), d[w]), d["cos"][pos], d["sin"][pos]) for x, w in (("q", "qw"), ("k", "kw")))
        K, V = d["K"].double(), d["V"].double()
        b = torch.arange(c["batch"], device="cuda")
        K[b, :, pos], V[b, :, pos] = k, d["v"].double()
        return q, k, K, V
    if op == "attn":
        return torch.stack([_attend(d["Q"][b].double().transpose(0, 1), _rows(d["K"], d.get("bt"), b, n),
                                    _rows(d["V"], d.get("bt"), b, n), n - 1).transpose(0, 1)
                            for b, n in enumerate(_lens(c))])
    if op == "prefill_attn":
        new, past = _chunks(c)
        outs, t = [], 0
        for b, (n, p) in enumerate(zip(new, past)):
            outs.append(_attend(d["Q"][t:t + n].double(), _rows(d["K"], d.get("bt"), b, p + n),
                                _rows(d["V"], d.get("bt"), b, p + n), p))
            t += n
        return torch.cat(outs)
    if op == "ffn":
        return _ffn(d["attn"].double(), d["residual"].double(), d["Wo"], d["pw"], d["Wg"], d["Wu"], d["Wd"])
    m = MODELS[c["model"]]
    if op == "prefill":
        new, past = _chunks(c)
    else:
        new, past = [1] * c["batch"], [n - 1 for n in _lens(c)]
    h, kv = d["hidden"].double(), d["kv"].double()
    for i, layer in enumerate(d["layers"]):
        h = _layer(m, h, layer, d["cos"], d["sin"], d["bt"], new, past, kv[i])
    if op != "step":
        return h, kv
    logits = torch.cat([_rms(h, d["final_w"]) @ w.double().T for w in d["lm_head"].split(16384)], -1)
    return h, logits, kv
