"""The work whose speed is measured, as a program that uses this package calls it.

`listed()` is a fixed list, `draw(rng)` gives one more case of the same ranges. The kinds:

  step       one token of the sparse read over a stack of layers (`sparse_decode_step_kernel`: index score, top-k,
             gather-free attend), every layer over a K/V cache and an index table of its own. A serving loop captures
             the stack in a HIP graph and replays it; the smallest one is a plain call.
  dense      the control: one token's full read of one layer (`dense_decode_step`).
  attend     the read of a given row list (`gather_attention`): sinks, a local window and uniform picks, unsorted.
  prefill    a causal prompt chunk of one layer (`full_attention`, T > 1), at the prompt's start or after a history.
  lightning  the lightning-indexer score of one decode query and its top-k by score.
  lightning_prefill   the T-query lightning score of a prompt chunk, causal.
  model      a prompt through the wrapped model (`LabRunner.prefill`): K/V and index tables written, logits returned.

Shapes: 8 KV groups, head_dim 128, index width 32, as in the Qwen3 shapes of bench.py; contexts from 1K to 128K, one
request to 32, 1 to 8 query heads per KV group; bfloat16 caches, bfloat16 or (trained banks) float32 index tables,
fp16 or bf16 lightning keys. Synthetic data, K, V, index keys and queries ~ N(0, 1).
"""
from __future__ import annotations

import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "attention-lab_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import attention_lab as al  # noqa: E402
from attention_lab import hip_score, hip_select  # noqa: E402

DEV = "cuda"
G, D, R = 8, 128, 32
RHO = 1 / 32
SINKS, WINDOW = 4, 128   # of the attend kind's row lists


def listed():
    return [
        # a short chat turn's single layer, called as it is: two launches, so the call itself is what there is to pay
        dict(name="step_short_call", kind="step", batch=1, heads=2, length=2048, layers=1, index="bf16", graph=False),
        # one request at 32K through all 28 layers of the 1.7B shape: latency per token
        dict(name="step_b1_32k", kind="step", batch=1, heads=2, length=32768, layers=28, index="bf16", graph=True),
        # batched serving at 32K, the benchmark's layer (four of its 36 layers; 1.1 GB of index tables a pass)
        dict(name="step_b16_32k", kind="step", batch=16, heads=4, length=32768, layers=4, index="bf16", graph=True),
        # long contexts, two requests, past what one list of 32K candidates holds
        dict(name="step_b2_128k", kind="step", batch=2, heads=2, length=131072, layers=4, index="bf16", graph=True),
        # a trained bank (float32 index table), an odd batch and an odd length
        dict(name="step_f32_b5_12k", kind="step", batch=5, heads=4, length=12345, layers=6, index="f32", graph=True),
        # the full read of a few requests of ordinary length
        dict(name="dense_b3_20k", kind="dense", batch=3, heads=2, length=20011),
        # the row-list read at its largest sweep point: 2048 picks + sinks + window out of 32K, 16 requests
        dict(name="attend_b16_k2048", kind="attend", batch=16, heads=2, length=32768, picks=2048),
        # an 8K prompt at once, 32 query heads
        dict(name="prefill_8k", kind="prefill", batch=1, heads=4, tokens=8192, history=0),
        # a ragged chunk deep into a long prompt, 16 query heads
        dict(name="prefill_chunk_30k", kind="prefill", batch=1, heads=2, tokens=1000, history=29011),
        # the lightning indexer's decode step over eight 128K contexts
        dict(name="lightning_b8_128k", kind="lightning", batch=8, groups=1, length=131072, heads=4, keys="f16"),
        # the lightning score of a prompt chunk after 7000 cached positions
        dict(name="lightning_prefill_3k", kind="lightning_prefill", batch=1, groups=8, tokens=3000, history=7000,
             heads=4, keys="f16"),
        # a prompt through four layers of the 1.7B shape, in the chunks a serving loop uses
        dict(name="model_prefill_3k", kind="model", layers=4, tokens=3003, chunk=1024),
    ]


def _log(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "dense", "attend", "prefill", "prefill", "lightning",
                       "lightning_prefill"])
    if kind == "step":
        length = _log(rng, 1024, 131072)
        batch = _log(rng, 1, max(1, min(32, 16 * 32768 // length)))
        index = rng.choice(["bf16", "bf16", "f32"])
        layers = max(1, min(28, (4 if index == "bf16" else 2) * 16 * 32768 // (batch * length)))
        return dict(kind=kind, batch=batch, heads=rng.choice([1, 2, 4, 4]), length=length,
                    layers=min(layers, _log(rng, 2, 28)), index=index, graph=True)
    if kind == "dense":
        length = _log(rng, 1024, 131072)
        return dict(kind=kind, batch=_log(rng, 1, max(1, min(32, 16 * 32768 // length))),
                    heads=rng.choice([1, 2, 4, 8]), length=length)
    if kind == "attend":
        length = _log(rng, 4096, 65536)
        return dict(kind=kind, batch=_log(rng, 1, 16), heads=rng.choice([1, 2, 4, 8]), length=length,
                    picks=_log(rng, 64, 2048))
    if kind == "prefill":
        tokens = _log(rng, 128, 8192)
        history = rng.choice([0, _log(rng, 64, 30000)]) if tokens <= 2048 else 0
        most = 8192 * 8192 // (tokens * (tokens + 2 * history))
        return dict(kind=kind, batch=_log(rng, 1, max(1, min(8, most))), heads=rng.choice([1, 2, 4]), tokens=tokens,
                    history=history)
    if kind == "lightning":
        length = _log(rng, 4096, 131072)
        return dict(kind=kind, batch=_log(rng, 1, 32), groups=rng.choice([1, 1, 8]), length=length,
                    heads=rng.choice([1, 2, 4, 8]), keys=rng.choice(["f16", "bf16"]))
    return dict(kind=kind, batch=1, groups=rng.choice([1, 8]), tokens=_log(rng, 256, 3000),
                history=_log(rng, 64, 7000), heads=rng.choice([1, 2, 4, 8]), keys=rng.choice(["f16", "bf16"]))


# ---------------------------------------------------------------------------------------------------------------------
# inputs: made on the GPU from the seed alone
# ---------------------------------------------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(gen, *shape, dtype=torch.bfloat16):
    return torch.randn(*shape, generator=gen, device=DEV, dtype=dtype)


def _keys_dtype(case):
    return torch.float16 if case["keys"] == "f16" else torch.bfloat16


class _Step:
    """A stack of layers at one token: caches, tables, weights, the step's plan and queries."""

    def __init__(self, case, seed):
        gen = _gen(seed)
        B, h, L, layers = case["batch"], case["heads"], case["length"], case["layers"]
        idx = torch.bfloat16 if case["index"] == "bf16" else torch.float32
        C = -(-L // 8) * 8
        self.k = _randn(gen, layers, B, G, C, D)
        self.v = _randn(gen, layers, B, G, C, D)
        self.z = _randn(gen, layers, B, G, R, C, dtype=idx)
        self.q = _randn(gen, layers, B, G, h, 1, D)
        self.q_pre = _randn(gen, layers, B, G, h, 1, D, dtype=idx)
        self.k_new = _randn(gen, layers, B, G, 1, D, dtype=idx)
        self.wk = _randn(gen, layers, G, R, D, dtype=torch.float32).mul_(0.02).to(idx)
        self.wq_t = _randn(gen, layers, G, h * D, R, dtype=torch.float32).mul_(0.02 / math.sqrt(R)).to(idx)
        self.request = al.prepare_request(B, G, C, valid_length=L, query_position=L - 1, rho=RHO, device=DEV)
        self.out = self.graph = None
        if case["graph"]:
            self.launch()   # grows the step's scratch, as a program does before it captures
            torch.cuda.synchronize()
            self.graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(self.graph):
                self.out = self.launch()

    def launch(self):
        rq, lay = self.request, self.request.layout
        return [al.sparse_decode_step_kernel(self.q[l], self.q_pre[l], self.k[l], self.v[l], self.z[l], self.wq_t[l],
                                             self.wk[l], rq.fixed_rows, rq.off_lo, lay.candidate_lo, lay.candidate_hi,
                                             rq.k, rq.selected_count, k_pre_new=self.k_new[l], write_col=rq.write_col)
                for l in range(self.q.shape[0])]

    def run(self):
        if self.graph is None:
            out = self.launch()
        else:
            self.graph.replay()
            out = self.out
        # what the step writes: every layer's output and the new key's index column
        return {"out": out, "index_column": self.z[..., self.request.write_col]}


def _qwen(seed, layers):
    from transformers import Qwen3Config, Qwen3ForCausalLM
    cfg = Qwen3Config(vocab_size=151936, hidden_size=2048, intermediate_size=6144, num_hidden_layers=layers,
                      num_attention_heads=16, num_key_value_heads=8, head_dim=128, max_position_embeddings=40960,
                      rope_theta=1_000_000.0, rms_norm_eps=1e-6, tie_word_embeddings=True, initializer_range=0.02,
                      attn_implementation="sdpa")
    torch.manual_seed(seed)
    with torch.device(DEV):
        model = Qwen3ForCausalLM(cfg)
    model = model.to(torch.bfloat16).eval()
    for p in model.parameters():
        p.requires_grad_(False)
    return model


def prepare(case, seed):
    kind = case["kind"]
    if kind == "step":
        return dict(kind=kind, step=_Step(case, seed))
    gen = _gen(seed)
    if kind == "model":
        from attention_lab.qwen_wrap import LabRunner, make_state, wrap_model
        model = _qwen(seed, case["layers"])
        state = make_state(model, case["tokens"], "sparse", r=R, seed=seed % 1000)
        runner = LabRunner(model, wrap_model(model), state)
        ids = torch.randint(0, 151936, (1, case["tokens"]), generator=gen, device=DEV)
        return dict(kind=kind, runner=runner, ids=ids, chunk=case["chunk"])
    B = case["batch"]
    if kind in ("lightning", "lightning_prefill"):
        KG, nh, dt = case["groups"], case["heads"], _keys_dtype(case)
        T = case.get("tokens", 0)
        L = case["length"] if kind == "lightning" else case["history"] + T
        keys = _randn(gen, B, KG, L, R, dtype=torch.float32).mul_(R ** -0.5).to(dt)
        lead = (B, KG) if kind == "lightning" else (B, KG, T)
        s = dict(kind=kind, keys=keys, q=_randn(gen, *lead, nh, R, dtype=torch.float32),
                 w=torch.rand(*lead, nh, generator=gen, device=DEV))
        if kind == "lightning":
            s["k"] = max(1, L // 32)
        else:   # scores past a query's position are never written: the program's buffer starts at zero
            s["q_pos0"] = case["history"]
            s["out"] = torch.zeros(B, KG, T, -(-L // 4) * 4, device=DEV)
        return s
    h = case["heads"]
    T = case.get("tokens", 1)
    L = case["history"] + T if kind == "prefill" else case["length"]
    C = -(-L // 8) * 8
    s = dict(kind=kind, q=_randn(gen, B, G, h, T, D), k=_randn(gen, B, G, C, D), v=_randn(gen, B, G, C, D), length=L)
    if kind == "attend":
        picks = torch.rand(B, G, L - SINKS - WINDOW, generator=gen, device=DEV).topk(case["picks"], dim=-1).indices
        fixed = torch.cat([torch.arange(SINKS, device=DEV), torch.arange(L - WINDOW, L, device=DEV)])
        rows = torch.cat([fixed.expand(B, G, -1), picks + SINKS], dim=-1)
        order = torch.rand(B, G, rows.shape[-1], generator=gen, device=DEV).argsort(dim=-1)
        s["rows"] = rows.gather(-1, order).to(torch.int32)
    return s


def run(s):
    kind = s["kind"]
    if kind == "step":
        return s["step"].run()
    if kind == "dense":
        return al.dense_decode_step(s["q"], s["k"], s["v"], s["length"])
    if kind == "attend":
        return al.gather_attention(s["q"], s["k"], s["v"], s["rows"])
    if kind == "prefill":
        return al.full_attention(s["q"], s["k"], s["v"], valid_length=s["length"])
    if kind == "lightning":
        scores = hip_score.score_lightning(s["keys"], s["q"], s["w"])
        values, indices = hip_select.topk(scores, s["k"])
        return {"scores": scores, "values": values, "indices": indices}
    if kind == "lightning_prefill":
        return hip_score.score_lightning_batched(s["keys"], s["q"], s["w"], q_pos0=s["q_pos0"], out=s["out"])
    runner = s["runner"]
    runner.rollback(0)
    logits = runner.prefill(s["ids"], s["chunk"])
    cache, n = runner.cache, s["ids"].shape[1]
    return {"logits": logits, "index": [z[..., :n] for z in cache.z], "k": [k[:, :, :n] for k in cache.k],
            "v": [v[:, :, :n] for v in cache.v]}


# ---------------------------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "step":
        B, h, L, layers = case["batch"], case["heads"], case["length"], case["layers"]
        lay = al.selection_layout(L)
        S = lay.selected_count(al.fixed_budget(L, RHO))
        e = 2 if case["index"] == "bf16" else 4
        row = lay.candidate_count * R * e + S * 2 * D * 2 + 2 * h * D * 2 + (h + 1) * D * e + R * e
        weights = G * (h * D * R + R * D) * e
        flops = 2 * lay.candidate_count * R + 4 * h * S * D + 2 * (h + 1) * D * R
        return dict(bytes=layers * (B * G * row + weights), flops=layers * B * G * flops)
    if kind == "dense":
        rows = case["batch"] * G
        return dict(bytes=rows * (case["length"] * 2 * D * 2 + 2 * case["heads"] * D * 2),
                    flops=rows * 4 * case["heads"] * case["length"] * D)
    if kind == "attend":
        rows, S = case["batch"] * G, SINKS + WINDOW + case["picks"]
        return dict(bytes=rows * (S * (2 * D * 2 + 4) + 2 * case["heads"] * D * 2),
                    flops=rows * 4 * case["heads"] * S * D)
    if kind == "prefill":
        T, P = case["tokens"], case["history"]
        rows = case["batch"] * G
        pairs = T * P + T * (T + 1) // 2
        return dict(bytes=rows * ((P + T) * 2 * D * 2 + 2 * case["heads"] * T * D * 2),
                    flops=rows * case["heads"] * pairs * 4 * D)
    if kind == "lightning":
        rows, L, nh = case["batch"] * case["groups"], case["length"], case["heads"]
        k = max(1, L // 32)
        return dict(bytes=rows * (L * R * 2 + L * 4 + k * 12 + nh * (R + 1) * 4), flops=rows * L * nh * (2 * R + 2))
    if kind == "lightning_prefill":
        rows, T, P, nh = case["batch"] * case["groups"], case["tokens"], case["history"], case["heads"]
        pairs = T * P + T * (T + 1) // 2
        return dict(bytes=rows * (pairs * 4 + (P + T) * R * 2 + T * nh * (R + 1) * 4),
                    flops=rows * pairs * nh * (2 * R + 2))
    T, layers, hidden, inner, vocab, heads = case["tokens"], case["layers"], 2048, 6144, 151936, 16
    params = hidden * (heads + 2 * G) * D + heads * D * hidden + 3 * hidden * inner
    attend = heads * (T * (T + 1) // 2) * 4 * D
    table = G * T * R * D * 2
    return dict(bytes=layers * (params * 2 + G * T * (2 * D + R) * 2) + vocab * hidden * 2 + T * hidden * 2 + vocab * 2,
                flops=layers * (2 * T * params + attend + table) + 2 * vocab * hidden)


def tolerance(case):
    """bfloat16 outputs: one rounding is 2^-9 of the value, 1.7e-3 over the norm; four times what the path is off
    `exact` by. A step's row list may differ by the near ties that the last fp32 bits of a score decide; one exchanged
    row changes its output row by about 1 / sqrt(S) of its norm."""
    kind = case["kind"]
    if kind == "step":
        return {"rel": 1e-2, "max": 0.5}
    if kind in ("dense", "attend"):
        return {"rel": 7e-3, "max": 0.03}
    if kind == "prefill":   # the weights are rounded to bfloat16 before the second product
        return {"rel": 1e-2, "max": 0.1}
    if kind == "lightning":   # the sums' order may swap near ties of the list
        return {"rel": 4e-6, "max": 1e-4, "differ": 5e-3}
    if kind == "lightning_prefill":
        return {"rel": 4e-6, "max": 1e-4}
    # model: a change of rounding in one layer travels through those after it; the same prompt in other chunks gives
    # logits 1.4e-2 apart (each chunk's products sum in another order)
    return {"rel": 3e-2, "max": 0.3}


# ---------------------------------------------------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------------------------------------------------
def _exact_step(case, seed):
    st = _Step(dict(case, graph=False), seed)
    lay, k = st.request.layout, st.request.k
    lo, hi, L = lay.candidate_lo, lay.candidate_hi, lay.legal_length
    layers, B, _, h = st.q.shape[:4]
    fixed = torch.tensor(lay.fixed_positions(), device=DEV).expand(B, G, -1)
    outs, cols = [], []
    for l in range(layers):
        u = torch.einsum("bgf,gfr->bgr", st.q_pre[l].double().reshape(B, G, h * D), st.wq_t[l].double())
        cols.append(torch.einsum("bge,gre->bgr", st.k_new[l, :, :, 0].double(), st.wk[l].double()))
        out = torch.empty(B, G, h, 1, D, dtype=torch.float64, device=DEV)
        for b in range(B):
            s = torch.einsum("gr,grm->gm", u[b], st.z[l, b, :, :, lo:hi].double())
            top = s.sort(dim=-1, descending=True, stable=True).indices[:, :k] + lo
            rows = torch.cat([fixed[b], top], dim=-1).unsqueeze(-1).expand(-1, -1, D)
            kk, vv = st.k[l, b].gather(1, rows).double(), st.v[l, b].gather(1, rows).double()
            p = torch.softmax(st.q[l, b, :, :, 0].double() @ kk.transpose(1, 2).contiguous() / math.sqrt(D), dim=-1)
            out[b, :, :, 0] = p @ vv
        outs.append(out)
    return {"out": outs, "index_column": torch.stack(cols)}


def _exact_attention(s):
    """dense, attend and prefill: query t of the T last positions reads the rows up to its own position."""
    q, L = s["q"], s["length"]
    B, _, h, T, _ = q.shape
    out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
    pos = torch.arange(L - T, L, device=DEV)
    step = max(1, (1 << 27) // (h * L))
    for b in range(B):
        for g in range(G):
            k, v = s["k"][b, g, :L], s["v"][b, g, :L]
            if "rows" in s:
                k, v = k[s["rows"][b, g].long()], v[s["rows"][b, g].long()]
            kt, v = k.double().t().contiguous(), v.double()
            for a in range(0, T, step):
                x = q[b, g, :, a:a + step].double() @ kt / math.sqrt(D)
                if "rows" not in s:
                    x.masked_fill_(torch.arange(L, device=DEV) > pos[a:a + step].unsqueeze(1), float("-inf"))
                out[b, g, :, a:a + step] = torch.softmax(x, dim=-1) @ v
    return out


def _exact_lightning(s):
    keys, q, w = s["keys"], s["q"], s["w"]
    B, KG, L, _ = keys.shape
    batched = q.dim() == 5
    if batched:
        out = torch.zeros(B, KG, q.shape[2], L, dtype=torch.float64, device=DEV)
        pos = s["q_pos0"] + torch.arange(q.shape[2], device=DEV)
    else:
        out = torch.zeros(B, KG, L, dtype=torch.float64, device=DEV)
    for b in range(B):
        for g in range(KG):
            kt = keys[b, g].double().t().contiguous()
            for i in range(q.shape[-2]):
                x = torch.relu(q[b, g, ..., i, :].double() @ kt)
                out[b, g] += (x * w[b, g, ..., i].double().unsqueeze(-1))
            if batched:
                out[b, g].masked_fill_(torch.arange(L, device=DEV) > pos.unsqueeze(1), 0.0)
    if batched:
        return out
    values, indices = out.sort(dim=-1, descending=True, stable=True)
    return {"scores": out, "values": values[..., :s["k"]].contiguous(), "indices": indices[..., :s["k"]].contiguous()}


def exact(case, seed):
    kind = case["kind"]
    if kind == "step":
        return _exact_step(case, seed)
    if kind == "model":
        return None
    s = prepare(case, seed)
    return _exact_lightning(s) if kind.startswith("lightning") else _exact_attention(s)
