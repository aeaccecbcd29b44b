"""Measured workloads: what a serving process has the framework compute.

One case is one model step, through the objects a program holds to make it:
`ModelWeights`, `PagedKV`, `Runner` and `DecodeGraphs`. Three kinds:

  decode   one token for each of `batch` sequences (DecodeGraphs.run), their
           contexts spread evenly from an eighth of `context` up to it; `limit`
           is the server's context limit (the width of its block table), `kv`
           the cache type ("native" bf16, or "fp8");
  prefill  `prompts` whole prompts in one packed step, spread evenly from an
           eighth of `longest` up to it, then the logits of their last tokens;
  chunk    the next `chunk` tokens of `sequences` sequences that already hold
           `history` tokens in the cache: a long prompt's next portion, or a
           few proposed tokens that speculative decoding verifies; logits of
           the last tokens (a portion) or of all of them (at most 16).

Models are the framework's presets with random weights and their first DEPTH
layers: bf16 rounding through random layers grows with every layer, and whole
stacks would differ by as much as a wrong kernel does. Stacks with routed
experts are not among them: a near tie in the choice of experts changes a
token's whole output, so two correct implementations cannot be compared.
"""
import dataclasses
import math
import random

import torch
import torch.nn.functional as F

from bee2bee_amd.engine.graphs import DecodeGraphs
from bee2bee_amd.engine.kv import PagedKV
from bee2bee_amd.engine.runner import Runner
from bee2bee_amd.models.spec import PRESETS
from bee2bee_amd.models.weights import ModelWeights

DEVICE = torch.device("cuda:0")
DTYPE = torch.bfloat16
DEPTH = 8         # layers of each stack (distilgpt2 has six)
VERIFY_ROWS = 16  # chunks up to this many tokens want the logits of each row


def spec_of(case):
    spec = PRESETS[case["model"]]
    return dataclasses.replace(spec, n_layers=min(DEPTH, spec.n_layers))


# ------------------------------------------------------------------- cases


def listed():
    return [
        # the smallest call: one user of the smallest model, a step of
        # launches and latency more than of work
        decode("distilgpt2", 1, 300, 1024),
        # one user of a small model on a short conversation
        decode("llama3.2-1b", 1, 1000, 4096),
        # one user of the flagship model: weights are read for one row
        decode("llama3-8b", 1, 3000, 4096),
        # two users deep in long documents: few rows, much cache
        decode("qwen2.5-7b", 2, 24000, 32768),
        # an ordinary moment of a chat server
        decode("llama3-8b", 24, 2000, 4096),
        # the flagship benchmark's batch: the cache outweighs the weights
        decode("llama3-8b", 1536, 1100, 2048),
        # a busy server with the 8-bit cache
        decode("zephyr-7b", 200, 3000, 4096, "fp8"),
        # a chat message to a small model: time to first token
        prefill("llama3.2-1b", 1, 57),
        # ordinary prompts of mixed length that arrived together
        prefill("llama3.2-3b", 9, 901),
        # a full admission step of long prompts
        prefill("qwen2.5-7b", 4, 4096),
        # a long document's next portion against what is already cached
        chunk("qwen2.5-7b", 1, 4096, 12288),
        # speculative decoding: the proposed tokens of a small batch
        chunk("llama3-8b", 16, 5, 1500),
    ]


def decode(model, batch, context, limit, kv="native"):
    return {"name": f"decode {model} b{batch} c{context} {kv}",
            "kind": "decode", "model": model, "batch": batch,
            "context": context, "limit": limit, "kv": kv}


def prefill(model, prompts, longest):
    return {"name": f"prefill {model} {prompts}x{longest}", "kind": "prefill",
            "model": model, "prompts": prompts, "longest": longest}


def chunk(model, sequences, tokens, history):
    return {"name": f"chunk {model} {sequences}x{tokens}+{history}",
            "kind": "chunk", "model": model, "sequences": sequences,
            "chunk": tokens, "history": history}


def draw(rng: random.Random):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["decode", "decode", "prefill", "chunk"])
    if kind == "decode":
        model = rng.choice(["distilgpt2", "llama3.2-1b", "llama3.2-3b",
                            "llama3-8b", "zephyr-7b", "qwen2.5-7b"])
        spec = PRESETS[model]
        limit = min(spec.max_seq_len, rng.choice([2048, 4096, 8192, 32768]))
        context = log_int(40, limit - 2)
        # at most the tokens in the cache of the largest listed case
        batch = log_int(1, max(1, min(1536, 1600000 // context)))
        kv = rng.choice(["native", "native", "native", "fp8"])
        case = decode(model, batch, context, limit, kv)
    elif kind == "prefill":
        model = rng.choice(["distilgpt2", "llama3.2-1b", "llama3.2-3b",
                            "llama3-8b", "zephyr-7b", "qwen2.5-7b"])
        longest = log_int(8, min(4096, PRESETS[model].max_seq_len - 1))
        prompts = log_int(1, max(1, min(64, 16384 // longest)))
        case = prefill(model, prompts, longest)
    else:
        model = rng.choice(["llama3.2-1b", "llama3.2-3b", "llama3-8b",
                            "qwen2.5-7b"])
        tokens = rng.choice([log_int(2, 8), log_int(64, 4096)])
        history = log_int(100, min(PRESETS[model].max_seq_len, 16384)
                          - tokens - 1)
        most = 64 if tokens <= VERIFY_ROWS else 8
        sequences = log_int(1, max(1, min(most, 4096 // tokens,
                                          200000 // history)))
        case = chunk(model, sequences, tokens, history)
    del case["name"]
    return case


def spread(n, longest):
    """n lengths, evenly from `longest` down to an eighth of it."""
    lo = max(1, longest // 8)
    return [longest - (longest - lo) * i // max(1, n - 1) for i in range(n)]


def lengths(case):
    """(tokens cached before the step, tokens of the step) per sequence."""
    if case["kind"] == "decode":
        return [(n - 1, 1) for n in spread(case["batch"], case["context"])]
    if case["kind"] == "prefill":
        return [(0, n) for n in spread(case["prompts"], case["longest"])]
    return [(case["history"], case["chunk"])] * case["sequences"]


# ----------------------------------------------------------------- prepare


@torch.no_grad()
def prepare(case, seed):
    spec = spec_of(case)
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    order = random.Random(seed)
    weights = ModelWeights(spec, DEVICE, DTYPE).random_init(seed=seed)
    # fresh weights have an embedding far smaller than what a layer adds and
    # an attention output lost beside the feed-forward's; trained stacks have
    # the three of one size
    weights.embed.normal_(0.0, 1.0, generator=gen)
    for layer in weights.layers:
        layer.wo *= 4.0
    # trained norms and biases are neither all ones nor all zeros
    for holder in [weights, *weights.layers]:
        for name in ("attn_norm", "mlp_norm", "final_norm"):
            w = getattr(holder, name, None)
            if w is not None:
                w.normal_(1.0, 0.1, generator=gen)
            b = getattr(holder, name + "_bias", None)
            if b is not None:
                b.normal_(0.0, 0.02, generator=gen)
        for name in ("wqkv_bias", "wo_bias", "w_gate_up_bias", "w_down_bias"):
            b = getattr(holder, name, None)
            if b is not None:
                b.normal_(0.0, 0.02, generator=gen)

    lens = lengths(case)
    order.shuffle(lens)
    totals = [old + new for old, new in lens]
    kv_dtype = case.get("kv", "native")
    kv = PagedKV(spec, DEVICE, DTYPE, n_blocks=1 + sum(
        -(-n // 256) for n in totals), block_size=256, kv_dtype=kv_dtype)
    # sequences that grew side by side: their pages alternate in the pool
    for s in range(len(totals)):
        kv.new_seq(s)
    for upto in range(256, max(totals) + 256, 256):
        for s, n in enumerate(totals):
            if upto - 256 < n:
                kv.extend_seq(s, min(n, upto))
    if case["kind"] != "prefill":
        # keys and values as the projections of unit-norm rows have them
        std = 0.02 * spec.hidden_size ** 0.5
        for cache in [*kv.k_cache, *kv.v_cache]:
            if kv_dtype == "fp8":
                rows = torch.empty(cache.shape, dtype=DTYPE, device=DEVICE)
                rows.normal_(0.0, std, generator=gen)
                cache.copy_(rows.to(torch.float8_e4m3fn).view(torch.uint8))
            else:
                cache.normal_(0.0, std, generator=gen)

    def ints(values):
        return torch.tensor(values, dtype=torch.int32, device=DEVICE)

    runner = Runner(spec, weights, kv, DEVICE, DTYPE)
    ids = torch.randint(0, spec.vocab_size, (sum(n for _, n in lens),),
                        generator=gen, device=DEVICE)
    positions = [p for old, new in lens for p in range(old, old + new)]
    state = {"case": case, "weights": weights, "kv": kv, "runner": runner,
             "ids": ids, "lens": lens, "table": kv.block_table(
                 list(range(len(lens))))}
    if case["kind"] == "decode":
        B, table = len(lens), state["table"]
        graphs = DecodeGraphs(runner, B, -(-case["limit"] // 256))
        graphs.positions.copy_(ints(positions))
        graphs.seq_lens.copy_(ints(totals))
        graphs.block_table[:, : table.shape[1]].copy_(table)
        graphs.input_ids.copy_(ids)
        graphs.run(B)       # captured when the server starts
        state["graphs"] = graphs
        return state
    cu = [0]
    for _, new in lens:
        cu.append(cu[-1] + new)
    state["positions"] = ints(positions)
    state["slots"] = ints([s for i, (old, new) in enumerate(lens)
                           for s in kv.slot_mapping(i, range(old, old + new))])
    state["cu"] = ints(cu)
    state["longest"] = max(new for _, new in lens)
    if case["kind"] == "chunk":
        state["seq_lens"] = ints(totals)
        state["query_lens"] = ints([new for _, new in lens])
    state["rows"] = torch.tensor(wanted_rows(case, lens), device=DEVICE)
    return state


def wanted_rows(case, lens):
    """Rows of the step whose logits are sampled from."""
    ends, total = [], 0
    for _, new in lens:
        total += new
        ends.append(total - 1)
    if case["kind"] == "chunk" and case["chunk"] <= VERIFY_ROWS:
        return list(range(total))
    return ends


@torch.no_grad()
def run(state):
    runner, case = state["runner"], state["case"]
    if case["kind"] == "decode":
        graphs = state["graphs"]
        graphs.input_ids.copy_(state["ids"])    # the tokens sampled last
        return {"logits": graphs.run(case["batch"])}
    more = {}
    if case["kind"] == "chunk":
        more = {"block_table": state["table"], "seq_lens": state["seq_lens"],
                "query_lens": state["query_lens"]}
    hidden = runner.forward_prefill(
        state["ids"], state["positions"], state["slots"], state["cu"],
        state["longest"], **more)
    out = {"hidden": hidden, "logits": runner.lm_head(hidden[state["rows"]])}
    if case["kind"] == "prefill":
        # a portion reads its own keys and values back; whole prompts leave
        # theirs for the steps that follow
        out["k"], out["v"] = state["kv"].k_cache, state["kv"].v_cache
    return out


# -------------------------------------------------------------------- work


def work(case):
    spec, lens = spec_of(case), lengths(case)
    H, I, L = spec.hidden_size, spec.intermediate_size, spec.n_layers
    qkv = spec.q_size + 2 * spec.kv_size
    mats = H * qkv + H * spec.q_size
    mats += (2 if spec.act_type == "gelu" else 3) * H * I
    T = sum(new for _, new in lens)
    rows = len(wanted_rows(case, lens)) if case["kind"] != "decode" else T
    pairs = sum(new * old + new * (new + 1) // 2 for old, new in lens)
    elem = 1 if case.get("kv") == "fp8" else 2
    weight = 2 * (L * mats + spec.vocab_size * H) + 2 * T * H
    cache = 2 * L * spec.kv_size * elem * sum(old + new for old, new in lens)
    hidden_out = 0 if case["kind"] == "decode" else 2 * T * H
    return {"bytes": weight + cache + hidden_out + 2 * rows * spec.vocab_size,
            "flops": 2 * L * mats * T + 2 * spec.vocab_size * H * rows
            + 4 * L * spec.q_size * pairs}


def tolerance(case):
    """bf16 activations and a bf16 residual through the whole stack: 0.007 to
    0.013 from `exact` as measured (0.024 with the 8-bit cache), so that two
    implementations differ by about as much."""
    return {"rel": 0.03, "max": 0.4}


# ------------------------------------------------------------------- exact


@torch.no_grad()
def exact(case, seed):
    """The same step in float64 with plain torch."""
    state = prepare(case, seed)
    state.pop("graphs", None)
    spec, W, kv, lens = (spec_of(case), state["weights"], state["kv"],
                         state["lens"])
    D = torch.float64
    nq, nkv, hd, eps = spec.n_heads, spec.n_kv_heads, spec.head_dim, \
        spec.rms_eps
    ids = state["ids"]
    pos = torch.tensor([p for old, new in lens
                        for p in range(old, old + new)], device=DEVICE)
    T, table = len(pos), state["table"].long()

    def norm(x, w, b):
        if spec.norm_type == "layernorm":
            return F.layer_norm(x, x.shape[-1:], w.to(D), b.to(D), eps)
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) \
            * w.to(D)

    def linear(x, w, b=None):
        y = x @ w.to(D).t()
        return y if b is None else y + b.to(D)

    def rotate(x):
        half = hd // 2
        freq = spec.rope_theta ** (
            -torch.arange(half, dtype=D, device=DEVICE) / half)
        a = pos.to(D)[:, None, None] * freq
        x1, x2 = x[..., :half], x[..., half:]
        return torch.cat([x1 * a.cos() - x2 * a.sin(),
                          x2 * a.cos() + x1 * a.sin()], -1)

    def cached(pool, s, n):
        """The first n rows of sequence s, [nkv, n, hd]."""
        pages = pool[table[s, : -(-n // 256)]]
        if pages.dtype == torch.uint8:
            pages = pages.view(torch.float8_e4m3fn)
        return pages.to(D).transpose(0, 1).reshape(nkv, -1, hd)[:, :n]

    def attention(q, k, v, layer):
        out, at = torch.empty(T, nq, hd, dtype=D, device=DEVICE), 0
        for s, (old, new) in enumerate(lens):
            kk = k[at : at + new].transpose(0, 1)
            vv = v[at : at + new].transpose(0, 1)
            if old:
                kk = torch.cat([cached(kv.k_cache[layer], s, old), kk], 1)
                vv = torch.cat([cached(kv.v_cache[layer], s, old), vv], 1)
            ahead = None
            if new > 1:
                ahead = torch.arange(old + new, device=DEVICE)[None] > \
                    torch.arange(old, old + new, device=DEVICE)[:, None]
            kk = kk.transpose(1, 2).contiguous()
            # heads at once while their scores are few
            step = nkv if new < 64 else 1
            for g in range(0, nkv, step):
                h = slice(g * (nq // nkv), (g + step) * (nq // nkv))
                qq = q[at : at + new, h].transpose(0, 1).reshape(step, -1, hd)
                sc = (qq @ kk[g : g + step]) * hd ** -0.5
                if ahead is not None:
                    sc.view(-1, new, old + new).masked_fill_(ahead, -math.inf)
                o = torch.softmax(sc, -1) @ vv[g : g + step]
                out[at : at + new, h] = o.view(-1, new, hd).transpose(0, 1)
            at += new
        return out.reshape(T, nq * hd)

    pools = ([], [])
    slots = state.get("slots")

    def keep(rows, pool, into):
        """The pages after the step, in float64."""
        pages = pool.to(D)
        pages[slots.long() // 256, :, slots.long() % 256] = rows
        into.append(pages.cpu())

    x = W.embed[ids].to(D)
    if spec.pos_type == "learned":
        x = x + W.pos_embed[pos].to(D)
    for i, lw in enumerate(W.layers):
        h = norm(x, lw.attn_norm, lw.attn_norm_bias)
        qkv = linear(h, lw.wqkv, lw.wqkv_bias)
        q, k, v = qkv.split([nq * hd, nkv * hd, nkv * hd], -1)
        q, k, v = (t.reshape(T, -1, hd) for t in (q, k, v))
        if spec.pos_type == "rope":
            q, k = rotate(q), rotate(k)
        if case["kind"] == "prefill":
            keep(k, kv.k_cache[i], pools[0])
            keep(v, kv.v_cache[i], pools[1])
        x = x + linear(attention(q, k, v, i), lw.wo, lw.wo_bias)
        h = norm(x, lw.mlp_norm, lw.mlp_norm_bias)
        z = linear(h, lw.w_gate_up, lw.w_gate_up_bias)
        if spec.act_type == "gelu":
            z = F.gelu(z, approximate="tanh")
        else:
            gate, up = z.chunk(2, -1)
            z = F.silu(gate) * up
        x = x + linear(z, lw.w_down, lw.w_down_bias)
        del h, qkv, q, k, v, z
    last = x if case["kind"] == "decode" else x[state["rows"]]
    logits = linear(norm(last, W.final_norm, W.final_norm_bias), W.lm_head)
    if case["kind"] == "decode":
        return {"logits": logits}
    out = {"hidden": x, "logits": logits}
    if case["kind"] == "prefill":
        out["k"], out["v"] = list(pools[0]), list(pools[1])
    return out
