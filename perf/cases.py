"""The work that a user of this framework has it do, as cases that can be timed: prompts, single-token steps, the greedy token
loop, a span of blocks of a split model and the op-level tensors, through the package's public entry points.

A case names an entry point ("kind"), a model or tensor shape, the mode (f16: the reference's --f16; otherwise f32, its default)
and the sizes of the call.  Weights come from the package's own generator, N(0, 0.02) as in bench.py, seeded per state; token ids
are uniform over the vocabulary like bench.py's.

Logits and not token ids are compared wherever the next id would be decided by sums in the last place: with random weights the
two largest of 32000 logits are often closer than that.  The one case that returns ids (the greedy loop) has an embedding and an
output head under which every token has a clear successor, as a trained model's confident predictions have.
"""
import math

import numpy as np
import torch

import rllama_amd

VOCAB = 32000
STD = 0.02

# dim, layers, heads, ffn width: the shapes of bench.py's workloads and of the test-suite
SMALL = dict(dim=1024, layers=8, heads=16, ffn=2816)      # the reference's CPU-runnable case
SHAPE_7B = dict(dim=4096, layers=32, heads=32, ffn=11008)
SHAPE_13B = dict(dim=5120, layers=40, heads=40, ffn=13824)
SHAPE_65B = dict(dim=8192, layers=80, heads=64, ffn=22016)


def listed():
    return [
        # one token of a small model, where launches and host round trips are what counts
        dict(name="decode-small", kind="decode", f16=True, **SMALL, pos=79),
        # the greedy token loop on the same model: 16 prompt ids, 64 new ones (the benchmark's smallest workload)
        dict(name="greedy-small", kind="greedy", f16=True, **SMALL, prompt=16, new=64),
        # one token of a chat in the middle of its answer, the next one drawn by the package's sampler from the 40 best
        dict(name="decode-7b-sampled", kind="decode", f16=True, **SHAPE_7B, pos=383, top_k=40),
        # the same step in the reference's default mode (no --f16), early in an answer
        dict(name="decode-7b-f32", kind="decode", f16=False, **SHAPE_7B, pos=100),
        # one token behind a long document
        dict(name="decode-13b-long", kind="decode", f16=True, **SHAPE_13B, pos=2111),
        # the reference's own protocol: a prompt of a few words
        dict(name="prompt-7b-short", kind="prompt", f16=True, **SHAPE_7B, n=8),
        # a chat turn: a few sentences, a ragged number of rows
        dict(name="prompt-7b-turn", kind="prompt", f16=True, **SHAPE_7B, n=131),
        # a page of text (the benchmark's prompt workload)
        dict(name="prompt-7b-page", kind="prompt", f16=True, **SHAPE_7B, n=1024),
        # a paragraph in the reference's default mode
        dict(name="prompt-7b-f32", kind="prompt", f16=False, **SHAPE_7B, n=200),
        # a document at the largest length the benchmark names
        dict(name="prompt-13b-document", kind="prompt", f16=True, **SHAPE_13B, n=2048),
        # a model split by percentage_to_gpu: the device's blocks, the residual stream in and out through host memory
        dict(name="layers-65b-split", kind="layers", f16=True, **SHAPE_65B, resident=4, n=256),
        # the op-level tensors as a host offloads a feed-forward block with them, result read back
        dict(name="ops-feed-forward", kind="ops", f16=True, dim=4096, ffn=11008, n=77),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _shape(rng, max_layers=32):
    """A shape between the small and the 13B one: heads of 64 or 128 dims, the package's ffn rule, fewer or more layers."""
    head_dim = rng.choice((64, 128, 128))
    heads = _log_int(rng, 8 if head_dim == 128 else 16, 40)
    dim = heads * head_dim
    return dict(dim=dim, layers=_log_int(rng, 4, max_layers), heads=heads, ffn=rllama_amd.llama_ffn_hidden(dim))


def draw(rng):
    kind = rng.choice(("decode", "decode", "decode", "prompt", "prompt", "prompt", "prompt", "greedy", "layers", "ops"))
    f16 = rng.random() < 0.75
    if kind == "decode":
        case = dict(kind=kind, f16=f16, **_shape(rng), pos=_log_int(rng, 1, 2111))
        if rng.random() < 0.3:
            case["top_k"] = rng.choice((10, 40, 100))
    elif kind == "prompt":
        case = dict(kind=kind, f16=f16, **_shape(rng), n=_log_int(rng, 2, 2048 if f16 else 300))
    elif kind == "greedy":
        case = dict(kind=kind, f16=f16, **SMALL, prompt=_log_int(rng, 1, 64), new=rng.randint(8, 64))
    elif kind == "layers":
        shape = rng.choice((SHAPE_7B, SHAPE_13B, SHAPE_65B))
        case = dict(kind=kind, f16=True, **shape, resident=rng.randint(2, 5), n=_log_int(rng, 1, 600))
    else:
        dim = 64 * _log_int(rng, 16, 80)
        case = dict(kind=kind, f16=f16, dim=dim, ffn=rllama_amd.llama_ffn_hidden(dim), n=_log_int(rng, 1, 512))
    return case


# ---------------------------------------------------------------------------------------------------------------------------

_context = None


def _ctx():
    """A program's one device context."""
    global _context
    if _context is None:
        _context = rllama_amd.Context(0)
    return _context


def _model(case, seed, max_seq_len):
    ctx = _ctx()
    settings = rllama_amd.DataSettings(ctx)
    if case["f16"]:
        settings = settings.force_f16()
    if "resident" in case:
        settings = settings.percentage_to_gpu((case["resident"] - 1) / (case["layers"] - 1))
    model = rllama_amd.Transformer(ctx, case["dim"], case["layers"], case["heads"], case["ffn"], VOCAB, max_seq_len, 1e-6, settings)
    model.fill_synthetic(seed, STD)
    return model


def _bits(t):
    return t.to(torch.float16).cpu().numpy().view(np.uint16)


def _clear_successors(model, seed):
    """Embedding and head under which token t is followed by another fixed token: the head's row of the successor has a part
    along t's embedding (a logit about 10 against a largest other one about 4)."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    emb = torch.randn(VOCAB, model.dim, generator=gen, device="cuda") * 0.5
    head = torch.randn(VOCAB, model.dim, generator=gen, device="cuda") * STD
    order = torch.randperm(VOCAB, generator=gen, device="cuda")
    head[order.roll(-1)] += emb[order] * (35.0 / model.dim)
    model.set_tensor(rllama_amd.TOK_EMB, 0, _bits(emb))
    model.set_tensor(rllama_amd.OUTPUT, 0, _bits(head))


def prepare(case, seed):
    kind = case["kind"]
    if kind == "ops":
        return _prepare_ops(case, seed)
    if kind == "layers":
        n, dim = case["n"], case["dim"]
        model = _model(case, seed, max(512, n))
        x = np.random.default_rng(seed).standard_normal((n, dim), dtype=np.float32)
        return dict(kind=kind, model=model, caches=model.make_caches(), x=x, last=model.last_layer_on_gpu())
    if kind == "greedy":
        model = _model(case, seed, 256)
        _clear_successors(model, seed)
        tokens = rllama_amd.synth_tokens(seed, case["prompt"], 3, VOCAB)
        return dict(kind=kind, model=model, caches=model.make_caches(), tokens=tokens, new=case["new"])
    if kind == "prompt":
        model = _model(case, seed, max(512, case["n"]))
        tokens = rllama_amd.synth_tokens(seed, case["n"], 3, VOCAB)
        return dict(kind=kind, model=model, caches=model.make_caches(), tokens=tokens)
    # decode: the caches hold the text so far
    pos = case["pos"]
    model = _model(case, seed, max(512, pos + 129))
    caches = model.make_caches()
    tokens = rllama_amd.synth_tokens(seed, pos + 1, 3, VOCAB)
    model.forward(tokens[:pos], 0, caches)
    sampler = None
    if "top_k" in case:
        sampler = rllama_amd.TokenSampler().temperature(0.8).top_k(case["top_k"]).repetition_penalty(1.1)
    return dict(kind=kind, model=model, caches=caches, token=tokens[pos:], text=tokens, pos=pos, sampler=sampler)


def _prepare_ops(case, seed):
    ctx = _ctx()
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def tensor(rows, cols, std):
        t = torch.randn(rows, cols, generator=gen, device="cuda") * std
        return rllama_amd.Tensor.from_numpy(ctx, _bits(t) if case["f16"] else t.cpu().numpy())

    n, d, f = case["n"], case["dim"], case["ffn"]
    return dict(kind="ops", f16=case["f16"], x=tensor(n, d, 1.0), w1=tensor(f, d, STD), w3=tensor(f, d, STD), w2=tensor(d, f, STD))


def run(state):
    kind = state["kind"]
    if kind == "ops":
        x, w1, w2, w3 = state["x"], state["w1"], state["w2"], state["w3"]
        if state["f16"]:
            mid = x.ffn_gate(w1, w3)
        else:
            mid = x.matrix_mul_transposed(w1).silu_mul(x.matrix_mul_transposed(w3))
        return mid.matrix_mul_transposed(w2).to_numpy()
    model, caches = state["model"], state["caches"]
    if kind == "layers":
        return model.forward_layers(state["x"], 0, caches, 0, state["last"])
    if kind == "greedy":
        tokens, new = state["tokens"], state["new"]
        ids, _, _ = model.generate_greedy(tokens, new, caches)
        # the step behind the last id: its logits rest on every cache row that the loop wrote
        logits = model.forward(ids[-1:], len(tokens) + new - 1, caches)
        return ids, logits
    if kind == "prompt":
        return model.forward(state["tokens"], 0, caches)
    logits = model.forward(state["token"], state["pos"], caches)
    if state["sampler"] is None:
        return logits
    # the candidates' ids are left out of what is compared: two probabilities that are nearly equal may change places
    _, probabilities, total = state["sampler"].candidates(logits, state["text"])
    return logits, probabilities, total


# ---------------------------------------------------------------------------------------------------------------------------


def _forward_work(case, n, past, layers, head):
    """Weights once, the cache rows of `past` positions read, n rows written; 2 flops per multiply-add, causal attention."""
    d, f, es = case["dim"], case["ffn"], 2 if case["f16"] else 4
    per_layer = 4 * d * d + 3 * d * f
    attended = n * past + n * (n + 1) / 2
    nbytes = layers * (per_layer * es + 2 * d * es * (past + n)) + (VOCAB * d * 2 + VOCAB * 4 if head else 2 * n * d * 4)
    flops = layers * (2.0 * n * per_layer + 4.0 * d * attended) + (2.0 * VOCAB * d if head else 0)
    return nbytes, flops


def work(case):
    kind = case["kind"]
    if kind == "ops":
        n, d, f, es = case["n"], case["dim"], case["ffn"], 2 if case["f16"] else 4
        return {"bytes": (3 * d * f + 2 * n * d) * es, "flops": 6.0 * n * d * f}
    if kind == "layers":
        calls = [_forward_work(case, case["n"], 0, case["resident"], False)]
    elif kind == "prompt":
        calls = [_forward_work(case, case["n"], 0, case["layers"], True)]
    elif kind == "decode":
        calls = [_forward_work(case, 1, case["pos"], case["layers"], True)]
    else:
        calls = [_forward_work(case, case["prompt"], 0, case["layers"], True)]
        calls += [_forward_work(case, 1, case["prompt"] + i, case["layers"], True) for i in range(case["new"])]
    return {"bytes": sum(c[0] for c in calls), "flops": sum(c[1] for c in calls)}


def tolerance(case):
    # Four times what one path differs from itself by with its sums in another order (prompts through the matrix cores against
    # the same prompts token by token; op-level products against float64).
    if case["kind"] == "ops":
        return {"rel": 4e-4, "max": 4e-3} if case["f16"] else {"rel": 5e-6, "max": 3e-5}
    layers, dim = case.get("resident", case["layers"]), case["dim"]
    if case["f16"]:
        # every product, activation and cache row is rounded to f16; another order of sums flips some of those roundings and the
        # flips add up through the layers: 4.4e-3 at 32 layers of dim 4096, 1.7e-3 at 9, 2.2e-3 at 20 of 2368, 0.8e-3 at 8 of 1024
        rel = 3e-3 * math.sqrt(layers * dim / 4096)
        if "top_k" in case:
            rel *= 1.6  # exp(logit / temperature): 6.7e-3 where the logits differ by 4.3e-3
    else:
        # no rounding points: 2.4e-5 at 32 layers of dim 4096, 1.4e-6 at 30 of 1408, 0.9e-6 at 7 of 1152
        rel = 1e-4 * math.sqrt(layers / 32) * (dim / 4096) ** 2
    return {"rel": rel, "max": 5 * rel}
