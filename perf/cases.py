"""The work that users of this package have it do, as measurable cases.

Encoders turn token ids into pooled embeddings, the flat index answers
queries, decoders take in prompts and then a token at a time. `listed` are
fixed sizes of these, `draw` gives others from the same ranges. Weights and
inputs are random, of the magnitudes that trained models and their caches
have; every model is of a size that this repository's presets or its
benchmark (`bench.py`) define, the decoders cut to the benchmark's eight
layers of width 4096 with 32768 tokens.
"""

from __future__ import annotations

import json
import math
import tempfile
from pathlib import Path

import numpy as np
import torch
import torch.nn.functional as F

from distllm_amd import ops
from distllm_amd.engine import LLMEngine
from distllm_amd.engine.engine import _Seq
from distllm_amd.models import ModelDims, build_model, get_dims
from distllm_amd.models.config import layered_preset

DEV = "cuda"
BLK = LLMEngine.BLK

# the decoder benchmark's layers (llama and Kanotar, 32 heads of 128)
WIDTH, HEADS, KV_HEADS, HEAD, FF, VOCAB, LAYERS = (
    4096, 32, 8, 128, 14336, 32768, 8)
Q_RANK, KV_RANK, LIMIT = 1536, 512, 7.0
MOST_TOKENS = 16384     # prompt tokens of one case, and of an engine step
MOST_CACHED = 131072    # cached tokens of one case


def listed() -> list[dict]:
    return [
        # a question of a retriever: one short text
        {"name": "embed-question", "kind": "text", "rows": 1, "longest": 24,
         "shortest": 24},
        # sentence buffers of the semantic-chunk embedder, padded together
        {"name": "embed-buffers", "kind": "text", "rows": 64,
         "longest": 203, "shortest": 40},
        # the benchmark's batch: 512 full sequences
        {"name": "embed-batch", "kind": "text", "rows": 512, "longest": 512,
         "shortest": 512},
        # proteins of a fasta file, lengths dispersed (packed path)
        {"name": "embed-proteins", "kind": "protein", "rows": 32,
         "longest": 1024, "shortest": 64},
        # a question against a corpus, and a batch of them (flat index)
        {"name": "search-question", "kind": "search", "rows": 1,
         "corpus": 250_000, "dim": 768, "top": 5},
        {"name": "search-batch", "kind": "search", "rows": 256,
         "corpus": 250_000, "dim": 768, "top": 10},
        # prompts of a generation run: retrieved passages and a question
        {"name": "prompts", "kind": "prompts", "rows": 16, "longest": 1024,
         "shortest": 256},
        # chat: one sequence, a token at a time; the same with 8-bit weights
        {"name": "decode-one", "kind": "decode", "rows": 1, "longest": 2048,
         "shortest": 2048, "weights": "bf16", "cache": "bf16"},
        {"name": "decode-one-fp8", "kind": "decode", "rows": 1,
         "longest": 1500, "shortest": 1500, "weights": "fp8",
         "cache": "bf16"},
        # a full batch of a generation run
        {"name": "decode-batch", "kind": "decode", "rows": 64,
         "longest": 2048, "shortest": 200, "weights": "bf16",
         "cache": "bf16"},
        # a decoder that is described layer by layer, through the engine
        {"name": "latent-prompts", "kind": "latent-prompts", "rows": 6,
         "longest": 2048, "shortest": 700, "window": 1024},
        {"name": "latent-decode", "kind": "latent-decode", "rows": 32,
         "longest": 2048, "shortest": 300, "window": 8192},
    ]


def _spread(rng, lo: int, hi: int) -> int:
    """A whole number from lo to hi, even over the logarithm."""
    return min(hi, max(lo, round(math.exp(
        rng.uniform(math.log(lo), math.log(hi + 0.5))))))


def draw(rng) -> dict:
    kind = rng.choice(["text", "text", "protein", "search", "prompts",
                       "decode", "decode", "latent-prompts",
                       "latent-decode"])
    if kind == "search":
        return {"kind": kind, "rows": _spread(rng, 1, 256),
                "corpus": _spread(rng, 20_000, 250_000),
                "dim": rng.choice([384, 768]),
                "top": rng.choice([1, 3, 5, 10, 20])}
    rows, longest, shortest = {
        "text": (512, 512, 8), "protein": (32, 1024, 30),
        "prompts": (32, 2048, 16), "decode": (128, 4096, 16),
        "latent-prompts": (8, 2048, 32), "latent-decode": (64, 4096, 16),
    }[kind]
    n = _spread(rng, shortest, longest)
    most = MOST_CACHED if kind.endswith("decode") else MOST_TOKENS
    if kind == "text":
        most = 512 * 512
    case = {"kind": kind, "rows": _spread(rng, 1, min(rows, most // n)),
            "longest": n}
    # batches of one length and of all sorts
    same = case["rows"] == 1 or rng.random() < 0.3
    case["shortest"] = n if same else rng.randint(shortest, n)
    if kind == "decode":
        case["weights"] = "fp8" if rng.random() < 0.25 else "bf16"
        case["cache"] = "fp8" if rng.random() < 0.25 else "bf16"
    if kind.startswith("latent"):
        case["window"] = rng.choice([1024, 8192])
    return case


def lengths(case: dict) -> list[int]:
    """Lengths of the case's sequences: evenly spread from its longest to
    its shortest, in an order that mixes them."""
    n, lo, hi = case["rows"], case["shortest"], case["longest"]
    if n == 1:
        return [hi]
    each = [hi - (hi - lo) * i // (n - 1) for i in range(n)]
    step = next(s for s in (7, 5, 3, 1) if math.gcd(s, n) == 1)
    return [each[i * step % n] for i in range(n)]


# ---- weights ----------------------------------------------------------------

def _generator(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(seed)


def _fill(shapes: dict, seed: int) -> dict[str, torch.Tensor]:
    """bf16 tensors: matrices of deviation 0.02, scales of norms around 1,
    biases around 0. Decoders have embeddings of deviation 1 and smaller
    output matrices of their 16 sublayers, so that a sublayer adds to the
    residual stream rather than replacing it, as in a trained model."""
    g = _generator(seed)
    out = {}
    for name, shape in shapes.items():
        t = torch.empty(shape, device=DEV, dtype=torch.float32)
        if len(shape) > 1:
            sd = 0.02
            if name in ("tok_emb", "embed"):
                sd = 1.0
            elif name.endswith((".wdown", ".mix.o", ".mlp.down")) or (
                    name.endswith(".wo") and "tok_emb" in shapes):
                sd = 0.005
            t.normal_(0.0, sd, generator=g)
        elif name.endswith(("_w", "norm")) or ".norm" in name:
            t.normal_(1.0, 0.1, generator=g)
        else:
            t.normal_(0.0, 0.02, generator=g)
        out[name] = t.to(torch.bfloat16)
    return out


def _encoder_dims(case: dict):
    return get_dims("pubmedbert-base" if case["kind"] == "text"
                    else "esm2-650m")


def _encoder_shapes(d) -> dict:
    H, I, bert = d.hidden_size, d.intermediate_size, d.arch == "bert"
    t = {"word_emb": (d.vocab_size, H)}
    if bert:
        t |= {"pos_emb": (d.max_position_embeddings, H),
              "type_emb": (d.type_vocab_size, H), "emb_ln_w": (H,),
              "emb_ln_b": (H,)}
    for i in range(d.num_layers):
        layer = {"wqkv": (3 * H, H), "bqkv": (3 * H,), "wo": (H, H),
                 "bo": (H,), "ln1_w": (H,), "ln1_b": (H,), "w1": (I, H),
                 "b1": (I,), "w2": (H, I), "b2": (H,), "ln2_w": (H,),
                 "ln2_b": (H,)}
        t |= {f"layers.{i}.{n}": s for n, s in layer.items()}
    if not bert:
        t |= {"final_ln_w": (H,), "final_ln_b": (H,)}
    return t


def _decoder_dims() -> ModelDims:
    return ModelDims(arch="llama", vocab_size=VOCAB, hidden_size=WIDTH,
                     num_layers=LAYERS, num_heads=HEADS,
                     num_kv_heads=KV_HEADS, intermediate_size=FF,
                     max_position_embeddings=16384)


def _decoder_shapes() -> dict:
    t = {"tok_emb": (VOCAB, WIDTH)}
    for i in range(LAYERS):
        layer = {"wqkv": ((HEADS + 2 * KV_HEADS) * HEAD, WIDTH),
                 "wo": (WIDTH, HEADS * HEAD), "in_norm": (WIDTH,),
                 "post_norm": (WIDTH,), "wgup": (2 * FF, WIDTH),
                 "wdown": (WIDTH, FF)}
        t |= {f"layers.{i}.{n}": s for n, s in layer.items()}
    return t | {"final_norm": (WIDTH,), "lm_head": (VOCAB, WIDTH)}


def _latent_dims(case: dict):
    return layered_preset(LAYERS, WIDTH, VOCAB, HEADS, HEAD, HEAD, Q_RANK,
                          KV_RANK, FF, [case["window"]], limit=LIMIT)


def _latent_shapes() -> dict:
    t = {"embed": (VOCAB, WIDTH), "head": (VOCAB, WIDTH),
         "final.norm": (WIDTH,)}
    for i in range(LAYERS):
        layer = {"norm1": (WIDTH,), "norm1b": (WIDTH,), "norm2": (WIDTH,),
                 "norm2b": (WIDTH,), "mix.dq": (Q_RANK, WIDTH),
                 "mix.dq.norm": (Q_RANK,),
                 "mix.uq": (HEADS * HEAD, Q_RANK),
                 "mix.dkv": (KV_RANK, WIDTH), "mix.dkv.norm": (KV_RANK,),
                 "mix.uk": (HEADS * HEAD, KV_RANK),
                 "mix.uv": (HEADS * HEAD, KV_RANK),
                 "mix.o": (WIDTH, HEADS * HEAD), "mlp.gate": (FF, WIDTH),
                 "mlp.up": (FF, WIDTH), "mlp.down": (WIDTH, FF)}
        t |= {f"l{i}.{n}": s for n, s in layer.items()}
    return t


def _built(dims, own: dict, raw: bool = False):
    """A model of these dims with these weights (raw: named as in a
    checkpoint)."""
    with torch.device(DEV):
        model = build_model(dims, device=DEV)
    with torch.no_grad():
        source = model.checkpoint(own) if raw else own
        for name, p in model.named_parameters():
            p.copy_(source[name])
    return model


# ---- inputs -----------------------------------------------------------------

def _padded_tokens(case: dict, seed: int):
    """Right-padded ids (words or, of proteins, residues) and their mask."""
    n = lengths(case)
    pad, end = {"text": (0, 30528), "protein": (1, 24),
                "prompts": (0, VOCAB)}[case["kind"]]
    ids = torch.randint(4, end, (len(n), max(n)), device=DEV,
                        generator=_generator(seed + 1))
    at = torch.arange(max(n), device=DEV)[None]
    mask = (at < torch.tensor(n, device=DEV)[:, None]).int()
    return torch.where(mask.bool(), ids, pad), mask


def _unit(x: torch.Tensor) -> torch.Tensor:
    return x / x.norm(dim=-1, keepdim=True)


def _corpus(case: dict, seed: int):
    """Unit embeddings around 64 topics, and queries close to some."""
    g = _generator(seed)

    def noise(n):
        return torch.randn(n, case["dim"], device=DEV, generator=g)

    topics = noise(64)

    def some(n):
        of = torch.randint(0, 64, (n,), device=DEV, generator=g)
        return _unit(0.7 * topics[of] + noise(n))

    return some(case["corpus"]), some(case["rows"])


def _paging(case: dict):
    """Block table and block count of sequences whose blocks follow one
    another; block 0 is reserved."""
    need = [-(-n // BLK) for n in lengths(case)]
    table = torch.zeros(len(need), max(need), dtype=torch.int32)
    at = 1
    for i, n in enumerate(need):
        table[i, :n] = torch.arange(at, at + n, dtype=torch.int32)
        at += n
    return table.to(DEV), at


def _cached(case: dict, seed: int, blocks: int) -> list[torch.Tensor]:
    """Keys and values (rows of unit deviation, as a normed input times
    matrices of deviation 0.02 has), layer by layer."""
    g = _generator(seed + 2)
    out = []
    for _ in range(2 * LAYERS):
        t = torch.randn(blocks, KV_HEADS, BLK, HEAD, device=DEV,
                        generator=g, dtype=torch.bfloat16)
        if case["cache"] == "fp8":
            t = t.to(torch.float8_e4m3fn).view(torch.uint8)
        out.append(t)
    return out


def _latents(case: dict, seed: int, blocks: int) -> list[torch.Tensor]:
    g = _generator(seed + 2)
    return [torch.randn(blocks, BLK, KV_RANK, device=DEV, generator=g,
                        dtype=torch.bfloat16) for _ in range(LAYERS)]


def _next_tokens(case: dict, seed: int) -> torch.Tensor:
    return torch.randint(4, VOCAB, (case["rows"],), device=DEV,
                         generator=_generator(seed + 1))


def _prompts(case: dict, seed: int) -> list[list[int]]:
    g = _generator(seed + 1)
    return [torch.randint(4, VOCAB, (n,), device=DEV, generator=g).tolist()
            for n in lengths(case)]


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    state = {"kind": kind}
    if kind in ("text", "protein"):
        d = _encoder_dims(case)
        state["model"] = _built(d, _fill(_encoder_shapes(d), seed))
        state["ids"], state["mask"] = _padded_tokens(case, seed)
    elif kind == "search":
        from datasets import Dataset

        from distllm_amd.rag.search import HipFlatIndex

        corpus, queries = _corpus(case, seed)
        with tempfile.TemporaryDirectory() as tmp:
            # the index file that a first run leaves beside the texts
            np.savez(Path(tmp) / "index.npz", embeddings=corpus.cpu().numpy(),
                     meta=json.dumps({"precision": "float32",
                                      "dim": case["dim"]}))
            Dataset.from_dict({"text": ["passage"]}).save_to_disk(
                str(Path(tmp) / "texts"))
            state["index"] = HipFlatIndex(Path(tmp) / "texts",
                                          Path(tmp) / "index.npz")
        state["queries"], state["top"] = queries.cpu().numpy(), case["top"]
    elif kind == "prompts":
        state["model"] = _built(_decoder_dims(),
                                _fill(_decoder_shapes(), seed))
        state["ids"], state["mask"] = _padded_tokens(case, seed)
        state["rows"] = torch.arange(case["rows"], device=DEV)
        state["last"] = state["mask"].sum(1) - 1
    elif kind == "decode":
        _prepare_decode(case, seed, state)
    else:
        _prepare_latent(case, seed, state)
    return state


@torch.no_grad()
def _prepare_decode(case: dict, seed: int, state: dict) -> None:
    """A decode step in a captured graph, as the engine keeps them."""
    model = _built(_decoder_dims(), _fill(_decoder_shapes(), seed))
    if case["weights"] == "fp8":
        model.enable_fp8_decode()
    table, blocks = _paging(case)
    cache = model.make_cache(blocks, BLK, "fp8_e4m3" if case["cache"] == "fp8"
                             else "bf16")
    for own, filled in zip(cache.k + cache.v, _cached(case, seed, blocks)):
        own.copy_(filled)
    tokens = _next_tokens(case, seed)
    ctx = torch.tensor(lengths(case), dtype=torch.int32, device=DEV)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            model.decode_step(tokens, cache, table, ctx)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        logits = model.decode_step(tokens, cache, table, ctx)
    state |= {"model": model, "cache": cache, "inputs": (tokens, table, ctx),
              "graph": graph, "logits": logits}


def _prepare_latent(case: dict, seed: int, state: dict) -> None:
    model = _built(_latent_dims(case), _fill(_latent_shapes(), seed), True)
    n = lengths(case)
    _, blocks = _paging(case)
    engine = LLMEngine(model, max_batch_size=case["rows"],
                       max_model_len=max(n), num_blocks=blocks - 1)
    state["engine"] = engine
    if case["kind"] == "latent-prompts":
        state["prompts"] = _prompts(case, seed)
        return
    engine.warm_graphs([case["rows"]])
    for own, filled in zip(engine.cache.layers,
                           _latents(case, seed, blocks)):
        own.copy_(filled)
    state["seqs"] = [_Seq(seq_id=i, prompt_ids=[], cached=m - 1,
                          blocks=engine.blockman.alloc(-(-m // BLK)))
                     for i, m in enumerate(n)]
    state["tokens"] = [[t] for t in _next_tokens(case, seed).tolist()]


# ---- one pass ---------------------------------------------------------------

@torch.no_grad()
def run(state: dict):
    kind = state["kind"]
    if kind in ("text", "protein"):
        hidden = state["model"](state["ids"], state["mask"])
        return ops.mean_pool(hidden, state["mask"], normalize=True)
    if kind == "search":
        found = state["index"].search(state["queries"], top_k=state["top"])
        return {"scores": np.array(found.total_scores, np.float32),
                "indices": np.array(found.total_indices, np.int64)}
    if kind == "prompts":
        hidden, kv = state["model"].prefill(state["ids"], state["mask"])
        last = hidden[state["rows"], state["last"]]
        return {"logits": state["model"].logits(last), "kv": kv}
    if kind == "decode":
        state["graph"].replay()
        return {"logits": state["logits"],
                "kv": list(zip(state["cache"].k, state["cache"].v))}
    engine = state["engine"]
    if kind == "latent-prompts":
        seqs = [_Seq(seq_id=i, prompt_ids=p)
                for i, p in enumerate(state["prompts"])]
        logits = engine.step([(s, s.prompt_ids) for s in seqs],
                             [[len(s.prompt_ids) - 1] for s in seqs])
        for s in seqs:
            engine.release(s)
    else:
        logits = engine.step(list(zip(state["seqs"], state["tokens"])),
                             [[0]] * len(state["seqs"]))
        for s in state["seqs"]:  # the same token again in the next pass
            s.cached -= 1
    return {"logits": logits, "latents": engine.cache.layers}


# ---- what a pass cannot do without --------------------------------------------

def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "search":
        n, q, d = case["corpus"], case["rows"], case["dim"]
        return {"bytes": 4 * d * (n + q) + 8 * q * case["top"],
                "flops": 2 * n * q * d}
    n = lengths(case)
    total = sum(n)
    if kind in ("text", "protein"):
        d = _encoder_dims(case)
        shapes = _encoder_shapes(d)
        H, L, bert = d.hidden_size, d.num_layers, kind == "text"
        per_layer = 4 * H * H + 2 * H * d.intermediate_size
        held = sum(math.prod(s) for k, s in shapes.items()
                   if k.startswith("layers") or k == "pos_emb")
        seen = min(total, d.vocab_size)
        return {"bytes": 2 * (held + seen * H) + 8 * total
                + 4 * len(n) * H,
                "flops": L * (2 * per_layer * total
                              + 4 * H * sum(m * m for m in n))}
    if kind in ("prompts", "decode"):
        layer = (WIDTH * (HEADS + 2 * KV_HEADS) * HEAD
                 + WIDTH * HEADS * HEAD + 3 * WIDTH * FF)
        head, kv = WIDTH * VOCAB, 2 * KV_HEADS * HEAD
        rows = total if kind == "prompts" else len(n)
        pairs = (sum(m * (m + 1) // 2 for m in n) if kind == "prompts"
                 else total)
        el = 1 if case.get("cache") == "fp8" else 2
        wel = 1 if case.get("weights") == "fp8" and len(n) <= 8 else 2
        return {"bytes": LAYERS * (wel * layer + el * kv * total)
                + 2 * head + 2 * WIDTH * rows + 4 * VOCAB * len(n),
                "flops": LAYERS * (2 * layer * rows
                                   + 4 * HEADS * HEAD * pairs)
                + 2 * head * len(n)}
    layer = (WIDTH * (Q_RANK + KV_RANK) + Q_RANK * HEADS * HEAD
             + HEADS * HEAD * WIDTH + 3 * WIDTH * FF)
    up, head = 2 * KV_RANK * HEADS * HEAD, WIDTH * VOCAB
    w = case["window"]
    if kind == "latent-prompts":
        rows = total
        pairs = sum(m * (m + 1) // 2 - max(0, m - w) * (m - w + 1) // 2
                    for m in n)
        dot = 4 * HEADS * HEAD
        cached = total
    else:  # in the latent space, where every head reads the same latent
        rows, pairs, dot = len(n), sum(min(m, w) for m in n), (
            4 * HEADS * KV_RANK)
        cached = pairs
    return {"bytes": LAYERS * 2 * (layer + up + KV_RANK * cached)
            + 2 * head + 2 * WIDTH * rows + 4 * VOCAB * len(n),
            "flops": LAYERS * (2 * (layer + up) * rows + dot * pairs)
            + 2 * head * len(n)}


def tolerance(case: dict):
    """About four times the distance between this package's outputs and
    those of `exact`: bf16 between the products of 12 post-normed, 33 and 8
    layers; new keys and values that are rounded to 8 bits may fall on the
    neighbouring number."""
    kind = case["kind"]
    if kind == "search":
        return {"rel": 2e-6, "differ": 0.01}
    rel = {"text": 0.013, "protein": 0.025, "prompts": 0.03,
           "decode": 0.03 if case.get("cache") == "fp8" else 0.02}
    return {"rel": rel.get(kind, 0.025), "max": 0.2, "differ": 0.01}


# ---- the same in 64 bits --------------------------------------------------------

def _linear(x, t, w, b=None):
    y = x @ t[w].double().T
    return y if b is None else y + t[b].double()


def _layer_norm(x, t, w, b, eps):
    return F.layer_norm(x, x.shape[-1:], t[w].double(), t[b].double(), eps)


def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _attend(q, k, v, hidden_keys):
    """q [B, S, H, D] against k, v [B, T, HKV, D]; hidden_keys broadcasts to
    [B, H, S, T]. A few heads at a time."""
    rep = q.shape[2] // k.shape[2]
    out = torch.empty_like(q)
    for h in range(0, q.shape[2], 4):
        kv = [h // rep] if rep >= 4 else list(range(h // rep, h // rep + 4
                                                    // rep))
        kk, vv = (x[:, :, kv].repeat_interleave(min(rep, 4), 2)
                  [:, :, : min(4, q.shape[2] - h)].transpose(1, 2)
                  for x in (k, v))
        qq = q[:, :, h: h + 4].transpose(1, 2)
        s = qq @ kk.transpose(2, 3) / math.sqrt(q.shape[3])
        p = s.masked_fill_(hidden_keys, -math.inf).softmax(-1)
        out[:, :, h: h + 4] = (p @ vv).transpose(1, 2)
    return out


def _rotated(x, pos):
    """Rotary positions over the two halves; x [B, S, H, D], pos [B, S]."""
    D = x.shape[-1]
    inv = 10000.0 ** (-torch.arange(0, D, 2, device=DEV,
                                    dtype=torch.float64) / D)
    ang = pos[..., None].double() * inv
    c, s = ang.cos()[:, :, None], ang.sin()[:, :, None]
    a, b = x[..., : D // 2], x[..., D // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _exact_encoder(case: dict, seed: int):
    d = _encoder_dims(case)
    t = _fill(_encoder_shapes(d), seed)
    bert = case["kind"] == "text"
    ids, mask = _padded_tokens(case, seed)
    H, eps = d.hidden_size, d.layer_norm_eps
    out = []
    for b in range(0, len(ids), 64):
        i, m = ids[b: b + 64], mask[b: b + 64].bool()
        B, S = i.shape
        pos = torch.arange(S, device=DEV).expand(B, S)
        x = t["word_emb"][i].double()
        if bert:
            x = x + t["pos_emb"][:S].double() + t["type_emb"][0].double()
            x = _layer_norm(x, t, "emb_ln_w", "emb_ln_b", eps)
        else:  # nothing is masked: the rescaling of token dropout
            x = x * (1 - 0.15 * 0.8)
        hidden = ~m[:, None, None]
        for n in range(d.num_layers):
            p = f"layers.{n}."
            h = x if bert else _layer_norm(x, t, p + "ln1_w", p + "ln1_b",
                                           eps)
            q, k, v = (y.reshape(B, S, d.num_heads, -1) for y in
                       _linear(h, t, p + "wqkv", p + "bqkv").split(H, -1))
            if not bert:
                q, k = _rotated(q, pos), _rotated(k, pos)
            y = _linear(_attend(q, k, v, hidden).reshape(B, S, H), t,
                        p + "wo", p + "bo")
            x = x + y
            if bert:
                h = x = _layer_norm(x, t, p + "ln1_w", p + "ln1_b", eps)
            else:
                h = _layer_norm(x, t, p + "ln2_w", p + "ln2_b", eps)
            x = x + _linear(F.gelu(_linear(h, t, p + "w1", p + "b1")), t,
                            p + "w2", p + "b2")
            if bert:
                x = _layer_norm(x, t, p + "ln2_w", p + "ln2_b", eps)
        if not bert:
            x = _layer_norm(x, t, "final_ln_w", "final_ln_b", eps)
        use = m.double()  # the mean leaves out the first and last token
        use[:, 0] = 0
        use.scatter_(1, m.sum(1, keepdim=True) - 1, 0.0)
        y = (x * use[..., None]).sum(1) / use.sum(1, keepdim=True).clamp(1)
        out.append(F.normalize(y, dim=-1))
    return torch.cat(out)


def _swiglu(h, t, pre, w):
    g, u = _linear(h, w, pre + "wgup").split(FF, -1)
    return _linear(F.silu(g) * u, w, pre + "wdown")


def _qkv(h, w, pre, pos):
    B, S, _ = h.shape
    qkv = _linear(h, w, pre + "wqkv").view(B, S, HEADS + 2 * KV_HEADS, HEAD)
    rot = _rotated(qkv[:, :, : HEADS + KV_HEADS], pos)
    return (rot[:, :, :HEADS], rot[:, :, HEADS:],
            qkv[:, :, HEADS + KV_HEADS:])


def _exact_prompts(case: dict, seed: int):
    t = _fill(_decoder_shapes(), seed)
    ids, mask = _padded_tokens(case, seed)
    parts = []
    for b in range(0, len(ids), 2):
        i, m = ids[b: b + 2], mask[b: b + 2].bool()
        B, S = i.shape
        pos = torch.arange(S, device=DEV).expand(B, S)
        hidden = (~m[:, None, None]
                  | (pos[0][None] > pos[0][:, None])[None, None])
        x, kv = t["tok_emb"][i].double(), []
        for n in range(LAYERS):
            p = f"layers.{n}."
            q, k, v = _qkv(_rms(x, t[p + "in_norm"], 1e-5), t, p, pos)
            kv.append((k, v))
            y = _attend(q, k, v, hidden).reshape(B, S, HEADS * HEAD)
            x = x + _linear(y, t, p + "wo")
            x = x + _swiglu(_rms(x, t[p + "post_norm"], 1e-5), t, p, t)
        last = x[torch.arange(B, device=DEV), m.sum(1) - 1]
        parts.append((_linear(_rms(last, t["final_norm"], 1e-5), t,
                              "lm_head"), kv))
    return {"logits": torch.cat([a for a, _ in parts]),
            "kv": [tuple(torch.cat([kv[n][j] for _, kv in parts])
                         for j in (0, 1)) for n in range(LAYERS)]}


def _eight_bits(w: torch.Tensor) -> torch.Tensor:
    """The numbers that a matrix has after 8-bit storage with a scale per
    row."""
    s = (w.float().abs().amax(1, keepdim=True) / 448.0).clamp_min(1e-12)
    q = (w.float() / s).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
    return q.double() * s.double()


def _exact_decode(case: dict, seed: int):
    t = _fill(_decoder_shapes(), seed)
    if case["weights"] == "fp8" and case["rows"] <= 8:
        for n in t:
            if n.startswith("layers") and t[n].dim() > 1:
                t[n] = _eight_bits(t[n])
    table, blocks = _paging(case)
    cached = _cached(case, seed, blocks)
    fp8 = case["cache"] == "fp8"
    n = torch.tensor(lengths(case), device=DEV)
    B = len(n)
    at = (n - 1)[:, None]
    where = table.long()[torch.arange(B, device=DEV), (n - 1) // BLK]
    x, kv = t["tok_emb"][_next_tokens(case, seed)].double()[:, None], []
    for i in range(LAYERS):
        p = f"layers.{i}."
        q, k, v = _qkv(_rms(x, t[p + "in_norm"], 1e-5), t, p, at)
        pages = []
        for old, new in ((cached[i], k), (cached[LAYERS + i], v)):
            if fp8:
                old = old.view(torch.float8_e4m3fn)
                new = new.to(torch.float8_e4m3fn)
            old = old.double()
            old[where, :, (n - 1) % BLK] = new[:, 0].double()
            pages.append(old)
        y = torch.empty(B, 1, HEADS * HEAD, dtype=torch.float64, device=DEV)
        for b in range(B):
            kk, vv = (pg[table[b].long()].transpose(0, 1)
                      .reshape(KV_HEADS, -1, HEAD)[:, : n[b]]
                      for pg in pages)
            qq = q[b, 0].view(KV_HEADS, HEADS // KV_HEADS, HEAD)
            s = qq @ kk.transpose(1, 2) / math.sqrt(HEAD)
            y[b, 0] = (s.softmax(-1) @ vv).reshape(-1)
        kv.append((None, None) if fp8 else tuple(pages))
        x = x + _linear(y, t, p + "wo")
        x = x + _swiglu(_rms(x, t[p + "post_norm"], 1e-5), t, p, t)
    return {"logits": _linear(_rms(x[:, 0], t["final_norm"], 1e-5), t,
                              "lm_head"), "kv": kv}


def _latent_layer(x, t, p, c, visible):
    """x [S, width] joined by a layer; c [T, rank] latents, visible [S, T]."""
    eps = 1e-5
    h = _rms(x, t[p + "norm1"], eps)
    q = _linear(_rms(_linear(h, t, p + "mix.dq"), t[p + "mix.dq.norm"], eps),
                t, p + "mix.uq").view(-1, HEADS, HEAD)
    k = _linear(c, t, p + "mix.uk").view(-1, HEADS, HEAD)
    v = _linear(c, t, p + "mix.uv").view(-1, HEADS, HEAD)
    y = _attend(q[None], k[None], v[None], ~visible[None, None])
    y = _linear(y.reshape(len(x), -1), t, p + "mix.o")
    x = x + _rms(y, t[p + "norm1b"], eps)
    h = _rms(x, t[p + "norm2"], eps)
    g = _linear(h, t, p + "mlp.gate").clamp(max=LIMIT)
    u = _linear(h, t, p + "mlp.up").clamp(-LIMIT, LIMIT)
    y = _linear(g * torch.sigmoid(1.702 * g) * (u + 1), t, p + "mlp.down")
    return x + _rms(y, t[p + "norm2b"], eps)


def _exact_latent(case: dict, seed: int):
    t = _fill(_latent_shapes(), seed)
    table, blocks = _paging(case)
    n, w = lengths(case), case["window"]
    prompts = case["kind"] == "latent-prompts"
    if prompts:
        tokens = _prompts(case, seed)
        pages = [torch.zeros(blocks, BLK, KV_RANK, dtype=torch.float64,
                             device=DEV) for _ in range(LAYERS)]
    else:
        tokens = [[i] for i in _next_tokens(case, seed).tolist()]
        pages = [c.double() for c in _latents(case, seed, blocks)]
    logits = []
    for b, m in enumerate(n):
        first = m - len(tokens[b])
        pos = torch.arange(m, device=DEV)
        ago = pos[first:, None] - pos[None]
        visible = (ago >= 0) & (ago < w)
        rows = table[b].long()[pos // BLK] * BLK + pos % BLK
        x = t["embed"][tokens[b]].double()
        for i in range(LAYERS):
            p, flat = f"l{i}.", pages[i].view(-1, KV_RANK)
            h = _rms(x, t[p + "norm1"], 1e-5)
            flat[rows[first:]] = _rms(_linear(h, t, p + "mix.dkv"),
                                      t[p + "mix.dkv.norm"], 1e-5)
            x = _latent_layer(x, t, p, flat[rows], visible)
        logits.append(_linear(_rms(x[-1:], t["final.norm"], 1e-5), t,
                              "head"))
    return {"logits": torch.cat(logits), "latents": pages}


@torch.no_grad()
def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind in ("text", "protein"):
        return _exact_encoder(case, seed)
    if kind == "search":
        corpus, queries = _corpus(case, seed)
        v, i = torch.topk(queries.double() @ corpus.double().T, case["top"])
        return {"scores": v, "indices": i}
    if kind == "prompts":
        return _exact_prompts(case, seed)
    if kind == "decode":
        return _exact_decode(case, seed)
    return _exact_latent(case, seed)
