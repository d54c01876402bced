"""The work a serving program has this package do, as measurable cases.

Kinds of case (``case["kind"]``):

* ``decode``: one paged-attention call of a decode step (one query row per
  sequence), optionally with decode rows that share a cached prefix.
* ``prefill``: one paged-attention call of prompt chunks, each at an offset
  into its sequence.
* ``step``: the decoder stack's forward over one packed batch (decode rows
  first, then prompt chunks), eager, as the engine runs every step that
  holds a chunk; with ``head`` the logits of each sequence's last row.
* ``graph``: a decode-only step of a whole model through
  ``ModelRunner.execute_model``, replaying the captured graph as the engine
  does.
* ``sample``: the fused greedy / temperature sampler over a batch of logits.

Sizes are those of the repository's benchmark (Qwen3-0.6B shape, the mixed
step under an 8192-token budget, the 151936-wide sampler, the tiny fp32
Llama) and of its tests (other head layouts, long contexts).

Context and chunk lengths are spread evenly over the case's range, so the
work of a case does not depend on the seed; their order, the block tables and
every value do.
"""

from __future__ import annotations

import math
import random
import sys
from pathlib import Path

import torch

_PKG = str(Path(__file__).resolve().parent.parent / "lite-vllm_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from litevllm import ops  # noqa: E402
from litevllm.cache.block_manager import BlockManager  # noqa: E402
from litevllm.config import (CacheConfig, EngineConfig, ModelConfig, SamplingParams,  # noqa: E402
                             SchedulerConfig)
from litevllm.engine.model_runner import ModelRunner  # noqa: E402
from litevllm.engine.sequence import SequenceGroup  # noqa: E402
from litevllm.layers.attention import AttentionMetadata  # noqa: E402
from litevllm.layers.sampler import Sampler  # noqa: E402
from litevllm.models.base import BaseModelForCausalLM  # noqa: E402

BS = 16
VOCAB = 151936
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}

SHAPES = {
    "qwen3": dict(model_type="qwen3", vocab_size=VOCAB, hidden_size=1024,
                  num_attention_heads=16, num_key_value_heads=8, head_dim=128,
                  intermediate_size=3072, rope_theta=1e6, rms_norm_eps=1e-6,
                  max_position_embeddings=40960, tie_word_embeddings=False),
    "tiny_llama": dict(model_type="llama", vocab_size=32000, hidden_size=256,
                       num_attention_heads=4, num_key_value_heads=2, head_dim=64,
                       intermediate_size=688, rope_theta=10000.0, rms_norm_eps=1e-6,
                       max_position_embeddings=4096, tie_word_embeddings=False),
}


# -- cases ---------------------------------------------------------------------

def _decode(name, heads, rows, lo, hi, dtype="bf16", shared=0, sharers=0):
    h, hkv, d = heads
    return dict(name=name, kind="decode", H=h, Hkv=hkv, D=d, dtype=dtype, rows=rows, ctx_lo=lo,
                ctx_hi=hi, shared=shared, sharers=sharers)


def _prefill(name, heads, chunks, len_lo, len_hi, off_lo, off_hi, dtype="bf16"):
    h, hkv, d = heads
    return dict(name=name, kind="prefill", H=h, Hkv=hkv, D=d, dtype=dtype, chunks=chunks,
                len_lo=len_lo, len_hi=len_hi, off_lo=off_lo, off_hi=off_hi)


def _step(name, shape, layers, rows, lo, hi, chunks, len_lo, len_hi, off_lo, off_hi, head,
          dtype="bf16"):
    return dict(name=name, kind="step", shape=shape, layers=layers, dtype=dtype, rows=rows,
                ctx_lo=lo, ctx_hi=hi, chunks=chunks, len_lo=len_lo, len_hi=len_hi, off_lo=off_lo,
                off_hi=off_hi, head=head)


def _graph(name, layers, rows, lo, hi, dtype="bf16"):
    return dict(name=name, kind="graph", shape="qwen3", layers=layers, dtype=dtype, rows=rows,
                ctx_lo=lo, ctx_hi=hi)


def _sample(name, rows, vocab, dtype="bf16"):
    return dict(name=name, kind="sample", rows=rows, vocab=vocab, dtype=dtype)


def listed():
    return [
        # one user's next token: latency of the attention call
        _decode("decode_one", (16, 8, 128), 1, 1500, 1500),
        # a full serving batch at the Qwen3-0.6B attention shape
        _decode("decode_256", (16, 8, 128), 256, 128, 2048),
        # a medium batch of a model with four query heads per kv head
        _decode("decode_gqa4", (32, 8, 128), 48, 256, 4096),
        # a few long documents, two kv heads of eight query heads each
        _decode("decode_long", (16, 2, 128), 5, 16000, 32768, dtype="fp16"),
        # a full batch, half of it on one cached 512-token system prompt
        _decode("decode_shared_256", (16, 8, 128), 256, 528, 2048, shared=32, sharers=128),
        # one fresh prompt: time to first token
        _prefill("prefill_one", (16, 8, 128), 1, 777, 777, 0, 0),
        # the chunks of a full mixed step
        _prefill("prefill_chunks", (16, 8, 128), 15, 512, 512, 0, 3072),
        # one decoder layer over a full mixed step (8192-token budget)
        _step("layer_mixed", "qwen3", 1, 192, 256, 4096, 15, 512, 512, 0, 3072, head=False),
        # a decode step of a full batch, from token ids to logits
        _graph("model_decode_256", 4, 256, 128, 2048),
        # the same for a handful of users
        _graph("model_decode_8", 4, 8, 128, 4096),
        # the sampler behind a full batch, half greedy, half temperature
        _sample("sample_256", 256, VOCAB),
        # the smallest model the repository runs end to end, in fp32: eight
        # short prompts from token ids to logits
        _step("tiny_llama_fp32", "tiny_llama", 2, 0, 0, 0, 8, 16, 64, 0, 0, head=True,
              dtype="fp32"),
    ]


HEADS = [(16, 8, 128), (16, 8, 128), (32, 8, 128), (16, 2, 128), (32, 4, 64), (8, 8, 128),
         (16, 4, 64)]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode"] * 4 + ["shared"] + ["prefill"] * 3 + ["step"] * 2 + ["graph"] * 2
                      + ["sample"] * 2 + ["tiny"])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16"])
    if kind == "decode":
        heads = rng.choice(HEADS)
        rows = _log(rng, 1, 256)
        hi = _log(rng, 48, min(32768, 280_000 // rows))
        c = _decode("", heads, rows, rng.randint(max(1, hi // 8), hi), hi, dtype=dtype)
    elif kind == "shared":
        heads = rng.choice(HEADS)
        rows = _log(rng, 16, 256)
        shared = rng.randint(8, 64)
        hi = rng.randint(shared * BS + 32, 2048)
        c = _decode("", heads, rows, shared * BS + rng.randint(1, 31), hi, dtype=dtype,
                    shared=shared, sharers=rng.randint(max(2, rows // 3), rows))
    elif kind == "prefill":
        heads = rng.choice(HEADS)
        chunks = _log(rng, 1, 15)
        hi = _log(rng, 20, 4096 if chunks == 1 else 512)
        off = rng.choice([0, rng.randint(1, 3072)])
        c = _prefill("", heads, chunks, rng.randint(max(2, hi // 4), hi), hi, 0, off, dtype=dtype)
    elif kind == "step":
        rows = rng.choice([0, _log(rng, 1, 192)])
        hi = _log(rng, 64, 4096)
        chunks = _log(rng, 1, 15)
        clen = _log(rng, 24, 512)
        off = rng.choice([0, rng.randint(1, 3072)])
        c = _step("", "qwen3", 1, rows, rng.randint(hi // 8, hi) if rows else 0,
                  hi if rows else 0, chunks, rng.randint(clen // 2, clen), clen, 0, off,
                  head=rng.random() < 0.3, dtype=dtype)
    elif kind == "graph":
        rows = _log(rng, 1, 256)
        hi = _log(rng, 64, min(8192, 280_000 // rows))
        c = _graph("", rng.randint(2, 4), rows, rng.randint(max(2, hi // 8), hi), hi)
    elif kind == "sample":
        c = _sample("", _log(rng, 1, 256), rng.choice([32000, 128256, VOCAB, VOCAB]),
                    dtype=rng.choice(["bf16", "bf16", "fp16", "fp32"]))
    else:
        rows = rng.choice([0, rng.randint(1, 8)])
        hi = rng.randint(16, 64)
        c = _step("", "tiny_llama", 2, rows, 8 if rows else 0, rng.randint(16, 256) if rows else 0,
                  rng.randint(1, 8), rng.randint(8, hi), hi, 0, 0, head=True, dtype="fp32")
    del c["name"]
    return c


# -- lengths -------------------------------------------------------------------

def _spread(n, lo, hi):
    """n lengths spread evenly over lo..hi."""
    return [lo + int((hi - lo) * (i + 0.5) / n) for i in range(n)]


def _decode_lens(case):
    lens = _spread(case["rows"], case["ctx_lo"], case["ctx_hi"])
    random.Random(3).shuffle(lens)   # which of them share a prefix
    return lens


def _chunk_lens(case):
    """(query tokens, offset) of every chunk."""
    lens = _spread(case["chunks"], case["len_lo"], case["len_hi"])
    offs = _spread(case["chunks"], case["off_lo"], case["off_hi"])
    random.Random(4).shuffle(offs)
    return list(zip(lens, offs))


def _blocks(n):
    return -(-n // BS)


# -- inputs --------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(shape, g, dtype, std=1.0):
    out = torch.empty(shape, dtype=dtype, device="cuda")
    return out.normal_(0.0, std, generator=g)


def _tables(nblocks, seed, shared=0, members=()):
    """Block tables over a shuffled pool that just fits them (block 0 is left
    out, as in a cache with a scratch block); the rows of ``members`` start
    with the same ``shared`` blocks.  Returns (tables, pool blocks)."""
    members = set(members)
    need = shared + sum(n - (shared if i in members else 0) for i, n in enumerate(nblocks))
    pool = list(range(1, need + 1))
    random.Random(seed).shuffle(pool)
    common, at = pool[:shared], shared
    tables = []
    for i, n in enumerate(nblocks):
        own = n - (shared if i in members else 0)
        tables.append((common if i in members else []) + pool[at:at + own])
        at += own
    return tables, need + 1


def _padded(tables):
    width = max(len(t) for t in tables)
    return torch.tensor([t + [0] * (width - len(t)) for t in tables], dtype=torch.int32)


def _attention_inputs(case, seed):
    """Sequences [(query tokens, context)], tables and tensors of one
    attention call."""
    shared, members = 0, ()
    if case["kind"] == "decode":
        lens = _decode_lens(case)
        order = list(range(len(lens)))
        random.Random(seed).shuffle(order)
        shared = case["shared"]
        members = [r for r, i in enumerate(order) if shared and i < case["sharers"]]
        seqs = [(1, lens[i]) for i in order]
    else:
        seqs = [(n, n + o) for n, o in _chunk_lens(case)]
        random.Random(seed).shuffle(seqs)
    tables, pool = _tables([_blocks(c) for _, c in seqs], seed, shared, members)
    g, dt = _gen(seed), DTYPES[case["dtype"]]
    T = sum(q for q, _ in seqs)
    query = _randn((T, case["H"], case["D"]), g, dt)
    kc = _randn((pool, BS, case["Hkv"], case["D"]), g, dt)
    vc = _randn((pool, BS, case["Hkv"], case["D"]), g, dt)
    return seqs, tables, members, query, kc, vc


def _cu(seqs):
    cu = [0]
    for q, _ in seqs:
        cu.append(cu[-1] + q)
    return cu


def _config(case):
    hf = dict(SHAPES[case["shape"]], num_hidden_layers=case["layers"])
    name = {"bf16": "bfloat16", "fp16": "float16", "fp32": "float32"}[case["dtype"]]
    return EngineConfig(
        model_config=ModelConfig(model="perf", dtype=name, load_format="dummy", hf_overrides=hf),
        cache_config=CacheConfig(block_size=BS),
        scheduler_config=SchedulerConfig(max_num_seqs=max(case["rows"], 1)), device="cuda",
        skip_tokenizer_init=True)


def _weights(case, seed):
    """Checkpoint tensors (q/k/v and gate/up apart, as checkpoints hold them):
    N(0, 0.02^2), norm weights around one."""
    s, g, dt = SHAPES[case["shape"]], _gen(seed + 1), DTYPES[case["dtype"]]
    hid, inter, d = s["hidden_size"], s["intermediate_size"], s["head_dim"]
    q, kv = s["num_attention_heads"] * d, s["num_key_value_heads"] * d
    w = {"model.embed_tokens.weight": _randn((s["vocab_size"], hid), g, dt, 0.02)}
    for i in range(case["layers"]):
        p = f"model.layers.{i}."
        for n, shape in (("self_attn.q_proj", (q, hid)), ("self_attn.k_proj", (kv, hid)),
                         ("self_attn.v_proj", (kv, hid)), ("self_attn.o_proj", (hid, q)),
                         ("mlp.gate_proj", (inter, hid)), ("mlp.up_proj", (inter, hid)),
                         ("mlp.down_proj", (hid, inter))):
            w[p + n + ".weight"] = _randn(shape, g, dt, 0.02)
        norms = [("input_layernorm", hid), ("post_attention_layernorm", hid)]
        if s["model_type"] == "qwen3":
            norms += [("self_attn.q_norm", d), ("self_attn.k_norm", d)]
        for n, size in norms:
            w[p + n + ".weight"] = 1.0 + _randn((size,), g, dt, 0.1)
    w["model.norm.weight"] = 1.0 + _randn((hid,), g, dt, 0.1)
    w["lm_head.weight"] = _randn((s["vocab_size"], hid), g, dt, 0.02)
    return w


def _model(config, weights):
    mc = config.model_config
    with torch.device("cuda"):
        model = BaseModelForCausalLM.get_model_cls(mc.model_type)(mc)
    model = model.to(dtype=mc.torch_dtype, device="cuda")
    model.load_weights(weights)
    return model.eval()


def _model_batch(case, seed):
    """Sequences [(query tokens, context)], decodes first, their tables, the
    token ids fed this step, and the cache [layers, 2, blocks, ...] before it."""
    lens = _decode_lens(case) if case["rows"] else []
    random.Random(seed).shuffle(lens)
    seqs = [(1, n) for n in lens]
    if case["kind"] == "step":
        chunks = [(n, n + o) for n, o in _chunk_lens(case)]
        random.Random(seed + 1).shuffle(chunks)
        seqs += chunks
    tables, pool = _tables([_blocks(c) for _, c in seqs], seed)
    s = SHAPES[case["shape"]]
    g = _gen(seed)
    ids = torch.randint(0, s["vocab_size"], (sum(q for q, _ in seqs),), generator=g, device="cuda")
    cache = _randn((case["layers"], 2, pool, BS, s["num_key_value_heads"], s["head_dim"]), g,
                   DTYPES[case["dtype"]])
    return seqs, tables, ids, cache


def prepare(case, seed):
    with torch.inference_mode():
        return dict(_PREPARE[case["kind"]](case, seed), kind=case["kind"])


def _prepare_attention(case, seed):
    seqs, tables, members, query, kc, vc = _attention_inputs(case, seed)
    st = dict(query=query, kc=kc, vc=vc, scale=case["D"] ** -0.5, kw={})
    st["bt"] = _padded(tables).cuda()
    st["ctx"] = torch.tensor([c for _, c in seqs], dtype=torch.int32).cuda()
    if case["kind"] == "prefill":
        st["kw"] = dict(cu_seqlens=torch.tensor(_cu(seqs), dtype=torch.int32).cuda(),
                        num_decodes=0, max_query_len=max(q for q, _ in seqs))
    elif members:
        st["kw"] = dict(prefix=ops.prefix_plan([(members, case["shared"])], len(seqs),
                                               case["H"] // case["Hkv"], torch.device("cuda")))
    return st


def _prepare_step(case, seed):
    seqs, tables, ids, cache = _model_batch(case, seed)
    model = _model(_config_resolved(case), _weights(case, seed))
    pos = torch.cat([torch.arange(c - q, c) for q, c in seqs])
    bt = _padded(tables)
    owner = torch.repeat_interleave(torch.arange(len(seqs)), torch.tensor([q for q, _ in seqs]))
    slots = bt[owner, pos // BS].to(torch.int64) * BS + pos % BS
    cu = _cu(seqs)
    bt, ctx = bt.cuda(), torch.tensor([c for _, c in seqs], dtype=torch.int32).cuda()
    meta = AttentionMetadata(block_tables=bt, context_lens=ctx,
                             cu_seqlens=torch.tensor(cu, dtype=torch.int32).cuda(),
                             num_decodes=case["rows"], max_query_len=max(q for q, _ in seqs))
    return dict(model=model, ids=ids, pos=pos.cuda(), slots=slots.cuda(), bt=bt, ctx=ctx,
                meta=meta, cache=cache, kv=[(c[0], c[1]) for c in cache], head=case["head"],
                last=torch.tensor([e - 1 for e in cu[1:]]).cuda())


def _config_resolved(case):
    config = _config(case)
    config.resolve()
    return config


def _prepare_graph(case, seed):
    seqs, tables, ids, cache = _model_batch(case, seed)
    config = _config_resolved(case)
    runner = ModelRunner(config)
    runner.model = _model(config, _weights(case, seed))
    runner.init_kv_cache(cache.shape[2])
    runner.kv_cache.storage.copy_(cache)
    blocks = BlockManager(BS, cache.shape[2], reserved_blocks=1)
    groups = []
    for i, ((_, ctx), table, tok) in enumerate(zip(seqs, tables, ids.tolist())):
        sg = SequenceGroup.create(f"r{i}", [1] * (ctx - 1), SamplingParams(temperature=0.0))
        seq = sg.seqs[0]
        seq.num_computed_tokens = ctx - 1
        seq.data.append_token(tok)
        # the tables of _tables, handed out by the allocator (from its end)
        blocks.gpu_allocator.free_list.extend(reversed(table))
        blocks.allocate(seq.seq_id, len(table))
        groups.append(sg)
    del cache
    runner.capture_decode_graphs()
    return dict(runner=runner, meta=runner.prepare_inputs(groups, blocks))


def _prepare_sample(case, seed):
    g = _gen(seed)
    rows, vocab = case["rows"], case["vocab"]
    logits = _randn((rows, vocab), g, DTYPES[case["dtype"]], 4.0)
    # a maximum half a unit above the rest, at a place of the row's own
    at = torch.randint(0, vocab, (rows, 1), generator=g, device="cuda")
    logits.scatter_(1, at, float("-inf"))
    logits.scatter_(1, at, logits.max(dim=1, keepdim=True).values + 0.5)
    temp = torch.zeros(rows, device="cuda")
    half = rows // 2
    temp[half:] = 0.5 + 0.5 * torch.rand(rows - half, generator=g, device="cuda")
    return dict(logits=logits, temp=temp, uniform=torch.rand(rows, generator=g, device="cuda"))


_PREPARE = {"decode": _prepare_attention, "prefill": _prepare_attention, "step": _prepare_step,
            "graph": _prepare_graph, "sample": _prepare_sample}


# -- one pass ------------------------------------------------------------------

def run(st):
    kind = st["kind"]
    if kind in ("decode", "prefill"):
        return ops.paged_attention(st["query"], st["kc"], st["vc"], st["bt"], st["ctx"],
                                   scale=st["scale"], **st["kw"])
    if kind == "sample":
        return Sampler.sample_batched(st["logits"], st["temp"], st["uniform"])
    if kind == "graph":
        runner = st["runner"]
        return {"logits": runner.execute_model(st["meta"]), "cache": runner.kv_cache.storage}
    with torch.inference_mode():
        if st["head"]:
            logits = st["model"](st["ids"], st["pos"], kv_caches=st["kv"],
                                 slot_mapping=st["slots"], block_tables=st["bt"],
                                 context_lens=st["ctx"], attn_metadata=st["meta"],
                                 logits_indices=st["last"])
            return {"logits": logits, "cache": st["cache"]}
        hidden, residual = st["model"].model(st["ids"], st["pos"], st["kv"], st["slots"],
                                             st["bt"], st["ctx"], True, st["meta"])
        return {"hidden": hidden, "residual": residual, "cache": st["cache"]}


# -- work ----------------------------------------------------------------------

def _attention_work(H, Hkv, D, es, decodes, chunks, shared=0, sharers=0):
    """Bytes and operations of attention over the given lengths: every key and
    value read once (a shared prefix once for all), q read, output written."""
    keys = sum(decodes) - max(sharers - 1, 0) * shared * BS + sum(n + o for n, o in chunks)
    rows = len(decodes) + sum(n for n, _ in chunks)
    pairs = sum(decodes) + sum(n * o + n * (n + 1) // 2 for n, o in chunks)
    blocks = sum(_blocks(c) for c in decodes) + sum(_blocks(n + o) for n, o in chunks)
    return (keys * Hkv * D * es * 2 + 2 * rows * H * D * es + 4 * blocks, 4 * H * D * pairs)


def work(case):
    kind, es = case["kind"], torch.empty(0, dtype=DTYPES[case["dtype"]]).element_size()
    if kind == "sample":
        n = case["rows"] * case["vocab"]
        return {"bytes": n * es + 16 * case["rows"], "flops": 4 * n}
    decodes = _decode_lens(case) if case.get("rows") else []
    chunks = _chunk_lens(case) if case.get("chunks") else []
    if kind in ("decode", "prefill"):
        b, f = _attention_work(case["H"], case["Hkv"], case["D"], es, decodes, chunks,
                               case.get("shared", 0), case.get("sharers", 0))
        return {"bytes": b, "flops": f}
    s = SHAPES[case["shape"]]
    H, Hkv, D = s["num_attention_heads"], s["num_key_value_heads"], s["head_dim"]
    hid, inter = s["hidden_size"], s["intermediate_size"]
    T = len(decodes) + sum(n for n, _ in chunks)
    ab, af = _attention_work(H, Hkv, D, es, decodes, chunks)
    ab -= 2 * T * H * D * es                     # q and the output stay inside the layer
    params = hid * D * (2 * H + 2 * Hkv) + 3 * hid * inter
    # a layer: its weights, the keys and values, the new rows of the cache
    nbytes = case["layers"] * (params * es + ab + 2 * T * Hkv * D * es)
    flops = case["layers"] * (2 * T * params + af)
    nbytes += T * (8 + hid * es)                 # token ids and their embeddings
    if kind == "graph" or case["head"]:
        seqs = len(decodes) + len(chunks)
        nbytes += (hid * s["vocab_size"] + seqs * s["vocab_size"]) * es
        flops += 2 * seqs * hid * s["vocab_size"]
    else:
        nbytes += 2 * T * hid * es               # hidden and residual
    return {"bytes": nbytes, "flops": flops}


# -- expected results ----------------------------------------------------------

def tolerance(case):
    kind, dt = case["kind"], case["dtype"]
    if kind == "sample":
        return "exact"
    if kind in ("decode", "prefill"):
        # the output rounded once; prompt chunks also round the weights
        # (2e-3 in bf16 and 2.5e-4 in fp16 against 64 bits)
        return {"bf16": {"rel": 8e-3, "max": 0.1}, "fp16": {"rel": 1e-3, "max": 0.0125}}[dt]
    # every layer rounds some ten intermediates to the model's type: logits
    # after four bf16 layers are 1.6e-2 off 64 bits, a layer's output 1e-2,
    # the fp32 model's logits 6e-7
    return {"bf16": {"rel": 3e-2, "max": 0.3}, "fp16": {"rel": 5e-3, "max": 0.05},
            "fp32": {"rel": 3e-6, "max": 3e-5}}[dt]


def _gather(cache, table, n):
    """The first n rows of a sequence in a paged cache [blocks, BS, Hkv, D],
    as fp64 [Hkv, n, D]."""
    idx = torch.tensor(table[:_blocks(n)], device="cuda")
    return cache[idx].reshape(-1, *cache.shape[2:])[:n].double().transpose(0, 1).contiguous()


def _attend(q, k, v, scale):
    """q [q, H, D] at the last q positions of k / v [Hkv, n, D], causal."""
    nq, H, D = q.shape
    hkv, n, _ = k.shape
    out = torch.empty_like(q)
    hide = (torch.arange(n, device="cuda")[None, :]
            > torch.arange(n - nq, n, device="cuda")[:, None])
    for h in range(H):
        kv = h // (H // hkv)
        s = (q[:, h] @ k[kv].t()) * scale
        out[:, h] = torch.softmax(s.masked_fill(hide, float("-inf")), dim=-1) @ v[kv]
    return out


def _norm(x, w, eps):
    return w * (x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps))


def _exact_model(case, seed):
    s = SHAPES[case["shape"]]
    seqs, tables, ids, cache = _model_batch(case, seed)
    w = {n: t.double() if t.dim() == 1 else t for n, t in _weights(case, seed).items()}
    H, Hkv, D, eps = (s["num_attention_heads"], s["num_key_value_heads"], s["head_dim"],
                      s["rms_norm_eps"])
    cu = _cu(seqs)
    T = cu[-1]
    pos = torch.cat([torch.arange(c - q, c) for q, c in seqs]).cuda().double()
    ang = pos[:, None] * (s["rope_theta"] ** (-torch.arange(0, D, 2, device="cuda").double() / D))
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]

    def linear(x, name):
        return x @ w[name + ".weight"].double().t()

    def rope(x):
        a, b = x.chunk(2, dim=-1)
        return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)

    res, out = w["model.embed_tokens.weight"][ids].double(), None
    for i in range(case["layers"]):
        p = f"model.layers.{i}."
        res = res if out is None else res + out
        x = _norm(res, w[p + "input_layernorm.weight"], eps)
        q = linear(x, p + "self_attn.q_proj").view(T, H, D)
        k = linear(x, p + "self_attn.k_proj").view(T, Hkv, D)
        v = linear(x, p + "self_attn.v_proj").view(T, Hkv, D)
        if s["model_type"] == "qwen3":
            q = _norm(q, w[p + "self_attn.q_norm.weight"], eps)
            k = _norm(k, w[p + "self_attn.k_norm.weight"], eps)
        q, k = rope(q), rope(k)
        att = torch.empty_like(q)
        for (nq, c), table, a in zip(seqs, tables, cu):
            kk, vv = _gather(cache[i, 0], table, c), _gather(cache[i, 1], table, c)
            kk[:, c - nq:] = k[a:a + nq].transpose(0, 1)
            vv[:, c - nq:] = v[a:a + nq].transpose(0, 1)
            att[a:a + nq] = _attend(q[a:a + nq], kk, vv, D ** -0.5)
        res = res + linear(att.reshape(T, H * D), p + "self_attn.o_proj")
        x = _norm(res, w[p + "post_attention_layernorm.weight"], eps)
        gate = linear(x, p + "mlp.gate_proj")
        out = linear(gate * torch.sigmoid(gate) * linear(x, p + "mlp.up_proj"), p + "mlp.down_proj")
    if case["kind"] == "step" and not case["head"]:
        return {"hidden": out, "residual": res, "cache": None}
    last = torch.tensor([e - 1 for e in cu[1:]], device="cuda")
    x = _norm((res + out)[last], w["model.norm.weight"], eps)
    return {"logits": linear(x, "lm_head"), "cache": None}


def exact(case, seed):
    if case["kind"] == "sample":     # token ids
        return None
    with torch.inference_mode():
        if case["kind"] in ("step", "graph"):
            return _exact_model(case, seed)
        seqs, tables, _, query, kc, vc = _attention_inputs(case, seed)
        out = torch.empty(query.shape, dtype=torch.float64, device="cuda")
        for (nq, c), table, a in zip(seqs, tables, _cu(seqs)):
            out[a:a + nq] = _attend(query[a:a + nq].double(), _gather(kc, table, c),
                                    _gather(vc, table, c), case["D"] ** -0.5)
        return out
