"""GPU parity of the four hot-path kernels against the CPU oracle.

Bars: packing, slot_mapping and KV scatter bit-exact; greedy argmax
bit-exact; temperature sampling bit-exact against oracle/sampler_ref.c at
the same uniforms; attention within 2e-2 max-abs and 1e-3 mean-abs of the
fp32 oracle on the same bf16 inputs (plus relative L2 <= 1e-2).
"""

from __future__ import annotations

import json
import math
import sys
import types
from pathlib import Path

import numpy as np
import pytest
import torch

from litevllm import ops, workloads
from oracle import attention as oatt
from oracle import packing as opack
from oracle import sampler as osamp
from oracle import scatter as oscat

pytestmark = pytest.mark.gpu

ATOL_MAX, ATOL_MEAN, REL_L2 = 2e-2, 1e-3, 1e-2


def _say(msg):
    print(f"[case] {msg}", flush=True)


def _check_attention(got: torch.Tensor, ref: torch.Tensor, what: str):
    got = got.float().cpu()
    err = (got - ref).abs()
    rel = (got - ref).norm() / ref.norm().clamp_min(1e-30)
    assert torch.isfinite(got).all(), f"{what}: non-finite output"
    assert err.max() <= ATOL_MAX, f"{what}: max-abs {err.max():.3e}"
    assert err.mean() <= ATOL_MEAN, f"{what}: mean-abs {err.mean():.3e}"
    assert rel <= REL_L2, f"{what}: rel-L2 {rel:.3e}"


# ---------------------------------------------------------------------------
# KV scatter
# ---------------------------------------------------------------------------

@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("strided", [False, True])
def test_kv_scatter_bit_exact(device, dtype, strided):
    _say(f"kv_scatter dtype={dtype} strided={strided}")
    g = torch.Generator().manual_seed(11)
    N, bs, Hkv, D, T = 64, 16, 8, 128, 300
    kc = torch.full((N, bs, Hkv, D), 3.5, dtype=dtype)
    vc = torch.full((N, bs, Hkv, D), -3.5, dtype=dtype)
    slots = torch.randperm(N * bs, generator=g)[:T].to(torch.int64)
    slots[::37] = -1
    if strided:
        qkv = torch.randn(T, (16 + 2 * Hkv) * D, generator=g).to(dtype)
        k = qkv[:, 16 * D:(16 + Hkv) * D].view(T, Hkv, D)
        v = qkv[:, (16 + Hkv) * D:].view(T, Hkv, D)
    else:
        k = torch.randn(T, Hkv, D, generator=g).to(dtype)
        v = torch.randn(T, Hkv, D, generator=g).to(dtype)
    kc_d, vc_d = kc.to(device), vc.to(device)
    if strided:
        qkv_d = qkv.to(device)
        k_d = qkv_d[:, 16 * D:(16 + Hkv) * D].view(T, Hkv, D)
        v_d = qkv_d[:, (16 + Hkv) * D:].view(T, Hkv, D)
    else:
        k_d, v_d = k.to(device), v.to(device)
    ops.kv_scatter(k_d, v_d, kc_d, vc_d, slots.to(device))
    torch.cuda.synchronize()
    kn, vn = kc.clone(), vc.clone()
    oscat.kv_scatter(k.contiguous().view(torch.int16).numpy() if dtype != torch.float32 else k.contiguous().numpy(),
                     v.contiguous().view(torch.int16).numpy() if dtype != torch.float32 else v.contiguous().numpy(),
                     kn.view(torch.int16).numpy() if dtype != torch.float32 else kn.numpy(),
                     vn.view(torch.int16).numpy() if dtype != torch.float32 else vn.numpy(),
                     slots.numpy())
    assert torch.equal(kc_d.cpu().view(torch.uint8), kn.view(torch.uint8))
    assert torch.equal(vc_d.cpu().view(torch.uint8), vn.view(torch.uint8))


def test_kv_scatter_config3_round_trip(device):
    _say("kv_scatter config3 round trip")
    step = workloads.mixed_step(seed=3)
    b = step.batch
    kc = torch.zeros_like(b.key_cache, device=device)
    vc = torch.zeros_like(b.value_cache, device=device)
    kc.fill_(7.0)
    vc.fill_(-7.0)
    slots = step.slot_mapping.to(device)
    ops.kv_scatter(step.key.to(device), step.value.to(device), kc, vc, slots)
    nb, bs = kc.shape[0], kc.shape[1]
    flat_k = kc.view(nb * bs, *kc.shape[2:])
    flat_v = vc.view(nb * bs, *vc.shape[2:])
    assert torch.equal(flat_k[slots].cpu(), step.key)
    assert torch.equal(flat_v[slots].cpu(), step.value)
    touched = torch.zeros(nb * bs, dtype=torch.bool, device=device)
    touched[slots] = True
    assert bool((flat_k[~touched] == 7.0).all()) and bool((flat_v[~touched] == -7.0).all())


# ---------------------------------------------------------------------------
# paged attention
# ---------------------------------------------------------------------------

def _run_attention(batch: workloads.PagedBatch, device, use_cu: bool):
    b = batch.to(device)
    return ops.paged_attention(b.query, b.key_cache, b.value_cache, b.block_tables,
                               b.context_lens, scale=b.scale,
                               cu_seqlens=b.cu_seqlens if use_cu else None,
                               num_decodes=b.num_decodes, max_query_len=b.max_query_len)


def _oracle(batch: workloads.PagedBatch):
    return oatt.mixed_attention(batch.query, batch.key_cache, batch.value_cache,
                                batch.block_tables, batch.cu_seqlens, batch.context_lens,
                                batch.scale)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("heads", [(16, 8, 128), (4, 2, 64), (8, 8, 128), (32, 4, 64),
                                   (16, 2, 128), (32, 8, 128), (16, 4, 64)])
def test_decode_small_shapes(device, dtype, heads):
    H, Hkv, D = heads
    _say(f"decode small dtype={dtype} H={H} Hkv={Hkv} D={D}")
    batch = workloads.paged_decode(seed=5, num_seqs=24, num_heads=H, num_kv_heads=Hkv,
                                   head_dim=D, ctx_lo=1, ctx_hi=700, dtype=dtype,
                                   scale_inputs=False, tail_fill=float("nan"),
                                   ctx_head=[1, 15, 16, 17, 256, 257, 512, 513])
    got = _run_attention(batch, device, use_cu=False)
    _check_attention(got, _oracle(batch), f"decode {dtype} {heads}")


@pytest.mark.parametrize("scaled", [True, False])
def test_decode_config2(device, scaled):
    _say(f"decode config2 scaled={scaled}")
    batch = workloads.paged_decode(seed=0, scale_inputs=scaled)
    got = _run_attention(batch, device, use_cu=False)
    _check_attention(got, _oracle(batch), f"config2 scaled={scaled}")


def test_decode_workspace_reuse_and_counter_reset(device):
    """Back-to-back calls of different shapes share one workspace; each is
    correct (stale partials of an earlier call are never read)."""
    _say("decode workspace reuse")
    for seed, n, lo, hi in ((21, 300, 1, 3000), (22, 7, 2000, 9000), (23, 64, 1, 40)):
        batch = workloads.paged_decode(seed=seed, num_seqs=n, ctx_lo=lo, ctx_hi=hi,
                                       scale_inputs=False)
        got = _run_attention(batch, device, use_cu=False)
        _check_attention(got, _oracle(batch), f"reuse seed={seed}")


def test_decode_long_contexts(device):
    """Rows of 16k-32k tokens among short ones: each workgroup walks many
    64-block groups, and a long row spreads over dozens of workgroup ranges,
    so the reduce takes its general (many-piece) merge path."""
    _say("decode long contexts")
    batch = workloads.paged_decode(seed=17, num_seqs=40, ctx_lo=1, ctx_hi=600,
                                   scale_inputs=False, tail_fill=float("nan"),
                                   ctx_head=[32768, 20000, 16385, 31999, 1])
    got = _run_attention(batch, device, use_cu=False)
    _check_attention(got, _oracle(batch), "long contexts")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("heads", [(16, 8, 128), (6, 3, 128), (20, 5, 64), (64, 8, 128),
                                   (8, 1, 64), (2, 2, 64)])
@pytest.mark.parametrize("kind", ["plain", "peaky", "small", "many"])
def test_decode_matrix_cores_one_rounding(device, dtype, heads, kind):
    """The matrix-core decode kernel rounds nothing to 16 bits but the output
    (K Q^T products are exact in fp32, the softmax weights enter V^T P^T as
    three parts: exact in bf16, within 2^-35 of the row's largest weight in
    fp16): each output is within half a unit in the last place
    of the fp64 result plus 2e-6 of the largest |value| for fp32 sums.  Block
    and 64-block edges, NaN past the context, softmaxes dominated by a few
    keys, values below the smallest normal fp16, and (rows past what its LDS
    holds) the vector kernel that takes over."""
    H, Hkv, D = heads
    _say(f"decode matrix cores {dtype} {heads} {kind}")
    if kind == "many":
        batch = workloads.paged_decode(seed=2, num_seqs=7300, num_heads=H, num_kv_heads=Hkv,
                                       head_dim=D, ctx_lo=1, ctx_hi=20, dtype=dtype,
                                       scale_inputs=False, tail_fill=float("nan"))
    else:
        batch = workloads.paged_decode(seed=3, num_seqs=19, num_heads=H, num_kv_heads=Hkv,
                                       head_dim=D, ctx_lo=1, ctx_hi=900, dtype=dtype,
                                       scale_inputs=False, tail_fill=float("nan"),
                                       ctx_head=[1, 15, 16, 17, 31, 33, 1023, 1024, 1025, 2500])
        if kind == "peaky":
            batch.query *= 8
        if kind == "small":
            batch.value_cache *= 2.0 ** -18
    got = _run_attention(batch, device, use_cu=False).double().cpu()
    G, ulp = H // Hkv, 2.0 ** (-9 if dtype == torch.bfloat16 else -12)
    tiny = 2.0 ** (-134 if dtype == torch.bfloat16 else -25)   # half the smallest step
    for r in range(0, batch.query.shape[0], 37 if kind == "many" else 1):
        n = int(batch.context_lens[r])
        blk = batch.block_tables[r, :-(-n // 16)].long()
        k = batch.key_cache[blk].reshape(-1, Hkv, D)[:n].double()
        v = batch.value_cache[blk].reshape(-1, Hkv, D)[:n].double()
        for h in range(H):
            p = torch.softmax(k[:, h // G] @ batch.query[r, h].double() * batch.scale, 0)
            ref = p @ v[:, h // G]
            bound = ulp * 2 * ref.abs().clamp_min(2.0 ** -14 if dtype == torch.float16 else 0)
            bound = torch.maximum(bound, torch.full_like(ref, tiny)) + 2e-6 * v.abs().max()
            err = (got[r, h] - ref).abs()
            assert (err <= bound).all(), (r, h, n, float((err / bound).max()))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("heads", [(16, 8, 128), (8, 8, 64), (16, 4, 64), (16, 2, 128)])
@pytest.mark.parametrize("kind", ["few rows", "many rows", "prefix", "chunks"])
def test_infinite_values(device, dtype, heads, kind):
    """An infinite V element the row can see makes its own dim of the row
    infinite (NaN where both signs meet) and touches no other dim: decode rows
    of one and of many pieces, rows with a shared prefix, and chunk rows in one
    and in several key ranges, each with a weight far below the row's largest
    among the infinite tokens (fp16 decode: under 2^-40)."""
    H, Hkv, D = heads
    G = H // Hkv
    _say(f"infinite values {dtype} {heads} {kind}")
    if kind == "chunks":
        batch = workloads.mixed_step(seed=5, num_decodes=0, num_chunks=1, chunk_len=20,
                                     off_lo=1500, off_hi=1500, num_heads=H, num_kv_heads=Hkv,
                                     head_dim=D, num_cache_slots=16 * 400, dtype=dtype).batch
    else:
        batch = workloads.paged_decode(seed=6, num_seqs=300 if kind == "many rows" else 5,
                                       num_heads=H, num_kv_heads=Hkv, head_dim=D, ctx_lo=90,
                                       ctx_hi=400, dtype=dtype, scale_inputs=False,
                                       ctx_head=[3000, 100, 97])
    plan = None
    if kind == "prefix":
        batch.block_tables[1:3, :4] = batch.block_tables[0, :4]
        plan = ops.prefix_plan([([0, 1, 2], 4)], 5, G, device) if dtype != torch.float32 else None

    def call():
        b = batch.to(device)
        cu = dict(cu_seqlens=b.cu_seqlens, max_query_len=b.max_query_len) if kind == "chunks" else {}
        return ops.paged_attention(b.query, b.key_cache, b.value_cache, b.block_tables,
                                   b.context_lens, scale=b.scale, num_decodes=b.num_decodes,
                                   prefix=plan, **cu).float().cpu()
    want = call()
    assert torch.isfinite(want).all()
    bt, kc, vc = batch.block_tables, batch.key_cache, batch.value_cache
    inf = float("inf")
    for r in range(bt.shape[0]):
        if kind == "prefix" and r == 0:
            continue                       # (its first blocks are the others' too)
        n = int(batch.context_lens[r]) - (19 if kind == "chunks" else 0)
        b0, b1, b2 = (int(bt[r, t // 16]) for t in (70, n - 1, 81))
        vc[b0, 70 % 16, :, 3] = inf
        vc[b1, (n - 1) % 16, :, 5] = -inf
        vc[b0, 70 % 16, 0, 7] = -inf
        vc[b1, (n - 1) % 16, 0, 7] = inf
        if kind not in ("chunks", "prefix"):
            # a token of little weight: its key against the row's first query head
            q = batch.query[r].float().view(Hkv, G, D).sum(1)
            kc[b2, 81 % 16] = (-q * 40 / q.square().sum(-1, keepdim=True).sqrt()).to(dtype)
            vc[b2, 81 % 16, :, 9] = inf
    want = want if kind in ("chunks", "prefix") else None
    got = call()
    if want is None:                       # the same keys with finite values
        vc.nan_to_num_(0.0, 0.0, 0.0)
        want = call()
    rows = slice(1, None) if kind == "prefix" else slice(None)
    got, want = got[rows], want[rows]
    assert (got[:, :, 3] == inf).all() and (got[:, :, 5] == -inf).all()
    assert got[:, :G, 7].isnan().all()
    special = torch.zeros(D, dtype=torch.bool)
    special[[3, 5]] = True
    if kind not in ("chunks", "prefix"):
        assert (got[:, :, 9] == inf).all()
        special[9] = True
    special = special.expand(H, D).clone()
    special[:G, 7] = True
    # other dims: the same weights and values, so one rounding of the output apart
    a, b = got[:, ~special], want[:, ~special]
    assert torch.isfinite(a).all()
    assert (a - b).norm() <= 2.0 ** -8 * b.norm()


@pytest.mark.parametrize("chunk,off", [(70, 0), (20, 1500)])
def test_chunk_scores_of_any_finite_size(device, chunk, off):
    """Split tiles tell a masked key by its position, not by its score: with
    every score -2^99 (and a scale that is 1/8 in log2 units, so its products
    are exact) a row's output is the mean of the values it sees."""
    _say(f"chunk scores of -2^99, {chunk} tokens at {off}")
    batch = workloads.mixed_step(seed=5, num_decodes=0, num_chunks=1, chunk_len=chunk, off_lo=off,
                                 off_hi=off, num_cache_slots=16 * 400).batch
    batch.query.fill_(2.0 ** 49)
    batch.key_cache.fill_(-2.0 ** 43)
    log2e = np.float32(1.4426950408889634)
    scale = np.float32(0.125) / log2e
    assert scale * log2e == np.float32(0.125)
    b = batch.to(device)
    got = ops.paged_attention(b.query, b.key_cache, b.value_cache, b.block_tables, b.context_lens,
                              scale=float(scale), cu_seqlens=b.cu_seqlens, num_decodes=0,
                              max_query_len=chunk).float().cpu()
    v = oatt.gather_sequence(batch.value_cache, batch.block_tables[0], chunk + off).float()
    mean = v.cumsum(0)[off:] / torch.arange(off + 1, off + chunk + 1)[:, None, None]
    want = mean.repeat_interleave(2, 1)
    assert (got - want).norm() <= 2.0 ** -8 * want.norm()


@torch.inference_mode()
def test_chunks_under_capture_use_no_pooled_scratch(device):
    """A captured chunk call keeps its keys in one range (the per-stream
    scratch may be replaced after the capture); replays, with eager split
    calls between them, equal the eager unsplit call."""
    _say("chunk call under capture")
    step = workloads.mixed_step(seed=3, num_decodes=0, num_chunks=1, chunk_len=33, off_lo=1500,
                                off_hi=1500, num_cache_slots=16 * 300).batch.to(device)

    def call(**kw):
        return ops.paged_attention(step.query, step.key_cache, step.value_cache,
                                   step.block_tables, step.context_lens, scale=step.scale,
                                   cu_seqlens=step.cu_seqlens, num_decodes=0, max_query_len=33,
                                   **kw)
    want = call(workspace=torch.empty(0, dtype=torch.uint8, device=device))
    split = call()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    for _ in range(3):
        out.zero_()
        ops._workspaces.clear()
        graph.replay()
        again = call()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(again, split)
    assert (split.float() - want.float()).norm() <= 2.0 ** -8 * want.float().norm()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("heads", [(16, 8, 128), (4, 2, 64), (16, 2, 128), (8, 8, 64)])
@pytest.mark.parametrize("lens", [[(1, 0), (2, 700)], [(31, 33), (32, 0), (33, 31)],
                                  [(63, 1), (64, 64), (65, 0), (129, 900)], [(5, 4200)],
                                  [(64, 960)], [(65, 1100), (3, 2300), (1, 0)], "full"])
def test_chunks_of_few_workgroups(device, dtype, heads, lens):
    """Chunks whose grid leaves the chip idle run on split key tiles (two
    wavefronts share 32 rows, 32 keys of each tile apiece), the emptiest with
    their keys in several ranges where scratch allows, fuller grids on whole
    tiles: lengths around a tile, rows with all keys in the first half of
    a tile, more than 64 tiles, NaN past the context.  Weights and outputs
    are rounded to 16 bits once each: 1.5 units in the last place of the
    largest |value| a row can see, and 2^-8 (2^-11) relative L2."""
    H, Hkv, D = heads
    if lens == "full":       # as many 128-row workgroups as take the whole tiles
        n = 400 // Hkv
        lens = [(17 + i % 40, (i * 37) % 90) for i in range(n)]
    _say(f"chunks {dtype} {heads} {lens[:4]}")
    g = torch.Generator().manual_seed(len(lens))
    nblk = [-(-(q + o) // 16) for q, o in lens]
    pool = sum(nblk) + 1
    perm = (torch.randperm(pool - 1, generator=g) + 1).to(torch.int32)
    bt, at = torch.zeros(len(lens), max(nblk), dtype=torch.int32), 0
    kc, vc = (torch.randn(pool, 16, Hkv, D, generator=g).to(dtype) for _ in range(2))
    for i, (n, (q, o)) in enumerate(zip(nblk, lens)):
        bt[i, :n] = perm[at:at + n]
        at += n
        if (q + o) % 16:
            kc[bt[i, n - 1], (q + o) % 16:] = float("nan")
            vc[bt[i, n - 1], (q + o) % 16:] = float("nan")
    cu = torch.tensor([0] + [q for q, _ in lens]).cumsum(0).to(torch.int32)
    ctx = torch.tensor([q + o for q, o in lens], dtype=torch.int32)
    query = torch.randn(int(cu[-1]), H, D, generator=g).to(dtype)
    scale = D ** -0.5
    got = ops.paged_attention(*(t.to(device) for t in (query, kc, vc, bt, ctx)), scale=scale,
                              cu_seqlens=cu.to(device), num_decodes=0,
                              max_query_len=max(q for q, _ in lens)).float().cpu()
    ref = oatt.mixed_attention(query, kc, vc, bt, cu, ctx, scale)
    ulp = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    # no scratch beyond what the call must have: keys in one range
    whole = ops.paged_attention(*(t.to(device) for t in (query, kc, vc, bt, ctx)), scale=scale,
                                cu_seqlens=cu.to(device), num_decodes=0,
                                max_query_len=max(q for q, _ in lens),
                                workspace=torch.empty(0, dtype=torch.uint8, device=device))
    assert (whole.float().cpu() - ref).norm() <= ulp * ref.norm()
    assert torch.isfinite(got).all()
    assert (got - ref).norm() <= ulp * ref.norm()
    assert (got - ref).abs().max() <= 1.5 * ulp * float(vc.nan_to_num(0).abs().max())


@pytest.mark.parametrize("path", ["native", "python"])
@torch.inference_mode()
def test_mixed_batch_under_capture_does_not_split(device, path, monkeypatch):
    """A captured mixed batch keeps its chunk's keys in one range whatever the
    per-stream scratch has grown to, as a call with a workspace of
    lv_paged_attention_workspace_size bytes does; with a larger one, and in
    eager calls, it splits."""
    _say(f"mixed batch under capture, {path}")
    if path == "python":
        monkeypatch.setattr(ops, "_native_module",
                            types.SimpleNamespace(paged_attention=lambda *a: None))
    step = workloads.mixed_step(seed=3, num_decodes=3, dec_lo=100, dec_hi=900, num_chunks=1,
                                chunk_len=20, off_lo=3000, off_hi=3000,
                                num_cache_slots=16 * 600).batch.to(device)
    geom = (4, 3, 23, 16, 128, 16, step.block_tables.shape[1], 20, step.query.dtype)
    plain = ops.paged_attention_workspace_size(*geom)

    def call(nbytes=None):
        ws = None if nbytes is None else torch.empty(nbytes, dtype=torch.uint8, device=device)
        return ops.paged_attention(step.query, step.key_cache, step.value_cache,
                                   step.block_tables, step.context_lens, scale=step.scale,
                                   cu_seqlens=step.cu_seqlens, num_decodes=3, max_query_len=20,
                                   workspace=ws)
    want, split = call(plain), call(plain + (1 << 24))
    assert not torch.equal(want, split)             # (another rounding of the weights)
    assert torch.equal(call(), split)
    ops._workspace(device, 1 << 26)                 # a pool grown by larger calls
    assert torch.equal(call(), split)
    graph = torch.cuda.CUDAGraph()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        pool = ops._workspace(device, 1 << 26)
    with torch.cuda.graph(graph, stream=stream):
        out = call()
    for _ in range(3):
        out.zero_()
        graph.replay()
        again = call()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(again, split)
    del pool


@pytest.mark.parametrize("heads,chunk,off", [
    ((16, 8, 128), 2048, 0), ((16, 8, 128), 2049, 0), ((16, 8, 128), 2049, 600),
    ((16, 8, 128), 3073, 0), ((8, 1, 128), 512, 0), ((8, 1, 128), 513, 0), ((4, 2, 64), 3000, 0)])
def test_chunks_around_the_line_of_split_tiles(device, heads, chunk, off):
    """One prompt just inside and past the sizes at which its workgroups stop
    running all at once (split tiles, from there on whole tiles unless the
    prompt is long and near its start), and past the last of them.  Weights
    and outputs are rounded to bf16 once each: 2^-8 relative L2."""
    H, Hkv, D = heads
    _say(f"chunks around the line {heads} {chunk} at {off}")
    batch = workloads.mixed_step(seed=chunk, num_decodes=0, num_chunks=1, chunk_len=chunk,
                                 off_lo=off, off_hi=off, num_heads=H, num_kv_heads=Hkv,
                                 head_dim=D, num_cache_slots=16 * 400).batch
    got = _run_attention(batch, device, use_cu=True).float().cpu()
    ref = _oracle(batch)
    assert torch.isfinite(got).all()
    assert (got - ref).norm() <= 2.0 ** -8 * ref.norm()


@pytest.mark.parametrize("rows,heads", [(1, (16, 8, 128)), (3, (16, 2, 128)), (7, (8, 8, 64)),
                                        (128, (16, 8, 128)), (129, (16, 8, 128))])
def test_decode_few_rows_of_many_pieces(device, rows, heads):
    """Rows cut into up to one piece per workgroup: the reduce kernel that
    takes a workgroup per (row, head) up to half as many rows as workgroups,
    and the other one just past that; empty, one-block and two-block rows
    among the long ones.  fp16 outputs round at 2^-11, so 3e-3 of the largest
    value and 1e-3 relative L2 bound one rounding plus fp32 merges."""
    H, Hkv, D = heads
    _say(f"decode few rows rows={rows} {heads}")
    batch = workloads.paged_decode(seed=rows, num_seqs=rows, num_heads=H, num_kv_heads=Hkv,
                                   head_dim=D, ctx_lo=1, ctx_hi=2000, dtype=torch.float16,
                                   scale_inputs=False, tail_fill=float("nan"),
                                   ctx_head=[5000, 17, 2050][:rows])
    got = _run_attention(batch, device, use_cu=False).float().cpu()
    ref = _oracle(batch)
    assert (got - ref).abs().max() <= 3e-3 * ref.abs().max()
    assert (got - ref).norm() <= 1e-3 * ref.norm()
    if rows > 3:     # a row without tokens is zero
        batch.context_lens[2] = 0
        got = _run_attention(batch, device, use_cu=False).float().cpu()
        assert (got[2] == 0).all() and torch.isfinite(got).all()


@pytest.mark.parametrize("heads", [(16, 8, 128), (8, 1, 64), (32, 4, 128)])
def test_decode_lockstep_interval_bit_identical(device, heads, monkeypatch):
    """The persistent kernel's wavefront lockstep barrier (LV_ATTN_SYNC,
    default every 4 blocks) moves no data: outputs are bit-identical with it
    off, at the default and at every 2 blocks; each run must also finish
    (every wavefront of a workgroup reaches the same barriers)."""
    H, Hkv, D = heads
    _say(f"decode lockstep interval H={H} Hkv={Hkv} D={D}")
    batch = workloads.paged_decode(seed=31, num_seqs=200, num_heads=H, num_kv_heads=Hkv,
                                   head_dim=D, ctx_lo=1, ctx_hi=1500, scale_inputs=False,
                                   ctx_head=[1, 2, 17, 33, 1024])
    outs = {}
    for sync in ("default", "0", "2"):
        if sync == "default":
            monkeypatch.delenv("LV_ATTN_SYNC", raising=False)
        else:
            monkeypatch.setenv("LV_ATTN_SYNC", sync)
        outs[sync] = _run_attention(batch, device, use_cu=False).cpu()
    monkeypatch.delenv("LV_ATTN_SYNC", raising=False)
    _check_attention(outs["default"], _oracle(batch), f"lockstep {heads}")
    assert torch.equal(outs["default"].view(torch.int16), outs["0"].view(torch.int16))
    assert torch.equal(outs["default"].view(torch.int16), outs["2"].view(torch.int16))


@pytest.mark.parametrize("knobs", [
    {"LV_ATTN_NBUF": "4"}, {"LV_ATTN_NT": "0"}, {"LV_ATTN_PERSIST_WGS": "97"},
    {"LV_ATTN_PERSIST_WGS": "1"}, {"LV_ATTN_PERSIST_WGS": "1024"},
    {"LV_ATTN_DECODE_KERNEL": "rows"},
    {"LV_ATTN_DECODE_KERNEL": "rows", "LV_ATTN_PART_TOKENS": "128"},
    {"LV_ATTN_CHUNK_KERNEL": "rows"}])
def test_attention_tuning_knobs(device, knobs, monkeypatch):
    """The per-call tuning knobs of lv_paged_attention (register buffers,
    load type, persistent grid -- one workgroup: every row whole; 1024: the
    40 rows cut into ranges of a few blocks, most rows in three or more
    pieces -- the fallback row kernels and their partition size) keep a
    mixed step within the attention bar; the two that change only prefetch
    depth or load type, of the vector kernel (run in fp32, where it takes the
    decode rows), leave it bit-identical."""
    _say(f"attention knobs {knobs}")
    vector = set(knobs) <= {"LV_ATTN_NBUF", "LV_ATTN_NT"}
    step = workloads.mixed_step(seed=13, num_decodes=40, dec_lo=1, dec_hi=2500, num_chunks=3,
                                chunk_len=90, off_hi=700, num_cache_slots=16 * 3000,
                                dtype=torch.float32 if vector else torch.bfloat16)
    base = _run_attention(step.batch, device, use_cu=True).cpu()
    for k, v in knobs.items():
        monkeypatch.setenv(k, v)
    got = _run_attention(step.batch, device, use_cu=True).cpu()
    for k in knobs:
        monkeypatch.delenv(k)
    _check_attention(got, _oracle(step.batch), f"knobs {knobs}")
    if vector:
        assert torch.equal(got.view(torch.int32), base.view(torch.int32))


def test_decode_matches_reference_restatement(device):
    """The literal _decode_fast restatement (gather over max_s, mask, einsum)."""
    _say("decode vs literal _decode_fast restatement")
    batch = workloads.paged_decode(seed=9, num_seqs=12, ctx_lo=1, ctx_hi=300, scale_inputs=False)
    got = _run_attention(batch, device, use_cu=False)
    ref = oatt.decode_attention(batch.query.float(), batch.key_cache.float(),
                                batch.value_cache.float(), batch.block_tables,
                                batch.context_lens, batch.scale)
    _check_attention(got, ref, "literal restatement")


@pytest.mark.parametrize("seed", [0, 1])
def test_mixed_step_small(device, seed):
    _say(f"mixed step small seed={seed}")
    step = workloads.mixed_step(seed=seed, num_decodes=12, dec_lo=1, dec_hi=600, num_chunks=4,
                                chunk_len=67, off_hi=300, num_cache_slots=16 * 400)
    got = _run_attention(step.batch, device, use_cu=True)
    _check_attention(got, _oracle(step.batch), f"mixed small seed={seed}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("heads", [(16, 8, 128), (4, 2, 64), (8, 8, 128), (32, 4, 64),
                                   (16, 2, 128), (32, 8, 128), (16, 4, 64)])
def test_chunks_all_shapes(device, dtype, heads):
    """Prefill chunks at unaligned offsets (MFMA path for bf16/fp16, per-row
    path for fp32), mixed with decodes, against the fp32 oracle."""
    H, Hkv, D = heads
    _say(f"chunks dtype={dtype} H={H} Hkv={Hkv} D={D}")
    step = workloads.mixed_step(seed=7, num_decodes=5, dec_lo=1, dec_hi=300, num_chunks=5,
                                chunk_len=97, off_lo=0, off_hi=400, num_heads=H,
                                num_kv_heads=Hkv, head_dim=D, num_cache_slots=16 * 300,
                                dtype=dtype)
    got = _run_attention(step.batch, device, use_cu=True)
    _check_attention(got, _oracle(step.batch), f"chunks {dtype} {heads}")


def test_chunk_lengths_and_offsets(device):
    """Chunk lengths 1..70 (ragged last query tile), offsets that are and
    are not block-aligned, a chunk ending exactly on a block edge."""
    _say("chunk lengths / offsets")
    g = torch.Generator().manual_seed(3)
    for chunk_len, off in ((1, 0), (2, 15), (31, 16), (32, 17), (33, 0), (64, 5), (70, 64), (16, 48)):
        step = workloads.mixed_step(seed=chunk_len * 100 + off, num_decodes=0, num_chunks=2,
                                    chunk_len=chunk_len, off_lo=off, off_hi=off,
                                    num_cache_slots=16 * 64)
        got = _run_attention(step.batch, device, use_cu=True)
        _check_attention(got, _oracle(step.batch), f"chunk len={chunk_len} off={off}")


def test_chunks_beyond_64_tiles(device):
    """Chunk rows whose keys run past 64 tiles of 64 keys (contexts beyond
    4096 tokens): the block ids each wavefront prefetches 64 tiles at a time
    are refilled mid-row.  One pair of chunks straddles the 4096-key edge,
    the other runs to ~12k keys (two refills)."""
    for seed, off_lo, off_hi, L in ((41, 3990, 3990, 130), (42, 8000, 12000, 96)):
        _say(f"chunks beyond 64 tiles off={off_lo}..{off_hi} len={L}")
        step = workloads.mixed_step(seed=seed, num_decodes=4, dec_lo=1, dec_hi=6000,
                                    num_chunks=2, chunk_len=L, off_lo=off_lo, off_hi=off_hi,
                                    num_cache_slots=16 * 4096)
        assert int(step.batch.context_lens.max()) > 64 * 64
        got = _run_attention(step.batch, device, use_cu=True)
        _check_attention(got, _oracle(step.batch), f"long chunks off={off_lo}")


def test_mixed_config3_full(device):
    """The full config-3 step: 192 decodes + 15 chunks of 512 at offsets up
    to 3072, 200k-slot cache, N(0,1) values."""
    _say("mixed config3 full")
    step = workloads.mixed_step(seed=0)
    got = _run_attention(step.batch, device, use_cu=True)
    _check_attention(got, _oracle(step.batch), "config3")


def test_prefill_only_offset_zero(device):
    _say("prefill only, offset 0")
    step = workloads.mixed_step(seed=4, num_decodes=0, num_chunks=3, chunk_len=100, off_lo=0,
                                off_hi=0, num_cache_slots=16 * 64)
    got = _run_attention(step.batch, device, use_cu=True)
    _check_attention(got, _oracle(step.batch), "prefill offset 0")


# ---------------------------------------------------------------------------
# sampler
# ---------------------------------------------------------------------------

def test_sampler_config4(device):
    _say("sampler config4")
    sb = workloads.sampler_batch(seed=0)
    got = ops.sample(sb.logits.to(device), sb.temperature.to(device), sb.uniform.to(device)).cpu()
    x = sb.logits.float().numpy()
    half = sb.logits.shape[0] // 2
    # greedy rows: the planted maximum, bit-exact with argmax
    assert torch.equal(got[:half], sb.planted[:half])
    assert np.array_equal(got[:half].numpy(), osamp.greedy(x[:half]))
    # temperature rows: bit-exact with the C restatement at the same uniforms
    ref = osamp.sample(x[half:], sb.temperature[half:].numpy(), sb.uniform[half:].numpy())
    assert np.array_equal(got[half:].numpy(), ref)


_SAMPLER_CHILD = r"""
import sys, numpy as np, torch
sys.path[:0] = sys.argv[1:3]
from litevllm import ops, workloads
sb = workloads.sampler_batch(seed=0)
d = torch.device("cuda:0")
ids = ops.sample(sb.logits.to(d), sb.temperature.to(d), sb.uniform.to(d)).cpu().numpy()
np.save(sys.argv[3], ids)
"""


@pytest.mark.parametrize("per_cu", ["1", "3", "32"])
def test_sampler_grid_knob_bit_identical(device, per_cu, tmp_path):
    """LV_SAMPLER_WGS_PER_CU (workgroups of the items kernel per CU, read
    once per process) only changes how segments are spread over
    wavefronts: config 4's ids are bit-identical to this process's default
    grid.  One child process per setting (the value is cached at first
    use)."""
    import os
    import subprocess
    import sys
    _say(f"sampler LV_SAMPLER_WGS_PER_CU={per_cu} (child process)")
    sb = workloads.sampler_batch(seed=0)
    want = ops.sample(sb.logits.to(device), sb.temperature.to(device),
                      sb.uniform.to(device)).cpu().numpy()
    root = Path(__file__).resolve().parent.parent
    out = tmp_path / "ids.npy"
    env = dict(os.environ, LV_SAMPLER_WGS_PER_CU=per_cu)
    subprocess.run([sys.executable, "-c", _SAMPLER_CHILD, str(root), str(root / "lite-vllm_amd"),
                    str(out)], env=env, check=True, timeout=240)
    assert np.array_equal(np.load(out), want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("V", [1, 7, 511, 512, 513, 32000, 151936])
def test_sampler_shapes(device, dtype, V):
    _say(f"sampler dtype={dtype} V={V}")
    g = torch.Generator().manual_seed(V)
    B = 12
    x = (torch.randn(B, V + 5, generator=g) * 3).to(dtype)[:, :V]   # row stride V + 5
    if V > 4:
        x[0, 1] = x[0, 3] = x[0].float().max() + 1   # tie: first index wins
        x[1, : V // 2] = float("-inf")
    temp = torch.tensor([0.0] * 4 + [0.6, 1.0, 1.7, 0.05, 1e-4, 2.0, 1.0, 1.0], dtype=torch.float32)
    uni = torch.rand(B, generator=g)
    uni[-2] = 0.0
    uni[-1] = float(np.nextafter(np.float32(1), np.float32(0)))
    xd = torch.empty(B, V + 5, dtype=dtype, device=device)[:, :V]
    xd.copy_(x)
    got = ops.sample(xd, temp.to(device), uni.to(device)).cpu().numpy()
    ref = osamp.sample(x.float().numpy(), temp.numpy(), uni.numpy())
    assert np.array_equal(got, ref)


# ---------------------------------------------------------------------------
# packing
# ---------------------------------------------------------------------------

KAT = json.loads((Path(__file__).parent / "golden" / "packing_kat.json").read_text())


def _pack_on_gpu(device, descs, blocks, toks, bs, max_blocks, dev_toks=None):
    T = int(np.asarray(descs)[:, 1].sum())
    out = ops.pack_inputs(torch.as_tensor(descs, dtype=torch.int32).to(device),
                          torch.as_tensor(blocks, dtype=torch.int32).to(device),
                          torch.as_tensor(toks, dtype=torch.int64).to(device), T, bs, max_blocks,
                          device_tokens=None if dev_toks is None else
                          torch.as_tensor(dev_toks, dtype=torch.int64).to(device))
    return {k: v.cpu().numpy() for k, v in out.items()}


@pytest.mark.parametrize("case", KAT["cases"], ids=lambda c: c["name"])
def test_pack_kat(device, case):
    _say(f"pack kat {case['name']}")
    recs = [opack.SeqRecord(s["prompt"], s["output"], s["num_computed"], s["blocks"])
            for s in case["seqs"]]
    descs, blocks, toks = opack.descriptors_from_records(recs)
    got = _pack_on_gpu(device, descs, blocks, toks, KAT["block_size"], case["packed"]["max_blocks"])
    for k in ("input_ids", "positions", "slot_mapping"):
        assert got[k].tolist() == case["reference"][k], k
    for k in ("cu_seqlens", "seq_start", "context_lens", "block_tables"):
        assert got[k].tolist() == case["packed"][k], k


@pytest.mark.parametrize("seed", range(4))
def test_pack_random(device, seed):
    _say(f"pack random seed={seed}")
    rng = np.random.default_rng(seed)
    B = int(rng.integers(1, 300))
    bs = 16
    descs, blocks, toks = [], [], []
    dev_toks = rng.integers(0, 151936, 50)
    for _ in range(B):
        if rng.random() < 0.6:
            n, q = int(rng.integers(0, 4000)), 1
        else:
            n, q = int(rng.integers(0, 3000)), int(rng.integers(1, 600))
        nb = (n + q + bs - 1) // bs - int(rng.random() < 0.1)
        tidx = int(rng.integers(0, 50)) if (q == 1 and rng.random() < 0.5) else -1
        descs.append([n, q, max(nb, 0), len(blocks), len(toks), tidx])
        blocks.extend(rng.integers(0, 12500, max(nb, 0)).tolist())
        toks.extend(rng.integers(0, 151936, q).tolist())
    descs = np.array(descs, dtype=np.int32)
    blocks = np.array(blocks, dtype=np.int32)
    toks = np.array(toks, dtype=np.int64)
    mb = int(descs[:, 2].max()) if B else 0
    got = _pack_on_gpu(device, descs, blocks, toks, bs, mb, dev_toks)
    ref = opack.expand_descriptors(descs, blocks, toks, bs, mb, device_tokens=dev_toks)
    for k in ref:
        assert np.array_equal(got[k], ref[k]), k


sys.path.insert(0, str(Path(__file__).parent / "golden"))
import packing_fixture  # noqa: E402


def test_pack_reference_fixtures(device):
    """Every schedule whose packed arrays the reference's own
    ModelRunner.prepare_inputs wrote (tests/golden/reference_packing.npz:
    40 decode-only and 40 prefill-only batches, block tables from its
    BlockManager, block sizes 8/16/32), replayed through lv_pack_inputs:
    bit-exact."""
    cases = packing_fixture.load_cases()
    _say(f"pack: {len(cases)} reference prepare_inputs fixtures")
    for case in cases:
        descs, blocks, toks = opack.descriptors_from_records(case["seqs"])
        mb = max(len(s.block_ids) for s in case["seqs"])
        got = _pack_on_gpu(device, descs, blocks, toks, case["block_size"], mb)
        for k in ("input_ids", "positions", "slot_mapping"):
            assert np.array_equal(got[k], case[k]), (case["name"], k)
        if not case["is_prefill"]:
            assert np.array_equal(got["block_tables"], case["block_tables"]), case["name"]
            assert np.array_equal(got["context_lens"], case["context_lens"]), case["name"]


def test_pack_config3(device):
    _say("pack config3")
    step = workloads.mixed_step(seed=2)
    mb = step.batch.block_tables.shape[1]
    got = _pack_on_gpu(device, step.descs.numpy(), step.block_ids.numpy(),
                       step.token_ids.numpy(), 16, mb)
    assert np.array_equal(got["slot_mapping"], step.slot_mapping.numpy())
    assert np.array_equal(got["positions"], step.positions.numpy())
    assert np.array_equal(got["input_ids"], step.token_ids.numpy())
    assert np.array_equal(got["cu_seqlens"], step.batch.cu_seqlens.numpy())
    assert np.array_equal(got["context_lens"], step.batch.context_lens.numpy())
    assert np.array_equal(got["block_tables"], step.batch.block_tables.numpy())
