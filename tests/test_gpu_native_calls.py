"""The native call path of litevllm.ops (litevllm/_native.so) against the
wrappers' own Python path: the same results bit for bit on the forms both
accept, the same refusals, and a None (nothing launched) for what is not of
the plain form."""

from __future__ import annotations

import types

import pytest
import torch

from litevllm import _hip, ops, workloads

pytestmark = pytest.mark.gpu

NAMES = ("kv_scatter", "paged_attention", "sample", "add_rms_norm", "qk_norm_rope_cache",
         "silu_mul", "linear")


def _calls(device):
    """(name, call) pairs; each call returns fresh tensors to compare."""
    b = workloads.mixed_step(seed=3, num_decodes=5, dec_lo=1, dec_hi=300, num_chunks=2,
                             chunk_len=33, off_hi=90, num_cache_slots=16 * 300).batch.to(device)
    bf = dict(device=device, dtype=torch.bfloat16)
    g = torch.Generator(device=device).manual_seed(5)
    wide = torch.randn(12, 4096, generator=g, **bf)
    w = torch.randn(1024, generator=g, **bf)
    wl = torch.randn(512, 1024, generator=g, **bf)
    pos, slots = torch.arange(12, device=device), torch.arange(12, device=device) * 3
    cos = torch.randn(64, 64, generator=g, **bf)
    temp = torch.tensor([0.0, 0.7, 1.0], device=device)
    uni = torch.tensor([0.0, 0.3, 0.9], device=device)

    def attention(**kw):
        return lambda: ops.paged_attention(b.query, b.key_cache, b.value_cache, b.block_tables,
                                           b.context_lens, scale=b.scale, cu_seqlens=b.cu_seqlens,
                                           max_query_len=b.max_query_len, **kw)

    def scatter():
        kc = torch.zeros(4, 16, 2, 64, **bf)
        vc = torch.zeros_like(kc)
        ops.kv_scatter(wide[:, :128].view(12, 2, 64), wide[:, 128:256].view(12, 2, 64), kc, vc,
                       slots)
        return torch.stack([kc, vc])

    def norm():
        r = wide[:, 1024:2048].clone()
        return torch.stack([ops.add_rms_norm(wide[:, :1024], w, 1e-6, residual=r), r])

    def rope():
        kc = torch.zeros(4, 16, 2, 128, **bf)
        vc = torch.zeros_like(kc)
        q = ops.qk_norm_rope_cache(wide[:, :1024], 4, 2, 128, cos, cos, pos, slots, kc, vc,
                                   q_norm_weight=w[:128])
        return torch.cat([q.flatten(), kc.flatten(), vc.flatten()])
    ws = torch.empty(1 << 24, dtype=torch.uint8, device=device)
    out = torch.empty(b.query.shape[0], 16, 256, **bf)[:, :, :128].contiguous()
    return [
        ("decode + chunks", attention(num_decodes=5)),
        ("attention, out and workspace", attention(num_decodes=5, out=out, workspace=ws)),
        ("attention, chunks only", attention()),
        ("decode with an empty plan",
         attention(num_decodes=5, prefix=ops.prefix_plan([], 5, 2, device))),
        ("scatter", scatter), ("norm", norm), ("rope", rope),
        ("sample", lambda: ops.sample(wide[:3], temp, uni)),
        ("greedy", lambda: ops.sample(wide[:3], temp * 0)),
        ("silu", lambda: ops.silu_mul(wide[:, :2048])),
        ("linear", lambda: ops.linear(wide[:, 1024:2048], wl)),
        ("linear silu", lambda: ops.linear(wide[:, 1024:2048], wl, activation="silu_mul")),
    ]


def _counting(taken, name, fn):
    def call(*a):
        r = fn(*a)
        taken.append((name, r))
        return r
    return call


def test_native_equals_python_path(device, monkeypatch):
    native = ops._native()
    taken = []
    counted = types.SimpleNamespace(**{
        n: _counting(taken, n, getattr(native, n))
        for n in NAMES})
    none = types.SimpleNamespace(**{n: (lambda *a: None) for n in NAMES})
    for what, call in _calls(device):
        monkeypatch.setattr(ops, "_native_module", none)
        want = call().clone()
        monkeypatch.setattr(ops, "_native_module", counted)
        taken.clear()
        got = call()
        print(f"[case] {what}", flush=True)
        if what != "greedy":          # (uniform omitted: the Python path makes the zeros)
            assert taken and taken[-1][1] is not None, what
        assert torch.equal(got.view(torch.int16) if got.dtype == torch.bfloat16 else got,
                           want.view(torch.int16) if want.dtype == torch.bfloat16 else want), what


def test_native_refuses_what_the_wrappers_refuse(device):
    native = ops._native()
    x = torch.randn(8, 1024, device=device, dtype=torch.bfloat16)
    w = torch.ones(1024, device=device, dtype=torch.bfloat16)
    for bad in [(x.cpu(), w), (x, w.cpu()), (x, w.float()), (x[:, ::2], w[:512]), (x.double(), w),
                (x, w[:512]), (x, torch.ones(2048, device=device, dtype=torch.bfloat16)[::2])]:
        assert native.add_rms_norm(*bad, 1e-6, None, None) is None
        with pytest.raises(RuntimeError):
            ops.add_rms_norm(*bad, 1e-6)
    assert native.linear(x, torch.ones(32, 512, device=device, dtype=torch.bfloat16), 0, None) is None
    assert native.silu_mul(x, x.float()) is None and native.kv_scatter(x, x, x, x, x) is None
    # what only the library refuses raises with its message
    with pytest.raises(RuntimeError, match="lv_linear failed"):
        ops.linear(x, torch.ones(31, 1024, device=device, dtype=torch.bfloat16))
    with pytest.raises(RuntimeError, match="lv_add_rms_norm failed"):
        native.add_rms_norm(x[:, 1:1021], w[:1020], 1e-6, None, None)
    # another stream has no scratch of its own yet: left to the wrapper, which makes it
    b = workloads.paged_decode(seed=1, num_seqs=2, ctx_lo=5, ctx_hi=40).to(device)
    args = (b.query, b.key_cache, b.value_cache, b.block_tables, b.context_lens)
    want = ops.paged_attention(*args, scale=b.scale)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        key = (torch.cuda.current_device(), side.cuda_stream, "attn")
        ops._workspaces.pop(key, None)
        rest = (None, b.scale, None, None, 1, None, None, None, None)
        assert native.paged_attention(*args, *rest) is None
        ops.paged_attention(*args, scale=b.scale)
        assert key in ops._workspaces
        got = native.paged_attention(*args, *rest)
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    assert ops._native() is native and _hip.load() is not None
