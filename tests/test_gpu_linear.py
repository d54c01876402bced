"""lv_linear (decode-sized linear layers on MFMA) against float32 products of
the same bf16/fp16 operands.

A library GEMM rounds the fp32 sum once to the dtype, so both lv_linear and
torch's GEMM sit within one rounding of the fp32 product (relative 2^-8 for
bf16); the bound used is 1.5 units in the last place of the output plus the
fp32 summation-order slack."""

from __future__ import annotations

import os

import pytest
import torch

from litevllm import ops

pytestmark = pytest.mark.gpu

SHAPES = [  # (N, K): qkv, o, gate_up, down of the Qwen3-0.6B shape, a small lm_head
    (4096, 1024), (1024, 2048), (6144, 1024), (1024, 3072), (32000, 1024)]


def _ulp(t: torch.Tensor, dtype: torch.dtype) -> torch.Tensor:
    """Spacing of `dtype` values at |t| (t in float32)."""
    mant = 8 if dtype == torch.bfloat16 else 11
    e = torch.floor(torch.log2(t.float().abs().clamp_min(1e-30)))
    return torch.pow(2.0, e - (mant - 1))


def _check(got: torch.Tensor, ref32: torch.Tensor, k: int, scale: torch.Tensor) -> None:
    err = (got.float() - ref32).abs()
    # output rounding (<= 1 ulp of the value; 1.5 allows the value near a
    # binade edge) + fp32 accumulation slack ~ k * 2^-24 * sum |x w|
    bound = 1.5 * _ulp(ref32, got.dtype) + k * 2.0 ** -22 * scale + 1e-6
    bad = err > bound
    assert not bad.any(), (f"{int(bad.sum())} of {err.numel()} beyond bound; "
                           f"max err {err.max():.3e}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m", [1, 7, 64, 200, 256])
@pytest.mark.parametrize("nk", SHAPES)
def test_linear_matches_fp32_product(dtype, m, nk):
    n, k = nk
    g = torch.Generator(device="cuda").manual_seed(m * 7 + n + k)
    x = torch.randn(m, k, device="cuda", generator=g).to(dtype)
    w = (torch.randn(n, k, device="cuda", generator=g) * k ** -0.5).to(dtype)
    assert ops.linear_supported(m, n, k, dtype)
    y = ops.linear(x, w)
    ref = x.float() @ w.float().T
    scale = x.float().abs() @ w.float().abs().T
    _check(y, ref, k, scale)
    torch.cuda.synchronize()


@pytest.mark.parametrize("cfg", ["0", "1", "2", "3"])
def test_every_tile_shape_gives_the_same_sums(cfg, monkeypatch):
    """Each forced tile configuration is within the bound of the fp32
    product; ragged m exercises the clamped rows."""
    n, k, m = 1024, 2048, 77
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn(m, k, device="cuda", generator=g).to(torch.bfloat16)
    w = (torch.randn(n, k, device="cuda", generator=g) * k ** -0.5).to(torch.bfloat16)
    monkeypatch.setenv("LV_LINEAR_CFG", cfg)
    y = ops.linear(x, w)
    monkeypatch.delenv("LV_LINEAR_CFG")
    ref = x.float() @ w.float().T
    _check(y, ref, k, x.float().abs() @ w.float().abs().T)


def test_strided_rows_and_out_buffer():
    n, k, m = 4096, 1024, 33
    x_big = torch.randn(m, k + 64, device="cuda").to(torch.bfloat16)
    x = x_big[:, 32:32 + k]
    w = (torch.randn(n, k, device="cuda") * k ** -0.5).to(torch.bfloat16)
    out_big = torch.full((m, n + 32), 7.0, device="cuda", dtype=torch.bfloat16)
    out = out_big[:, :n]
    ops.linear(x, w, out=out)
    ref = x.float() @ w.float().T
    _check(out, ref, k, x.float().abs() @ w.float().abs().T)
    assert torch.all(out_big[:, n:] == 7.0)


def test_unsupported_shapes_raise_and_report():
    assert not ops.linear_supported(8, 100, 1024, torch.bfloat16)   # n % 32
    assert not ops.linear_supported(8, 100, 1024, torch.bfloat16, "silu_mul")
    assert not ops.linear_supported(8, 1024, 1000, torch.bfloat16)  # k % 128
    assert not ops.linear_supported(8, 1024, 1024, torch.float32)
    x = torch.randn(8, 1000, device="cuda").to(torch.bfloat16)
    w = torch.randn(1024, 1000, device="cuda").to(torch.bfloat16)
    with pytest.raises(RuntimeError, match="no kernel"):
        ops.linear(x, w)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m", [1, 64, 200, 256])
@pytest.mark.parametrize("cfg", ["0", "1"])
def test_silu_mul_epilogue_equals_plain_then_silu_mul(dtype, m, cfg, monkeypatch):
    """The fused gate|up + SiLU form gives exactly lv_silu_mul of the plain
    product (same k order of the sums), and is within rounding of the fp32
    composition silu(x g^T) * (x u^T)."""
    inter, k = 3072, 1024
    g = torch.Generator(device="cuda").manual_seed(m + 11)
    x = torch.randn(m, k, device="cuda", generator=g).to(dtype)
    w = (torch.randn(2 * inter, k, device="cuda", generator=g) * k ** -0.5).to(dtype)
    assert ops.linear_supported(m, inter, k, dtype, "silu_mul")
    monkeypatch.setenv("LV_LINEAR_SILU_CFG", cfg)
    fused = ops.linear(x, w, activation="silu_mul")
    monkeypatch.delenv("LV_LINEAR_SILU_CFG")
    plain = ops.linear(x, w)
    assert torch.equal(fused, ops.silu_mul(plain))
    ref = x.float() @ w.float().T
    gate, up = ref[:, :inter], ref[:, inter:]
    want = torch.nn.functional.silu(gate) * up
    err = (fused.float() - want).abs()
    tol = (4 * _ulp(want, dtype) + 4 * _ulp(up, dtype) * (gate.abs() + 1)
           + 2 * _ulp(gate, dtype) * up.abs() + 1e-5)
    assert (err <= tol).all(), err.max()


@pytest.mark.parametrize("m", [1, 31, 32, 33, 320])
@pytest.mark.parametrize("nk", [(512, 256), (33, 4), (31, 36), (256, 688), (1, 60), (100, 2052)])
def test_linear_f32_matches_fp64(m, nk):
    """fp32 products and sums: k 2^-24 of sum |x w| bounds any order of the
    sum.  Edges of the 32 x 32 tiles, a last half chunk (k % 8 == 4), strided
    rows; nothing is written past the output's columns."""
    n, k = nk
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k + 4, device="cuda", generator=g)[:, 4:]
    w = torch.randn(n, k + 8, device="cuda", generator=g)[:, :k]
    buf = torch.full((m, n + 3), 7.0, device="cuda")
    y = ops.linear_f32(x, w, out=buf[:, :n])
    ref = x.double() @ w.double().T
    bound = (k + 1) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    assert ((y.double() - ref).abs() <= bound).all()
    assert (buf[:, n:] == 7.0).all()


def test_linear_f32_forms_left_to_the_library():
    """The layer runs what lv_linear_f32 has no kernel for on the library, and
    keeps autograd; the op itself refuses such operands."""
    from litevllm.models.llama import Linear
    lin = Linear(256, 64, bias=False).cuda()
    x = torch.randn(9, 257, device="cuda")
    assert ops.linear_f32_if_plain(x[:, 1:], lin.weight) is None     # rows off 16 bytes
    with pytest.raises(RuntimeError, match="16-byte aligned"):
        ops.linear_f32(x[:, 1:], lin.weight.detach())
    with torch.inference_mode():
        y = lin(x[:, 1:])
        z = lin(x[:, :256].contiguous())
    for got, a in ((y, x[:, 1:]), (z, x[:, :256])):
        ref = a.double() @ lin.weight.detach().double().T
        assert (got.double() - ref).norm() <= 1e-6 * ref.norm()
    lin(x[:, :256].contiguous()).sum().backward()
    assert lin.weight.grad is not None


def _layer_and_reference(dtype, k=512, n=64):
    from litevllm.models.llama import Linear
    torch.manual_seed(3)
    lin = Linear(k, n, bias=False).to(device="cuda", dtype=dtype)
    ref = torch.nn.Linear(k, n, bias=False).to(device="cuda", dtype=dtype)
    ref.load_state_dict(lin.state_dict())
    return lin, ref


@pytest.mark.parametrize("dtype,m", [(torch.float32, 9), (torch.bfloat16, 300)])
def test_layer_is_nn_linear_to_autograd_autocast_and_transforms(dtype, m):
    """Without reverse-mode gradients too, whatever else follows a call by the
    dispatcher gets nn.Linear's product: tangents, autocast's type, traces that
    record the product, vmap, dispatch and function modes, lazy negation."""
    import torch.autograd.forward_ad as fwd
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode
    lin, ref = _layer_and_reference(dtype)
    x, t = (torch.randn(m, 512, device="cuda", dtype=dtype) for _ in range(2))
    tol = 1e-5 if dtype == torch.float32 else 2.0 ** -7

    def close(a, b):
        assert a.dtype == b.dtype and (a - b).float().norm() <= tol * b.float().norm()
    with torch.no_grad():
        close(lin(x), ref(x))
        with fwd.dual_level():
            d = fwd.unpack_dual(lin(fwd.make_dual(x, t)))
            close(d.primal, ref(x))
            close(d.tangent, ref(t))
        y, dy = torch.func.jvp(lin, (x,), (t,))
        close(dy, ref(t))
        other = torch.float16 if dtype == torch.bfloat16 else torch.bfloat16
        with torch.autocast("cuda", dtype=other):
            assert lin(x).dtype == ref(x).dtype == other
        traced = torch.jit.trace(lin, (x,))
        close(traced(t), ref(t))
        compiled = torch.compile(lin, backend="eager", fullgraph=True)
        close(compiled(t), ref(t))
        batch = torch.stack([x, t])
        close(torch.func.vmap(lin)(batch), torch.func.vmap(ref)(batch))
        seen = []

        class Functions(TorchFunctionMode):
            def __torch_function__(self, func, types, args=(), kwargs=None):
                seen.append(func)
                return func(*args, **(kwargs or {}))

        class Ops(TorchDispatchMode):
            def __torch_dispatch__(self, func, types, args=(), kwargs=None):
                seen.append(func)
                return func(*args, **(kwargs or {}))
        with Functions():
            lin(x)
        assert torch.nn.functional.linear in seen
        seen.clear()
        with Ops():
            lin(x)
        assert seen
        if dtype == torch.float32:
            z = torch.complex(t, x).conj().imag          # -x, not yet negated
            assert z.is_neg()
            close(lin(z), ref(z))


@pytest.mark.parametrize("dtype,m", [(torch.float32, 9), (torch.bfloat16, 300),
                                     (torch.float16, 300)])
@torch.inference_mode()
def test_layer_takes_every_row_layout_of_nn_linear(dtype, m, monkeypatch):
    """Rows that overlap, lie off 16-byte boundaries or are columns, and a
    weight that is a view: the library's product, as nn.Linear has it.  With
    LV_DECODE_GEMM_ROWS = 0 every call is."""
    from litevllm.models import llama
    lin, ref = _layer_and_reference(dtype)
    wide = torch.randn(m, 520, device="cuda", dtype=dtype)
    forms = {"contiguous": wide[:, :512].contiguous(), "strided": wide[:, :512],
             "off 16 bytes": wide[:, 1:513], "one row repeated": wide[:1, :512].expand(m, 512),
             "overlapping": wide.flatten().as_strided((m, 512), (8, 1)),
             "columns": wide[:, :512].t().contiguous().t()}
    for name, x in forms.items():
        print(f"[case] {dtype} {name}", flush=True)
        a, b = lin(x), ref(x)
        assert (a - b).float().norm() <= 2.0 ** (-20 if dtype == torch.float32 else -7) * \
            b.float().norm()
        mlp = llama.GatedMLP(512, 512).to(device="cuda", dtype=dtype)
        up = torch.nn.functional.linear(x, mlp.gate_up_proj.weight)
        want = torch.nn.functional.linear(
            torch.nn.functional.silu(up[:, :512]) * up[:, 512:], mlp.down_proj.weight)
        if m > 256 or dtype == torch.float32:
            got = mlp(x)
            assert (got - want).float().norm() <= 2.0 ** -6 * want.float().norm()
    calls = []
    monkeypatch.setattr(llama.ops, "linear", lambda *a, **k: calls.append(a))
    monkeypatch.setattr(llama.ops, "linear_if_plain", lambda *a, **k: calls.append(a))
    monkeypatch.setattr(llama, "DECODE_GEMM_ROWS", 0)
    assert torch.equal(lin(forms["contiguous"]), ref(forms["contiguous"])) and not calls


@torch.inference_mode()
def test_gated_mlp_runs_the_hooks_of_its_projection():
    from litevllm.models.llama import GatedMLP
    mlp = GatedMLP(256, 256).cuda().bfloat16()
    x = torch.randn(300, 256, device="cuda", dtype=torch.bfloat16)
    want, seen = mlp(x), []
    mlp.gate_up_proj.register_forward_hook(lambda mod, args, out: seen.append(out.shape))
    got = mlp(x)
    assert seen == [(300, 512)]
    assert (got - want).float().norm() <= 2.0 ** -6 * want.float().norm()


@torch.inference_mode()
def test_layer_products_leave_graphs_and_slow_sizes_to_the_library():
    """Inside library_products nn.Linear makes the layer's product, in the
    warm-up and in the capture, equal on every replay to its eager one; a
    program's own capture takes the route of its own warm-up; sizes whose
    workgroups do not run at once are the library's."""
    lin, ref = _layer_and_reference(torch.float32)
    x = torch.randn(9, 512, device="cuda")
    own = ops.linear_if_plain(x, lin.weight)
    with ops.library_products():
        assert ops.linear_if_plain(x, lin.weight) is None
        assert torch.equal(lin(x), ref(x))
    assert torch.equal(lin(x), own)
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=stream):
        y = lin(x)
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(y, own)
    graph = torch.cuda.CUDAGraph()
    with ops.library_products(), torch.cuda.graph(graph, stream=stream):
        y = lin(x)
    for _ in range(3):
        x.normal_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.allclose(y, ref(x), rtol=0, atol=1e-5 * float(x.abs().max()))
    for m, n, k, act, own in ((320, 6144, 1024, None, True), (384, 6144, 1024, None, False),
                              (300, 512, 256, None, False), (300, 1024, 512, "silu_mul", True),
                              (300, 512, 512, "silu_mul", False)):
        x, w = (torch.randn(r, k, device="cuda", dtype=torch.bfloat16) for r in (m, n))
        assert (ops.linear_if_plain(x, w, act) is not None) == own, (m, n, k, act)


@torch.inference_mode()
@pytest.mark.parametrize("dtype,m", [(torch.float32, 9), (torch.bfloat16, 9), (torch.bfloat16, 300)])
def test_layer_with_a_bias_or_a_parametrized_weight(dtype, m):
    from torch.nn.utils import parametrize
    from litevllm.models.llama import Linear

    class Half(torch.nn.Module):
        def forward(self, w):
            return w * 0.5
    x = torch.randn(m, 512, device="cuda", dtype=dtype)
    for bias in (False, True):
        lin = Linear(512, 64, bias=bias).to(device="cuda", dtype=dtype)
        want = torch.nn.functional.linear(x, lin.weight * 0.5, lin.bias)
        parametrize.register_parametrization(lin, "weight", Half())
        got = lin(x)
        assert (got - want).float().norm() <= 2.0 ** -7 * want.float().norm()
