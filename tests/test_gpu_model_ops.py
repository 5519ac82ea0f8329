"""The element-wise kernels of a single-token decode step (RMSNorm, silu * mul,
rotary tables, argmax) against the model code's own tensor ops, and the
wrapped modules' route for inputs the kernels do not serve."""
import math

import pytest
import torch
from torch.autograd import forward_ad

pytestmark = pytest.mark.gpu

DTYPES = [torch.bfloat16, torch.float16]


def _ulp_close(got, want, ulps=1):
    """Equal, or neighbouring values of the dtype: the fp32 values before the
    rounding differ in the order of a sum or in the last bit of an exp."""
    i = lambda t: torch.where(t.view(torch.int16) < 0, -32768 - t.view(torch.int16).int(),
                              t.view(torch.int16).int())
    assert (i(got) - i(want)).abs().max().item() <= ulps


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H", [8, 72, 4096, 4104, 8192, 8200, 28672])
def test_rms_norm(dtype, H):
    from laprune_amd._ops import ops
    from transformers.models.llama.modeling_llama import LlamaRMSNorm
    g = torch.Generator(device="cuda").manual_seed(H)
    m = LlamaRMSNorm(H, eps=1e-5).to("cuda", dtype)
    with torch.no_grad():
        m.weight.normal_(1.0, 0.3, generator=g)
        x = torch.randn((3, 1, H), generator=g, device="cuda").mul(2.5).to(dtype)
        out = torch.empty_like(x)
        ops().rms_norm(x, m.weight, m.variance_epsilon, out)
        # two roundings: a last-bit difference of the first may move the second
        _ulp_close(out, m(x), 2)


def test_rms_norm_of_no_columns_is_refused():
    from laprune_amd._ops import ops
    x, w = (torch.empty(s, dtype=torch.bfloat16, device="cuda") for s in ((2, 1, 0), (0,)))
    with pytest.raises(RuntimeError, match="rms_norm"):
        ops().rms_norm(x, w, 1e-5, torch.empty_like(x))


def test_empty_batches_run_the_models_code():
    layer = _layer()
    x = torch.empty((0, 1, 64), dtype=torch.bfloat16, device="cuda")
    with torch.no_grad():
        for f in _calls(layer, x):
            assert f(x).shape == x.shape


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n", [2, 510, 514, 14336])
def test_silu_mul(dtype, n):
    from laprune_amd._ops import ops
    g = torch.Generator(device="cuda").manual_seed(n)
    a = torch.randn((2, 1, n), generator=g, device="cuda").mul(6).to(dtype)
    b = torch.randn((2, 1, n), generator=g, device="cuda").to(dtype)
    a.view(-1)[0] = -math.inf
    a.view(-1)[1] = math.nan
    out = torch.empty_like(a)
    ops().silu_mul(a, b, out)
    want = torch.nn.functional.silu(a) * b
    assert torch.equal(out.isnan(), want.isnan())
    ok = ~want.isnan()
    _ulp_close(out[ok], want[ok], 2)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("freq", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("D", [2, 64, 128, 256])
def test_rope_tables(dtype, freq, D):
    from laprune_amd._ops import ops
    f = (1.0 / 500000.0 ** (torch.arange(0, D, 2, device="cuda").float() / D)).to(freq)
    pos = torch.tensor([[0], [1], [8191], [131071]], device="cuda")
    cos = torch.empty((4, 1, D), dtype=dtype, device="cuda")
    sin = torch.empty_like(cos)
    ops().rope_tables(pos, f, 1.25, cos, sin)
    a = (pos.float() * f.float())[:, None]
    a = torch.cat((a, a), -1)
    _ulp_close(cos, (a.cos() * 1.25).to(dtype))
    _ulp_close(sin, (a.sin() * 1.25).to(dtype))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("V,stride,copy", [(1, 1, True), (7, 9, False), (8, 8, True),
                                           (8191, 8191, True), (8193, 8200, False),
                                           (8200, 8200, True), (65544, 65544, False),
                                           (128256, 128256, True)])
def test_argmax_rows(dtype, V, stride, copy):
    from laprune_amd._ops import ops
    g = torch.Generator(device="cuda").manual_seed(V)
    x = torch.randn((6, stride), generator=g, device="cuda").to(dtype)[:, :V]
    x[1] = -math.inf
    x[2] = 0.0
    x[2, V // 2:] = -0.0
    x[3, V // 3] = math.nan
    x[3, V - 1] = math.nan
    x[4, V // 2:] = 50.0  # ties: the first
    x[5] = -0.0
    x[5, V - 1] = 0.0     # equal to -0: the first
    out = torch.empty((6, 1), dtype=torch.long, device="cuda")
    to = torch.full((6, V), 9.0, dtype=dtype, device="cuda") if copy else None
    ops().argmax_rows(x, out, to)
    if copy:
        assert torch.equal(to.view(torch.int16), x.contiguous().view(torch.int16))
    f = x.cpu().float()
    want = [next(i for i, v in enumerate(r.tolist())
                 if (math.isnan(v) if r.isnan().any() else v == r.max().item())) for r in f]
    assert out[:, 0].tolist() == want


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("N,K", [(1, 8), (7, 64), (8, 2048), (9, 2056), (1001, 2040),
                                 (64, 4096), (6, 14336), (4099, 520)])
def test_gemv(dtype, N, K):
    """Against the products in 64 bits: the fp32 sum of K exact products errs by
    at most K * 2^-24 of the sum of their magnitudes, the rounding by half a
    unit of the dtype; the fused MLP part equals its unfused ops on the
    kernel's own projections (silu's exp may differ in its last bit)."""
    from laprune_amd._ops import ops
    g = torch.Generator(device="cuda").manual_seed(N * 7 + K)
    x = torch.randn((1, 1, K), generator=g, device="cuda").to(dtype)
    w = torch.randn((2, N, K), generator=g, device="cuda").mul(0.1).to(dtype)
    got = torch.empty((2, 1, 1, N), dtype=dtype, device="cuda")
    for i in range(2):
        ops().gemv(x, w[i], got[i])
    want = w.double() @ x.double().view(K)
    mag = w.double().abs() @ x.double().abs().view(K)
    half = 2.0 ** (-8 if dtype is torch.bfloat16 else -11)
    err = (got.view(2, N).double() - want).abs()
    assert (err <= want.abs() * half + mag * K * 2.0 ** -24 * (1 + half) + 2.0 ** -25).all()
    glu = torch.empty((1, 1, N), dtype=dtype, device="cuda")
    ops().gemv_glu(x, w[0], w[1], glu)
    _ulp_close(glu, torch.nn.functional.silu(got[0]) * got[1], 2)


@pytest.mark.parametrize("N,K,own", [(8192, 64, True), (8200, 64, False), (151936, 384, False),
                                     (8200, 512, True), (64, 8, True)])
def test_short_rows_keep_the_librarys_product(N, K, own):
    """The projection kernel takes one token where it is the faster one."""
    from laprune_amd.llama import _one_vector
    x = torch.zeros((1, 1, K), dtype=torch.bfloat16, device="cuda")
    w = torch.zeros((N, K), dtype=torch.bfloat16, device="cuda")
    with torch.no_grad():
        assert _one_vector(x, w) == own


def test_wrapped_modules_keep_the_models_code_elsewhere():
    """Prompt lengths, gradients and fp32 run the class's own forward; the expected
    values come from a copy that was never wrapped."""
    import copy
    from laprune_amd.llama import _fuse_decode_ops
    from transformers import LlamaConfig, LlamaForCausalLM
    torch.manual_seed(0)
    cfg = LlamaConfig(vocab_size=64, hidden_size=64, intermediate_size=96, num_hidden_layers=1,
                      num_attention_heads=2, num_key_value_heads=1)
    model = LlamaForCausalLM(cfg).to("cuda", torch.bfloat16).eval()
    plain = copy.deepcopy(model)
    _fuse_decode_ops(model)
    pos = torch.arange(5, device="cuda")[None]

    def run(m, x, p):
        layer = m.model.layers[0]
        return [layer.input_layernorm(x), layer.mlp(x), layer.self_attn.o_proj(x), m.lm_head(x),
                *m.model.rotary_emb(x, p)]

    for dt, T, grad in ((torch.bfloat16, 5, False), (torch.bfloat16, 1, True),
                        (torch.float32, 1, False), (torch.bfloat16, 1, False)):
        model.to(dt), plain.to(dt)
        assert not any("forward" in m.__dict__ for m in plain.modules())
        x = torch.randn((1, T, 64), device="cuda", dtype=dt)
        with torch.set_grad_enabled(grad):
            want, got = run(plain, x, pos[:, :T]), run(model, x, pos[:, :T])
        for a, b in zip(got, want):
            assert a.dtype == b.dtype and a.requires_grad == b.requires_grad
            if dt is torch.bfloat16 and T == 1 and not grad:
                # roundings to bf16 of fp32 sums in another order
                torch.testing.assert_close(a, b, rtol=2 ** -6, atol=2 ** -9)
            else:
                assert torch.equal(a, b)


def _layer(I=96):
    from laprune_amd.llama import _fuse_decode_ops
    from transformers import LlamaConfig, LlamaForCausalLM
    torch.manual_seed(0)
    cfg = LlamaConfig(vocab_size=64, hidden_size=64, intermediate_size=I, num_hidden_layers=1,
                      num_attention_heads=2, num_key_value_heads=1)
    model = LlamaForCausalLM(cfg).to("cuda", torch.bfloat16).eval()
    _fuse_decode_ops(model)
    return model.model.layers[0]


@pytest.mark.parametrize("B", [1, 3])
def test_hooks_on_the_activation_run(B):
    """The fused MLP leaves the activation's call out, unless something waits for it
    or stands in its place."""
    x = torch.randn((B, 1, 64), device="cuda", dtype=torch.bfloat16)
    with torch.no_grad():
        mlp, seen = _layer().mlp, []
        h = mlp.act_fn.register_forward_hook(lambda m, i, o: seen.append(o) or 2 * o)
        want = mlp.down_proj(2 * torch.nn.functional.silu(mlp.gate_proj(x)) * mlp.up_proj(x))
        assert torch.equal(mlp(x), want) and len(seen) == 1
        h.remove()
        mlp.act_fn.forward = lambda t: 0 * t
        assert not mlp(x).any()
        del mlp.act_fn.forward
        h = torch.nn.modules.module.register_module_forward_hook(
            lambda m, i, o: seen.append(m) if m is mlp.act_fn else None)
        mlp(x)
        h.remove()
        assert seen[-1] is mlp.act_fn


def _calls(layer, x):
    yield from (lambda t: layer.mlp(t), lambda t: layer.input_layernorm(t),
                lambda t: layer.self_attn.o_proj(t))


@pytest.mark.parametrize("B", [1, 3])
def test_forward_mode_tangents_pass_through(B):
    layer = _layer()
    x, t = torch.randn((2, B, 1, 64), device="cuda", dtype=torch.bfloat16)
    with torch.no_grad():
        for f in _calls(layer, x):
            with forward_ad.dual_level():
                got = forward_ad.unpack_dual(f(forward_ad.make_dual(x, t)))
            want = torch.func.jvp(f, (x,), (t,))
            assert torch.equal(got.primal, want[0]) and torch.equal(got.tangent, want[1])
            assert got.tangent.any()


def test_vmap_passes_through():
    layer = _layer()
    xs = torch.randn((5, 1, 1, 64), device="cuda", dtype=torch.bfloat16)
    with torch.no_grad():
        for f in _calls(layer, xs):
            got = torch.vmap(f)(xs)
            # bf16 results of fp32 sums in another order
            torch.testing.assert_close(got, torch.stack([f(x) for x in xs]), rtol=2 ** -6,
                                       atol=2 ** -9)


def test_modes_and_traces_see_the_models_ops():
    from torch.utils.flop_counter import FlopCounterMode
    layer = _layer().requires_grad_(False)
    x = torch.randn((1, 1, 64), device="cuda", dtype=torch.bfloat16)
    with torch.no_grad():
        with FlopCounterMode(display=False) as c:
            layer.mlp(x)
        assert c.get_total_flops() == 3 * 2 * 64 * 96
        traced = torch.jit.trace(lambda t: layer.mlp(t), x, check_trace=False)
        assert "laprune::" not in str(traced.graph)
        from torch.fx.experimental.proxy_tensor import make_fx
        graph = make_fx(lambda t: layer.mlp(t))(x).graph
        assert not any("laprune" in str(n.target) for n in graph.nodes)
        compiled = torch.compile(layer.mlp, backend="eager", fullgraph=True)
        torch.testing.assert_close(compiled(x), layer.mlp(x), rtol=2 ** -6, atol=2 ** -9)


def test_weights_of_another_class_keep_their_product():
    class Doubled(torch.Tensor):
        @classmethod
        def __torch_function__(cls, func, types, args=(), kwargs=None):
            plain = [a.as_subclass(torch.Tensor) if isinstance(a, Doubled) else a for a in args]
            out = func(*plain, **(kwargs or {}))
            return 2 * out if func is torch.nn.functional.linear else out

    layer = _layer()
    x = torch.randn((1, 1, 64), device="cuda", dtype=torch.bfloat16)
    with torch.no_grad():
        for mod in (layer.self_attn.o_proj, layer.mlp.gate_proj):
            w = mod.weight.detach()
            del mod.weight
            mod.weight = w.as_subclass(Doubled)
            assert torch.equal(mod(x), 2 * torch.nn.functional.linear(x, w))
        g, u = mod(x), layer.mlp.up_proj(x)
        torch.testing.assert_close(layer.mlp(x), layer.mlp.down_proj(
            torch.nn.functional.silu(g) * u), rtol=2 ** -6, atol=2 ** -9)
