"""GPU parity at realistic magnitudes: codebooks with the statistics of
trained residual-ordered ones (stage norms 11.5 -> 2.2, absolute maximum
near 9-10; tests/_synth.residual_codebooks) instead of N(0, 0.02).

Covered bit for bit against the oracle: the LUT builder (both forms, fp32 and
fp16 codebooks), the fused G = 4 scorer on codes that real keys produce, the
greedy encode on all its kernels, the codebook manager's serving methods, and
the one-launch decode step's selection.  The fp16 table's range is checked too (no entry overflows).
"""
import numpy as np
import pytest
import torch

from _forms import encode_forms
from _synth import c3_keys, residual_codebooks

pytestmark = pytest.mark.gpu

Hq, Hkv, D = 32, 8, 128


def _np_u16(t):
    return t.detach().cpu().contiguous().view(torch.int16).numpy().view(np.uint16)


def _query(seed, n=Hq):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(n, D, generator=g) * (torch.rand(D, generator=g) * 2.5 + 0.5)).bfloat16()


@pytest.fixture(scope="module")
def cb():
    return residual_codebooks(41)


@pytest.fixture(scope="module")
def K(dev):
    from laprune_amd import aq_kernels as K
    return K


@pytest.fixture(params=["mfma", "dpp"])
def lut_impl(request, monkeypatch):
    monkeypatch.setenv("LAPRUNE_LUT_IMPL", request.param)
    return request.param


@pytest.mark.parametrize("cdt", [torch.float32, torch.float16])
def test_lut_residual_codebooks(dev, K, orc, cb, lut_impl, cdt):
    q = _query(42)
    cbx = cb.to(cdt)
    lut = K.aq_lut_build(q.to(dev), cbx.to(dev), G=4, layout="gmkg")
    torch.cuda.synchronize()
    want = orc.lut_to_gmkg(orc.lut_build(q.float().numpy(), cbx.float().numpy()), 4)
    got = _np_u16(lut)
    assert np.array_equal(got, want)
    vals = np.abs(orc.h_vals(want.reshape(-1)))
    assert np.isfinite(vals).all() and vals.max() < 65504
    print(f"LUT |max| {vals.max():.1f} ({cdt})")


def test_score_residual_codebooks_real_codes(dev, K, orc, cb):
    """Codes from encoding keys (skewed entry use, as real caches have), the
    fused scorer through lap_lut_score_grouped's G = 4 path."""
    from laprune_amd import _native as N
    T = 8192
    keys = c3_keys(43, Hkv=Hkv, n_tok=T).reshape(Hkv * T, D)
    prep = K.aq_encode_prepare(cb.to(dev))
    codes, _ = K.aq_encode_greedy(keys.to(dev), cb.to(dev), prep)
    codes = codes.view(Hkv, T, 32)
    q = _query(44)
    lut = K.aq_lut_build(q.to(dev), cb.to(dev), G=4, layout="gmkg")
    out = torch.empty(Hq, T, dtype=torch.float16, device=dev)
    N.call("lap_lut_score_grouped", N.ptr(lut), N.LUT_GMKG, N.ptr(codes), codes.stride(0),
           codes.stride(1), Hkv, 4, T, 32, 256, N.ptr(out), N.stream_of(out))
    torch.cuda.synchronize()
    lut_h = orc.lut_build(q.float().numpy(), cb.numpy())
    want = orc.score_grouped(lut_h, codes.cpu().numpy(), 4)
    assert np.array_equal(_np_u16(out), want)
    used = np.bincount(codes.cpu().numpy()[:, :, 0].ravel(), minlength=256)
    print(f"stage-0 entries used: {int((used > 0).sum())} of 256")


@encode_forms(64, 128, 256)
def test_encode_residual_codebooks(dev, K, orc, form):
    """C3-shaped keys (norms about 28 at head dim 128) against residual codebooks,
    on every encode kernel."""
    cb = residual_codebooks(41, form)
    x = c3_keys(45, D=form)
    codes, rn = K.aq_encode_greedy(x.to(dev), cb.to(dev))
    torch.cuda.synchronize()
    want_c, want_r = orc.encode(x.numpy(), cb.numpy())
    assert np.array_equal(codes.cpu().numpy(), want_c)
    assert np.array_equal(rn.cpu().numpy().view(np.uint32), want_r.view(np.uint32))
    print(f"D = {form}: mean residual norm {float(want_r.mean()):.3f} "
          f"of key norm {float(np.linalg.norm(x.numpy(), axis=1).mean()):.3f}")


def test_encode_residual_codebooks_large_launch(dev, K, orc, cb):
    """40,000 rows take the wide kernel on a 256-CU device; sampled rows checked."""
    g = torch.Generator().manual_seed(46)
    N = 40000
    x = (torch.randn(N, D, generator=g) * (torch.rand(D, generator=g) * 3.5 + 0.5))
    codes, rn = K.aq_encode_greedy(x.to(dev), cb.to(dev))
    torch.cuda.synchronize()
    rows = np.unique(np.concatenate([np.arange(64), np.arange(N - 64, N),
                                     torch.randperm(N, generator=g)[:256].numpy()]))
    want_c, want_r = orc.encode(x.numpy()[rows], cb.numpy())
    assert np.array_equal(codes.cpu().numpy()[rows], want_c)
    assert np.array_equal(rn.cpu().numpy()[rows].view(np.uint32), want_r.view(np.uint32))


def test_manager_residual_codebooks(dev, orc, cb):
    from laprune_amd.aq_kv import AQLayerCodebookManager, AQLayerConfig
    cfg = AQLayerConfig(M=32, K=256, d=D, heads_per_group=4, num_heads=Hkv)
    m = AQLayerCodebookManager({0: cfg}, device=dev)
    m.set_codebooks(0, 0, cb)
    q = _query(47, n=Hkv * 4).half()
    codes = torch.randint(0, 256, (Hkv, 3000, 32), generator=torch.Generator().manual_seed(48),
                          dtype=torch.uint8)
    got = m.approx_inner_product_multihead_gqa(0, q.to(dev), codes.to(dev), 4)
    want = orc.score_grouped(orc.lut_build(q.float().numpy(), cb.numpy()), codes.numpy(), 4)
    assert np.array_equal(_np_u16(got), want)
    x = c3_keys(49, Hkv=1, n_tok=300)
    got_c = m.encode_keys_batch(0, 0, x.to(dev), icm_iters=0)
    assert np.array_equal(got_c.cpu().numpy(), orc.encode(x.numpy(), cb.numpy())[0])


def test_decode_step_residual_codebooks(dev, orc, cb):
    """The one-launch step at T = 16384 with codes of real keys and a
    realistic query: the selected indices bit for bit against the oracle."""
    from laprune_amd import aq_kernels as K
    from laprune_amd.retrieval import RetrievalConfig, SparseDecoder
    T = 16384
    keys = c3_keys(50, Hkv=Hkv, n_tok=T)  # [Hkv * T, D]
    codes, _ = K.aq_encode_greedy(keys.to(dev), cb.to(dev))
    codes = codes.view(1, Hkv, T, 32)
    kk = keys.view(1, Hkv, T, D).bfloat16().to(dev)
    gv = torch.Generator(device=dev).manual_seed(51)
    vv = torch.randn((1, Hkv, T, D), generator=gv, device=dev).bfloat16()
    q = _query(52).view(1, Hq, 1, D)
    cfg = RetrievalConfig(topk=1024, sink_size=4, local_window=64, select="group",
                          score_dtype=torch.bfloat16)
    dec = SparseDecoder(cb.to(dev), 1, Hq, Hkv, D, T, cfg, dtype=torch.bfloat16)
    dec.step(q.to(dev), codes, kk, vv)
    torch.cuda.synchronize()
    sel = dec.selected().cpu().numpy()[0]
    p = dec.plan(T, T)
    s = orc.score_grouped(orc.lut_build(q[0, :, 0].float().numpy(), cb.numpy()),
                          codes[0].cpu().numpy(), 4)
    want = orc.topk(s, p["k"], 4, p["cand_start"], p["cand_end"], key_bf16=True)
    assert np.array_equal(sel.astype(np.int64), want)
    assert dec.fused_status() == (0, 0)
