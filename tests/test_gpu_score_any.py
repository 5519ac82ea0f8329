"""The scorer for any group size (score_any_kernel): scores bit-exact against the
oracle at the edges of its stages (1024 tokens) and of its 1, 2, 4 and 8 stages
per workgroup, and the decode step's selection against the path that code rows
without 16-byte alignment take (per-head scores, then their top-k)."""
import numpy as np
import pytest
import torch

from _synth import gaussian_codebooks, gen

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K(dev):
    from laprune_amd import aq_kernels
    return aq_kernels


@pytest.mark.parametrize("G,Hkv,T", [
    (1, 8, 1), (2, 3, 1023), (3, 2, 1024), (3, 2, 1025), (5, 1, 2049), (6, 4, 40000),
    (7, 8, 33333), (8, 2, 5000), (8, 8, 131073), (1, 8, 131073), (4, 2, 1500),
    # more than four heads: both sides of the sizes that keep one head per workgroup
    (8, 3, 1), (5, 1, 512), (5, 1, 513), (7, 33, 1023), (6, 32, 1024), (8, 32, 1025),
    (5, 16, 2049), (8, 1, 32768), (8, 1, 32769)])
def test_scores(dev, K, orc, G, Hkv, T):
    print(f"G={G} Hkv={Hkv} T={T}", flush=True)
    g = gen(T)
    lut = (torch.randn(Hkv * G, 32, 256, generator=g) * 0.3).half()
    codes = torch.randint(0, 256, (Hkv, T + 5, 32), generator=g, dtype=torch.uint8)
    dl, dc = lut.to(dev), codes.to(dev)[:, :T]
    got = K.aq_lut_gather_gqa(dl, dc, G, 0, 32)
    if G <= 4:
        assert torch.equal(K.aq_lut_gather_grouped(dl, dc, G), got)
    want = orc.score_grouped(lut.numpy().view(np.uint16), codes[:, :T].numpy(), G)
    assert np.array_equal(got.cpu().numpy().view(np.uint16), want.view(np.uint16))


@pytest.mark.parametrize("select", ["group", "head"])
@pytest.mark.parametrize("G,Hkv,T,k,ragged", [(1, 8, 3000, 100, False), (2, 2, 40001, 700, False),
                                              (5, 2, 9000, 64, True), (8, 4, 33000, 2048, False),
                                              (7, 4, 34567, 1024, True), (8, 1, 70, 9, False)])
def test_step_selection(dev, G, Hkv, T, k, ragged, select):
    """A step over aligned code rows and over the same codes at a pitch of 33
    bytes select the same tokens and attend alike."""
    from laprune_amd.retrieval import RetrievalConfig, SparseDecoder
    print(f"G={G} Hkv={Hkv} T={T} {select}", flush=True)
    B, D = 2, 64
    g = gen(T + G)
    cb = gaussian_codebooks(3, D).to(dev)
    q = torch.randn(B, Hkv * G, 1, D, generator=g).bfloat16().to(dev)
    kk = torch.randn(B, Hkv, T, D, generator=g).bfloat16().to(dev)
    codes = torch.randint(0, 256, (B, Hkv, T, 32), generator=g, dtype=torch.uint8).to(dev)
    odd = torch.zeros(B, Hkv, T, 33, dtype=torch.uint8, device=dev)
    odd[..., :32] = codes
    cfg = RetrievalConfig(topk=k, select=select, score_dtype=torch.bfloat16)
    lens = [T, T // 2] if ragged else [T, T]
    outs = []
    for c in (codes, odd[..., :32]):
        dec = SparseDecoder(cb, B, Hkv * G, Hkv, D, T, cfg)
        o = dec.step(q, c, kk, kk, t_codes=[n - n % 8 for n in lens], t_total=lens).clone()
        outs.append((o, dec.selected().clone()))
    assert torch.equal(outs[0][1], outs[1][1])
    assert torch.equal(outs[0][0], outs[1][0])


@pytest.mark.parametrize("score_dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("select", ["group", "head"])
@pytest.mark.parametrize("G", [1, 3, 7, 8])
def test_step_selection_with_nan_scores(dev, orc, G, select, score_dtype):
    """A group's key is the largest of its heads' keys, a NaN head's among them (a
    positive NaN ranks above every score, a negative one below), whichever path the
    code rows' alignment takes."""
    from laprune_amd.retrieval import RetrievalConfig, SparseDecoder
    print(f"G={G} {select} {score_dtype}", flush=True)
    Hkv, T, D, k = 2, 3000, 64, 40
    g = gen(G)
    lut = (torch.randn(Hkv * G, 32, 256, generator=g) * 0.3).half()
    codes = torch.randint(0, 255, (1, Hkv, T, 32), generator=g, dtype=torch.uint8)
    pos = torch.tensor([150, 1023, 1024, 1700, 2047, 2900])
    neg = torch.tensor([160, 1022, 1025, 2500])
    lut[:, 0, 255] = float("-inf")       # tokens with entry 255: -inf in every head but
    lut[G - 1, 0, 255] = float("nan")    # the last of group 0, and the first of group 1
    lut[G, 0, 255] = float("nan")
    lut[0, 1, 255] = -torch.tensor(float("nan")).half()
    codes[:, :, pos, 0] = 255
    codes[:, :, neg, 1] = 255
    q = torch.randn(1, Hkv * G, 1, D, generator=g).bfloat16().to(dev)
    kk = torch.randn(1, Hkv, T, D, generator=g).bfloat16().to(dev)
    odd = torch.zeros(1, Hkv, T, 33, dtype=torch.uint8, device=dev)
    odd[..., :32] = codes.to(dev)
    cfg = RetrievalConfig(topk=k, select=select, score_dtype=score_dtype)
    got = []
    for c in (codes.to(dev), odd[..., :32]):
        dec = SparseDecoder(gaussian_codebooks(3, D).to(dev), 1, Hkv * G, Hkv, D, T, cfg)
        dec.lut.copy_(lut)
        p = dec.plan(T, T)
        dec.last_k = p["k"]
        dec._decode_step(q[:, :, 0], c, kk, kk, T, T, p, None, 0, 0, 0)
        got.append(dec.selected()[0].cpu().numpy())
    assert np.array_equal(got[0], got[1])
    s = orc.score_grouped(lut.numpy().view(np.uint16), codes[0].numpy(), G)
    want = orc.topk(s, k, 1 if select == "head" else G, p["cand_start"], p["cand_end"],
                    key_bf16=score_dtype == torch.bfloat16)
    assert np.array_equal(got[0], want)
    if select == "group":
        assert np.isin(pos.numpy(), got[0][0]).all() and np.isin(pos.numpy(), got[0][1]).all()
