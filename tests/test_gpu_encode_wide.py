"""Every encode kernel, forced at the sizes where it can go wrong: codes and residual
norms equal the oracle's bit for bit.  At head dims 64 and 128 the wide kernel (256
rows per workgroup) and the split kernel (16 or 32 rows), at 64 also the exact one
(one row); at 256 the bf16 MFMA kernel (16 rows), or, for entry counts that are no
multiple of 16, the VALU kernel.

A coarse search may only rule entries out, so every case whose magnitudes leave
its range (rows past 2^15, non-finite rows, codebook norms that are zero, tiny,
past 2^12 or not finite) has to fall back to the contract's distances and give the
same codes.
"""
import numpy as np
import pytest
import torch

from _forms import encode_forms
from _synth import gen, residual_codebooks

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K(dev):
    from laprune_amd import aq_kernels
    return aq_kernels


def _check(K, orc, dev, x, cb, what):
    print(what, flush=True)
    codes, rn = K.aq_encode_greedy(x.to(dev), cb.to(dev))
    torch.cuda.synchronize()
    want_c, want_r = orc.encode(x.numpy(), cb.numpy())
    assert np.array_equal(codes.cpu().numpy(), want_c), what
    got = rn.cpu().numpy()
    assert np.array_equal(got, want_r, equal_nan=True), what


@encode_forms(64, 128, 256)
@pytest.mark.parametrize("N", [1, 15, 17, 32, 33, 255, 256, 257, 513])
def test_row_edges(dev, K, orc, form, N):
    D = form
    x = torch.randn(N, D, generator=gen(N)) * 3
    _check(K, orc, dev, x, residual_codebooks(7, D), f"N={N} D={D}")


@encode_forms(64, 128, 256)
@pytest.mark.parametrize("Kc,M", [(4, 3), (16, 8), (32, 2), (48, 65), (60, 5), (64, 1), (100, 33),
                                  (224, 2), (240, 40), (252, 66), (256, 70)])
def test_entry_and_stage_edges(dev, K, orc, form, Kc, M):
    D = form
    x = torch.randn(70, D, generator=gen(Kc)) * 3
    _check(K, orc, dev, x, residual_codebooks(3, D, M, Kc), f"K={Kc} M={M} D={D}")


@encode_forms(128, 256)
@pytest.mark.parametrize("scale", [1e-30, 1e-6, 2e-3, 40.0, 900.0, 4e5, 1e20])
def test_scales(dev, K, orc, form, scale):
    """Rows and codebooks alike, each alone, and far from each other."""
    x = torch.randn(64, form, generator=gen(1))
    cb = residual_codebooks(5, form)[:4]
    _check(K, orc, dev, x * scale, cb * scale, f"both x {scale}")
    _check(K, orc, dev, x * scale, cb, f"rows x {scale}")
    _check(K, orc, dev, x, cb * scale, f"codebooks x {scale}")


@encode_forms(64, 128, 256)
@pytest.mark.parametrize("Kc", [256, 60])
def test_out_of_range_rows_and_stages(dev, K, orc, form, Kc):
    x = torch.randn(96, form, generator=gen(2)) * 3
    x[3] = 0
    x[17, 5] = float("nan")
    x[33, 0] = float("inf")
    x[34, form - 1] = -float("inf")
    x[50] *= 1e4
    x[95] = 1e19  # its squared norm overflows
    cb = residual_codebooks(11, form)[:6, :Kc].clone()
    _check(K, orc, dev, x, cb, "rows")
    cb[1, 40] = float("nan")
    cb[2, 3, 7] = float("inf")
    cb[3] = 0
    cb[4, Kc - 56] *= 1e6
    _check(K, orc, dev, x, cb, "rows and stages")


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("M", [1, 2, 3, 8])
@pytest.mark.parametrize("polls", [0, 1, 2])
def test_waits_that_give_up(dev, K, orc, monkeypatch, polls, M, D):
    """The wide kernel's waits end after a bounded number of polls.  With a
    bound that no stage's fragments can meet, or that some waves meet, the
    contract's distances decide and the codes stay the oracle's."""
    monkeypatch.setenv("LAPRUNE_ENCODE_TILE", "1")
    monkeypatch.setenv("LAPRUNE_ENCODE_EXACT", "0")
    monkeypatch.setenv("LAPRUNE_ENCODE_POLLS", str(polls))
    x = torch.randn(300, D, generator=gen(polls + M)) * 3
    _check(K, orc, dev, x, residual_codebooks(23, D, M), f"polls={polls} M={M} D={D}")


@encode_forms(64, 128, 256)
def test_ties(dev, K, orc, form):
    """Equal entries, across halves, tiles and pairs of tiles: the lowest wins."""
    cb = residual_codebooks(13, form)[:5].clone()
    for m, (a, b) in enumerate([(3, 4), (2, 37), (5, 64), (7, 255), (0, 128)]):
        cb[m, b] = cb[m, a]
    x = cb[0, torch.randint(0, 256, (80,), generator=gen(4))].clone()
    x += 0.05 * torch.randn(80, form, generator=gen(5))
    for m, a in enumerate([3, 2, 5, 7, 0]):
        x[m] = cb[:m, 9].sum(0) + cb[m, a]
    _check(K, orc, dev, x, cb, "ties")


@encode_forms(128, 256)
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("off", [0, 1])
def test_strided_keys(dev, K, orc, form, dt, off):
    """A token range of a [B, H, T, D] cache, its rows aligned or not, and
    code rows at an odd pitch."""
    from laprune_amd import _native as N
    B, H, T, D, t0, t1 = 2, 3, 60, form, 7, 58
    buf = torch.randn(B * H * T * (D + off) + off, generator=gen(6)).to(dt).to(dev)
    k = buf[off:].view(B, H, T, D + off)[..., :D]
    cb = residual_codebooks(17, D)[:9].contiguous().to(dev)
    prep = K.aq_encode_prepare(cb)
    codes = torch.full((B, H, T, 11), 99, dtype=torch.uint8, device=dev)
    N.call("lap_encode_keys", N.ptr(k), N.dtype_code(dt), k.stride(0), k.stride(1), k.stride(2),
           B, H, t0, t1, D, N.ptr(cb), 9, 256, N.ptr(prep), prep.numel(), N.ptr(codes),
           codes.stride(0), codes.stride(1), codes.stride(2), None, N.stream_of(k))
    torch.cuda.synchronize()
    rows = k[:, :, t0:t1].float().cpu().reshape(-1, D)
    want, _ = orc.encode(rows.numpy(), cb.cpu().numpy())
    got = codes.cpu()
    assert np.array_equal(got[:, :, t0:t1, :9].reshape(-1, 9).numpy(), want)
    got[:, :, t0:t1, :9] = 99
    assert bool((got == 99).all()), "codes written outside the range"


@encode_forms(64, 128, 256)
def test_device_ranges(dev, K, orc, form):
    """Per-sequence ranges read on the device: rows past a range are left alone."""
    from laprune_amd.cache import DecodeKVCache
    cb = residual_codebooks(19, form)[:8].contiguous().to(dev)
    c = DecodeKVCache(cb, 3, 4, form, 200, group_size=64)
    c.k.copy_(torch.randn(c.k.shape, generator=gen(8)))
    c.codes.fill_(77)
    ranges = [(0, 0), (100, 164), (5, 30)]
    c.encode_ranges(torch.tensor(ranges, dtype=torch.int32, device=dev))
    torch.cuda.synchronize()
    got = c.codes.cpu().numpy()
    for b, (lo, hi) in enumerate(ranges):
        want = np.full_like(got[b], 77)
        if hi > lo:
            w, _ = orc.encode(c.k[b, :, lo:hi].float().cpu().reshape(-1, form).numpy(),
                              cb.cpu().numpy())
            want[:, lo:hi] = w.reshape(4, hi - lo, 8)
        assert np.array_equal(got[b], want), b
