"""The encode's coarse searches, restated on the CPU (test only).

At head dim 256 the GPU encode (csrc/encode.hip) prunes each stage's candidates
with bf16 MFMA distances G_k = (rn + cn_k) - 2 bf16(r).bf16(C_k) and a proven
error bound eps_k; entry k survives unless G_k - eps_k > min_j (G_j + eps_j),
and only survivors get the exact fp32 recheck.  Along the oracle's own
encode trajectory this test recomputes the shortlist in float64 with the
kernel's eps formula, checks that the exact argmin (the oracle's code)
always survives, and reports survivors per row and stage for N(0, 0.02)
codebooks and for residual-ordered ones of trained magnitude.

At head dims 64 and 128 (csrc/encode_wide.h) scores of fp16 rows against scaled
fp16 entries rule out what lies 2 eps below the row's best.  Restated with every
subnormal fp16 input flushed, the scores stay within eps of the unrounded ones and
the oracle's code survives, over rows and codebooks of all magnitudes.
"""
import math

import numpy as np
import pytest

from oracle import orc

from _synth import c3_keys, gaussian_codebooks, residual_codebooks


def _bf16(a):
    b = np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)
    b = (b + 0x7FFF + ((b >> 16) & 1)) & 0xFFFF0000  # round to nearest even
    return b.view(np.float32).astype(np.float64)


def _shortlist_sizes(x, cb):
    codes, _ = orc.encode(x, cb)
    r = x.astype(np.float32).copy()
    n, M = codes.shape
    sizes = np.zeros((n, M), np.int64)
    cn = (cb.astype(np.float64) ** 2).sum(-1)  # [M, K]
    for m in range(M):
        rn = (r.astype(np.float64) ** 2).sum(-1)[:, None]
        dm = _bf16(r) @ _bf16(cb[m]).T
        A = rn + cn[m][None, :]
        G = A - 2 * dm
        eps = (1.0078125 * 2.0 ** -6 * np.sqrt(rn) * np.sqrt(cn[m])[None, :]
               + 2.0 ** -21 * (np.abs(A) + 2 * np.abs(dm))
               + 2.0 ** -116 * (1 + np.sqrt(rn) + np.sqrt(cn[m])[None, :]))
        U = (G + eps).min(axis=1, keepdims=True)
        keep = ~(G - eps > U)
        assert keep[np.arange(n), codes[:, m]].all(), m  # the exact argmin survives
        sizes[:, m] = keep.sum(1)
        r = (r - cb[m][codes[:, m]]).astype(np.float32)
    return sizes


@pytest.mark.parametrize("kind", ["gaussian", "residual"])
def test_encode_shortlist_c3(kind):
    x = c3_keys(60).numpy()
    cb = (gaussian_codebooks(61) if kind == "gaussian" else residual_codebooks(61)).numpy()
    s = _shortlist_sizes(x, cb)
    assert s.min() >= 1
    first, last = s[:, 0].mean(), s[:, -1].mean()
    print(f"{kind}: survivors per row and stage mean {s.mean():.2f}, p99 "
          f"{np.percentile(s, 99):.0f}, max {s.max()}; stage 0 {first:.2f}, stage 31 {last:.2f}")


def _f16_flushed(a):
    y = np.asarray(a, np.float32).astype(np.float16).astype(np.float64)
    return np.where(np.abs(y) < 2.0 ** -14, 0.0, y)


def _h_parts(h):
    """Sum of the three fp16 parts of h / 64, times 64, subnormal parts flushed."""
    x, total = (np.asarray(h, np.float64) / 64).astype(np.float32), 0.0
    for _ in range(3):
        part = x.astype(np.float16).astype(np.float32)
        total = total + _f16_flushed(part)
        x = x - part
    return 64 * total


def test_parts_of_the_norm():
    """What the three parts lose, flushes included, is what the bound allows them."""
    h = 2.0 ** np.random.default_rng(1).uniform(-40, 20, 200000)
    h = np.concatenate([h, 2.0 ** np.arange(-40, 21.0), 64 * 2.0 ** -14 - 2.0 ** np.arange(-30, -10.0)])
    h = h.astype(np.float32).astype(np.float64)
    lost = np.abs(_h_parts(h) - h)
    assert (lost <= np.minimum(h, 2.0 ** -8) * (1 + 2.0 ** -10) + 2.0 ** -19).all()
    assert lost.max() > 2.0 ** -9  # not covered by the other terms' 2^-18


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("rows", [1e-6, 2e-3, 1.0, 900.0])
@pytest.mark.parametrize("books", [1e-30, 1e-6, 2e-3, 1.0, 90.0])
def test_fp16_search_bound(D, rows, books):
    x = (c3_keys(62, n_tok=4, D=D) * rows).numpy()
    cb = (residual_codebooks(63, D)[:6] * books).numpy()
    codes, _ = orc.encode(x, cb)
    r = x.astype(np.float32).copy()
    for m in range(cb.shape[0]):
        c = cb[m].astype(np.float64)
        cn = (c ** 2).sum(-1).astype(np.float32).astype(np.float64)
        cmax = cn.max()
        b = 9 - math.frexp(math.sqrt(cmax))[1] + 1 if cmax > 0 else 0
        sc = 2.0 ** min(max(b, -20), 60)
        cq = _f16_flushed(c * sc)
        d_ = np.sqrt(((c * sc - cq) ** 2).sum(-1).max()) * 1.001
        cc, h = math.sqrt(cmax) * sc * 1.001, 0.5 * cmax * sc * 1.001
        e1 = 2.05 * (d_ + (2.0 ** -11 + 2.0 ** -15 + 2.0 ** -17) * (cc + d_))
        e0 = 2.05 * (math.sqrt(D) * 2.0 ** -14 * (1 + 2.0 ** -8) * (cc + d_) + 2.0 ** -15 * h +
                     2.0 ** -18 + 1.01 * min(h, 2.0 ** -8))
        rr = r.astype(np.float64)
        rn = (rr ** 2).sum(-1)
        eps2 = np.sqrt(rn) * e1 + e0 + rn * 2.05 * sc * 2.0 ** -22
        A = _f16_flushed(r) @ cq.T - _h_parts(0.5 * sc * cn)
        exact = rr @ (c * sc).T - 0.5 * sc * cn
        ok = (eps2 < 2.0 ** 60) & (rn < 2.0 ** 30)
        assert (np.abs(A - exact).max(1) <= eps2 / 2)[ok].all(), m
        keep = A >= A.max(1, keepdims=True) - eps2[:, None]
        assert keep[np.arange(len(r)), codes[:, m]][ok].all(), m
        r = (r - cb[m][codes[:, m]]).astype(np.float32)
