"""CPU check of the encoder's ranking bound: wherever the best approximate
similarity (two fp16 terms per codebook row, fp32 keys as two fp16 terms, fp32
sums, the code in the low six bits) leads the second by more than kGapSlack
times the key's norm, the exactly scored maximum is the same code.

The arithmetic of csrc/sphkv_encode.hip is restated in numpy; the slack itself
is read from that file.
"""
import os
import re

import numpy as np
import pytest

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "spherical-kv_amd", "csrc", "sphkv_encode.hip")
F = np.float32


def _constant(name):
    return float(re.search(rf"constexpr float {name} = ([0-9.e-]+)f;", open(SRC).read()).group(1))


def _rtz16(x):
    """fp32 -> fp16, rounded towards zero."""
    h = np.asarray(x, F).astype(np.float16)
    over = np.abs(h.astype(F)) > np.abs(np.asarray(x, F))
    return np.where(over, np.nextafter(h, np.float16(0)), h)


def _split(x):
    hi = _rtz16(x)
    return hi.astype(F), _rtz16(np.asarray(x, F) - hi.astype(F)).astype(F)


def _ranked(x, cb, fp32):
    """Approximate similarities [n, C] with the code in their low six bits, and
    the unit (norm) that the slack is taken in."""
    r = np.sqrt((x.astype(np.float64) ** 2).sum(-1)).astype(F)
    chi, clo = _split(cb)
    if fp32:
        xh, xl = _split(x * (F(256) / r)[:, None])
        terms, unit = [(chi, xh), (clo, xh), (chi, xl)], np.full(len(x), 256, F)
    else:
        terms, unit = [(chi, x.astype(F)), (clo, x.astype(F))], r
    s = np.zeros((len(x), len(cb)), F)
    for c, k in terms:
        for i in range(cb.shape[1]):
            s = (s + c[None, :, i] * k[:, None, i]).astype(F)
    code = np.arange(len(cb), dtype=np.uint32)
    bits = (s.view(np.uint32) & ~np.uint32(63)) | (16 * (code // 16) + code % 16)
    return bits.view(F), unit


def _exact(x, cb, fp32):
    den = np.sqrt((x.astype(np.float64) ** 2).sum(-1)).astype(F) + F(1e-8)
    d = (x.astype(F) / den[:, None]).astype(F)
    s = np.zeros((len(x), len(cb)), np.float64)
    for i in range(cb.shape[1]):                       # an fma chain: one rounding per step
        s = (s + d[:, None, i].astype(np.float64) * cb[None, :, i].astype(np.float64)).astype(F).astype(np.float64)
    return s


def test_slack_covers_both_similarities_errors():
    # twice the largest distance between an approximate similarity and norm x
    # exact one, with a fifth to spare
    c = (1 + _constant("kUnitTol")) ** 0.5             # longest row that is ranked
    for g, products in ((16, 16), (32, 32)):
        row = 2.0 ** -20 + 2.0 ** -24 * g ** 0.5       # two fp16 terms (the second may be denormal)
        key = 2.0 ** -19                               # fp32 keys' two terms, without low x low
        sums = 3 * products * 2.0 ** -24               # three products per dimension
        code = 63 * 2.0 ** -23                         # at the bottom of a binade
        chain = (products + 2) * 2.0 ** -24            # the exact chain and its directions
        eps = c * (row + key + sums + code + chain)
        assert 2 * eps <= 0.8 * _constant("kGapSlack"), (g, eps)


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("g,C", [(16, 64), (32, 8)])
def test_ranking_stands_past_the_slack(g, C, fp32):
    # the first and the last code as the two best, their gap around the slack,
    # rows as long as are ranked, best similarities just above a power of two
    rng, slack = np.random.default_rng(g + fp32), _constant("kGapSlack")
    n, kept, worst = 400, 0, 0.0
    for _ in range(40):
        cb = rng.standard_normal((C, g)).astype(F)
        cb *= (np.sqrt(1 + 0.099 * rng.choice([-1, 1, 1], C)) / np.linalg.norm(cb, axis=1)).astype(F)[:, None]
        a, b = (0, C - 1) if rng.random() < 0.5 else (C - 1, 0)
        v = rng.standard_normal(g)
        v -= cb[a] * (v @ cb[a]) / (cb[a] @ cb[a])
        cb[a] *= F(1.048 / np.linalg.norm(cb[a]))
        cb[b] = cb[a] + (1e-3 * v).astype(F)
        x = cb[a].astype(np.float64)[None] * np.exp2(rng.integers(-6, 6, n))[:, None]
        x = x / np.linalg.norm(cb[a]) ** 2 * (1 + 10.0 ** rng.uniform(-7, -3, n))[:, None]      # <x, c_a> just above 2^k
        x += (rng.uniform(-1, 1, n) * 0.2 * np.linalg.norm(x, axis=1))[:, None] * (v / np.linalg.norm(v))
        x = x.astype(F if fp32 else np.float16)
        top, unit = _ranked(x, cb, fp32)
        order = np.sort(top, axis=1)
        clear = order[:, -1] - order[:, -2] > F(slack) * unit
        s = _exact(x, cb, fp32)
        worst = max(worst, np.abs(top.astype(np.float64) / unit[:, None] - s).max())
        kept += int(clear.sum())
        assert (top.argmax(1) == s.argmax(1))[clear].all()
    assert kept > 1000 and 2 * worst <= slack


@pytest.mark.parametrize("g", [16, 32])
def test_ranked_fp32_keys_have_the_length_that_the_slack_is_taken_in(g):
    # the fp32 norm in the kernel's order (8 chains of fused multiply-adds, a
    # float64 product and sum rounded once), from keys whose squares underflow
    rng, least = np.random.default_rng(g), _constant("kMinNorm")
    x = rng.standard_normal((20000, g))
    x = (x / np.linalg.norm(x, axis=1, keepdims=True) * 10.0 ** rng.uniform(-23.5, -15, (20000, 1))).astype(F)
    acc = np.zeros((len(x), 8), F)
    for d in range(0, g, 8):
        acc = (x[:, d:d + 8].astype(np.float64) ** 2 + acc).astype(F)
    s = acc[:, 0]
    for lane in range(1, 8):
        s = s + acc[:, lane]
    r, true = np.sqrt(s), np.linalg.norm(x.astype(np.float64), axis=1)
    ranked = (r > 0) & (r >= F(least))
    off = np.abs(true[ranked] / r[ranked] - 1)
    assert ranked.sum() > 1000 and off.max() < 1e-6
    assert np.abs(true[r > 0] / r[r > 0] - 1).max() > 0.5          # what the limit keeps out
