"""The specialised kernels' lookup tables, restated: bucket of x = the step of the grid that fp32
``x + magic`` rounds to, code or level count = base + (x >= thr).  Every bucket of [-1, 1] (or [0, 1])
must hold at most one change, lie inside the LDS array, and give the exact count or code at and around
every change and bucket edge."""

from __future__ import annotations

import numpy as np
import pytest

from adamw4bit_amd import quantization as q

SLOTS = 514
F = np.float32


def count_less(cb, x):
    return (cb[None, :] < x[:, None]).sum(1)


def nearest(cb, x, floor):
    i = count_less(cb, x)
    lo, hi = np.maximum(i - 1, 0), np.minimum(i, 15)
    code = np.where(np.abs(x - cb[lo]) < np.abs(cb[hi] - x), lo, hi)
    return np.maximum(code, 1) if floor else code


def around(values, ulps=6):
    out = []
    for v in values:
        a = b = F(v)
        out.append(a)
        for _ in range(ulps):
            a, b = np.nextafter(a, F(-4)), np.nextafter(b, F(4))
            out += [a, b]
    return np.array(out, dtype=F)


CASES = [(c, kind) for c in range(5) for kind in ("levels", "nearest")] + [(q.CB_DYN4, "floored")]


@pytest.mark.parametrize("codebook,kind", CASES)
def test_one_change_per_bucket(codebook, kind):
    cb = np.array(q.CODEBOOK_VALUES[codebook], dtype=F)
    signed = cb[0] < 0
    f = (lambda x: count_less(cb, x)) if kind == "levels" else (lambda x: nearest(cb, x, kind == "floored"))
    mids = (cb[1:].astype(np.float64) + cb[:-1]) / 2
    for inv in (16, 32, 64, 128, 256, 512):
        magic = F(1.5 * 2 ** 23 / inv)
        zero = inv if signed else 0
        slots = 2 * inv + 1 if signed else inv + 1
        if slots > SLOTS:
            pytest.fail("no bucket width holds one change each")
        edges = (np.arange(-inv if signed else 0, inv) + 0.5) / inv
        x = np.unique(np.concatenate([around(cb), around(mids), around(edges), around([0.0, 1.0]),
                                      np.linspace(-1 if signed else 0, 1, 20001, dtype=F)]))
        x = x[(x <= 1) & (x >= (-1 if signed else 0))]
        bucket = (x + magic).view(np.int32) - magic.view(np.int32) + zero
        assert bucket.min() == 0 and bucket.max() == slots - 1  # inside the table
        value = f(x)
        assert (np.diff(bucket) >= 0).all() and (np.diff(value) >= 0).all()
        base = np.array([value[bucket == b].min() for b in range(slots)])
        top = np.array([value[bucket == b].max() for b in range(slots)])
        if (top - base <= 1).all():
            break
    # threshold: the first sampled x of the bucket with the higher value (the samples hold every change's
    # two neighbours, so it is the first float too)
    thr = np.array([x[(bucket == b) & (value == base[b] + 1)].min() if top[b] > base[b] else np.nan for b in range(slots)])
    assert np.array_equal(base[bucket] + (x >= thr[bucket]), value)
