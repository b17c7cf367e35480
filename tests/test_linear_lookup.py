"""The specialised kernels' lookup tables as the library builds them (aw4_linear_tables), read the way the
kernels read them: entry = bits of the fp32 sum x + magic, less those of magic, plus the entry of 0; code or
level count = base + (x >= threshold).  Every x of [-1, 1] (or [0, 1]) must lie inside the table and the LDS
array, and give the exact count or code at and around every level, midpoint and bucket edge."""

from __future__ import annotations

import numpy as np
import pytest

from adamw4bit_amd import _lib
from adamw4bit_amd import quantization as q

F = np.float32


@pytest.fixture(scope="module")
def tables():
    return _lib.linear_tables()


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


def entry_of(table, x):
    return (x + table["magic"]).view(np.int32) - table["magic"].reshape(1).view(np.int32) + table["zero"]


def samples(cb, signed):
    lo = -1 if signed else 0
    mids = (cb[1:].astype(np.float64) + cb[:-1]) / 2
    edges = (np.arange(lo * 1024, 1024) + 0.5) / 1024  # every bucket edge of widths from 1/16 to 1/512, and between
    edges = np.concatenate([edges, *((np.arange(lo * n, n) + 0.5) / n for n in (16, 32, 64, 128, 256, 512))])
    x = np.unique(np.concatenate([around(cb), around(mids), around(edges, 2), around([0.0, 1.0, -1.0]),
                                  F([1e-45, 1e-38, 1e-20]), np.linspace(lo, 1, 200001, dtype=F)]))
    return x[(x <= 1) & (x >= lo)]


# (lookup-table id, codebook, what it gives): round-to-nearest per codebook, dyn4 with the zero floor, level counts
CASES = [(cb, cb, "nearest") for cb in range(5)] + [(5, q.CB_DYN4, "floored")] + [(6 + cb, cb, "levels") for cb in range(5)]


@pytest.mark.parametrize("lut,codebook,kind", CASES)
def test_table_gives_every_code_and_count(tables, lut, codebook, kind):
    cb = np.array(q.CODEBOOK_VALUES[codebook], dtype=F)
    signed = bool(cb[0] < 0)
    t = tables[lut]
    assert 0 < t["count"] <= _lib.LINEAR_SLOTS and (t["zero"] > 0) == signed and t["reserved"] == 0
    x = samples(cb, signed)
    entry = entry_of(t, x)
    assert entry.min() == 0 and entry.max() == t["count"] - 1  # inside the table, and every end of it reached
    assert (np.diff(entry) >= 0).all()
    e = t["entries"][entry]
    got = e["base"].astype(np.int64) + (x >= e["threshold"])
    want = count_less(cb, x) if kind == "levels" else nearest(cb, x, kind == "floored")
    wrong = np.flatnonzero(got != want)
    assert not len(wrong), (x[wrong[:5]], got[wrong[:5]], want[wrong[:5]])


def test_entries_keep_their_indexes_in_range(tables):
    """Whatever x: base + 1 within the codes or level counts where a threshold can be reached, and the entries
    behind the last one used are never read as codes beyond them either."""
    for lut in range(_lib.NUM_LUTS):
        t = tables[lut]
        e = t["entries"]
        top = 16 if lut >= 6 else 15
        assert (e["base"].astype(np.int64) + np.isfinite(e["threshold"]) * (e["threshold"] <= 1)).max() <= top, lut


def test_second_moments_lie_in_every_table(tables):
    """Second moments are looked up by |x|, in tables of either kind."""
    for lut in range(_lib.NUM_LUTS):
        t = tables[lut]
        x = samples(np.array(q.CODEBOOK_VALUES[q.CB_DYN4], dtype=F), False)
        entry = entry_of(t, x)
        assert entry.min() == t["zero"] and entry.max() == t["count"] - 1


@pytest.mark.parametrize("field,change", [("magic", 2.0), ("zero", 1), ("count", -1), ("threshold", None)])
def test_planted_fault_is_found(tables, field, change):
    """The check above fails on a table with one field off (planted in a copy)."""
    wrong = tables.copy()
    t = wrong[6 + q.CB_NF4]
    if field == "threshold":
        k = int(np.flatnonzero(np.isfinite(t["entries"]["threshold"][:t["count"]]))[3])
        t["entries"]["threshold"][k] = np.nextafter(t["entries"]["threshold"][k], F(4))
    elif field == "magic":
        t["magic"] *= F(change)
    else:
        t[field] += change
    with pytest.raises((AssertionError, IndexError)):
        test_table_gives_every_code_and_count(wrong, 6 + q.CB_NF4, q.CB_NF4, "levels")
