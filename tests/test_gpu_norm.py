"""The gradient-norm pass and the clip's host side: many gradients, gradients of many segments, values that are
not finite, the fused unscaling, and a clip table reused while gradients move, change or come and go."""

from __future__ import annotations

import math

import numpy as np
import pytest
import torch

import adamw4bit_amd as aw
from adamw4bit_amd import _lib
from tests import gpu_helpers as H

pytestmark = pytest.mark.gpu

CODES = {torch.float32: _lib.F32, torch.bfloat16: _lib.BF16, torch.float16: _lib.F16}


def norm_pass(grads, max_norm=1.0, inv_scale=None):
    """(norm, coefficient, found_inf) of the library's pass over `grads`, as floats."""
    rows = np.zeros(len(grads), dtype=_lib.TENSOR)
    rows["grad"] = [g.data_ptr() for g in grads]
    rows["numel"] = [g.numel() for g in grads]
    rows["grad_dtype"] = [CODES[g.dtype] for g in grads]
    rows["flags"] = [_lib.TENSOR_VEC_ALIGNED if g.data_ptr() % (4 * g.element_size()) == 0 else 0 for g in grads]
    out = torch.full((4,), 7.0, device=H.DEVICE)
    q, stream = out.data_ptr(), torch.cuda.current_stream().cuda_stream
    if inv_scale is None:
        _lib.clip_coefficient(rows, max_norm, q, q + 4, stream)
    else:
        out[3] = inv_scale
        _lib.unscale_clip_coefficient(rows, q + 12, max_norm, q, q + 4, q + 8, stream)
    return out[:3].tolist()


def norm_of(grads, dtype):
    """The norm of the gradients' norms, each rounded to its dtype (the pass adds up in float64; so does this)."""
    per = torch.stack([g.double().square().sum().sqrt().float().to(dtype) for g in grads])
    return float(per.double().square().sum().sqrt().float().to(dtype))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("count,numel", [(31, 1000), (33, 8195), (255, 1000), (256, 9000), (257, 1000), (1000, 129), (5000, 96)])
def test_many_gradients(count, numel, dtype):
    """Fewer and more gradients than the pass counts in one level, of one segment and of several, twice."""
    gen = torch.Generator(device=H.DEVICE).manual_seed(count)
    stride = -(-numel // 8) * 8
    flat = (torch.randn(count, stride, generator=gen, device=H.DEVICE) * 0.1).to(dtype)
    grads = [flat[i, :numel] for i in range(count)]
    want = norm_of(grads, dtype)
    for k in range(6):
        got = norm_pass(grads)
        assert got[0] == want, (count, numel, k, got, want)
        assert norm_pass(grads, inv_scale=1.0)[0::2] == [want, 0.0]


def test_many_gradients_do_not_draw_one_after_another():
    """20,000 gradients of 64 values: atomics on one address follow one another at 13-14 ns, 275 us for as many
    gradients; counted in runs the pass took 84 us.  The bound is 8 ns a gradient."""
    count = 20000
    flat = torch.randn(count, 64, device=H.DEVICE)
    rows = np.zeros(count, dtype=_lib.TENSOR)
    rows["grad"] = flat.data_ptr() + 256 * np.arange(count, dtype=np.uint64)
    rows["numel"], rows["flags"] = 64, _lib.TENSOR_VEC_ALIGNED
    out = torch.zeros(4, device=H.DEVICE)
    q, stream = out.data_ptr(), torch.cuda.current_stream().cuda_stream
    times = []
    for _ in range(20):
        torch.cuda.synchronize()
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda._sleep(2_000_000)  # the host is ahead of the GPU: the events enclose the pass alone
        a.record()
        _lib.clip_coefficient(rows, 1.0, q, q + 4, stream)
        b.record()
        torch.cuda.synchronize()
        times.append(a.elapsed_time(b) * 1e3)
    print(f"norm pass of {count} gradients: {min(times):.1f} us", flush=True)
    assert min(times) < 8e-3 * count, times


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_loads_through_and_past_the_caches(dtype):
    """160 * 2^20 values, the most that are read through the caches, and one more; the gradients one value off
    their alignment too.  Against the sums of 2^20 values each, added in float64."""
    most = 160 << 20
    gen = torch.Generator(device=H.DEVICE).manual_seed(9)
    flat = torch.empty(most + 8, device=H.DEVICE, dtype=dtype).normal_(generator=gen)
    for sizes, shift in (((most - 3, 3), 0), ((most - 3, 4), 0), ((most, 1), 1)):
        a = flat[shift:shift + sizes[0]]
        grads = [a, flat[most + 4 - sizes[1]:most + 4]]
        sq = math.fsum(float(c.double().square().sum()) for c in a.split(1 << 20))
        per = [torch.tensor(math.sqrt(sq), dtype=torch.float64).float().to(dtype).double(),
               grads[1].double().square().sum().sqrt().float().to(dtype).double().cpu()]
        want = float(torch.stack(per).square().sum().sqrt().float().to(dtype))
        for _ in range(2):
            # the order of the float64 sums differs: a relative 2^-40 at most, one rounding of the norm where it is a tie
            got = norm_pass(grads)[0]
            assert abs(got - want) <= H.ULP16.get(dtype, 2.0 ** -23) * want, (sizes, got, want)


@pytest.mark.parametrize("bad", [math.inf, -math.inf, math.nan])
@pytest.mark.parametrize("where", ["first segment", "inside", "last segment of a cut gradient", "second gradient"])
def test_unscaling_finds_values_that_are_not_finite(where, bad):
    """2,048 segments of one gradient and 41 of a cut one, so that the flags are read eight at a time and singly
    and published through counters of two levels; then the same gradients without the value."""
    sizes = (1 << 24, 8192 * 40 + 5)
    gen = torch.Generator(device=H.DEVICE).manual_seed(3)
    grads = [torch.randn(n, generator=gen, device=H.DEVICE) * 256.0 for n in sizes]
    t, i = {"first segment": (0, 0), "inside": (0, 8192 * 500 + 17), "last segment of a cut gradient": (1, sizes[1] - 1),
            "second gradient": (1, 8192 * 3 + 1)}[where]
    want = norm_of([g / 256.0 for g in grads], torch.float32)
    for _ in range(5):  # every staging buffer, and the first one again
        kept = float(grads[t][i])
        grads[t][i] = bad
        norm, coef, found = norm_pass(grads, max_norm=2.0, inv_scale=1 / 256)
        assert found == 1.0 and (math.isnan(norm) and math.isnan(coef) if math.isnan(bad) else norm == math.inf and coef == 0.0)
        assert norm_pass(grads)[0] == math.inf or math.isnan(bad)
        grads[t][i] = kept
        norm, coef, found = norm_pass(grads, max_norm=2.0, inv_scale=1 / 256)
        assert found == 0.0 and norm == want and 0.0 < coef < 1.0


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("value", [math.inf, math.nan, 0.0, "overflow"])
def test_clip_returns_torchs_norm_of_special_values(value, dtype):
    """Infinite, NaN and zero gradients, and a norm beyond the dtype: norm and coefficient as torch's clip has them."""
    grads = [torch.ones(300, device=H.DEVICE, dtype=dtype), torch.zeros(5000, device=H.DEVICE, dtype=dtype)]
    if value == "overflow":
        grads = [torch.full((4096,), torch.finfo(dtype).max / 2, device=H.DEVICE, dtype=dtype)]
    elif value == 0.0:
        grads[0].zero_()
    else:
        grads[1][4321] = value
    params = [torch.nn.Parameter(torch.zeros_like(g)) for g in grads]
    for p, g in zip(params, grads):
        p.grad = g
    opt = aw.ZEEDENAdamW4Bit(params, optimized=True)
    total = opt.clip_grad_norm_(1.0)
    coef = opt._grad_clip[1][1].to(dtype)
    opt.zero_grad()
    per = torch.stack([g.double().square().sum().sqrt().float().to(dtype) for g in grads])
    want = per.double().square().sum().sqrt().float().to(dtype)
    assert total.dtype == dtype and total.shape == ()
    assert torch.equal(total, want) or (bool(total.isnan()) and bool(want.isnan()))
    want_coef = torch.clamp(1.0 / (want.cpu() + 1e-6), max=1.0)
    assert torch.equal(coef.cpu(), want_coef) or (bool(coef.isnan()) and bool(want_coef.isnan()))
    for p, g in zip(params, grads):
        p.grad = g
    if value in (math.inf, math.nan, "overflow") and not bool(want.isfinite()):
        with pytest.raises(RuntimeError, match="non-finite"):
            opt.clip_grad_norm_(1.0, error_if_nonfinite=True)


@pytest.mark.parametrize("count", [3, 20])
def test_reused_clip_table_follows_the_gradients(count):
    """Clip and step with the tables kept between calls against an optimizer that makes them anew each time:
    gradients at the same addresses, moved, off their alignment, strided, missing, back again, and parameters of
    another dtype."""
    gen = torch.Generator().manual_seed(count)
    sizes = [((64, 128), (1000,), (33, 7), (4097,))[i % 4] for i in range(count)]
    pairs = []
    for _ in range(2):
        g0 = torch.Generator().manual_seed(1)
        params = [torch.nn.Parameter((torch.randn(s, generator=g0) * 0.02).to(H.DEVICE)) for s in sizes]
        pairs.append((params, aw.ZIPSRAdamW4Bit(params, optimized=True, quant_rng_seed=5)))

    def aligned(s, dtype):
        return torch.randn(s, generator=gen).to(dtype).to(H.DEVICE)

    def shifted(s, dtype):
        n = math.prod(s)
        return torch.randn(n + 1, generator=gen).to(dtype).to(H.DEVICE)[1:].view(s)

    def strided(s, dtype):
        return torch.randn(s + (2,), generator=gen).to(dtype).to(H.DEVICE)[..., 0]

    reused = 0
    kinds = ["aligned", "same", "same", "aligned", "shifted", "shifted", "same", "missing", "same", "aligned", "strided",
             "aligned", "same", "bf16", "same", "aligned", "shifted"]
    for k, kind in enumerate(kinds):
        if kind == "bf16":
            for params, _ in pairs:
                for p in params[::2]:
                    p.grad = None
                    p.data = p.data.to(torch.bfloat16)
        if kind != "same":
            make = {"shifted": shifted, "strided": strided}.get(kind, aligned)
            for i, (a, b) in enumerate(zip(pairs[0][0], pairs[1][0])):
                g = None if kind == "missing" and i == 1 else make(sizes[i], a.dtype)
                a.grad, b.grad = g, g
        (pa, oa), (pb, ob) = pairs
        before = oa._clip_plan
        ob._clip_plan = ob._launch_plan = None
        na, nb = oa.clip_grad_norm_(1.0), ob.clip_grad_norm_(1.0)
        reused += int(before is not None and oa._clip_plan is before)
        assert na.dtype == nb.dtype and torch.equal(na, nb), (k, kind)
        assert float(oa._grad_clip[1][1]) == float(ob._grad_clip[1][1]), (k, kind)
        oa.step()
        ob.step()
        for i, (a, b) in enumerate(zip(pa, pb)):
            assert torch.equal(H.bits(a), H.bits(b)), (k, kind, i)
            sa, sb = H.state_of(oa, a), H.state_of(ob, b)
            assert sa["step"] == sb["step"] and all(torch.equal(H.bits(sa[x]), H.bits(sb[x])) for x in sa if x != "step")
    assert reused == 11, reused  # every pass but the first, those around a missing or strided gradient and the cast
