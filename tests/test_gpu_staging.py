"""The staging buffers of a step's launch table and of the gradient-norm pass: their first use on a device
waits for none of the work queued before it, and the norm pass's counters are right from the first pass on,
whatever used the buffer before."""

from __future__ import annotations

import ctypes
import os
import shutil
import tempfile

import numpy as np
import pytest
import torch

import adamw4bit_amd as aw
from adamw4bit_amd import _lib
from tests import gpu_helpers as H

pytestmark = pytest.mark.gpu


@pytest.fixture
def fresh_library():
    """A copy of the library with no buffers yet (the session's own has grown them in earlier tests)."""
    with tempfile.TemporaryDirectory() as tmp:
        path = shutil.copy(_lib.LIBRARY, os.path.join(tmp, "libfresh.so"))
        lib = ctypes.CDLL(path)
    for name, (restype, argtypes) in _lib.SIGNATURES.items():
        fn = getattr(lib, name)
        fn.restype, fn.argtypes = restype, argtypes
    yield lib
    torch.cuda.synchronize()


def step_table(count, numel=4096):
    """The launch table of a ZE-EDEN step over `count` tensors, its optimizer and the tables of other lengths."""
    gen = torch.Generator().manual_seed(count)
    params = [torch.nn.Parameter((torch.randn(numel, generator=gen) * 0.02).to(H.DEVICE)) for _ in range(count)]
    for p in params:
        p.grad = (torch.randn(numel, generator=gen) * 1e-3).to(H.DEVICE)
    opt = aw.ZEEDENAdamW4Bit(params, optimized=True)
    captured = []
    regular = _lib.fused_step
    _lib.fused_step = lambda t, st: (captured.append(np.array(t)), regular(t, st))
    try:
        opt.step()
    finally:
        _lib.fused_step = regular
    return opt, params, captured[-1]


def queue_work():
    """An event behind some tens of milliseconds of queued products."""
    a = torch.ones(8192, 8192, device=H.DEVICE, dtype=torch.bfloat16)
    b = torch.empty_like(a)
    for _ in range(60):
        torch.mm(a, a, out=b)
    event = torch.cuda.Event()
    event.record()
    return event, (a, b)


@pytest.mark.parametrize("call", ["step", "clip"])
def test_first_use_of_the_buffers_does_not_wait_for_queued_work(fresh_library, call):
    print(f"staging: first {call} behind queued work", flush=True)
    lib = fresh_library
    opt, params, table = step_table(40)
    stream = torch.cuda.current_stream().cuda_stream
    out = torch.zeros(4, device=H.DEVICE)
    one = np.array(table[:1])
    assert lib.aw4_fused_step(one.ctypes.data, 1, stream) == 0  # the device's first call: the codebook tables
    torch.cuda.synchronize()

    def run(rows):
        if call == "step":
            return lib.aw4_fused_step(rows.ctypes.data, len(rows), stream)
        q = out.data_ptr()
        return lib.aw4_clip_coefficient(rows.ctypes.data, len(rows), 1.0, q, q + 12, stream)

    queue_work()[0].synchronize()  # the product's own first call
    for k in range(4):  # every buffer
        event, keep = queue_work()
        assert run(table) == 0
        assert not event.query(), f"buffer {k}: the host waited for the queued work"
        event.synchronize()
    torch.cuda.synchronize()


def test_norm_counters_of_buffers_that_steps_used_first(fresh_library):
    """Every buffer stages a step first; then norm passes of few and of many segments, each through every
    buffer, so that counters are made, grown and used again."""
    print("staging: norm passes after steps", flush=True)
    lib = fresh_library
    opt, params, table = step_table(40)
    stream = torch.cuda.current_stream().cuda_stream
    for _ in range(4):
        assert lib.aw4_fused_step(table.ctypes.data, len(table), stream) == 0
    for sizes in ([5], [8192 * 40 + 3] * 3 + [7] * 200, [8192 * 70 - 3], [11] * 3000, [5]):
        grads = [torch.full((n,), 2.0, device=H.DEVICE) for n in sizes]
        rows = np.zeros(len(sizes), dtype=_lib.TENSOR)
        rows["grad"], rows["numel"], rows["grad_dtype"] = [g.data_ptr() for g in grads], sizes, _lib.F32
        per = [torch.tensor(float(n) * 4.0, dtype=torch.float64).sqrt().float().double() for n in sizes]
        want = torch.stack(per).square().sum().sqrt().float()
        for k in range(9):
            out = torch.zeros(4, device=H.DEVICE)
            q = out.data_ptr()
            assert lib.aw4_clip_coefficient(rows.ctypes.data, len(rows), 1.0, q, q + 12, stream) == 0
            assert float(out[0]) == float(want), (len(sizes), k, float(out[0]), float(want))
