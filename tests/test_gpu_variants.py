"""Specialised kernels by dtype and scheme pair, at the sizes where a dispatch or a tile can go wrong:
whole tiles, a last tile of a few blocks, a single 4-bit tensor of the smallest size, fp32-state tensors
in the same launch, and launches of two to twelve tiles per wave.  Against the oracle, with the bars of
``test_gpu_step`` (codes, scales and fp32 state bit-exact; parameters within the bars of ``gpu_helpers``)."""

from __future__ import annotations

import pytest
import torch

import adamw4bit_amd as aw
from adamw4bit_amd import _lib
from adamw4bit_amd import quantization as q
from oracle import reference_step as ref
from tests import gpu_helpers as H
from tests.test_gpu_step import compare_pair, gpu_encode, log, moment_desc, run_pair, stream

pytestmark = pytest.mark.gpu

# 4 whole tiles, 1 block past a whole tile, 1 block short of one, many tiles (one per wave), fp32 state
SHAPES = [(4096,), (33, 128), (71, 128), (1056, 2048), (4097,), (129,), (3,)]


def fp16_safe(shape, gen):
    return H.heavy_tailed(shape, gen, row_mu=-5.0)


@pytest.mark.parametrize("m1,m2,eden", [("nf4", "dyn4_nz", True), ("nf4", "dyn4_upd_sr_fp32read", False),
                                        ("nf4_sr", "dyn4_upd_sr_fp32read", False)])
def test_fp16_recipe_kernels_match_oracle(m1, m2, eden):
    """fp16 parameters and gradients under the recipes' schemes."""
    log(f"fp16 {m1} / {m2} eden={eden} x 3 steps")
    make = lambda ps: aw.QuantizedAdamW(ps, lr=1e-3, weight_decay=0.1, m1_quant_scheme=m1, m2_quant_scheme=m2,  # noqa: E731
                                        use_eden_m2=eden, quant_rng_seed=3, optimized=True)
    out = run_pair(make, SHAPES, torch.float16, 3, seed=3, zero_block_frac=0.02, grad_fn=fp16_safe)
    compare_pair(*out, f"fp16 {m1}/{m2}", steps=3)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m1,m2", [("nf4", "dyn4_nz"), ("sdyn4", "lin4_nz"), ("nf4", "dyn4")])
def test_round_to_nearest_pairs_match_oracle(m1, m2, dtype):
    """Round-to-nearest first and second moments without EDEN: the optimized step's pairs of them."""
    log(f"round-to-nearest {m1} / {m2} {dtype} x 3 steps")
    make = lambda ps: aw.QuantizedAdamW(ps, lr=1e-3, weight_decay=0.1, m1_quant_scheme=m1, m2_quant_scheme=m2,  # noqa: E731
                                        optimized=True)
    out = run_pair(make, SHAPES, dtype, 3, seed=None, zero_block_frac=0.02, grad_fn=fp16_safe)
    compare_pair(*out, f"{m1}/{m2} {dtype}", steps=3)


@pytest.mark.parametrize("m2,eden", [("fp32", False), ("dyn4_upd_sr_fp32read", True)])
def test_fp16_ablations_match_oracle(m2, eden):
    """fp16 with an fp32 second moment, and with EDEN on the update-SR one."""
    log(f"fp16 nf4 / {m2} eden={eden} x 3 steps")
    make = lambda ps: aw.QuantizedAdamW(ps, lr=1e-3, weight_decay=0.1, m1_quant_scheme="nf4", m2_quant_scheme=m2,  # noqa: E731
                                        use_eden_m2=eden, quant_rng_seed=3, optimized=True)
    out = run_pair(make, SHAPES, torch.float16, 3, seed=3, zero_block_frac=0.02, grad_fn=fp16_safe)
    compare_pair(*out, f"fp16 nf4/{m2}", steps=3)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shapes", [[(1030, 1021), (1, 3), (1024,), (4,), (5,), (513, 2047)],  # a launch of their own
                                    [(1030, 1021), (64, 128), (1024,), (2049, 511)],             # beside a block launch
                                    [(3,), (1000,)]])                                           # few, and nothing else
@pytest.mark.parametrize("betas", [(0.9, 0.95), (0.4, 0.45)])
def test_fp32_state_launches_match_oracle(shapes, dtype, betas):
    """fp32-state tensors in launches of their own: whole and cut tiles, the last quad of 1 to 3 values,
    both lerp forms."""
    log(f"fp32-state launches {dtype} {betas} {shapes}")
    make = lambda ps: aw.ZIPSRAdamW4Bit(ps, lr=1e-3, betas=betas, weight_decay=0.1, quant_rng_seed=5, optimized=True)  # noqa: E731
    out = run_pair(make, shapes, dtype, 2, seed=5, grad_fn=fp16_safe)
    compare_pair(*out, f"fp32 state {dtype}", steps=2)


def test_fp32_state_launch_with_misaligned_and_clipped_gradients():
    """Gradients and parameters off a 16-byte boundary (single accesses), clipped in the same step, against
    aligned copies of them stepped the same way."""
    gen = torch.Generator().manual_seed(2)
    n = 1025 * 1023
    init, grad = torch.randn(n, generator=gen) * 0.02, torch.randn(n, generator=gen)
    got = []
    for shift in (0, 1):
        p = torch.nn.Parameter(torch.zeros(n + 4, device=H.DEVICE)[shift:shift + n].copy_(init))
        p.grad = torch.zeros(n + 4, device=H.DEVICE)[shift:shift + n].copy_(grad)
        assert (p.data_ptr() % 16 == 0) == (shift == 0)
        opt = aw.ZEEDENAdamW4Bit([p], optimized=True)
        for _ in range(2):
            opt.clip_grad_norm_(1.0)
            opt.step()
        got.append((p.detach().cpu(), opt.state[p]["m1"].cpu(), opt.state[p]["m2"].cpu()))
    for a, b in zip(*got):
        assert torch.equal(H.bits(a), H.bits(b))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_fp32_state_beside_a_large_block_launch(dtype):
    """A block launch of 32 tiles per CU and more, with fewer and more fp32-state tiles than the few that
    join it in grid order."""
    for extra in ([(4095,)], [(4095,)] * 5):
        log(f"fp32-state tiles beside 2048x4096 {dtype} {len(extra)}")
        make = lambda ps: aw.ZIPSRAdamW4Bit(ps, lr=1e-3, weight_decay=0.1, quant_rng_seed=5, optimized=True)  # noqa: E731
        out = run_pair(make, [(2048, 4096)] + extra, dtype, 2, seed=5)
        compare_pair(*out, f"fp32 state beside blocks {dtype}", steps=2)


@pytest.mark.parametrize("blocks", [1, 7, 8, 9, 33, 8 * 4 * 256 * 8 + 5])
@pytest.mark.parametrize("mode,eden", [("nf4", False), ("dyn4_nz", True), ("nf4_sr", False), ("dyn4_upd_sr_fp32read", False)])
def test_codec_sizes_match_oracle(mode, eden, blocks):
    """aw4_quantize and aw4_dequantize from one block to more tiles than a wave each: whole and cut tiles."""
    log(f"codec {mode} {blocks} blocks")
    gen = torch.Generator().manual_seed(blocks)
    values = H.heavy_tailed((blocks, 128), gen).reshape(-1)
    if mode.startswith("dyn4"):
        values = values.square()
    values[:128] = 0.0
    draws = torch.rand(blocks, 128, generator=gen) if "sr" in mode else None
    codes, scales = gpu_encode(values, mode, eden, True, draws)
    expect, expect_scales = ref.encode(values, mode, eden=eden, draws=draws, usr_sqrt="cr")
    assert torch.equal(q.unpack_4bit_codes(codes, numel=values.numel()), expect)
    assert torch.equal(H.bits(scales), H.bits(expect_scales))
    packed, sc = codes.to(H.DEVICE), scales.to(H.DEVICE)
    out = torch.full((values.numel() + 64,), 7.0, device=H.DEVICE)
    _lib.dequantize(moment_desc(mode, eden, True, packed, sc), values.numel(), out.data_ptr(), stream())
    torch.cuda.synchronize()
    levels = q.codebook_tensor(mode)
    assert torch.equal(H.bits(out[:values.numel()]), H.bits(levels[expect.long()] * expect_scales.repeat_interleave(128)))
    assert bool((out[values.numel():] == 7.0).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("sizes", [[1], [3], [8191, 8193, 5], [4096 * 4096], [1 << 18] * 9 + [1000001],
                                   [257 * (i % 7 + 1) for i in range(156)],   # the most rows launch arguments hold
                                   [257 * (i % 7 + 1) for i in range(157)],   # one more: a staged table
                                   [40_000_003, 11, 30_000_000],
                                   # runs of 32 segments: more and fewer than one, parts of one at both ends
                                   [8192 * 33, 5, 8192 * 40 + 1, 8192 * 32, 8192 * 70 - 3]])
def test_clip_norm_sizes(sizes, dtype):
    """The norm pass over segments of 2^13 to 2^15 values, cut ones, many gradients and one; twice, since
    its counters must be zero again.  The same gradients one value off their alignment, too."""
    gen = torch.Generator(device=H.DEVICE).manual_seed(len(sizes))
    for shift in (0, 1):
        params = []
        for n in sizes:
            p = torch.nn.Parameter(torch.zeros(n, device=H.DEVICE, dtype=dtype))
            p.grad = torch.randn(n + 4, generator=gen, device=H.DEVICE).to(dtype)[shift:shift + n]
            params.append(p)
        opt = aw.ZEEDENAdamW4Bit(params, optimized=True)
        per = [p.grad.double().square().sum().sqrt().float().to(dtype) for p in params]
        want = torch.stack([x.double() for x in per]).square().sum().sqrt().float().to(dtype)
        for _ in range(6):  # every staging slot, and the first one again
            norm = opt.clip_grad_norm_(1.0)
            opt._grad_clip = None  # no step: drop the pending clip
            torch.cuda.synchronize()
            assert torch.equal(norm, want), (sizes, float(norm), float(want))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m2", ["dyn4_proxy_la_upd_sr", "dyn4_vproxy_la_upd_sr", "dyn4_upd_sr"])
def test_16bit_research_kernels_match_oracle(m2, dtype):
    """16-bit parameters under the code-storing lookahead and the read-back second moments."""
    log(f"{dtype} nf4 / {m2} x 3 steps")
    make = lambda ps: aw.QuantizedAdamW(ps, lr=1e-3, weight_decay=0.1, m1_quant_scheme="nf4", m2_quant_scheme=m2,  # noqa: E731
                                        quant_rng_seed=3, optimized=True)
    out = run_pair(make, SHAPES, dtype, 3, seed=3, zero_block_frac=0.02, grad_fn=fp16_safe)
    compare_pair(*out, f"{dtype} nf4/{m2}", steps=3)


def launches(params, opt):
    """How many kernels a step of `opt` launches: the launch after the k-th is made to fail."""
    lib = _lib.library()
    for k in range(1, 8):
        for p in params:
            p.grad = torch.zeros_like(p)
        lib.aw4_inject_launch_failure(k)
        try:
            opt.step()
            return k
        except _lib.HipLaunchIncomplete:
            opt._inconsistent = None  # the test's own failure; the state is thrown away
        finally:
            lib.aw4_inject_launch_failure(-1)
    raise AssertionError("more launches than the test tries")


@pytest.mark.parametrize("dtype,m2,tiles,expect", [
    (torch.float32, "dyn4_sr", 1, 2),  # the generic kernel, whose fp32-state tile takes longer than a launch
    (torch.bfloat16, "dyn4_upd_sr_fp32read", 1, 1), (torch.bfloat16, "dyn4_upd_sr_fp32read", 2, 1),
    (torch.bfloat16, "dyn4_upd_sr_fp32read", 3, 2), (torch.float16, "dyn4_upd_sr_fp32read", 2, 1),
    (torch.float32, "dyn4_upd_sr", 2, 1), (torch.float32, "dyn4_upd_sr", 3, 2),
    (torch.float32, "dyn4_upd_sr_fp32read", 15, 1), (torch.float32, "dyn4_upd_sr_fp32read", 16, 2),
    (torch.float32, "dyn4_proxy_la_upd_sr", 15, 1), (torch.float32, "dyn4_proxy_la_upd_sr", 16, 2)])
def test_few_fp32_state_tiles_join_a_large_block_launch(dtype, m2, tiles, expect):
    """A launch of their own beside 8,192 block tiles costs 5-6 us, more than one or two tiles of a wave take in a
    specialised kernel."""
    params = [torch.nn.Parameter(torch.zeros(n, device=H.DEVICE, dtype=dtype)) for n in [8192 * 1024] + [1000] * tiles]
    opt = aw.QuantizedAdamW(params, m1_quant_scheme="nf4", m2_quant_scheme=m2, quant_rng_seed=1, optimized=True)
    assert launches(params, opt) == expect


# Every instance beside the recipes' fp32 and bf16 ones (those: test_gpu_step, test_gpu_fullsize).
INSTANCES = ([("nf4", "dyn4_nz", True, torch.float16), ("nf4", "dyn4_upd_sr_fp32read", False, torch.float16),
              ("nf4_sr", "dyn4_upd_sr_fp32read", False, torch.float16), ("nf4", "fp32", False, torch.float16),
              ("nf4", "dyn4_upd_sr_fp32read", True, torch.float16)]
             + [("sdyn4", "lin4_nz", False, dt) for dt in (torch.float32, torch.bfloat16, torch.float16)]
             + [("nf4", m2, False, dt) for m2 in ("dyn4_upd_sr", "dyn4_proxy_la_upd_sr")
                for dt in (torch.float32, torch.bfloat16, torch.float16)])


def instance(m1, m2, eden):
    return lambda ps: aw.QuantizedAdamW(ps, lr=1e-3, weight_decay=0.1, m1_quant_scheme=m1, m2_quant_scheme=m2,
                                        use_eden_m2=eden, quant_rng_seed=3, optimized=True)


@pytest.mark.parametrize("m1,m2,eden,dtype", INSTANCES)
def test_two_tiles_per_wave_match_oracle(m1, m2, eden, dtype):
    """32 tiles per CU, two for each wave, and a last tile of each tensor that is cut: the second tile's inputs are
    loaded during the first one's encode."""
    log(f"two tiles per wave {m1} / {m2} eden={eden} {dtype}")
    out = run_pair(instance(m1, m2, eden), [(2048, 4096), (33, 128), (71, 128)], dtype, 2, seed=3, zero_block_frac=0.02,
                   grad_fn=fp16_safe)
    compare_pair(*out, f"two tiles {m1}/{m2} {dtype}", steps=2)


def steps_of(make, shapes, dtype, shift, steps=2):
    """Parameters and state after `steps` on the GPU, parameters and gradients `shift` values off a 16-byte boundary."""
    params = []
    gen = torch.Generator(device=H.DEVICE).manual_seed(1)
    for s in shapes:
        n = s[0] * s[1]
        flat = torch.zeros(n + 8, device=H.DEVICE, dtype=dtype)
        flat[shift:n + shift].normal_(0.0, 0.02, generator=gen)
        params.append(torch.nn.Parameter(flat[shift:n + shift].view(s)))
    opt = make(params)
    for _ in range(steps):
        for p in params:
            n = p.numel()
            flat = torch.zeros(n + 8, device=H.DEVICE, dtype=dtype)
            # rows of magnitudes from e^-9 to e^-3, as heavy-tailed as an embedding's gradients
            g = flat[shift:n + shift].normal_(generator=gen).view(p.shape)
            g.mul_(torch.empty(p.shape[0], 1, device=H.DEVICE).uniform_(-9.0, -3.0, generator=gen).exp_().to(dtype))
            p.grad = g
        opt.step()
        for p in params:
            p.grad = None
    out = []
    for p in params:
        st = opt.state[p]
        out += [p.detach()] + [st[k] for k in ("m1", "m2", "m1_code", "m2_code") if k in st]
        out += [st[k].absmax for k in ("m1_quant_state", "m2_quant_state") if st.get(k) is not None]
    return out


@pytest.mark.parametrize("m1,m2,eden,dtype,rows", [case + (8200,) for case in INSTANCES]
                         + [case + (98400,) for case in INSTANCES if "upd_sr" in case[1]])
def test_more_tiles_per_wave_match_generic_kernel(m1, m2, eden, dtype, rows):
    """Three and four tiles per wave (128 tiles per CU), and twelve (1,536) of the kernels that take so many,
    against the generic kernel, which steps the same tensors one value off their alignment: bit for bit."""
    log(f"{rows} x 4096 {m1} / {m2} eden={eden} {dtype} against the generic kernel")
    shapes = [(rows, 4096), (33, 128)]
    got = steps_of(instance(m1, m2, eden), shapes, dtype, 0)
    want = steps_of(instance(m1, m2, eden), shapes, dtype, 1)
    assert len(got) == len(want)
    for i, (a, b) in enumerate(zip(got, want)):
        view = {4: torch.int32, 2: torch.int16, 1: torch.uint8}[a.element_size()]
        assert torch.equal(a.contiguous().view(-1).view(view), b.contiguous().view(-1).view(view)), i
