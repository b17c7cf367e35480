"""Specialised kernels by dtype and scheme pair, at the sizes where a dispatch or a tile can go wrong:
whole tiles, a last tile of a few blocks, a single 4-bit tensor of the smallest size, fp32-state tensors
in the same launch, and a launch of more than one tile per wave.  Against the oracle, with the bars of
``test_gpu_step`` (codes, scales and fp32 state bit-exact; parameters within the bars of ``gpu_helpers``)."""

from __future__ import annotations

import pytest
import torch

import adamw4bit_amd as aw
from tests import gpu_helpers as H
from tests.test_gpu_step import compare_pair, log, run_pair

pytestmark = pytest.mark.gpu

# 4 whole tiles, 1 block past a whole tile, 1 block short of one, many tiles, fp32 state
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
