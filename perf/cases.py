"""Performance cases of the 4-bit AdamW step: the calls a training program makes, over the sizes,
data types and options it makes them with.

A step case is an optimizer resumed at step 100 (4-bit codes and block scales, or fp32 state where a
tensor is below 4,096 values or not a multiple of 128), a gradient for every parameter, and one pass
is ``optimizer.step()``, with ``clip_grad_norm_`` before it where the program clips.  Parameters and
state lie in flat buffers (one per kind), so that a pass's whole result is a few tensors.  A codec
case is the stand-alone encode and decode of one moment.

Recipes are ``zeeden`` and ``zipsr`` (the two optimizer classes), ``mixed`` (ZIP-SR with an nf4_sr
head and ablations of its second moment, as ``bench.py`` groups them) or ``m1/m2`` (QuantizedAdamW
with those schemes).  Shapes are written ``RxC`` or ``N``, separated by spaces.
"""

from __future__ import annotations

import math

import numpy as np
import torch

import adamw4bit_amd as aw
from adamw4bit_amd import _lib, quantization
from adamw4bit_amd.quantization import QuantState

LR, BETA1, BETA2, EPS, DECAY = 1e-4, 0.9, 0.95, 1e-8, 0.1
STEP0 = 100          # the step count the optimizer resumes at
BLOCK, MIN_4BIT = 128, 4096
ALIGN = 1024         # flat buffers hold each tensor at a multiple of this many values

LAYER = "4096x4096 1024x4096 1024x4096 4096x4096 14336x4096 14336x4096 4096x14336 4096 4096"  # Llama-3-8B's
EMBEDDING = "128256x4096"
GPT2_LAYER = "768 768 768x2304 2304 768x768 768 768 768 768x3072 3072 3072x768 768"
GPT2_SMALL = "50257x768 1024x768 " + " ".join([GPT2_LAYER] * 12) + " 768 768"
TINY_LAYER = "64 64 64x192 192 64x64 64 64 64 64x256 256 256x64 64"
TINY_GPT2 = "128x64 64x64 " + " ".join([TINY_LAYER] * 2) + " 64 64 128x64"
ODD = "1000x1001 2049x1023 513x255x9 50257x33 4097 1000 129 50x256 3072x768 96x511 1001 7"

NF4 = (-1.0, -0.696192801, -0.525073111, -0.394917488, -0.284441411, -0.1847734, -0.091049999, 0.0, 0.0795802996,
       0.160930201, 0.246112302, 0.337915212, 0.4407098, 0.562617004, 0.722956777, 1.0)
SDYN4 = (-0.887499988, -0.662500024, -0.4375, -0.212499991, -0.0775000006, -0.0325000025, -0.00549999997, 0.0,
         0.00549999997, 0.0325000025, 0.0775000006, 0.212499991, 0.4375, 0.662500024, 0.887499988, 1.0)
DYN4 = (0.0, 0.00325000007, 0.00774999941, 0.0212500002, 0.0437499993, 0.0662500039, 0.0887499973, 0.15625, 0.268750012,
        0.381249994, 0.493750006, 0.606250048, 0.71875, 0.831249952, 0.943750024, 1.0)
LIN4 = tuple(float(np.float32(v)) for v in torch.linspace(0, 1, 16, dtype=torch.float32).tolist())
DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}


def levels_of(scheme: str):
    return NF4 if scheme.startswith("nf4") else SDYN4 if scheme.startswith("sdyn4") else (
        LIN4 if scheme.startswith("lin4") else DYN4)


def step_case(name, recipe, dtype, shapes, clip=0.0):
    return dict(name=name, kind="step", recipe=recipe, dtype=dtype, shapes=shapes, clip=clip)


def listed():
    return [
        # the smallest steps: a tiny GPT-2 trained with clipping (29 tensors, 120K values) and one square
        # matrix; the host and the launches set their time
        step_case("tiny_gpt2_zipsr_clip", "zipsr", "fp32", TINY_GPT2, 1.0),
        step_case("zeeden_fp32_1024", "zeeden", "fp32", "1024x1024"),
        # one ordinary weight matrix
        step_case("zipsr_fp32_4096", "zipsr", "fp32", "4096x4096"),
        # GPT-2 small trained the way the reference's trainer does, gradients clipped to norm 1
        step_case("gpt2_small_zeeden_clip", "zeeden", "fp32", GPT2_SMALL, 1.0),
        # GPT-2 small under plain round-to-nearest moments, the ablation both recipes are compared with
        step_case("gpt2_small_nf4_dyn4_nz", "nf4/dyn4_nz", "fp32", GPT2_SMALL),
        # two layers of Llama-3-8B with bf16 parameters and gradients: one rank's shard of a larger model
        step_case("llama_layers_zipsr_bf16", "zipsr", "bf16", LAYER + " " + LAYER),
        # the largest: embedding and one layer of Llama-3-8B in fp32
        step_case("llama_embed_layer_zipsr_fp32", "zipsr", "fp32", EMBEDDING + " " + LAYER),
        # the mixed-scheme bf16 set: fp32 and EDEN second moments between ZIP-SR tensors, an nf4_sr head
        step_case("llama_mixed_bf16", "mixed", "bf16", LAYER + " " + EMBEDDING),
        # fp16 parameters and gradients (a model held in half precision)
        step_case("llama_layer_zeeden_fp16", "zeeden", "fp16", LAYER),
        # a model whose sizes are no multiples of 128 (convolutions, odd heads, biases): mostly fp32 state
        step_case("odd_sizes_zipsr_fp32", "zipsr", "fp32", ODD),
        # a research second moment, stored for the next step's preconditioner
        step_case("llama_layer_proxy_lookahead", "nf4/dyn4_proxy_la_upd_sr", "fp32", LAYER),
        # encode and decode of one moment on their own (a checkpoint converted, state inspected)
        dict(name="codec_nf4_16m", kind="codec", scheme="nf4", numel=1 << 24),
    ]


RECIPES = ("zeeden", "zipsr", "zeeden", "zipsr", "mixed", "nf4/dyn4_nz", "nf4_sr/dyn4_upd_sr_fp32read",
           "sdyn4/dyn4", "nf4/lin4", "nf4/fp32", "nf4/dyn4_proxy_la_upd_sr")


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    if rng.random() < 0.1:
        return dict(kind="codec", scheme=rng.choice(["nf4", "nf4_sr", "dyn4_nz", "dyn4_sr", "sdyn4"]),
                    numel=BLOCK * size(32, 1 << 20))
    recipe = rng.choice(RECIPES)
    dtype = rng.choice(["fp32", "fp32", "bf16", "bf16", "fp16"])
    budget = size(5_000, 300_000_000)  # values in all
    if recipe == "nf4/dyn4_proxy_la_upd_sr":
        budget = min(budget, 150_000_000)
    ragged = rng.random() < 0.3
    shapes = []
    for _ in range(size(1, 24)):
        kind = rng.random()
        if kind < 0.3:
            shape = (size(1, 16384),)
        else:
            rows, cols = size(16, 16384), size(16, 16384)
            shape = (rows, cols if ragged else max(BLOCK, cols // BLOCK * BLOCK))
        n = math.prod(shape)
        if n <= budget:
            shapes.append("x".join(map(str, shape)))
            budget -= n
    if not shapes:
        shapes = [str(budget)]
    return dict(kind="step", recipe=recipe, dtype=dtype, shapes=" ".join(shapes), clip=rng.choice([0.0, 0.0, 1.0]))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def tensors_of(case):
    """Per tensor: shape, numel, first-moment scheme, second-moment scheme, EDEN on the second moment
    (the effective ones: fp32 state below 4,096 values or off the 128-value block)."""
    out = []
    shapes = [tuple(int(d) for d in s.split("x")) for s in case["shapes"].split()]
    recipe = case["recipe"]
    for i, shape in enumerate(shapes):
        n = math.prod(shape)
        if recipe == "zeeden":
            m1, m2, eden = "nf4", "dyn4_nz", True
        elif recipe == "zipsr":
            m1, m2, eden = "nf4", "dyn4_upd_sr_fp32read", False
        elif recipe == "mixed":
            m1, m2, eden = "nf4", "dyn4_upd_sr_fp32read", False
            if i % 5 == 2:
                m2 = "fp32"
            elif i % 5 == 4:
                eden = True
            if i == len(shapes) - 1:
                m1, m2, eden = "nf4_sr", "dyn4_upd_sr_fp32read", False
        else:
            (m1, m2), eden = recipe.split("/"), False
        if n < MIN_4BIT or n % BLOCK:
            m1 = m2 = "fp32"
        out.append((shape, n, m1, m2, eden))
    return out


def layout_of(case):
    """Where each tensor's parts start in the flat buffers, and the buffers' lengths: p and g in values,
    codes in bytes, scales and fp32 state in floats."""
    sizes = dict(p=0, m1_codes=0, m1_scales=0, m2_codes=0, m2_scales=0, m1=0, m2=0)
    places = []
    for _, n, m1, m2, _ in tensors_of(case):
        padded = -(-n // ALIGN) * ALIGN
        at = dict(p=sizes["p"])
        sizes["p"] += padded
        for key, scheme in (("m1", m1), ("m2", m2)):
            if scheme == "fp32":
                at[key] = sizes[key]
                sizes[key] += padded
            else:
                at[key + "_codes"], at[key + "_scales"] = sizes[key + "_codes"], sizes[key + "_scales"]
                sizes[key + "_codes"] += padded // 2
                sizes[key + "_scales"] += padded // BLOCK
        places.append(at)
    return places, {k: v for k, v in sizes.items() if v}


def encode(values, scheme):
    """Nearest codes (packed, the even value in the low nibble) and block scales of a moment."""
    levels = torch.tensor(levels_of(scheme), device=values.device)
    blocks = values.view(-1, BLOCK)
    scale = blocks.abs().amax(1).clamp_min(1e-12)
    code = torch.bucketize((blocks / scale[:, None]).view(-1), (levels[1:] + levels[:-1]) / 2, out_int32=True).to(torch.uint8)
    if scheme == "dyn4_nz":
        code.clamp_(min=1)
    return code[0::2] | code[1::2] << 4, scale


def decode64(codes, scales, scheme):
    levels = torch.tensor(levels_of(scheme), device=codes.device, dtype=torch.float32).double()
    x = torch.stack((levels[(codes & 15).long()], levels[(codes >> 4).long()]), 1)
    return (x.view(-1, BLOCK) * scales.double()[:, None]).view(-1)


def inputs(case, seed, device="cuda"):
    """The flat parameters, gradients and state, made from the seed alone.  Gradients are Student-t(3)
    values times a log-normal magnitude per row, as an embedding's or a projection's are; the moments
    are those of such gradients, and every hundredth block of a 4-bit tensor has had no gradient."""
    gen = torch.Generator(device=device).manual_seed(1000 + seed)
    dtype = DTYPES[case["dtype"]]
    mu = -5.0 if dtype == torch.float16 else -7.0  # fp16 gradients are kept above its subnormals
    tensors = tensors_of(case)
    places, sizes = layout_of(case)
    flat = {k: torch.zeros(v, device=device, dtype=dtype if k == "p" else torch.uint8 if k.endswith("codes") else
                           torch.float32) for k, v in sizes.items()}
    grad = torch.zeros(sizes["p"], device=device, dtype=dtype)

    def normal(n):
        return torch.randn(n, generator=gen, device=device)

    for (shape, n, m1, m2, _), at in zip(tensors, places):
        flat["p"][at["p"]:at["p"] + n] = (normal(n) * 0.02).to(dtype)
        rows = shape[0] if len(shape) > 1 else 1
        size = torch.exp(normal(rows) + mu).repeat_interleave(n // rows)
        chi2 = normal(n).square_()
        for _ in range(2):
            chi2.addcmul_(*(2 * [normal(n)]))
        g = normal(n).div_(chi2.div_(3.0).sqrt_()).mul_(size)
        del chi2
        a = normal(n).mul_(0.4).mul_(size)
        b = size.square_().mul_(1.5 * torch.rand(n, generator=gen, device=device) + 0.05).addcmul_(g, g, value=0.1)
        if m1 != "fp32":
            still = (torch.rand(n // BLOCK, generator=gen, device=device) < 0.01)[:, None]
            for v in (g, a, b):
                v.view(-1, BLOCK).masked_fill_(still, 0.0)
        grad[at["p"]:at["p"] + n] = g.to(dtype)
        for key, scheme, v in (("m1", m1, a), ("m2", m2, b)):
            if scheme == "fp32":
                flat[key][at[key]:at[key] + n] = v
            else:
                codes, scales = encode(v, scheme)
                flat[key + "_codes"][at[key + "_codes"]:at[key + "_codes"] + n // 2] = codes
                flat[key + "_scales"][at[key + "_scales"]:at[key + "_scales"] + n // BLOCK] = scales
                del codes
    return flat, grad


def codec_inputs(case, seed, device="cuda"):
    gen = torch.Generator(device=device).manual_seed(1000 + seed)
    n = case["numel"]
    values = torch.randn(n, generator=gen, device=device) * 1e-3
    if case["scheme"].startswith("dyn4"):
        values.square_()
    stored = torch.randint(0, 256, (n // 2,), generator=gen, device=device, dtype=torch.uint8)
    stored_scales = torch.rand(n // BLOCK, generator=gen, device=device) * 1e-2
    return values, stored, stored_scales


# ---------------------------------------------------------------------------
# The program's handles, one pass, and its cost
# ---------------------------------------------------------------------------

def moment(scheme, codes, scales):
    codebook, rounding, floor = quantization.SCHEMES[scheme]
    m = np.zeros((), dtype=_lib.MOMENT)
    m["codes"], m["scales"], m["codebook"], m["rounding"] = codes.data_ptr(), scales.data_ptr(), codebook, rounding
    m["flags"] = (_lib.MOMENT_ZERO_FLOOR if floor else 0) | _lib.MOMENT_GUARDS
    m["rng_seed"], m["sr_bias"], m["sr_bias_rcp"], m["sr_eps"] = 7, 1.0, 1.0, EPS
    return m


def prepare(case, seed):
    if case["kind"] == "codec":
        values, stored, stored_scales = codec_inputs(case, seed)
        n = case["numel"]
        out = dict(codes=torch.empty_like(stored), scales=torch.empty_like(stored_scales), values=torch.empty_like(values))
        return dict(kind="codec", n=n, values=values, stored=(stored, stored_scales), out=out,
                    enc=moment(case["scheme"], out["codes"], out["scales"]), dec=moment(case["scheme"], stored, stored_scales))
    flat, grad = inputs(case, seed)
    tensors = tensors_of(case)
    places, _ = layout_of(case)
    params = []
    for (shape, n, *_), at in zip(tensors, places):
        p = torch.nn.Parameter(flat["p"][at["p"]:at["p"] + n].view(shape))
        p.grad = grad[at["p"]:at["p"] + n].view(shape)
        params.append(p)
    hyper = dict(lr=LR, betas=(BETA1, BETA2), eps=EPS, weight_decay=DECAY, optimized=True)
    recipe = case["recipe"]
    if recipe == "zeeden":
        opt = aw.ZEEDENAdamW4Bit(params, **hyper)
    elif recipe == "zipsr":
        opt = aw.ZIPSRAdamW4Bit(params, quant_rng_seed=0, **hyper)
    elif recipe == "mixed":
        groups = [dict(params=[p], m1_quant_scheme="nf4",
                       m2_quant_scheme="fp32" if i % 5 == 2 and i < len(params) - 1 else "dyn4_upd_sr_fp32read",
                       use_eden_m2=i % 5 == 4 and i < len(params) - 1) for i, p in enumerate(params)]
        opt = aw.QuantizedAdamW(groups, m1_quant_scheme="nf4", m2_quant_scheme="dyn4_upd_sr_fp32read", quant_rng_seed=0,
                                **hyper)
        opt.set_m1_quant_scheme_for_parameters([params[-1]], "nf4_sr")
    else:
        m1, m2 = recipe.split("/")
        opt = aw.QuantizedAdamW(params, m1_quant_scheme=m1, m2_quant_scheme=m2, quant_rng_seed=0, **hyper)
    for p, (shape, n, m1, m2, _), at in zip(params, tensors, places):
        state = opt.state[p]
        state["step"] = STEP0
        for key, scheme in (("m1", m1), ("m2", m2)):
            if scheme == "fp32":
                state[key] = flat[key][at[key]:at[key] + n].view(shape)
                continue
            codes = flat[key + "_codes"][at[key + "_codes"]:at[key + "_codes"] + n // 2]
            scales = flat[key + "_scales"][at[key + "_scales"]:at[key + "_scales"] + n // BLOCK]
            state[key + "_code"] = codes
            state[key + "_quant_state"] = QuantState(absmax=scales, shape=p.shape, dtype=torch.float32, blocksize=BLOCK,
                                                     packed=True)
    return dict(kind="step", opt=opt, clip=case["clip"], flat=flat, grad=grad)


def run(state):
    if state["kind"] == "codec":
        stream = torch.cuda.current_stream().cuda_stream
        _lib.quantize(state["values"].data_ptr(), state["n"], state["enc"], stream)
        _lib.dequantize(state["dec"], state["n"], state["out"]["values"].data_ptr(), stream)
        return state["out"]
    out = dict(state["flat"])
    if state["clip"]:
        out["norm"] = state["opt"].clip_grad_norm_(state["clip"])
    state["opt"].step()
    return out


def work(case):
    """Bytes: parameters read and written, gradients read, and of each moment the codes and scales, or
    the fp32 state, read and written.  A few dozen operations per value, none of them a product of
    matrices."""
    if case["kind"] == "codec":
        n = case["numel"]
        return {"bytes": n * (4 + 0.5 + 4 / BLOCK) * 2, "flops": 8.0 * n}
    size = 4 if case["dtype"] == "fp32" else 2
    total = values = 0
    for _, n, m1, m2, _ in tensors_of(case):
        values += n
        total += n * (3 * size + sum(8 if m == "fp32" else 1 + 8 / BLOCK for m in (m1, m2)))
    return {"bytes": total, "flops": 40.0 * values}


def tolerance(case):
    """Codes and round-to-nearest scales are the same for every correct fp32 implementation; fp32
    parameters and scales differ by single roundings (EPS-sized updates of N(0, 0.02) values), 16-bit
    parameters by a rounding of a few values."""
    if case["kind"] == "codec" or case["dtype"] == "fp32":
        return {"rel": 1e-6, "max": 1e-4}
    return {"rel": 1e-3, "max": 4e-2}


def exact(case, seed):
    """One pass in 64 bits: the parameters, the fp32 state, the absmax scales and the gradient norm.  Codes,
    and scales calibrated to them (EDEN), have no value there."""
    if case["kind"] == "codec":
        values, stored, stored_scales = codec_inputs(case, seed)
        return dict(codes=None, scales=values.double().view(-1, BLOCK).abs().amax(1).clamp_min(1e-12),
                    values=decode64(stored, stored_scales, case["scheme"]))
    flat, grad = inputs(case, seed)
    tensors = tensors_of(case)
    places, _ = layout_of(case)
    out = {k: None if k.endswith("codes") else v.double() for k, v in flat.items()}
    coef = 1.0
    if case["clip"]:
        norm = math.sqrt(sum(float(grad[at["p"]:at["p"] + n].double().square().sum()) for (_, n, *_), at in
                             zip(tensors, places)))
        out["norm"] = torch.tensor(norm, dtype=torch.float64)
        coef = min(1.0, case["clip"] / (norm + 1e-6))
    step = STEP0 + 1
    for (_, n, s1, s2, eden), at in zip(tensors, places):
        g = grad[at["p"]:at["p"] + n].double().mul_(coef)
        new = {}
        for key, scheme, beta, target in (("m1", s1, BETA1, g), ("m2", s2, BETA2, g.square())):
            if scheme == "fp32":
                m = flat[key][at[key]:at[key] + n].double()
            else:
                c, s = at[key + "_codes"], at[key + "_scales"]
                m = decode64(flat[key + "_codes"][c:c + n // 2], flat[key + "_scales"][s:s + n // BLOCK], scheme)
            m = new[key] = m.mul_(beta).add_(target, alpha=1 - beta)
            if scheme == "fp32":
                out[key][at[key]:at[key] + n] = m
            elif key == "m1" or not eden:
                out[key + "_scales"][s:s + n // BLOCK] = m.view(-1, BLOCK).abs().amax(1).clamp_min(1e-12)
        den = new["m2"].div_(1 - BETA2 ** step).sqrt_().add_(EPS)
        p = out["p"][at["p"]:at["p"] + n]
        p.mul_(1 - LR * DECAY).addcdiv_(new["m1"], den, value=-LR / (1 - BETA1 ** step))
    if any(eden and s2 != "fp32" for *_, s2, eden in tensors):
        out["m2_scales"] = None
    return out
