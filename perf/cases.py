"""The work that a user has this library do, as a list of cases to be timed.

A case is a dict of plain values; its "call" says which of the public entry points it goes through:

  train    FusedSoftcappedCrossEntropy.apply(...) and .backward(): the loss head of one training step
  norm     FusedNormSoftcappedCrossEntropy with the weight's scale taken on the device (amax_scale) in the same step
  micro    ce_forward / ce_backward of a few micro-batches under one WeightCache: gradient accumulation
  eval     softcapped_cross_entropy: the loss alone, of a validation batch
  score    target_probability: what the rows give their targets, for ensembles and for ranking short texts
  weight   amax_scale, quantize_e4m3, transpose_copy: both fp8 layouts of a weight, for a caller's own GEMMs

Sizes: N rows (tokens), d hidden units, V vocabulary columns (50304 is GPT-2's 50257 padded; "vocab" is how many of them
take part).  Rows have unit RMS, weights are normal, targets are Zipf-distributed or uniform over the real vocabulary --
the values of slowrun_amd.configs -- and everything is drawn on the GPU from the seed alone.
"""
import math

import torch
import torch.nn.functional as F

from slowrun_amd import cuda_kernels as ck

REAL_VOCAB = 50257
X_S, W_S, GRAD_S = 100 / 448, 1.6 / 448, 0.75 / 448          # the trainer's fixed fp8 scales (tiny/train.py:188-190)
MTP = (1.0, 0.5, 0.25, 0.125)                                 # weights of the prediction offsets
MOST_FLOPS = 6.0 * 65536 * 2560 * 50304                       # of one drawn case: the largest listed training step


def _case(name, call, N, d, V, **more):
    c = dict(name=name, call=call, N=N, d=d, V=V, vocab=min(REAL_VOCAB, V), dtype="bf16", operands="e4m3", cap=15.0, reduction="mean", offsets=1,
             keep=True, ignored=0.0, hot=0.0, zipf=True, fixed_scales=False, device_scales=False, micro=1)
    c.update(more)
    return c


def listed():
    return [
        # a unit test or a toy model: the smallest training step, bound by launches
        _case("train_toy", "train", 1000, 256, 4096, zipf=False),
        # the small fp32 configuration: float32 hidden states, weight and gradients
        _case("train_fp32", "train", 2048, 768, 50304, dtype="fp32", zipf=False),
        # the tiny track's device batch as its trainer calls the head: three offsets, per-row losses, fixed scales
        _case("train_tiny_mtp", "train", 32768, 1024, 50304, offsets=3, reduction="none", fixed_scales=True, zipf=False),
        # the 2.7B model's head on one GPU's share of the batch: the headline
        _case("train_2p7b", "train", 65536, 2560, 50304),
        # ragged rows, masked prompts and padding (12 % ignored), a few rows that saturate the cap
        _case("train_irregular", "train", 30011, 2560, 50304, ignored=0.12, hot=0.001, zipf=False),
        # a large multilingual vocabulary under a higher cap
        _case("train_large_vocab", "train", 16384, 4096, 131072, vocab=131072, cap=30.0, zipf=False),
        # a trainer short of memory: nothing N x V is held between forward and backward
        _case("train_recompute", "train", 8192, 2560, 50304, keep=False),
        # final norm fused into the head, the weight's scale taken from the weight in every step
        _case("norm_device_scale", "norm", 4096, 1600, 50304, device_scales=True),
        # two micro-batches between optimizer steps, the weight quantised once
        _case("micro_steps", "micro", 2048, 1024, 50304, micro=2),
        # a validation batch in the reference's eval arithmetic (bf16 GEMM, padded columns sliced off)
        _case("eval_bf16", "eval", 16384, 1024, 50304, operands="bf16", reduction="none"),
        # one short text scored by a large head: all of the weight for a few rows
        _case("score_short", "score", 61, 2560, 50304, operands="bf16"),
        # an fp8 copy of a weight and its transpose
        _case("weight_fp8", "weight", 1, 2560, 50304),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    while True:
        call = rng.choice(("train", "train", "train", "norm", "micro", "eval", "score", "weight"))
        lo, hi = {"train": (256, 65536), "norm": (256, 32768), "micro": (256, 8192), "eval": (512, 65536), "score": (1, 4096), "weight": (1, 1)}[call]
        N = min(hi, max(lo, round(_log(rng, lo, hi))))
        if rng.random() < 0.4 and N >= 512:
            N = N // 256 * 256                                 # whole batches of whole sequences
        d = round(_log(rng, 256, 4096) / 16) * 16
        V = round(_log(rng, 4096, 131072))
        V = V if rng.random() < 0.3 else (V + 63) // 64 * 64   # most vocabularies are padded
        V = 50304 if rng.random() < 0.4 else min(V, 131072)
        more = dict(vocab=min(REAL_VOCAB, V) if V <= 65536 else V, dtype="fp32" if rng.random() < 0.2 else "bf16", zipf=rng.random() < 0.5,
                    cap=30.0 if rng.random() < 0.2 else 15.0)
        if call in ("train", "norm"):
            more.update(offsets=rng.choice((1, 1, 2, 3)), keep=rng.random() < 0.75, ignored=rng.choice((0.0, 0.0, 0.12)), device_scales=call == "norm")
        if call == "train":
            more.update(hot=rng.choice((0.0, 0.0, 0.001)), fixed_scales=rng.random() < 0.3)
        if call == "micro":
            more.update(micro=rng.choice((2, 3)))
        if call in ("eval", "score"):
            more.update(operands=rng.choice(("bf16", "e4m3")))
        more["reduction"] = "none" if more.get("offsets", 1) > 1 or call == "score" else rng.choice(("mean", "none"))
        c = _case("", call, N, d, V, **more)
        del c["name"]
        if work(c)["flops"] <= MOST_FLOPS:
            return c


def _targets(c, n, gen):
    if c["zipf"]:
        p = (torch.arange(c["vocab"], dtype=torch.float64, device="cuda") + 1.0) ** -1.1
        y = torch.multinomial(p / p.sum(), n, True, generator=gen)
    else:
        y = torch.randint(0, c["vocab"], (n,), device="cuda", generator=gen)
    if c["ignored"]:
        y[torch.rand(n, device="cuda", generator=gen) < c["ignored"]] = -1
    return y


def prepare(c, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = torch.float32 if c["dtype"] == "fp32" else torch.bfloat16
    N, d, V, grad = c["N"], c["d"], c["V"], c["call"] in ("train", "norm")
    s = dict(case=c)
    w = torch.randn(d, V, device="cuda", generator=gen).mul_(d ** -0.5)
    s["w_s"] = W_S if c["fixed_scales"] else float(w.abs().max()) / 448
    s["w"] = w.to(dtype).requires_grad_(grad)
    del w
    if c["call"] == "weight":
        return s
    s["x"], s["y"] = [], []
    for _ in range(c["micro"]):
        x = torch.randn(N, d, device="cuda", generator=gen)
        if c["call"] != "norm":
            x = F.rms_norm(x, (d,))
        if c["hot"]:
            x[torch.rand(N, device="cuda", generator=gen) < c["hot"]] *= 50.0
        s["x_s"] = X_S if c["fixed_scales"] else float(F.rms_norm(x, (d,)).abs().max() if c["call"] == "norm" else x.abs().max()) / 448
        s["x"].append(x.to(dtype).requires_grad_(grad))
        s["y"].append(_targets(c, N, gen))
    if c["offsets"] > 1:
        s["mtp"] = torch.tensor(MTP[: c["offsets"]], device="cuda")
    if c["call"] == "micro":
        s["cache"] = ck.WeightCache()
        s["go"] = torch.ones((), device="cuda") if c["reduction"] == "mean" else torch.full((N,), 1.0 / N, device="cuda")
    return s


def run(s):
    c, w = s["case"], s["w"]
    if c["call"] == "weight":
        scale = ck.amax_scale(w)
        q = ck.quantize_e4m3(w, scale)
        qt = torch.empty(w.shape[1], w.shape[0], dtype=q.dtype, device=q.device)
        ck.transpose_copy(q, qt)
        return scale, q.view(torch.uint8), qt.view(torch.uint8)
    x, y, cap = s["x"][0], s["y"][0], c["cap"]
    if c["call"] == "eval":
        ops = dict(operand_dtype=torch.bfloat16) if c["operands"] == "bf16" else dict(x_s=s["x_s"], w_s=s["w_s"])
        return ck.softcapped_cross_entropy(x, w, y, cap=cap, vocab_size=c["vocab"], reduction=c["reduction"], **ops)
    if c["call"] == "score":
        ops = dict(operand_dtype=torch.bfloat16) if c["operands"] == "bf16" else dict(x_s=s["x_s"], w_s=s["w_s"])
        return ck.target_probability(x, w, y, cap=cap, vocab_size=c["vocab"], **ops)
    if c["call"] == "micro":
        out = []
        s["cache"].invalidate()                                # the optimizer has stepped
        for x, y in zip(s["x"], s["y"]):
            loss, saved, _lse, _argmax, _n = ck.ce_forward(x, w, y, s["x_s"], s["w_s"], cap, c["reduction"], keep_dlogits=True, weight_cache=s["cache"])
            dx, dw = ck.ce_backward(saved, y, s["go"], x.shape[0], x.shape[1], w.shape[1], s["x_s"], s["w_s"], cap, 1.0, c["reduction"], x.dtype, w.dtype,
                                    keep_dlogits=True, weight_cache=s["cache"], cache_generation=s["cache"].generation)
            out.append((loss, dx, dw))
        return out
    x.grad = w.grad = None
    mtp = s.get("mtp")
    if c["call"] == "norm":
        w_s = ck.amax_scale(w.detach()) if c["device_scales"] else s["w_s"]
        out = ck.FusedNormSoftcappedCrossEntropy.apply(x, y, mtp, w, s["x_s"], w_s, GRAD_S, 1.0, cap, c["reduction"], None, c["keep"])
    else:
        out = ck.FusedSoftcappedCrossEntropy.apply(x, y, mtp, w, s["x_s"], s["w_s"], GRAD_S, 1.0, cap, c["reduction"], c["keep"])
    (out if c["reduction"] == "mean" else out.mean()).backward()
    return out.detach(), x.grad, w.grad


def work(c):
    """Inputs read once and outputs written once; two flops per multiply-add of the logits and, in training, of dX and dW."""
    N, d, V, eb = c["N"], c["d"], c["V"], 4 if c["dtype"] == "fp32" else 2
    if c["call"] == "weight":
        return {"bytes": d * V * (eb + 2.0) + 4, "flops": 2.0 * d * V}
    if c["call"] in ("eval", "score"):
        return {"bytes": (N * d + d * c["vocab"]) * eb + N * 12.0, "flops": 2.0 * N * d * c["vocab"]}
    return {"bytes": c["micro"] * (N * (2.0 * d * eb + 12) + d * V * eb) + float(d * V * eb), "flops": c["micro"] * 6.0 * N * d * V}


def tolerance(c):
    """Four times what was measured between two ways of computing the same thing: training against the other backward mode
    and against an fp32 evaluation in torch (rel 2.5e-3, max 1.7e-2 with bf16 gradients: their rounding and the e4m3 dlogits;
    7e-4 and 4e-3 with fp32 ones), the forward-only calls against the same call with d summed in another order."""
    if c["call"] == "weight":
        return "exact"                                         # bytes of an exactly defined cast, and a maximum
    if c["call"] in ("eval", "score"):
        if c["operands"] == "bf16":                            # the logits are rounded to bf16: in a rare row the target's falls to the other side
            return {"rel": 1e-4, "max": 0.02}
        return {"rel": 1e-5, "max": 1e-4} if c["call"] == "eval" else {"rel": 1e-4, "max": 4e-4}        # loss; exp(-loss)
    return {"rel": 0.01, "max": 0.07} if c["dtype"] == "bf16" else {"rel": 0.003, "max": 0.02}
