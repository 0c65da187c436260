"""What the performance of this library is measured on: the calls that an FP8 MoE model makes through the
public entry points, training and inference, from one decode step to the largest training shapes.

A case is a dict of plain values; its "op" names the group of calls that a layer makes together.
listed() gives the standing cases, draw() more of the same ranges, prepare() what a program holds
before the calls, run() the calls, work() the compulsory traffic, tolerance() what may differ.
"""
import math

import torch

from linghe_amd import configs
from linghe_amd.quant.block import triton_batch_blockwise_quant, triton_block_quant, triton_blockwise_quant
from linghe_amd.quant.group import triton_group_quant
from linghe_amd.utils.gather import triton_batch_block_pad_permute_with_indices
from linghe_amd.utils.norm import (
    triton_rms_norm_and_block_quant_forward,
    triton_rms_norm_backward,
    triton_rms_norm_forward,
    triton_rms_norm_fp32_gemm_block_quant_forward,
)
from linghe_amd.utils.silu import (
    build_expert_plan,
    triton_batch_weighted_silu_and_block_quant_backward,
    triton_batch_weighted_silu_and_block_quant_forward,
    triton_silu_and_block_quant_backward,
    triton_silu_and_block_quant_forward,
    triton_weighted_silu_backward,
    triton_weighted_silu_forward,
)


def listed():
    return [
        # one decode step of a batch of 32 sequences: the layer's row-wise quantisers, where latency counts
        dict(name="infer_decode_32", op="infer", M=32, n=2048, f=1536, pow2=False),
        # a prefill chunk of ragged length through the same calls
        dict(name="infer_prefill_3001", op="infer", M=3001, n=4096, f=1536, pow2=False),
        # pre-attention / pre-MLP norm of a training step, both code layouts (the benchmark's headline shape)
        dict(name="norm_quant_8192x2048", op="norm_quant", M=8192, n=2048, pow2=False),
        # the same at the largest hidden size and batch of the benchmark
        dict(name="norm_quant_16384x7168", op="norm_quant", M=16384, n=7168, pow2=False),
        # activation recompute: row-wise codes in the forward, transposed ones from the saved statistic in the
        # backward, power-of-two scales, rows not a multiple of 128
        dict(name="norm_recompute_4104x5120", op="norm_recompute", M=4104, n=5120, pow2=True),
        # bf16 training step of the layers kept out of FP8: RMSNorm and weighted SwiGLU, forward and backward
        dict(name="bf16_step_8192", op="bf16_step", M=8192, n=2048, f=2048, wbf16=False),
        # dense MLP / shared expert of a training step: SwiGLU + quant forward and backward
        dict(name="swiglu_step_8192x2048", op="swiglu_step", M=8192, f=2048, pow2=False),
        # routed experts of a training step: 8192 tokens, top-8 of 256 experts, Zipf-distributed load
        dict(name="experts_step_256", op="experts_step", tokens=8192, topk=8, experts=256, f=512, counts_seed=1003,
             plan=True, wbf16=False, pow2=False),
        # token dispatch to 32 experts, top-2 (forward), and the gradient's quantiser on the same rows (backward)
        dict(name="dispatch_32", op="dispatch", tokens=16384, topk=2, experts=32, n=2048, counts_seed=1101, pow2=False),
        # a linear layer of a training step: activation in both layouts and the weight in 128x128 blocks
        dict(name="linear_8192x2048", op="linear", M=8192, n=2048, out=4096, pow2=False),
        # norm + router logits + quant with a bf16 router weight
        dict(name="router_bf16_8192", op="router", M=8192, N=256, K=2048, fp32=False, pow2=False),
        # the same with the fp32 router weight that a mixed-precision optimiser keeps, on a wider model
        dict(name="router_fp32_4096", op="router", M=4096, N=256, K=4096, fp32=True, pow2=False),
    ]


def _log(rng, lo, hi, multiple=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(multiple, int(round(v / multiple)) * multiple)


def _draw_one(rng):
    op = rng.choice(["infer", "norm_quant", "norm_recompute", "bf16_step", "swiglu_step", "experts_step", "dispatch",
                     "linear", "router"])
    pow2 = rng.random() < 0.3
    width = lambda lo, hi: _log(rng, lo, hi, 128)  # noqa: E731
    if op == "infer":
        return dict(op=op, M=_log(rng, 1, 4096), n=width(1024, 7168), f=width(512, 4096), pow2=pow2)
    if op in ("norm_quant", "norm_recompute"):
        # sequence lengths are even or padded more often than not
        return dict(op=op, M=_log(rng, 256, 16384, rng.choice([1, 8, 128, 128, 1024])), n=width(512, 7168), pow2=pow2)
    if op == "bf16_step":
        return dict(op=op, M=_log(rng, 256, 16384, rng.choice([1, 128])), n=width(512, 7168), f=width(512, 4096),
                    wbf16=rng.random() < 0.3)
    if op == "swiglu_step":
        return dict(op=op, M=_log(rng, 256, 16384, 128), f=width(512, 6144), pow2=pow2)
    if op == "experts_step":
        experts = rng.choice([8, 16, 32, 64, 128, 256])
        return dict(op=op, tokens=_log(rng, 256, 16384), topk=rng.choice([1, 2, 4, 6, 8]), experts=experts,
                    f=width(256, 2048), counts_seed=rng.randrange(1 << 20), plan=rng.random() < 0.5,
                    wbf16=rng.random() < 0.3, pow2=pow2)
    if op == "dispatch":
        return dict(op=op, tokens=_log(rng, 256, 16384), topk=rng.choice([1, 2, 4, 6, 8]),
                    experts=rng.choice([8, 16, 32, 64, 128, 256]), n=width(1024, 7168),
                    counts_seed=rng.randrange(1 << 20), pow2=pow2)
    if op == "linear":
        return dict(op=op, M=_log(rng, 256, 16384, 16), n=width(512, 7168), out=width(512, 8192), pow2=pow2)
    return dict(op="router", M=_log(rng, 128, 16384, 128), N=rng.choice([128, 256, 256, 384, 512]),
                K=width(1024, 7168), fp32=rng.random() < 0.5, pow2=pow2)


def draw(rng):
    """A case of the ranges above that moves no more bytes, and multiplies no more, than the largest listed ones."""
    most = {k: max(work(c)[k] for c in listed()) for k in ("bytes", "flops")}
    while True:
        case = _draw_one(rng)
        w = work(case)
        if all(w[k] <= most[k] for k in most):
            return case


def _counts(case):
    """Rows per expert: Zipf popularity with a few experts that no token chose."""
    experts = case["experts"]
    return configs.zipf_counts(case["tokens"] * case["topk"], experts, seed=case["counts_seed"],
                               n_empty=max(1, experts // 64))


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape, scale=1.0, dtype=torch.bfloat16):
        return torch.randn(*shape, generator=gen, device="cuda").mul_(scale).to(dtype)

    def uniform(*shape, bf16=False):
        return torch.rand(*shape, generator=gen, device="cuda").to(torch.bfloat16 if bf16 else torch.float32)

    def hidden(M, n):
        """A residual stream: normal entries, a few channels a hundred times larger, as in trained models."""
        x = normal(M, n)
        x[:, torch.randperm(n, generator=gen, device="cuda")[:8]] *= 100.0
        return x

    def gate_up(M, f):
        x = normal(M, 2 * f)
        x.view(-1)[torch.randint(0, x.numel(), (max(1, x.numel() // 1000),), generator=gen, device="cuda")] *= 50.0
        return x

    def gamma(n):
        return (1.0 + 0.1 * torch.randn(n, generator=gen, device="cuda")).to(torch.bfloat16)

    op, s = case["op"], dict(case)
    if op == "infer":
        s.update(x=hidden(case["M"], case["n"]), gamma=gamma(case["n"]), h=gate_up(case["M"], case["f"]),
                 a=normal(case["M"], case["n"]))
    elif op in ("norm_quant", "norm_recompute"):
        s.update(x=hidden(case["M"], case["n"]), gamma=gamma(case["n"]))
    elif op == "bf16_step":
        M, n, f = case["M"], case["n"], case["f"]
        s.update(x=hidden(M, n), gamma=gamma(n), dy=normal(M, n, scale=1e-3), h=gate_up(M, f),
                 weight=uniform(M, 1, bf16=case["wbf16"]), dh=normal(M, f, scale=1e-3))
    elif op == "swiglu_step":
        s.update(h=gate_up(case["M"], case["f"]), dh=normal(case["M"], case["f"], scale=1e-3))
    elif op in ("experts_step", "dispatch"):
        counts = _counts(case)
        # which expert is popular differs from input to input; the sizes of the outputs do not
        order = torch.randperm(case["experts"], generator=torch.Generator().manual_seed(seed)).tolist()
        s["splits"] = splits = [counts[i] for i in order]
        s["counts"] = torch.tensor(splits, dtype=torch.int64, device="cuda")
        if op == "experts_step":
            M = sum(splits)
            s.update(h=gate_up(M, case["f"]), dh=normal(M, case["f"], scale=1e-3),
                     weight=uniform(M, 1, bf16=case["wbf16"]))
        else:
            padded = [(c + 15) // 16 * 16 for c in splits]
            s["padded"], s["padded_counts"] = padded, torch.tensor(padded, dtype=torch.int64, device="cuda")
            # every routed row names a random token; the padding entries behind an expert's rows are 0
            index = torch.randint(0, case["tokens"], (sum(padded),), generator=gen, device="cuda", dtype=torch.int32)
            start = torch.tensor([0] + padded[:-1]).cumsum(0).cuda()
            expert = torch.repeat_interleave(torch.arange(case["experts"], device="cuda"), s["padded_counts"])
            place = torch.arange(sum(padded), device="cuda") - start[expert]
            s["indices"] = torch.where(place < s["counts"][expert], index, torch.zeros_like(index))
            s.update(x=normal(case["tokens"], case["n"]), probs=uniform(case["tokens"], case["experts"]),
                     dy=normal(sum(padded), case["n"], scale=1e-3))
    elif op == "linear":
        s.update(x=normal(case["M"], case["n"]), w=normal(case["out"], case["n"], scale=0.02))
    else:
        s.update(x=hidden(case["M"], case["K"]), gamma=gamma(case["K"]),
                 w=normal(case["N"], case["K"], scale=0.02, dtype=torch.float32 if case["fp32"] else torch.bfloat16))
    return s


def run(state):
    s = state
    op, pow2 = s["op"], s.get("pow2", False)
    if op == "infer":
        q, scale, rms, _, _ = triton_rms_norm_and_block_quant_forward(s["x"], s["gamma"], round_scale=pow2, output_mode=0)
        a = triton_group_quant(s["a"], round_scale=pow2)
        h = triton_silu_and_block_quant_forward(s["h"], round_scale=pow2, output_mode=0)
        return q, scale, rms, a, h[:2]
    if op == "norm_quant":
        return triton_rms_norm_and_block_quant_forward(s["x"], s["gamma"], round_scale=pow2)
    if op == "norm_recompute":
        q, scale, rms, _, _ = triton_rms_norm_and_block_quant_forward(s["x"], s["gamma"], round_scale=pow2, output_mode=0)
        again = triton_rms_norm_and_block_quant_forward(s["x"], s["gamma"], rms=rms, round_scale=pow2, output_mode=1)
        return q, scale, rms, again[3], again[4]
    if op == "bf16_step":
        y, rms = triton_rms_norm_forward(s["x"], s["gamma"])
        h = triton_weighted_silu_forward(s["h"], s["weight"])
        dh, dweight = triton_weighted_silu_backward(s["dh"], s["h"], s["weight"])
        dx, dgamma = triton_rms_norm_backward(s["dy"], s["x"], s["gamma"], rms=rms)
        return y, rms, h, dh, dweight, dx, dgamma
    if op == "swiglu_step":
        return (triton_silu_and_block_quant_forward(s["h"], round_scale=pow2),
                triton_silu_and_block_quant_backward(s["dh"], s["h"], round_scale=pow2))
    if op == "experts_step":
        plan = build_expert_plan(s["counts"], s["splits"]) if s["plan"] else None
        return (triton_batch_weighted_silu_and_block_quant_forward(s["h"], s["weight"], s["counts"], s["splits"],
                                                                   round_scale=pow2, plan=plan),
                triton_batch_weighted_silu_and_block_quant_backward(s["dh"], s["h"], s["weight"], s["counts"],
                                                                    s["splits"], round_scale=pow2, plan=plan))
    if op == "dispatch":
        return (triton_batch_block_pad_permute_with_indices(s["x"], s["counts"], s["indices"], s["splits"],
                                                            probs=s["probs"], round_scale=pow2),
                triton_batch_blockwise_quant(s["dy"], s["padded_counts"], s["padded"], round_scale=pow2))
    if op == "linear":
        return triton_blockwise_quant(s["x"], round_scale=pow2), triton_block_quant(s["w"], round_scale=pow2)
    y, rms, logits, q, scale, _, _ = triton_rms_norm_fp32_gemm_block_quant_forward(s["x"], s["gamma"], s["w"],
                                                                                   round_scale=pow2)
    return y, rms, logits, q, scale


def work(case):
    """Every input read once, every output written once; the only operations counted are the router's products
    (the element-wise arithmetic of the other calls is below 30 operations a byte)."""
    op, flops = case["op"], 0
    if op == "infer":
        M, n, f = case["M"], case["n"], case["f"]
        rw = [configs.rw_rmsnorm_quant(M, n, 0), configs.rw_swiglu_fwd(M, f, 0), (2 * M * n, M * n + 4 * M * (n // 128))]
    elif op == "norm_quant":
        rw = [configs.rw_rmsnorm_quant(case["M"], case["n"])]
    elif op == "norm_recompute":
        rw = [configs.rw_rmsnorm_quant(case["M"], case["n"], 0), configs.rw_rmsnorm_quant(case["M"], case["n"], 1)]
    elif op == "bf16_step":
        M, n, f = case["M"], case["n"], case["f"]
        rw = [(2 * M * n + 2 * n, 2 * M * n + 4 * M), configs.rw_rmsnorm_bwd(M, n), configs.rw_weighted_silu(M, f, False),
              configs.rw_weighted_silu(M, f, True)]
    elif op == "swiglu_step":
        rw = [configs.rw_swiglu_fwd(case["M"], case["f"]), configs.rw_swiglu_bwd(case["M"], case["f"])]
    elif op == "experts_step":
        M, counts = case["tokens"] * case["topk"], _counts(case)
        rw = [configs.rw_batched_swiglu_fwd(M, case["f"], counts), configs.rw_batched_swiglu_bwd(M, case["f"], counts)]
    elif op == "dispatch":
        n, counts = case["n"], _counts(case)
        routed, padded = sum(counts), sum((c + 15) // 16 * 16 for c in counts)
        blocks = sum((c + 127) // 128 for c in counts)
        once = min(routed, case["tokens"])  # a token that several experts take is read once
        rw = [(2 * once * n + 4 * padded + 4 * routed, 2 * padded * n + 4 * padded * (n // 128) + 4 * blocks * n + 4 * padded),
              (2 * padded * n, 2 * padded * n + 4 * padded * (n // 128) + 4 * blocks * n)]
    elif op == "linear":
        M, n, out = case["M"], case["n"], case["out"]
        rw = [(2 * M * n, 2 * M * n + 4 * M * (n // 128) + 4 * ((M + 127) // 128) * n), (2 * out * n, out * n)]
    else:
        M, N, K = case["M"], case["N"], case["K"]
        rw = [(2 * M * K + (4 if case["fp32"] else 2) * N * K, 3 * M * K + 4 * M * N + 4 * (K // 128) * M + 4 * M)]
        flops = 2.0 * M * N * K
    return {"bytes": float(sum(r + w for r, w in rw)), "flops": float(flops)}


def tolerance(case):
    """The plain quantisers are exact.  Behind a floating-point sum or a sigmoid two correct evaluations differ in
    the last bit of a scale or a value, which moves a few codes in ten thousand by one step (an eighth of the
    value).  Measured against the same expressions in 64 bits: codes behind an RMSNorm 9e-4 (rows with outlier
    channels have most of their codes among the smallest), behind a SwiGLU 1.8e-4, bf16 results one rounding."""
    op = case["op"]
    if op in ("dispatch", "linear"):
        return "exact"
    if op == "bf16_step":
        return {"rel": 2e-3, "max": 0.016}
    return {"rel": 7e-4 if op in ("swiglu_step", "experts_step") else 3e-3, "max": 0.13}


def exact(case, seed):
    """What run() returns, in 64-bit arithmetic and plain torch: scales and values unrounded, codes the FP8 value
    nearest to the 64-bit quotient."""
    s, f64, fp8, fmax = prepare(case, seed), torch.float64, torch.float8_e4m3fn, 448.0
    op, pow2 = case["op"], case.get("pow2", False)

    def scale_of(amax):
        scale = (amax / fmax).clamp_min(1e-30)
        return torch.exp2(torch.ceil(torch.log2(scale))) if pow2 else scale

    def codes(v):
        return v.to(fp8).to(f64)

    def rows(v):  # codes [M, n], scales [M, n/128]
        g = v.view(v.shape[0], -1, 128)
        scale = scale_of(g.abs().amax(2))
        return codes((g / scale[:, :, None]).view(v.shape)), scale

    def columns(v):  # codes [n, M], scales [ceil(M/128), n]
        M, n = v.shape
        g = torch.nn.functional.pad(v, (0, 0, 0, -M % 128)).view(-1, 128, n)
        scale = scale_of(g.abs().amax(1))
        return codes((g / scale[:, None, :]).view(-1, n)[:M].t().contiguous()), scale

    def both(v):
        q, scale = rows(v)
        return q, scale.t().contiguous(), *columns(v)

    def experts(v, splits):  # the flat pieces of the experts one after the other
        out, pos = [[], [], [], []], 0
        for p in splits:
            for k, piece in enumerate(both(v[pos:pos + p]) if p else ()):
                out[k].append(piece if k in (0, 3) else piece.reshape(-1))
            pos += p
        return [torch.cat(o) for o in out]

    def norm(x, gamma):
        x = x.to(f64)
        r = 1.0 / torch.sqrt((x * x).mean(1) + 1e-6)
        return x * r[:, None] * gamma.to(f64), r

    def silu(h, weight=None):
        h1, h2 = h.to(f64).chunk(2, 1)
        y = torch.sigmoid(h1) * h1 * h2
        return y if weight is None else y * weight.to(f64).view(-1, 1)

    def silu_back(dh, h, weight=None):
        h1, h2 = h.to(f64).chunk(2, 1)
        sig, d = torch.sigmoid(h1), dh.to(f64)
        w = 1.0 if weight is None else weight.to(f64).view(-1, 1)
        dx = torch.cat([d * w * h2 * sig * (1.0 + h1 * (1.0 - sig)), d * w * sig * h1], 1)
        return dx, None if weight is None else (d * sig * h1 * h2).sum(1).view(weight.shape)

    def swap(t):  # scales of row-wise codes, one row per 128 columns
        return t[0], t[1].t().contiguous()

    if op == "infer":
        y, r = norm(s["x"], s["gamma"])
        return (*swap(rows(y)), r, rows(s["a"].to(f64)), swap(rows(silu(s["h"]))))
    if op in ("norm_quant", "norm_recompute"):
        y, r = norm(s["x"], s["gamma"])
        q, scale, qt, st = both(y)
        return q, scale, r, qt, st
    if op == "bf16_step":
        y, r = norm(s["x"], s["gamma"])
        dh, dweight = silu_back(s["dh"], s["h"], s["weight"])
        x, d = s["x"].to(f64), s["dy"].to(f64)
        xhat, g = x * r[:, None], d * s["gamma"].to(f64)
        dx = (g - xhat * (g * xhat).mean(1, keepdim=True)) * r[:, None]
        return y, r, silu(s["h"], s["weight"]), dh, dweight, dx, (d * xhat).sum(0)
    if op == "swiglu_step":
        return both(silu(s["h"])), both(silu_back(s["dh"], s["h"])[0])
    if op == "experts_step":
        n = case["f"]
        q, scale, qt, st = experts(silu(s["h"], s["weight"]), s["splits"])
        dx, dweight = silu_back(s["dh"], s["h"], s["weight"])
        dq, dscale, dqt, dst = experts(dx, s["splits"])
        return ((q, scale.view(-1, n // 128), qt.view(-1, n), st),
                (dq, dscale.view(-1, n // 64), dweight, dqt.view(-1, 2 * n), dst))
    if op == "dispatch":
        n, index = case["n"], s["indices"].long()
        starts = [sum(s["padded"][:e]) for e in range(case["experts"])]
        real = torch.zeros(len(index), dtype=torch.bool, device="cuda")
        probs = torch.zeros(len(index), dtype=f64, device="cuda")
        for e, (at, c) in enumerate(zip(starts, s["splits"])):
            real[at:at + c] = True
            probs[at:at + c] = s["probs"][index[at:at + c], e].to(f64)
        v = torch.where(real[:, None], s["x"][index].to(f64), torch.zeros((), dtype=f64, device="cuda"))
        q, scale, qt, st = experts(v, s["padded"])
        dq, dscale, dqt, dst = experts(s["dy"].to(f64), s["padded"])
        return ((q, scale.view(-1, n // 128), qt.view(-1, n), st, probs), (dq, dscale, dqt, dst.reshape(-1)))
    if op == "linear":
        w = s["w"].to(f64).view(case["out"] // 128, 128, case["n"] // 128, 128)
        scale = scale_of(w.abs().amax((1, 3)))
        return both(s["x"].to(f64)), (codes(w / scale[:, None, :, None]).view(s["w"].shape), scale)
    y, r = norm(s["x"], s["gamma"])
    return (y, r, y @ s["w"].to(f64).t(), *swap(rows(y)))
