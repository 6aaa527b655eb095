"""What the speed of this framework is measured on: the quantized linear layers of a diffusion transformer, through the
entry points a model calls (``SVDQW4A4Linear``, ``fused_gelu_mlp``, ``fused_qkv_norm_rottary``, the linear-attention pair,
``AWQW4A16Linear``), from one row to the largest batches of the repository's own benchmark.

A pass is one call of one layer (or fused pair of layers) on activations that are already on the GPU.  Weights are loaded
and converted once, as a model does at load time; they are drawn like those of a quantized checkpoint (normal weights, one
scale per group), activations like a transformer's (normal, one channel in a hundred 20 times as large).

Kinds of case:

``linear``   one ``SVDQW4A4Linear`` forward: M rows, K -> N, rank R, INT4 or NVFP4
``mlp``      ``fused_gelu_mlp``: K -> N -> K with the GELU and the second layer's quantization in the first one's epilogue
``qkv``      ``fused_qkv_norm_rottary``: K -> N = 3 x heads x 128, q | k | v in one bf16 tensor or (``split``) three fp16 ones
``litela``   linear attention: projection with relu(q) and the vk sums in its epilogue, then vk times q
``awq``      ``AWQW4A16Linear`` on 1 .. 8 rows
"""

from __future__ import annotations

import math

import torch

from nunchaku_amd import packing
from nunchaku_amd.models.linear import AWQW4A16Linear, SVDQW4A4Linear
from nunchaku_amd.ops import fused_gelu_mlp, fused_qkv_norm_rottary, linearattn_vk_mul_q, svdq_gemm_w4a4

E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)


def listed():
    return [
        # The modulation vectors of a block (six of them, 3072 wide) for one image: once per block and step, pure latency
        # and weight traffic.
        dict(name="awq_modulation_1row", kind="awq", M=1, K=3072, N=18432),
        # The smallest layer of the benchmark: a few hundred tokens (a low-resolution image or a prompt), hidden size 3072.
        dict(name="linear_int4_256", kind="linear", M=256, K=3072, N=3072, R=32, fp4=False),
        # The same layer in NVFP4 on a ragged token count.
        dict(name="linear_nvfp4_300", kind="linear", M=300, K=3072, N=3072, R=32, fp4=True),
        # QKV projection of a prompt's tokens next to the image's, q | k | v side by side; an odd token count.
        dict(name="qkv_int4_505", kind="qkv", M=505, K=3072, N=9216, R=32, fp4=False, split=False),
        # The MLP of a quarter-size image in NVFP4, odd token count.
        dict(name="mlp_nvfp4_1157", kind="mlp", M=1157, K=3072, N=12288, R=32, fp4=True),
        # Linear attention at 4096 tokens, 72 heads of 32.
        dict(name="litela_int4_4096", kind="litela", B=1, T=4096, K=2304, N=6912, R=32, fp4=False),
        # The full-size image (4096 + 512 tokens) of a double block: QKV with q, k, v apart for the attention kernel ...
        dict(name="qkv_int4_4608", kind="qkv", M=4608, K=3072, N=9216, R=32, fp4=False, split=True),
        # ... the first MLP layer by itself, the benchmark's headline ...
        dict(name="linear_int4_4608", kind="linear", M=4608, K=3072, N=12288, R=32, fp4=False),
        # ... and the whole MLP.
        dict(name="mlp_int4_4608", kind="mlp", M=4608, K=3072, N=12288, R=32, fp4=False),
        # The two projections of a single block in NVFP4: wide output, long contraction.
        dict(name="linear_nvfp4_4608_wide", kind="linear", M=4608, K=3072, N=21504, R=32, fp4=True),
        dict(name="linear_nvfp4_4608_long", kind="linear", M=4608, K=15360, N=3072, R=32, fp4=True),
        # Four images in a batch, stock branch with a user's low-rank adapter appended (rank 128): the largest.
        dict(name="linear_int4_18432_r128", kind="linear", M=18432, K=3072, N=12288, R=128, fp4=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Another case of the same ranges: 16 .. 9216 tokens (any number), widths 1024 .. 15360 in steps of 128, ranks 16 .. 128,
    both precisions; no more work than the largest listed one."""
    most = 2.0 * 18432 * 3072 * 12288
    kind = rng.choice(["linear", "linear", "linear", "mlp", "mlp", "qkv", "qkv", "litela", "awq"])
    while True:
        fp4 = rng.random() < 0.4
        R = rng.choice([16, 32, 32, 32, 48, 64, 128])
        M = _log_int(rng, 16, 9216)
        if kind == "awq":
            return dict(kind="awq", M=rng.randint(1, 8), K=64 * _log_int(rng, 16, 64), N=128 * _log_int(rng, 16, 160))
        if kind == "linear":
            c = dict(kind="linear", M=M, K=128 * _log_int(rng, 8, 120), N=128 * _log_int(rng, 8, 168), R=R, fp4=fp4)
            ops = 2.0 * M * c["K"] * c["N"]
        elif kind == "mlp":
            k = 128 * _log_int(rng, 8, 32)
            c = dict(kind="mlp", M=M, K=k, N=4 * k, R=R, fp4=fp4)
            ops = 4.0 * M * c["K"] * c["N"]
        elif kind == "qkv":
            split = rng.random() < 0.5
            if split:
                M = max(256, M // 256 * 256)  # one tensor per q, k, v holds padded tokens: whole blocks
            k = 128 * _log_int(rng, 8, 32)
            c = dict(kind="qkv", M=M, K=k, N=3 * k, R=R, fp4=fp4, split=split)
            ops = 2.0 * M * c["K"] * c["N"]
        else:
            B = rng.choice([1, 1, 2])
            T = 256 * rng.choice([1, 2, 4, 4, 8, 16, 16])
            k = 128 * rng.randint(8, 20)
            c = dict(kind="litela", B=B, T=T, K=k, N=3 * k, R=R, fp4=False)
            ops = 2.0 * B * T * c["K"] * c["N"]
        if ops * (2.0 if fp4 else 1.0) <= most:
            return c


# ---- inputs -----------------------------------------------------------------------------------------------------------


def _int4_weights(N, K, g, dev):
    """Codes and scales of normal weights, one scale per 64 of a row; the storage order of a checkpoint permutes elements
    among themselves, which a sample of independent weights need not follow."""
    w = torch.randn(N * K // 64, 64, generator=g, device=dev)
    s = (0.02 / 7.0 * w.abs().amax(1)).to(torch.bfloat16)
    q = (0.02 * w / s.float()[:, None]).round_().clamp_(-7, 7).to(torch.int8).view(N, K)
    return (q[:, 0::2] & 15) | (q[:, 1::2] << 4), s.view(K // 64, N)


def _nvfp4_weights(N, K, g, dev):
    w = 0.02 * torch.randn(N * K // 16, 16, generator=g, device=dev)
    amax = w.abs().amax(1)
    wt = (amax.max() / (6.0 * 448.0)).to(torch.bfloat16)
    s = (amax / 6.0 / wt.float()).clamp_(max=448.0).to(torch.float8_e4m3fn)
    v = w / (s.float() * wt.float())[:, None].clamp_min(1e-30)
    grid = torch.tensor(E2M1, device=dev)
    code = torch.bucketize(v.abs(), (grid[1:] + grid[:-1]) / 2).to(torch.uint8)
    code |= (v < 0).to(torch.uint8) << 3
    code = code.view(N, K)
    return (code[:, 0::2] | (code[:, 1::2] << 4)).view(torch.int8), s.view(K // 16, N), wt.view(1)


def _layer(K, N, R, fp4, g, dev, act_unsigned=False):
    def normal(*shape):
        return (0.02 * torch.randn(*shape, generator=g, device=dev)).to(torch.bfloat16)

    m = SVDQW4A4Linear(K, N, rank=R, precision="nvfp4" if fp4 else "int4", act_unsigned=act_unsigned, device=dev)
    sd = dict(
        smooth_factor=(0.5 + 1.5 * torch.rand(K, generator=g, device=dev)).to(torch.bfloat16),
        smooth_factor_orig=torch.ones(K, dtype=torch.bfloat16, device=dev),
        proj_down=normal(K, R), proj_up=normal(N, R), bias=normal(N),
    )
    if fp4:
        sd["qweight"], sd["wscales"], sd["wtscale"] = _nvfp4_weights(N, K, g, dev)
        sd["wcscales"] = torch.ones(N, dtype=torch.bfloat16, device=dev)
    else:
        sd["qweight"], sd["wscales"] = _int4_weights(N, K, g, dev)
    m.load_state_dict(sd)
    m.native_tensors()  # the load-time conversion to the layouts of the kernels
    return m


def _activations(M, K, g, dev):
    x = torch.randn(M, K, generator=g, device=dev)
    x[:, torch.randperm(K, generator=g, device=dev)[: math.ceil(K / 100)]] *= 20.0
    return x.to(torch.bfloat16)


class _Norm:
    def __init__(self, weight):
        self.weight = weight


def prepare(case, seed):
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(seed)
    kind, K, N = case["kind"], case["K"], case["N"]
    state = {"case": case}
    if kind == "awq":
        m = AWQW4A16Linear(K, N, device=dev)
        w = 0.02 * torch.randn(K // 64, N, 64, generator=g, device=dev)
        lo, hi = w.amin(-1), w.amax(-1)
        s = ((hi - lo) / 15).to(torch.bfloat16)
        q = ((w - lo[..., None]) / s.float()[..., None]).round_().clamp_(0, 15).to(torch.uint8).view(-1)
        m.load_state_dict(dict(qweight=(q[0::2] | (q[1::2] << 4)).view(torch.int32).view(N // 4, K // 2), wscales=s, wzeros=lo.to(torch.bfloat16),
                               bias=(0.02 * torch.randn(N, generator=g, device=dev)).to(torch.bfloat16)))
        state.update(m=m, x=torch.randn(case["M"], K, generator=g, device=dev).to(torch.bfloat16))
        return state
    R, fp4 = case["R"], case["fp4"]
    state["m"] = _layer(K, N, R, fp4, g, dev)
    if kind == "litela":
        state["x"] = _activations(case["B"] * case["T"], K, g, dev)
        return state
    M = case["M"]
    state["x"] = _activations(M, K, g, dev).view(1, M, K)
    if kind == "mlp":
        state["m2"] = _layer(N, K, R, fp4, g, dev, act_unsigned=not fp4)
    if kind == "qkv":
        M_pad = (M + 255) // 256 * 256
        ang = 6.283 * torch.rand(M_pad, 64, generator=g, device=dev)
        # (the (sin, cos) pairs of a packed table stay adjacent: random angles in any order are such a table)
        state["rotary"] = packing.repack_rotemb(torch.stack((ang.sin(), ang.cos()), dim=-1).view(M_pad, 128))
        state["nq"] = _Norm((1.0 + 0.2 * torch.randn(128, generator=g, device=dev)).to(torch.bfloat16))
        state["nk"] = _Norm((1.0 + 0.2 * torch.randn(128, generator=g, device=dev)).to(torch.bfloat16))
        if case["split"]:  # the attention's inputs, which a model keeps
            state["out"] = tuple(torch.empty(1, N // 384, M_pad, 128, dtype=torch.float16, device=dev) for _ in range(3))
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear" or kind == "awq":
        return state["m"](state["x"])
    if kind == "mlp":
        return fused_gelu_mlp(state["x"], state["m"], state["m2"])
    if kind == "qkv":
        return fused_qkv_norm_rottary(state["x"], state["m"], state["nq"], state["nk"], state["rotary"],
                                      output=state.get("out"), attn_tokens=case["M"] if case["split"] else 0)
    m = state["m"]
    t = m.native_tensors()
    B, T, N = case["B"], case["T"], case["N"]
    act, asc, la = m.quantize(state["x"])
    q = torch.empty(B, T, N // 3, dtype=torch.bfloat16, device=act.device)
    vk = torch.empty(B, N // 96, 33, 32, dtype=torch.float32, device=act.device)
    svdq_gemm_w4a4(act=act, wgt=t["qweight"], ascales=asc, wscales=t["wscales"], lora_act_in=la, lora_up=t["proj_up"], bias=t["bias"],
                   out_vk=vk, out_linearattn=q)
    return linearattn_vk_mul_q(q, vk), vk


def _layer_work(M, K, N, R, fp4, x_in=True, out=True):
    scales = K * N / 16 if fp4 else 2.0 * K * N / 64
    return (K * N / 2.0 + scales + 2.0 * R * (K + N) + 2.0 * (K + N) + (2.0 * M * K if x_in else 0) + (2.0 * M * N if out else 0),
            2.0 * M * K * N + 2.0 * M * R * (K + N))


def work(case):
    kind, K, N = case["kind"], case["K"], case["N"]
    if kind == "awq":
        M = case["M"]
        return {"bytes": N * K / 2.0 + 4.0 * N * K / 64 + 2.0 * N + 2.0 * M * (K + N), "flops": 2.0 * M * N * K}
    R, fp4 = case["R"], case["fp4"]
    if kind == "mlp":
        b1, f1 = _layer_work(case["M"], K, N, R, fp4, out=False)
        b2, f2 = _layer_work(case["M"], N, K, R, fp4, x_in=False)
        return {"bytes": b1 + b2, "flops": f1 + f2}
    if kind == "litela":
        M = case["B"] * case["T"]
        b, f = _layer_work(M, K, N, R, fp4, out=False)
        heads = N // 96
        return {"bytes": b + 2.0 * M * N / 3 + 4.0 * case["B"] * heads * 33 * 32, "flops": f + 4.0 * M * heads * 33 * 32}
    b, f = _layer_work(case["M"], K, N, R, fp4)
    if kind == "qkv":
        b += 4.0 * case["M"] * 128
    return {"bytes": b, "flops": f}


def tolerance(case):
    # Largest differences between the path and itself with its sums in another order (tiles split along K in 1, 2 or 3 parts),
    # and between it and a 64-bit evaluation rounded to bf16 at the end, over both precisions, K = 3072 and 12288, ranks 32 and
    # 128: relative 5e-5, one element 7.3e-3 (a bf16 value that rounds the other way).  In the MLP such a value can also move
    # a 4-bit code of the second layer's input: 2.4e-4 and 1.1e-2.  Four times that.
    if case["kind"] == "mlp":
        return {"rel": 1e-3, "max": 0.045}
    return {"rel": 2e-4, "max": 0.03}
