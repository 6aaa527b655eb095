"""``fused_gelu_mlp`` and ``fused_qkv_norm_rottary`` with the signatures of nunchaku/ops/fused.py:10-110."""

from __future__ import annotations

import ctypes

import torch

from .. import _native as nv
from .. import packing
from . import gemm as _gemm_op
from .gemm import svdq_gemm_w4a4
from .quantize import svdq_quantize_w4a4_act_fuse_lora


def fused_gelu_mlp(x: torch.Tensor, fc1, fc2, pad_size: int = 256) -> torch.Tensor:
    """fc1 -> GELU -> fc2 with the GELU, fc2's activation quantization (unsigned INT4 after a
    +0.171875 shift) and fc2's low-rank down projection fused into fc1's GEMM epilogue
    (nunchaku/ops/fused.py:10-47).  All launches come from one call into the host extension once the layers are converted."""
    c1, c2 = fc1._call, fc2._call
    if c1 is not None and c2 is not None:
        y = nv.host().gelu_mlp(c1.handle, fc1, c2.handle, fc2, x, pad_size, _gemm_op.K_SPLIT or 0, _gemm_op.NO_ALLOC)
        if y is not None:
            return y
    # the first call, one on changed parameters, or one the extension has no fast way for: convert and check
    batch_size, seq_len, channels = x.shape
    M = batch_size * seq_len
    x2 = x.view(M, channels)
    if pad_size % 256 != 0:
        raise ValueError("pad_size must be a multiple of 256")
    if fc1.out_features != fc2.in_features or fc1.precision != fc2.precision:
        raise ValueError(f"fc2 ({fc2}) does not take what fc1 ({fc1}) gives")
    if M == 0:
        return x.new_empty(batch_size, seq_len, fc2.out_features)
    c1 = fc1._prepared(x2)
    dev = c1.device
    c2 = fc2._blocks(dev)
    y = nv.host().gelu_mlp(c1.handle, fc1, c2.handle, fc2, x, pad_size, _gemm_op.K_SPLIT or 0, _gemm_op.NO_ALLOC)
    if y is not None:
        return y
    t1, t2 = c1.tensors, c2.tensors
    fp4 = fc1.precision == "nvfp4"
    act, ascales, lora_act = svdq_quantize_w4a4_act_fuse_lora(x2, lora_down=t1["proj_down"], smooth=t1["smooth_factor"], fp4=fp4, pad_size=pad_size)
    M_pad = act.shape[0]
    qout = torch.empty(M_pad, packing.act_nbytes_per_row(fc2.in_features, fp4), dtype=torch.uint8, device=dev)
    oscales = torch.empty(fc2.in_features // fc2.group_size, M_pad, dtype=ascales.dtype, device=dev)
    lora_out = torch.empty(M_pad, fc2.rank, dtype=torch.float32, device=dev)
    svdq_gemm_w4a4(
        act=act, wgt=t1["qweight"], qout=qout, ascales=ascales, wscales=t1["wscales"], oscales=oscales, lora_act_in=lora_act, lora_up=t1["proj_up"],
        lora_down=t2["proj_down"], lora_act_out=lora_out, bias=t1["bias"], smooth_factor=t2["smooth_factor"], fp4=fp4, alpha=fc1.alpha,
        wcscales=t1["wcscales"], act_unsigned=fc1.act_unsigned, lora_scales=fc1.lora_scales,
    )
    output = torch.empty(M, fc2.out_features, dtype=x.dtype, device=dev)
    fc2.forward_quant(qout, oscales, lora_out, output)
    return output.view(batch_size, seq_len, -1)


def fused_qkv_norm_rottary(x: torch.Tensor, proj, norm_q, norm_k, rotary_emb: torch.Tensor, output=None, attn_tokens: int = 0):
    """QKV projection with the RMS norm of q and k (per 128-wide head) and the rotary embedding fused
    into the GEMM epilogue (nunchaku/ops/fused.py:50-110).  ``norm_q`` / ``norm_k`` are modules with a
    bf16 ``weight`` of 128 elements, ``rotary_emb`` is the table packed by ``pack_rotemb``.

    ``output``: None or a bf16 tensor: q | k | v side by side, one row per token.  A tuple (q, k, v) of
    fp16 [1, heads, tokens_pad, 128] tensors: the three apart, per head, rows from ``attn_tokens`` on
    masked (see ``svdq_gemm_w4a4``)."""
    batch_size, seq_len, channels = x.shape
    x2 = x.view(batch_size * seq_len, channels)
    c = proj._call
    if c is None:
        c = proj._prepared(x2)
    if output is None or isinstance(output, tuple):
        rot = packing.native(rotary_emb, "rotemb")
        y = nv.host().qkv_norm_rope(c.handle, proj, x, norm_q.weight, norm_k.weight, rot, output, attn_tokens, _gemm_op.NORM_EPS, _gemm_op.K_SPLIT or 0,
                                    _gemm_op.NO_ALLOC)
        if y is not None:
            return y
    c = proj._prepared(x2)
    quantized_x, ascales, lora_act = proj.quantize(x2)
    t = c.tensors
    common = dict(
        act=quantized_x, wgt=t["qweight"], ascales=ascales, wscales=t["wscales"], lora_act_in=lora_act, lora_up=t["proj_up"],
        bias=t["bias"], fp4=proj.precision == "nvfp4", alpha=proj.alpha, wcscales=t["wcscales"], norm_q=norm_q.weight,
        norm_k=norm_k.weight, rotary_emb=rotary_emb, lora_scales=proj.lora_scales,
    )
    if isinstance(output, tuple):
        if len(output) != 3:
            raise ValueError("a tuple `output` is (q, k, v)")
        svdq_gemm_w4a4(**common, out_q=output[0], out_k=output[1], out_v=output[2], attn_tokens=attn_tokens)
        return output
    if output is None:
        output = torch.empty(quantized_x.shape[0], proj.out_features, dtype=x.dtype, device=x.device)
    svdq_gemm_w4a4(**common, out=output)
    # (the reference views the padded buffer directly, which only works for token counts that need no padding)
    return output[: batch_size * seq_len].view(batch_size, seq_len, -1)


def linearattn_vk_mul_q(q: torch.Tensor, vk: torch.Tensor, num_tokens: int | None = None, eps: float = 1e-6) -> torch.Tensor:
    """Second half of the linear attention: ``q[b, t, h] <- (vk[b, h, :32] @ q[b, t, h]) / (vk[b, h, 32] . q[b, t, h] + eps)``
    in place (kernels::linearattn_vk_mul_q, gemm_w4a4_launch_impl.cuh:427-448).  q bf16 [B, tokens_pad, heads * 32]
    (``out_linearattn`` of ``svdq_gemm_w4a4``), vk fp32 [B, heads, 33, 32] (its ``out_vk``); only the first
    ``num_tokens`` rows of every batch entry are touched (all by default, as in the reference)."""
    if getattr(q, "is_cuda", False) and nv.host().vk_mul_q(q, vk, num_tokens, eps):  # (the plain case, with the same checks)
        return q
    nv.require_gpu(q, "q")
    nv.require_gpu(vk, "vk")
    if q.dim() != 3 or vk.dim() != 4 or q.dtype != torch.bfloat16 or vk.dtype != torch.float32:
        raise ValueError("q is bf16 [B, tokens_pad, heads * 32] and vk fp32 [B, heads, 33, 32]")
    B, tokens_pad, width = q.shape
    heads = vk.shape[1]
    if tuple(vk.shape) != (B, heads, 33, 32) or width != heads * 32 or vk.device != q.device:
        raise ValueError(f"vk has shape {tuple(vk.shape)}; q [{B}, {tokens_pad}, {width}] takes [{B}, {width // 32}, 33, 32] on the same device")
    num_tokens = tokens_pad if num_tokens is None else int(num_tokens)
    with torch.cuda.device(q.device):
        nv.check(nv.lib().svdq_linearattn_vk_mul_q(q.data_ptr(), vk.data_ptr(), B, num_tokens, tokens_pad, heads, ctypes.c_float(eps),
                                                   nv.stream_ptr(q.device)))
    return q
