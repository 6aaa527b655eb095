"""What the library would do with a GEMM call (csrc/internal_api.h, ``svdq_gemm_plan_of``): which kernel, and how it divides the
work.  Needs no GPU."""

import ctypes

from nunchaku_amd import _native as nv


class Plan(ctypes.Structure):
    """Mirror of ``svdq_gemm_plan``."""

    _fields_ = [(n, ctypes.c_int32) for n in ("few_rows", "row_blocks", "full_blocks", "half_blocks", "kparts", "workgroups", "shared_tiles", "columns", "shared_rows", "copied_ranks", "low_blocks")]

    def __repr__(self):
        return "Plan(" + ", ".join(f"{n}={getattr(self, n)}" for n, _ in self._fields_ if getattr(self, n)) + ")"


class Tile(ctypes.Structure):
    """Mirror of ``svdq_gemm_tile``."""

    _fields_ = [(n, ctypes.c_int32) for n in ("row", "rows", "column_block", "part", "row_block", "tile")]


def plan_of(args: nv.GemmArgs, rows: int = 0, compute_units: int = 256) -> Plan:
    """``rows``: of a call without ``out`` whose caller reads only these."""
    plan = Plan()
    nv.check(nv.lib().svdq_gemm_plan_of(ctypes.byref(args), ctypes.c_int64(rows), compute_units, ctypes.byref(plan)))
    return plan


def tile_of(plan: Plan, N: int, block: int) -> Tile:
    tile = Tile()
    nv.lib().svdq_gemm_int4_tile(ctypes.byref(plan), ctypes.c_int64(N), block, ctypes.byref(tile))
    return tile


def call(kind: str, M: int, K: int, N: int, R: int, fp4: bool, k_split: int = 0, aligned: bool = True, R_down: int = 48, with_out: bool = True,
         vk_rows: int = 256) -> nv.GemmArgs:
    """The argument block of a call as the Python operators make it; the addresses are never followed.  ``aligned`` False: a bias
    2 bytes off, which the few-rows kernel does not take."""
    P, M_pad = 1 << 20, (M + 255) // 256 * 256
    a = nv.GemmArgs(act=P, ascales=P, wgt=P, wscales=P, colnorm=P if fp4 else None, bias=P if aligned else P + 2, wcscales=P if fp4 else None, M_pad=M_pad, N=N, K=K,
                    M_out=M, N_out=N, R_up=R, alpha=1.0, fp4=int(fp4), k_split=k_split)
    if R:
        a.lora_act_in = a.lora_up = P
    if kind == "next":
        a.M_out = M_pad
        a.qout = a.oscales = a.next_smooth_rcp = P
        if R_down:
            a.next_lora_down = a.next_lora_act_out = P
            a.R_down = R_down
    if kind != "split" and with_out:
        a.out = P
    else:
        a.M_out = a.N_out = 0
    if kind == "silu":
        a.fuse_silu = 1
    if kind in ("rope", "split"):
        a.norm_q = a.norm_k = a.rotary_emb = P
        a.rot_rows = M_pad
    if kind == "split":
        a.out_q = a.out_k = a.out_v = P
        a.qkv_head_stride = (ctypes.c_int64 * 3)(*[M_pad * 128] * 3)
        a.qkv_rows, a.attn_tokens = M_pad, M
    if kind == "litela":
        a.out_vk, a.vk_rows, a.M_out, a.N_out = P, vk_rows, M_pad, N // 3
    return a
