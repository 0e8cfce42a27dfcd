"""Dense causal prefill attention on MI355X (libstarkv_hip.so, starkv_prefill_attention).

The attention half of the STAR-KV layer's prefill (starkv_serve/attention.py:219-251 in
the reference, which hands the lifted K and V to vLLM's flash_attn_varlen_func with
causal=True): every prompt attends to itself, no cached context.
"""
import ctypes
from typing import List, Optional

import torch

from starkv_serve import _hip


def block_list(query_lens: List[int]) -> List[int]:
    """The kernel's workgroup rows, (prompt, query block) pairs flattened, from the
    library's host helper starkv_prefill_block_list (the query block size is the
    kernel's): the blocks with the most keys first."""
    cu = [0]
    for L in query_lens:
        if L < 0:
            raise ValueError(f"negative prompt length {L}")
        cu.append(cu[-1] + int(L))
    lib = _hip.lib()
    cu_c = (ctypes.c_int32 * len(cu))(*cu)
    n = lib.starkv_prefill_block_list(cu_c, len(query_lens), None, 0)
    buf = (ctypes.c_int32 * (2 * max(n, 1)))()
    if n < 0 or lib.starkv_prefill_block_list(cu_c, len(query_lens), buf, n) != n:
        raise RuntimeError("starkv_prefill_block_list failed")
    return list(buf)[:2 * n]


def prompt_tables(query_lens: List[int], device) -> tuple:
    """(cu_seqlens [P + 1], blocks [num_blocks, 2]) int32 on `device`, in one upload."""
    cu = [0]
    for L in query_lens:
        cu.append(cu[-1] + int(L))
    meta = torch.tensor(cu + block_list(query_lens), dtype=torch.int32).to(device, non_blocking=True)
    return meta[:len(cu)], meta[len(cu):].view(-1, 2)


def prefill_lift(k_codes: torch.Tensor, v_codes: torch.Tensor, cu_seqlens: torch.Tensor, k_up: torch.Tensor,
                 k_offsets: torch.Tensor, k_widths: torch.Tensor, cos_sin: torch.Tensor) -> tuple:
    """The step's lifted keys and the V codes in fp16 (V's product's left operand), in one
    launch (starkv_prefill_lift): K [T, H_kv, 128] = RoPE(codes @ U), formed in fp32 and
    rounded once to fp16.

    k_codes [T, W], v_codes [T, r_v] (bf16, fp16 or fp32, contiguous rows); k_up [W, 128]
    fp32, rank-major; cos_sin [positions, 128] covering the longest prompt. fp16 V codes
    are returned as they are."""
    T = k_codes.shape[0]
    _hip.require_cuda(k_codes, v_codes, cu_seqlens, k_up, k_offsets, k_widths, cos_sin)
    key = torch.empty(T, k_offsets.numel(), 128, dtype=torch.float16, device=k_codes.device)
    if v_codes.dtype != k_codes.dtype:
        v_codes = v_codes.to(torch.float16)
    v16 = None
    if v_codes.dtype != torch.float16:
        v16 = torch.empty(v_codes.shape, dtype=torch.float16, device=v_codes.device)
    _hip.ops().prefill_lift(k_codes, v_codes, cu_seqlens, k_up, k_offsets, k_widths, cos_sin, key, v16)
    return key, v_codes if v16 is None else v16


def prefill_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, query_lens: List[int], scale: float,
                      out: Optional[torch.Tensor] = None, tables: Optional[tuple] = None) -> torch.Tensor:
    """Causal attention of each prompt to itself.

    q [T, H_q, 128] (bf16, fp16 or fp32); k, v [T, H_kv, 128] (converted to fp16 once
    here when they are not); query_lens: the prompts' token counts (host ints, summing to
    T); tables: their ``prompt_tables``, when the caller has them. Returns ``out``
    [T, H_q, 128] (new, in q's dtype, when not given)."""
    T, Hq, D = q.shape
    assert D == 128 and k.shape == v.shape and k.shape[0] == T and k.shape[2] == D and Hq % k.shape[1] == 0
    assert sum(query_lens) == T
    if out is None:
        out = torch.empty_like(q)
    if T == 0:
        return out
    _hip.require_cuda(q, k, v, out)
    if k.dtype == v.dtype and k.dtype in (torch.bfloat16, torch.float32) and k.stride(-1) == v.stride(-1) == 1:
        kv = torch.empty((2, *k.shape), dtype=torch.float16, device=k.device)
        _hip.ops().prefill_to_half(k, v, kv[0], kv[1])
        k, v = kv[0], kv[1]
    k, v = k.to(torch.float16), v.to(torch.float16)
    q = q if q.stride(-1) == 1 else q.contiguous()
    k, v = k.contiguous(), v.contiguous()
    cu_d, blk_d = prompt_tables(query_lens, q.device) if tables is None else tables
    _hip.ops().prefill(q, k, v, cu_d, blk_d, float(scale), out)
    return out
