"""The decoder layers' operations around the attention, on MI355X (csrc/model_ops.hip): RoPE
with the cache write of an uncompressed layer, the SiLU gate, and the weight products of a
decode step's few tokens (the reference runs these in vLLM's stock Llama,
starkv_serve/model.py:77-106 there)."""
from typing import Optional

import torch
from torch.autograd import forward_ad
from torch.utils._python_dispatch import is_in_torch_dispatch_mode

from starkv_serve import _hip
from starkv_serve.kernels.paged_decode import _as_i32

_FLOATS = (torch.bfloat16, torch.float16, torch.float32)


def _rows_ok(t: torch.Tensor) -> bool:
    """[T, heads, 128] rows that 16-byte loads can take."""
    step = 16 // t.element_size()
    return (t.dim() == 3 and t.shape[2] == 128 and t.stride(2) == 1 and t.stride(0) % step == 0
            and t.stride(1) % step == 0 and t.data_ptr() % 16 == 0)


def _traced() -> bool:
    """Under torch.compile (which cannot look into ``_plain``), torch.jit.trace or a dispatch mode (make_fx, fake
    tensors): what is recorded there are torch's operations."""
    return torch.compiler.is_compiling() or torch.jit.is_tracing() or is_in_torch_dispatch_mode()


def _plain(t: torch.Tensor) -> bool:
    """Not a subclass (a tracer's tensor), a transform's wrapper (vmap, jvp) or a dual tensor."""
    return (type(t) in (torch.Tensor, torch.nn.Parameter) and not torch._C._functorch.is_functorch_wrapped_tensor(t)
            and forward_ad.unpack_dual(t).tangent is None)


def rope_fits(cos_sin: torch.Tensor, positions: torch.Tensor, *rows: torch.Tensor) -> bool:
    """Whether the kernel takes these rows (q, and k and v): GPU tensors of one dtype, no gradient
    wanted in either direction, not traced or mapped."""
    if _traced() or (torch.is_grad_enabled() and any(t.requires_grad for t in rows)):
        return False
    if not all(_plain(t) for t in (cos_sin, positions, *rows)):
        return False
    return (all(t.is_cuda and t.dtype == rows[0].dtype and t.dtype in _FLOATS and _rows_ok(t) for t in rows)
            and all(t.device == rows[0].device for t in (cos_sin, positions, *rows)) and cos_sin.dtype in _FLOATS
            and cos_sin.dim() == 2 and cos_sin.shape[1] == 128 and cos_sin.is_contiguous()
            and cos_sin.data_ptr() % 16 == 0 and positions.dim() == 1 and positions.is_contiguous()
            and positions.dtype in (torch.int32, torch.int64) and positions.numel() == rows[0].shape[0])


def rope(positions: torch.Tensor, x: torch.Tensor, cos_sin: torch.Tensor) -> torch.Tensor:
    """x [T, H, 128] rotated at `positions` (fp32 arithmetic, x's dtype out)."""
    out = torch.empty(x.shape, dtype=x.dtype, device=x.device)
    if x.numel():
        _hip.ops().rope_qkv(x, None, None, positions, cos_sin, out, None, None, None, None, None, None)
    return out


def rope_write_fits(cos_sin: torch.Tensor, positions: torch.Tensor, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor,
                    k_cache: torch.Tensor, v_cache: torch.Tensor, slots: torch.Tensor) -> bool:
    """Whether ``rope_write`` may stand for the rotations and ``write_kv_full``: rows the kernel takes, and caches
    and slots that write_kv_full accepts (it refuses the others itself)."""
    bs = k_cache.shape[1]
    return (all(t.device == q.device for t in (k_cache, v_cache, slots))
            and k_cache.dtype == v_cache.dtype == q.dtype and q.dtype in (torch.bfloat16, torch.float16)
            and k_cache.shape == v_cache.shape and k_cache.shape[2:] == k.shape[1:] == v.shape[1:]
            and k_cache.stride() == v_cache.stride() and k_cache.stride(-1) == 1
            and all(s % 8 == 0 for s in k_cache.stride()[:3]) and (k_cache.data_ptr() | v_cache.data_ptr()) % 16 == 0
            and bs >= 16 and bs & (bs - 1) == 0 and rope_fits(cos_sin, positions, q, k, v))


def rope_write(positions: torch.Tensor, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, cos_sin: torch.Tensor,
               k_cache: torch.Tensor, v_cache: torch.Tensor, slots: torch.Tensor, keep_k: bool, half: bool) -> tuple:
    """An uncompressed layer's step in one launch: q and k rotated, k and v into their slots
    (``write_kv_full``). Returns (q, k when `keep_k`, and with `half` k and v in fp16, the
    prefill attention's operands)."""
    q_out = torch.empty(q.shape, dtype=q.dtype, device=q.device)
    k_out = torch.empty(k.shape, dtype=k.dtype, device=k.device) if keep_k else None
    kv16 = torch.empty((2, *k.shape), dtype=torch.float16, device=k.device) if half else (None, None)
    slots = slots.contiguous() if slots.dtype == torch.int64 else _as_i32(slots)
    _hip.ops().rope_qkv(q, k, v, positions, cos_sin, q_out, k_out, k_cache, v_cache, slots, kv16[0], kv16[1])
    return q_out, k_out, kv16[0], kv16[1]


def silu_mul(gate_up: torch.Tensor) -> torch.Tensor:
    """silu(gate) * up of gate_up [T, 2 I] (bf16 / fp16, I a multiple of 8)."""
    T, w = gate_up.shape
    out = torch.empty(T, w // 2, dtype=gate_up.dtype, device=gate_up.device)
    _hip.ops().silu_mul(gate_up, out)
    return out


def slots_fit(block_table: torch.Tensor, positions: torch.Tensor) -> bool:
    """Whether ``decode_slots`` takes this step: GPU tensors of a decode step's types, not traced or mapped."""
    return (not _traced() and positions.is_cuda and block_table.device == positions.device
            and positions.dtype == torch.int64 and positions.is_contiguous()
            and block_table.dtype in (torch.int32, torch.int64) and block_table.shape[0] >= positions.shape[0]
            and _plain(positions) and _plain(block_table))


def decode_slots(block_table: torch.Tensor, positions: torch.Tensor, block_size: int) -> tuple:
    """(slot_mapping int64, seq_lens int32) of a decode step at `positions` [n] int64."""
    slots = torch.empty_like(positions)
    lens = torch.empty(positions.shape, dtype=torch.int32, device=positions.device)
    _hip.ops().decode_slots(block_table, positions, int(block_size), slots, lens)
    return slots, lens


def greedy_fits(logits: torch.Tensor, tokens: torch.Tensor) -> bool:
    """Whether ``greedy_step`` takes these logits: rows that 16-byte loads can take."""
    return (tokens.dtype == torch.int64 and logits.dtype in _FLOATS and logits.stride(1) == 1
            and logits.stride(0) % 8 == 0 and logits.data_ptr() % 16 == 0)


def greedy_step(logits: torch.Tensor, tokens: torch.Tensor, positions: torch.Tensor) -> None:
    """tokens [n] = logits.argmax(-1) (the first of equals), positions [n] += 1, in place."""
    _hip.ops().greedy_step(logits, tokens, positions)


def few_fits(x: torch.Tensor, w: torch.Tensor, norm_weight: Optional[torch.Tensor] = None,
             residual: Optional[torch.Tensor] = None) -> bool:
    """Whether ``few_linear`` takes these operands, on one device: rows that 16-byte loads can take, K a multiple of a matrix
    step, no gradient wanted in either direction, not traced or mapped."""
    tensors = [t for t in (x, w, norm_weight, residual) if t is not None]
    if _traced() or (torch.is_grad_enabled() and any(t.requires_grad for t in tensors)):
        return False
    return (all(t.device == x.device and _plain(t) and t.stride(-1) == 1 and t.dtype == x.dtype for t in tensors)
            and all(t.stride(0) % 8 == 0 and t.data_ptr() % 16 == 0 for t in (x, w))
            and (norm_weight is None or norm_weight.data_ptr() % 16 == 0)
            and bool(_hip.lib().starkv_few_linear_fits(x.shape[0], x.shape[1])))


def few_linear(x: torch.Tensor, w: torch.Tensor, norm_weight: Optional[torch.Tensor] = None, eps: float = 0.0,
               h_out: Optional[torch.Tensor] = None, gate: bool = False,
               residual: Optional[torch.Tensor] = None) -> torch.Tensor:
    """x [n, K] @ w^T for n <= 16 tokens (starkv_few_linear): with `norm_weight` (bf16) x is
    normalised first (`h_out` receives it), `gate` gives silu(first half) * second half of w's
    rows, `residual` is added."""
    N = w.shape[0] // 2 if gate else w.shape[0]
    out = torch.empty(x.shape[0], N, dtype=x.dtype, device=x.device)
    mode = 2 if gate else 1 if residual is not None else 0
    _hip.ops().few_linear(x, w, norm_weight, float(eps), h_out, mode, residual, out)
    return out
