"""W8A16 group-128 operators and the HBM-resident expert dispatcher.

Drop-in for qwen35_deploy/operators/int8.py: same names, argument meaning and
error text.  The arithmetic runs in gfx950 HIP kernels (gemv.hip, gemm.hip,
route.hip) reached through the C ABI; there is no host or PyTorch fallback.

The reference's byte-budgeted host expert cache (ExpertCache, int8.py:51-124)
has no counterpart: the whole expert bank is resident in HBM, so an
Int8Experts module holds device tensors and builds its decode descriptor
table on the device without a host synchronisation.
"""
import functools

import torch

from .. import _lib
from . import w8a8 as _w8a8  # noqa: F401  (module-global swap target, cli.py:37-39)


def _require_int8_pair(q, scale):
    if q.dtype != torch.int8 or scale.dtype != torch.float32:
        raise ValueError('Invalid INT8 group geometry')
    if not (q.is_cuda and scale.is_cuda):
        raise ValueError('Invalid INT8 group geometry')
    if not (q.is_contiguous() and scale.is_contiguous()):
        raise ValueError('Invalid INT8 group geometry')


def linear(x, q, scale, large_tile=False):
    """y = x . bf16(q * s)^T with fp32 accumulation (int8.py:26-37).

    x: CUDA bf16/fp16 [..., K]; q int8 [N, K]; scale fp32 [N, K/128].
    One or two rows run the HBM-streaming GEMV, more the MFMA tiles their size
    selects; large_tile is taken like the reference's flag and has no effect.
    """
    if not x.is_cuda or x.dtype not in (torch.float16, torch.bfloat16):
        raise ValueError('W8A16 requires CUDA FP16/BF16 activations')
    n, k = q.shape
    shape = x.shape
    if k % 128 or shape[-1] != k or scale.shape != (n, k // 128):
        raise ValueError('Invalid INT8 group geometry')
    _require_int8_pair(q, scale)
    x = x.contiguous()
    out = x.new_empty((*shape[:-1], n))
    _lib.call('lm_w8a16_linear', x.data_ptr(), q.data_ptr(), scale.data_ptr(), out.data_ptr(),
              x.numel() // k, n, k, _lib.dtype_code(x.dtype), 1 if large_tile else 0,
              _lib.stream(x.device))
    return out


class Int8Linear(torch.nn.Module):
    """nn.Linear replacement holding int8 weights and fp32 group scales (int8.py:40-48)."""

    def __init__(self, q, scale):
        super().__init__()
        self.register_buffer('q', q)
        self.register_buffer('scale', scale)
        self.large_prefill_tile = False

    def forward(self, x):
        buffers = self._buffers  # skips two module attribute searches
        if 'q' in buffers and 'scale' in buffers:
            return linear(x, buffers['q'], buffers['scale'], self.large_prefill_tile)
        return linear(x, self.q, self.scale, self.large_prefill_tile)


def _check_weights(weights, experts):
    if not weights.is_cuda or weights.numel() < experts:
        raise ValueError('Expected CUDA routing weights of every selected expert')
    return weights.contiguous()


def grouped_linear(x, table, experts, n, field, shared):
    """W8A16 grouped decode GEMV over a device descriptor table (int8.py:233-237).

    table: CUDA int64 [experts, 5] = [gate_up.q, gate_up.s, down.q, down.s, slot]
    data pointers; row e reads x row 0 if shared else row e.
    """
    if not x.is_cuda or x.dtype not in (torch.float16, torch.bfloat16):
        raise ValueError('W8A16 requires CUDA FP16/BF16 activations')
    x, table = x.contiguous(), _lib.device_table(table, experts)
    out = torch.empty((experts, n), dtype=x.dtype, device=x.device)
    _lib.call('lm_w8a16_grouped_gemv', x.data_ptr(), table.data_ptr(), out.data_ptr(),
              experts, n, x.shape[-1], field, int(bool(shared)), _lib.dtype_code(x.dtype),
              _lib.stream(x.device))
    return out


def ordered_reduce(values, table, weights, out=None):
    """Decode combine (int8.py:240-250): acc = T(acc + T(v_e * w[slot_e])).

    values [E_sel, N] (bf16 or fp16, T) in ascending-expert table order;
    weights [1, top_k] (bf16, fp16 or fp32); returns [1, N] in T.
    """
    experts, n = values.shape
    table, weights = _lib.device_table(table, experts), _check_weights(weights, experts)
    if out is None:
        out = torch.empty((1, n), dtype=values.dtype, device=values.device)
    _lib.call('lm_ordered_reduce', values.contiguous().data_ptr(), table.data_ptr(),
              weights.data_ptr(), _lib.dtype_code(weights.dtype), out.data_ptr(), n, experts,
              _lib.dtype_code(values.dtype), _lib.stream(values.device))
    return out


def swiglu(gu):
    """T(T(silu(gate)) * up) over the two halves of the last dim, T = gu.dtype."""
    gu = gu.contiguous()
    half = gu.shape[-1] // 2
    out = torch.empty((*gu.shape[:-1], half), dtype=gu.dtype, device=gu.device)
    _lib.call('lm_swiglu', gu.data_ptr(), out.data_ptr(), gu.numel() // gu.shape[-1], half,
              _lib.dtype_code(gu.dtype), _lib.stream(gu.device))
    return out


def _selection(ids):
    """The selected ids of one token as (flat contiguous tensor, element size)."""
    if not ids.is_cuda:
        raise ValueError('Expected CUDA routing IDs')
    if ids.dtype is not torch.int64 and ids.dtype is not torch.int32:
        ids = ids.to(torch.int64)
    return ids.reshape(-1).contiguous(), 8 if ids.dtype is torch.int64 else 4


def _bank_args(gate_up, down):
    gq, gs, dq, ds = gate_up['q'], gate_up['scale'], down['q'], down['scale']
    return (gq.data_ptr(), gs.data_ptr(), dq.data_ptr(), ds.data_ptr(), gq.stride(0),
            gs.stride(0), dq.stride(0), ds.stride(0))


def build_descriptors(gate_up, down, ids):
    """Decode descriptor table for one token, sorted by expert id (int8.py:164-179).

    Returns an int64 [top_k, 5] table of (gate_up.q, gate_up.s, down.q,
    down.s) data pointers of each selected expert of the HBM bank plus its
    slot, built on the device (no host read of the routing ids), by one kernel
    for a token's.  Ids in host memory give the same table there; the operators
    take it only on the GPU.
    """
    if not ids.is_cuda or ids.numel() > _RANKED_IDS:
        experts, slots = torch.sort(ids.reshape(-1), stable=True)
        experts = experts.to(torch.int64).clamp(0, gate_up['q'].shape[0] - 1)
        columns = [t.data_ptr() + experts * (t.stride(0) * t.element_size())
                   for t in (gate_up['q'], gate_up['scale'], down['q'], down['scale'])]
        return torch.stack([*columns, slots], dim=1)
    flat, size = _selection(ids)
    n = flat.numel()
    table = torch.empty((n, 5), dtype=torch.int64, device=flat.device)
    _lib.call('lm_expert_table', flat.data_ptr(), size, n, gate_up['q'].shape[0],
              *_bank_args(gate_up, down), table.data_ptr(), _lib.stream(flat.device))
    return table


# The kernel compares every id with every other: 10 us for 64 ids, 52 for 512, 400
# for 4096, where the sort and its arithmetic take about 90.
_RANKED_IDS = 512


@functools.lru_cache(maxsize=None)
def _decode_fits(n, hidden, intermediate):
    return bool(_lib.lib().lm_w8a16_experts_decode_fits(n, hidden, intermediate))


# The operators that the two-launch decode computes.
_w8a16_decode = (build_descriptors, grouped_linear, swiglu, ordered_reduce)


class Int8Experts(torch.nn.Module):
    """HF Qwen3_5MoeExperts replacement over an HBM-resident int8 bank (int8.py:127-210).

    gate_up = {'q': int8 [E, 2I, H], 'scale': fp32 [E, 2I, H/128]} and
    down = {'q': int8 [E, H, I], 'scale': fp32 [E, H, I/128]}, all on the GPU.
    forward(x, top_k_index, top_k_weights) keeps the HF contract
    (Experts.forward, HF:733-757):
      * M > 1 rows: prefill_pipeline.run if one is attached, else the
        device-planned routed MoE (gpu_routes.routed_moe);
      * M == 1: grouped decode - module-level grouped_linear (W8A16, or W8A8
        after `int8.grouped_linear = w8a8.grouped_linear`), SwiGLU, and the
        ordered bf16 combine in ascending expert order; while none of these
        module-level operators is replaced, in two fused launches with the
        same results.
    """

    def __init__(self, layer, gate_up, down, cache=None):
        super().__init__()
        self.layer, self.gate_up, self.down, self.cache = layer, gate_up, down, cache
        self.prefill_pipeline = None
        self.large_tile = False
        for bank in (gate_up, down):
            if not (bank['q'].is_cuda and bank['scale'].is_cuda):
                raise ValueError('Int8Experts needs an HBM-resident bank')

    def forward(self, x, top_k_index, top_k_weights):
        if x.shape[0] > 1:
            if self.prefill_pipeline is not None:
                return self.prefill_pipeline.run(self.layer, x, top_k_index, top_k_weights)
            from ..runtime import gpu_routes
            banks = [self.gate_up['q'], self.gate_up['scale'], self.down['q'], self.down['scale']]
            return gpu_routes.routed_moe(x, top_k_weights, top_k_index.contiguous(), banks,
                                         self.large_tile)
        hidden, intermediate, n = x.shape[-1], self.down['q'].shape[-1], top_k_index.numel()
        if ((build_descriptors, grouped_linear, swiglu, ordered_reduce) == _w8a16_decode
                and _decode_fits(n, hidden, intermediate)):
            return self._decode(x, top_k_index, n, top_k_weights, hidden, intermediate)
        table = build_descriptors(self.gate_up, self.down, top_k_index)
        experts = table.shape[0]
        gu = grouped_linear(x, table, experts, 2 * intermediate, 0, True)
        h = swiglu(gu)
        values = grouped_linear(h, table, experts, hidden, 2, False)
        return ordered_reduce(values, table, top_k_weights)

    def _decode(self, x, ids, n, weights, hidden, intermediate):
        """One token, W8A16: gate_up + SwiGLU, then down + combine, two launches
        with the results of the separate operators."""
        if not x.is_cuda or x.dtype not in (torch.float16, torch.bfloat16):
            raise ValueError('W8A16 requires CUDA FP16/BF16 activations')
        flat, size = _selection(ids)
        x, weights = x.contiguous(), _check_weights(weights, n)
        h = x.new_empty((n, intermediate))
        out = x.new_empty((1, hidden))
        _lib.call('lm_w8a16_experts_decode', x.data_ptr(), flat.data_ptr(), size, n,
                  self.gate_up['q'].shape[0], *_bank_args(self.gate_up, self.down),
                  weights.data_ptr(), _lib.dtype_code(weights.dtype), h.data_ptr(),
                  out.data_ptr(), hidden, intermediate, _lib.dtype_code(x.dtype),
                  _lib.stream(x.device))
        return out
