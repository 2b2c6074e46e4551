"""INT4 group-wise weight quantisation with a fused dequant-GEMM.

Keeps the reference's "int4" format (nanoserve/quant.py:53-80): per output
row, groups of `group_size` consecutive input features share a float32 scale
and a uint8 zero point, codes are round(w / scale) + zero clamped to [0, 15],
and two codes share a byte (even input index in the low nibble).  The
quantiser is setup-time tensor code and follows the reference step for step,
so checkpoints quantised either way are interchangeable.

The difference is the forward.  The reference's QuantLinear expands the whole
weight to fp16 on every call and then runs F.linear (quant.py:149-158); here
`Int4Linear.forward` calls `ns_int4_linear`, which never writes the expanded
weight: up to FUSED_MAX_ROWS rows it dequantises each weight in registers on
its way into the MFMA, above that (prefill chunks) a tiled GEMM dequantises
each weight tile once per 64- or 128-token tile.
"""

from __future__ import annotations

import functools
import itertools

import torch
import torch.nn as nn
import torch.nn.functional as F

from . import _lib

# Up to this many rows ns_int4_linear dequantises inside its MFMA tiles (and
# can fuse the input RMSNorm and the rotary + cache-write epilogue); above it
# the library runs its tiled GEMM, which shares each dequantised weight tile
# among 128 tokens (each 64-row tile of the register path would repeat the
# dequantisation of its weight tile).
FUSED_MAX_ROWS = 128

# "auto" takes the dequantise + library GEMM steps instead of the tiled GEMM
# for layers whose K is at least LONG_K above LONG_K_TILED_MAX_ROWS rows, but
# only inside a graph capture.  The tiled GEMM's time grows with its K steps
# per workgroup, and past 1024 tokens the long-K layers have too many tiles to
# split that far: graph-replayed on MI355X, down_proj (K 4864, N 896, residual)
# takes 31.0 / 33.4 us tiled / dequantise + hipBLASLt at 1088 tokens, 41.2 /
# 39.3 at 2048 and 65.4 / 52.0 at 4096; K 8192, N 2048 67.7 / 64.0 at 1088 and
# 99.5 / 83.1 at 2048; K 14336, N 3584 163 / 142 and 286 / 212.
# Called eagerly, the steps' four to five launches and tensor ops cost more
# host time than the single launch saves on the device: the c5 engine (eager
# prefill chunks of up to 2048 tokens) measured TTFT p50 17.0-18.5 ms with
# them against 13.9-14.1 ms with the tiled GEMM, and 1% fewer output tokens/s.
# Short-K layers keep the tiled GEMM everywhere (gate|up at 2048 tokens 64.0
# against 94.5 us).
LONG_K = 2048
LONG_K_TILED_MAX_ROWS = 1024

# Dequantised-weight scratch per (device, stream), grown on demand.
_dequant_scratch: dict[tuple[int, int], torch.Tensor] = {}


@torch.inference_mode()
def int4_dequantize(qweight: torch.Tensor, scales: torch.Tensor, zeros: torch.Tensor, group_size: int,
                    dtype: torch.dtype, out: torch.Tensor | None = None) -> torch.Tensor:
    """The model-dtype weight [N, K] of an INT4 layer (reference dequantize_int4, bit for bit)."""
    N, half_k = qweight.shape
    K = 2 * half_k
    if out is None:
        out = torch.empty((N, K), dtype=dtype, device=qweight.device)
    elif out.shape != (N, K) or out.dtype != dtype or not out.is_contiguous():
        raise ValueError(f"out must be a contiguous [{N}, {K}] {dtype} tensor")
    rc = _lib.load().ns_int4_dequantize(out.data_ptr(), qweight.data_ptr(), scales.data_ptr(), zeros.data_ptr(),
                                        N, K, group_size, _lib.DTYPE_CODES[dtype],
                                        torch.cuda.current_stream(qweight.device).cuda_stream)
    _lib.check(rc, "ns_int4_dequantize")
    return out


def _scratch_key(device: torch.device) -> tuple[int, int]:
    return (device.index if device.index is not None else torch.cuda.current_device(),
            torch.cuda.current_stream(device).cuda_stream)


def _scratch_ready(device: torch.device, N: int, K: int, dtype: torch.dtype) -> bool:
    """Whether this stream's weight scratch already holds an N x K weight (no allocation needed)."""
    buf = _dequant_scratch.get(_scratch_key(device))
    return buf is not None and buf.numel() >= N * K * torch.tensor([], dtype=dtype).element_size()


def _scratch_weight(device: torch.device, N: int, K: int, dtype: torch.dtype) -> torch.Tensor:
    key = _scratch_key(device)
    buf = _dequant_scratch.get(key)
    need = N * K * torch.tensor([], dtype=dtype).element_size()
    if buf is None or buf.numel() < need:
        buf = torch.empty(need, dtype=torch.uint8, device=device)
        _dequant_scratch[key] = buf
    return buf[:need].view(dtype).view(N, K)


@torch.no_grad()
def quantize_int4_groupwise(w: torch.Tensor, group_size: int = 128):
    """w [out, in] -> (packed uint8 [out, in/2], scales f32 [out, G], zeros uint8 [out, G]).

    Same steps as the reference (quant.py:53-80): scale = (max - min) / 15
    clamped to 1e-8, zero = round(-min / scale) clamped to [0, 15],
    code = clamp(round(w / scale) + zero, 0, 15), round half to even.
    """
    out_f, in_f = w.shape
    if in_f % group_size != 0:
        raise ValueError(f"a weight with {in_f} input features splits into no whole number of {group_size}-wide groups")
    if in_f % 2 != 0:
        raise ValueError(f"INT4 packing stores input features in pairs per byte; {in_f} is odd")
    g = in_f // group_size
    wg = w.to(torch.float32).reshape(out_f, g, group_size)
    w_max = wg.amax(dim=2, keepdim=True)
    w_min = wg.amin(dim=2, keepdim=True)
    scale = ((w_max - w_min) / 15.0).clamp(min=1e-8)
    zero = (-w_min / scale).round().clamp(0, 15)
    q = ((wg / scale).round() + zero).clamp(0, 15).to(torch.uint8).reshape(out_f, in_f)
    packed = (q[:, 0::2] | (q[:, 1::2] << 4)).contiguous()
    return packed, scale.squeeze(2).contiguous(), zero.squeeze(2).to(torch.uint8).contiguous()


# The tiled GEMM's split layout depends on M only through its tile counts
# (ceil(M/128) and ceil(M/64) token tiles).  From 512 tiles of 128 x 128 it
# always takes those, and their last round repeats every 512 token tiles (two
# workgroups per CU on 256 CUs), so multiples of 64 rows up to twice that cover
# every token count.
_SPLITK_SCAN_ROWS = 2 * 512 * 128


@functools.lru_cache(maxsize=256)
def splitk_workspace_bytes(N: int, K: int) -> int:
    """Workspace bytes that cover every token count of an N x K layer.

    The fused kernel (1..FUSED_MAX_ROWS rows) splits K while its tiles are few;
    the tiled GEMM (above) splits the tiles of a last dispatch round that
    leaves slots of the device idle, which can happen at any token count, so
    the scan runs over every multiple of 64 rows up to the point where the
    GEMM's layouts repeat.  It depends on the two sizes alone and is kept by
    them: a model's layers share a handful of sizes (2.9 ms a scan of 3584 x
    14336, 0.6 ms of 896 x 896).
    """
    lib = _lib.load()
    rows = list(range(1, FUSED_MAX_ROWS + 1))
    rows += range(3 * 64, _SPLITK_SCAN_ROWS + 1, 64)
    return max(int(lib.ns_int4_linear_splitk_workspace_size(m, N, K)) for m in rows)


# One split-K workspace per device serves every Int4Linear on it: their calls
# run in stream order (the engine's eager steps and graph replays share one
# stream) and a workspace's arrival counters are back at zero after each call,
# so no call sees another's state.  A module keeps the buffer it was given; a
# module that needs more than the current buffer gets a new, larger one, and
# the old one stays with the modules (and captured graphs) that hold it.
_splitk_shared: dict[int, torch.Tensor] = {}


def _shared_splitk_workspace(device: torch.device, nbytes: int) -> torch.Tensor:
    key = device.index if device.index is not None else torch.cuda.current_device()
    ws = _splitk_shared.get(key)
    if ws is None or ws.numel() < nbytes:
        ws = torch.zeros(nbytes, dtype=torch.uint8, device=device)
        _splitk_shared[key] = ws
    return ws


def int4_linear(x: torch.Tensor, qweight: torch.Tensor, scales: torch.Tensor, zeros: torch.Tensor,
                bias: torch.Tensor | None, group_size: int, out: torch.Tensor | None = None,
                residual: torch.Tensor | None = None, silu_mul: bool = False,
                norm_weight: torch.Tensor | None = None, norm_eps: float = 1e-6,
                method: str = "auto", workspace: torch.Tensor | None = None) -> torch.Tensor:
    """x [..., K] -> [..., N] through ns_int4_linear (HIP; no CPU fallback).

    norm_weight: RMS-normalise the rows of x with this [K] weight inside the
    same launch first (the reference's RMSNorm before the projection; K must
    be a multiple of 128 and at most 1024).
    workspace: a zeroed uint8 buffer of splitk_workspace_bytes(N, K) bytes;
    given, long-K layers split their K loop over several workgroups per tile
    when their tiles alone would leave CUs idle (ns_int4_linear_splitk, both
    kernels).  Calls that overlap in time must not share one.
    method: "fused" (ns_int4_linear: the register-dequant kernel up to
    FUSED_MAX_ROWS rows, the tiled GEMM above; above FUSED_MAX_ROWS the
    RMSNorm runs first as its own op), "dequant" (ns_int4_dequantize, then a
    library GEMM and the same epilogue as tensor ops: the reference's
    QuantLinear steps) or "auto": "fused", except for layers with K >= LONG_K
    above LONG_K_TILED_MAX_ROWS rows when the call is recorded into a graph
    (whose replays carry none of the host work) and an eager call on the
    stream already took the weight scratch, which capture cannot allocate:
    those take the dequantised weight through the library GEMM too, with a
    residual added by the GEMM itself (torch.addmm with the residual as its
    input, written straight into the output: one rounding of
    residual + x·W^T instead of the reference's two, within the same bound).
    residual: [..., N] added to the result in the same launch (the reference's
    `residual + o_proj(x)`, rounded as two tensor ops).  silu_mul: the weight's
    rows are interleaved (gate, up) pairs and the result is
    silu(gate) * up, [..., N/2] (the reference SwiGLU, rounded per op).
    """
    lib = _lib.load()
    N, half_k = qweight.shape
    K = 2 * half_k
    if x.shape[-1] != K:
        raise ValueError(f"x has {x.shape[-1]} features, the weight {K}")
    if x.dtype not in (torch.float16, torch.bfloat16):
        raise TypeError(f"int4_linear computes in fp16 or bf16, got {x.dtype}")
    if not (x.is_cuda and qweight.is_cuda and scales.is_cuda and zeros.is_cuda):
        raise ValueError("int4_linear needs GPU tensors (the HIP path has no CPU fallback)")
    if qweight.dtype != torch.uint8 or zeros.dtype != torch.uint8 or scales.dtype != torch.float32:
        raise TypeError("qweight/zeros must be uint8 and scales float32")
    if not (qweight.is_contiguous() and scales.is_contiguous() and zeros.is_contiguous()):
        raise ValueError("quantised weight tensors must be contiguous")
    if bias is not None and (bias.dtype != x.dtype or bias.shape != (N,) or not bias.is_contiguous()):
        raise ValueError(f"bias must be a contiguous [{N}] {x.dtype} tensor")
    if silu_mul and residual is not None:
        raise ValueError("silu_mul and residual are separate epilogues")
    lead = x.shape[:-1]
    x2 = x.reshape(-1, K)
    if x2.stride(1) != 1 or x2.stride(0) % 8 != 0 or x2.data_ptr() % 16 != 0:
        x2 = x2.contiguous()
    M = x2.shape[0]
    n_out = N // 2 if silu_mul else N
    epilogue = _lib.NS_EPILOGUE_SILU_MUL if silu_mul else _lib.NS_EPILOGUE_NONE
    res_ptr = None
    if residual is not None:
        res = residual.reshape(-1, N)
        if res.shape[0] != M or res.dtype != x.dtype or not res.is_contiguous():
            raise ValueError(f"residual must be a contiguous [{M}, {N}] {x.dtype} tensor")
        res_ptr = res.data_ptr()
        epilogue = _lib.NS_EPILOGUE_RESIDUAL
    if out is None:
        out = torch.empty((M, n_out), dtype=x.dtype, device=x.device)
    elif out.shape != (M, n_out) or out.dtype != x.dtype or not out.is_contiguous():
        raise ValueError(f"out must be a contiguous [{M}, {n_out}] {x.dtype} tensor")
    if method not in ("auto", "fused", "dequant"):
        raise ValueError(f"unknown method {method!r}")
    blas_epilogue = False
    if (method == "auto" and K >= LONG_K and M > LONG_K_TILED_MAX_ROWS
            and torch.cuda.is_current_stream_capturing() and _scratch_ready(x.device, N, K, x.dtype)):
        method = "dequant"
        blas_epilogue = residual is not None and bias is None
    if method == "dequant":
        w = _scratch_weight(x.device, N, K, x.dtype)
        int4_dequantize(qweight, scales, zeros, group_size, x.dtype, out=w)
        xin = x2 if norm_weight is None else F.rms_norm(x2, (K,), norm_weight, norm_eps)
        if blas_epilogue:
            # Graph-replayed on MI355X, down_proj + residual at 1024 / 2048
            # tokens: 32.7 / 40.9 us, against 33.8 / 42.2 for the reference's
            # steps (the GEMM, then the add and a copy as tensor ops).
            torch.addmm(res, xin, w.t(), out=out)
            return out.view(*lead, n_out)
        y = F.linear(xin, w, bias)
        if silu_mul:
            y = F.silu(y[:, 0::2]) * y[:, 1::2]
        if residual is not None:
            y = res + y
        out.copy_(y)
        return out.view(*lead, n_out)
    nw_ptr = None
    if norm_weight is not None:
        if norm_weight.shape != (K,) or norm_weight.dtype != x.dtype or not norm_weight.is_contiguous():
            raise ValueError(f"norm_weight must be a contiguous [{K}] {x.dtype} tensor")
        if M > FUSED_MAX_ROWS:
            # The tiled GEMM does not fuse the RMSNorm: normalise as its own op
            # (the reference's separate RMSNorm, torch's fused kernel).
            x2 = F.rms_norm(x2, (K,), norm_weight, norm_eps).contiguous()
        else:
            nw_ptr = norm_weight.data_ptr()
    stream = torch.cuda.current_stream(x.device).cuda_stream
    if workspace is not None:
        if workspace.dtype != torch.uint8 or not workspace.is_cuda or workspace.data_ptr() % 256 != 0:
            raise ValueError("workspace must be a 256-byte aligned uint8 GPU tensor")
        rc = lib.ns_int4_linear_splitk(out.data_ptr(), x2.data_ptr(), x2.stride(0),
                                       qweight.data_ptr(), scales.data_ptr(), zeros.data_ptr(),
                                       bias.data_ptr() if bias is not None else None, res_ptr, epilogue,
                                       nw_ptr, float(norm_eps), M, N, K, group_size, _lib.DTYPE_CODES[x.dtype],
                                       workspace.data_ptr(), workspace.numel(), stream)
        _lib.check(rc, "ns_int4_linear_splitk")
        return out.view(*lead, n_out)
    rc = lib.ns_int4_linear(out.data_ptr(), x2.data_ptr(), x2.stride(0),
                            qweight.data_ptr(), scales.data_ptr(), zeros.data_ptr(),
                            bias.data_ptr() if bias is not None else None, res_ptr, epilogue,
                            nw_ptr, float(norm_eps),
                            M, N, K, group_size, _lib.DTYPE_CODES[x.dtype], stream)
    _lib.check(rc, "ns_int4_linear")
    return out.view(*lead, n_out)


def rope_pair_order(num_heads: int, head_dim: int) -> torch.Tensor:
    """Row order of a q|k|v weight for ns_int4_linear_rope_cache: new row r is original row order[r].

    Each head's rows are regrouped in 16-row tiles; tile i holds dims
    [8i, 8i+8) then [D/2 + 8i, D/2 + 8i + 8), so the MFMA result puts every
    dim and its rotate_half partner in lanes 32 apart."""
    D = head_dim
    if D % 16 != 0:
        raise ValueError(f"head_dim must be a multiple of 16, got {D}")
    j = torch.arange(16)
    tiles = torch.stack([torch.where(j < 8, 8 * i + j, D // 2 + 8 * i + (j - 8)) for i in range(D // 16)])
    per_head = tiles.reshape(-1)
    return (torch.arange(num_heads).unsqueeze(1) * D + per_head).reshape(-1)


def int4_qkv_rope_cache(x: torch.Tensor, qkv: "Int4Linear", cos: torch.Tensor, sin: torch.Tensor,
                        k_cache: torch.Tensor, v_cache: torch.Tensor, slot_mapping: torch.Tensor,
                        norm=None) -> torch.Tensor:
    """q' for attention, with k' and v written to the cache: one ns_int4_linear_rope_cache launch.

    qkv is a rope-paired q|k|v module (Int4Linear.rope_pairs); x [T, K];
    cos/sin [T, 1, D] or [T, D] in x's dtype; norm an RMSNorm-like module run
    in the same launch.  Above FUSED_MAX_ROWS tokens (prefill chunks) this is
    the dequantised-weight projection followed by ns_rope_reshape_and_cache.
    Returns q' as a contiguous [T, Hq, D] tensor."""
    from .rotary import rope_reshape_and_cache

    Hq, Hkv, D = qkv.rope_heads
    T, K = x.shape
    if T > FUSED_MAX_ROWS or not qkv.fuses_norm:
        y = qkv(x, norm=norm)
        q, k, v = y[:, :Hq * D].view(T, Hq, D), y[:, Hq * D:(Hq + Hkv) * D].view(T, Hkv, D), y[:, (Hq + Hkv) * D:].view(T, Hkv, D)
        return rope_reshape_and_cache(q, k, v, cos, sin, k_cache, v_cache, slot_mapping)
    lib = _lib.load()
    cs, sn = cos.reshape(T, D), sin.reshape(T, D)
    if not (x.dtype == cos.dtype == sin.dtype == k_cache.dtype == v_cache.dtype):
        raise TypeError("x, cos, sin and the caches must share one dtype")
    if cs.stride(1) != 1 or sn.stride(0) != cs.stride(0) or sn.stride(1) != 1:
        raise ValueError("cos and sin must be [T, D] rows with one token stride")
    if k_cache.dim() != 4 or v_cache.shape != k_cache.shape or k_cache.shape[2:] != (Hkv, D):
        raise ValueError(f"caches must be [num_blocks, block_size, {Hkv}, {D}]")
    if not (k_cache.is_contiguous() and v_cache.is_contiguous()):
        raise ValueError("caches must be contiguous")
    if slot_mapping.shape != (T,) or slot_mapping.dtype not in (torch.int32, torch.int64):
        raise ValueError(f"slot_mapping must be a [{T}] int32/int64 tensor")
    x2 = x if (x.stride(1) == 1 and x.stride(0) % 8 == 0 and x.data_ptr() % 16 == 0) else x.contiguous()
    slots = slot_mapping if slot_mapping.is_contiguous() else slot_mapping.contiguous()
    out = torch.empty((T, Hq, D), dtype=x.dtype, device=x.device)
    rc = lib.ns_int4_linear_rope_cache(
        out.data_ptr(), x2.data_ptr(), x2.stride(0),
        qkv.qweight.data_ptr(), qkv.scales.data_ptr(), qkv.zeros.data_ptr(),
        None if qkv.bias is None else qkv.bias.data.data_ptr(),
        None if norm is None else norm.weight.data.data_ptr(), 1e-6 if norm is None else float(norm.variance_epsilon),
        cs.data_ptr(), sn.data_ptr(), cs.stride(0),
        k_cache.data_ptr(), v_cache.data_ptr(), slots.data_ptr(), int(slots.dtype == torch.int64),
        T, K, qkv.group_size, Hq, Hkv, D, k_cache.shape[1], k_cache.shape[0],
        _lib.DTYPE_CODES[x.dtype], torch.cuda.current_stream(x.device).cuda_stream)
    _lib.check(rc, "ns_int4_linear_rope_cache")
    return out


class Int4Linear(nn.Module):
    """Drop-in nn.Linear whose weight lives as INT4 groups (reference QuantLinear, int4 mode).

    Buffers and their shapes match the reference module (quant.py:131-135):
    qweight [out, in/2] uint8, scales [out, in/gs] float32, zeros [out, in/gs]
    uint8, plus an optional bias in the compute dtype.
    """

    def __init__(self, in_features: int, out_features: int, bias: bool, group_size: int, dtype, device) -> None:
        super().__init__()
        if in_features % group_size != 0:
            raise ValueError(f"Int4Linear needs in_features ({in_features}) to be a multiple of group_size ({group_size})")
        self.in_features = in_features
        self.out_features = out_features
        self.group_size = group_size
        self.compute_dtype = dtype
        g = in_features // group_size
        self.register_buffer("qweight", torch.zeros(out_features, in_features // 2, dtype=torch.uint8, device=device))
        self.register_buffer("scales", torch.zeros(out_features, g, dtype=torch.float32, device=device))
        self.register_buffer("zeros", torch.zeros(out_features, g, dtype=torch.uint8, device=device))
        self.bias = nn.Parameter(torch.zeros(out_features, dtype=dtype, device=device)) if bias else None
        # Rows interleaved as (gate, up) pairs whose output is silu(gate) * up.
        self.silu_mul = False
        # (num_heads, num_kv_heads, head_dim) when the rows are q|k|v in
        # rotary-pair order (rope_pairs); forward() then restores row order.
        self.rope_heads: tuple[int, int, int] | None = None
        self.rope_inverse: torch.Tensor | None = None
        # Split-K workspace (taken on first use from the device's shared one;
        # the INT4 layers' calls run in stream order, so they never overlap).
        self._splitk_ws: torch.Tensor | None = None
        self._splitk_checked = False

    @classmethod
    def from_linear(cls, lin: nn.Linear, group_size: int = 128) -> "Int4Linear":
        w = lin.weight.data
        m = cls(lin.in_features, lin.out_features, lin.bias is not None, group_size, w.dtype, w.device)
        packed, s, z = quantize_int4_groupwise(w, group_size)
        m.qweight.copy_(packed)
        m.scales.copy_(s)
        m.zeros.copy_(z)
        if lin.bias is not None:
            m.bias.data.copy_(lin.bias.data)
        return m

    def forward(self, x: torch.Tensor, residual: torch.Tensor | None = None, norm=None) -> torch.Tensor:
        """self(norm(x)) (+ residual); `norm` is an RMSNorm-like module (weight,
        variance_epsilon) applied inside the launch when the shape allows."""
        if norm is not None and not self.fuses_norm:
            x, norm = norm(x), None
        if self.rope_heads is not None and residual is not None:
            raise ValueError("a rope-paired q|k|v projection takes no residual")
        if not self._splitk_checked:
            n = splitk_workspace_bytes(self.out_features, self.in_features)
            if n and torch.cuda.is_current_stream_capturing():
                # A new workspace's zero fill would be recorded into the graph
                # (and rerun by every replay); the first call belongs before capture.
                raise RuntimeError(
                    f"Int4Linear({self.in_features}, {self.out_features}) takes its split-K workspace "
                    "on first use: call it once before graph capture")
            self._splitk_ws = _shared_splitk_workspace(self.qweight.device, n) if n else None
            self._splitk_checked = True
        y = int4_linear(x, self.qweight, self.scales, self.zeros,
                        None if self.bias is None else self.bias.data, self.group_size,
                        residual=residual, silu_mul=self.silu_mul,
                        norm_weight=None if norm is None else norm.weight.data,
                        norm_eps=1e-6 if norm is None else norm.variance_epsilon,
                        workspace=self._splitk_ws)
        return y if self.rope_inverse is None else y.index_select(-1, self.rope_inverse)

    @property
    def fuses_norm(self) -> bool:
        """Whether to RMS-normalise this layer's input inside its own launch.

        The kernel can when K is a multiple of 128 up to 1024: each wave scales
        its slice of x by the norm weight as it loads it and the rows' sums of
        squares meet with the partial products, so the norm costs no pass of
        its own.  Graph-replayed on MI355X, fused against torch's norm plus
        the GEMM: q|k|v (1152 outputs) 3.6 / 4.0 / 4.9 us against 5.5 / 6.3 /
        7.2 at 1 / 32 / 64 tokens, gate|up (9728 outputs) 6.0 / 8.3 / 12.8 us
        against 7.0 / 9.6 / 13.3."""
        return self.in_features % 128 == 0 and self.in_features <= 1024

    @classmethod
    def gate_up_pairs(cls, gate: "Int4Linear", up: "Int4Linear") -> "Int4Linear":
        """One module computing silu(gate(x)) * up(x): rows interleaved gate_0, up_0, gate_1, ..."""
        if gate.bias is not None or up.bias is not None or gate.qweight.shape != up.qweight.shape:
            raise ValueError("gate/up must be bias-free projections of one shape")
        m = cls(gate.in_features, 2 * gate.out_features, False, gate.group_size, gate.compute_dtype,
                gate.qweight.device)
        for name in ("qweight", "scales", "zeros"):
            a, b = getattr(gate, name), getattr(up, name)
            getattr(m, name).copy_(torch.stack([a, b], dim=1).reshape(-1, a.shape[1]))
        m.silu_mul = True
        return m

    @classmethod
    def rope_pairs(cls, qkv: "Int4Linear", num_heads: int, num_kv_heads: int, head_dim: int) -> "Int4Linear":
        """The q|k|v module with its rows in rotary-pair order (rope_pair_order),
        for int4_qkv_rope_cache; calling it still returns rows in q|k|v order."""
        heads = num_heads + 2 * num_kv_heads
        if qkv.out_features != heads * head_dim or qkv.silu_mul:
            raise ValueError("rope_pairs needs a q|k|v projection of (Hq + 2 Hkv) * D rows")
        order = rope_pair_order(heads, head_dim).to(qkv.qweight.device)
        m = cls(qkv.in_features, qkv.out_features, qkv.bias is not None, qkv.group_size, qkv.compute_dtype,
                qkv.qweight.device)
        for name in ("qweight", "scales", "zeros"):
            getattr(m, name).copy_(getattr(qkv, name).index_select(0, order))
        if qkv.bias is not None:
            m.bias.data.copy_(qkv.bias.data.index_select(0, order))
        m.rope_heads = (num_heads, num_kv_heads, head_dim)
        m.rope_inverse = torch.argsort(order)
        return m

    def extra_repr(self) -> str:
        extra = ", silu(gate)*up pairs" if self.silu_mul else ""
        return f"in={self.in_features}, out={self.out_features}, int4 group={self.group_size}{extra}"


def _int4_sites(model: nn.Module, group_size: int, skip: tuple[str, ...]) -> list[tuple[nn.Module, str]]:
    """(owner, attribute) of every nn.Linear that quantize_model converts.

    A linear qualifies when no entry of `skip` occurs in its dotted path (so a
    skipped module's whole subtree stays as it is), its in_features is a whole
    number of groups and its out_features a whole number of the kernels'
    16-row tiles.  The list is complete before anything is replaced, so the
    walk never meets a module it created."""
    sites = []
    for owner_path, owner in model.named_modules():
        for attr, child in owner.named_children():
            path = f"{owner_path}.{attr}" if owner_path else attr
            if not isinstance(child, nn.Linear) or any(tag in path for tag in skip):
                continue
            if child.in_features % group_size == 0 and child.out_features % 16 == 0:
                sites.append((owner, attr))
    return sites


def _resident_bytes(model: nn.Module) -> int:
    """Bytes of the distinct storages behind the model's parameters and buffers.

    Counting storages rather than tensors charges tied weights (an lm_head
    that shares the embedding) and views once each."""
    sizes: dict[tuple[str, int], int] = {}
    for tensor in itertools.chain(model.parameters(), model.buffers()):
        storage = tensor.untyped_storage()
        sizes[(str(tensor.device), storage.data_ptr())] = storage.nbytes()
    return sum(sizes.values())


def quantize_model(model: nn.Module, group_size: int = 128, skip: tuple[str, ...] = ("lm_head",)) -> dict:
    """Convert the model's eligible nn.Linear layers to Int4Linear in place.

    The reference's int4 mode of quantize_model (nanoserve/quant.py:165-199):
    same eligibility by name (`skip` substrings) and by shape, and a report
    under the same keys, which its loader and benchmarks read: mode,
    group_size, layers_quantized, weight_mib_before / _after, compression
    (before / after) and freed_mib.  Linears the kernels cannot take (in
    features not a multiple of group_size, out features not a multiple of 16)
    stay in the model's dtype.
    """
    mib = float(2**20)
    sites = _int4_sites(model, group_size, skip)
    resident_before = _resident_bytes(model)
    for owner, attr in sites:
        setattr(owner, attr, Int4Linear.from_linear(getattr(owner, attr), group_size))
    resident_after = _resident_bytes(model)
    report = dict(mode="int4", group_size=group_size, layers_quantized=len(sites))
    report.update(weight_mib_before=resident_before / mib, weight_mib_after=resident_after / mib)
    report["compression"] = resident_before / resident_after if resident_after else 0.0
    report["freed_mib"] = report["weight_mib_before"] - report["weight_mib_after"]
    return report
