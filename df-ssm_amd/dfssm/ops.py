"""Single-operator wrappers over the C ABI, taking torch tensors on the GPU.

These are the operator-level entry points (scaffold GEMM, RMSNorm+quantize, conv step, SSM step,
bit/embedding tiling). Every call launches on torch's current stream and raises on any error;
there is no CPU fallback. Arguments that are not contiguous are copied; all copies of a call stay bound
to names until its launch, so that the allocator cannot give one's memory to the next.
"""
from __future__ import annotations

import threading

import torch

from . import _C


def _need(t: torch.Tensor, dtype, name: str):
    if isinstance(t, torch.Tensor) and t.is_cuda and t.dtype is dtype:
        return
    if not isinstance(t, torch.Tensor) or t.device.type != "cuda":
        raise TypeError(f"{name} must be a CUDA (HIP) tensor")
    if t.dtype != dtype:
        raise TypeError(f"{name} must be {dtype}, got {t.dtype}")


def tile_bits(packed: torch.Tensor, rows: int, k: int) -> torch.Tensor:
    """(rows, k/32) int32 sign-bit words -> tiled copy for the scaffold kernels."""
    _need(packed, torch.int32, "packed")
    if not packed.is_contiguous() or packed.numel() != rows * (k // 32):
        raise ValueError("packed must be a contiguous (rows, k/32) int32 tensor")
    out = torch.empty(_C.lib().dfssm_tiled_bits_bytes(rows, k) // 4, dtype=torch.int32, device=packed.device)
    _C.check(_C.lib().dfssm_tile_bits(packed.data_ptr(), out.data_ptr(), rows, k, _C.stream()), "tile_bits")
    return out


def scaffold_gemm(tiled_bits: torch.Tensor, q: torch.Tensor, N: int, xscale=None, wscale=None, want_y=False):
    """int32 acc (M, N) = q (M, K) int8 x sign-bit matrix^T; optionally y fp16 (M, N)."""
    _need(q, torch.int8, "q")
    M, K = q.shape
    acc = torch.empty(M, N, dtype=torch.int32, device=q.device)
    y = torch.empty(M, N, dtype=torch.float16, device=q.device) if want_y else None
    q = q.contiguous()
    _C.check(_C.lib().dfssm_scaffold_gemm(
        tiled_bits.data_ptr(), q.data_ptr(), _C.ptr(xscale), _C.ptr(wscale), M, N, K,
        acc.data_ptr(), _C.ptr(y), _C.stream()), "scaffold_gemm")
    return (acc, y) if want_y else acc


SCAFFOLD_WORKSPACE_BYTES = 64 << 10   # DFSSM_SCAFFOLD_WORKSPACE_BYTES
SCAFFOLD_ERROR_OFFSET = 1024          # DFSSM_SCAFFOLD_ERROR_OFFSET
SCAFFOLD_WORKSPACE_STREAMS = 64       # streams whose workspaces are kept
_scaffold_ws = {}
_scaffold_ws_lock = threading.Lock()


def _new_scaffold_workspace(device) -> torch.Tensor:
    return torch.zeros(SCAFFOLD_WORKSPACE_BYTES // 4, dtype=torch.int32, device=device)


def scaffold_workspace(device) -> torch.Tensor:
    """The exchange workspace of dfssm_scaffold_lora_gemm for calls on torch's current stream of `device`,
    zeroed on that stream at allocation. Calls that share one must not overlap, so every stream has its
    own; those of the last SCAFFOLD_WORKSPACE_STREAMS streams are kept. A stream that is being captured
    gets a new one at each call, owned by its graph and zeroed at every replay: a kept one would tie
    the graph's replays to whatever runs on the capture's stream then."""
    return _stream_workspace(device, _C.stream())


def _stream_workspace(device, stream: int) -> torch.Tensor:
    dev = device if isinstance(device, torch.device) else torch.device(device)
    if stream and torch.cuda.is_current_stream_capturing():  # (the null stream cannot be captured)
        return _new_scaffold_workspace(dev)
    if dev.index is None:
        dev = torch.device(dev.type, torch.cuda.current_device())
    key = (dev, stream)
    ws = _scaffold_ws.get(key)
    if ws is None:
        with _scaffold_ws_lock:
            ws = _scaffold_ws.get(key)
            if ws is None:
                while len(_scaffold_ws) >= SCAFFOLD_WORKSPACE_STREAMS:  # (freed in its stream's order)
                    del _scaffold_ws[next(iter(_scaffold_ws))]
                ws = _scaffold_ws[key] = _new_scaffold_workspace(dev)
    return ws


def scaffold_error(workspace: torch.Tensor) -> int:
    """The workspace's error word (synchronizes): non-zero after a call whose wait timed out."""
    return int(workspace[SCAFFOLD_ERROR_OFFSET // 4].item())


def scaffold_lora_gemm(tiled_bits: torch.Tensor, wscale: torch.Tensor, q: torch.Tensor, xscale: torch.Tensor,
                       xn: torch.Tensor, lA: torch.Tensor, lA_s: torch.Tensor, lBq: torch.Tensor, N: int,
                       workspace="auto"):
    """One projection with its LoRA (dfssm_scaffold_lora_gemm): returns (acc int32 (M, N),
    y fp16 (M, N), lora_h fp16 (M, 16)). q (M, K) int8 with fp16 scales xscale (M,), xn (M, K) fp16,
    lA (N, 16) int8, lA_s (N,) fp16, lBq (16, K) fp16, wscale (N,) fp16. workspace: "auto" (the
    current stream's exchange workspace: one launch at M <= 4; in a capture one more, which clears it),
    None (no workspace) or an int32 tensor of SCAFFOLD_WORKSPACE_BYTES, zeroed before its first use and
    used by calls that do not overlap."""
    _need(q, torch.int8, "q")
    _need(xn, torch.float16, "xn")
    _need(lBq, torch.float16, "lBq")
    _need(lA, torch.int8, "lA")
    M, K = q.shape
    if xn.shape != (M, K) or lBq.shape != (16, K) or lA.shape != (N, 16):
        raise ValueError("shape mismatch: q/xn (M, K), lBq (16, K), lA (N, 16)")
    acc = torch.empty(M, N, dtype=torch.int32, device=q.device)
    y = torch.empty(M, N, dtype=torch.float16, device=q.device)
    h = torch.empty(M, 16, dtype=torch.float16, device=q.device)
    stream = _C.stream()
    if isinstance(workspace, str):
        if workspace != "auto":
            raise ValueError('workspace must be "auto", None or a tensor')
        workspace = _stream_workspace(q.device, stream) if M <= 4 else None  # (unused by more rows)
    elif workspace is not None:
        _need(workspace, torch.int32, "workspace")
        if workspace.numel() * 4 < SCAFFOLD_WORKSPACE_BYTES:
            raise ValueError(f"workspace must hold {SCAFFOLD_WORKSPACE_BYTES} bytes")
    wscale, q, xscale, xn = wscale.contiguous(), q.contiguous(), xscale.contiguous(), xn.contiguous()
    lA, lA_s, lBq = lA.contiguous(), lA_s.contiguous(), lBq.contiguous()
    _C.check(_C.lib().dfssm_scaffold_lora_gemm(
        tiled_bits.data_ptr(), wscale.data_ptr(), q.data_ptr(), xscale.data_ptr(), xn.data_ptr(), lA.data_ptr(),
        lA_s.data_ptr(), lBq.data_ptr(), M, N, K, h.data_ptr(), acc.data_ptr(), y.data_ptr(), _C.ptr(workspace), stream), "scaffold_lora_gemm")
    return acc, y, h


def rmsnorm_quantize(x: torch.Tensor, w: torch.Tensor):
    """x (M, K) fp16, w (K) fp32 -> (xn fp16 (M, K), q int8 (M, K), scale fp16 (M,))."""
    _need(x, torch.float16, "x")
    _need(w, torch.float32, "w")
    M, K = x.shape
    xn = torch.empty(M, K, dtype=torch.float16, device=x.device)
    q = torch.empty(M, K, dtype=torch.int8, device=x.device)
    s = torch.empty(M, dtype=torch.float16, device=x.device)
    x, w = x.contiguous(), w.contiguous()
    _C.check(_C.lib().dfssm_rmsnorm_quantize(x.data_ptr(), w.data_ptr(), M, K,
                                             xn.data_ptr(), q.data_ptr(), s.data_ptr(), _C.stream()),
             "rmsnorm_quantize")
    return xn, q, s


def conv_step(conv_state: torch.Tensor, xbc: torch.Tensor, conv_w: torch.Tensor, conv_b: torch.Tensor) -> None:
    """In place: conv_state (B, C, 3) fp16 and xbc (B, C) fp16 (row stride honoured)."""
    for t, n in ((conv_state, "conv_state"), (xbc, "xBC"), (conv_w, "conv_weight"), (conv_b, "conv_bias")):
        _need(t, torch.float16, n)
    B, C = xbc.shape
    if conv_state.shape != (B, C, 3) or not conv_state.is_contiguous():
        raise ValueError(f"conv_state must be contiguous ({B}, {C}, 3)")
    if xbc.stride(1) != 1:
        raise ValueError("xBC rows must be contiguous")
    conv_w, conv_b = conv_w.contiguous(), conv_b.contiguous()
    _C.check(_C.lib().dfssm_conv_step(conv_state.data_ptr(), xbc.data_ptr(), xbc.stride(0), conv_w.data_ptr(),
                                      conv_b.data_ptr(), B, C, _C.stream()), "conv_step")


def ssm_step(h: torch.Tensor, xbc: torch.Tensor, dt: torch.Tensor, dt_bias, A_log, D, y_out: torch.Tensor) -> None:
    """h (B, H, P, N) fp32 in place; xbc rows x|B|C fp16; dt (B, H) fp16; y_out (B, H*P) fp16."""
    _need(h, torch.float32, "h_state")
    _need(xbc, torch.float16, "xBC")
    _need(dt, torch.float16, "dt")
    _need(y_out, torch.float16, "y_out")
    for t, n in ((dt_bias, "dt_bias"), (A_log, "A_log"), (D, "D")):
        _need(t, torch.float32, n)
    B, H, P, N = h.shape
    if not h.is_contiguous() or xbc.stride(1) != 1 or dt.stride(1) != 1 or y_out.stride(1) != 1:
        raise ValueError("h_state must be contiguous and xBC / dt / y_out rows contiguous")
    dt_bias, A_log, D = dt_bias.contiguous(), A_log.contiguous(), D.contiguous()
    _C.check(_C.lib().dfssm_ssm_step(h.data_ptr(), xbc.data_ptr(), xbc.stride(0), dt.data_ptr(), dt.stride(0),
                                     dt_bias.data_ptr(), A_log.data_ptr(), D.data_ptr(), y_out.data_ptr(),
                                     y_out.stride(0), B, H, P, N, _C.stream()), "ssm_step")
