"""Dense 16-bit layers for the non-LLM model families (BERT, Whisper, CLIP/T5 text encoders, UNet /
MMDiT, VAE, TTS): plain library GEMMs on hipBLASLt (few rows by matrices it is slow on: lin16.hip) with the bias folded into
the GEMM, fp32 accumulation into the residual stream, and the library's act16 activations.

On CPU everything runs in fp32 (the numerics oracle for the tests)."""
from __future__ import annotations

import numpy as np
import torch
import torch.nn.functional as F

from .linear import ACT_DTYPE, _fp32_out_ok


def model_dtype(device) -> torch.dtype:
    return ACT_DTYPE if torch.device(device).type == "cuda" else torch.float32


def to_dev(a, device, dtype) -> torch.Tensor:
    if isinstance(a, torch.Tensor):
        return a.to(device=device, dtype=dtype).contiguous()
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).to(device).to(dtype).contiguous()


def few_rows_parts(M: int, N: int, K: int) -> int:
    """Parts of K that csrc/kernels/lin16.hip sums for M rows, or 0 where the library multiplies.

    Measured with weights in no cache (bf16, f16 alike; us, here / library): long K and few columns, where the library's choice
    degrades beyond K = 16384: 4096 x 17408 0.75 of the library's time at one row, 0.34-0.4 beyond 32, x 28672 0.96 and 0.4-0.47,
    3072 0.65-0.9 and 0.3-0.6, 2048 0.25-0.6, 1024 0.22-0.7, 128-512 0.22-1.0; but 64 x 49152 1.06-1.4 beyond 32 rows, 5120 x
    20480 49-56 / 50-53 to 16 rows, 8192 x 20480 66-89 / 59-65 to 32. Many columns and up to 8 rows: 24576-32768 x 512-2304
    0.67-1.0, 28672-32768 x 4096 0.84-0.98; 24576 x 4096 1.1, any x 5120 and 8192 up to 1.4, and beyond 32768 columns the library is
    as good or better at most widths (51200 x 1280 1.14-1.25, 256000 x 2304 1.07-1.17). Parts make one workgroup per compute unit
    (4096 columns: 1 / 2 / 4 / 8 parts 148 / 80 / 50 / 52 us)."""
    if N % 64 or K % 32 or not 0 < M <= 64:
        return 0
    if K > 16384 and N <= 4096:
        return min(8, 256 // (N // 64)) if N >= 128 or K <= 32768 or M <= 32 else 0
    return 1 if 24576 <= N <= 32768 and M <= 8 and K <= (4096 if N >= 28672 else 2304) else 0


def _few_rows(x: torch.Tensor, w: torch.Tensor, out: torch.Tensor, acc: bool) -> bool:
    """out (fp32) (+)= x w^T by lin16.hip where few_rows_parts takes it; False: nothing done, the library's product answers (or
    refuses) as for any other shape: operands of other devices or widths, rows of x that overlap (a row stride below K, as
    expanded rows and sliding windows have), and graphs that would need a gradient are its business."""
    if not (x.is_cuda and x.dim() == 2 and x.dtype == w.dtype and x.dtype in (torch.float16, torch.bfloat16)):
        return False
    M, K = x.shape
    N_ = w.shape[0]
    parts = few_rows_parts(M, N_, K)
    if not parts or w.device != x.device or out.device != x.device or x.device.index != torch.cuda.current_device() \
            or tuple(w.shape) != (N_, K) or (torch.is_grad_enabled() and (x.requires_grad or w.requires_grad or out.requires_grad)):
        return False
    ldx = x.stride(0) if M > 1 else K
    if x.stride(1) != 1 or ldx < K or ldx % 8 or x.data_ptr() % 16 or not w.is_contiguous() or w.data_ptr() % 16 \
            or out.dtype != torch.float32 or out.shape != (M, N_) or out.stride(1) != 1 or out.stride(0) < N_:
        return False
    from .. import _native as N
    part = torch.empty(parts, M, N_, dtype=torch.float32, device=x.device) if parts > 1 else None
    N.kcall("mxk_lin16", x.data_ptr(), ldx, w.data_ptr(), out.data_ptr(), out.stride(0), N.ptr(part), parts, M, N_, K,
            int(x.dtype == torch.float16), int(acc), N.stream_ptr())
    return True


class Dense:
    """y = x W^T + b with W [N, K] in the model dtype; bias kept in both dtypes."""

    __slots__ = ("w", "b", "b32", "wt")

    def __init__(self, w, b=None, device="cpu", dtype=torch.float32):
        self.w = to_dev(w, device, dtype)
        self.wt = self.w.t()
        self.b = to_dev(b, device, dtype) if b is not None else None
        self.b32 = to_dev(b, device, torch.float32) if b is not None else None

    @property
    def n(self) -> int:
        return self.w.shape[0]

    def __call__(self, x: torch.Tensor, act: str | None = None) -> torch.Tensor:
        y = torch.addmm(self.b, x, self.wt) if self.b is not None else x @ self.wt
        if act == "gelu":
            y = F.gelu(y)
        elif act == "silu":
            y = F.silu(y)
        elif act == "gelu_tanh":
            y = F.gelu(y, approximate="tanh")
        return y

    def f32(self, x: torch.Tensor) -> torch.Tensor:
        """fp32 output (hipBLASLt 16-bit x 16-bit -> fp32 where the build supports it)."""
        if x.dtype == torch.float32:
            return self(x)
        out = torch.empty(x.shape[0], self.n, dtype=torch.float32, device=x.device)
        if _fp32_out_ok(x.dtype):
            if self.b32 is not None:
                out.copy_(self.b32.expand_as(out))
                torch.addmm(out, x, self.wt, out_dtype=torch.float32, out=out)
            else:
                torch.mm(x, self.wt, out_dtype=torch.float32, out=out)
            return out
        out.copy_(self(x))
        return out

    def into(self, x: torch.Tensor, out: torch.Tensor) -> torch.Tensor:
        """out (fp32, contiguous, preallocated) = x W^T + b: 16-bit operands with the fp32 accumulator written as is,
        fp32 operands in plain fp32. `out` is written in place; under capture the parts of a few rows' product (_few_rows)
        come from the graph's own pool, so a captured graph sees static addresses."""
        if x.dtype == torch.float32:
            if self.b32 is not None:
                torch.addmm(self.b32, x, self.wt, out=out)
            else:
                torch.mm(x, self.wt, out=out)
            return out
        if self.b32 is None and _few_rows(x, self.w, out, False):
            return out
        if _fp32_out_ok(x.dtype):
            if self.b32 is not None:
                out.copy_(self.b32.expand_as(out))
                torch.addmm(out, x, self.wt, out_dtype=torch.float32, out=out)
            else:
                torch.mm(x, self.wt, out_dtype=torch.float32, out=out)
            return out
        out.copy_(self(x))
        return out

    def acc(self, x: torch.Tensor, acc: torch.Tensor) -> torch.Tensor:
        """acc (fp32) += x W^T + b — the residual add fused as GEMM beta = 1."""
        if x.dtype == torch.float32 and acc.is_contiguous():
            if self.b32 is not None:
                acc.add_(self.b32)
            torch.addmm(acc, x, self.wt, out=acc)
            return acc
        if x.dtype != torch.float32 and _fp32_out_ok(x.dtype) and acc.is_contiguous():
            if self.b32 is not None:
                acc.add_(self.b32)
            if not _few_rows(x, self.w, acc, True):
                torch.addmm(acc, x, self.wt, out_dtype=torch.float32, out=acc)
            return acc
        acc.add_(self(x).float())
        return acc


_BMM_OUT_DTYPE: dict = {}


def bmm_f32(a: torch.Tensor, b: torch.Tensor, out: torch.Tensor | None = None) -> torch.Tensor:
    """fp32 batched product a @ b; 16-bit operands keep the fp32 accumulator where the library exposes it."""
    if a.dtype == torch.float32:
        return torch.bmm(a, b, out=out) if out is not None else torch.bmm(a, b)
    ok = _BMM_OUT_DTYPE.get(a.dtype)
    if ok is None:
        try:
            torch.bmm(a[:1, :1], b[:1], out_dtype=torch.float32)
            ok = True
        except Exception:
            ok = False
        _BMM_OUT_DTYPE[a.dtype] = ok
    if ok:
        return torch.bmm(a, b, out_dtype=torch.float32, out=out) if out is not None else \
            torch.bmm(a, b, out_dtype=torch.float32)
    r = torch.bmm(a, b).float()
    if out is not None:
        out.copy_(r)
        return out
    return r


def layernorm(x: torch.Tensor, w, b, eps: float, out_dtype) -> torch.Tensor:
    """fp32 [M, H] -> layer-normed in out_dtype (norm.hip on GPU)."""
    from . import core as K
    out = torch.empty(x.shape, dtype=out_dtype, device=x.device)
    K.layernorm(x, w, b, eps, out)
    return out
