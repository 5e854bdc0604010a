"""Dense 16-bit layers for the non-LLM model families (BERT, Whisper, CLIP/T5 text encoders, UNet /
MMDiT, VAE, TTS): plain library GEMMs on hipBLASLt (bf16 products of long K or many columns: dense16.hip; few rows by other
matrices the library is slow on: lin16.hip) with the bias folded into the GEMM, fp32 accumulation into the residual stream, and the
library's act16 activations.

On CPU everything runs in fp32 (the numerics oracle for the tests)."""
from __future__ import annotations

import functools

import numpy as np
import torch
import torch.nn.functional as F

from .linear import ACT_DTYPE, CU_COUNT, _fp32_out_ok


def model_dtype(device) -> torch.dtype:
    return ACT_DTYPE if torch.device(device).type == "cuda" else torch.float32


def to_dev(a, device, dtype) -> torch.Tensor:
    if isinstance(a, torch.Tensor):
        return a.to(device=device, dtype=dtype).contiguous()
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).to(device).to(dtype).contiguous()


def few_rows_parts(M: int, N: int, K: int) -> int:
    """Parts of K that csrc/kernels/lin16.hip sums for M rows, or 0 where the library multiplies. It is asked after dense16.hip (takes_dense16), so
    what comes here is f16, and of bf16 long K with few columns or fewer than 2^24 weights, many columns by short K, K that is no whole 64s, and rows of
    `out` off 16 bytes.

    Measured with weights in no cache, against the library (bf16, f16 alike; us, here / library): long K and few columns, where the library's choice
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


# dense16.hip's tiles (16-row units, 16-column units of a wave): us a 64-wide k-tile and a round of workgroups, us to fill and drain a
# round, share of a round that its first workgroup takes, us and us a MB for the sum of parts, us for parts behind whole tiles. Fitted to
# 6300 measurements (26 shapes 1024 x 2048 .. 151936 x 1536, 1 to 4000 rows, weights in no cache): the pick is 1.5 % slower than the best
# of them on average.
_D16_COST = {(8, 8): (1.352, 16.3, 0.68, 1.0, 0.075, 3.7), (7, 8): (1.245, 14.4, 0.69, 1.1, 0.087, 2.6), (6, 8): (1.18, 11.2, 0.68, 2.8, 0.095, 0.0),
             (5, 8): (1.11, 8.4, 0.66, 3.5, 0.116, 0.0), (8, 6): (1.083, 12.8, 0.69, 1.0, 0.097, 0.0), (6, 6): (0.977, 8.7, 0.65, 2.6, 0.118, 0.0),
             (8, 4): (0.872, 8.1, 0.65, 3.4, 0.106, 0.0), (5, 4): (0.578, 7.2, 0.62, 2.1, 0.184, 0.0), (4, 4): (0.527, 6.0, 0.62, 1.9, 0.247, 0.0),
             (2, 4): (0.5, 3.4, 0.48, 2.8, 0.246, 0.9)}


@functools.lru_cache(maxsize=4096)
def dense16_plan(M: int, N_: int, K: int, Fn: int = 0):
    """(16-row units, 16-column units, whole tiles, parts of K of the others) of dense16.hip's tiles for M rows by N_ columns and Fn gated
    ones. Parts of K keep every compute unit at work where tiles leave some idle; only plain columns can have them. One round of parts
    at most, so their sums take at most 64 MB.

    Up to 64 rows the weights' bytes bound the product: 64-row tiles, 256 columns wide where 128 make more than one round of workgroups
    and these do not (us, 128 / 256 wide: 28672 x 4096 45 / 54, 40992 x 4096 74 / 64, 50304 x 2048 41 / 39.5, 128256 x 4096 177 / 194); by long K
    in up to 8 parts (4096 x 20480 at 33 rows 1 / 4 / 8 parts 120 / 46 / 38)."""
    nk = K // 64

    def tiles(mi, nj):
        return -(-M // (32 * mi)), -(-N_ // (32 * nj)), -(-2 * Fn // (32 * nj))
    if M <= 64:
        _, n, g = tiles(2, 4)
        if not Fn and K >= 2 * N_:
            return 2, 4, 0, max(1, min(8, CU_COUNT // n, nk))
        wide = sum(tiles(2, 8)[1:])
        return (2, 8, wide, 1) if n + g > CU_COUNT >= wide else (2, 4, n + g, 1)
    floor = (2 * K * (N_ + 2 * Fn + M) + 4 * M * N_ + 2 * M * Fn) / 5.6e6 + 4  # us: every byte once
    best = None
    for (mi, nj), (a, fill, first, e1, e2, e3) in _D16_COST.items():
        m, n, g = tiles(mi, nj)
        t = m * (n + g)
        for parts in (1, 2, 3, 4, 6, 8):
            whole = t if parts == 1 else t // CU_COUNT * CU_COUNT
            rest = t - whole
            if parts > 1 and (not rest or rest > m * n or parts > nk or rest * parts > CU_COUNT):
                continue

            def rounds(w):
                full, rem = divmod(w, CU_COUNT)
                return full + (first + (1 - first) * rem / CU_COUNT if rem else 0.0)
            us = rounds(whole) * nk * a + -(-whole // CU_COUNT) * fill
            if rest:
                us += rounds(rest * parts) * -(-nk // parts) * a + fill + e1 + (e3 if whole else 0.0) + e2 * rest * parts * min(M, 32 * mi) * 32 * nj * 8e-6
            us = (us ** 4 + floor ** 4) ** 0.25
            if best is None or us < best[0]:
                best = us, (mi, nj, whole, parts)
    return best[1]


# the same tiles with 16-bit outputs of 12 to 64 k-tiles (encoders; weights in the last-level cache): us a k-tile and a round, us to fill and
# store a round, share of a round that its first workgroup takes; plain, with GELU, and fp32 parts of K. Fitted to 2800 measurements (384 x 384
# .. 4096 x 1024, 64 to 24000 rows): picks are 0.1 % slower than the best of them on average, parts 0.7 %.
_D16_ENC_COST = (
    {(8, 8): (1.27, 8.49, 0.73), (7, 8): (1.12, 7.74, 0.74), (6, 8): (0.967, 6.9, 0.74), (5, 8): (0.851, 5.91, 0.74), (8, 6): (0.971, 6.65, 0.73),
     (6, 6): (0.785, 5.38, 0.73), (8, 4): (0.728, 4.65, 0.72), (5, 4): (0.476, 3.63, 0.75), (4, 4): (0.409, 3.25, 0.75), (2, 8): (0.614, 2.79, 0.67),
     (2, 4): (0.369, 1.66, 0.69)},
    {(8, 8): (1.11, 19.6, 0.82), (7, 8): (0.955, 17.1, 0.82), (6, 8): (0.823, 15.3, 0.81), (5, 8): (0.742, 12.9, 0.81), (8, 6): (0.825, 15.0, 0.82),
     (6, 6): (0.642, 11.9, 0.81), (8, 4): (0.607, 10.3, 0.82), (5, 4): (0.425, 7.18, 0.8), (4, 4): (0.36, 6.04, 0.83), (2, 8): (0.599, 5.53, 0.76),
     (2, 4): (0.281, 3.76, 0.83)},
    {(8, 8): (1.41, 13.7, 0.64), (7, 8): (1.23, 12.4, 0.67), (6, 8): (1.03, 11.0, 0.7), (5, 8): (0.899, 9.64, 0.69), (8, 6): (1.1, 11.0, 0.63),
     (6, 6): (0.839, 8.76, 0.66), (8, 4): (0.877, 8.06, 0.57), (5, 4): (0.571, 6.02, 0.62), (4, 4): (0.529, 5.21, 0.58), (2, 8): (0.573, 5.21, 0.67),
     (2, 4): (0.322, 3.38, 0.69)})


def _enc_tile(M: int, N_: int, K: int, kind: int, parts: int = 1):
    """(estimated us, 16 * row units + column units) of the best tile."""
    best = None
    for (mi, nj), (a, fill, first) in _D16_ENC_COST[kind].items():
        full, rem = divmod(-(-M // (32 * mi)) * -(-N_ // (32 * nj)) * parts, CU_COUNT)
        us = (full + (first + (1 - first) * rem / CU_COUNT if rem else 0.0)) * (-(-K // 64 // parts) * a + fill)
        if best is None or us < best[0]:
            best = us, 16 * mi + nj
    return best


ENC_SMALL_ROWS = 448  # where tiles do not take the widths


def small_rows(hidden: int, ffn: int) -> int:
    """Packed rows up to which encoder.hip's 16-column GEMMs are faster than the library's (they read a layer's weights once per 64 rows, so rows
    x weights decide; beyond 64 M weights a layer the library's tiles win at any row count). They run the layers up to here where dense16.hip's
    tiles do not take the widths (no whole 64s), and up to 64 rows where they do; the tiles' undivided products keep their fp32 sums up to here.

    Whole embed calls, us, one call / library GEMMs issued from Python (110 us a layer at least), all widths by these two: 384 x 1536, 12 layers, 448 rows
    679 / 1433; 768 x 3072, 12 layers, 64 rows 657 / 1374, 384 1161 / 1363, 512 1275 / 1356, 640 1488 / 1354; 1024 x 4096, 24
    layers, 64 rows 1428 / 2631, 256 2263 / 2605, 320 2857 / 2624; 1280 x 5120, 8 layers, 128 rows 828 / 910, 192 940 / 906; 1536 x
    6144, 8 layers, 96 rows 813 / 958, 128 994 / 952; 2048 x 8192, 8 layers, 48 rows 899 / 963, 128 1388 / 947; 3072 x 12288, 4
    layers, 16 rows 596 / 534, 256 2320 / 883."""
    weights = 4 * hidden * hidden + 2 * hidden * ffn
    return min(ENC_SMALL_ROWS, 3_200_000_000 // weights) if weights <= 64_000_000 else 0


@functools.lru_cache(maxsize=1024)
def encoder_plan(M: int, H: int, Fn: int) -> tuple:
    """Tiles (and parts of K) of an encoder layer's q|k|v, output, up and down products for M rows, as encoder.hip takes them. Parts that the
    LayerNorm adds up cost it 4 bytes a number each, an undivided product's sums 2 bytes where the library rounded them to 16 bits too; up to
    `small_rows` they are one fp32 part, as the 16-column GEMMs had them."""
    kind = 2 if M <= small_rows(H, Fn) else 0

    def narrow(K):
        best = None
        for parts in (1, 2, 3, 4, 8):
            if parts > K // 64 or parts > 1 and M * H * parts > 1 << 25:
                break
            us, tile = _enc_tile(M, H, K, 2 if parts > 1 else kind, parts)
            us += M * H * (4 * parts if parts > 1 or kind else 2) / 4e6
            if best is None or us < best[0]:
                best = us, (tile, parts)
        return best[1]
    return (_enc_tile(M, 3 * H, H, 0)[1], *narrow(H), _enc_tile(M, Fn, H, 1)[1], *narrow(Fn))


def takes_dense16(M: int, N_: int, K: int) -> bool:
    """Whether x w^T (bf16, fp32 out) runs dense16.hip. Measured beside the library's products in a graph, weights in no cache, us
    (library / here): long K, whose columns leave compute units idle or to products the library splits badly, 4096 x 20480 at 4 / 64 / 240 /
    944 / 1768 rows 56 / 35, 127 / 39, 225 / 58, 233 / 146, 381 / 241 (2351 and 3069 rows 333 / 336, 370 / 372), 5120 x 13824 at 64 / 101 / 693 / 3289
    47 / 34, 63 / 38, 123 / 96, 681 / 344 (up to 16 rows even), 2048 x 10240 at 64 / 512 / 2123 23 / 18, 49 / 37, 102 / 88 (8 rows 12.5 / 14), 1536 x 9216
    at 121 / 891 20 / 17, 43 / 36 (75 rows 15.4 / 16.4). Many columns by up to 64 rows: 28672 x 4096 at 5 / 33 rows 60 / 45, 50 / 46, 32000 60 / 53, 65536
    119 / 101, 123 / 103, 128256 187 / 181, 208 / 191, 50304 x 2048 48 / 40, 50 / 42, 151936 x 1536 161 / 89, 112 / 105; by up to 16 rows also 24576 x
    3072 49 / 30 (33 rows 32.2 / 32.3) and 25000 x 5120 69 / 47 (33 rows 50 / 52). The rest is the library's: 2048 x 2048 .. 4096 x 4096 are 5 to
    20 % slower here, 8192 x 8192 0.84 to 1.17, wide matrices by 65 to 300 rows 0.8 to 1.0, by more rows 0.9 to 1.5 as its choice falls.
    Where the lines lie within these, here against there (lin16.hip for few rows): few rows by 2048 columns and fewer 1.01 to 1.16 (2048 x 20480
    at 1 / 33 / 48 rows 1.16, 1.00, 0.96; 3072 x 49152 at 8 / 12 1.02, 0.98), 128 x 131072 at 128 rows 1.20, 1024 x 16384 at 64 1.09; more than 900 rows by K
    up to 8960 0.83 to 1.12, 0.99 on average; one round of 256 x 192 tiles 0.96 to 1.15 (1800 x 5120 x 13824 1.10; three of 32 0.57), all other
    tiles of 216 products of more rows and longer K 0.86 on average, 1.05 at most; many columns by K of 1024 and less 1.0 to 1.28 beyond 32000
    columns (100352 x 512 at 16 rows 1.16), by 1280 and more than 16 rows 1.04 to 1.07."""
    if K % 64 or N_ % 4 or M <= 0 or K < 64:
        return False
    if K >= 2 * N_:
        if M < 96 and N_ * K < 1 << 24 or N_ * K < 12 << 20 or N_ < 256:
            return False
        if M < 64:
            return K > 16384 and (M >= 40 or N_ >= 3072 and (K <= 32768 or M > 8))
        if M < 96:
            return K > 16384 or N_ > 1024
        if M <= 900:
            return True
        mi, nj, whole, parts = dense16_plan(M, N_, K)
        return K >= 9216 and not (mi == 8 and nj == 6 and parts == 1 and -(-M // 256) * -(-N_ // 192) <= CU_COUNT)
    if N_ >= 24576 and M <= 64:
        if K <= 2048:
            return K >= (1280 if M <= 16 else 1536) or N_ <= 32000 and 576 <= K <= 1024
        return K <= 4096 and N_ >= 28672 or K <= 5120 and M <= 16
    return False


def takes_gated16(M: int, N_: int, K: int, Fn: int) -> bool:
    """Whether a projection's N_ plain columns and its gated unit of Fn features run as one launch of dense16.hip. us, the library's product
    and the gating kernel / here: 12320 + 2 x 14336 columns x 4096 at 1 / 33 / 112 / 322 / 703 / 2062 rows 76 / 64, 78 / 67, 92 / 88, 214 / 143, 334 / 227,
    733 / 641, 6176 + 2 x 8192 x 2048 at 5 / 33 / 310 / 1693 / 3557 38 / 22, 29 / 23, 50 / 47, 197 / 158, 407 / 307 (184 rows 41 / 42), 9000 + 2 x 20000 x
    6144 134 / 111, 145 / 110, 194 / 165 (239 rows); 3000 + 2 x 5632 x 2048 even up to 64 rows (20 / 20 and 20.6 / 21.5), 465 rows 52 / 40.
    Fewer gated columns than plain ones are left apart between 64 and 1000 rows from K = 2048 on (twelve such of 48 widths and heights 1.02 to 1.27 of
    the two launches, 0.98 on average; narrower K 0.6 to 0.95), and so are up to 64 rows by fewer than 16384 columns (3840 + 2 x 5120 x 2560 1.17 to
    1.28). Of 1244 products beyond 64 rows that are taken 2 % are slower by more than 1.05, 768 + 2 x 24576 x 3072 at 80 rows by 1.14; 0.85 on average."""
    if M <= 0 or K % 64 or K < 512 or N_ <= 0 or N_ % 4 or Fn % 8 or Fn <= 0:
        return False
    n = N_ + 2 * Fn
    if M <= 64:
        return n >= 16384 and n * K >= 1 << 25
    return n * K >= 1 << 22 and (2 * Fn >= N_ or K < 2048 or M > 1000)


def _dense16(x: torch.Tensor, w: torch.Tensor, out: torch.Tensor, acc: bool, bias, gated=None) -> bool:
    """out (fp32) (+)= x w^T + bias by dense16.hip; gated = (first gate row of w, first up row, features, gate bias, up bias, 16-bit out): out
    takes the first out.shape[1] rows' products alone. False: nothing done; as for _few_rows, operands that the kernel cannot read as they
    lie and graphs that need a gradient are the library's business."""
    if not (x.is_cuda and x.dim() == 2 and out.dim() == 2 and x.dtype == w.dtype == torch.bfloat16):
        return False
    M, K = x.shape
    N_ = out.shape[1]
    if not (takes_gated16(M, N_, K, gated[2]) if gated else takes_dense16(M, N_, K)):
        return False
    if w.device != x.device or out.device != x.device or x.device.index != torch.cuda.current_device() or w.shape[1] != K \
            or (w.shape[0] < N_ if gated else w.shape[0] != N_) \
            or (torch.is_grad_enabled() and (x.requires_grad or w.requires_grad or out.requires_grad)):
        return False
    ldx, ldo = (x.stride(0), out.stride(0)) if M > 1 else (K, N_)
    if x.stride(1) != 1 or not K <= ldx <= 1 << 22 or ldx % 8 or x.data_ptr() % 16 or not w.is_contiguous() or w.data_ptr() % 16 or K > 1 << 22 \
            or out.dtype != torch.float32 or out.shape[0] != M or out.stride(1) != 1 or ldo < N_ or ldo % 4 or out.data_ptr() % 16:
        return False
    g = (0, 0, 0, None, None, None, 0)
    if gated:
        gate, up, Fn, gate_b, up_b, gout = gated
        ldg = gout.stride(0) if M > 1 else Fn
        if gout.dtype != x.dtype or gout.device != x.device or tuple(gout.shape) != (M, Fn) or gout.stride(1) != 1 or ldg < Fn or ldg % 8 \
                or gout.data_ptr() % 16 or gate < N_ or up < gate + Fn or up + Fn > w.shape[0] or w.numel() * 2 >= 1 << 32 \
                or any(b is not None and (b.dtype != torch.float32 or b.numel() != Fn or not b.is_contiguous() or b.data_ptr() % 16 or b.device != x.device)
                       for b in (gate_b, up_b)):
            return False
    if bias is not None and (bias.dtype != torch.float32 or bias.numel() != N_ or not bias.is_contiguous() or bias.data_ptr() % 16 or bias.device != x.device):
        return False
    from .. import _native as N
    mi, nj, whole, parts = dense16_plan(M, N_, K, gated[2] if gated else 0)
    part = None
    if parts > 1:
        m, cols = -(-M // (32 * mi)), 32 * nj
        t = m * (-(-N_ // cols) + (-(-2 * gated[2] // cols) if gated else 0))
        try:
            part = torch.empty((t - whole) * parts * 32 * mi * cols, dtype=torch.float32, device=x.device)
        except torch.cuda.OutOfMemoryError:
            whole, parts = t, 1  # (whole tiles need no room)
    if gated:
        g = (Fn, gate, up, N.ptr(gate_b), N.ptr(up_b), gout.data_ptr(), ldg)
    N.kcall("mxk_dense16", 4 if gated else int(acc), 16 * mi + nj, x.data_ptr(), ldx, w.data_ptr(), K, M, N_, K, N.ptr(bias), out.data_ptr(), ldo,
            whole, parts, N.ptr(part), *g, N.stream_ptr())
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
        if _dense16(x, self.w, out, False, self.b32) or self.b32 is None and _few_rows(x, self.w, out, False):
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

    def gated(self, x: torch.Tensor, out: torch.Tensor, gate: int, up: int, gate_b, up_b, gout: torch.Tensor) -> bool:
        """out (fp32 [T, n]) = x times the first n rows of W and gout (16-bit [T, F]) = silu(x W[gate:gate + F]^T + gate_b) (x W[up:up + F]^T +
        up_b) in one launch, without the gated unit's operands in memory; False where that is not done (nothing is written)."""
        return self.b32 is None and _dense16(x, self.w, out, False, None, (gate, up, gout.shape[1], gate_b, up_b, gout))

    def acc(self, x: torch.Tensor, acc: torch.Tensor) -> torch.Tensor:
        """acc (fp32) += x W^T + b — the residual add fused as GEMM beta = 1."""
        if x.dtype == torch.float32 and acc.is_contiguous():
            if self.b32 is not None:
                acc.add_(self.b32)
            torch.addmm(acc, x, self.wt, out=acc)
            return acc
        if acc.is_contiguous() and _dense16(x, self.w, acc, True, self.b32):
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
