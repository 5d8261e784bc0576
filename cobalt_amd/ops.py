"""Operator-level Python surface over the C ABI: dequant / gemv / gemm / linear on a
PackedMatrix.  torch is used for device memory and the current stream only.  The operators a
model calls per token are in the extension module (csrc/cbk_torch.cpp)."""
from __future__ import annotations

import ctypes
from typing import Optional

import torch

from . import _lib
from .format import PackedMatrix

def _stream_ptr(device) -> int:
    return torch.cuda.current_stream(device).cuda_stream


def _require_gpu(pm: PackedMatrix, *tensors):
    if pm.blob.device.type != "cuda":
        raise _lib.CbkError("the packed matrix must live on the GPU (PackedMatrix.to('cuda')); "
                            "this package has no CPU execution path")
    for t in tensors:
        if t is not None and t.device != pm.blob.device:
            raise _lib.CbkError(f"tensor on {t.device}, packed matrix on {pm.blob.device}")


def workspace_for(pm: PackedMatrix, M: int) -> Optional[torch.Tensor]:
    """A scratch tensor large enough for any operator at M activation rows, or None: for callers
    that keep one and pass it as `workspace` (the operators allocate their own without it)."""
    need = _lib.lib().cbk_workspace_bytes(ctypes.byref(pm.desc()), int(M))
    return torch.empty(need, dtype=torch.uint8, device=pm.blob.device) if need else None


def dequant(pm: PackedMatrix, dtype=torch.float32, row0: int = 0, nrows: Optional[int] = None,
            with_col_scale: bool = True) -> torch.Tensor:
    """W_hat[row0:row0+nrows] as a dense tensor (bit-exact float32 formula, one cast)."""
    return _lib.native().dequant(pm.native(), dtype, row0, pm.K - row0 if nrows is None else nrows, bool(with_col_scale))


def gemv(pm, x, bias=None, out_dtype=None, workspace=None):
    """Decode path (at most 16 activation rows)."""
    return _lib.native().matmul(0, pm.native(), x, bias, out_dtype, workspace)


def gemm(pm, x, bias=None, out_dtype=None, workspace=None):
    """Prefill path."""
    return _lib.native().matmul(1, pm.native(), x, bias, out_dtype, workspace)


def linear(pm, x, bias=None, out_dtype=None, workspace=None):
    """y = x @ W_hat.T (+ bias): decode kernel up to 8 rows, prefill kernel above."""
    return _lib.native().matmul(2, pm.native(), x, bias, out_dtype, workspace)


def linear_act(pm, x, act: str, bias=None, out_dtype=None):
    """First half of a gated MLP on a gate/up matrix (rows 2i gate, 2i+1 up):
    y[..., i] = act(t[..., 2i]) * t[..., 2i+1] with t = x @ W_hat.T (+ bias), act 'gelu_tanh' or
    'silu' (EPI_GEGLU_BF16 / EPI_SWIGLU_BF16, src/cobaltkernel/csrc/cobalt_gemm.cuh:30-33)."""
    if act not in _lib.ACT_CODE:
        raise ValueError(f"act must be one of {sorted(_lib.ACT_CODE)}, got {act!r}")
    return _lib.native().linear_act(pm.native(), x, _lib.ACT_CODE[act], bias, out_dtype)


def gemv_batch(pms, xs, biases=None, out_dtype=None):
    """Independent decode GEMVs in one launch pair: ys[i] = xs[i] @ W_hat_i.T (+ biases[i]).
    All xs share the number of rows (<= 16) and the dtype; at most 8 matrices."""
    if len(pms) == 0:
        return []
    return _lib.native().gemv_batch([pm.native() for pm in pms], list(xs), None if biases is None else list(biases), out_dtype)


class PackJob:
    """A matrix being packed on the GPU: `pm` describes it already (its zero-point flags and survivor
    count are provisional), `finish()` waits for the kernel, raises if the arrays do not fit the
    layout, and completes the description."""

    def __init__(self, mask_bits, q, scale, zero, col_scale, layout, bits=None, group=None, keep=None, fix_zero=True,
                 cs_splits=(0, 0), tiled=True):
        from . import format as F
        bits, group, kpb = F.canon(layout, bits, group, keep)
        if layout in F._SPARSE:
            raise NotImplementedError("the variable-length SPARSE4* layouts are read, not produced, by this package")
        if q.device.type != "cuda":
            raise _lib.CbkError("ops.pack_raw packs on the GPU; use format.pack_raw for tensors on the CPU")
        K, N = q.shape
        if N % 128 or N % group:
            raise ValueError(f"N={N} must be a multiple of 128 and of the group size")
        blob, (o_data, o_scale, o_zero, o_cs), cs_rows, data_bytes, self._pending = _lib.native().pack_begin(
            mask_bits, q, scale, zero, col_scale, layout, bits, group, kpb, bool(fix_zero), tiled)
        offs = {"data": o_data, "scale": o_scale, "zero": o_zero}
        if cs_rows:
            offs["col_scale"] = o_cs
        self.pm = PackedMatrix(blob, offs, K, N, layout, bits, group, kpb, cs_rows, tuple(cs_splits), data_bytes,
                               K * (N // F.BLOCK) * kpb, 0, F.FLAG_TILED16 if tiled else 0).validate()

    def finish(self) -> PackedMatrix:
        from . import format as F
        pm = self.pm
        wrong, pm.n_zero_fixed, z_max, n_mask = _lib.native().pack_end(self._pending)
        if wrong & 2:
            raise ValueError(f"{F.LAYOUT_NAME[pm.layout]} stores the zero point as the code of a pruned column, and a zero point "
                             f"of this matrix is above {(1 << pm.bits) - 1}: such a column would not dequantise to 0 (pack with "
                             f"fix_zero=True, or keep a bitmap layout)")
        if wrong & 1:
            raise ValueError(f"{F.LAYOUT_NAME[pm.layout]} needs exactly {pm.keep} survivors in every aligned block of "
                             f"{F.BLOCK} columns; the mask has a block with another count")
        if pm.layout in F._DENSE:
            pm.n_survivors = n_mask
        pm.flags |= F.zero_flags(z_max, pm.bits)
        return pm


def pack_raw(mask_bits, q, scale, zero, col_scale, layout, bits=None, group=None, keep=None, fix_zero=True,
             cs_splits=(0, 0), tiled=True) -> PackedMatrix:
    """RAW arrays on the GPU -> PackedMatrix on the GPU, written by the library's packing kernel
    (rows, scale, zero point, and the re-derivation of zero points that are off the code grid,
    src/cobaltkernel/pack_cobalt.py:55-87), in the tiled order the decode kernel streams (`tiled`)
    or the reference's row-major order.  Same arguments and same bytes as `format.pack_raw`
    (which is torch and runs anywhere)."""
    return PackJob(mask_bits, q, scale, zero, col_scale, layout, bits, group, keep, fix_zero, cs_splits, tiled).finish()


def unpack(pm: PackedMatrix):
    """(mask_bits uint8 [K, N/8], q uint8 [K, N]) of a packed matrix of any layout on the GPU: the
    inverse of `pack_raw` up to the zero-point repair (a dense layout returns its stored codes,
    the zero point at pruned columns, and an all-ones mask)."""
    _require_gpu(pm)
    q = torch.empty(pm.K, pm.N, dtype=torch.uint8, device=pm.blob.device)
    mask = torch.empty(pm.K, pm.N // 8, dtype=torch.uint8, device=pm.blob.device)
    d = pm.desc()
    _lib.check(_lib.lib().cbk_unpack(ctypes.byref(d), q.data_ptr(), mask.data_ptr(), _stream_ptr(pm.blob.device)), "cbk_unpack")
    return mask, q


def with_group_offsets(pm: PackedMatrix) -> PackedMatrix:
    """A SPARSE4 matrix as SPARSE4X: the same mask words and code bytes, plus, behind the mask
    plane of every row, the table of 16-bit byte offsets of its groups' codes that SPARSE4X / 4E
    rows carry (pack_cobalt.py:201-250: the running sum of ceil(survivors / 2) over the groups
    before), padded to 16 bytes.  Two bytes per group (0.125 bits per weight) more; with them the
    rows are served by the 16-row matrix-core stream kernel instead of the row kernel, which has
    to sum the offsets of every row itself.  Runs on the device the matrix is on."""
    from . import format as F
    if pm.layout != F.SPARSE4:
        raise ValueError("only SPARSE4 rows lack the offset table")
    K, N, G = pm.K, pm.N, pm.G
    dev = pm.device
    data = pm.array("data")
    ro = pm.array("row_off").to(torch.int64) & 0xFFFFFFFF                     # [K + 1]
    nm = N // 8
    gp = (2 * G + 15) // 16 * 16
    ar = lambda n: torch.arange(n, device=dev, dtype=torch.int64)
    mask = data[ro[:K, None] + ar(nm)[None, :]]                               # [K, N / 8]
    popc = torch.tensor([bin(i).count("1") for i in range(256)], dtype=torch.int64, device=dev)
    cnt = popc[mask.to(torch.int64)].view(K, G, pm.group // 8).sum(-1)
    gbytes = (cnt + 1) // 2
    goff = torch.cumsum(gbytes, 1) - gbytes
    if int(goff.max()) >= 1 << 16:
        raise ValueError("a row's codes exceed the 16-bit offsets of SPARSE4X")
    total = int(ro[K])
    new_ro = ro + ar(K + 1) * gp
    if int(new_ro[K]) >= 1 << 32:
        raise ValueError("the image would exceed 32-bit row offsets")
    out = torch.zeros(total + K * gp + F.BLOB_TAIL, dtype=torch.uint8, device=dev)
    out[new_ro[:K, None] + ar(nm)[None, :]] = mask
    gb = torch.stack([goff & 0xFF, goff >> 8], -1).to(torch.uint8).view(K, 2 * G)
    out[new_ro[:K, None] + nm + ar(2 * G)[None, :]] = gb
    clen = ro[1:] - ro[:K] - nm                                               # code bytes (with padding) of every row
    row = torch.repeat_interleave(ar(K), clen)
    within = ar(int(clen.sum())) - torch.repeat_interleave(torch.cumsum(clen, 0) - clen, clen)
    out[new_ro[row] + nm + gp + within] = data[ro[row] + nm + within]
    cs = pm.array("col_scale").view(pm.cs_rows, N) if pm.cs_rows else None
    res = F.from_arrays(out, pm.array("scale").view(K, G), pm.array("zero").view(K, G), cs, K, N, F.SPARSE4X,
                        pm.bits, pm.group, None, row_off=new_ro.to(torch.int32), cs_splits=pm.cs_splits, device=dev)
    res.n_survivors = pm.n_survivors
    return res


def transcode(pm: PackedMatrix, layout: int, bits=None, group=None, keep=None, tiled=True) -> PackedMatrix:
    """The same weights in another fixed-stride layout (same codes, scales, zero points and column
    scales; every weight dequantises to the same value).  The use: a survivor-stream matrix
    (SPARSE4*, which the row kernel serves at about a tenth of the matrix-core kernels' rate)
    as DENSE4, one bit per weight more for the fast kernels."""
    from . import format as F
    mask, q = unpack(pm)
    rm = pm.to_rowmajor() if pm.tiled else pm
    cs = rm.array("col_scale").view(rm.cs_rows, rm.N) if rm.cs_rows else None
    out = pack_raw(None if pm.layout in F._DENSE else mask, q, rm.array("scale").view(rm.K, rm.G), rm.array("zero").view(rm.K, rm.G),
                   cs, layout, bits, group, keep, fix_zero=False, cs_splits=rm.cs_splits, tiled=tiled)
    out.n_survivors = pm.n_survivors
    return out
