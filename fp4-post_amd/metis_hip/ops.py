"""Tensor-level entry points over the C ABI: quantize, dequantize, fused norm+quant, GEMMs.

All functions take CUDA (ROCm) tensors, enqueue on torch's current stream and return tensors;
PyTorch is used only to own device memory and streams.
"""
from __future__ import annotations

import ctypes
import functools
from dataclasses import dataclass

import torch

from . import _lib
from ._lib import B16, DTYPE_BF16, DTYPE_F32, F32, MODE_P32, MODE_PB16, U8, check, load

BLOCK = 16
_workspaces: dict = {}
# Derived copies of a cached weight cost memory beside its packed form (0.5625 B per parameter): the decode layout
# (0.5625 B) for decode-sized batches, and the tiled binary16 expansions (2 B each: one per arithmetic the layer runs in,
# one more per arithmetic for the transposed operand of the NV recipe).  Memory-bound deployments switch them off:
# without the tiled copies, binary32-arithmetic GEMMs run on the packed operands, and bf16-arithmetic GEMMs expand the
# weight on every call instead of once.  A plain unsplit product has the same bits either way; a low-rank term joins
# the binary32 sum at another point on the pipelined kernel than on the packed one (1e-6 relative in binary32).
decode_layout_weights = True
tiled_weight_copies = True
# Decode-sized activations (fewer than 256 rows, a multiple of 256 columns) leave the round-to-nearest quantizers in the
# decode layout as well: written by the quantizer's second launch, read by the decode-sized GEMM as whole lines.
decode_layout_activations = True


@dataclass
class PackedNVFP4:
    """NVFP4 tensor: value[i, k] = e2m1(codes) * e4m3(scales[i, k // 16]) * unit.

    `codes` [rows, cols/2] uint8 (element 2j in the low nibble), `scales` [rows, cols/16] uint8
    (float8_e4m3fn bytes), `unit` float32[1] on the device.  (rows, cols) is the logical shape in
    the packed orientation: for column-blocked packing of x[R, C] it is (C, R).
    """
    codes: torch.Tensor
    scales: torch.Tensor
    unit: torch.Tensor
    rows: int
    cols: int
    mode: int = MODE_P32
    expanded: torch.Tensor | None = None      # cached exact f16 expansion e2m1 * e4m3 * 2^-8, see expand()
    tiled: torch.Tensor | None = None         # exact binary16 expansion in the pipelined GEMM's tiled layout, see expand_tiled()
    tiled_pb16: torch.Tensor | None = None    # the reference's bf16 dequantized values in the same layout (bf16 arithmetic)
    transposed: "PackedNVFP4 | None" = None   # cached column-blocked packing of the same source tensor (dgrad operand)
    persistent: bool = False                  # lives across calls (a cached weight): worth keeping its tiled expansion
    shared: bool = False                      # an activation read by several GEMMs (a q/k/v or gate/up group): likewise, while it lives
    rht: int | None = None                    # NV recipe: the packed values are those of the ROTATED tensor (sign mask of the rotation)
    tiled_t: torch.Tensor | None = None       # tiled expansion of the transposed tensor (contraction over this tensor's rows)
    tiled_t_pb16: torch.Tensor | None = None
    # deferred scale bytes: the quantizer stopped after its first launch and parked the block maxima here; `scales` and
    # `unit` are produced on first access (one more launch), unless a consumer that forms the bytes itself
    # (expand_tiled) got there first and wrote the unit
    deferred: torch.Tensor | None = None
    decode_layout: torch.Tensor | None = None  # a persistent weight in the layout the decode-sized kernel streams as whole lines

    def dequantize(self, dtype: torch.dtype = torch.bfloat16) -> torch.Tensor:
        return dequantize(self, dtype)

    def held_bytes(self) -> dict:
        """Device bytes this tensor holds right now, by part: the packed form and every derived copy built so far."""
        d = self.__dict__
        parts = {"packed": self.codes.numel() + (d["_scales"].numel() if d.get("_scales") is not None else 0)}
        for name in ("expanded", "tiled", "tiled_pb16", "tiled_t", "tiled_t_pb16", "decode_layout", "deferred"):
            t = d.get(name)
            if t is not None:
                parts[name] = t.numel() * t.element_size()
        if self.transposed is not None:
            parts["transposed"] = sum(self.transposed.held_bytes().values())
        return parts

    def _materialize(self) -> None:
        d = self.__dict__
        scales = torch.empty(self.rows, self.cols // BLOCK, dtype=torch.uint8, device=self.codes.device)
        rc = load().metis_nvfp4_deferred_scales(d["deferred"].data_ptr(), self.rows, self.cols, self.mode, scales.data_ptr(),
                                                d["_unit"].data_ptr(), _stream())
        if rc:
            check(rc, "metis_nvfp4_deferred_scales", (self.rows, self.cols))
        d["_scales"], d["_unit_ready"] = scales, True


def _packed_scales(self):
    d = self.__dict__
    s = d.get("_scales")
    if s is None and d.get("deferred") is not None:
        self._materialize()
        s = d["_scales"]
    return s


def _packed_unit(self):
    d = self.__dict__
    if d.get("deferred") is not None and not d.get("_unit_ready", False):
        self._materialize()
    return d.get("_unit")


PackedNVFP4.scales = property(_packed_scales, lambda self, v: self.__dict__.__setitem__("_scales", v))
PackedNVFP4.unit = property(_packed_unit, lambda self, v: self.__dict__.__setitem__("_unit", v))


@dataclass
class CenteredNVFP4:
    """Mean-mode activation: value[i, k] = mean[k] + deq(residual)[i, k] (the column mean over tokens stays in
    high precision, only the centred residual is NVFP4).  `mean` is float32 [cols] in binary32 arithmetic,
    bf16 [cols] in bf16 arithmetic."""
    residual: PackedNVFP4
    mean: torch.Tensor
    mean32: torch.Tensor | None = None       # the same values as float32 when the producer had them at hand
    pending: tuple | None = None             # (what it was made with, partial sums of a rank-r projection) from the same launch

    @property
    def center32(self) -> torch.Tensor:
        return self.mean32 if self.mean32 is not None else self.mean

    @property
    def rows(self) -> int:
        return self.residual.rows

    @property
    def cols(self) -> int:
        return self.residual.cols

    def dequantize(self, dtype: torch.dtype = torch.bfloat16) -> torch.Tensor:
        return self.mean.to(dtype).unsqueeze(0) + dequantize(self.residual, dtype)


@dataclass
class LowRankNVFP4:
    """"svd"-mode activation: value = us @ deq(vt) + deq(residual) (reference src/Metis/Metis/bitlinear.py:296-303).
    `us` [rows, r] is U (after its QDQ) times diag(s), in the arithmetic's type; `vt` is V after its QDQ, kept packed
    (its QDQ is the packed tensor's dequantization), so that products with a packed weight run on the packed GEMM;
    `residual` packs x - ker.  `dense` (when the producer wrote it) is the reference's own tensor ker + QDQ(x - ker)."""
    residual: PackedNVFP4
    us: torch.Tensor
    vt: PackedNVFP4
    dense: torch.Tensor | None = None

    @property
    def rows(self) -> int:
        return self.residual.rows

    @property
    def cols(self) -> int:
        return self.residual.cols

    def dequantize(self, dtype: torch.dtype = torch.bfloat16) -> torch.Tensor:
        if self.dense is not None:
            return self.dense.to(dtype)
        # without the dense tensor: a library product in the arithmetic's type (agrees with the kernel's ker to rounding)
        return (self.us @ dequantize(self.vt, self.us.dtype)).to(dtype) + dequantize(self.residual, dtype)


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)
_raw_device = getattr(torch._C, "_cuda_getDevice", None)


def _stream() -> int:
    """Handle of torch's current stream on the current device (the raw getters skip the Stream object and the check for an
    initialised runtime, which a device tensor implies: this is called several times per layer)."""
    if _raw_stream is not None and _raw_device is not None:
        return _raw_stream(_raw_device())
    return torch.cuda.current_stream().cuda_stream


# Sizes that depend on the shape alone; a library call costs as much host time as an allocation.
@functools.lru_cache(maxsize=4096)
def _deferred_bytes(rows: int, cols: int) -> int:
    return int(load().metis_nvfp4_deferred_bytes(rows, cols))


@functools.lru_cache(maxsize=4096)
def _decode_operand_bytes(rows: int, cols: int) -> int:
    return int(load().metis_nvfp4_decode_operand_bytes(rows, cols))


@functools.lru_cache(maxsize=4096)
def _decode_weight_bytes(rows: int, cols: int) -> int:
    return int(load().metis_nvfp4_decode_weight_bytes(rows, cols))


@functools.lru_cache(maxsize=4096)
def _expand_tiled_bytes(rows: int, cols: int) -> int:
    return int(load().metis_nvfp4_expand_tiled_bytes(rows, cols))


@functools.lru_cache(maxsize=4096)
def _column_mean_bytes(cols: int) -> int:
    return int(load().metis_column_mean_workspace_bytes(cols))


@functools.lru_cache(maxsize=4096)
def _rmsnorm_colmean_bytes(rows: int, cols: int, device_index: int) -> int:
    return max(int(load().metis_rmsnorm_colmean_workspace_bytes(rows, cols)), 16)        # depends on the device's CU count only


@functools.lru_cache(maxsize=4096)
def _rmsnorm_backward_bytes(rows: int, cols: int, device_index: int) -> int:
    return int(load().metis_rmsnorm_backward_workspace_bytes(rows, cols))                # likewise


@functools.lru_cache(maxsize=4096)
def _lowrank_backward_bytes(L_: int, N: int, K: int, R: int, device_index: int) -> int:
    return int(load().metis_lowrank_backward_workspace_bytes(L_, N, K, R))


@functools.lru_cache(maxsize=4096)
def _quant_workspace_bytes(rows: int, cols: int) -> int:
    return int(load().metis_nvfp4_workspace_bytes(rows, cols))


@functools.lru_cache(maxsize=4096)
def _lowrank_rows_workspace_bytes(M: int, R: int, K: int, device_index: int) -> int:
    return int(load().metis_lowrank_project_rows_workspace_bytes(M, R, K))       # depends on the device's CU count only


def _workspace(rows: int, cols: int, device: torch.device, zeroed: bool = False, tensors: int = 1) -> torch.Tensor:
    """Scratch of a quantizer's call (for `tensors` packings of [rows, cols]): kept per stream, grown as needed, zero when first used.
    A captured call gets memory of its graph's pool that nobody else is handed, and takes no kept area: a fill recorded into a graph
    has not run when the next eager call comes, a replay may run beside eager work of the stream it was captured on, and a kept
    area is freed when it grows, whatever graph still writes to it.  zeroed: the call reads words that have to be zero (a maximum
    taken over the grid); the others write every word that they read."""
    need = tensors * _quant_workspace_bytes(rows, cols)
    if torch.cuda.is_current_stream_capturing():
        return _captured_workspace(need, device, zeroed)
    return _kept_workspace(need, device, tensors)


def _captured_workspace(need: int, device: torch.device, zeroed: bool) -> torch.Tensor:
    ws = torch.empty(need, dtype=torch.uint8, device=device)
    return ws.fill_(0) if zeroed else ws                           # (a fill kernel: no memset is recorded into a graph)


def _kept_workspace(need: int, device: torch.device, tensors: int = 1) -> torch.Tensor:
    key = (device.index, _stream(), tensors)
    ws = _workspaces.get(key)
    if ws is None or ws.numel() < need:
        ws = torch.empty(max(need, 1 << 20), dtype=torch.uint8, device=device).fill_(0)
        _workspaces[key] = ws
    return ws


def _as_2d_bf16(x: torch.Tensor) -> torch.Tensor:
    if not x.is_cuda:
        raise _lib.MetisHipError("metis_hip ops need a ROCm device tensor; there is no CPU path")
    if x.dtype != torch.bfloat16:
        x = x.to(torch.bfloat16)
    x2 = x if x.dim() == 2 else x.reshape(-1, x.shape[-1])
    return x2 if x2.is_contiguous() else x2.contiguous()


def _bf16_row(c: torch.Tensor) -> torch.Tensor:
    """A vector of one value per column as contiguous bf16 [cols] (what a mean of this library already is)."""
    if c.dim() == 1 and c.dtype == torch.bfloat16 and c.is_contiguous():
        return c
    return c.reshape(-1).to(torch.bfloat16).contiguous()


def _as_2d_for_quant(x: torch.Tensor, mode: int) -> tuple[torch.Tensor, int]:
    """(2-D contiguous tensor, kernel mode).  bf16 tensors go to the bf16 kernels.  In binary32 arithmetic any
    other dtype is quantized from its binary32 values (they need not be bf16 values); in bf16 arithmetic the
    tensor is first cast to bf16, as the reference casts to its compute dtype."""
    if mode == MODE_P32 and x.dtype != torch.bfloat16:
        if not x.is_cuda:
            raise _lib.MetisHipError("metis_hip ops need a ROCm device tensor; there is no CPU path")
        x2 = x.to(torch.float32).reshape(-1, x.shape[-1])
        return (x2 if x2.is_contiguous() else x2.contiguous()), _lib.MODE_P32_F32
    return _as_2d_bf16(x), mode


def quantize(x: torch.Tensor, mode: int = MODE_P32, *, col: bool = False, sr: bool = False,
             noise: torch.Tensor | None = None, seed: int = 0, offset: int = 0,
             center: torch.Tensor | TokenMean | None = None, resident: bool = False, spin_limit: int = 0,
             deferred: bool = False, pad_rows: int | None = None, checked: bool = False) -> PackedNVFP4:
    """NVFP4-quantize x (flattened to [R, C]).

    col=False: blocks of 16 along C -> PackedNVFP4 of shape (R, C).
    col=True : blocks of 16 along R, written transposed -> shape (C, R).
    sr=True  : stochastic rounding; `noise` (same shape as x, float32 for P32 / bf16 for PB16)
               overrides the internal Philox stream keyed by (seed, offset).
    center   : [C] vector subtracted from every row first (the reference's mean mode), in the arithmetic's
               dtype: the packed tensor is that of x - center.  A TokenMean: the column mean of x itself, formed in the
               same launch and left in it (deferred, bf16 arithmetic, see token_mean_applies; checked: the caller has just asked it of x).
    resident : round-to-nearest rows of a bf16 tensor as ONE launch (metis_nvfp4_quant_row_resident), same bytes: a
               workgroup that gives up waiting for the grid's maximum after `spin_limit` polls (0: library default)
               leaves its scale bytes to the last workgroup.
    deferred : round-to-nearest rows of a bf16 tensor: only the first of the two launches now (codes, parked block
               maxima); `scales` and `unit` of the result appear on first access, or never if the only consumer is
               expand_tiled, which forms the bytes itself.  Same bits either way.
    pad_rows : col=True: pack as if x had pad_rows rows, those beyond its own with a zero residual (equal to the centre,
               zero without one); no copy of x is made.  Only without caller noise.
    """
    x2, kmode = _as_2d_for_quant(x, mode)
    if isinstance(center, TokenMean):
        if not deferred or col or sr or kmode != MODE_PB16 or pad_rows is not None:
            raise ValueError("a TokenMean centre: bf16 arithmetic, rows, round to nearest, scale bytes deferred")
        return _quantize_token_mean(x2, center, checked and x2 is x)
    rows, cols = x2.shape
    if pad_rows is not None and pad_rows != rows:
        return _quantize_col_padded(x2, kmode, mode, pad_rows, col, sr, noise, seed, offset, center)
    blocked = rows if col else cols
    if blocked % BLOCK:
        raise ValueError(f"NVFP4 block shape (1, 16) does not divide tensor shape {tuple(x.shape)}")
    prow, pcol = (cols, rows) if col else (rows, cols)
    dev = x2.device
    packed = ((U8, prow, pcol // 2), (U8, prow, pcol // BLOCK), (F32, 1))
    if (deferred and not col and not sr and (center is None or kmode == MODE_PB16) and kmode in (MODE_P32, MODE_PB16)
            and x2.stride(0) == cols and rows * cols > 0):
        cen = None
        if center is not None:
            cen = center.reshape(-1).to(device=dev, dtype=torch.bfloat16).contiguous()
            if cen.numel() != cols:
                raise ValueError(f"center must have one value per column ({cols}), got {cen.numel()}")
        size = _deferred_bytes(rows, cols)
        new = _lib.call("metis_nvfp4_quant_row_deferred", dev.index, (packed[0], packed[2], (U8, size)),
                        (x2, rows, cols, kmode, cen, "0", "2", size, _stream()))
        if new.__class__ is int:
            check(new, "metis_nvfp4_quant_row_deferred", x.shape)
        return PackedNVFP4(new[0], None, new[1], prow, pcol, mode, deferred=new[2])
    ws = _workspace(rows, cols, dev, zeroed=resident)
    tail = ("0", "1", "2", ws, ws.numel(), _stream())
    if center is not None:
        cen = center.reshape(-1).to(device=dev, dtype=torch.bfloat16 if mode == MODE_PB16 else torch.float32).contiguous()
        if cen.numel() != cols:
            raise ValueError(f"center must have one value per column ({cols}), got {cen.numel()}")
        nz = None
        if sr and noise is not None:
            nz = noise.reshape(rows, cols).to(torch.bfloat16 if mode == MODE_PB16 else torch.float32).contiguous()
        name = "metis_nvfp4_quant_centered"
        new = _lib.call(name, dev.index, packed, (x2, rows, cols, x2.stride(0), kmode, cen, int(sr), int(col), nz, seed & (2 ** 64 - 1), offset, *tail))
    elif sr:
        nz = None
        if noise is not None:
            want = torch.bfloat16 if mode == MODE_PB16 else torch.float32
            nz = noise.reshape(rows, cols).to(want).contiguous()
        name = "metis_nvfp4_quant_sr_col" if col else "metis_nvfp4_quant_sr_row"
        new = _lib.call(name, dev.index, packed, (x2, rows, cols, x2.stride(0), kmode, nz, seed & (2 ** 64 - 1), offset, *tail))
    elif resident and not col and kmode in (MODE_P32, MODE_PB16) and x2.stride(0) == cols:
        name = "metis_nvfp4_quant_row_resident"
        new = _lib.call(name, dev.index, packed, (x2, rows, cols, kmode, "0", "1", "2", ws, ws.numel(), int(spin_limit), _stream()))
    elif (decode_layout_activations and not col and kmode in (MODE_P32, MODE_PB16) and 0 < rows < 256 and cols % 256 == 0
          and x2.stride(0) == cols):
        name = "metis_nvfp4_quant_row_decode"
        new = _lib.call(name, dev.index, packed + ((U8, _decode_weight_bytes(rows, cols)),),
                        (x2, rows, cols, kmode, "0", "1", "2", "3", ws, ws.numel(), _stream()))
    else:
        name = "metis_nvfp4_quant_col" if col else "metis_nvfp4_quant_row"
        new = _lib.call(name, dev.index, packed, (x2, rows, cols, x2.stride(0), kmode, *tail))
    if new.__class__ is int:
        check(new, name, x.shape)
    return PackedNVFP4(new[0], new[1], new[2], prow, pcol, mode, decode_layout=new[3] if len(new) > 3 else None)


def _quantize_col_padded(x2, kmode, mode, pad_rows, col, sr, noise, seed, offset, center) -> PackedNVFP4:
    rows, cols = x2.shape
    if not col or noise is not None or pad_rows < rows:
        raise ValueError("pad_rows: column blocks of at least as many rows as the tensor has, without caller noise")
    if pad_rows % BLOCK:
        raise ValueError(f"NVFP4 block shape (1, 16) does not divide tensor shape {(cols, pad_rows)}")
    dev = x2.device
    cen = None
    if center is not None:
        cen = center.reshape(-1).to(device=dev, dtype=torch.bfloat16 if mode == MODE_PB16 else torch.float32).contiguous()
        if cen.numel() != cols:
            raise ValueError(f"center must have one value per column ({cols}), got {cen.numel()}")
    ws = _workspace(pad_rows, cols, dev)
    new = _lib.call("metis_nvfp4_quant_col_padded", dev.index, ((U8, cols, pad_rows // 2), (U8, cols, pad_rows // BLOCK), (F32, 1)),
                    (x2, rows, pad_rows, cols, x2.stride(0), kmode, cen, int(sr), seed & (2 ** 64 - 1), offset, "0", "1", "2", ws, ws.numel(), _stream()))
    if new.__class__ is int:
        check(new, "metis_nvfp4_quant_col_padded", (rows, cols))
    return PackedNVFP4(*new, cols, pad_rows, mode)


def quantize_dequantize(x: torch.Tensor, mode: int = MODE_P32) -> tuple[PackedNVFP4, torch.Tensor]:
    """(quantize(x, mode), its dequantized bf16 tensor) of a bf16 tensor with round to nearest, from one call of two
    launches: the second forms scale bytes and dequantized values in one pass over the codes.  Same bytes as
    quantize() followed by dequantize()."""
    if x.dtype != torch.bfloat16 or mode not in (MODE_P32, MODE_PB16):
        p = quantize(x, mode)
        return p, dequantize(p, torch.bfloat16)
    x2 = _as_2d_bf16(x)
    rows, cols = x2.shape
    if cols % BLOCK:
        raise ValueError(f"NVFP4 block shape (1, 16) does not divide tensor shape {tuple(x.shape)}")
    dev = x2.device
    codes = torch.empty(rows, cols // 2, dtype=torch.uint8, device=dev)
    scales = torch.empty(rows, cols // BLOCK, dtype=torch.uint8, device=dev)
    unit = torch.empty(1, dtype=torch.float32, device=dev)
    out = torch.empty(rows, cols, dtype=torch.bfloat16, device=dev)
    ws = _workspace(rows, cols, dev)
    rc = load().metis_nvfp4_quant_dequant_row(x2.data_ptr(), rows, cols, mode, codes.data_ptr(), scales.data_ptr(), unit.data_ptr(),
                                              out.data_ptr(), ws.data_ptr(), ws.numel(), _stream())
    if rc:
        check(rc, "metis_nvfp4_quant_dequant_row", x.shape)
    return PackedNVFP4(codes, scales, unit, rows, cols, mode), out


def quantize_dequantize_f32(x: torch.Tensor) -> tuple[PackedNVFP4, torch.Tensor]:
    """quantize_dequantize of a binary32 tensor in binary32 arithmetic: (quantize(x), its dequantized binary32 tensor)."""
    if x.dtype != torch.float32 or not x.is_cuda:
        raise ValueError("quantize_dequantize_f32: a float32 device tensor")
    x2 = x.reshape(-1, x.shape[-1])
    x2 = x2 if x2.is_contiguous() else x2.contiguous()
    rows, cols = x2.shape
    if cols % BLOCK:
        raise ValueError(f"NVFP4 block shape (1, 16) does not divide tensor shape {tuple(x.shape)}")
    dev = x2.device
    codes = torch.empty(rows, cols // 2, dtype=torch.uint8, device=dev)
    scales = torch.empty(rows, cols // BLOCK, dtype=torch.uint8, device=dev)
    unit = torch.empty(1, dtype=torch.float32, device=dev)
    out = torch.empty(rows, cols, dtype=torch.float32, device=dev)
    ws = _workspace(rows, cols, dev)
    rc = load().metis_nvfp4_quant_dequant_row_f32(x2.data_ptr(), rows, cols, codes.data_ptr(), scales.data_ptr(), unit.data_ptr(), out.data_ptr(),
                                                  ws.data_ptr(), ws.numel(), _stream())
    if rc:
        check(rc, "metis_nvfp4_quant_dequant_row_f32", x.shape)
    return PackedNVFP4(codes, scales, unit, rows, cols, MODE_P32), out


@functools.lru_cache(maxsize=4096)
def _roundtrip_scratch(rows: int, cols: int, kmode: int, device_index: int) -> int | None:
    """Bytes of zeroed scratch that the round trip of this shape reads (0: a small tensor), None if it is too large; depends on the device's
    capacity only."""
    need = ctypes.c_size_t(0)
    rc = load().metis_nvfp4_roundtrip_applies(rows, cols, kmode, ctypes.addressof(need))
    if rc and rc != _lib.E_TOO_LARGE:
        check(rc, "metis_nvfp4_roundtrip", (rows, cols))
    return None if rc else need.value


# Elements from which a captured round trip takes the grid-wide maximum.  In a graph its area is cleared in every replay, a launch of its
# own (about 2 us): with it 768 x 4096 10.5 us in bf16 and 12.8 in binary32 where the two launches of the packed form take 9.8 and 11.7;
# 1024 x 4096 10.6 and 14.2 against 11.1 and 14.4, 4096 x 4096 19.2 and 30.0 against 22.6 and 32.6.
_ROUNDTRIP_CAPTURED = 1 << 22


def roundtrip(x: torch.Tensor, spin_limit: int = 0) -> torch.Tensor | None:
    """dequantize(quantize(x)) of a bf16 tensor in bf16 arithmetic or a binary32 tensor in binary32 arithmetic, round to nearest: the
    same values in x's shape and type, from one launch that packs nothing.  None where half of the device's registers do not hold
    the tensor's codes, and in a capture where the packed form is faster.  spin_limit: polls for the grid's maximum before a
    workgroup leaves its values to the last one (0: the library's limit)."""
    x2 = x if (x.dim() == 2 and x.is_contiguous()) else x.reshape(-1, x.shape[-1]).contiguous()
    rows, cols = x2.shape
    kmode = MODE_PB16 if x.dtype == torch.bfloat16 else _lib.MODE_P32_F32
    need = _roundtrip_scratch(rows, cols, kmode, x.device.index or 0)
    if need is None:
        return None
    ws = None
    if need and torch.cuda.is_current_stream_capturing():
        if rows * cols < _ROUNDTRIP_CAPTURED:
            return None
        ws = _captured_workspace(need, x.device, True)
    elif need:
        ws = _kept_workspace(need, x.device)
    new = _lib.call("metis_nvfp4_roundtrip", x.device.index, ((B16 if kmode == MODE_PB16 else F32, *x.shape),),
                    (x2, rows, cols, kmode, "0", ws, need, int(spin_limit), _stream()))
    if new.__class__ is int:
        check(new, "metis_nvfp4_roundtrip", x.shape)
    return new[0]


def quantize_lowrank_residual(x: torch.Tensor, us: torch.Tensor, vt: torch.Tensor, mode: int = MODE_P32,
                              dense: bool = False) -> tuple[PackedNVFP4, torch.Tensor | None]:
    """The packed residual QDQ(x - ker) with ker = us @ vt formed in registers (the "svd" mode of the activation
    decomposition, src/Metis/Metis/bitlinear.py:296-303), and with dense=True also ker + QDQ(x - ker).
    MODE_P32: us, vt binary32, x bf16 or binary32, dense binary32; MODE_PB16: all bf16.  x [rows, cols], us [rows, r],
    vt [r, cols], r a multiple of 16.  ker sums its r products in the order k = 0 .. r-1 with fused multiply-adds."""
    if not x.is_cuda:
        raise RuntimeError("metis_hip kernels need tensors on the GPU")
    x2 = x.reshape(-1, x.shape[-1]).contiguous()
    rows, cols = x2.shape
    r = us.shape[-1]
    want = torch.float32 if mode == MODE_P32 else torch.bfloat16
    if mode not in (MODE_P32, MODE_PB16) or us.dtype != want or vt.dtype != want:
        raise ValueError("the factors come in the arithmetic's type: binary32 for MODE_P32, bf16 for MODE_PB16")
    if x2.dtype != torch.bfloat16 and not (mode == MODE_P32 and x2.dtype == torch.float32):
        raise ValueError(f"unsupported tensor type {x2.dtype} for this arithmetic")
    if tuple(us.shape) != (rows, r) or tuple(vt.shape) != (r, cols):
        raise ValueError(f"factors {tuple(us.shape)} x {tuple(vt.shape)} do not give {tuple(x2.shape)}")
    if cols % BLOCK or r % BLOCK or r == 0:
        raise ValueError(f"NVFP4 block shape (1, 16) does not divide {tuple(x.shape)} or the rank {r}")
    us, vt = us.contiguous(), vt.contiguous()
    dev = x2.device
    ws = _workspace(rows, cols, dev)
    specs = ((U8, rows, cols // 2), (U8, rows, cols // BLOCK), (F32, 1))
    if dense:
        specs += ((F32 if want == torch.float32 else B16, rows, cols),)
    new = _lib.call("metis_nvfp4_quant_lowrank_residual", dev.index, specs,
                    (x2, DTYPE_F32 if x2.dtype == torch.float32 else DTYPE_BF16, us, vt, rows, cols, r, mode, "0", "1", "2", "3" if dense else None,
                     ws, ws.numel(), _stream()))
    if new.__class__ is int:
        check(new, "metis_nvfp4_quant_lowrank_residual", (rows, cols, r))
    return PackedNVFP4(new[0], new[1], new[2], rows, cols, mode), new[3] if dense else None


def _check_bf16_copy(copy: torch.Tensor | None, x2: torch.Tensor, kmode: int) -> None:
    if copy is not None and (kmode != _lib.MODE_P32_F32 or copy.dtype != torch.bfloat16 or copy.shape != x2.shape or not copy.is_contiguous()
                             or copy.device != x2.device):
        raise ValueError("bf16_copy: a contiguous bfloat16 tensor of the flattened shape, for a binary32 tensor in binary32 arithmetic")


def quantize_both_sr(x: torch.Tensor, mode: int = MODE_P32, *, seed: int = 0, offset_row: int = 0,
                     offset_col: int = 0, pad_rows: int | None = None,
                     bf16_copy: torch.Tensor | None = None, center: torch.Tensor | None = None) -> tuple[PackedNVFP4, PackedNVFP4]:
    """(quantize(x, sr=True, offset=offset_row), quantize(x, col=True, sr=True, offset=offset_col)) from ONE pass over x:
    the two packings of an output gradient that the input-gradient and weight-gradient products contract.  Same
    bytes as the two calls.  Both dimensions of x flattened to [R, C] have to be multiples of 16; with pad_rows, that
    and C: the column packing is that of x filled up with zero rows to pad_rows, the row packing that of x.
    bf16_copy (a binary32 x in binary32 arithmetic): bf16 [R, C], contiguous: the same pass leaves x.to(bfloat16) in it.
    center: [C] subtracted from every row first, as in quantize; in bf16 arithmetic, or of a binary32 x in binary32 arithmetic."""
    x2, kmode = _as_2d_for_quant(x, mode)
    if center is not None:
        if bf16_copy is not None or kmode == MODE_P32:
            raise ValueError("quantize_both_sr: a centre in bf16 arithmetic or for a binary32 tensor, and without bf16_copy")
        center = center.reshape(-1).to(device=x2.device, dtype=torch.bfloat16 if kmode == MODE_PB16 else torch.float32).contiguous()
        if center.numel() != x2.shape[1]:
            raise ValueError(f"center must have one value per column ({x2.shape[1]}), got {center.numel()}")
    _check_bf16_copy(bf16_copy, x2, kmode)
    have, cols = x2.shape
    rows = have if pad_rows is None else pad_rows
    if rows < have:
        raise ValueError("pad_rows: at least as many rows as the tensor has")
    if rows % BLOCK or cols % BLOCK:
        raise ValueError(f"NVFP4 block shape (1, 16) does not divide tensor shape {tuple(x.shape)} both ways")
    dev = x2.device
    specs = ((U8, rows, cols // 2), (U8, rows, cols // BLOCK), (F32, 1), (U8, cols, rows // 2), (U8, cols, rows // BLOCK), (F32, 1))
    ws = _workspace(rows, cols, dev, tensors=2)
    seeds, outs = (seed & (2 ** 64 - 1), offset_row, offset_col), ("0", "1", "2", "3", "4", "5")
    if not rows * cols:
        new = tuple([torch.empty(*size, dtype=torch.uint8 if kind == U8 else torch.float32, device=dev) for kind, *size in specs])
    elif center is not None:
        name = "metis_nvfp4_quant_sr_both_centered"
        new = _lib.call(name, dev.index, specs, (x2, have, rows, cols, x2.stride(0), kmode, center, *seeds, *outs, ws, ws.numel(), _stream()))
    elif bf16_copy is not None:
        name = "metis_nvfp4_quant_sr_both_copy"
        new = _lib.call(name, dev.index, specs, (x2, have, rows, cols, x2.stride(0), *seeds, *outs, bf16_copy, ws, ws.numel(), _stream()))
    else:
        name = "metis_nvfp4_quant_sr_both_padded"
        new = _lib.call(name, dev.index, specs, (x2, have, rows, cols, x2.stride(0), kmode, *seeds, *outs, ws, ws.numel(), _stream()))
    if new.__class__ is int:
        check(new, name, x.shape)
    cr, sr_, ur, cc, sc, uc = new
    if have != rows:
        cr, sr_ = cr[:have], sr_[:have]
    return PackedNVFP4(cr, sr_, ur, have, cols, mode), PackedNVFP4(cc, sc, uc, cols, rows, mode)


def dequantize(p: PackedNVFP4, dtype: torch.dtype = torch.bfloat16) -> torch.Tensor:
    if dtype not in (torch.bfloat16, torch.float32):
        raise ValueError("dequantize: dtype must be bfloat16 or float32")
    out = torch.empty(p.rows, p.cols, dtype=dtype, device=p.codes.device)
    rc = load().metis_nvfp4_dequant(p.codes.data_ptr(), p.scales.data_ptr(), p.unit.data_ptr(), p.rows, p.cols,
                                    p.mode, out.data_ptr(), DTYPE_F32 if dtype == torch.float32 else DTYPE_BF16,
                                    _stream())
    if rc:
        check(rc, "metis_nvfp4_dequant", (p.rows, p.cols))
    if p.rht is not None:                     # packed in the rotated domain: back to the tensor's own
        out = hadamard16(out, p.rht, inverse=True)
    return out


def hadamard16(x: torch.Tensor, sign_mask: int, inverse: bool = False) -> torch.Tensor:
    """Tiled random Hadamard rotation along the last dimension, tiles of 16: (x * sign) H, or the rotation back
    (x H) / 16 * sign (reference bitlinear.py:195-202).  bf16 or float32, same dtype out."""
    if x.dtype not in (torch.bfloat16, torch.float32) or not x.is_cuda:
        raise ValueError("hadamard16: bf16 or float32 device tensor")
    cols = x.shape[-1]
    x2 = x.reshape(-1, cols)
    if not x2.is_contiguous():
        x2 = x2.contiguous()
    out = torch.empty_like(x2)
    rc = load().metis_hadamard16(x2.data_ptr(), x2.shape[0], cols, cols, DTYPE_F32 if x.dtype == torch.float32 else DTYPE_BF16,
                                 int(inverse), int(sign_mask), out.data_ptr(), cols, _stream())
    if rc:
        check(rc, "metis_hadamard16", tuple(x.shape))
    return out.reshape(x.shape)


def quantize_rht(x: torch.Tensor, mode: int, sign_mask: int, *, sr: bool = False, seed: int = 0, offset: int = 0,
                 bf16_copy: torch.Tensor | None = None) -> PackedNVFP4:
    """Row quantizer of the ROTATED tensor (NV recipe): rotation and quantization in one pass over x.  The result
    carries `rht` = sign_mask; its dequantize() and tiled expansions rotate back.  bf16_copy: as in quantize_both_sr."""
    x2, kmode = _as_2d_for_quant(x, mode)
    _check_bf16_copy(bf16_copy, x2, kmode)
    rows, cols = x2.shape
    if cols % BLOCK:
        raise ValueError(f"last dimension {cols} is not a multiple of {BLOCK}")
    dev = x2.device
    codes = torch.empty(rows, cols // 2, dtype=torch.uint8, device=dev)
    scales = torch.empty(rows, cols // BLOCK, dtype=torch.uint8, device=dev)
    unit = torch.empty(1, dtype=torch.float32, device=dev)
    ws = _workspace(rows, cols, dev)
    if bf16_copy is not None:
        rc = load().metis_nvfp4_quant_row_rht_copy(x2.data_ptr(), rows, cols, x2.stride(0), int(sign_mask), int(sr), int(seed), int(offset),
                                                   codes.data_ptr(), scales.data_ptr(), unit.data_ptr(), bf16_copy.data_ptr(), ws.data_ptr(),
                                                   ws.numel(), _stream())
        if rc:
            check(rc, "metis_nvfp4_quant_row_rht_copy", (rows, cols))
        return PackedNVFP4(codes, scales, unit, rows, cols, MODE_P32, rht=int(sign_mask))
    rc = load().metis_nvfp4_quant_row_rht(x2.data_ptr(), rows, cols, x2.stride(0), kmode, int(sign_mask), int(sr), int(seed), int(offset),
                                          codes.data_ptr(), scales.data_ptr(), unit.data_ptr(), ws.data_ptr(), ws.numel(), _stream())
    if rc:
        check(rc, "metis_nvfp4_quant_row_rht", (rows, cols))
    return PackedNVFP4(codes, scales, unit, rows, cols, MODE_PB16 if mode == MODE_PB16 else MODE_P32, rht=int(sign_mask))


def column_sum(x: torch.Tensor, out_dtype: torch.dtype = torch.float32) -> torch.Tensor:
    """Sum over the rows of x flattened to [R, C] -> [C] (binary32 accumulation; bf16 or float32 in and out)."""
    return column_mean(x, out_dtype, _sum_only=True)


def column_mean(x: torch.Tensor, out_dtype: torch.dtype = torch.float32, _sum_only: bool = False) -> torch.Tensor:
    """Mean over the rows of x flattened to [R, C] -> [C] (binary32 accumulation; bf16 or float32 in and out)."""
    if not x.is_cuda:
        raise _lib.MetisHipError("metis_hip ops need a ROCm device tensor; there is no CPU path")
    if x.dtype not in (torch.bfloat16, torch.float32) or out_dtype not in (torch.bfloat16, torch.float32):
        raise ValueError("column_mean: bfloat16 or float32 tensors only")
    x2 = x.reshape(-1, x.shape[-1])
    if not x2.is_contiguous():
        x2 = x2.contiguous()
    rows, cols = x2.shape
    out = torch.empty(cols, dtype=out_dtype, device=x2.device)
    L = load()
    ws = torch.empty(_column_mean_bytes(cols), dtype=torch.uint8, device=x2.device)
    fn = L.metis_column_sum if _sum_only else L.metis_column_mean
    rc = fn(x2.data_ptr(), rows, cols, x2.stride(0), DTYPE_F32 if x2.dtype == torch.float32 else DTYPE_BF16,
            out.data_ptr(), DTYPE_F32 if out_dtype == torch.float32 else DTYPE_BF16, ws.data_ptr(), ws.numel(), _stream())
    check(rc, "metis_column_sum" if _sum_only else "metis_column_mean", x.shape)
    return out


def column_mean_running(x: torch.Tensor, cached: torch.Tensor | None, cached_count: int,
                        out_dtype: torch.dtype = torch.float32) -> tuple[torch.Tensor, torch.Tensor]:
    """(me, me as float32) with me = (cached * cached_count + mean(x) * rows) / (cached_count + rows), each operation
    rounded to out_dtype (cached None: me = mean(x)).  One reduction and one small kernel; in float32 both results
    are the same tensor."""
    if not x.is_cuda:
        raise _lib.MetisHipError("metis_hip ops need a ROCm device tensor; there is no CPU path")
    if x.dtype not in (torch.bfloat16, torch.float32) or out_dtype not in (torch.bfloat16, torch.float32):
        raise ValueError("column_mean_running: bfloat16 or float32 tensors only")
    x2 = x.reshape(-1, x.shape[-1])
    if not x2.is_contiguous():
        x2 = x2.contiguous()
    rows, cols = x2.shape
    if cached is not None:
        cached = cached.reshape(-1).to(device=x2.device, dtype=out_dtype).contiguous()
        if cached.numel() != cols:
            raise ValueError(f"cached mean has {cached.numel()} values, the tensor {cols} columns")
    out = torch.empty(cols, dtype=out_dtype, device=x2.device)
    out32 = out if out_dtype == torch.float32 else torch.empty(cols, dtype=torch.float32, device=x2.device)
    L = load()
    ws = torch.empty(_column_mean_bytes(cols), dtype=torch.uint8, device=x2.device)
    rc = L.metis_column_mean_running(x2.data_ptr(), rows, cols, x2.stride(0), DTYPE_F32 if x2.dtype == torch.float32 else DTYPE_BF16,
                                     None if cached is None else cached.data_ptr(), int(cached_count), out.data_ptr(),
                                     None if out32 is out else out32.data_ptr(),
                                     DTYPE_F32 if out_dtype == torch.float32 else DTYPE_BF16, ws.data_ptr(), ws.numel(), _stream())
    if rc:
        check(rc, "metis_column_mean_running", x.shape)
    return out, out32


@functools.lru_cache(maxsize=4096)
def _token_mean_takes(rows: int, cols: int, after_norm: int, device_index: int) -> bool:
    return bool(load().metis_token_mean_quant_applies(rows, cols, after_norm))       # depends on the device's CU count only


TOKEN_MEAN_MAX_ROWS = 768


def token_mean_applies(x2: torch.Tensor, after_norm: bool) -> bool:
    """quantize() with a TokenMean centre takes this tensor: few rows (a decode step, a short prompt), contiguous bf16.  Beyond 768 rows a
    narrow tensor's strips are too few workgroups for the work (times beside the kernel, token_mean_quant.hip)."""
    return (x2.is_cuda and x2.dtype == torch.bfloat16 and x2.dim() == 2 and 0 < x2.shape[0] <= TOKEN_MEAN_MAX_ROWS and x2.shape[1] % 32 == 0
            and x2.is_contiguous() and x2.data_ptr() % 16 == 0
            and _token_mean_takes(x2.shape[0], x2.shape[1], int(after_norm), x2.device.index or 0))


@dataclass
class TokenMean:
    """A centre that quantize() forms itself in the launch that subtracts it: the column mean of the tensor over its rows, as
    column_mean_running(x, cached, cached_count, bfloat16) gives it -- or, after_norm, as rmsnorm_colmean does of its normed tensor.
    v (bf16 [r, cols], optional): the same launch leaves the partial sums of x . v^T for project_and_operand(..., pending=)."""
    after_norm: bool = False
    cached: torch.Tensor | None = None
    cached_count: int = 0
    v: torch.Tensor | None = None
    # results
    mean: torch.Tensor | None = None
    mean32: torch.Tensor | None = None
    pending: torch.Tensor | None = None


def _quantize_token_mean(x2: torch.Tensor, tm: TokenMean, checked: bool) -> PackedNVFP4:
    if not (checked or token_mean_applies(x2, tm.after_norm)):
        raise ValueError("a TokenMean centre: outside the call's domain (see token_mean_applies)")
    after_norm, cached, cached_count, v = tm.after_norm, tm.cached, tm.cached_count, tm.v
    rows, cols = x2.shape
    dev = x2.device
    if cached is not None:
        cached = cached.to(device=dev, dtype=torch.bfloat16).contiguous()
        if cached.numel() != cols:
            raise ValueError(f"cached mean has {cached.numel()} values, the tensor {cols} columns")
    size = _deferred_bytes(rows, cols)
    specs = ((B16, cols), (F32, cols), (U8, rows, cols // 2), (F32, 1), (U8, size))
    R = need = 0
    pending = None
    if v is not None:
        v = v.contiguous()
        R = v.shape[0]
        if v.dtype != torch.bfloat16 or v.shape[1] != cols or v.device != dev:
            raise ValueError("TokenMean: v is bfloat16 [r, cols] on the tensor's device")
        need = _lowrank_workspace_bytes(rows, R, cols)
        specs += ((U8, need),)
        pending = "5"
    new = _lib.call("metis_token_mean_quant_deferred", dev.index, specs,
                    (x2, rows, cols, after_norm, cached, int(cached_count), "0", "1", "2", "4", size, v, R, pending, need, _stream()))
    if new.__class__ is int:
        check(new, "metis_token_mean_quant_deferred", (rows, cols, R))
    me, me32, codes, unit, parked = new[:5]
    pending = None if v is None else new[5]
    tm.mean, tm.mean32, tm.pending = me, me32, pending
    return PackedNVFP4(codes, None, unit, rows, cols, MODE_PB16, deferred=parked)


def matvec(p: PackedNVFP4, v: torch.Tensor | None = None, alpha: float = 1.0, *, out: torch.Tensor | None = None,
           split: torch.Tensor | None = None, split_col: int = 0, z: torch.Tensor | None = None,
           beta: float = 0.0) -> torch.Tensor | None:
    """y[i] = alpha * sum_k deq(p)[i, k] * v[k] (+ beta * z[i]) in binary32 (v=None: all ones, i.e. row sums).

    Returns y as float32 [rows] (written into `out` when given).  With `split` (a bf16 matrix with at least
    split_col + 3 columns) y is also stored as three bf16 terms hi + mid + lo in columns split_col..+2 of
    its rows; with split given and out=None nothing else is allocated and None is returned."""
    dev = p.codes.device
    vp = None
    if v is not None:
        v = v.reshape(-1).to(device=dev, dtype=torch.float32).contiguous()
        if v.numel() != p.cols:
            raise ValueError(f"vector length {v.numel()} does not match the packed tensor's {p.cols} columns")
        vp = v.data_ptr()
    if out is None and (split is None or z is not None):
        out = torch.empty(p.rows, dtype=torch.float32, device=dev)
    if z is not None:
        if split is not None:
            raise ValueError("matvec: the affine tail and the split output are separate entry points")
        z = z.reshape(-1).to(device=dev, dtype=torch.float32).contiguous()
        if z.numel() != p.rows:
            raise ValueError(f"z must have one value per packed row ({p.rows}), got {z.numel()}")
        rc = load().metis_nvfp4_matvec_affine(p.codes.data_ptr(), p.scales.data_ptr(), p.unit.data_ptr(), p.rows, p.cols, vp,
                                              float(alpha), z.data_ptr(), float(beta), out.data_ptr(), _stream())
        if rc:
            check(rc, "metis_nvfp4_matvec_affine", (p.rows, p.cols))
        return out
    sp, sld = None, 0
    if split is not None:
        if split.dtype != torch.bfloat16 or split.dim() != 2 or split.shape[0] != p.rows or split.stride(1) != 1:
            raise ValueError("split must be a bf16 matrix with one row per packed row and unit column stride")
        sp, sld = split.data_ptr(), split.stride(0)
    rc = load().metis_nvfp4_matvec(p.codes.data_ptr(), p.scales.data_ptr(), p.unit.data_ptr(), p.rows, p.cols, vp,
                                   float(alpha), None if out is None else out.data_ptr(), sp, sld, int(split_col), _stream())
    if rc:
        check(rc, "metis_nvfp4_matvec", (p.rows, p.cols))
    return out


def rank_one_operands(n: int, k: int, first: tuple | None, second: tuple | None = None):
    """(t [n, 32], u [k, 32]) bf16 with t u^T = a1 b1^T (+ a2 b2^T) to binary32 precision; first = (a1 [n], b1 [k]),
    second = (a2, b2) or None.  They go into linear_fwd as its low-rank operands."""
    pairs = [pr for pr in (first, second) if pr is not None]
    if not pairs:
        raise ValueError("rank_one_operands: at least one (a, b) pair")
    dev = pairs[0][0].device
    ptrs, keep = [], []
    for a, b in pairs:
        a = a.reshape(-1).to(torch.float32).contiguous()
        b = b.reshape(-1).to(torch.float32).contiguous()
        if a.numel() != n or b.numel() != k:
            raise ValueError("rank_one_operands: a must have n values and b must have k")
        keep += [a, b]
        ptrs += [a.data_ptr(), b.data_ptr()]
    while len(ptrs) < 4:
        ptrs.append(None)
    t = torch.empty(n, 32, dtype=torch.bfloat16, device=dev)
    u = torch.empty(k, 32, dtype=torch.bfloat16, device=dev)
    rc = load().metis_rank_one_operands(ptrs[0], ptrs[1], ptrs[2], ptrs[3], n, k, t.data_ptr(), u.data_ptr(), _stream())
    if rc:
        check(rc, "metis_rank_one_operands", (n, k))
    return t, u


def expand(p: PackedNVFP4) -> torch.Tensor:
    """Exact binary16 expansion e2m1(code) * e4m3(scale) * 2^-8 of a packed tensor, cached on it.

    Costs 2 B/element of HBM; it is what the compute-bound GEMM path consumes (MFMA and LDS reads only
    in its inner loop)."""
    if p.expanded is None:
        out = torch.empty(p.rows, p.cols, dtype=torch.float16, device=p.codes.device)
        rc = load().metis_nvfp4_expand_f16(p.codes.data_ptr(), p.scales.data_ptr(), p.rows, p.cols, out.data_ptr(), _stream())
        if rc:
            check(rc, "metis_nvfp4_expand_f16", (p.rows, p.cols))
        p.expanded = out
    return p.expanded


def expand_tiled(p: PackedNVFP4, cache: bool = True, mode: int = MODE_P32, center: torch.Tensor | None = None) -> torch.Tensor:
    """16-bit expansion of a packed tensor in the tiled layout of the pipelined GEMM (uint8 buffer): exact binary16
    values e2m1 * e4m3 * 2^-8 (mode P32) or the reference's bf16 dequantized values, unit included (mode PB16).
    cache=True keeps it on the packed tensor (weights); activations are expanded per call.
    center (bf16 [cols], mode PB16): p packs a centred residual; the operand is the mean mode's center + QDQ(x - center)
    rounded to bf16, the tensor the reference multiplies with in bf16 arithmetic."""
    dev, spec = p.codes.device.index, ((U8, _expand_tiled_bytes(p.rows, p.cols)),)
    d = p.__dict__
    lazy = d.get("deferred") is not None and d.get("_scales") is None and p.rht is None and p.cols % 32 == 0
    if center is not None:
        if mode != MODE_PB16 or p.rht is not None:
            raise ValueError("a centre goes into the bf16-arithmetic operand of an unrotated tensor")
        center = _bf16_row(center)
        if center.numel() != p.cols:
            raise ValueError(f"center must have {p.cols} values, got {center.numel()}")
        key = (center.data_ptr(), center._version)
        kept = d.get("_tiled_centered")
        if cache and kept is not None and kept[0] == key:
            return kept[1]
        if lazy:
            new = _lib.call("metis_nvfp4_expand_tiled_deferred", dev, spec, (p.codes, d["deferred"], p.rows, p.cols, p.mode, mode, center, d["_unit"], "0", _stream()))
            d["_unit_ready"] = True
        else:
            new = _lib.call("metis_nvfp4_expand_tiled_centered", dev, spec, (p.codes, p.scales, p.unit, p.rows, p.cols, center, "0", _stream()))
        if new.__class__ is int:
            check(new, "metis_nvfp4_expand_tiled_centered", (p.rows, p.cols))
        out = new[0]
        if cache:
            d["_tiled_centered"] = (key, out, center)                 # (the centre is kept alive with its address)
        return out
    have = p.tiled_pb16 if mode == MODE_PB16 else p.tiled
    if have is not None:
        return have
    if lazy:
        # the scale bytes were never written: this kernel forms them from the parked block maxima, and writes the unit
        new = _lib.call("metis_nvfp4_expand_tiled_deferred", dev, spec, (p.codes, d["deferred"], p.rows, p.cols, p.mode, mode, None, d["_unit"], "0", _stream()))
        if new.__class__ is int:
            check(new, "metis_nvfp4_expand_tiled_deferred", (p.rows, p.cols))
        d["_unit_ready"] = True
    elif p.rht is not None:                   # NV recipe: the operand holds the values rotated back
        new = _lib.call("metis_nvfp4_expand_tiled_rht", dev, spec, (p.codes, p.scales, p.unit, p.rows, p.cols, mode, p.rht, 1, 0, "0", _stream()))
    else:
        new = _lib.call("metis_nvfp4_expand_tiled", dev, spec, (p.codes, p.scales, p.unit, p.rows, p.cols, mode, "0", _stream()))
    if new.__class__ is int:
        check(new, "metis_nvfp4_expand_tiled", (p.rows, p.cols))
    out = new[0]
    if cache and (tiled_weight_copies or not p.persistent):
        if mode == MODE_PB16:
            p.tiled_pb16 = out
        else:
            p.tiled = out
    return out


def expand_tiled_transposed(p: PackedNVFP4, cache: bool = False, mode: int = MODE_P32) -> torch.Tensor:
    """expand_tiled of the TRANSPOSED tensor: the operand [cols, rows] of a GEMM that contracts over this tensor's
    rows (rows % 32 == 0); a rotated tensor (NV recipe) is rotated back block by block on the way."""
    have = p.tiled_t_pb16 if mode == MODE_PB16 else p.tiled_t
    if have is not None:
        return have
    L = load()
    out = torch.empty(L.metis_nvfp4_expand_tiled_bytes(p.cols, p.rows), dtype=torch.uint8, device=p.codes.device)
    rc = L.metis_nvfp4_expand_tiled_rht(p.codes.data_ptr(), p.scales.data_ptr(), p.unit.data_ptr(), p.rows, p.cols, mode,
                                        p.rht or 0, int(p.rht is not None), 1, out.data_ptr(), _stream())
    if rc:
        check(rc, "metis_nvfp4_expand_tiled_rht", (p.rows, p.cols))
    if cache and (tiled_weight_copies or not p.persistent):
        if mode == MODE_PB16:
            p.tiled_t_pb16 = out
        else:
            p.tiled_t = out
    return out


def decode_operand(p: PackedNVFP4, mode: int = MODE_P32, center: torch.Tensor | None = None, rotate: int | None = None) -> torch.Tensor:
    """The activation of a decode-sized call (rows < 256, cols % 256 == 0) as ready 16-bit MFMA operands for
    metis_linear_fwd_grouped_operand: exact binary16 values (mode P32), the reference's bf16 dequantized values (mode
    PB16), or with `center` (bf16 [cols], PB16) the mean mode's center + QDQ(x - center) rounded to bf16.
    rotate (sign mask): the call multiplies with a weight packed in the rotated domain (NV recipe); the operand then
    holds the activation's dequantized blocks rotated forward and scaled by 1/16, which gives the product with the
    weight rotated back."""
    L = load()
    out = torch.empty(L.metis_nvfp4_decode_operand_bytes(p.rows, p.cols), dtype=torch.uint8, device=p.codes.device)
    if rotate is not None:
        if center is not None or p.rht is not None:
            raise ValueError("a rotated operand is built from an unrotated, uncentred activation")
        d = p.__dict__
        lazy = d.get("deferred") is not None and d.get("_scales") is None
        rc = L.metis_nvfp4_decode_operand_rht(p.codes.data_ptr(), None if lazy else p.scales.data_ptr(),
                                              d["_unit"].data_ptr() if lazy else p.unit.data_ptr(),
                                              d["deferred"].data_ptr() if lazy else None, p.rows, p.cols, p.mode, mode, int(rotate),
                                              out.data_ptr(), _stream())
        if rc:
            check(rc, "metis_nvfp4_decode_operand_rht", (p.rows, p.cols))
        if lazy:
            d["_unit_ready"] = True
        return out
    if center is not None:
        center = center.reshape(-1).to(torch.bfloat16).contiguous()
        if center.numel() != p.cols:
            raise ValueError(f"center must have {p.cols} values, got {center.numel()}")
    d = p.__dict__
    if d.get("deferred") is not None and d.get("_scales") is None:
        # the scale bytes were never written: this kernel forms them from the parked block maxima, and writes the unit
        rc = L.metis_nvfp4_decode_operand_deferred(p.codes.data_ptr(), d["deferred"].data_ptr(), p.rows, p.cols, p.mode, mode,
                                                   None if center is None else center.data_ptr(), d["_unit"].data_ptr(),
                                                   out.data_ptr(), _stream())
        if rc:
            check(rc, "metis_nvfp4_decode_operand_deferred", (p.rows, p.cols))
        d["_unit_ready"] = True
        return out
    rc = L.metis_nvfp4_decode_operand(p.codes.data_ptr(), p.scales.data_ptr(), p.unit.data_ptr(), p.rows, p.cols, mode,
                                      None if center is None else center.data_ptr(), out.data_ptr(), _stream())
    if rc:
        check(rc, "metis_nvfp4_decode_operand", (p.rows, p.cols))
    return out


def grouped_operand_applies(a: PackedNVFP4, weights, ranks, center: torch.Tensor | None, reference_rounding: bool) -> bool:
    """Whether linear_fwd_grouped(a, members, center=center, reference_rounding=...) reads the activation as ready
    operands (decode_operand): bf16 arithmetic on every tensor, decode-sized shapes in wide runs.  weights: the
    members' packed weights, ranks: the widths of their low-rank terms (0 without)."""
    M, K = a.rows, a.cols
    if not (reference_rounding and 0 < M < 256 and a.mode == MODE_PB16 and K % 256 == 0 and len(weights) <= 4
            and (center is None or center.dtype == torch.bfloat16)):
        return False
    for b, r in zip(weights, ranks):
        if b.mode != MODE_PB16 or b.rht is not None or not _decode_kernel_takes(M, b.rows, K, r) or b.scales.data_ptr() % 8:
            return False
    return True


def project_and_operand_applies(x2: torch.Tensor, v: torch.Tensor, s: torch.Tensor, p: PackedNVFP4) -> bool:
    """project_and_operand takes these: the decode-sized domain of lowrank_project (with s), and a packed form of the
    same shape whose quantizer call deferred its scale bytes, never materialized since."""
    M, K = x2.shape
    R = v.shape[0]
    d = p.__dict__
    return bool(x2.is_cuda and x2.dtype == torch.bfloat16 and v.dtype == torch.bfloat16 and s.dtype == torch.bfloat16
                and 0 < M < 256 and K % 256 == 0 and v.shape[1] == K and R % 32 == 0 and 0 < R <= 256 and s.numel() == R
                and x2.stride(1) == 1 and x2.stride(0) % 8 == 0 and x2.data_ptr() % 16 == 0
                and p.rows == M and p.cols == K and p.rht is None
                and d.get("deferred") is not None and d.get("_scales") is None)


def project_and_operand(x2: torch.Tensor, v: torch.Tensor, s: torch.Tensor, p: PackedNVFP4, mode: int = MODE_PB16,
                        center: torch.Tensor | None = None, pending: torch.Tensor | None = None, rotate: int | None = None,
                        checked: bool = False):
    """(xv, t, operand) = lowrank_project(x2, v, s) and decode_operand(p, mode, center) of one decode-sized activation
    in two launches instead of three: the projection's finishing step rides in the operand launch.  Same bits.
    pending: the projection's partial sums as quantize_project_decode left them (the first of the two launches already
    ran beside the quantizer): one launch.  rotate (sign mask): the operand of decode_operand(p, mode, rotate=...).
    checked: the caller has just asked project_and_operand_applies."""
    if rotate is not None and center is not None:
        raise ValueError("a rotated operand takes no centre")
    if not checked and not project_and_operand_applies(x2, v, s, p):
        raise ValueError("project_and_operand: outside the call's domain (see project_and_operand_applies)")
    M, K = x2.shape
    R = v.shape[0]
    dev = x2.device
    v = v.contiguous()
    s = s.contiguous()
    if center is not None:
        center = _bf16_row(center)
        if center.numel() != K:
            raise ValueError(f"center must have {K} values, got {center.numel()}")
    need = _lowrank_workspace_bytes(M, R, K)
    if pending is not None and (pending.numel() < need or pending.device != dev):
        raise ValueError("project_and_operand: `pending` is not what quantize_project_decode or a TokenMean's call leaves for these shapes")
    specs = ((B16, M, R), (B16, M, R), (U8, _decode_operand_bytes(M, K)))
    d = p.__dict__
    new = _lib.call("metis_decode_prepare_deferred", dev.index, specs if pending is not None else specs + ((U8, need),),
                    (None if pending is not None else x2, x2.stride(0), v, R, s, "0", "1", "3" if pending is None else pending, need,
                     p.codes, d["deferred"], M, K, p.mode, mode, center, d["_unit"], "2", rotate is not None, int(rotate or 0), _stream()))
    if new.__class__ is int:
        check(new, "metis_decode_prepare_deferred", (M, K, R))
    xv, t, out = new[:3]
    d["_unit_ready"] = True
    return xv, t, out


def decode_weight(p: PackedNVFP4, cache: bool = True) -> torch.Tensor | None:
    """The packed weight in the decode layout (same 0.5625 B per element): rows in tiles of 32, K in steps of 256, the
    pieces of a wave's 64 lanes side by side, so that the decode-sized kernel's loads cover whole lines.  None when
    K % 256 != 0.  Kept on a persistent (cached) weight."""
    if p.decode_layout is not None:
        return p.decode_layout
    if p.cols % 256:
        return None
    L = load()
    out = torch.empty(L.metis_nvfp4_decode_weight_bytes(p.rows, p.cols), dtype=torch.uint8, device=p.codes.device)
    rc = L.metis_nvfp4_decode_weight(p.codes.data_ptr(), p.scales.data_ptr(), p.rows, p.cols, out.data_ptr(), _stream())
    if rc:
        check(rc, "metis_nvfp4_decode_weight", (p.rows, p.cols))
    if cache:
        p.decode_layout = out
    return out


def dense_expand_tiled(x: torch.Tensor, mode: int = MODE_P32, col_scale: torch.Tensor | None = None) -> torch.Tensor:
    """A dense [rows, cols] bf16 or float32 tensor as a tiled GEMM operand (see expand_tiled): binary16 values in mode
    P32 (pair it with a unit of 2^-8, see gemm_tiled), bf16 values in mode PB16.  col_scale (bf16 [cols]) multiplies
    column k first."""
    if x.dim() != 2 or x.dtype not in (torch.bfloat16, torch.float32) or not x.is_cuda:
        raise ValueError("dense_expand_tiled: a 2-D bf16 or float32 device tensor")
    if x.stride(1) != 1 or x.data_ptr() % 16 or x.stride(0) % (4 if x.dtype == torch.float32 else 8):
        x = x.contiguous()
    rows, cols = x.shape
    L = load()
    out = torch.empty(L.metis_nvfp4_expand_tiled_bytes(rows, cols), dtype=torch.uint8, device=x.device)
    cs = None if col_scale is None else col_scale.to(torch.bfloat16).contiguous()
    rc = L.metis_dense_expand_tiled(x.data_ptr(), rows, cols, x.stride(0), DTYPE_F32 if x.dtype == torch.float32 else DTYPE_BF16,
                                    None if cs is None else cs.data_ptr(), mode, out.data_ptr(), _stream())
    if rc:
        check(rc, "metis_dense_expand_tiled", (rows, cols))
    return out


@functools.lru_cache(maxsize=4096)
def _tiled_workspace_bytes(M: int, N: int, K: int, mode: int, device_index: int) -> int:
    return int(load().metis_linear_tiled_workspace_bytes(M, N, K, mode))


def gemm_tiled(ax: torch.Tensor, a_unit: torch.Tensor, bx: torch.Tensor, b_unit: torch.Tensor, M: int, N: int, K: int, *,
               mode: int = MODE_P32, t: torch.Tensor | None = None, u: torch.Tensor | None = None,
               bias: torch.Tensor | None = None, out_dtype: torch.dtype = torch.bfloat16, split_k: bool = True) -> torch.Tensor:
    """out[M, N] = A B^T (+ t u^T + bias) on tiled 16-bit operands ax [M, K], bx [N, K] (see expand_tiled); mode P32:
    binary16 operands, the product times a_unit * b_unit; mode PB16: bf16 operands that hold their units, the
    reference's bf16 roundings in the epilogue."""
    dev = ax.device
    r = 0
    if t is not None:
        t = t.to(torch.bfloat16).contiguous()
        u = u.to(torch.bfloat16).contiguous()
        r = t.shape[1]
        if t.shape != (M, r) or u.shape != (N, r):
            raise ValueError("low-rank operands must be t[M, r], u[N, r]")
    bias_f32 = bias is not None and bias.dtype == torch.float32
    if bias is not None:
        bias = bias.contiguous() if bias_f32 else bias.to(torch.bfloat16).contiguous()
    need = _tiled_workspace_bytes(M, N, K, mode, dev.index or 0) if split_k else 0
    f32 = out_dtype == torch.float32
    specs = ((F32 if f32 else B16, M, N), (U8, need)) if need else ((F32 if f32 else B16, M, N),)
    new = _lib.call("metis_linear_fwd_tiled", dev.index, specs,
                    (ax, a_unit, bx, b_unit, M, N, K, t, u, r, bias, bias_f32, "0", DTYPE_F32 if f32 else DTYPE_BF16, mode, "1" if need else None, need, _stream()))
    if new.__class__ is int:
        check(new, "metis_linear_fwd_tiled", (M, N, K))
    return new[0]


def linear_fwd_tiled(a: PackedNVFP4, b: PackedNVFP4, *, t: torch.Tensor | None = None, u: torch.Tensor | None = None,
                     bias: torch.Tensor | None = None, out_dtype: torch.dtype = torch.bfloat16,
                     a_tiled: torch.Tensor | None = None, reference_rounding: bool = False,
                     split_k: bool = True, center: torch.Tensor | None = None, batch: "_TiledBatch | None" = None) -> torch.Tensor | None:
    """linear_fwd on tiled 16-bit expansions: b's is cached on b when b is persistent, a's is made here unless given.
    batch: the product is queued there, for the launch that runs them all (linear_fwd_tiled_grouped); no output is returned.

    reference_rounding (both operands packed in bf16 arithmetic): operands are the reference's bf16 dequantized
    values and the epilogue rounds where the reference's all-bf16 forward rounds; otherwise exact products.
    center (bf16 [K], with reference_rounding): `a` packs the centred residual of the mean mode and the activation
    operand is the reference's bf16 tensor center + QDQ(x - center)."""
    if a.cols != b.cols:
        raise ValueError(f"contraction mismatch: {a.cols} vs {b.cols}")
    mode = MODE_P32
    if reference_rounding:
        if a.mode != MODE_PB16 or b.mode != MODE_PB16:
            raise ValueError("reference_rounding needs both operands packed in bf16 arithmetic")
        mode = MODE_PB16
    elif center is not None:
        raise ValueError("a centre inside the operand belongs to reference_rounding")
    bx = expand_tiled(b, cache=b.persistent, mode=mode)
    ax = a_tiled if a_tiled is not None else expand_tiled(a, cache=a.shared, mode=mode, center=center)
    if batch is not None:
        return batch.add(bx, b, t, u, bias)
    return gemm_tiled(ax, a.unit, bx, b.unit, a.rows, b.rows, a.cols, mode=mode, t=t, u=u, bias=bias, out_dtype=out_dtype,
                      split_k=split_k)


def tiled_group_applies(a: PackedNVFP4, weights, reference_rounding: bool) -> bool:
    """Whether linear_fwd would run every product of this activation with `weights` on the tiled kernel in one format, so
    that linear_fwd_tiled_grouped can run them in one launch: 256 rows or more, all of them in the reference's bf16
    roundings, or all of them exact (cached weights with a kept expansion, or weights in the rotated domain)."""
    if not (a.rows >= 256 and a.cols % 32 == 0 and a.rht is None and 0 < len(weights) <= 4 and all(b.cols == a.cols for b in weights)):
        return False
    rounded = [reference_rounding and a.mode == MODE_PB16 and b.mode == MODE_PB16 for b in weights]
    return all(rounded) or (not any(rounded) and all(b.rht is not None or _tiled_applies(a, b) for b in weights))


def linear_fwd_tiled_grouped(a: PackedNVFP4, members, out_dtype: torch.dtype = torch.bfloat16, center: torch.Tensor | None = None,
                             reference_rounding: bool = False) -> list[torch.Tensor]:
    """[linear_fwd_tiled(a, b, t=t, u=u, bias=bias, ...) for (b, t, u, bias) in members] in one launch, with the same bits: a
    projection group at prefill size (tiled_group_applies).  t may be a column slice of a stacked projection.  center: as
    linear_fwd_tiled."""
    if not tiled_group_applies(a, [m[0] for m in members], reference_rounding):
        raise ValueError("linear_fwd_tiled_grouped: outside the call's domain (see tiled_group_applies)")
    return _linear_fwd_tiled_grouped(a, members, out_dtype, center, reference_rounding)


def _linear_fwd_tiled_grouped(a: PackedNVFP4, members, out_dtype, center, reference_rounding) -> list[torch.Tensor]:
    mode = MODE_PB16 if (reference_rounding and a.mode == MODE_PB16 and members[0][0].mode == MODE_PB16) else MODE_P32
    if center is not None and mode != MODE_PB16:
        raise ValueError("a centre inside the operand belongs to reference_rounding")
    ax = expand_tiled(a, cache=False, mode=mode, center=center)
    batch = _TiledBatch(a, ax, out_dtype, mode)
    for b, t, u, bias in members:
        linear_fwd_tiled(a, b, t=t, u=u, bias=bias, out_dtype=out_dtype, a_tiled=ax, reference_rounding=mode == MODE_PB16, center=center, batch=batch)
    return batch.run()


class _TiledBatch:
    """Products of one tiled activation that run as one launch."""

    def __init__(self, a: PackedNVFP4, ax: torch.Tensor, out_dtype: torch.dtype, mode: int):
        self.a, self.ax, self.out_dtype, self.mode = a, ax, out_dtype, mode
        self.members: list = []                                    # as _lib.call takes them
        self.rows: list[int] = []

    def add(self, bx, b, t, u, bias) -> None:
        M = self.a.rows
        r = ldt = 0
        if t is not None:
            if t.dtype != torch.bfloat16:
                t = t.to(torch.bfloat16)
            if u.dtype != torch.bfloat16 or not u.is_contiguous():
                u = u.to(torch.bfloat16).contiguous()
            r = t.shape[1]
            if t.shape != (M, r) or u.shape != (b.rows, r):
                raise ValueError("low-rank operands must be t[M, r], u[N, r]")
            if t.stride(1) != 1 or t.stride(0) % 8 or t.data_ptr() % 16:
                t = t.contiguous()
            ldt = t.stride(0)
        bias_f32 = bias is not None and bias.dtype == torch.float32
        if bias is not None:
            bias = bias.contiguous() if bias_f32 else bias.to(torch.bfloat16).contiguous()
        self.members.append((bx, None, b.unit, t, u, r, bias, _OUT[len(self.rows)], b.rows, bias_f32, ldt, None))
        self.rows.append(b.rows)

    def run(self) -> list[torch.Tensor]:
        a, dev, count = self.a, self.ax.device, len(self.rows)
        need = _tiled_group_workspace_bytes(a.rows, a.cols, tuple(self.rows), dev.index or 0)
        f32 = self.out_dtype == torch.float32
        specs = [(F32 if f32 else B16, a.rows, n) for n in self.rows]
        if need:
            specs.append((U8, need))
        new = _lib.call("metis_linear_fwd_tiled_grouped", dev.index, tuple(specs),
                        (self.ax, a.unit, a.rows, a.cols, self.members, count, DTYPE_F32 if f32 else DTYPE_BF16, self.mode, _OUT[count] if need else None, need,
                         _stream()))
        if new.__class__ is int:
            check(new, "metis_linear_fwd_tiled_grouped", (a.rows, a.cols, self.rows))
        return list(new[:count])


@functools.lru_cache(maxsize=4096)
def _tiled_group_workspace_bytes(M: int, K: int, ns: tuple, device_index: int) -> int:
    arr = (_lib.LinearMember * len(ns))()
    for i, n in enumerate(ns):
        arr[i].N = n
    return int(load().metis_linear_tiled_grouped_workspace_bytes(M, K, ctypes.cast(arr, ctypes.c_void_p), len(ns)))


def rmsnorm_quantize(x: torch.Tensor, gamma: torch.Tensor, eps: float, mode: int = MODE_P32,
                     want_normed: bool = True, deferred: bool = False):
    """Fused RMSNorm -> NVFP4.  Returns (normed bf16 or None, PackedNVFP4).  deferred: as in quantize (one launch; scale
    bytes and unit on first access, or formed by expand_tiled)."""
    x2 = _as_2d_bf16(x)
    rows, cols = x2.shape
    if cols % BLOCK:
        raise ValueError(f"NVFP4 block shape (1, 16) does not divide tensor shape {tuple(x.shape)}")
    g = gamma.to(device=x2.device, dtype=torch.bfloat16).contiguous()
    dev = x2.device
    # the packed tensor's parts, then the normed tensor if it is wanted
    normed = "4" if want_normed else None
    extra = ((B16, rows, cols),) if want_normed else ()
    codes, unit = (U8, rows, cols // 2), (F32, 1)
    if deferred and rows * cols > 0:
        size = _deferred_bytes(rows, cols)
        name = "metis_rmsnorm_nvfp4_quant_deferred"
        new = _lib.call(name, dev.index, (codes, unit, (U8, size), *extra), (x2, g, float(eps), rows, cols, mode, "3" if want_normed else None, "0", "2", size, _stream()))
        if new.__class__ is int:
            check(new, name, x.shape)
        return new[3].reshape(x.shape) if want_normed else None, PackedNVFP4(new[0], None, new[1], rows, cols, mode, deferred=new[2])
    ws = _workspace(rows, cols, dev)
    decode = decode_layout_activations and 0 < rows < 256 and cols % 256 == 0
    specs = (codes, (U8, rows, cols // BLOCK), unit, (U8, _decode_weight_bytes(rows, cols) if decode else 0), *extra)
    if decode:
        name = "metis_rmsnorm_nvfp4_quant_decode"
        new = _lib.call(name, dev.index, specs, (x2, g, float(eps), rows, cols, mode, normed, "0", "1", "2", "3", ws, ws.numel(), _stream()))
    else:
        name = "metis_rmsnorm_nvfp4_quant"
        new = _lib.call(name, dev.index, specs, (x2, g, float(eps), rows, cols, mode, normed, "0", "1", "2", ws, ws.numel(), _stream()))
    if new.__class__ is int:
        check(new, name, x.shape)
    return (new[4].reshape(x.shape) if want_normed else None,
            PackedNVFP4(new[0], new[1], new[2], rows, cols, mode, decode_layout=new[3] if decode else None))


def rmsnorm(x: torch.Tensor, gamma: torch.Tensor, eps: float) -> torch.Tensor:
    """The normed bf16 [R, C] of rmsnorm_colmean alone.  C <= 4096."""
    x2 = _as_2d_bf16(x)
    rows, cols = x2.shape
    g = gamma.to(device=x2.device, dtype=torch.bfloat16).contiguous()
    new = _lib.call("metis_rmsnorm", x2.device.index, ((B16, rows, cols),), (x2, g, float(eps), rows, cols, "0", _stream()))
    if new.__class__ is int:
        check(new, "metis_rmsnorm", x.shape)
    return new[0]


def rmsnorm_colmean(x: torch.Tensor, gamma: torch.Tensor, eps: float, mean_dtype: torch.dtype = torch.float32,
                    cached: torch.Tensor | None = None, cached_count: int = 0):
    """RMSNorm for the mean mode: (normed bf16 [R, C], column mean of normed over its rows in mean_dtype, the same as
    float32) from one pass over x plus one small kernel.  cached / cached_count: the weighted running mean of
    single-token decode calls, as column_mean_running.  C <= 4096."""
    x2 = _as_2d_bf16(x)
    rows, cols = x2.shape
    if cols % BLOCK:
        raise ValueError(f"NVFP4 block shape (1, 16) does not divide tensor shape {tuple(x.shape)}")
    if mean_dtype not in (torch.bfloat16, torch.float32):
        raise ValueError("rmsnorm_colmean: the mean is bfloat16 or float32")
    dev = x2.device
    g = gamma.to(device=dev, dtype=torch.bfloat16).contiguous()
    f32 = mean_dtype == torch.float32
    size = _rmsnorm_colmean_bytes(rows, cols, dev.index or 0)
    if cached is not None:
        cached = cached.reshape(-1).to(device=dev, dtype=mean_dtype).contiguous()
        if cached.numel() != cols:
            raise ValueError(f"cached mean must have one value per column ({cols}), got {cached.numel()}")
    specs = ((B16, rows, cols), (U8, size), (F32 if f32 else B16, cols))
    new = _lib.call("metis_rmsnorm_colmean", dev.index, specs if f32 else specs + ((F32, cols),),
                    (x2, g, float(eps), rows, cols, "0", "2", DTYPE_F32 if f32 else DTYPE_BF16, cached, int(cached_count), None if f32 else "3", "1", size, _stream()))
    if new.__class__ is int:
        check(new, "metis_rmsnorm_colmean", x.shape)
    return new[0], new[2], new[2] if f32 else new[3]


def rmsnorm_backward_applies(x: torch.Tensor, g: torch.Tensor, gamma: torch.Tensor) -> bool:
    """rmsnorm_backward takes these: bf16 device tensors of the same non-empty shape, a wave per row."""
    cols = x.shape[-1]
    return bool(x.is_cuda and x.dtype == torch.bfloat16 and g.dtype == torch.bfloat16 and gamma.dtype == torch.bfloat16
                and g.device == x.device and gamma.device == x.device and g.shape == x.shape and cols % BLOCK == 0
                and 0 < cols <= 4096 and x.numel() > 0)


def rmsnorm_backward(x: torch.Tensor, g: torch.Tensor, gamma: torch.Tensor, eps: float, want_gamma: bool = True):
    """(gradient of x, gradient of gamma or None) of y = bf16(bf16(x rstd) gamma) for the gradient g of y, all bf16: one
    pass over x and g, binary32 arithmetic, column sums in a fixed order rounded once."""
    def dense(t, cols):
        t = t.reshape(-1, cols)
        t = t if t.is_contiguous() else t.contiguous()
        return t if t.data_ptr() % 16 == 0 else t.clone()
    cols = x.shape[-1]
    x2, g2 = dense(x, cols), dense(g, cols)
    gm = dense(gamma, cols)
    rows = x2.shape[0]
    need = _rmsnorm_backward_bytes(rows, cols, x.device.index or 0) if want_gamma else 0
    specs = ((B16, rows, cols), (B16, cols), (U8, need)) if want_gamma else ((B16, rows, cols),)
    new = _lib.call("metis_rmsnorm_backward", x.device.index, specs,
                    (x2, g2, gm, float(eps), rows, cols, "0", "1" if want_gamma else None, DTYPE_BF16, "2" if want_gamma else None, need, _stream()))
    if new.__class__ is int:
        check(new, "metis_rmsnorm_backward", x.shape)
    return new[0].reshape(x.shape), new[1] if want_gamma else None


@functools.lru_cache(maxsize=16)
def _device_cus(device_index: int) -> int:
    return int(torch.cuda.get_device_properties(device_index).multi_processor_count)


def _tiled_applies(a: PackedNVFP4, b: PackedNVFP4) -> bool:
    """The pipelined GEMM on tiled binary16 expansions pays when the weight-side expansion is reused across calls
    (a cached weight) and the batch fills a 256-row tile; the activation side is expanded per call (2.56 B/element,
    about 2 % of the GEMM's time at such shapes)."""
    if not ((b.persistent and tiled_weight_copies) or b.tiled is not None):
        return False
    M, N, K = a.rows, b.rows, a.cols
    return M >= 256 and N >= 256 and K % 32 == 0 and K >= 128


@functools.lru_cache(maxsize=4096)
def _linear_workspace_bytes(M: int, N: int, K: int, device_index: int) -> int:
    return int(load().metis_linear_workspace_bytes(M, N, K))          # depends on the device's CU count only


@functools.lru_cache(maxsize=4096)
def _lowrank_workspace_bytes(M: int, R: int, K: int) -> int:
    return int(load().metis_lowrank_project_workspace_bytes(M, R, K))


@functools.lru_cache(maxsize=4096)
def _grouped_plan(M: int, K: int, ns: tuple, device_index: int) -> tuple[int, bool]:
    """(split-K scratch bytes, whether a centre can ride inside the launch) of a grouped call; shape-only queries."""
    arr = (_lib.LinearMember * len(ns))()
    for i, n in enumerate(ns):
        arr[i].N = n
    ap = ctypes.cast(arr, ctypes.c_void_p)
    L = load()
    need = int(L.metis_linear_grouped_workspace_bytes(M, K, ap, len(ns)))
    return need, bool(L.metis_linear_grouped_centered_supported(M, K, ap, len(ns), int(need > 0)))


@functools.lru_cache(maxsize=4096)
def _grouped_centre_fits_unsplit(M: int, K: int, ns: tuple, device_index: int) -> bool:
    arr = (_lib.LinearMember * len(ns))()
    for i, n in enumerate(ns):
        arr[i].N = n
    return bool(load().metis_linear_grouped_centered_supported(M, K, ctypes.cast(arr, ctypes.c_void_p), len(ns), 0))


def _gemm_workspace(M: int, N: int, K: int, device: torch.device) -> torch.Tensor | None:
    """Split-K scratch for an M x N output contracted over K, or None when the shape is not split.

    Taken from torch's caching allocator per call (stream-ordered, so overlapping streams and captured
    graphs each get their own) rather than cached here."""
    if M >= 256 and N < 256:
        return None
    need = _linear_workspace_bytes(M, N, K, device.index or 0)
    return torch.empty(need, dtype=torch.uint8, device=device) if need else None


def nv_decode_applies(a: PackedNVFP4, weights, ranks) -> bool:
    """A decode-sized call against weights packed in the rotated domain (NV recipe) runs on the decode-sized kernel,
    the rotation carried by the activation's operand: one rotation for all members, an unrotated activation, the
    kernel's shapes in wide runs."""
    masks = {b.rht for b in weights}
    return bool(len(masks) == 1 and None not in masks and a.rht is None and len(weights) <= 4 and a.cols % 256 == 0
                and all(_decode_kernel_takes(a.rows, b.rows, a.cols, r) for b, r in zip(weights, ranks))
                and all(b.scales.data_ptr() % 8 == 0 for b in weights))


def nv_operand_mode(a: PackedNVFP4, weights, reference_rounding: bool) -> int:
    """The format of the rotated operand of a decode-sized NV-recipe call: the reference's bf16 values when the call
    follows its all-bf16 evaluation (every tensor packed in bf16 arithmetic), exact binary16 otherwise."""
    return MODE_PB16 if (reference_rounding and a.mode == MODE_PB16 and all(b.mode == MODE_PB16 for b in weights)) else MODE_P32


def _decode_kernel_takes(M: int, N: int, K: int, r: int) -> bool:
    """Shapes of the decode-sized kernel (waves split K over packed operands streamed from global memory)."""
    return 0 < M < 256 and K % 64 == 0 and N % 4 == 0 and r % 32 == 0


def linear_fwd(a: PackedNVFP4, b: PackedNVFP4, *, t: torch.Tensor | None = None, u: torch.Tensor | None = None,
               bias: torch.Tensor | None = None, out_dtype: torch.dtype = torch.bfloat16,
               expanded: bool | None = None, split_k: bool = True, tiled: bool | None = None,
               reference_rounding: bool = False, a_operand: torch.Tensor | None = None) -> torch.Tensor:
    """out[M, N] = deq(a)[M, K] . deq(b)[N, K]^T (+ t[M, r] . u[N, r]^T) (+ bias[N]).

    tiled=None picks the pipelined kernel on tiled binary16 expansions when b is a cached weight and the shape is
    large (see _tiled_applies), or when the product is large enough to pay for expansions made for this one call
    (_tiled_backward_pays); True / False force the choice.  Same products either way; a plain unsplit product has the
    same bits, a low-rank term joins the binary32 sum at another point (1e-6 relative in binary32).
    reference_rounding: the forward of a layer whose arithmetic is bf16 (both operands packed in that mode): follow the
    reference's all-bf16 evaluation (twice-rounded bf16 operands, residual product and bias add rounded to bf16): the
    pipelined kernel from 256 rows on, the decode-sized kernel below (shapes it does not take get exact products).

    split_k=False withholds the split-K workspace: the contraction then runs unsplit in one launch.

    expanded=True runs on cached exact f16 expansions of a and b (2 B/element extra HBM, inner loop of
    MFMA + LDS reads only); the default works on the packed operands directly.
    a_operand: as in linear_fwd_grouped (a decode-sized call in bf16 arithmetic)."""
    if a.cols != b.cols:
        raise ValueError(f"contraction mismatch: {a.cols} vs {b.cols}")
    if (tiled is None and not expanded and b.rht is not None
            and nv_decode_applies(a, [b], [0 if t is None else t.shape[1]])):
        # NV recipe at decode size: the packed rotated weight is streamed as it is, the activation's operand is rotated
        return _linear_fwd_grouped(a, [(b, t, u, bias)], out_dtype=out_dtype, split_k=split_k,
                                   reference_rounding=reference_rounding, a_operand=a_operand)[0]
    if a.rht is not None or b.rht is not None:
        # NV recipe: only the tiled operands know how to rotate a block back
        if a.cols % 32:
            raise ValueError("a rotated operand needs a contraction that is a multiple of 32")
        tiled = True
    rounded = reference_rounding and a.mode == MODE_PB16 and b.mode == MODE_PB16
    faithful = rounded and (a.rows >= 256 or tiled) and a.cols % 32 == 0
    if tiled is None:
        tiled = faithful or (not expanded and (_tiled_applies(a, b) or _tiled_backward_pays(a.rows, b.rows, a.cols, a.codes.device.index or 0)))
    if tiled:
        return linear_fwd_tiled(a, b, t=t, u=u, bias=bias, out_dtype=out_dtype, reference_rounding=faithful, split_k=split_k)
    M, N, K = a.rows, b.rows, a.cols
    if rounded and not expanded and _decode_kernel_takes(M, N, K, 0 if t is None else t.shape[1]):
        return _linear_fwd_grouped(a, [(b, t, u, bias)], out_dtype=out_dtype, split_k=split_k, reference_rounding=True,
                                   a_operand=a_operand)[0]
    dev = a.codes.device
    r = 0
    if t is not None:
        t = t.to(torch.bfloat16).contiguous()
        u = u.to(torch.bfloat16).contiguous()
        r = t.shape[1]
        if t.shape != (M, r) or u.shape != (N, r):
            raise ValueError("low-rank operands must be t[M, r], u[N, r]")
    bias_f32 = bias is not None and bias.dtype == torch.float32     # e.g. bias + W^ me of the mean mode
    if bias is not None:
        bias = bias.contiguous() if bias_f32 else bias.to(torch.bfloat16).contiguous()
    out = torch.empty(M, N, dtype=out_dtype, device=dev)
    dt = DTYPE_F32 if out_dtype == torch.float32 else DTYPE_BF16
    tp = None if t is None else t.data_ptr()
    up = None if u is None else u.data_ptr()
    bp = None if bias is None else bias.data_ptr()
    if expanded is None:
        # measured on MI355X: the packed kernel (expansion inside the K loop, 16 KiB/step of operand traffic)
        # is within 5 % of the expanded one at 8192x4096x14336 and faster on smaller shapes, so it is the default
        expanded = False
    if expanded and bias_f32:
        raise ValueError("the expanded-operand path takes a bf16 bias")
    if expanded:
        ae, be = expand(a), expand(b)
        rc = load().metis_linear_fwd_expanded(ae.data_ptr(), a.unit.data_ptr(), be.data_ptr(), b.unit.data_ptr(), M, N, K,
                                              tp, up, r, bp, out.data_ptr(), dt, _stream())
        if rc:
            check(rc, "metis_linear_fwd_expanded", (M, N, K))
        return out
    ws = _gemm_workspace(M, N, K, dev) if split_k else None
    if bias_f32:
        rc = load().metis_linear_fwd_f32bias(a.codes.data_ptr(), a.scales.data_ptr(), a.unit.data_ptr(), b.codes.data_ptr(),
                                             b.scales.data_ptr(), b.unit.data_ptr(), M, N, K, tp, up, r, bp, out.data_ptr(), dt,
                                             None if ws is None else ws.data_ptr(), 0 if ws is None else ws.numel(), _stream())
        if rc:
            check(rc, "metis_linear_fwd_f32bias", (M, N, K))
        return out
    if ws is not None:
        rc = load().metis_linear_fwd_ws(a.codes.data_ptr(), a.scales.data_ptr(), a.unit.data_ptr(), b.codes.data_ptr(),
                                        b.scales.data_ptr(), b.unit.data_ptr(), M, N, K, tp, up, r, bp, out.data_ptr(), dt,
                                        ws.data_ptr(), ws.numel(), _stream())
        if rc:
            check(rc, "metis_linear_fwd_ws", (M, N, K))
        return out
    rc = load().metis_linear_fwd(a.codes.data_ptr(), a.scales.data_ptr(), a.unit.data_ptr(), b.codes.data_ptr(),
                                 b.scales.data_ptr(), b.unit.data_ptr(), M, N, K, tp, up, r, bp, out.data_ptr(), dt, _stream())
    if rc:
        check(rc, "metis_linear_fwd", (M, N, K))
    return out


ONE_PASS_RANKS = (32, 64, 96, 128, 192, 256)      # of lowrank_project from 256 rows on: the kernel holds a row's R sums in registers


class FactorStack:
    """V (or s) of up to four members of a projection group on top of each other, each where it is: what lowrank_project takes
    for one pass over their common x (lowrank_stack_applies).  Nothing is copied, so nothing is outdated by a write to a member."""

    def __init__(self, parts):
        self.parts = parts
        self.shape = (sum([p.shape[0] for p in parts]), *parts[0].shape[1:])


def _lowrank_operands(x2: torch.Tensor, v: torch.Tensor, s: torch.Tensor | None) -> bool:
    """The operands have a form that the library's projection kernels read (shapes aside)."""
    M, K = x2.shape
    return (x2.is_cuda and x2.dtype == torch.bfloat16 and v.dtype == torch.bfloat16 and M > 0 and K % 64 == 0 and v.shape[1] == K
            and x2.stride(1) == 1 and x2.stride(0) % 8 == 0 and x2.data_ptr() % 16 == 0 and (s is None or s.dtype == torch.bfloat16))


def _one_pass_takes(x2: torch.Tensor, v: torch.Tensor, s: torch.Tensor | None) -> bool:
    """A projection of 256 rows or more runs on the one-pass kernel: ranks 32, 64 and 128 always; 96, 192 and 256, which have few
    stages of the wide tile in flight and fetch all of V again for every row tile, up to a bound on the work.  Microseconds,
    kernel | library product and its multiplication by s:
        R = 96   4096 x 8960 22 | 35, 8000 x 3584 24 | 21, 16384 x 3584 30 | 28, 16384 x 8960 96 | 67, 16384 x 18944 200 | 144
        R = 192  800 x 18944 35 | 72, 4096 x 3584 23 | 27, 8000 x 1536 22 | 24, 8000 x 3584 39 | 31, 16384 x 18944 359 | 215
        R = 256  800 x 18944 38 | 87, 2103 x 3584 21 | 25, 4096 x 3584 28 | 24, 8000 x 3584 47 | 37, 16384 x 18944 469 | 252
    The library product also takes what the kernel does not read there (rows that overlap, an unaligned V) and what autograd records."""
    R = v.shape[0]
    if R in (32, 64, 128):
        return True
    if R not in ONE_PASS_RANKS:
        return False
    M, K = x2.shape
    return ((M <= 1024 or M * K * R <= (5 * 10 ** 9 if R == 96 else 3 * 10 ** 9)) and x2.stride(0) >= K and (v.data_ptr() % 16 == 0 or not v.is_contiguous())
            and not (torch.is_grad_enabled() and (x2.requires_grad or v.requires_grad or (s is not None and s.requires_grad))))


def lowrank_stack_applies(x2: torch.Tensor, factors) -> bool:
    """lowrank_project takes the (v, s) pairs of a projection group as FactorStacks: 256 rows or more, every member's own projection
    and the sum of the ranks on the one-pass kernel.  Column for column the bits of the members' own projections."""
    M, K = x2.shape
    if M < 256 or len(factors) > 4:
        return False
    total = 0
    for v, s in factors:
        if v.shape[1] != K or v.dtype != torch.bfloat16 or s.dtype != torch.bfloat16 or not _one_pass_takes(x2, v, s):
            return False
        total += v.shape[0]
    return total in ONE_PASS_RANKS and _lowrank_operands(x2, *factors[0])


def _lowrank_project_stack(x2: torch.Tensor, v: FactorStack, s: FactorStack):
    (M, K), R = x2.shape, v.shape[0]
    factors = [(a if a.is_contiguous() else a.contiguous(), b if b.is_contiguous() else b.contiguous(), a.shape[0]) for a, b in zip(v.parts, s.parts)]
    need = _lowrank_rows_workspace_bytes(M, R, K, x2.device.index or 0)
    specs = ((B16, M, R), (B16, M, R))
    new = _lib.call("metis_lowrank_project_rows_grouped", x2.device.index, specs + ((U8, need),) if need else specs,
                    (x2, x2.stride(0), M, K, factors, len(factors), "0", "1", "2" if need else None, need, _stream()))
    if new.__class__ is int:
        check(new, "metis_lowrank_project_rows_grouped", (M, [f[2] for f in factors], K))
    return new[0], new[1]


def lowrank_project(x2: torch.Tensor, v: "torch.Tensor | FactorStack", s: "torch.Tensor | FactorStack | None" = None):
    """Rank-r projection of the low-rank branch: xv = x2[M, K] . v[R, K]^T in bf16 (binary32 accumulation) and, with
    `s` [R], t = bf16(xv * s): returns xv or (xv, t).  Decode-sized batches (M < 256, R <= 256) run on the library's
    split-K kernel, larger ones on its one-pass kernel (_one_pass_takes); other shapes are a torch matmul.  FactorStacks (lowrank_stack_applies): the members' columns side by side."""
    if isinstance(v, FactorStack):
        return _lowrank_project_stack(x2, v, s)
    M, K = x2.shape
    R = v.shape[0]
    common = _lowrank_operands(x2, v, s)
    small = common and M < 256 and R % 32 == 0 and 0 < R <= 256
    large = common and M >= 256 and _one_pass_takes(x2, v, s)
    if not (small or large):
        xv = torch.matmul(x2, v.T)
        return xv if s is None else (xv, xv * s.to(xv.dtype))
    v = v.contiguous()
    specs = ((B16, M, R),)
    tp = None
    if s is not None:
        s, specs, tp = s.contiguous(), ((B16, M, R), (B16, M, R)), "1"
    if large:
        name, need = "metis_lowrank_project_rows_ws", _lowrank_rows_workspace_bytes(M, R, K, x2.device.index or 0)
    else:
        name, need = "metis_lowrank_project", _lowrank_workspace_bytes(M, R, K)
    scratch = _OUT[len(specs)] if need else None
    new = _lib.call(name, x2.device.index, specs + ((U8, need),) if need else specs,
                    (x2, x2.stride(0), v, M, R, K, s, "0", tp, scratch, need, _stream()))
    if new.__class__ is int:
        check(new, name, (M, R, K))
    return new[0] if s is None else (new[0], new[1])


def quantize_project_applies(x2: torch.Tensor, v: torch.Tensor, mode: int) -> bool:
    """quantize_project takes this activation: a contiguous bf16 [M, K] from 256 to 65536 rows, K a multiple of 64, a bf16
    V of 32 or 64 rows."""
    M, K = x2.shape
    return (x2.is_cuda and x2.dtype == torch.bfloat16 and v.dtype == torch.bfloat16 and 256 <= M <= 65536 and K % 64 == 0
            and v.shape[0] in (32, 64) and v.shape[1] == K and x2.is_contiguous() and x2.data_ptr() % 16 == 0
            and mode in (MODE_P32, MODE_PB16))


def quantize_project(x2: torch.Tensor, v: torch.Tensor, s: torch.Tensor, mode: int = MODE_P32):
    """(quantize(x2, mode, deferred=True), xv, t) from ONE pass over the activation: the packed tensor that feeds the
    residual branch and the rank-r projection xv = x2 . v^T, t = bf16(xv * s) of the low-rank branch (lowrank_project).
    The packed tensor has the bytes of quantize(); xv is the K-sliced sum of lowrank_project."""
    if not quantize_project_applies(x2, v, mode):
        raise ValueError("quantize_project: shape or dtype outside the kernel's domain (see quantize_project_applies)")
    M, K = x2.shape
    R = v.shape[0]
    dev = x2.device
    v = v.contiguous()
    s = s.to(torch.bfloat16).contiguous()
    size, need = _deferred_bytes(M, K), _lowrank_rows_workspace_bytes(M, R, K, dev.index or 0)
    specs = ((B16, M, R), (B16, M, R), (U8, M, K // 2), (F32, 1), (U8, size))
    new = _lib.call("metis_nvfp4_quant_project_deferred", dev.index, specs + ((U8, need),) if need else specs,
                    (x2, M, K, mode, v, R, s, "0", "1", "2", "4", size, "5" if need else None, need, _stream()))
    if new.__class__ is int:
        check(new, "metis_nvfp4_quant_project_deferred", (M, K, R))
    return PackedNVFP4(new[2], None, new[3], M, K, mode, deferred=new[4]), new[0], new[1]


def quantize_project_decode_applies(x2: torch.Tensor, v: torch.Tensor, mode: int) -> bool:
    """quantize_project_decode takes this activation: a contiguous bf16 [M, K] of fewer than 256 rows, K a multiple of
    256 (what the consumer of the pending sums, project_and_operand, needs), a bf16 V of 32 to 128 rows."""
    M, K = x2.shape
    return bool(x2.is_cuda and x2.dtype == torch.bfloat16 and v.dtype == torch.bfloat16 and 0 < M < 256 and K % 256 == 0
                and v.shape[0] % 32 == 0 and 0 < v.shape[0] <= 128 and v.shape[1] == K and x2.is_contiguous()
                and x2.data_ptr() % 16 == 0 and mode in (MODE_P32, MODE_PB16))


def quantize_project_decode(x2: torch.Tensor, v: torch.Tensor, mode: int = MODE_PB16):
    """(quantize(x2, mode, deferred=True), pending) from ONE launch over a decode-sized activation: the packed tensor and
    the partial sums of its rank-r projection x2 . v^T, which project_and_operand(..., pending=pending) finishes in the
    launch that also builds the GEMM operands.  Same bits as the separate calls."""
    if not quantize_project_decode_applies(x2, v, mode):
        raise ValueError("quantize_project_decode: outside the call's domain (see quantize_project_decode_applies)")
    M, K = x2.shape
    R = v.shape[0]
    dev = x2.device
    v = v.contiguous()
    size, need = _deferred_bytes(M, K), _lowrank_workspace_bytes(M, R, K)
    new = _lib.call("metis_decode_quant_project_deferred", dev.index, ((U8, M, K // 2), (F32, 1), (U8, size), (U8, need)),
                    (x2, M, K, mode, "0", "2", size, v, R, "3", need, _stream()))
    if new.__class__ is int:
        check(new, "metis_decode_quant_project_deferred", (M, K, R))
    return PackedNVFP4(new[0], None, new[1], M, K, mode, deferred=new[2]), new[3]


def lowrank_contract_tokens(a: torch.Tensor, b: torch.Tensor, out_dtype: torch.dtype = torch.bfloat16,
                            transpose: bool = False) -> torch.Tensor:
    """sum_l a[l, C] b[l, R] -> [C, R] (or [R, C] with transpose): the rank-r products of the backward pass that
    contract over tokens, bf16 operands, binary32 accumulation.  R in 32 / 64 / 128 on the library's kernel; other
    shapes are a torch matmul."""
    Lt, C = a.shape
    R = b.shape[1]
    ok = (a.is_cuda and a.dtype == torch.bfloat16 and b.dtype == torch.bfloat16 and b.shape[0] == Lt and Lt > 0 and R in (32, 64, 128)
          and C % 8 == 0 and a.stride(1) == 1 and a.stride(0) % 8 == 0 and a.data_ptr() % 16 == 0
          and out_dtype in (torch.bfloat16, torch.float32))
    if not ok:
        out = torch.matmul(a.T, b).to(out_dtype)
        return out.T.contiguous() if transpose else out
    b = b.contiguous()
    L = load()
    out = torch.empty((R, C) if transpose else (C, R), dtype=out_dtype, device=a.device)
    need = int(L.metis_lowrank_tokens_workspace_bytes(Lt, C, R))
    ws = torch.empty(need, dtype=torch.uint8, device=a.device)
    rc = L.metis_lowrank_contract_tokens(a.data_ptr(), a.stride(0), b.data_ptr(), Lt, C, R, out.data_ptr(),
                                         DTYPE_F32 if out_dtype == torch.float32 else DTYPE_BF16, int(transpose),
                                         ws.data_ptr(), need, _stream())
    if rc:
        check(rc, "metis_lowrank_contract_tokens", (Lt, C, R))
    return out


def lowrank_scale_grad(g: torch.Tensor, xv: torch.Tensor, out_dtype: torch.dtype = torch.float32) -> torch.Tensor:
    """sum_l bf16(g[l, :] * xv[l, :]) -> [R]: the gradient of s in y = s * (x V^T), as (g * xv).sum(0, dtype=float32) on bf16
    tensors computes it (the product rounded to bf16), in one launch and a fixed summation order; out_dtype bfloat16
    rounds the binary32 sum once, as .to(bfloat16) would."""
    R = g.shape[-1]
    if not (g.is_cuda and g.dtype == torch.bfloat16 and xv.dtype == torch.bfloat16 and g.shape == xv.shape and g.dim() == 2
            and R % 8 == 0 and g.is_contiguous() and xv.is_contiguous() and g.data_ptr() % 16 == 0 and xv.data_ptr() % 16 == 0
            and out_dtype in (torch.float32, torch.bfloat16)):
        return (g * xv).sum(dim=0, dtype=torch.float32).to(out_dtype)
    out = torch.empty(R, dtype=out_dtype, device=g.device)
    rc = load().metis_lowrank_scale_grad(g.data_ptr(), xv.data_ptr(), g.shape[0], R, out.data_ptr(),
                                         DTYPE_F32 if out_dtype == torch.float32 else DTYPE_BF16, _stream())
    if rc:
        check(rc, "metis_lowrank_scale_grad", tuple(g.shape))
    return out


def lowrank_backward(dy: torch.Tensor, t: torch.Tensor, x: torch.Tensor, gxv: torch.Tensor, gt: torch.Tensor, xv: torch.Tensor,
                     scale_dtype: torch.dtype = torch.float32):
    """(lowrank_contract_tokens(dy, t), lowrank_contract_tokens(x, gxv, transpose=True), lowrank_scale_grad(gt, xv, scale_dtype)): the
    gradients of a layer's U, V and s, none of which needs another, side by side in two launches instead of five.  Same bits."""
    L_, N = dy.shape
    K, R = x.shape[1], t.shape[1]
    skinny = (t, gxv, gt, xv)
    ok = (dy.is_cuda and dy.dtype == torch.bfloat16 and x.dtype == torch.bfloat16 and x.shape[0] == L_ and L_ > 0 and R in (32, 64, 128)
          and all(m.dtype == torch.bfloat16 and m.shape == (L_, R) and m.is_contiguous() and m.data_ptr() % 16 == 0 for m in skinny)
          and all(m.shape[1] % 8 == 0 and m.stride(1) == 1 and m.stride(0) % 8 == 0 and m.data_ptr() % 16 == 0 for m in (dy, x))
          and scale_dtype in (torch.float32, torch.bfloat16))
    if not ok:
        return (lowrank_contract_tokens(dy, t), lowrank_contract_tokens(x, gxv, transpose=True), lowrank_scale_grad(gt, xv, out_dtype=scale_dtype))
    need = _lowrank_backward_bytes(L_, N, K, R, dy.device.index or 0)
    f32 = scale_dtype == torch.float32
    new = _lib.call("metis_lowrank_backward", dy.device.index, ((B16, N, R), (B16, R, K), (F32 if f32 else B16, R), (U8, need)),
                    (dy, dy.stride(0), t, N, x, x.stride(0), gxv, K, L_, R, "0", DTYPE_BF16, "1", DTYPE_BF16, gt, xv, "2",
                     DTYPE_F32 if f32 else DTYPE_BF16, "3", need, _stream()))
    if new.__class__ is int:
        check(new, "metis_lowrank_backward", (L_, N, K, R))
    return new[0], new[1], new[2]


def linear_fwd_grouped(a: PackedNVFP4, members, out_dtype: torch.dtype = torch.bfloat16,
                       center: torch.Tensor | None = None, split_k: bool = True,
                       reference_rounding: bool = False, a_operand: torch.Tensor | None = None, checked: bool = False) -> list[torch.Tensor]:
    return _linear_fwd_grouped(a, members, out_dtype, center, split_k, reference_rounding, a_operand, checked)


def _grouped_members(members, M: int, K: int, out_dtype: torch.dtype, decode_layout: bool):
    """(members, specs of their outputs) of a grouped call as _lib.call takes them.  decode_layout: cached weights are streamed in that
    layout (whole lines per load instruction) by the decode-sized kernel."""
    words, specs = [], []
    kind = F32 if out_dtype == torch.float32 else B16
    for i, (b, t, u, bias) in enumerate(members):
        if b.cols != K:
            raise ValueError(f"contraction mismatch: {K} vs {b.cols}")
        r = ldt = 0
        if t is not None:
            if t.dtype != torch.bfloat16:
                t = t.to(torch.bfloat16)
            if u.dtype != torch.bfloat16 or not u.is_contiguous():
                u = u.to(torch.bfloat16).contiguous()
            r = t.shape[1]
            if t.shape != (M, r) or u.shape != (b.rows, r):
                raise ValueError("low-rank operands must be t[M, r], u[N, r]")
            # a column slice of a stacked projection is taken as it is by the single-launch path
            if not t.is_contiguous():
                if M < 256 and K % 64 == 0 and t.stride(1) == 1 and t.stride(0) % 8 == 0 and t.data_ptr() % 16 == 0:
                    ldt = t.stride(0)
                else:
                    t = t.contiguous()
        bias_f32 = bias is not None and bias.dtype == torch.float32
        if bias is not None:
            bias = bias.contiguous() if bias_f32 else bias.to(torch.bfloat16).contiguous()
        words.append((b.codes, b.scales, b.unit, t, u, r, bias, _OUT[i], b.rows, bias_f32, ldt,
                      decode_weight(b) if (decode_layout and b.persistent) else None))
        specs.append((kind, M, b.rows))
    return words, specs


_OUT = tuple([chr(ord("0") + i) for i in range(32)])              # the new tensors of a call, by position


def _linear_fwd_grouped(a: PackedNVFP4, members, out_dtype: torch.dtype = torch.bfloat16,
                        center: torch.Tensor | None = None, split_k: bool = True,
                        reference_rounding: bool = False, a_operand: torch.Tensor | None = None, checked: bool = False) -> list[torch.Tensor]:
    """[linear_fwd(a, b, t=t, u=u, bias=bias) for (b, t, u, bias) in members] in one call: a projection group
    (q/k/v, gate/up) that shares one packed activation.  Decode-sized batches run as a single launch.

    reference_rounding (every operand packed in bf16 arithmetic): the reference's all-bf16 evaluation, as in
    linear_fwd; shapes the decode-sized kernel does not take are served member by member.  A bf16 `center` then goes
    into the activation operand itself (the reference's bf16 tensor center + QDQ(x - center)); a float32 centre keeps
    exact products with the centre's share accumulated in binary32.

    center (mean mode: `a` packs the centred residual X - center): every output row also receives deq(b) . center,
    inside the same launch where the shape allows, else through matvec and a binary32 bias.

    a_operand: decode_operand(a, MODE_PB16, center) when the caller has it already (project_and_operand); read only
    where grouped_operand_applies says the call reads ready operands (checked: the caller has just asked it)."""
    M, K = a.rows, a.cols
    dev = a.codes.device
    if len(members) >= len(_OUT):                              # (beyond four members every one is a launch of its own)
        rest = (out_dtype, center, split_k, reference_rounding, a_operand)
        return _linear_fwd_grouped(a, members[:16], *rest) + _linear_fwd_grouped(a, members[16:], *rest)
    if a_operand is not None and split_k and (checked or grouped_operand_applies(a, [m[0] for m in members], [0 if m[1] is None else m[1].shape[1] for m in members],
                                                                     center, reference_rounding)):
        # the usual decode step: every question below has its answer
        words, specs = _grouped_members(members, M, K, out_dtype, decode_layout_weights)
        need, _ = _grouped_plan(M, K, tuple([m[0].rows for m in members]), dev.index or 0)
        return _grouped_call("metis_linear_fwd_grouped_operand", dev, words, specs, need,
                             (a_operand, a.__dict__["_unit"], M, K, words, len(members), DTYPE_F32 if out_dtype == torch.float32 else DTYPE_BF16, MODE_PB16))
    rounded = (reference_rounding and (center is None or center.dtype == torch.bfloat16) and a.mode == MODE_PB16
               and all(m[0].mode == MODE_PB16 for m in members))
    takes = len(members) <= 4 and all(_decode_kernel_takes(M, m[0].rows, K, 0 if m[1] is None else m[1].shape[1]) for m in members)
    # NV recipe: weights packed in the rotated domain.  The decode-sized kernel streams them as they are and the
    # activation's operand carries the rotation (decode_operand(rotate=...)); callers check nv_decode_applies first
    rotate = None
    masks = {m[0].rht for m in members}
    if masks != {None}:
        if len(masks) != 1 or a.rht is not None or center is not None or not takes or K % 256 \
                or any(m[0].scales.data_ptr() % 8 for m in members):
            raise ValueError("rotated weights: one rotation for all members of a decode-sized call on an unrotated, uncentred "
                             "activation (see nv_decode_applies); other calls take the tiled GEMM")
        rotate = masks.pop()
    # ready operands (built once for the group): wide runs only
    operand = grouped_operand_applies(a, [m[0] for m in members], [0 if m[1] is None else m[1].shape[1] for m in members],
                                      center, reference_rounding)
    if rounded and center is not None and not operand:
        if M >= 256 and K % 32 == 0:
            ax = expand_tiled(a, cache=a.shared, mode=MODE_PB16, center=center)
            return [linear_fwd_tiled(a, b, t=t, u=u, bias=bias, out_dtype=out_dtype, a_tiled=ax, reference_rounding=True, split_k=split_k)
                    for b, t, u, bias in members]
        rounded = False                                        # exact products, the centre's share in binary32
    if rounded and not takes:
        return [linear_fwd(a, b, t=t, u=u, bias=bias, out_dtype=out_dtype, split_k=split_k, reference_rounding=True)
                for b, t, u, bias in members]
    words, specs = _grouped_members(members, M, K, out_dtype, takes and M < 256 and decode_layout_weights)
    # split-K scratch (long K, few columns) and whether a centre fits the launch: functions of the shape alone
    ns = tuple(m[0].rows for m in members)
    need, centre_ok = _grouped_plan(M, K, ns, dev.index or 0) if split_k else (0, _grouped_centre_fits_unsplit(M, K, ns, dev.index or 0))
    dt = DTYPE_F32 if out_dtype == torch.float32 else DTYPE_BF16
    if rotate is not None:
        op_mode = MODE_PB16 if rounded else MODE_P32          # (nv_operand_mode: what a caller that brings a_operand built it in)
        aop = a_operand if a_operand is not None else decode_operand(a, op_mode, None, rotate=rotate)
        return _grouped_call("metis_linear_fwd_grouped_operand", dev, words, specs, need, (aop, a.unit, M, K, words, len(members), dt, op_mode))
    if operand:
        # (a quantizer call that deferred its scale bytes never gets them: the operand kernel forms them on the way)
        aop = a_operand if a_operand is not None else decode_operand(a, MODE_PB16, center)
        return _grouped_call("metis_linear_fwd_grouped_operand", dev, words, specs, need, (aop, a.unit, M, K, words, len(members), dt, MODE_PB16))
    # the activation's decode layout (written by its quantizer) in place of the row-major packing: wide runs only
    a_dec = a.decode_layout if (takes and K % 256 == 0 and all(m[0].scales.data_ptr() % 8 == 0 for m in members)) else None
    a_codes, a_scales = (a_dec, None) if a_dec is not None else (a.codes, a.scales)
    if center is not None:
        center = center.reshape(-1).to(device=dev, dtype=torch.float32).contiguous()
        if center.numel() != K:
            raise ValueError(f"center must have {K} values, got {center.numel()}")
        aligned = center.data_ptr() % 16 == 0 and all(m[0].scales.data_ptr() % 8 == 0 for m in members) and a.scales.data_ptr() % 8 == 0
        if aligned and centre_ok:
            return _grouped_call("metis_linear_fwd_grouped_centered", dev, words, specs, need,
                                 (a_codes, a_scales, a.unit, M, K, words, len(members), dt, center))
        # two passes: W^ center as a binary32 bias per member
        shifted = []
        for b, t, u, bias in members:
            w_mean = matvec(b, center)
            shifted.append((b, t, u, w_mean if bias is None else w_mean + bias.float()))
        return _linear_fwd_grouped(a, shifted, out_dtype)
    return _grouped_call("metis_linear_fwd_grouped_bf16" if rounded else "metis_linear_fwd_grouped", dev, words, specs, need,
                         (a_codes, a_scales, a.unit, M, K, words, len(members), dt))


def _grouped_call(name: str, dev: torch.device, words: list, specs: list, need: int, args: tuple) -> list[torch.Tensor]:
    """The launch of a grouped product with its split-K scratch; the members' outputs."""
    count = len(specs)
    if need:
        specs.append((U8, need))
    new = _lib.call(name, dev.index, tuple(specs), args + (_OUT[count] if need else None, need, _stream()))
    if new.__class__ is int:
        check(new, name, (args[2] if "operand" in name else args[3], [w[8] for w in words]))
    return list(new[:count])


def _tiled_backward_pays(M: int, N: int, K: int, device_index: int) -> bool:
    """Whether a backward product out[M, N] over a contraction of K goes to the pipelined kernel on tiled expansions made
    for this one call: from about 2e11 flop on, with at least one 256 x 256 tile per compute unit, the faster GEMM pays
    for writing the expansions.  Microseconds, packed | tiled with both operands expanded | with the weight's
    expansion kept: 8192 x 4096 over 14336 826 | 791 | 754, 14336 x 4096 over 8192 851 | 797, 18944 x 3584 over 2112 301 | 277; below
    either bound the two are close and the order varies: 4096 x 1536 over 8960 152 | 144 | 136, 8960 x 1536 over 4096
    115 | 119, 2103 x 3584 over 18944 307 | 315 | 273, 4096 x 3584 over 18944 496 | 494 | 451.  Plain products keep their
    bits; with a low-rank term the binary32 sums are taken in another order."""
    return (tiled_weight_copies and M >= 256 and N >= 256 and K % 32 == 0 and 2.0 * M * N * K >= 2e11
            and (M // 256) * (N // 256) >= _device_cus(device_index))


def linear_dgrad(dy: PackedNVFP4, wt: PackedNVFP4, out_dtype: torch.dtype = torch.bfloat16) -> torch.Tensor:
    """grad_input[L, K] from dY packed along N [L, N] and W packed along N (column-blocked) [K, N]."""
    if dy.cols != wt.cols:
        raise ValueError(f"contraction mismatch: {dy.cols} vs {wt.cols}")
    L, N, K = dy.rows, dy.cols, wt.rows
    if dy.mode == wt.mode and _tiled_backward_pays(L, K, N, dy.codes.device.index or 0):
        return linear_fwd(dy, wt, out_dtype=out_dtype, tiled=True)          # out = deq(dy) . deq(wt)^T: the same product
    return _packed_product("dgrad", dy, wt, (L, K, N), (L, N, K), out_dtype)


def linear_wgrad(dyt: PackedNVFP4, xt: PackedNVFP4, out_dtype: torch.dtype = torch.float32) -> torch.Tensor:
    """grad_weight[N, K] from dY and X both packed along tokens: dyt [N, L], xt [K, L]."""
    if dyt.cols != xt.cols:
        raise ValueError(f"contraction mismatch: {dyt.cols} vs {xt.cols}")
    N, L, K = dyt.rows, dyt.cols, xt.rows
    if dyt.mode == xt.mode and _tiled_backward_pays(N, K, L, dyt.codes.device.index or 0):
        return linear_fwd(dyt, xt, out_dtype=out_dtype, tiled=True)
    return _packed_product("wgrad", dyt, xt, (N, K, L), (L, N, K), out_dtype)


def _packed_product(which: str, a: PackedNVFP4, b: PackedNVFP4, product: tuple, shape: tuple, out_dtype: torch.dtype) -> torch.Tensor:
    """metis_linear_dgrad / _wgrad with the split-K scratch of the product [M, N] over K; shape: the entry point's own three sizes."""
    dev = a.codes.device
    M, N, K = product
    need = 0 if (M >= 256 and N < 256) else _linear_workspace_bytes(M, N, K, dev.index or 0)
    f32 = out_dtype == torch.float32
    specs = ((F32 if f32 else B16, M, N),)
    args = (a.codes, a.scales, a.unit, b.codes, b.scales, b.unit, *shape, "0", DTYPE_F32 if f32 else DTYPE_BF16)
    if need:
        name = f"metis_linear_{which}_ws"
        new = _lib.call(name, dev.index, specs + ((U8, need),), args + ("1", need, _stream()))
    else:
        name = f"metis_linear_{which}"
        new = _lib.call(name, dev.index, specs, args + (_stream(),))
    if new.__class__ is int:
        check(new, name, shape)
    return new[0]
