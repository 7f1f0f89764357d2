"""Python face of the gfx950 kernel library: one function per kernel entry point.

Each function checks devices, dtypes and shapes on the host, then calls the flat C ABI
through ctypes on the current HIP stream. There is no CPU fallback: without the library
or without a GPU these functions raise.
"""

from __future__ import annotations

import ctypes
import functools
import importlib.util
import os
import sys
import time
import warnings
from typing import Dict, Optional, Union

import torch

from . import build as _build

# (the last two: a storing product leaves gelu of its float32 sums; a gated product gelu_tanh(gate) * up)
F32, BF16, BF16_GELU, BF16_GEGLU, BF16_TILES = 0, 1, 2, 3, 4
PAGE_SIZE = 64          # tokens per cache page: the width of a wavefront
COMPUTE_UNITS = 256     # of the chip
MAX_HEAD_DIM = 256          # of the matrix-core attention kernels
MAX_PLAIN_HEAD_DIM = 1024   # of the plain attention kernels, which serve what the others do not take

_lib = None


class KernelError(RuntimeError):
    pass


class _ProfiledLibrary:
    """The kernel library with every call bracketed by two events on the current stream.
    Nothing is waited for at a launch (a host that waits lets the GPU's clock drop, which would
    rescale every figure): the events are read when the report is asked for, as the reference's
    per-kernel profile does (native/src/v2_runtime.cpp:27590-27728)."""
    CAPACITY = 1 << 16

    def __init__(self, lib):
        self._library = lib
        self._pending = []          # (name, first event, second event)
        self._totals: Dict[str, Dict[str, float]] = {}
        self.overflow = 0

    def __getattr__(self, name):
        entry = getattr(self._library, name)
        if not name.startswith("fw_") or name in ("fw_last_error", "fw_abi_version") or name.endswith(("_plan", "_fits", "_tiles", "_floats", "_slots")):
            return entry

        def timed(*args):
            if len(self._pending) >= self.CAPACITY or torch.cuda.is_current_stream_capturing():
                self.overflow += 1
                return entry(*args)
            first, second = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            first.record()
            began = time.perf_counter()
            status = entry(*args)
            host_ms = (time.perf_counter() - began) * 1e3
            second.record()
            self._pending.append((name, first, second))
            total = self._totals.setdefault(name, {"calls": 0, "gpu_ms": 0.0, "host_launch_ms": 0.0, "max_us": 0.0})
            total["calls"] += 1
            total["host_launch_ms"] += host_ms
            return status
        return timed

    def report(self) -> Dict[str, Dict[str, float]]:
        torch.cuda.synchronize()
        for name, first, second in self._pending:
            ms = first.elapsed_time(second)
            total = self._totals[name]
            total["gpu_ms"] += ms
            total["max_us"] = max(total["max_us"], ms * 1e3)
        self._pending = []
        return {name: dict(total) for name, total in sorted(self._totals.items(), key=lambda item: -item[1]["gpu_ms"])}


_profiled: Optional[_ProfiledLibrary] = None


def kernel_profile(enable: bool = True) -> None:
    """Switches the per-kernel profile on or off (also switched on by FLYWEIGHT_KERNEL_PROFILE=1
    in the environment, as in the reference). While it is on, steps are not recorded into graphs."""
    global _profiled
    if enable and _profiled is None:
        _profiled = _ProfiledLibrary(library())
    elif not enable:
        _profiled = None


def kernel_profile_active() -> bool:
    return _profiled is not None


def kernel_profile_report() -> Dict[str, Dict[str, float]]:
    """Entry point -> calls, GPU milliseconds between its two events, host milliseconds inside
    the launching call, the longest single call in microseconds; sorted by GPU time."""
    return _profiled.report() if _profiled is not None else {}


_C_TYPES = {"int": ctypes.c_int, "float": ctypes.c_float, "size_t": ctypes.c_size_t, "long long": ctypes.c_longlong}


def _declare(lib) -> None:
    """Gives every entry point the argument types that the kernels' header declares: addresses and numbers then go
    through as they are. Wrapped one by one (an object per argument, about twenty of them a launch) they were a sixth of
    what the host spends on a launch, and a short prompt's step, some hundred launches, is bound by that."""
    for name, arguments in _build.declarations():
        entry = getattr(lib, name)
        entry.restype = ctypes.c_int
        entry.argtypes = [ctypes.c_void_p if "*" in argument else _C_TYPES[argument.rpartition(" ")[0]] for argument in arguments]


def library():
    """Loads (building first if nothing is built) the kernel library."""
    global _lib
    if _profiled is not None:
        return _profiled
    if _lib is None:
        path = _build.ensure_built()
        lib = ctypes.CDLL(path)
        lib.fw_last_error.restype = ctypes.c_char_p
        lib.fw_abi_version.restype = ctypes.c_int
        wanted = _build.abi_version()       # compared first: a library of another interface may lack what is declared now
        if lib.fw_abi_version() != wanted:
            raise KernelError(f"{path}: kernel library ABI {lib.fw_abi_version()} != {wanted}; rebuild it")
        _declare(lib)
        _lib = lib
        _load_native(lib)
        if os.environ.get("FLYWEIGHT_KERNEL_PROFILE", "")[:1] == "1":
            kernel_profile(True)
            return _profiled
    return _lib


# The launches of a prompt's step as functions of a native module (csrc/launch): checks, allocations and the call in one. The general paths below serve whatever
# it hands back (NotImplemented), everything while kernels are timed one by one, and everything where it could not be built.
_native = None
_NATIVE_ENTRIES = ("fw_gemm_rows", "fw_gemm_medium", "fw_gemm_mfma_big_tile", "fw_rmsnorm_rows", "fw_shortconv", "fw_qk_norm_rope_kv_write", "fw_attention_prefill",
                   "fw_last_error")


def _load_native(lib) -> None:
    global _native
    _native = None
    module = sys.modules.get(_build.LAUNCH_NAME)
    if module is None:
        try:
            spec = importlib.util.spec_from_file_location(_build.LAUNCH_NAME, _build.ensure_launch_built())
            module = importlib.util.module_from_spec(spec)
            spec.loader.exec_module(module)
        except (RuntimeError, OSError, ImportError) as error:
            warnings.warn(f"the native launches cannot be had; steps with prompts take longer on the host: {error}")
            return
        sys.modules[_build.LAUNCH_NAME] = module
    module.bind({name: ctypes.cast(getattr(lib, name), ctypes.c_void_p).value for name in _NATIVE_ENTRIES}, KernelError, torch.OutOfMemoryError)
    _native = module


def native_launches() -> bool:
    """Whether launches go through the native module."""
    return _native is not None and _profiled is None


def library_path() -> str:
    library()
    return _lib._name


def _check(status: int) -> None:
    if status:
        raise KernelError(library().fw_last_error().decode("utf-8", "replace"))


def _code(dtype: torch.dtype) -> int:
    if dtype == torch.float32:
        return F32
    if dtype == torch.bfloat16:
        return BF16
    raise KernelError(f"kernels take float32 or bfloat16, not {dtype}")


def _dev(*tensors: Optional[torch.Tensor]) -> None:
    for t in tensors:
        if t is not None and not (t.is_cuda and t.is_contiguous()):
            raise KernelError("kernels need contiguous tensors" if t.is_cuda else "kernels run on the GPU only; got a CPU tensor")


def _dev_rows(t: torch.Tensor, name: str) -> None:
    """A matrix whose rows may lie apart (a view of some columns of wider rows), each row contiguous."""
    if not t.is_cuda:
        raise KernelError("kernels run on the GPU only; got a CPU tensor")
    if t.dim() != 2 or t.stride(1) != 1:
        raise KernelError(f"{name} must be a matrix with contiguous rows")


def _stride(t: torch.Tensor) -> int:
    """Elements between the rows of a matrix (of a single row: its width)."""
    return t.stride(0) if t.shape[0] > 1 else max(t.shape[1], t.stride(0))


def _p(t: Optional[torch.Tensor]) -> Optional[int]:
    return None if t is None else t.data_ptr()


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)
_device = getattr(torch._C, "_cuda_getDevice", torch.cuda.current_device)      # (the tensors at hand have initialised the GPU)


def _stream() -> int:
    """The current HIP stream of the current device (asked for at every launch: a graph
    capture or a caller's stream context changes it)."""
    return _raw_stream(_device()) if _raw_stream is not None else torch.cuda.current_stream().cuda_stream


def _want(t: torch.Tensor, dtype: torch.dtype, name: str) -> None:
    if t.dtype != dtype:
        raise KernelError(f"{name} must be {dtype}, found {t.dtype}")


# ---------------------------------------------------------------------------------------
def embed_rows(table: torch.Tensor, ids: torch.Tensor, out: Optional[torch.Tensor] = None, scale: float = 1.0,
               places_table: Optional[torch.Tensor] = None, places: Optional[torch.Tensor] = None, copies: int = 1) -> torch.Tensor:
    """table[ids] * scale as float32 rows (``copies`` > 1: [rows, copies, hidden], every row that many times); with ``places_table`` and ``places`` (int32, one per row, checked against
    the table by the caller) plus places_table[places], not scaled."""
    _dev(table, ids, out, places_table, places)
    _want(ids, torch.int32, "ids")
    vocab, hidden = table.shape
    if (places_table is None) != (places is None):
        raise KernelError("embed_rows: a table of places and the rows' places come together")
    if places is not None:
        _want(places, torch.int32, "places")
        if places_table.dim() != 2 or places_table.shape[1] != hidden or places.numel() < ids.numel():
            raise KernelError(f"embed_rows: the table of places is {tuple(places_table.shape)} beside rows of {hidden}, {places.numel()} places for {ids.numel()} rows")
    rows = ids.numel()
    if out is None:
        out = torch.empty((rows, hidden) if copies == 1 else (rows, copies, hidden), dtype=torch.float32, device=table.device)
    _want(out, torch.float32, "out")
    if copies < 1 or out.shape != ((rows, hidden) if copies == 1 else (rows, copies, hidden)):
        raise KernelError(f"embed_rows: out is {tuple(out.shape)}, expected {(rows, hidden)} ({copies} copies)")
    _check(library().fw_embed_rows(_p(table), _code(table.dtype), _p(ids), _p(out), rows, hidden, vocab,
                                   float(scale), _p(places_table), _code(places_table.dtype) if places_table is not None else F32,
                                   _p(places), places_table.shape[0] if places_table is not None else 0, int(copies), _stream()))
    return out


def scale_softcap_(x: torch.Tensor, scale: float = 1.0, cap: float = 0.0) -> torch.Tensor:
    """In place on float32: x * scale, then with ``cap`` > 0 cap * tanh(x / cap)."""
    _dev(x)
    _want(x, torch.float32, "x")
    if cap < 0:
        raise KernelError("scale_softcap: the cap must not be negative")
    _check(library().fw_scale_softcap(_p(x), int(x.numel()), float(scale), float(cap), _stream()))
    return x


def rmsnorm_rows(x: torch.Tensor, weight: torch.Tensor, eps: float, out_dtype: torch.dtype,
                 row_index: Optional[torch.Tensor] = None, one_centered: bool = False,
                 out: Optional[torch.Tensor] = None) -> torch.Tensor:
    if _native is not None and _profiled is None and out is None and x.is_cuda and (out_dtype == torch.bfloat16 or out_dtype == torch.float32):
        made = _native.rmsnorm(x, weight, row_index, out_dtype == torch.bfloat16, eps, one_centered, _stream())
        if made is not NotImplemented:
            return made
    _dev(x, weight, row_index, out)
    _want(x, torch.float32, "x")
    _want(weight, torch.float32, "weight")
    hidden = x.shape[-1]
    if weight.shape != (hidden,):
        raise KernelError(f"rmsnorm: weight is {tuple(weight.shape)}, row width is {hidden}")
    rows = x.numel() // hidden if row_index is None else row_index.numel()
    if row_index is not None:
        _want(row_index, torch.int32, "row_index")
    if out is None:
        out = torch.empty(rows, hidden, dtype=out_dtype, device=x.device)
    elif out.shape != (rows, hidden) or out.dtype != out_dtype:
        raise KernelError("rmsnorm: out has the wrong shape or dtype")
    _check(library().fw_rmsnorm_rows(x.data_ptr(), weight.data_ptr(), out.data_ptr(), _code(out_dtype), _p(row_index), rows, hidden, float(eps), 1 if one_centered else 0,
                                     _stream()))
    return out


def gemm_generic(a: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor] = None,
                 out_dtype: Optional[torch.dtype] = None, accumulate_into: Optional[torch.Tensor] = None,
                 out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """a [M, K] . w [N, K]^T (+ bias). With ``accumulate_into`` (float32 [M, N]) the
    product is added to it in place: the residual sum in float32."""
    _dev(a, w, bias, accumulate_into, out)
    M, K = a.shape
    N, K2 = w.shape
    if K != K2:
        raise KernelError(f"gemm: a is {tuple(a.shape)} but w is {tuple(w.shape)}")
    if bias is not None:
        _want(bias, torch.float32, "bias")
        if bias.shape != (N,):
            raise KernelError(f"gemm: bias is {tuple(bias.shape)}, expected {(N,)}")
    if accumulate_into is not None:
        _want(accumulate_into, torch.float32, "accumulate_into")
        if accumulate_into.shape != (M, N):
            raise KernelError(f"gemm: destination is {tuple(accumulate_into.shape)}, expected {(M, N)}")
        target, mode, code = accumulate_into, 1, F32
    else:
        out_dtype = out_dtype or a.dtype
        if out is None:
            out = torch.empty((M, N), dtype=out_dtype, device=a.device)
        if out.shape != (M, N) or out.dtype != out_dtype:
            raise KernelError("gemm: out has the wrong shape or dtype")
        target, mode, code = out, 0, _code(out_dtype)
    if _float32_ok(a, w):
        _check(library().fw_gemm_float32(_p(a), _p(w), _p(bias), _p(target), code, mode, M, N, K, _stream()))
    else:
        _check(library().fw_gemm_generic(_p(a), _code(a.dtype), _p(w), _code(w.dtype), _p(bias), _p(target), code, mode,
                                         M, N, K, _stream()))
    return target


@functools.lru_cache(maxsize=4096)
def float32_normed_takes(gated: bool, rows: int, features: int, k: int) -> bool:
    """Whether a float32 product of few rows takes their RMS norm in front (``gemm_float32_normed``)."""
    return bool(library().fw_gemm_float32_normed_takes(2 if gated else 0, rows, features, k))


def gemm_float32_normed(x: torch.Tensor, norm_weight: torch.Tensor, eps: float, one_centered: bool, w: torch.Tensor, bias: Optional[torch.Tensor] = None, *,
                        row_index: Optional[torch.Tensor] = None, gated: bool = False) -> torch.Tensor:
    """``rmsnorm_rows`` followed by the product with ``w`` (``gated``: silu(gate) * up of [gate rows; up rows]), float32 throughout, in one kernel and bit
    for bit as the two give it; ``float32_normed_takes`` says which shapes."""
    _dev(x, norm_weight, w, bias, row_index)
    for name, t in (("x", x), ("norm_weight", norm_weight), ("w", w)) + ((("bias", bias),) if bias is not None else ()):
        _want(t, torch.float32, name)
    if x.dim() != 2 or w.dim() != 2 or x.shape[1] != w.shape[1] or norm_weight.shape != (x.shape[1],):
        raise KernelError(f"gemm_float32_normed: x is {tuple(x.shape)}, w {tuple(w.shape)}, the norm's weight {tuple(norm_weight.shape)}")
    if row_index is not None:
        _want(row_index, torch.int32, "row_index")
    rows = x.shape[0] if row_index is None else row_index.numel()
    features = w.shape[0] // 2 if gated else w.shape[0]
    if (gated and w.shape[0] % 2) or (bias is not None and bias.shape != (w.shape[0],)):
        raise KernelError("gemm_float32_normed: gate and up rows are even in number, a bias has a value per row of w")
    if eps <= 0.0:
        raise KernelError("gemm_float32_normed: eps must be positive")
    out = torch.empty((rows, features), dtype=torch.float32, device=x.device)
    _check(library().fw_gemm_float32_normed(_p(x), _p(norm_weight), _p(row_index), float(eps), int(one_centered), _p(w), _p(bias), _p(out), 2 if gated else 0, rows,
                                            features, x.shape[1], _stream()))
    return out


def _float32_ok(a: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether the product runs on the float32 matrix instruction, whose lanes read four k at once; other operands and
    other K take the plain FMA tiles (one row, 1,024 outputs: 464 us against 9; 301 rows: 523 against 38)."""
    return (a.dtype == torch.float32 and w.dtype == torch.float32 and a.shape[1] % 4 == 0
            and a.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0)


def swiglu(gate_up: torch.Tensor, out_dtype: Optional[torch.dtype] = None,
           out: Optional[torch.Tensor] = None, gelu: bool = False) -> torch.Tensor:
    """silu(gate) * up of [rows, gate | up] (``gelu``: the tanh form of gelu in place of silu); the input may be float32
    beside a bfloat16 output."""
    _dev(gate_up, out)
    out_dtype = out_dtype or gate_up.dtype
    rows, width = gate_up.shape
    if width % 2:
        raise KernelError("swiglu: the input holds gate and up halves; its width must be even")
    inter = width // 2
    if out is None:
        out = torch.empty((rows, inter), dtype=out_dtype, device=gate_up.device)
    if out.shape != (rows, inter) or out.dtype != out_dtype:
        raise KernelError("swiglu: out has the wrong shape or dtype")
    _check(library().fw_swiglu(_p(gate_up), _code(gate_up.dtype), _p(out), _code(out_dtype), rows, inter, int(gelu), _stream()))
    return out


def rope_table(positions: torch.Tensor, inv_freq: torch.Tensor):
    """cos and sin [rows, half] (float32) of position * inv_freq (float64)."""
    _dev(positions, inv_freq)
    _want(positions, torch.int32, "positions")
    _want(inv_freq, torch.float64, "inv_freq")
    rows, half = positions.numel(), inv_freq.numel()
    cos = torch.empty((rows, half), dtype=torch.float32, device=positions.device)
    sin = torch.empty_like(cos)
    _check(library().fw_rope_table(_p(positions), _p(inv_freq), _p(cos), _p(sin), rows, half, _stream()))
    return cos, sin


def query_temperature(positions: torch.Tensor, coef: float, every: int) -> torch.Tensor:
    """float32 [rows]: 1 + coef * ln(floor((position + 1) / every) + 1)."""
    _dev(positions)
    _want(positions, torch.int32, "positions")
    out = torch.empty((positions.numel(),), dtype=torch.float32, device=positions.device)
    _check(library().fw_query_temperature(_p(positions), _p(out), positions.numel(), float(coef), int(every), _stream()))
    return out


def shortconv(bcx: torch.Tensor, taps: torch.Tensor, conv_bias: Optional[torch.Tensor], state: torch.Tensor,
              row_seg: torch.Tensor, seg_row0: torch.Tensor, seg_slot: torch.Tensor, segments: int,
              out_dtype: Optional[torch.dtype] = None, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """state [slots, H, L-1] is read and updated in place. ``bcx`` may be float32 beside a
    bfloat16 output."""
    if _native is not None and _profiled is None and out is None and bcx.is_cuda and (out_dtype == torch.bfloat16 or out_dtype == torch.float32):
        made = _native.shortconv(bcx, taps, conv_bias, state, row_seg, seg_row0, seg_slot, segments, out_dtype == torch.bfloat16, _stream())
        if made is not NotImplemented:
            return made
    _dev(bcx, taps, conv_bias, state, row_seg, seg_row0, seg_slot, out)
    out_dtype = out_dtype or bcx.dtype
    rows, width = bcx.shape
    hidden, kernel = taps.shape
    if width != 3 * hidden:
        raise KernelError(f"shortconv: input width {width} is not 3 x {hidden}")
    _want(taps, torch.float32, "taps")
    _want(state, torch.float32, "state")
    if state.dim() != 3 or state.shape[1:] != (hidden, kernel - 1):
        raise KernelError(f"shortconv: state is {tuple(state.shape)}, expected [slots, {hidden}, {kernel - 1}]")
    if conv_bias is not None:
        _want(conv_bias, torch.float32, "conv_bias")
        if conv_bias.shape != (hidden,):
            raise KernelError("shortconv: bias has the wrong shape")
    if (row_seg.dtype != torch.int32 or seg_row0.dtype != torch.int32 or seg_slot.dtype != torch.int32 or row_seg.numel() < rows
            or seg_row0.numel() <= segments or seg_slot.numel() < segments):
        for name, t, n in (("row_seg", row_seg, rows), ("seg_row0", seg_row0, segments + 1), ("seg_slot", seg_slot, segments)):
            _want(t, torch.int32, name)
            if t.numel() < n:
                raise KernelError(f"shortconv: {name} holds {t.numel()} entries, needs {n}")
    if out is None:
        out = torch.empty(rows, hidden, dtype=out_dtype, device=bcx.device)
    elif out.shape != (rows, hidden) or out.dtype != out_dtype:
        raise KernelError("shortconv: out has the wrong shape or dtype")
    _check(library().fw_shortconv(bcx.data_ptr(), _code(bcx.dtype), out.data_ptr(), _code(out_dtype), taps.data_ptr(), _p(conv_bias), state.data_ptr(),
                                  row_seg.data_ptr(), seg_row0.data_ptr(), seg_slot.data_ptr(), rows, segments, hidden, kernel, state.shape[0], _stream()))
    return out


def _check_pages(k_pages: torch.Tensor, v_pages: torch.Tensor, kv_heads: int, head_dim: int, dtype: torch.dtype,
                 v_dim: Optional[int] = None):
    pages = k_pages.shape[0]
    v_dim = head_dim if v_dim is None else v_dim
    if k_pages.shape != (pages, kv_heads, PAGE_SIZE, head_dim):
        raise KernelError(f"K pages are {tuple(k_pages.shape)}, expected [pages, {kv_heads}, {PAGE_SIZE}, {head_dim}]")
    if v_pages.shape != (pages, kv_heads, v_dim, PAGE_SIZE):
        raise KernelError(f"V pages are {tuple(v_pages.shape)}, expected [pages, {kv_heads}, {v_dim}, {PAGE_SIZE}]")
    if k_pages.dtype != dtype or v_pages.dtype != dtype:
        raise KernelError(f"cache pages are {k_pages.dtype}/{v_pages.dtype} but activations are {dtype}")
    return pages


def qk_norm_rope_kv_write(qkv: torch.Tensor, num_heads: int, num_kv_heads: int, head_dim: int,
                          q_norm_weight: Optional[torch.Tensor], k_norm_weight: Optional[torch.Tensor], eps: float,
                          cos: Optional[torch.Tensor], sin: Optional[torch.Tensor], rotary_dim: int,
                          k_pages: torch.Tensor, v_pages: torch.Tensor, block_table: torch.Tensor,
                          row_seg: torch.Tensor, row_pos: torch.Tensor, write_kv: bool = True,
                          v_dim: Optional[int] = None, interleaved: bool = False, q_only: bool = False,
                          q_row_scale: Optional[torch.Tensor] = None) -> torch.Tensor:
    """The output and the cache take the pages' dtype; ``qkv`` may be float32 beside bfloat16 pages, and its rows may lie
    apart (some columns of wider rows).
    ``q_row_scale`` (float32 [rows]): a factor on each row's finished queries.
    ``v_dim``: the size of a value head where it is not ``head_dim``. ``interleaved``: channel 2i turns
    with channel 2i + 1 instead of channel i with channel i + rotary_dim / 2."""
    if _native is not None and _profiled is None and qkv.is_cuda:
        made = _native.qk_norm(qkv, num_heads, num_kv_heads, head_dim, q_norm_weight, k_norm_weight, eps, cos, sin, rotary_dim, k_pages, v_pages, block_table, row_seg,
                               row_pos, write_kv, head_dim if v_dim is None else v_dim, interleaved, q_only, q_row_scale, PAGE_SIZE, _stream())
        if made is not NotImplemented:
            return made
    _dev(q_norm_weight, k_norm_weight, cos, sin, k_pages, v_pages, block_table, row_seg, row_pos)
    _dev_rows(qkv, "qkv")
    rows, width = qkv.shape
    v_dim = head_dim if v_dim is None else int(v_dim)
    expected = num_heads * head_dim if q_only else (num_heads + num_kv_heads) * head_dim + num_kv_heads * v_dim
    if width != expected or (q_only and write_kv):
        raise KernelError(f"qk_norm_rope: qkv width {width} != {expected} (queries alone: {q_only}; they bring nothing to store)")
    pages = _check_pages(k_pages, v_pages, num_kv_heads, head_dim, k_pages.dtype, v_dim)
    for w in (q_norm_weight, k_norm_weight):
        if w is not None:
            _want(w, torch.float32, "norm weight")
            if w.shape != (head_dim,):
                raise KernelError("qk_norm_rope: a head norm weight must be [head_dim]")
    if rotary_dim:
        for t in (cos, sin):
            _want(t, torch.float32, "rotation table")
            if t.shape != (rows, rotary_dim // 2):
                raise KernelError(f"qk_norm_rope: rotation table is {tuple(t.shape)}, expected {(rows, rotary_dim // 2)}")
    _want(block_table, torch.int32, "block_table")
    _want(row_seg, torch.int32, "row_seg")
    _want(row_pos, torch.int32, "row_pos")
    if block_table.dim() != 2 or row_seg.numel() < rows or row_pos.numel() < rows:
        raise KernelError("qk_norm_rope: batch index arrays are too short")
    q_out = torch.empty((rows, num_heads * head_dim), dtype=k_pages.dtype, device=qkv.device)
    _row_scale(q_row_scale, rows)
    _check(library().fw_qk_norm_rope_kv_write(
        _p(qkv), _code(qkv.dtype), _stride(qkv), _p(q_out), _code(k_pages.dtype), _p(q_norm_weight), _p(k_norm_weight), float(eps), _p(cos), _p(sin),
        rotary_dim, _p(k_pages), _p(v_pages), _p(block_table), block_table.shape[1], _p(row_seg), _p(row_pos), rows,
        num_heads, num_kv_heads, head_dim, v_dim, PAGE_SIZE, pages, int(write_kv), int(interleaved), int(q_only), _p(q_row_scale), _stream()))
    return q_out


def _row_scale(q_row_scale: Optional[torch.Tensor], rows: int) -> None:
    if q_row_scale is not None:
        _dev(q_row_scale)
        _want(q_row_scale, torch.float32, "q_row_scale")
        if q_row_scale.numel() < rows:
            raise KernelError(f"a factor per row: {q_row_scale.numel()} for {rows} rows")


def _sinks(sinks: Optional[torch.Tensor], num_heads: int, keep_first: int, window: int, chunk: int,
           slopes: Optional[torch.Tensor] = None):
    """Checks what the mask and the softmax take beyond a window: ``keep_first`` first keys that stay seen
    (beside a window only), one more term exp(sinks[head]) in the denominator (float32 [heads]) and a bias by
    distance (``slopes`` float32 [heads]: slopes[head] * (row's position - key's position) is taken off a score)."""
    if slopes is not None:
        _dev(slopes)
        _want(slopes, torch.float32, "slopes")
        if slopes.shape != (num_heads,):
            raise KernelError(f"attention: slopes are {tuple(slopes.shape)}, expected one per head ({num_heads})")
    if keep_first < 0 or (keep_first and chunk):
        raise KernelError(f"attention: {keep_first} first keys are kept beside a window, not beside chunks")
    if sinks is not None:
        _dev(sinks)
        _want(sinks, torch.float32, "sinks")
        if sinks.shape != (num_heads,):
            raise KernelError(f"attention: sinks are {tuple(sinks.shape)}, expected one per head ({num_heads})")
    return int(keep_first) if window else 0, _p(sinks), _p(slopes)


def attention_generic(q: torch.Tensor, num_heads: int, num_kv_heads: int, head_dim: int, k_pages: torch.Tensor,
                      v_pages: torch.Tensor, block_table: torch.Tensor, row_seg: torch.Tensor, row_pos: torch.Tensor,
                      scale: float, window: int = 0, v_dim: Optional[int] = None, chunk: int = 0,
                      softcap: float = 0.0, keep_first: int = 0, sinks: Optional[torch.Tensor] = None,
                      slopes: Optional[torch.Tensor] = None) -> torch.Tensor:
    """``v_dim``: the size of a value head (and of a head's output) where it is not ``head_dim``.
    ``chunk`` > 0: a row sees only the keys of its own chunk of that many positions; ``softcap`` c > 0:
    score <- c tanh(score / c)."""
    _dev(q, k_pages, v_pages, block_table, row_seg, row_pos)
    rows = q.shape[0]
    v_dim = head_dim if v_dim is None else int(v_dim)
    if q.shape != (rows, num_heads * head_dim):
        raise KernelError(f"attention: q is {tuple(q.shape)}, expected {(rows, num_heads * head_dim)}")
    pages = _check_pages(k_pages, v_pages, num_kv_heads, head_dim, q.dtype, v_dim)
    _want(block_table, torch.int32, "block_table")
    _want(row_seg, torch.int32, "row_seg")
    _want(row_pos, torch.int32, "row_pos")
    if block_table.dim() != 2 or row_seg.numel() < rows or row_pos.numel() < rows:
        raise KernelError("attention: batch index arrays are too short")
    out = torch.empty((rows, num_heads * v_dim), dtype=q.dtype, device=q.device)
    _check(library().fw_attention_generic(
        _p(q), _p(out), _code(q.dtype), _p(k_pages), _p(v_pages), _p(block_table), block_table.shape[1], _p(row_seg),
        _p(row_pos), rows, num_heads, num_kv_heads, head_dim, v_dim, float(scale), int(window), int(chunk),
        float(softcap), *_sinks(sinks, num_heads, keep_first, window, chunk, slopes), PAGE_SIZE, pages, _stream()))
    return out


def argmax_rows(logits: torch.Tensor, out: Optional[torch.Tensor] = None, also: Optional[torch.Tensor] = None,
                advance: Optional[torch.Tensor] = None) -> torch.Tensor:
    """The id of each row's largest logit (ties: the lowest id), int32 [rows], into ``out`` if
    given and into ``also`` as well; ``advance[r]`` goes up by one (all contiguous int32 of at
    least ``rows`` elements)."""
    _dev(logits)
    _want(logits, torch.float32, "logits")
    rows, vocab = logits.shape
    ids = out if out is not None else torch.empty((rows,), dtype=torch.int32, device=logits.device)
    for name, target in (("out", out), ("also", also), ("advance", advance)):
        if target is not None:
            _dev(target)
            _want(target, torch.int32, name)
            if target.numel() < rows or not target.is_contiguous():
                raise KernelError(f"argmax_rows: {name} must be contiguous and hold {rows} ids")
    workspace = torch.empty((max(rows, 1), 64), dtype=torch.int64, device=logits.device)       # best key of each part
    _check(library().fw_argmax_rows(_p(logits), _p(ids), _p(also), _p(advance), _p(workspace), rows, vocab, _stream()))
    return ids


def sample_rows(logits: torch.Tensor, settings: torch.Tensor, states: torch.Tensor, out: Optional[torch.Tensor] = None,
                also: Optional[torch.Tensor] = None, advance: Optional[torch.Tensor] = None) -> torch.Tensor:
    """The next token of every row, drawn on the device (fw_sample_rows): ``settings`` float32
    [rows, 4] = temperature (0: greedy), top_k (0: all), top_p, min_p; ``states`` int64 [rows], the
    rows' xorshift64* generators, moved on in place by the rows that draw. ``out`` / ``also`` /
    ``advance`` as for ``argmax_rows``."""
    _dev(logits, settings, states)
    _want(logits, torch.float32, "logits")
    _want(settings, torch.float32, "settings")
    _want(states, torch.int64, "states")
    rows, vocab = logits.shape
    if settings.numel() < 4 * rows or states.numel() < rows or not settings.is_contiguous() or not states.is_contiguous():
        raise KernelError(f"sample_rows: settings must hold [{rows}, 4] and states [{rows}], contiguous")
    ids = out if out is not None else torch.empty((rows,), dtype=torch.int32, device=logits.device)
    for name, target in (("out", out), ("also", also), ("advance", advance)):
        if target is not None:
            _dev(target)
            _want(target, torch.int32, name)
            if target.numel() < rows or not target.is_contiguous():
                raise KernelError(f"sample_rows: {name} must be contiguous and hold {rows} ids")
    _check(library().fw_sample_rows(_p(logits), _p(settings), _p(states), _p(ids), _p(also), _p(advance), rows, vocab, _stream()))
    return ids


def fill_zero(t: torch.Tensor) -> None:
    _dev(t)
    _check(library().fw_fill_zero(_p(t), int(t.numel() * t.element_size()), _stream()))


def fill_zero_pieces(first: torch.Tensor, pieces: int, stride_bytes: int) -> None:
    """Clears ``pieces`` runs of memory the size of ``first`` (contiguous), ``stride_bytes`` apart,
    beginning with ``first`` itself: the caller vouches that all of them lie in one allocation."""
    _dev(first)
    _check(library().fw_fill_zero_pieces(_p(first), int(pieces), int(first.numel() * first.element_size()),
                                         int(int(stride_bytes)), _stream()))


def gather_rows(rows: torch.Tensor, index: torch.Tensor) -> torch.Tensor:
    """rows[index] for float32 rows and an int32 index on the device (the embedding kernel: a
    table of rows is a table of rows)."""
    return embed_rows(rows, index)


def skinny_takes(M: int, N: int, K: int) -> bool:
    """Whether a product of up to 16 rows goes to the kernel without rings of operands in LDS (fw_gemm_skinny): with a short K, as far as
    its narrow loads of W do not show. Storing, from memory, us (skinny / waves that split K): 16 features over K 256 2.2 / 2.9, 2,048
    over 768 at 16 rows 3.8 / 4.0, over 1,024 at 8 4.2 / 4.3, at 16 4.6 / 4.4; 12,288 over 512 6.0 / 6.1, over 1,024 9.0 / 8.2."""
    return N <= 16384 and K <= (512 if N > 8192 else 1024 if M <= 8 else 768)


@functools.lru_cache(maxsize=4096)
def rows_fit(mode: int, M: int, N: int, K: int) -> bool:
    """Whether a product of more than 64 rows, its weights in operand tiles, goes to the kernel whose waves split K."""
    return M <= ROWS_MAX and bool(library().fw_gemm_rows_round_fits(mode, M, N, K))


def _fast_gemm(a: torch.Tensor, w: torch.Tensor, bias, target: torch.Tensor, out_code: int, mode: int, N: int,
               w_tiled: Optional[torch.Tensor] = None) -> None:
    """bfloat16 operands on the matrix cores: up to 16 rows of a short K the skinny kernel; up to 64 rows, and with weights in operand tiles as long as its tiles are one
    round over the chip, the product whose waves split K; the tiled ones beyond, with weights in operand tiles the large tile that ``large_tile`` names."""
    M, K = a.shape
    if M <= DECODE_MAX_ROWS and skinny_takes(M, N, K):
        _check(library().fw_gemm_skinny(_p(a), _p(w), _p(bias), _p(target), out_code, mode, M, N, K, _stream()))
        return
    if w_tiled is not None and M > MEDIUM_MAX_ROWS:
        tile = large_tile(mode, M, N, K)
        if tile is not None:
            if rows_fit(mode, M, N, K):     # where the tiles could be read they have to be w's
                _tiled_for(w, w_tiled)
            rows, columns, each, slices, need_bytes, need_counters = tile
            workspace_at = counters_at = None
            if need_bytes:
                workspace = torch.empty(need_bytes // 4, dtype=torch.float32, device=a.device)
                workspace_at, counters_at = workspace.data_ptr(), _medium_counters(a.device, need_counters).data_ptr()
            _check(library().fw_gemm_mfma_big_tile(a.data_ptr(), w.data_ptr(), None if bias is None else bias.data_ptr(), target.data_ptr(), out_code, mode, M, N, K,
                                                   rows, columns, each, slices, workspace_at, need_bytes, counters_at, need_counters, _stream()))
            return
    if M <= MEDIUM_MAX_ROWS or (w_tiled is not None and rows_fit(mode, M, N, K)):
        if out_code == BF16_GEGLU:      # that product is told by its unit, not by the output's type
            gemm_medium_into(a, w, bias, target, BF16, mode, N, w_tiled=w_tiled, glu=GEGLU)
        else:
            gemm_medium_into(a, w, bias, target, out_code, mode, N, w_tiled=w_tiled)
        return
    kind, columns = tiled_plan(mode, M, N, K)
    if kind == "deep":
        _check(library().fw_gemm_mfma_deep(_p(a), _p(w), _p(bias), _p(target), out_code, mode, M, N, K, columns, _stream()))
        return
    if kind in ("split", "bigsplit"):
        need_bytes, need_counters = (_split_needs if kind == "split" else _big_split_needs)(mode, M, N, K)[:2]
        workspace = torch.empty(need_bytes // 4, dtype=torch.float32, device=a.device)
        counters = _medium_counters(a.device, need_counters)
        entry = library().fw_gemm_mfma_split if kind == "split" else library().fw_gemm_mfma_big_split
        _check(entry(_p(a), _p(w), _p(bias), _p(target), out_code, mode, M, N, K, _p(workspace), ctypes.c_size_t(need_bytes), _p(counters),
                     counters.numel(), _stream()))
        return
    entry = library().fw_gemm_mfma_big if kind == "big" else library().fw_gemm_mfma
    _check(entry(_p(a), _p(w), _p(bias), _p(target), out_code, mode, M, N, K, _stream()))


def _split_needs(mode: int, M: int, N: int, K: int):
    """(bytes of workspace, counters) of the product that cuts K over workgroups; zeros where it does not take the shape."""
    need_bytes, need_counters = ctypes.c_size_t(0), ctypes.c_int(0)
    _check(library().fw_gemm_mfma_split_plan(mode, M, N, K, ctypes.byref(need_bytes), ctypes.byref(need_counters)))
    return need_bytes.value, need_counters.value


def _big_split_needs(mode: int, M: int, N: int, K: int):
    """(bytes of workspace, counters, slices of K) of the product that cuts K over workgroups on large tiles; zeros where it does not take the shape."""
    slices, need_bytes, need_counters = ctypes.c_int(0), ctypes.c_size_t(0), ctypes.c_int(0)
    _check(library().fw_gemm_mfma_big_split_plan(mode, M, N, K, ctypes.byref(slices), ctypes.byref(need_bytes), ctypes.byref(need_counters)))
    return need_bytes.value, need_counters.value, slices.value


# What the tiled products take, us: start + rounds * round + tiles / 256 * tile + K / 1,024 * (rounds * walk + tiles / 256 * fill), rounds those of
# their tiles over the 256 compute units (a round that is little full is a little faster). By mode: storing, adding, gated. Fitted to 2,200
# shapes (the large tiles: 852, when their loop changed) of 65 to 16,384 rows by 32 to 16,384 features over K 32 to 12,288, the weights from memory, to 4 to 12 % (mean square), with no part
# below zero: parts that were, fitted to shapes of few rounds, made many rounds over a short K free.
_TIME_DEEP = {0: {128: (3.2, 9.1, 1.4, 4.76, 3.28), 64: (2.6, 3.9, 1.2, 3.56, 1.54)},
              1: {128: (2.7, 10.4, 1.9, 4.84, 2.64), 64: (2.4, 4.5, 1.3, 3.62, 1.26)}}
_TIME_DEEP_FEW_ROWS = 1.25     # 64 columns, a long K, at most three rows of tiles sharing what they read of the weights (256 x 2,112 over 7,872: 53 us, by the parts alone 38)
# ... through registers, where two workgroups share a compute unit, two parts more: for each pair of rounds (a gated product's third round
# and those behind it: half a pair each), for 1,024 k of it
_TIME_TILES = {0: {128: (5.1, 0.0, 1.5, 6.32, 2.84, 6.2, 0.92), 64: (0.0, 0.3, 0.8, 3.64, 1.42, 6.2, 2.54)},
               1: {128: (0.3, 0.0, 6.1, 5.87, 1.06, 11.7, 3.78), 64: (0.0, 1.1, 1.3, 2.55, 2.66, 5.1, 3.81)},
               2: {64: (3.2, 0.8, 0.5, 5.52, 1.82, 2.8, 3.67)}}
_TIME_RAGGED = 3.0       # ... adding into features that end inside a tile of 64, and the same with K cut: a branch and a load an element
_TIME_BIG = {0: {128: (2.3, 2.8, 3.2, 0.301, 0.099), 256: (4.1, 2.3, 7.0, 0.219, 0.114)},     # by the tile's rows; walk and fill by 32 x 32 of its area
             1: {128: (0.9, 5.1, 3.8, 0.301, 0.111), 256: (5.5, 0.9, 14.8, 0.217, 0.118)}, 2: {256: (1.8, 5.7, 1.6, 0.239, 0.095)}}
_TIME_BIG_ODD = 4.0      # a round more of gated products with an odd number of features, which leave element by element
# ... with K cut: start, a slice's part in the sum at the end, 1,024 k of a slice in each round and for 256 workgroups, 256 workgroups
_TIME_SPLIT = {0: (8.3, 0.44, 4.6, 3.4, 1.5), 1: (7.3, 0.55, 4.8, 4.55, 4.0), 2: (8.3, 0.77, 8.7, 3.96, 2.5)}

# ... large tiles with K cut: start, a slice's part in the sum at the end, 256 workgroups, 1,024 k of a slice and for 256 workgroups
_TIME_BIG_SPLIT = {0: (8.4, 1.9, 5.5, 5.0, 8.6), 1: (10.6, 1.6, 5.6, 5.8, 7.9)}


def _tiled_time(tiles: int, K: int, start: float, each_round: float, each_tile: float, walk: float, fill: float, each_pair: float = 0.0,
                walk_pair: float = 0.0, gated: bool = False) -> float:
    rounds = -(-tiles // DEEP_ROUND)
    pairs = max(1.0, rounds / 2) if gated else -(-rounds // 2)
    share = tiles / DEEP_ROUND
    return (start + rounds * each_round + share * each_tile + pairs * each_pair
            + K / 1024 * (rounds * walk + share * fill + pairs * walk_pair))


def _tiled_times(mode: int, M: int, N: int, K: int):
    """The estimated time of every product on tiles of both operands that takes the shape, by (kind, columns)."""
    lib = library()
    wide, narrow = -(-M // 128) * -(-N // 128), -(-M // 128) * -(-N // 64)
    columns = 64 if mode == 2 or wide < DEEP_ROUND or (wide == DEEP_ROUND and K < LONG_K) else 128        # as fw_gemm_mfma chooses
    ragged = _TIME_RAGGED if mode == 1 and N % 64 else 0.0
    times = {("tiles", 0): _tiled_time(narrow if columns == 64 else wide, K, *_TIME_TILES[mode][columns], gated=mode == 2) + (ragged if columns == 64 else 0.0)}
    if mode != 2:
        for columns in (128, 64):
            tiles = lib.fw_gemm_mfma_deep_tiles(mode, M, N, K, columns)
            if tiles:
                few = columns == 64 and M <= 384 and K > 2560
                times["deep", columns] = _tiled_time(tiles, K, *_TIME_DEEP[mode][columns]) * (_TIME_DEEP_FEW_ROWS if few else 1.0)
    if M > BIG_MIN_ROWS:
        rows, columns = ctypes.c_int(0), ctypes.c_int(0)
        tiles = lib.fw_gemm_mfma_big_plan(mode, M, N, K, ctypes.byref(rows), ctypes.byref(columns))
        if tiles:
            start, each_round, each_tile, walk, fill = _TIME_BIG[mode][rows.value]
            area = rows.value * (256 if mode == 2 else columns.value) / 1024        # (a gated tile has gate and up columns)
            if mode == 2:
                each_round += _TIME_BIG_ODD if N % 2 else 0.0
            times["big", 0] = _tiled_time(tiles, K, start, each_round, each_tile, walk * area, fill * area)
    need_bytes, tiles = _split_needs(mode, M, N, K)
    if need_bytes:
        slices = need_bytes // (tiles * 128 * (128 if mode == 2 else 64) * 4)
        start, each, walk, fill, all_at_once = _TIME_SPLIT[mode]
        workgroups = tiles * slices
        share = workgroups / DEEP_ROUND
        times["split", 0] = (start + ragged + each * slices + share * all_at_once
                             + K / 1024 / slices * (walk * -(-workgroups // DEEP_ROUND) + fill * share))
    if mode != 2 and M > BIG_MIN_ROWS:
        need_bytes, tiles, slices = _big_split_needs(mode, M, N, K)
        if slices:
            start, each, all_at_once, walk, fill = _TIME_BIG_SPLIT[mode]
            share = tiles * slices / DEEP_ROUND
            times["bigsplit", 0] = start + each * slices + share * all_at_once + K / 1024 / slices * (walk + fill * share)
    return times


@functools.lru_cache(maxsize=4096)
def tiled_plan(mode: int, M: int, N: int, K: int):
    """Which of the products on tiles of both operands takes a shape, as (kind, columns of its tiles or 0): "big" (256 or 128 rows by up to
    256 columns), "bigsplit" (128 rows by 256, K cut over workgroups), "deep" (128 rows by 128 or 64, the waves split K), "tiles" (128 rows, through
    registers), "split" (those with K cut over workgroups). The least estimated time decides. Fixed numbers of
    tiles were 10 % above the fastest in the geometric mean, adding products of up to 2,048 features held to the tiles whose waves split K 5 %; K cut
    over workgroups takes 1,111 rows by 2,048 features over K 8,192 in 50 us against 60 on the tiles whose waves split K."""
    times = _tiled_times(mode, M, N, K)
    return min(times, key=times.get)


# The large tiles one by one, us, by (rows, columns, workgroups on a compute unit): start + rounds * round + tiles / 256 * tile + K / 1,024 * (rounds * walk +
# tiles / 256 * fill) + MB of weights * memory, rounds those of the tiles over the 256 compute units (over 512 places where two workgroups share one). Fitted to
# 420 shapes a mode (65 to 4,096 rows by 64 to 14,000 features over K 256 to 10,752, the weights from memory, no launch in the time) to 2.4 to 11 % (mean square).
_TIME_LARGE = {
    0: {(64, 128, 1): (1.479, 2.7, 0.387, 3.672, 1.243, 0.132), (64, 128, 2): (2.751, 0.488, 0.848, 3.974, 2.614, 0.122), (128, 128, 1): (2.133, 2.631, 1.925, 5.279, 1.699, 0.102),
        (128, 128, 2): (3.379, 0.0, 2.127, 6.304, 3.248, 0.071), (192, 128, 1): (2.607, 2.755, 2.626, 7.1, 2.099, 0.048), (64, 192, 1): (1.898, 2.731, 0.665, 4.762, 1.757, 0.176),
        (128, 192, 1): (2.073, 3.337, 1.99, 7.08, 1.83, 0.124), (128, 256, 1): (2.277, 3.438, 2.524, 8.98, 2.227, 0.135), (192, 192, 1): (2.267, 3.91, 3.176, 9.708, 2.078, 0.042),
        (192, 256, 1): (1.621, 5.112, 3.981, 12.299, 2.613, 0.049), (256, 192, 1): (1.774, 4.865, 3.937, 12.25, 2.695, 0.032), (256, 256, 1): (1.564, 6.259, 5.049, 15.86, 3.458, 0.02),
        (256, 320, 1): (0.0, 8.431, 3.819, 20.043, 4.24, 0.163)},
    1: {(64, 128, 1): (1.548, 2.711, 0.962, 3.716, 1.22, 0.147), (64, 128, 2): (2.46, 0.722, 1.346, 4.101, 2.628, 0.134), (128, 128, 1): (1.304, 3.83, 2.21, 5.427, 1.382, 0.115),
        (128, 128, 2): (1.934, 1.583, 3.413, 6.501, 2.787, 0.08), (192, 128, 1): (0.752, 5.218, 3.532, 7.165, 1.608, 0.073), (64, 192, 1): (1.554, 3.171, 1.097, 4.877, 1.585, 0.206),
        (128, 192, 1): (1.169, 4.72, 2.821, 7.253, 1.656, 0.135), (128, 256, 1): (1.68, 4.487, 5.011, 9.231, 1.665, 0.151), (192, 192, 1): (1.434, 5.569, 5.932, 9.822, 1.757, 0.049),
        (192, 256, 1): (0.797, 7.165, 7.688, 12.428, 2.505, 0.053), (256, 192, 1): (0.951, 6.927, 7.95, 12.431, 2.596, 0.003), (256, 256, 1): (0.0, 9.246, 10.769, 16.027, 3.126, 0.002),
        (256, 320, 1): (0.0, 10.509, 10.441, 20.3, 3.87, 0.144)},
    2: {(64, 128, 1): (1.537, 2.467, 0.0, 3.851, 1.227, 0.112), (64, 128, 2): (2.328, 0.577, 0.346, 4.133, 2.77, 0.106), (128, 128, 1): (1.606, 3.179, 0.278, 5.465, 1.516, 0.095),
        (128, 128, 2): (1.835, 1.195, 0.853, 6.48, 3.039, 0.082), (192, 128, 1): (1.821, 3.503, 0.574, 7.149, 1.813, 0.069), (64, 192, 1): (1.519, 2.702, 0.0, 5.07, 1.556, 0.141),
        (128, 192, 1): (1.393, 3.791, 0.244, 7.286, 1.741, 0.105), (128, 256, 1): (1.358, 3.944, 0.448, 9.29, 1.927, 0.109), (192, 192, 1): (1.796, 4.198, 0.672, 9.826, 1.84, 0.058),
        (192, 256, 1): (1.5, 5.095, 0.671, 12.494, 2.431, 0.049), (256, 192, 1): (1.514, 5.132, 0.447, 12.374, 2.544, 0.037), (256, 256, 1): (1.951, 5.817, 1.116, 15.924, 3.445, 0.013),
        (256, 320, 1): (1.562, 6.131, 1.696, 20.857, 3.561, 0.095)}}
# ... with K cut over workgroups: start, a slice's part in the sum at the end, 256 workgroups, 1,024 k of a slice and for 256 workgroups, MB of weights
_TIME_LARGE_CUT = {0: {(64, 128): (5.054, 0.448, 4.393, 3.678, 0.047, 0.083), (128, 128): (6.172, 0.703, 6.135, 5.315, 0.43, 0.068)},
                   1: {(64, 128): (6.096, 0.4, 3.895, 3.5, 0.874, 0.069), (128, 128): (7.824, 0.499, 5.709, 5.176, 0.861, 0.069)}}
# ... of the product whose waves split K (fw_gemm_rows): start, 1,024 k, and for 256 rows, for 4,096 rows of W, a million outputs, and 1,024 k of them
_TIME_ROWS = {0: (3.585, 0.562, 0.112, 1.194, 4.492, 3.142), 1: (3.719, 0.601, 0.108, 1.152, 4.71, 2.926),
              2: (4.209, 0.786, 0.139, 1.173, 3.606, 2.155)}
_TIME_OLDER = 1.05       # what the products of `_tiled_times` took of those shapes, by their estimates
_LARGE_LEAST_SLICE = 384     # k


@functools.lru_cache(maxsize=4096)
def _fastest_large(mode: int, rows64: int, N: int, K: int):
    """The large tile with the least estimated time for (rows64 - 1) * 64 + 1 to rows64 * 64 rows, its needs (``large_tile``) and that time: a tile's rows are a multiple of 64."""
    M, k, megabytes = rows64 * 64, K / 1024, N * (2 if mode == 2 else 1) * K * 2e-6
    best, least = None, 1e30
    for (rows, columns, each), (start, each_round, each_tile, walk, fill, memory) in _TIME_LARGE[mode].items():
        tiles = -(-M // rows) * -(-N // (columns // 2 if mode == 2 else columns))
        rounds, share = -(-tiles // (DEEP_ROUND * each)), tiles / DEEP_ROUND
        if mode == 2 and N % 2:
            each_round += _TIME_BIG_ODD
        time = start + rounds * each_round + share * each_tile + k * (rounds * walk + share * fill) + megabytes * memory
        if time < least:
            best, least = (rows, columns, each, 1), time
    for (rows, columns), (start, each_slice, all_at_once, walk, fill, memory) in _TIME_LARGE_CUT.get(mode, {}).items():
        tiles = -(-M // rows) * -(-N // columns)
        for slices in range(2, 9):
            if tiles * slices > DEEP_ROUND or K < slices * _LARGE_LEAST_SLICE:
                break
            share = tiles * slices / DEEP_ROUND
            time = start + slices * each_slice + share * all_at_once + k / slices * (walk + fill * share) + megabytes * memory
            if time < least and -(-K // slices // 64) * 64 * (slices - 1) < K:
                best, least = (rows, columns, 1, slices), time
    need_bytes, need_counters = ctypes.c_size_t(0), ctypes.c_int(0)
    _check(library().fw_gemm_mfma_big_tile_needs(mode, M, N, K, *best, ctypes.byref(need_bytes), ctypes.byref(need_counters)))
    return (*best, need_bytes.value, need_counters.value), least


@functools.lru_cache(maxsize=4096)
def _fastest_older(mode: int, rows128: int, N: int, K: int) -> float:
    """... and of ``tiled_plan``'s products, whose tiles (and the lines between them) are multiples of 128 rows."""
    return min(_tiled_times(mode, rows128 * 128, N, K).values())


@functools.lru_cache(maxsize=4096)
def large_tile(mode: int, M: int, N: int, K: int):
    """The large tile that takes a product of more than 64 rows by weights that a model holds (they come with their operand tiles; a bare product keeps to
    ``tiled_plan``, whose sums its callers know by the kernel's name): (rows, columns, workgroups on a compute unit, slices of K, bytes of workspace, counters),
    or None where the product whose waves split K or one of ``tiled_plan`` is estimated to be faster. Chosen so, the 420 shapes a mode take 1.8 (storing,
    adding) and 1.0 % (gated) more than with the fastest product each, and 12, 13 and 26 % less than without these tiles; no shape loses more than 15 %
    (adding 2,048 x 1,024 over K 1,024 13.3 -> 10.3 us, 801 x 2,048 over 7,168 43.3 -> 36.1, gated 500 x 4,608 over 1,024 24.8 -> 16.4, 2,048 x 4,608 55 -> 38).
    The estimates are kept by 64 (128) rows, since nearly every prompt has a length of its own: 400 lengths up to 2,048 took 17 to 23 us a product on the host
    when each was searched for anew, 4 to 6 now."""
    if K % 32 or K > 1 << 22 or N > 1 << 20:
        return None
    tile, least = _fastest_large(mode, -(-M // 64), N, K)
    if rows_fit(mode, M, N, K):
        start, walk, by_rows, by_width, outputs, by_outputs = _TIME_ROWS[mode]
        k, width = K / 1024, N * (2 if mode == 2 else 1)
        other = start + k * (walk + by_rows * M / 256 + by_width * width / 4096) + M * width * 1e-6 * (outputs + by_outputs * k)
    else:
        other = _TIME_OLDER * _fastest_older(mode, -(-M // 128), N, K)
    return None if other <= least else tile


MEDIUM_MAX_ROWS = 64
# Beyond 64 rows the waves-split-K product (gemm_rows.hip) is taken for weights in operand tiles while its tiles, of at most 64 x 64, are one round over the 256
# compute units; measured against the tiled products, every weight from memory: adding 2,048 features (K 8,192) at 128 / 256 / 512
# rows 20.6 / 26.2 / 34.8 against 25.0 / 30.6 / 44.1 us, K 2,048 8.2 / 10.6 / 14.3 against 14.8 / 15.1 / 18.9; storing 3,072 features at
# 256 rows 14.4 against 18.1, 6,144 at 128 rows 15.3 against 18.9. With two rounds it loses (6,144 features at 192 rows 25.9 against
# 17.3, 3,072 at 384 rows 24.4 against 18.3, 16,384 gated at 128 rows 35 against 27), and so it does with a long K where the others' tiles
# fill their round (fw_gemm_rows_round_fits).
ROWS_MAX = 1024
DEEP_ROUND = 256          # tiles of a round: one per compute unit
BIG_MIN_ROWS = 128       # up to here a 256-row tile would be at least half empty (the head at 128 rows: 110 vs 78 us)
_MEDIUM_COUNTERS = {}


TICKET_COUNTERS = 1 << 20      # 4 MB per device


def _medium_counters(device: torch.device, count: int) -> torch.Tensor:
    """Zeroed int32 counters for the tickets of the kernels whose last workgroup finishes the
    work of the others (products whose K is cut over workgroups, decode attention), one set per device: each kernel
    leaves them at zero, and calls on one device follow each other in stream order (work on
    several streams of one device at once would need a set per stream). The set is allocated
    once and never replaced: recorded graphs hold its address."""
    have = _MEDIUM_COUNTERS.get(device.index)
    if have is None:
        if torch.cuda.is_current_stream_capturing():
            raise KernelError("the ticket counters must exist before a graph is captured (prepare_device)")
        have = _MEDIUM_COUNTERS[device.index] = torch.zeros(TICKET_COUNTERS, dtype=torch.int32, device=device)
    if count > have.numel():
        raise KernelError(f"a kernel asks for {count} ticket counters; the device's set holds {have.numel()}")
    return have


def prepare_device(device: torch.device) -> None:
    """Allocates what kernels keep between calls on this device; a model does this when its
    weights arrive, so that nothing is allocated for the first time inside a graph capture."""
    _medium_counters(torch.device(device), 0)


def tile_weights(w: torch.Tensor) -> Optional[torch.Tensor]:
    """``w`` [rows, K] bfloat16 once more in operand tiles, [ceil(rows / 16), K / 32, 4, 16, 8]: what the
    decode products read as whole contiguous kilobytes per wave (see fw_gemm_decode). None where the
    layout does not apply (K no multiple of 32, another dtype)."""
    if w.dtype != torch.bfloat16 or w.dim() != 2 or w.shape[1] % 32 or not w.is_cuda:
        return None
    rows, K = w.shape
    padded = (rows + 15) // 16 * 16
    if padded != rows:
        w = torch.cat([w, torch.zeros((padded - rows, K), dtype=w.dtype, device=w.device)])
    return w.view(padded // 16, 16, K // 32, 4, 8).permute(0, 2, 3, 1, 4).contiguous()


class ExpertWeights:
    """The weights [rows, K] of every expert, held once for ``grouped_gemm``: in operand tiles where that layout applies (``tile_weights``), which steps of
    a few places an expert stream in whole kilobytes and the other products read as they read rows; else one behind the other. ``pieces``: called with an
    expert's number."""

    def __init__(self, experts: int, pieces):
        first = pieces(0).contiguous()
        rows, K = first.shape
        self.shape = (experts, rows, K)
        self.rows = self.tiled = None
        laid = tile_weights(first)
        if laid is None:
            self.rows = torch.stack([first, *(pieces(e) for e in range(1, experts))])
        elif rows % 16:             # experts that meet inside a tile
            self.tiled = tile_weights(torch.cat([first, *(pieces(e) for e in range(1, experts))]))
        else:
            self.tiled = laid.new_empty((experts * laid.shape[0], *laid.shape[1:]))
            for e, own in enumerate(self.tiled.chunk(experts)):
                own.copy_(laid if e == 0 else tile_weights(pieces(e).contiguous()))

    @property
    def held(self) -> torch.Tensor:
        return self.rows if self.tiled is None else self.tiled


@functools.lru_cache(maxsize=4096)
def _tiled_shape(rows: int, K: int) -> Optional[torch.Size]:
    return None if K % 32 else torch.Size(((rows + 15) // 16, K // 32, 4, 16, 8))


def _tiled_for(w: torch.Tensor, w_tiled: Optional[torch.Tensor]) -> Optional[torch.Tensor]:
    """``w_tiled`` if it is ``w`` in operand tiles (checked by its shape), else an error."""
    if w_tiled is None:
        return None
    rows, K = w.shape
    if (w_tiled.dtype != torch.bfloat16 or w_tiled.shape != _tiled_shape(rows, K) or not w_tiled.is_contiguous()
            or w_tiled.get_device() != w.get_device()):
        raise KernelError(f"weights in operand tiles for w {tuple(w.shape)} are bfloat16 [{(rows + 15) // 16}, {K // 32}, 4, 16, 8], "
                          f"found {tuple(w_tiled.shape)}")
    return w_tiled


# K from which a product that stores or adds up to 1,024 / 2,048 / 4,095 / 4,096 features splits it over workgroups, by the most rows
_LONG_K = ((8, (12288, 10240, 12288, 1 << 30)), (11, (8192, 10240, 8192, 12288)), (16, (6144, 6144, 6144, 12288)), (32, (10240, 10240, 6144, 10240)),
           (48, (16384, 16384, 12288, 1 << 30)), (64, (16384, 10240, 6144, 1 << 30)))


@functools.lru_cache(maxsize=4096)      # (asked at every launch: 0.2 to 0.7 us of the host's time worked out)
def medium_splits_k(mode: int, M: int, N: int, K: int) -> bool:
    """Whether a product of up to 64 rows goes to the kernel that splits K over workgroups (fw_gemm_medium, several workgroups on a
    compute unit) and not to the one whose waves do (fw_gemm_rows, tiles of up to 64 x 64, one workgroup on a compute unit). The
    latter loses, every weight from memory, us (splitting / waves):

    * with more than one round of its largest tiles: storing 20,480 features over K 2,048 at 17 / 64 rows 19.1 / 24.0, 29.3 / 30.8,
      65,536 at 64 rows 62 / 70, gated 10,752 over 2,048 22.5 / 24.6, 28.0 / 31.3 (not over K 2,056, in row-major order: 32.7 / 30.9);
    * with a short K on wide tiles: gated 4,608 over 1,024 at 32 rows 8.5 / 8.9, over 1,536 10.5 / 11.1, storing 16,384 over 1,024 at 17
      rows 9.4 / 10.8, 8,192 over 2,048 8.9 / 9.4 (10,240 over 2,048 leave the former's second round empty: 13.6 / 12.4);
    * with a long K and few tiles: adding 2,048 features over K 8,192 at 16 rows 12.0 / 13.0, over 12,288 13.1 / 18.3, at 32 rows
      15.2 / 18.2, at 64 21.3 / 23.3, over 10,240 at 64 19.5 / 20.4 but at 48 18.6 / 17.6; 1,024 over 10,240 at 32 rows 13.0 /
      14.6, at 64 17.3 / 14.1; 2,560, whose tiles of 16 leave a third of the chip without work, over 6,144 at 32 rows 12.0 /
      13.9; where the slices of K are more than a round they lose again (3,072 over 8,192 at 32 rows 20.3 / 17.2). Fewer rows
      pay the exchange later: adding 2,048 over 8,192 at 10 rows 11.9 / 11.7 (a decode step of 9 requests, 16 such products, 814 / 804,
      of 12 831 / 831, of 16 865 / 882), over 12,288 13.5 / 16.7; 1,024 over 6,144 at 9 rows 9.1 / 9.0, over 8,192 9.7 / 11.0. Up to
      eight rows come here in row-major order alone: 2,048 over 8,192 at 1 / 8 rows 13.2 / 11.0, 13.0 / 12.0, over 12,288
      15.4 / 14.9, 15.3 / 16.8, 4,096 over 12,288 26.9 / 22.5."""
    if mode == 2:
        return K % 32 == 0 and (N > 8192 or (N > 4096 and M > DECODE_MAX_ROWS and K <= (1536 if M <= 48 else 1024)))
    if N > 16384:
        return True
    if N > 4096:
        if M <= DECODE_MAX_ROWS:
            return False
        if M <= 32:
            return K <= 1024 or (K <= 2048 and not 8192 < N <= 12288)
        return N > 8192 and K <= (1024 if N > 12288 and M <= 48 else 512)
    tiles = -(-N // 32)
    if tiles * ((COMPUTE_UNITS + tiles // 2) // tiles) > COMPUTE_UNITS or (N <= 512 and M > DECODE_MAX_ROWS):
        return False
    least = next(by_features for rows, by_features in _LONG_K if M <= rows)
    return K >= least[0 if N <= 1024 else 1 if N <= 2048 else 2 if N < 4096 else 3]


@functools.lru_cache(maxsize=4096)
def _medium_plan(mode: int, M: int, N: int, K: int):
    """What the product that splits K over workgroups needs of a shape: bytes of workspace, counters, rows of sums of squares."""
    need_bytes, need_counters, squares_rows = ctypes.c_size_t(0), ctypes.c_int(0), ctypes.c_int(0)
    _check(library().fw_gemm_medium_plan(M, N, K, mode, ctypes.byref(need_bytes), ctypes.byref(need_counters), ctypes.byref(squares_rows)))
    return need_bytes.value, need_counters.value, squares_rows.value


@functools.lru_cache(maxsize=4096)
def _few_plan(mode: int, M: int, N: int, K: int):
    """Of a product of a few dozen rows: whether K is split over workgroups, then its bytes of workspace, counters and rows of sums of squares, and the rows
    of sums of squares of the kernel whose waves split K."""
    squares_rows = library().fw_gemm_rows_square_tiles(M, N)
    if M <= MEDIUM_MAX_ROWS and medium_splits_k(mode, M, N, K):
        return (True, *_medium_plan(mode, M, N, K), squares_rows)
    return False, 0, 0, 0, squares_rows


def gemm_medium_into(a: torch.Tensor, w: torch.Tensor, bias, target: torch.Tensor, out_code: int, mode: int, N: int,
                     next_norm_weight: Optional[torch.Tensor] = None, next_one_centered: bool = False,
                     squares: Optional[torch.Tensor] = None, eps: float = 0.0, w_tiled: Optional[torch.Tensor] = None,
                     glu: Optional[tuple] = None):
    """The product for 1..64 rows (more where nothing is prepared). With
    ``squares`` ``a`` holds prepared activations (x * w of an RMS norm) and the rows' 1/rms is
    formed from those sums. With ``next_norm_weight`` (accumulating product) returns what the
    norm after it needs: (activations x * w_next, sums of squares)."""
    M, K = a.shape
    stride = 16 if M <= DECODE_MAX_ROWS else 64
    squares_at, squares_rows = None, 0
    if squares is not None:
        if squares.dtype != torch.float32 or squares.dim() != 2 or squares.shape[1] != stride or not squares.is_contiguous():
            raise KernelError(f"gemm_medium: sums of squares for {M} rows are float32 [n, {stride}]")
        squares_at, squares_rows = squares.data_ptr(), squares.shape[0]
    operand, tiled = (w, 0) if w_tiled is None else (_tiled_for(w, w_tiled), 1)
    splits_k, need_bytes, need_counters, prepared_rows, whole_rows = _few_plan(mode, M, N, K)
    target_at = target.data_ptr()
    splits_k = splits_k and target_at % 16 == 0
    next_activations = next_squares = weight_at = activations_at = next_at = None
    if next_norm_weight is not None:
        device = a.device
        next_activations = torch.empty(M, N, dtype=torch.bfloat16, device=device)
        next_squares = torch.empty(prepared_rows if splits_k else whole_rows, stride, dtype=torch.float32, device=device)
        weight_at, activations_at, next_at = next_norm_weight.data_ptr(), next_activations.data_ptr(), next_squares.data_ptr()
    bias_at = None if bias is None else bias.data_ptr()
    limit, alpha, shift = _SWIGLU if glu is None else _glu(glu)
    if splits_k:
        workspace_at = counters_at = None
        counters_len = 0
        if need_bytes:
            workspace = torch.empty(need_bytes // 4, dtype=torch.float32, device=a.device)
            counters = _medium_counters(a.device, need_counters)
            workspace_at, counters_at, counters_len = workspace.data_ptr(), counters.data_ptr(), counters.numel()
        _check(library().fw_gemm_medium(a.data_ptr(), operand.data_ptr(), tiled, bias_at, target_at, out_code, mode, M, N, K,
                                        workspace_at, need_bytes, counters_at, counters_len, weight_at, 1 if next_one_centered else 0, activations_at, next_at,
                                        squares_at, squares_rows, float(eps), limit, alpha, shift, _stream()))
    else:
        _check(library().fw_gemm_rows(a.data_ptr(), operand.data_ptr(), tiled, bias_at, target_at, out_code, mode, M, N, K,
                                      weight_at, 1 if next_one_centered else 0, activations_at, next_at, squares_at, squares_rows, float(eps), limit, alpha, shift,
                                      _stream()))
    if next_norm_weight is not None:
        return next_activations, next_squares
    return None


@functools.lru_cache(maxsize=8192)
def _native_plan(few: bool, tiled: bool, mode: int, M: int, N: int, K: int):
    """How the native module launches a product: (0, *_few_plan) or (1, *large_tile), None for the general path. ``few``: the product of a few dozen rows was
    asked for by name."""
    if K % 8 or M < 1:
        return None
    if not few:
        if M <= DECODE_MAX_ROWS and skinny_takes(M, N, K):
            return None
        tile = large_tile(mode, M, N, K) if tiled and M > MEDIUM_MAX_ROWS else None
        if tile is not None:
            return (1, *tile)
        if M > MEDIUM_MAX_ROWS and not (tiled and rows_fit(mode, M, N, K)):
            return None
    elif M > MEDIUM_MAX_ROWS:
        return None
    return (0, *_few_plan(mode, M, N, K))


def _native_product(few: bool, a: torch.Tensor, w: torch.Tensor, w_tiled, bias, target, mode: int, out_dtype, gelu: bool = False, glu=None,
                    next_norm_weight=None, next_one_centered: bool = False, squares=None, eps: float = 0.0):
    """A product through the native module: what ``gemm_medium`` (``few``), ``gemm`` or ``gemm_swiglu`` return, or NotImplemented."""
    if not a.is_cuda or a.dim() != 2 or w.dim() != 2 or (out_dtype != torch.bfloat16 and out_dtype != torch.float32):
        return NotImplemented
    M, K = a.shape
    rows = w.shape[0]
    plan = _native_plan(few, w_tiled is not None, mode, M, rows // 2 if mode == 2 else rows, K)
    if plan is None:
        return NotImplemented
    tickets = plan[6] if plan[0] else plan[3]
    counters = _medium_counters(a.device, tickets) if tickets else None
    rounded = out_dtype == torch.bfloat16
    code = BF16 if rounded else F32
    if gelu:
        code = BF16_GELU
    elif glu == GEGLU and plan[0]:      # (the products of few rows are told by the unit, not by the output's type)
        code, glu = BF16_GEGLU, None
    limit, alpha, shift = _SWIGLU if glu is None else _glu(glu)
    return _native.product(a, w, w_tiled, bias, target, mode, code, rounded, next_norm_weight, next_one_centered, squares, eps, limit, alpha, shift, plan, counters,
                           _stream())


def gemm_medium(a: torch.Tensor, w: torch.Tensor, epilogue: int, *, bias: Optional[torch.Tensor] = None,
                out_dtype: Optional[torch.dtype] = None, accumulate_into: Optional[torch.Tensor] = None,
                squares: Optional[torch.Tensor] = None, eps: float = 0.0,
                next_norm_weight: Optional[torch.Tensor] = None, next_one_centered: bool = False,
                w_tiled: Optional[torch.Tensor] = None, glu: Optional[tuple] = None, gelu: bool = False):
    """The medium product with the fused decode product's conventions (EPILOGUE_STORE /
    ACCUMULATE / SWIGLU): returns the output, or for an accumulation with ``next_norm_weight``
    what the norm after it needs. ``glu`` (with EPILOGUE_SWIGLU): (limit, alpha, shift) of a gated
    unit with clamped halves instead of SwiGLU."""
    if _native is not None and _profiled is None and epilogue in (0, 1, 2) and (not gelu or (epilogue == EPILOGUE_STORE and (out_dtype or torch.bfloat16) == torch.bfloat16)):
        made = _native_product(True, a, w, w_tiled, bias, accumulate_into, epilogue,
                               torch.bfloat16 if epilogue == EPILOGUE_SWIGLU else torch.float32 if epilogue == EPILOGUE_ACCUMULATE else out_dtype or torch.bfloat16,
                               gelu, glu if epilogue == EPILOGUE_SWIGLU else None, next_norm_weight, next_one_centered, squares, eps)
        if made is not NotImplemented:
            return made
    _dev(a, w, bias, accumulate_into, squares, next_norm_weight)
    _want(a, torch.bfloat16, "a")
    _want(w, torch.bfloat16, "w")
    M, K = a.shape
    w_rows, w_k = w.shape
    kinds = 2 if epilogue == EPILOGUE_SWIGLU else 1
    if not 1 <= M <= MEDIUM_MAX_ROWS or w_k != K or w_rows % kinds or K % 8 or epilogue not in (0, 1, 2):
        raise KernelError(f"gemm_medium: a is {tuple(a.shape)}, w is {tuple(w.shape)}, epilogue {epilogue}")
    N = w_rows // kinds
    if bias is not None and (bias.dtype != torch.float32 or bias.shape != (w_rows,)):
        raise KernelError("gemm_medium: bias must be float32, one entry per row of w")
    if next_norm_weight is not None and (epilogue != EPILOGUE_ACCUMULATE or next_norm_weight.dtype != torch.float32
                                         or next_norm_weight.shape != (N,)):
        raise KernelError("gemm_medium: only the accumulating product prepares the next norm, whose weight is float32 [N]")
    if epilogue == EPILOGUE_ACCUMULATE:
        _want(accumulate_into, torch.float32, "accumulate_into")
        if accumulate_into.shape != (M, N):
            raise KernelError(f"gemm_medium: destination is {tuple(accumulate_into.shape)}, expected {(M, N)}")
        left = gemm_medium_into(a, w, bias, accumulate_into, F32, 1, N, next_norm_weight, next_one_centered, squares, eps, w_tiled=w_tiled)
        return accumulate_into if left is None else left
    out_dtype = torch.bfloat16 if epilogue == EPILOGUE_SWIGLU else (out_dtype or torch.bfloat16)
    out = torch.empty(M, N, dtype=out_dtype, device=a.device)
    if gelu and (epilogue != EPILOGUE_STORE or out_dtype != torch.bfloat16):
        raise KernelError("gemm_medium: gelu goes with a storing product of bfloat16")
    gemm_medium_into(a, w, bias, out, BF16_GELU if gelu else _code(out_dtype), epilogue, N, squares=squares, eps=eps, w_tiled=w_tiled, glu=glu)
    return out


def gemm_deep(a: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor] = None,
              out_dtype: Optional[torch.dtype] = None, accumulate_into: Optional[torch.Tensor] = None,
              columns: int = 128) -> torch.Tensor:
    """a [M, K] . w [N, K]^T (+ bias) on 128 x 128 tiles whose waves split K (fw_gemm_mfma_deep),
    whatever the dispatch of ``gemm`` would choose: bfloat16 operands, K a multiple of 64."""
    _dev(a, w, bias, accumulate_into)
    _want(a, torch.bfloat16, "a")
    _want(w, torch.bfloat16, "w")
    M, K = a.shape
    N = w.shape[0]
    if w.shape[1] != K or (bias is not None and (bias.dtype != torch.float32 or bias.shape != (N,))):
        raise KernelError(f"gemm_deep: a is {tuple(a.shape)}, w is {tuple(w.shape)}; bias is float32 [N]")
    if accumulate_into is not None:
        _want(accumulate_into, torch.float32, "accumulate_into")
        if accumulate_into.shape != (M, N):
            raise KernelError(f"gemm_deep: destination is {tuple(accumulate_into.shape)}, expected {(M, N)}")
        target, mode = accumulate_into, 1
    else:
        target, mode = torch.empty((M, N), dtype=out_dtype or a.dtype, device=a.device), 0
    _check(library().fw_gemm_mfma_deep(_p(a), _p(w), _p(bias), _p(target), _code(target.dtype), mode, M, N, K, int(columns), _stream()))
    return target


def _fast_ok(a: torch.Tensor, w: torch.Tensor) -> bool:
    return (a.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and a.shape[0] >= 1 and a.shape[1] % 8 == 0
            and a.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0)


# ---- dispatch: which kernel serves a call ------------------------------------------------
def gemm(a: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor] = None,
         out_dtype: Optional[torch.dtype] = None, accumulate_into: Optional[torch.Tensor] = None,
         w_tiled: Optional[torch.Tensor] = None, gelu: bool = False) -> torch.Tensor:
    """a [M, K] . w [N, K]^T (+ bias): bfloat16 operands go to the matrix-core kernels,
    everything else (float32, mixed) to the generic float32 one. ``w_tiled``: ``w`` once more in
    operand tiles (``tile_weights``), for the kernels of few rows that read it so. ``gelu``: the error-function gelu of
    the float32 sums, rounded once (the matrix-core products form it as they store)."""
    if gelu and accumulate_into is not None:
        raise KernelError("gemm: gelu goes with a product that stores")
    if _native is not None and _profiled is None and a.dtype == torch.bfloat16 and (not gelu or (out_dtype or a.dtype) == torch.bfloat16):
        made = _native_product(False, a, w, w_tiled, bias, accumulate_into, 0 if accumulate_into is None else 1,
                               out_dtype or a.dtype if accumulate_into is None else torch.float32, gelu)
        if made is not NotImplemented:
            return made
    if gelu and (not _fast_ok(a, w) or (out_dtype or a.dtype) != torch.bfloat16):
        return gelu_rows(gemm(a, w, bias, out_dtype=torch.float32, w_tiled=w_tiled), out_dtype or a.dtype)
    if not _fast_ok(a, w):
        return gemm_generic(a, w, bias, out_dtype=out_dtype, accumulate_into=accumulate_into)
    _dev(a, w, bias, accumulate_into)
    M, K = a.shape
    N, K2 = w.shape
    if K != K2:
        raise KernelError(f"gemm: a is {tuple(a.shape)} but w is {tuple(w.shape)}")
    if bias is not None and (bias.dtype != torch.float32 or bias.shape != (N,)):
        raise KernelError("gemm: bias must be float32 [N]")
    if accumulate_into is not None:
        _want(accumulate_into, torch.float32, "accumulate_into")
        if accumulate_into.shape != (M, N):
            raise KernelError(f"gemm: destination is {tuple(accumulate_into.shape)}, expected {(M, N)}")
        _fast_gemm(a, w, bias, accumulate_into, F32, 1, N, w_tiled)
        return accumulate_into
    out_dtype = out_dtype or a.dtype
    out = torch.empty((M, N), dtype=out_dtype, device=a.device)
    _fast_gemm(a, w, bias, out, BF16_GELU if gelu else _code(out_dtype), 0, N, w_tiled)
    return out


def gemm_swiglu(a: torch.Tensor, w_gate_up: torch.Tensor, w_tiled: Optional[torch.Tensor] = None, gelu: bool = False) -> torch.Tensor:
    """silu(a . gate^T) * (a . up^T) with w_gate_up = [gate rows; up rows]: [M, I] in a's dtype (``gelu``: the tanh form of gelu
    in place of silu).
    The activation is formed from the float32 sums inside the product's kernel; where the operands fit none of those the
    [M, 2I] intermediate is float32 and a second kernel forms it."""
    if _native is not None and _profiled is None and a.dtype == torch.bfloat16:
        made = _native_product(False, a, w_gate_up, w_tiled, None, None, 2, torch.bfloat16, glu=GEGLU if gelu else None)
        if made is not NotImplemented:
            return made
    rows2, K = w_gate_up.shape
    if rows2 % 2:
        raise KernelError("gemm_swiglu: the operand holds gate and up rows; their number must be even")
    if _fast_ok(a, w_gate_up):
        _dev(a, w_gate_up)
        if a.shape[1] != K:
            raise KernelError(f"gemm_swiglu: a is {tuple(a.shape)} but w is {tuple(w_gate_up.shape)}")
        out = torch.empty((a.shape[0], rows2 // 2), dtype=torch.bfloat16, device=a.device)
        _fast_gemm(a, w_gate_up, None, out, BF16_GEGLU if gelu else BF16, 2, rows2 // 2, w_tiled)
        return out
    if _float32_ok(a, w_gate_up) and not gelu:
        _dev(a, w_gate_up)
        if a.shape[1] != K:
            raise KernelError(f"gemm_swiglu: a is {tuple(a.shape)} but w is {tuple(w_gate_up.shape)}")
        out = torch.empty((a.shape[0], rows2 // 2), dtype=torch.float32, device=a.device)
        _check(library().fw_gemm_float32(_p(a), _p(w_gate_up), _p(None), _p(out), F32, 2, a.shape[0], rows2 // 2, K, _stream()))
        return out
    return swiglu(gemm_generic(a, w_gate_up, out_dtype=torch.float32), out_dtype=a.dtype, gelu=gelu)


# ---- fused products for decode steps of up to 16 rows --------------------------------------------
EPILOGUE_STORE, EPILOGUE_ACCUMULATE, EPILOGUE_SWIGLU, EPILOGUE_CONV = 0, 1, 2, 3


GEGLU = "gelu_tanh"       # in place of a clamped unit's three numbers
_SWIGLU = (0.0, 1.0, 0.0)


def _glu(glu):
    """The three numbers a gated epilogue takes: (0, 1, 0) is SwiGLU, (-1, 1, 0) the same around the tanh form of gelu
    (``GEGLU``); else (limit > 0, alpha, shift)."""
    if glu is None or glu == GEGLU:
        return float(0.0 if glu is None else -1.0), float(1.0), float(0.0)
    limit, alpha, shift = glu
    if not limit > 0:
        raise KernelError("a gated unit with clamped halves needs a positive limit")
    return float(limit), float(alpha), float(shift)
DECODE_MAX_ROWS = 16
LONG_K = 4096
LONG_K_TILED_ROWS = 8


def gemm_decode_fits(rows: int, features: int, k: int, epilogue: int) -> bool:
    return bool(library().fw_gemm_decode_fits(int(rows), int(features), int(k), int(epilogue)))


def gemm_decode(a: torch.Tensor, w: torch.Tensor, epilogue: int, *, bias: Optional[torch.Tensor] = None,
                norm_weight: Optional[torch.Tensor] = None, eps: float = 0.0, one_centered: bool = False,
                row_index: Optional[torch.Tensor] = None, out_dtype: Optional[torch.dtype] = None,
                accumulate_into: Optional[torch.Tensor] = None, taps: Optional[torch.Tensor] = None,
                conv_bias: Optional[torch.Tensor] = None, state: Optional[torch.Tensor] = None,
                seg_slot: Optional[torch.Tensor] = None, squares: Optional[torch.Tensor] = None,
                next_norm_weight: Optional[torch.Tensor] = None, next_one_centered: bool = False,
                w_tiled: Optional[torch.Tensor] = None, glu: Optional[tuple] = None, gelu: bool = False):
    """One kernel for (optional RMS norm of float32 rows) -> product with bfloat16 ``w`` -> epilogue.
    ``glu`` (with EPILOGUE_SWIGLU): (limit, alpha, shift) of a gated unit with clamped halves. ``gelu`` (EPILOGUE_STORE,
    bfloat16, no norm in front): the error-function gelu of the sums is stored.
    With ``norm_weight`` ``a`` holds float32 rows (gathered through ``row_index`` if given), else
    bfloat16 activations. With ``next_norm_weight`` the accumulating epilogue also leaves what
    the norm after it needs, and the call returns (activations x * w_next, sums of squares);
    a later call takes those as ``a`` and ``squares`` (with ``eps``) and skips the norm's
    arithmetic. See fw_gemm_decode in fw_kernels.h for the epilogues."""
    _dev(a, w, bias, norm_weight, row_index, accumulate_into, taps, conv_bias, state, seg_slot, squares, next_norm_weight)
    _want(w, torch.bfloat16, "w")
    normed = norm_weight is not None
    if squares is not None and (normed or squares.dtype != torch.float32 or squares.dim() != 2 or squares.shape[1] != 16
                                or not squares.is_contiguous()):
        raise KernelError("gemm_decode: sums of squares are float32 [tiles, 16] and replace the norm")
    rows = row_index.numel() if (normed and row_index is not None) else a.shape[0]
    K = a.shape[1]
    tiles = {EPILOGUE_SWIGLU: 2, EPILOGUE_CONV: 3}.get(epilogue, 1)
    if w.shape[1] != K or w.shape[0] % tiles:
        raise KernelError(f"gemm_decode: a is {tuple(a.shape)} but w is {tuple(w.shape)}")
    N = w.shape[0] // tiles
    if normed:
        _want(a, torch.float32, "a")
        _want(norm_weight, torch.float32, "norm_weight")
        if norm_weight.shape != (K,):
            raise KernelError("gemm_decode: the norm weight must be [K]")
        if row_index is not None:
            _want(row_index, torch.int32, "row_index")
    else:
        _want(a, torch.bfloat16, "a")
    if bias is not None and (bias.dtype != torch.float32 or bias.shape != (w.shape[0],)):
        raise KernelError("gemm_decode: bias must be float32, one entry per row of w")
    kernel_size = 0
    if epilogue == EPILOGUE_CONV:
        _want(taps, torch.float32, "taps")
        _want(state, torch.float32, "state")
        _want(seg_slot, torch.int32, "seg_slot")
        kernel_size = taps.shape[1]
        if taps.shape != (N, kernel_size) or state.dim() != 3 or state.shape[1:] != (N, kernel_size - 1):
            raise KernelError("gemm_decode: taps must be [N, L] and state [slots, N, L - 1]")
        if seg_slot.numel() < rows or (conv_bias is not None and conv_bias.shape != (N,)):
            raise KernelError("gemm_decode: seg_slot or the convolution bias has the wrong size")
    if epilogue == EPILOGUE_ACCUMULATE:
        _want(accumulate_into, torch.float32, "accumulate_into")
        if accumulate_into.shape != (rows, N):
            raise KernelError(f"gemm_decode: destination is {tuple(accumulate_into.shape)}, expected {(rows, N)}")
        target, out_dtype = accumulate_into, torch.float32
    else:
        out_dtype = out_dtype or torch.bfloat16
        target = torch.empty((rows, N), dtype=out_dtype, device=a.device)
    next_activations = next_squares = None
    if next_norm_weight is not None and (epilogue != EPILOGUE_ACCUMULATE or next_norm_weight.dtype != torch.float32
                                         or next_norm_weight.shape != (N,)):
        raise KernelError("gemm_decode: only the accumulating product prepares the next norm, whose weight is float32 [N]")
    if epilogue == EPILOGUE_ACCUMULATE and K >= LONG_K and N <= 4096 and not (w_tiled is not None and rows <= LONG_K_TILED_ROWS):
        # few features and a long K: the products of a few dozen rows (from operand tiles only beyond eight rows:
        # 2,048 features over K 8,192 at 8 rows 11.8 us on this one, at 12 / 16 rows 14.1 / 14.7 against 11.8 / 11.7)
        left = gemm_medium_into(a, w, bias, target, F32, 1, N, next_norm_weight, next_one_centered, w_tiled=w_tiled)
        return target if left is None else left
    if next_norm_weight is not None:
        next_activations = torch.empty((rows, N), dtype=torch.bfloat16, device=a.device)
        next_squares = torch.empty((library().fw_gemm_decode_accumulate_tiles(N), 16), dtype=torch.float32, device=a.device)
    prologue = 1 if normed else (2 if squares is not None else 0)
    if gelu and (epilogue != EPILOGUE_STORE or out_dtype != torch.bfloat16 or prologue):
        raise KernelError("gemm_decode: gelu goes with a plain storing product of bfloat16")
    w_tiled = _tiled_for(w, w_tiled)
    _check(library().fw_gemm_decode(
        prologue, _p(a), _p(norm_weight), _p(row_index), float(eps), int(one_centered),
        _p(w if w_tiled is None else w_tiled), int(w_tiled is not None), _p(bias),
        _p(target), BF16_GELU if gelu else _code(out_dtype), int(epilogue), rows, N, K, _p(taps), _p(conv_bias), _p(state), _p(seg_slot),
        int(kernel_size), _p(next_norm_weight), int(next_one_centered), _p(next_activations), _p(next_squares),
        _p(squares), 0 if squares is None else squares.shape[0], *_glu(glu), _stream()))
    if next_norm_weight is not None:
        return next_activations, next_squares
    return target


DECODE_SPLIT_PAGES = 4


QUERY_TILE = 64


def query_tiles(seg_row0):
    """Cuts the rows of each segment into tiles of up to 64 that never span two segments:
    (segment of each tile, first row of each tile), as lists."""
    tile_seg, tile_row0 = [], []
    for seg in range(len(seg_row0) - 1):
        for row in range(seg_row0[seg], seg_row0[seg + 1], QUERY_TILE):
            tile_seg.append(seg)
            tile_row0.append(row)
    return tile_seg, tile_row0


def decode_splits(max_context: int, window: int = 0, chunk: int = 0, keep_first: int = 0) -> int:
    """Into how many workgroups at most the keys that a row sees are cut: runs of 4 pages."""
    blocks = (max_context + PAGE_SIZE - 1) // PAGE_SIZE
    span = min((n for n in (window, chunk) if n > 0), default=0)     # the most keys a row sees, where bounded
    if span > 0:
        blocks = min(blocks, (span + PAGE_SIZE - 2) // PAGE_SIZE + 1 + (keep_first + PAGE_SIZE - 1) // PAGE_SIZE)
    return max(1, (blocks + DECODE_SPLIT_PAGES - 1) // DECODE_SPLIT_PAGES)


def attention_prefill(q: torch.Tensor, num_heads: int, num_kv_heads: int, head_dim: int, k_pages: torch.Tensor,
                      v_pages: torch.Tensor, block_table: torch.Tensor, tile_seg: torch.Tensor, tile_row0: torch.Tensor,
                      seg_row0: torch.Tensor, row_pos: torch.Tensor, scale: float, window: int = 0,
                      heads_together: int = 0, out: Optional[torch.Tensor] = None, v_dim: Optional[int] = None,
                      chunk: int = 0, softcap: float = 0.0, keep_first: int = 0, sinks: Optional[torch.Tensor] = None,
                      slopes: Optional[torch.Tensor] = None, halves: bool = False, paired: bool = False) -> torch.Tensor:
    """``heads_together``: query heads of a kv group per workgroup (0 and 1: one; 4 up to head_dim 64). ``halves`` (up
    to head_dim 64): two heads per workgroup, whose two halves share a tile's pages out and merge. ``paired`` (head_dim and v_dim both
    64 or both 128, an even number of heads a group): two heads per workgroup, whose loop has three pages in flight; with ``halves`` or without. Only the rows of the given tiles are written (into ``out`` if given)."""
    if _native is not None and _profiled is None and out is None and q.is_cuda:
        made = _native.prefill(q, num_heads, num_kv_heads, head_dim, k_pages, v_pages, block_table, tile_seg, tile_row0, seg_row0, row_pos, scale, window, heads_together,
                               head_dim if v_dim is None else v_dim, chunk, softcap, keep_first, sinks, slopes, (1 if halves else 0) + (2 if paired else 0), PAGE_SIZE,
                               _stream())
        if made is not NotImplemented:
            return made
    _dev(q, k_pages, v_pages, block_table, tile_seg, tile_row0, seg_row0, row_pos)
    _want(q, torch.bfloat16, "q")
    rows = q.shape[0]
    v_dim = head_dim if v_dim is None else int(v_dim)
    if q.shape != (rows, num_heads * head_dim):
        raise KernelError(f"attention: q is {tuple(q.shape)}, expected {(rows, num_heads * head_dim)}")
    pages = _check_pages(k_pages, v_pages, num_kv_heads, head_dim, torch.bfloat16, v_dim)
    for name, t in (("block_table", block_table), ("tile_seg", tile_seg), ("tile_row0", tile_row0),
                    ("seg_row0", seg_row0), ("row_pos", row_pos)):
        _want(t, torch.int32, name)
    if block_table.dim() != 2 or row_pos.numel() < rows or tile_seg.numel() != tile_row0.numel():
        raise KernelError("attention: batch index arrays are inconsistent")
    if out is None:
        out = torch.empty((rows, num_heads * v_dim), dtype=q.dtype, device=q.device)
    elif out.shape != (rows, num_heads * v_dim) or out.dtype != q.dtype or not out.is_contiguous():
        raise KernelError("attention: out must be bfloat16 [rows, heads * v_dim]")
    _check(library().fw_attention_prefill(
        _p(q), _p(out), _p(k_pages), _p(v_pages), _p(block_table), block_table.shape[1], _p(tile_seg), _p(tile_row0),
        tile_seg.numel(), _p(seg_row0), _p(row_pos), rows, num_heads, num_kv_heads, head_dim, v_dim, float(scale),
        int(window), int(chunk), float(softcap), *_sinks(sinks, num_heads, keep_first, window, chunk, slopes), PAGE_SIZE, pages,
        int(heads_together), int(halves) + (2 if paired else 0), _stream()))
    return out


def _work(decode_work: Optional[torch.Tensor]):
    if decode_work is not None:
        _dev(decode_work)
        _want(decode_work, torch.int32, "decode_work")
        if decode_work.numel() < 1:
            raise KernelError("attention_decode: decode_work holds one int32")
    return _p(decode_work)


def attention_decode(q: torch.Tensor, num_heads: int, num_kv_heads: int, head_dim: int, k_pages: torch.Tensor,
                     v_pages: torch.Tensor, block_table: torch.Tensor, row_seg: torch.Tensor, row_pos: torch.Tensor,
                     scale: float, max_context: int, window: int = 0, out: Optional[torch.Tensor] = None,
                     decode_work: Optional[torch.Tensor] = None, v_dim: Optional[int] = None, chunk: int = 0,
                     softcap: float = 0.0, keep_first: int = 0, sinks: Optional[torch.Tensor] = None,
                      slopes: Optional[torch.Tensor] = None) -> torch.Tensor:
    """One row per request; ``max_context`` bounds position + 1 of every row (the host knows it).
    ``decode_work``: one int32 on the device, the runs of 4 pages that the rows see together (the
    sum of ceil((position + 1) / 256)), or, where the rows are equally long, those of the longest as a negative number: the kernel shares
    the work out by it (fewer, longer workgroups once there are more runs than about as many as compute units); without it, one
    run per workgroup."""
    _dev(q, k_pages, v_pages, block_table, row_seg, row_pos)
    _want(q, torch.bfloat16, "q")
    rows = q.shape[0]
    v_dim = head_dim if v_dim is None else int(v_dim)
    if q.shape != (rows, num_heads * head_dim):
        raise KernelError(f"attention: q is {tuple(q.shape)}, expected {(rows, num_heads * head_dim)}")
    pages = _check_pages(k_pages, v_pages, num_kv_heads, head_dim, torch.bfloat16, v_dim)
    for name, t in (("block_table", block_table), ("row_seg", row_seg), ("row_pos", row_pos)):
        _want(t, torch.int32, name)
    if block_table.dim() != 2 or row_seg.numel() < rows or row_pos.numel() < rows:
        raise KernelError("attention: batch index arrays are too short")
    keep_first, sinks_at, slopes_at = _sinks(sinks, num_heads, keep_first, window, chunk, slopes)
    splits = decode_splits(max_context, window, chunk, keep_first)
    partial = torch.empty((rows, num_heads, splits, v_dim + 4), dtype=torch.float32, device=q.device)
    if out is None:
        out = torch.empty((rows, num_heads * v_dim), dtype=q.dtype, device=q.device)
    elif out.shape != (rows, num_heads * v_dim) or out.dtype != q.dtype or not out.is_contiguous():
        raise KernelError("attention: out must be bfloat16 [rows, heads * v_dim]")
    group = num_heads // num_kv_heads
    tickets = _medium_counters(q.device, rows * num_kv_heads * ((group + 15) // 16))
    _check(library().fw_attention_decode(
        _p(q), _p(out), _p(partial), splits, int(max_context), _work(decode_work), _p(tickets), tickets.numel(), _p(k_pages), _p(v_pages),
        _p(block_table),
        block_table.shape[1], _p(row_seg), _p(row_pos), rows, num_heads, num_kv_heads, head_dim, v_dim, float(scale),
        int(window), int(chunk), float(softcap), keep_first, sinks_at, slopes_at, PAGE_SIZE, pages, _stream()))
    return out


def attention_decode_fused(qkv: torch.Tensor, num_heads: int, num_kv_heads: int, head_dim: int,
                           q_norm_weight: Optional[torch.Tensor], k_norm_weight: Optional[torch.Tensor], eps: float,
                           cos: Optional[torch.Tensor], sin: Optional[torch.Tensor], rotary_dim: int, k_pages: torch.Tensor,
                           v_pages: torch.Tensor, block_table: torch.Tensor, row_seg: torch.Tensor, row_pos: torch.Tensor,
                           scale: float, max_context: int, window: int = 0, write_kv: bool = True,
                           decode_work: Optional[torch.Tensor] = None, v_dim: Optional[int] = None, chunk: int = 0,
                           softcap: float = 0.0, interleaved: bool = False, q_only: bool = False, keep_first: int = 0,
                           sinks: Optional[torch.Tensor] = None, slopes: Optional[torch.Tensor] = None,
                           q_row_scale: Optional[torch.Tensor] = None) -> torch.Tensor:
    """One row per request, from the step's raw projections ``qkv`` (float32 [rows, (heads + 2 kv
    heads) * head_dim]): per-head norm and rotation of queries and keys, the new keys and values
    into their pages, and the split-key attention, in one kernel. Returns bfloat16 [rows, heads *
    head_dim]; the same numbers as ``qk_norm_rope_kv_write`` followed by ``attention_decode``."""
    _dev(qkv, q_norm_weight, k_norm_weight, cos, sin, k_pages, v_pages, block_table, row_seg, row_pos)
    _want(qkv, torch.float32, "qkv")
    rows, width = qkv.shape
    v_dim = head_dim if v_dim is None else int(v_dim)
    expected = num_heads * head_dim if q_only else (num_heads + num_kv_heads) * head_dim + num_kv_heads * v_dim
    if width != expected or (q_only and write_kv):
        raise KernelError(f"attention_decode_fused: qkv width {width} != {expected} (queries alone: {q_only}; they bring nothing to store)")
    pages = _check_pages(k_pages, v_pages, num_kv_heads, head_dim, torch.bfloat16, v_dim)
    for w in (q_norm_weight, k_norm_weight):
        if w is not None:
            _want(w, torch.float32, "norm weight")
            if w.shape != (head_dim,):
                raise KernelError("attention_decode_fused: a head norm weight must be [head_dim]")
    if rotary_dim:
        for t in (cos, sin):
            _want(t, torch.float32, "rotation table")
            if t.shape != (rows, rotary_dim // 2):
                raise KernelError(f"attention_decode_fused: rotation table is {tuple(t.shape)}, expected {(rows, rotary_dim // 2)}")
    for name, t in (("block_table", block_table), ("row_seg", row_seg), ("row_pos", row_pos)):
        _want(t, torch.int32, name)
    if block_table.dim() != 2 or row_seg.numel() < rows or row_pos.numel() < rows:
        raise KernelError("attention: batch index arrays are too short")
    keep_first, sinks_at, slopes_at = _sinks(sinks, num_heads, keep_first, window, chunk, slopes)
    splits = decode_splits(max_context, window, chunk, keep_first)
    partial = torch.empty((rows, num_heads, splits, v_dim + 4), dtype=torch.float32, device=qkv.device)
    out = torch.empty((rows, num_heads * v_dim), dtype=torch.bfloat16, device=qkv.device)
    group = num_heads // num_kv_heads
    tickets = _medium_counters(qkv.device, rows * num_kv_heads * ((group + 15) // 16))
    _row_scale(q_row_scale, rows)
    _check(library().fw_attention_decode_fused(
        _p(qkv), _p(q_norm_weight), _p(k_norm_weight), float(eps), _p(cos), _p(sin), int(rotary_dim), int(write_kv), _p(out),
        _p(partial), splits, int(max_context), _work(decode_work), _p(tickets), tickets.numel(), _p(k_pages), _p(v_pages), _p(block_table),
        block_table.shape[1], _p(row_seg), _p(row_pos), rows, num_heads, num_kv_heads, head_dim, v_dim, float(scale), int(window),
        int(chunk), float(softcap), int(interleaved), int(q_only), keep_first, sinks_at, slopes_at, _p(q_row_scale), PAGE_SIZE, pages,
        _stream()))
    return out


def attention_is_tiled(head_dim: int) -> bool:
    """Whether bfloat16 attention with this head size runs on the matrix-core kernels (which
    work on tiles of QUERY_TILE rows)."""
    return head_dim % 16 == 0 and 16 <= head_dim <= MAX_HEAD_DIM


def prompt_halves(tiles: int, num_heads: int, num_kv_heads: int, widest: int, keys: int) -> bool:
    """Whether a prompt's attention takes the form of two heads a workgroup (fw_attention_prefill), whose two halves share the
    pages out: ``tiles`` tiles of rows, of which the rows see up to ``keys`` keys, heads of up to ``widest`` channels.
    It is asked where the heads of a group are not taken two by two (``prompt_pairs``): heads of 48 channels, or keys and values of 48 and 64.
    Its workgroups have a compute unit each, those of the form of one head share one by two to four. So it pays where
    its rounds over the chip are full, and where rows see enough keys for the merge at the end to be little. us, one head /
    halves, heads of 48: 32 heads in 8 groups, 2,048 rows (2 rounds) behind 0 / 2,048 / 30,720 keys 53.5 / 54.1, 120 / 109, 1,050 /
    850; 1,500 rows (1.5 rounds) behind 3,072 100 / 121; 1,700 (1.7) behind 2,048 108 / 100; 777 (0.8) behind 0 / 512 19.5 / 19.5,
    27.6 / 26.7; 6,000 (5.9) behind 4,096 642 / 642, 3,500 (3.4) 333 / 345; 16 heads in 8 groups, 777 rows (0.4) behind 2,048 45.0 /
    45.7, 2,048 rows (1) behind 0 / 30,720 38.1 / 35.1, 544 / 438; keys of 64 and values of 48, 32 heads, 2,048 rows behind 0 / 2,048 53.1 /
    54.2, 119 / 109, 6,000 behind 4,096 639 / 647; keys of 48 and values of 64, 16 heads, 2,048 rows behind 2,048 76 / 64. Over 52 such prompts
    the rule's choice takes 0.1 % more than the better one. With an odd number of heads a group one wave
    in so many idles (24 in 8 groups of 64 channels, 2,048 rows behind 8,192 223 / 267), and heads of 32 channels leave LDS less to bound
    (2,048 rows behind 8,192 188 / 213)."""
    group = num_heads // num_kv_heads
    if not 32 < widest <= 64 or group % 2:
        return False
    workgroups = tiles * num_kv_heads * (group // 2)
    rounds = -(-workgroups // COMPUTE_UNITS)
    if 2 * workgroups <= COMPUTE_UNITS:
        return keys >= 16384
    fill, least = ((0.5, 1280), (0.84, 1280), (0.95, 3072))[min(rounds, 3) - 1]
    return workgroups >= fill * rounds * COMPUTE_UNITS and keys >= least


# us of the paired form: a workgroup of four waves per page while it has a compute unit to itself, while two share one, and of many in line for
# two places a unit; eight waves per page; start, end (and merge) of either
_PAIRED = {64: (0.93, 1.2, 1.32, 0.73, 4.0, 7.0), 128: (1.6, 2.2, 2.4, 1.09, 4.0, 8.5)}


def prompt_pairs(tiles: int, num_heads: int, num_kv_heads: int, head_dim: int, v_dim: int, keys: int, context: int):
    """Whether a prompt's attention takes the heads of a group two by two (fw_attention_prefill), and if so whether in halves: None, False or True.
    ``tiles`` tiles of rows, of which the rows see up to ``keys`` keys, the last of them ``context`` if no window held it. It does where its kernel is built (heads of 64 or 128 channels, an even number a
    group); with heads of 64 from 640 keys on: in front of that its two operands in flight have no page to hide behind (us, one head a workgroup / two by two:
    37 rows 6.4 / 7.0, 300 9.9 / 10.8, 500 12.9 / 13.7, 777 17.4 / 16.6, 2,048 45 / 39, behind 2,048 keys 104 / 85, 16 heads behind 30,720 442 / 359).
    Heads of 128: 16 in 4 groups, 37 rows 8.9 / 8.8, 1,111 rows 36.5 / 27.2, 2,048 44.7 / 29.0 with a window of 1,024, behind 4,096 keys 187 / 104.
    Eight waves a workgroup (halves) or four by the estimated time of either: pages of a tile run from what the last tile sees down to what the first one does;
    the longest workgroup, or all of them over the places there are, or two rounds in line (us, four / eight: 32 heads, 777 rows 18.6 / 17.6, 1,500
    30.7 / 27.5, 3,000 65 / 78, 1,300 behind 2,048 66 / 71; 16 heads, 4,096 rows 71 / 64, 2,048 behind 30,720 462 / 359)."""
    group = num_heads // num_kv_heads
    if head_dim != v_dim or head_dim not in _PAIRED or group % 2 or tiles < 1 or (head_dim == 64 and keys < 640):
        return None
    alone, shared, many, eight, start, start_eight = _PAIRED[head_dim]
    workgroups = tiles * num_kv_heads * (group // 2)
    longest, last = -(-keys // 64), -(-context // 64)
    full = min(tiles, max(1, last - longest + 1))           # tiles that see as much as the last one does; a page less each from there on
    least = max(1, longest - (tiles - full))
    total = (full * longest + (tiles - full) * (longest - 1 + least) / 2) * (workgroups // tiles)
    four = start + max(longest * (alone if workgroups <= COMPUTE_UNITS else shared), total * many / (2 * COMPUTE_UNITS) if workgroups > 2 * COMPUTE_UNITS else 0.0)
    rounds = -(-workgroups // COMPUTE_UNITS)
    halves = start_eight + longest * eight
    if rounds == 2:         # the workgroup that ends its round first, and the first of the next
        halves = max(halves, 2 * (start_eight + eight * max(least, min(longest, longest + full - tiles * COMPUTE_UNITS / workgroups))))
    elif rounds > 2:
        halves = max(halves, rounds * start_eight + total * eight / COMPUTE_UNITS)
    return halves < four


def attention(q: torch.Tensor, num_heads: int, num_kv_heads: int, head_dim: int, k_pages: torch.Tensor,
              v_pages: torch.Tensor, block_table: torch.Tensor, ctx, scale: float, window: int = 0,
              tile_seg: Optional[torch.Tensor] = None, tile_row0: Optional[torch.Tensor] = None,
              decode_work: Optional[torch.Tensor] = None, v_dim: Optional[int] = None, chunk: int = 0,
              softcap: float = 0.0, keep_first: int = 0, sinks: Optional[torch.Tensor] = None,
                      slopes: Optional[torch.Tensor] = None) -> torch.Tensor:
    """bfloat16 with a head size in steps of 16 runs on the matrix cores: the split-key decode
    kernel for segments of one row (all of them, or those a mixed step begins with: a single row
    would hold a 64-row tile of the prompt kernel and walk its whole context alone), the tiled
    kernel for the rest (``tile_seg``, ``tile_row0``: the tiles of ``query_tiles`` in the order
    workgroups take them, those of the leading single rows in front; ``decode_work``: see
    ``attention_decode``); float32 and everything else on the generic kernel. ``v_dim``: the size of a
    value head (and of a head's output) where it is not ``head_dim``."""
    v_dim = head_dim if v_dim is None else int(v_dim)
    fast = q.dtype == torch.bfloat16 and attention_is_tiled(head_dim) and attention_is_tiled(v_dim)
    if fast and ctx.all_decode:
        return attention_decode(q, num_heads, num_kv_heads, head_dim, k_pages, v_pages, block_table, ctx.row_seg,
                                ctx.row_pos, scale, ctx.max_context, window, decode_work=decode_work, v_dim=v_dim,
                                chunk=chunk, softcap=softcap, keep_first=keep_first, sinks=sinks, slopes=slopes)
    if fast:
        if tile_seg is None or tile_row0 is None:
            raise KernelError("attention: the tiled kernel needs the step's query tiles")
        single = getattr(ctx, "decode_prefix", 0)       # leading segments of one row: rows and tiles 0 .. single - 1
        lengths = getattr(ctx, "new_lengths", None)     # what each segment sees in the end; the single rows' contexts are not the tiles'
        keys = min([n for n in (window, chunk) if n] + [max(lengths[single:]) if lengths else ctx.max_context])
        context = max(lengths[single:]) if lengths else ctx.max_context
        halves = prompt_pairs(tile_seg.numel() - single, num_heads, num_kv_heads, head_dim, v_dim, keys, context)
        paired = halves is not None
        if not paired:
            halves = prompt_halves(tile_seg.numel() - single, num_heads, num_kv_heads, max(head_dim, v_dim), keys)
        if single == 0:
            return attention_prefill(q, num_heads, num_kv_heads, head_dim, k_pages, v_pages, block_table, tile_seg,
                                     tile_row0, ctx.seg_row0, ctx.row_pos, scale, window, halves=halves, paired=paired, v_dim=v_dim,
                                     chunk=chunk, softcap=softcap, keep_first=keep_first, sinks=sinks, slopes=slopes)
        out = torch.empty((q.shape[0], num_heads * v_dim), dtype=q.dtype, device=q.device)
        attention_decode(q[:single], num_heads, num_kv_heads, head_dim, k_pages, v_pages, block_table, ctx.row_seg,
                         ctx.row_pos, scale, ctx.max_context, window, out=out[:single], decode_work=decode_work, v_dim=v_dim,
                         chunk=chunk, softcap=softcap, keep_first=keep_first, sinks=sinks, slopes=slopes)
        return attention_prefill(q, num_heads, num_kv_heads, head_dim, k_pages, v_pages, block_table,
                                 tile_seg[single:], tile_row0[single:], ctx.seg_row0, ctx.row_pos, scale, window,
                                 halves=halves, paired=paired, out=out, v_dim=v_dim, chunk=chunk, softcap=softcap,
                                 keep_first=keep_first, sinks=sinks, slopes=slopes)
    return attention_generic(q, num_heads, num_kv_heads, head_dim, k_pages, v_pages, block_table, ctx.row_seg,
                             ctx.row_pos, scale, window, v_dim=v_dim, chunk=chunk, softcap=softcap, keep_first=keep_first, sinks=sinks, slopes=slopes)


# ---- attention whose weights are sigmoids and whose heads mix them ------------------------------------------
SIGMOID_MAX_HEADS = 256         # of the plain kernel (the matrix-core kernels: see sigmoid_attention_is_tiled)
SIGMOID_DECODE_WORKGROUPS = 256     # one per compute unit: up to here every page of a row gets a workgroup of its own


def sigmoid_attention_is_tiled(num_heads: int, head_dim: int, v_dim: int) -> bool:
    """Whether bfloat16 runs on the matrix-core kernels: up to 16 heads, sizes in steps of 16, all heads of 16 rows in LDS."""
    return bool(library().fw_sigmoid_attention_fits(int(num_heads), int(head_dim), int(v_dim)))


def _sigmoid_checks(num_heads: int, num_kv_heads: int, head_dim: int, v_dim: int, k_pages: torch.Tensor, v_pages: torch.Tensor,
                    block_table: torch.Tensor, row_seg: Optional[torch.Tensor], row_pos: torch.Tensor, rows: int, bias: torch.Tensor,
                    mix: torch.Tensor, gate: Optional[torch.Tensor]):
    _dev(k_pages, v_pages, block_table, row_seg, row_pos, bias, mix)
    pages = _check_pages(k_pages, v_pages, num_kv_heads, head_dim, k_pages.dtype, v_dim)
    for name, t in (("block_table", block_table), ("row_seg", row_seg), ("row_pos", row_pos)):
        if t is not None:
            _want(t, torch.int32, name)
    if block_table.dim() != 2 or (row_seg is not None and row_seg.numel() < rows) or row_pos.numel() < rows:
        raise KernelError("sigmoid_attention: batch index arrays are too short")
    for name, t, shape in (("bias", bias, (num_heads,)), ("mix", mix, (num_heads, num_heads))):
        _want(t, torch.float32, name)
        if t.shape != shape:
            raise KernelError(f"sigmoid_attention: {name} is {tuple(t.shape)}, expected {shape}")
    if gate is not None:
        _dev_rows(gate, "gate")
        if gate.dtype != torch.float32 or gate.shape != (rows, num_heads * v_dim):
            raise KernelError(f"sigmoid_attention: the gate is {tuple(gate.shape)} {gate.dtype}, expected {(rows, num_heads * v_dim)} float32")
    return pages


def sigmoid_attention_generic(q: torch.Tensor, num_heads: int, num_kv_heads: int, head_dim: int, v_dim: int, k_pages: torch.Tensor,
                              v_pages: torch.Tensor, block_table: torch.Tensor, row_seg: torch.Tensor, row_pos: torch.Tensor,
                              scale: float, window: int, bias: torch.Tensor, mix: torch.Tensor,
                              gate: Optional[torch.Tensor] = None) -> torch.Tensor:
    """a_g = sigmoid(q_g . k * scale + bias[g]) over the visible keys, heads mixed by ``mix`` [heads, heads], the weighted
    sums of the values times sigmoid(``gate``) (float32 [rows, heads * v_dim], rows may lie apart; None: no gate)."""
    rows = q.shape[0]
    _dev(q)
    if q.shape != (rows, num_heads * head_dim) or q.dtype != k_pages.dtype:
        raise KernelError(f"sigmoid_attention: q is {tuple(q.shape)} {q.dtype}, expected {(rows, num_heads * head_dim)} {k_pages.dtype}")
    pages = _sigmoid_checks(num_heads, num_kv_heads, head_dim, v_dim, k_pages, v_pages, block_table, row_seg, row_pos, rows, bias, mix, gate)
    out = torch.empty((rows, num_heads * v_dim), dtype=q.dtype, device=q.device)
    _check(library().fw_sigmoid_attention_generic(
        _p(q), _p(out), _code(q.dtype), _p(k_pages), _p(v_pages), _p(block_table), block_table.shape[1], _p(row_seg), _p(row_pos), rows,
        num_heads, num_kv_heads, head_dim, v_dim, float(scale), int(window), _p(bias), _p(mix), _p(gate),
        _stride(gate) if gate is not None else 0, PAGE_SIZE, pages, _stream()))
    return out


def sigmoid_attention_prefill(q: torch.Tensor, num_heads: int, num_kv_heads: int, head_dim: int, v_dim: int, k_pages: torch.Tensor,
                              v_pages: torch.Tensor, block_table: torch.Tensor, tile_seg: torch.Tensor, tile_row0: torch.Tensor,
                              seg_row0: torch.Tensor, row_pos: torch.Tensor, scale: float, window: int, bias: torch.Tensor,
                              mix: torch.Tensor, gate: Optional[torch.Tensor] = None, out: Optional[torch.Tensor] = None,
                              max_context: int = 0, parts: int = 0) -> torch.Tensor:
    """The same on the matrix cores for the rows of the given tiles (of up to 64 rows; ``attention_prefill``).
    ``max_context`` bounds position + 1 of every row (0: what the block table holds). ``parts``: workgroups that share the keys of
    16 rows (0: as many as fill the chip)."""
    rows = q.shape[0]
    _dev(q, tile_seg, tile_row0, seg_row0)
    _want(q, torch.bfloat16, "q")
    for name, t in (("tile_seg", tile_seg), ("tile_row0", tile_row0), ("seg_row0", seg_row0)):
        _want(t, torch.int32, name)
    if q.shape != (rows, num_heads * head_dim) or k_pages.dtype != torch.bfloat16 or tile_seg.numel() != tile_row0.numel():
        raise KernelError(f"sigmoid_attention: q is {tuple(q.shape)}, pages {k_pages.dtype}, {tile_seg.numel()} / {tile_row0.numel()} tiles")
    pages = _sigmoid_checks(num_heads, num_kv_heads, head_dim, v_dim, k_pages, v_pages, block_table, None, row_pos, rows, bias, mix, gate)
    if out is None:
        out = torch.empty((rows, num_heads * v_dim), dtype=q.dtype, device=q.device)
    elif out.shape != (rows, num_heads * v_dim) or out.dtype != q.dtype or not out.is_contiguous():
        raise KernelError("sigmoid_attention: out must be bfloat16 [rows, heads * v_dim]")
    floats, counters = ctypes.c_longlong(0), ctypes.c_int(0)
    parts = library().fw_sigmoid_attention_prefill_plan(tile_seg.numel(), num_heads, head_dim, v_dim, int(window),
                                                        int(max_context) or block_table.shape[1] * PAGE_SIZE, int(parts),
                                                        ctypes.byref(floats), ctypes.byref(counters))
    partial = torch.empty((floats.value,), dtype=torch.float32, device=q.device) if parts > 1 else None
    tickets = _medium_counters(q.device, counters.value)
    _check(library().fw_sigmoid_attention_prefill(
        _p(q), _p(out), _p(partial), int(floats.value), _p(tickets), tickets.numel(), parts, _p(k_pages), _p(v_pages), _p(block_table), block_table.shape[1], _p(tile_seg), _p(tile_row0), tile_seg.numel(),
        _p(seg_row0), _p(row_pos), rows, num_heads, num_kv_heads, head_dim, v_dim, float(scale), int(window), _p(bias), _p(mix),
        _p(gate), _stride(gate) if gate is not None else 0, PAGE_SIZE, pages, _stream()))
    return out


def sigmoid_decode_splits(rows: int, max_context: int, window: int):
    """(workgroups a row's visible pages are cut into at most, pages each of them takes)."""
    blocks = (max_context + PAGE_SIZE - 1) // PAGE_SIZE
    if window > 0:
        blocks = min(blocks, (window + PAGE_SIZE - 2) // PAGE_SIZE + 1)
    each = max(1, rows * blocks // SIGMOID_DECODE_WORKGROUPS)
    return (blocks + each - 1) // each, each


def sigmoid_attention_decode(num_heads: int, num_kv_heads: int, head_dim: int, v_dim: int, k_pages: torch.Tensor, v_pages: torch.Tensor,
                             block_table: torch.Tensor, row_seg: torch.Tensor, row_pos: torch.Tensor, scale: float, window: int,
                             bias: torch.Tensor, mix: torch.Tensor, max_context: int, gate: Optional[torch.Tensor] = None,
                             q: Optional[torch.Tensor] = None, qkv: Optional[torch.Tensor] = None, qk_norm: bool = True, eps: float = 0.0,
                             write_kv: bool = True, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """One row per request on the matrix cores; ``max_context`` bounds position + 1 of every row. From finished queries
    ``q`` (bfloat16), or from the raw projections ``qkv`` (float32 [rows, q | k | v], rows may lie apart): queries and keys of a
    head divided by their root mean square (``qk_norm``, ``eps``) and the new keys and values stored (``write_kv``) in the same
    kernel."""
    if (q is None) == (qkv is None):
        raise KernelError("sigmoid_attention: finished queries or raw projections, one of the two")
    rows = (q if q is not None else qkv).shape[0]
    if q is not None:
        _dev(q)
        _want(q, torch.bfloat16, "q")
        if q.shape != (rows, num_heads * head_dim):
            raise KernelError(f"sigmoid_attention: q is {tuple(q.shape)}, expected {(rows, num_heads * head_dim)}")
    else:
        _dev_rows(qkv, "qkv")
        _want(qkv, torch.float32, "qkv")
        expected = (num_heads + num_kv_heads) * head_dim + num_kv_heads * v_dim
        if qkv.shape != (rows, expected):
            raise KernelError(f"sigmoid_attention: qkv is {tuple(qkv.shape)}, expected {(rows, expected)}")
    if k_pages.dtype != torch.bfloat16:
        raise KernelError("sigmoid_attention: the matrix-core kernels work on a bfloat16 cache")
    pages = _sigmoid_checks(num_heads, num_kv_heads, head_dim, v_dim, k_pages, v_pages, block_table, row_seg, row_pos, rows, bias, mix, gate)
    splits, each = sigmoid_decode_splits(rows, max_context, window)
    partial = torch.empty((rows, splits, num_heads * v_dim), dtype=torch.float32, device=k_pages.device) if splits > 1 else None
    tickets = _medium_counters(k_pages.device, rows)
    if out is None:
        out = torch.empty((rows, num_heads * v_dim), dtype=torch.bfloat16, device=k_pages.device)
    elif out.shape != (rows, num_heads * v_dim) or out.dtype != torch.bfloat16 or not out.is_contiguous():
        raise KernelError("sigmoid_attention: out must be bfloat16 [rows, heads * v_dim]")
    _check(library().fw_sigmoid_attention_decode(
        _p(q), _p(qkv), _stride(qkv) if qkv is not None else 0, int(qk_norm), float(eps), int(write_kv), _p(out), _p(partial), splits,
        each, int(max_context), _p(tickets), tickets.numel(), _p(k_pages), _p(v_pages), _p(block_table), block_table.shape[1], _p(row_seg),
        _p(row_pos), rows, num_heads, num_kv_heads, head_dim, v_dim, float(scale), int(window), _p(bias), _p(mix), _p(gate),
        _stride(gate) if gate is not None else 0, PAGE_SIZE, pages, _stream()))
    return out


def sigmoid_attention(q: torch.Tensor, num_heads: int, num_kv_heads: int, head_dim: int, v_dim: int, k_pages: torch.Tensor,
                      v_pages: torch.Tensor, block_table: torch.Tensor, ctx, scale: float, window: int, bias: torch.Tensor,
                      mix: torch.Tensor, gate: Optional[torch.Tensor] = None, tile_seg: Optional[torch.Tensor] = None,
                      tile_row0: Optional[torch.Tensor] = None) -> torch.Tensor:
    """The step's rows: bfloat16 in sizes the matrix-core kernels take goes to the decode kernel for segments of one row
    (all of them, or those a mixed step begins with) and to the tiled kernel for the rest; everything else to the plain one."""
    if q.dtype != torch.bfloat16 or not sigmoid_attention_is_tiled(num_heads, head_dim, v_dim):
        return sigmoid_attention_generic(q, num_heads, num_kv_heads, head_dim, v_dim, k_pages, v_pages, block_table, ctx.row_seg, ctx.row_pos,
                                         scale, window, bias, mix, gate)
    rows = q.shape[0]
    single = rows if ctx.all_decode else getattr(ctx, "decode_prefix", 0)
    out = torch.empty((rows, num_heads * v_dim), dtype=q.dtype, device=q.device)
    if single:
        sigmoid_attention_decode(num_heads, num_kv_heads, head_dim, v_dim, k_pages, v_pages, block_table, ctx.row_seg, ctx.row_pos, scale,
                                 window, bias, mix, ctx.max_context, gate=gate[:single] if gate is not None else None, q=q[:single],
                                 out=out[:single])
    if single < rows:
        if tile_seg is None or tile_row0 is None:
            raise KernelError("sigmoid_attention: the tiled kernel needs the step's query tiles")
        sigmoid_attention_prefill(q, num_heads, num_kv_heads, head_dim, v_dim, k_pages, v_pages, block_table, tile_seg[single:],
                                  tile_row0[single:], ctx.seg_row0, ctx.row_pos, scale, window, bias, mix, gate, out=out,
                                  max_context=ctx.max_context)
    return out


# ---- the gated delta rule -----------------------------------------------------------------------------
def _delta_inputs(name: str, proj, a, taps, conv_state, A_log, dt_bias, seg_row0, seg_slot, segments: int, heads: int, kv_heads: int, dim: int,
                  vdim: int, decay_per_head: bool):
    """Checks what the gated delta rule's kernels are given; (rows, floats between rows, channels, taps, decays of a row)."""
    _dev(proj, taps, conv_state, A_log, dt_bias, seg_row0, seg_slot)
    _dev_rows(a, "a")
    rows, stride = proj.shape
    channels = 2 * kv_heads * dim + heads * vdim
    count = taps.shape[1]
    if proj.dtype != a.dtype or not proj.is_contiguous() or a.dim() != 2 or a.stride(1) != 1:
        raise KernelError(f"{name}: the projections and the decays' arguments come in one dtype, rows contiguous")
    decays = heads if decay_per_head else heads * dim
    if a.shape != (rows, decays):
        raise KernelError(f"{name}: a is {tuple(a.shape)}, expected {(rows, decays)} (a view of wider rows will do)")
    for what, t, shape in (("taps", taps, (channels, count)), ("A_log", A_log, (heads,)), ("dt_bias", dt_bias, (decays,))):
        _want(t, torch.float32, what)
        if t.shape != shape or not t.is_contiguous():
            raise KernelError(f"{name}: {what} is {tuple(t.shape)}, expected {shape}")
    _want(conv_state, torch.float32, "conv_state")
    if conv_state.dim() != 3 or conv_state.shape[1:] != (channels, count - 1) or not conv_state.is_contiguous():
        raise KernelError(f"{name}: the convolutions' state is {tuple(conv_state.shape)}, expected [slots, {channels}, {count - 1}]")
    for what, t, n in (("seg_row0", seg_row0, segments + 1), ("seg_slot", seg_slot, segments)):
        _want(t, torch.int32, what)
        if t.numel() < n:
            raise KernelError(f"{name}: {what} holds {t.numel()} entries, needs {n}")
    return rows, stride, channels, count, decays


def delta_prepare(proj: torch.Tensor, beta_col: int, a: torch.Tensor, taps: torch.Tensor, conv_state: torch.Tensor,
                  A_log: torch.Tensor, dt_bias: torch.Tensor, row_seg: torch.Tensor, seg_row0: torch.Tensor,
                  seg_slot: torch.Tensor, segments: int, heads: int, kv_heads: int, dim: int, vdim: int,
                  decay_per_head: bool = False):
    """From a step's projections to what the recurrence reads. ``proj`` [rows, >= channels + ...]:
    its first ``channels`` = 2 kv_heads dim + heads vdim columns are q | k | v before their short
    convolutions, columns ``beta_col`` .. + heads the write strengths before the sigmoid; ``a``
    [rows, heads dim] the decays' arguments. ``conv_state`` [slots, channels, taps - 1] is read and
    moved on. ``decay_per_head``: one decay for all key channels of a head (``a`` [rows, heads],
    ``dt_bias`` [heads]). Returns float32 records [rows, heads, delta_record_floats(dim, vdim)]: per row and head
    q | k | g | beta | v as the recurrence reads them (q and k of the head's group)."""
    _dev(row_seg)
    _want(row_seg, torch.int32, "row_seg")
    if row_seg.numel() < proj.shape[0]:
        raise KernelError(f"delta_prepare: row_seg holds {row_seg.numel()} entries, needs {proj.shape[0]}")
    rows, stride, channels, count, decays = _delta_inputs("delta_prepare", proj, a, taps, conv_state, A_log, dt_bias, seg_row0, seg_slot,
                                                          segments, heads, kv_heads, dim, vdim, decay_per_head)
    records = torch.empty((rows, heads, delta_record_floats(dim, vdim)), dtype=torch.float32, device=proj.device)
    _check(library().fw_delta_prepare(_p(proj), _code(proj.dtype), stride, int(beta_col), _p(a), a.stride(0) if rows > 1 else max(decays, a.stride(0)),
                                      _p(taps), _p(conv_state), _p(A_log), _p(dt_bias), _p(row_seg), _p(seg_row0), _p(seg_slot),
                                      _p(records), rows, int(segments), heads, kv_heads, dim, vdim, count, conv_state.shape[0],
                                      int(decay_per_head), _stream()))
    return records


def delta_record_floats(dim: int, vdim: int) -> int:
    """Floats of what one token brings to one head of the recurrence: q | k | g (dim rounded up to a
    multiple of 4 each) | beta and three unused | v (vdim rounded up likewise)."""
    return 3 * ((dim + 3) // 4 * 4) + 4 + (vdim + 3) // 4 * 4


def _delta_state(name: str, state: torch.Tensor, heads: int, dim: int, vdim: int) -> None:
    _dev(state)
    _want(state, torch.float32, "state")
    if state.dim() != 4 or state.shape[1:] != (heads, vdim, dim):
        raise KernelError(f"{name}: the state is {tuple(state.shape)}, expected [slots, {heads}, {vdim}, {dim}]")


def gated_delta_rule(records: torch.Tensor, state: torch.Tensor, seg_row0: torch.Tensor, seg_slot: torch.Tensor,
                     segments: int, heads: int, dim: int, vdim: int, spread: bool = False) -> torch.Tensor:
    """The recurrence over each segment's rows (``spread``: large heads on twice the workgroups, for prompts).
    ``records`` [rows, heads, delta_record_floats]: what
    ``delta_prepare`` made. ``state`` [slots, heads, vdim, dim] float32 (the matrix transposed) is read
    at a segment's start and written at its end. Returns [rows, heads vdim]."""
    _dev(records, state, seg_row0, seg_slot)
    rows = records.shape[0]
    _want(records, torch.float32, "records")
    if records.shape != (rows, heads, delta_record_floats(dim, vdim)) or not records.is_contiguous():
        raise KernelError(f"gated_delta_rule: records are {tuple(records.shape)}, expected {(rows, heads, delta_record_floats(dim, vdim))}")
    _delta_state("gated_delta_rule", state, heads, dim, vdim)
    for name, t, n in (("seg_row0", seg_row0, segments + 1), ("seg_slot", seg_slot, segments)):
        _want(t, torch.int32, name)
        if t.numel() < n:
            raise KernelError(f"gated_delta_rule: {name} holds {t.numel()} entries, needs {n}")
    out = torch.empty((rows, heads * vdim), dtype=torch.float32, device=records.device)
    _check(library().fw_gated_delta_rule(_p(records), _p(state), _p(out), _p(seg_row0), _p(seg_slot), rows, int(segments), heads,
                                         dim, vdim, state.shape[0], int(spread), _stream()))
    return out


def delta_chunks(proj: torch.Tensor, beta_col: int, a: torch.Tensor, taps: torch.Tensor, conv_state: torch.Tensor, A_log: torch.Tensor,
                 dt_bias: torch.Tensor, state: torch.Tensor, seg_row0: torch.Tensor, seg_slot: torch.Tensor, segments: int, heads: int,
                 kv_heads: int, dim: int, vdim: int, decay_per_head: bool = False) -> torch.Tensor:
    """``delta_prepare`` and ``gated_delta_rule`` at once for steps with long segments, float32 projections: sixteen tokens of a segment at a
    time as matrix products (float32 throughout; other sums than token by token). Returns [rows, heads vdim]."""
    rows, stride, channels, count, decays = _delta_inputs("delta_chunks", proj, a, taps, conv_state, A_log, dt_bias, seg_row0, seg_slot,
                                                          segments, heads, kv_heads, dim, vdim, decay_per_head)
    _want(proj, torch.float32, "proj")
    _delta_state("delta_chunks", state, heads, dim, vdim)
    lib = library()
    packets = torch.empty((lib.fw_delta_chunk_slots(rows, int(segments)), heads, lib.fw_delta_packet_floats(dim, vdim)), dtype=torch.float32,
                          device=proj.device)
    out = torch.empty((rows, heads * vdim), dtype=torch.float32, device=proj.device)
    _check(lib.fw_delta_chunks(_p(proj), stride, int(beta_col), _p(a), a.stride(0) if rows > 1 else max(decays, a.stride(0)), _p(taps),
                               _p(conv_state), _p(A_log), _p(dt_bias), _p(seg_row0), _p(seg_slot), _p(packets), _p(state), _p(out), rows,
                               int(segments), heads, kv_heads, dim, vdim, count, min(conv_state.shape[0], state.shape[0]),
                               int(decay_per_head), _stream()))
    return out


def gated_head_norm(o: torch.Tensor, gate: torch.Tensor, weight: torch.Tensor, heads: int, vdim: int, eps: float,
                    out_dtype: torch.dtype, gate_silu: bool = False) -> torch.Tensor:
    # ``weight`` [vdim] serves every head; [heads * vdim] gives each head its own
    """Per head: o / rms(o) * weight * sigmoid(gate) (``gate_silu``: times gate * sigmoid(gate)); ``o`` float32 [rows, heads vdim], ``gate``
    [rows, heads vdim] (float32, or bfloat16 beside a bfloat16 output; a view of wider rows will do)."""
    _dev(o, weight)
    _dev_rows(gate, "gate")
    _want(o, torch.float32, "o")
    _want(weight, torch.float32, "weight")
    rows = o.shape[0]
    per_head = weight.shape == (heads * vdim,) and heads > 1
    if o.shape != (rows, heads * vdim) or gate.shape != o.shape or (weight.shape != (vdim,) and not per_head) or not o.is_contiguous() or gate.stride(1) != 1:
        raise KernelError(f"gated_head_norm: o {tuple(o.shape)}, gate {tuple(gate.shape)}, weight {tuple(weight.shape)} do not fit {heads} x {vdim}")
    out = torch.empty((rows, heads * vdim), dtype=out_dtype, device=o.device)
    _check(library().fw_gated_head_norm(_p(o), _p(gate), _code(gate.dtype), gate.stride(0) if rows > 1 else max(heads * vdim, gate.stride(0)), _p(weight), int(per_head), _p(out), _code(out_dtype), rows,
                                        heads, vdim, float(eps), int(gate_silu), _stream()))
    return out


# ---- sublayers whose output is normed --------------------------------------------------------------------
def norm_scale_add_(x: torch.Tensor, a: torch.Tensor, weight: torch.Tensor, eps: float, mult: float, *,
                    b: Optional[torch.Tensor] = None, scale_a: float = 1.0, scale_b: float = 1.0,
                    one_centered: bool = False, rounded_dtype: Optional[torch.dtype] = None) -> Optional[torch.Tensor]:
    """x += mult * rmsnorm(scale_a a + scale_b b) * w in place (float32 rows; ``b`` optional). With
    ``rounded_dtype`` the new x is also returned in that dtype (what the next products read)."""
    _dev(x, a, b, weight)
    rows, hidden = x.shape
    for name, t in (("x", x), ("a", a), ("b", b)):
        if t is not None:
            _want(t, torch.float32, name)
            if t.shape != (rows, hidden) or not t.is_contiguous():
                raise KernelError(f"norm_scale_add: {name} is {tuple(t.shape)}, expected {(rows, hidden)}")
    _want(weight, torch.float32, "weight")
    if weight.shape != (hidden,):
        raise KernelError(f"norm_scale_add: weight is {tuple(weight.shape)}, row width is {hidden}")
    rounded = torch.empty((rows, hidden), dtype=rounded_dtype, device=x.device) if rounded_dtype is not None else None
    _check(library().fw_norm_scale_add(_p(x), _p(a), _p(b), float(scale_a), float(scale_b), _p(weight),
                                       int(one_centered), float(eps), float(mult), _p(rounded),
                                       _code(rounded_dtype) if rounded_dtype is not None else F32, rows, hidden, _stream()))
    return rounded


def round_rows(x: torch.Tensor, dtype: torch.dtype) -> torch.Tensor:
    """float32 rows in the activation dtype (float32: the rows themselves)."""
    _want(x, torch.float32, "x")
    if dtype == torch.float32:
        return x
    _dev(x)
    out = torch.empty(x.shape, dtype=torch.bfloat16, device=x.device)
    _check(library().fw_round_rows(_p(x), _p(out), int(x.numel()), _stream()))
    return out


def clamped_glu(gate_up: torch.Tensor, limit: float, alpha: float, shift: float, out_dtype: torch.dtype) -> torch.Tensor:
    """[rows, gate | up] -> min(gate, limit) * sigmoid(alpha * that) * (clamp(up, +-limit) + shift)."""
    _dev(gate_up)
    rows, width = gate_up.shape
    if width % 2 or not gate_up.is_contiguous():
        raise KernelError("clamped_glu: the input holds gate and up halves, contiguous")
    out = torch.empty((rows, width // 2), dtype=out_dtype, device=gate_up.device)
    _check(library().fw_clamped_glu(_p(gate_up), _code(gate_up.dtype), _p(out), _code(out_dtype), rows, width // 2,
                                    float(limit), float(alpha), float(shift), _stream()))
    return out


def gemm_clamped_glu(a: torch.Tensor, w_gate_up: torch.Tensor, limit: float, alpha: float, shift: float) -> Optional[torch.Tensor]:
    """clamped_glu(a . [gate | up]^T) in bfloat16 for more than 64 rows by weights that a model holds, the unit in the product's epilogue; None where no large
    tile takes the product (``large_tile``)."""
    rows2, K = w_gate_up.shape
    M = a.shape[0]
    if rows2 % 2 or a.shape[1] != K or M <= MEDIUM_MAX_ROWS or not _fast_ok(a, w_gate_up) or not limit > 0.0:
        return None
    tile = large_tile(2, M, rows2 // 2, K)
    if tile is None:
        return None
    _dev(a, w_gate_up)
    out = torch.empty((M, rows2 // 2), dtype=torch.bfloat16, device=a.device)
    _check(library().fw_gemm_mfma_big_tile_clamped(a.data_ptr(), w_gate_up.data_ptr(), out.data_ptr(), M, rows2 // 2, K, *tile[:3], limit, alpha, shift, _stream()))
    return out


# ---- a sublayer between two norms, layer norm, the gate on a second token table ------------------------------
NEXT_NOTHING, NEXT_ROUNDED, NEXT_RMS, NEXT_CENTERED = 0, 1, 2, 3


def layernorm_rows(x: torch.Tensor, weight: torch.Tensor, eps: float, out_dtype: torch.dtype,
                   row_index: Optional[torch.Tensor] = None, bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """(x - mean) / sqrt(mean((x - mean)^2) + eps) * weight (+ bias) over float32 rows (gathered through
    ``row_index`` if given), in ``out_dtype``."""
    _dev(x, weight, row_index, bias)
    _want(x, torch.float32, "x")
    hidden = x.shape[-1]
    for name, t in (("weight", weight), ("bias", bias)):
        if t is not None:
            _want(t, torch.float32, name)
            if t.shape != (hidden,):
                raise KernelError(f"layernorm: {name} is {tuple(t.shape)}, row width is {hidden}")
    rows = x.numel() // hidden if row_index is None else row_index.numel()
    if row_index is not None:
        _want(row_index, torch.int32, "row_index")
    out = torch.empty((rows, hidden), dtype=out_dtype, device=x.device)
    _check(library().fw_layernorm_rows(_p(x), _p(weight), _p(bias), _p(out), _code(out_dtype), _p(row_index), rows, hidden,
                                       float(eps), _stream()))
    return out


def norm_add_norm_(x: torch.Tensor, a: torch.Tensor, weight: torch.Tensor, centered: bool, eps: float, *,
                   bias: Optional[torch.Tensor] = None, mult: float = 1.0, next_kind: int = NEXT_NOTHING,
                   next_weight: Optional[torch.Tensor] = None, next_bias: Optional[torch.Tensor] = None, next_eps: float = 0.0,
                   next_dtype: Optional[torch.dtype] = None, next_out: Optional[torch.Tensor] = None) -> Optional[torch.Tensor]:
    """x += mult * (norm(a) * weight + bias) in place (float32 rows; ``bias`` optional; ``centered``: the row's mean is
    taken off before its root mean square). What reads x next is formed from the new rows in the same kernel and
    returned: ``NEXT_ROUNDED`` the rows in ``next_dtype``, ``NEXT_RMS`` / ``NEXT_CENTERED`` their norm with ``next_weight``,
    ``next_bias`` (optional) and ``next_eps``, into ``next_out`` if given (rows may lie apart); ``NEXT_NOTHING`` returns None."""
    _dev(x, a, weight, bias, next_weight, next_bias)
    rows, hidden = x.shape
    for name, t in (("x", x), ("a", a)):
        _want(t, torch.float32, name)
        if t.shape != (rows, hidden):
            raise KernelError(f"norm_add_norm: {name} is {tuple(t.shape)}, expected {(rows, hidden)}")
    for name, t in (("weight", weight), ("bias", bias), ("next_weight", next_weight), ("next_bias", next_bias)):
        if t is not None:
            _want(t, torch.float32, name)
            if t.shape != (hidden,):
                raise KernelError(f"norm_add_norm: {name} is {tuple(t.shape)}, row width is {hidden}")
    if next_kind not in (NEXT_NOTHING, NEXT_ROUNDED, NEXT_RMS, NEXT_CENTERED):
        raise KernelError(f"norm_add_norm: unknown kind {next_kind} of what follows")
    if next_kind >= NEXT_RMS and next_weight is None:
        raise KernelError("norm_add_norm: the norm that follows needs its weight")
    out = None
    if next_kind != NEXT_NOTHING:
        out = next_out
        if out is None:
            out = torch.empty((rows, hidden), dtype=next_dtype or torch.float32, device=x.device)
        _dev_rows(out, "next_out")
        if out.shape != (rows, hidden) or (next_dtype is not None and out.dtype != next_dtype):
            raise KernelError(f"norm_add_norm: next_out is {tuple(out.shape)} {out.dtype}, expected {(rows, hidden)} {next_dtype}")
    _check(library().fw_norm_add_norm(_p(x), _p(a), _p(weight), _p(bias), float(mult), int(centered), float(eps),
                                      int(next_kind), _p(next_weight), _p(next_bias), float(next_eps), _p(out),
                                      _code(out.dtype) if out is not None else F32, _stride(out) if out is not None else 0, rows, hidden,
                                      _stream()))
    return out


def place_rows(x: torch.Tensor, out: torch.Tensor, col0: int = 0, twice: bool = False) -> torch.Tensor:
    """float32 rows (which may lie apart) into columns ``col0`` .. of the wider rows ``out``, in its dtype; ``twice``: once
    more behind them."""
    _dev(out)
    _dev_rows(x, "x")
    _want(x, torch.float32, "x")
    if x.dim() != 2 or out.dim() != 2 or out.shape[0] != x.shape[0]:
        raise KernelError(f"place_rows: {tuple(x.shape)} into {tuple(out.shape)}")
    _check(library().fw_place_rows(_p(x), _stride(x), _p(out), _code(out.dtype), x.shape[0], x.shape[1], out.shape[1], int(col0), int(twice), _stream()))
    return out


def gelu_rows(z: torch.Tensor, out_dtype: torch.dtype) -> torch.Tensor:
    """z Phi(z) (the error-function gelu) of float32 values, in ``out_dtype``."""
    _dev(z)
    _want(z, torch.float32, "z")
    out = torch.empty(z.shape, dtype=out_dtype, device=z.device)
    _check(library().fw_gelu_rows(_p(z), _p(out), _code(out_dtype), int(z.numel()), _stream()))
    return out


def gelu_gate_rows(z: torch.Tensor, table: torch.Tensor, ids: torch.Tensor, col0: int, out_dtype: torch.dtype) -> torch.Tensor:
    """gelu_tanh(z) * table[ids][:, col0 : col0 + width]: ``z`` float32 [rows, width], ``table`` [entries,
    columns], ``ids`` int32 [rows] (checked against the table by the caller)."""
    _dev(z, table, ids)
    _want(z, torch.float32, "z")
    _want(ids, torch.int32, "ids")
    rows, width = z.shape
    if table.dim() != 2 or col0 < 0 or col0 + width > table.shape[1] or ids.numel() < rows:
        raise KernelError(f"gelu_gate_rows: columns {col0}..{col0 + width} of a table {tuple(table.shape)}, {ids.numel()} ids for {rows} rows")
    out = torch.empty((rows, width), dtype=out_dtype, device=z.device)
    _check(library().fw_gelu_gate_rows(_p(z), width, _p(table), _code(table.dtype), table.shape[0], table.shape[1], int(col0), _p(ids),
                                       _p(out), _code(out_dtype), rows, width, _stream()))
    return out


# ---- attention over a cached latent ------------------------------------------------------------------------
def latent_norm_write(raw: torch.Tensor, weight: torch.Tensor, eps: float, k_pages: torch.Tensor, v_pages: torch.Tensor,
                      block_table: torch.Tensor, row_seg: torch.Tensor, row_pos: torch.Tensor, rot: int = 0,
                      cos: Optional[torch.Tensor] = None, sin: Optional[torch.Tensor] = None, turn: Optional[int] = None,
                      interleaved: bool = True) -> None:
    """The step's latents ``raw`` (float32 [rows, rank + rot]; a view of some columns of wider rows will do): the first
    rank columns RMS-normed times ``weight`` and stored at each row's position in a cache of one key/value head; the last
    ``rot`` columns (a key part all heads share) turned by the row's angles (``interleaved``: neighbouring channels paired,
    else channel i with channel i + turn / 2; ``cos``, ``sin`` float32 [rows, turn / 2]) and stored behind the latent in the keys' layout, whose head then has rank + rot channels."""
    _dev(weight, k_pages, v_pages, block_table, row_seg, row_pos, cos, sin)
    _dev_rows(raw, "raw")
    _want(raw, torch.float32, "raw")
    _want(weight, torch.float32, "weight")
    rows, rank = raw.shape[0], raw.shape[1] - int(rot)
    if weight.shape != (rank,):
        raise KernelError(f"latent_norm_write: weight is {tuple(weight.shape)}, the latent has {rank} channels")
    turn = int(rot) if turn is None else int(turn)      # the first so many channels of the part are turned, the rest pass
    if turn:
        for t in (cos, sin):
            if t is None or t.dtype != torch.float32 or t.shape != (rows, turn // 2):
                raise KernelError(f"latent_norm_write: {turn} turned channels need float32 tables {(rows, turn // 2)}")
    pages = _check_pages(k_pages, v_pages, 1, rank + int(rot), k_pages.dtype, rank)
    for name, t in (("block_table", block_table), ("row_seg", row_seg), ("row_pos", row_pos)):
        _want(t, torch.int32, name)
    if block_table.dim() != 2 or row_seg.numel() < rows or row_pos.numel() < rows:
        raise KernelError("latent_norm_write: batch index arrays are too short")
    _check(library().fw_latent_norm_write(_p(raw), raw.stride(0) if rows > 1 else max(rank + int(rot), raw.stride(0)), 0, _p(weight),
                                          float(eps), _p(k_pages), _p(v_pages), _code(k_pages.dtype), _p(block_table),
                                          block_table.shape[1], _p(row_seg), _p(row_pos), rows, rank, int(rot), turn, int(interleaved), _p(cos), _p(sin),
                                          PAGE_SIZE, pages, _stream()))


def head_linear(x: torch.Tensor, w: torch.Tensor, out_dtype: torch.dtype, gate: Optional[torch.Tensor] = None,
                in_head: Optional[int] = None, out: Optional[torch.Tensor] = None, out_head: Optional[int] = None) -> torch.Tensor:
    """A map per head: ``x`` [rows, heads K] (rows may lie apart), ``w`` [heads, N, K] -> [rows, heads N], with
    ``gate`` (float32 [rows, heads N], or [rows, heads]: one number a head; rows may lie apart) times its sigmoid. ``in_head``: a head's vector in ``x`` holds
    that many channels of which the map reads the first K; ``out`` with ``out_head``: the results go to the first N
    channels of each head's vector of ``out_head`` channels in the rows of ``out``."""
    _dev(w)
    _dev_rows(x, "x")
    heads, N, K = w.shape
    rows = x.shape[0]
    in_head = K if in_head is None else int(in_head)
    if x.shape[1] != heads * in_head or in_head < K:
        raise KernelError(f"head_linear: x is {tuple(x.shape)}, the weight {tuple(w.shape)}, a head's vector {in_head}")
    if gate is not None:
        _dev_rows(gate, "gate")
        if gate.shape not in ((rows, heads * N), (rows, heads)) or gate.dtype != torch.float32:
            raise KernelError(f"head_linear: the gate is {tuple(gate.shape)} {gate.dtype}, expected {(rows, heads * N)} or {(rows, heads)} float32")
    out_head = N if out_head is None else int(out_head)
    if out is None:
        out = torch.empty((rows, heads * out_head), dtype=out_dtype, device=x.device)
    elif out.shape != (rows, heads * out_head) or out.dtype != out_dtype or not out.is_contiguous() or not out.is_cuda:
        raise KernelError(f"head_linear: out is {tuple(out.shape)} {out.dtype}, expected {(rows, heads * out_head)} {out_dtype}")
    if out_head < N or (gate is not None and out_head != N):
        raise KernelError("head_linear: a head's outputs do not fit its vector (a gate goes with outputs side by side)")

    def stride(t: torch.Tensor, width: int) -> int:
        return t.stride(0) if rows > 1 else max(width, t.stride(0))

    _check(library().fw_head_linear(_p(x), _code(x.dtype), stride(x, heads * in_head), _p(w), _code(w.dtype), _p(gate),
                                    stride(gate, gate.shape[1]) if gate is not None else 0,
                                    int(gate is not None and gate.shape[1] == heads and N > 1), _p(out), _code(out_dtype), rows, heads, N, K,
                                    in_head, out_head, heads * out_head, _stream()))
    return out


def rotate_place(x: torch.Tensor, heads: int, col0: int, rot: int, cos: torch.Tensor, sin: torch.Tensor, out: torch.Tensor,
                 out_col0: int, turn: Optional[int] = None, interleaved: bool = True) -> torch.Tensor:
    """Channels col0 .. col0 + rot - 1 of every head's vector in ``x`` [rows, heads * in_head], neighbouring channels
    (``interleaved``; else channels i and i + turn / 2) turned by the row's angles (``cos``, ``sin`` float32 [rows, rot / 2]), stored from channel ``out_col0`` of the head's
    vector in ``out`` [rows, heads * out_head]."""
    _dev(x, cos, sin, out)
    rows = x.shape[0]
    if x.dim() != 2 or out.dim() != 2 or x.shape[1] % heads or out.shape[1] % heads or out.shape[0] != rows:
        raise KernelError(f"rotate_place: {tuple(x.shape)} -> {tuple(out.shape)} with {heads} heads")
    turn = int(rot) if turn is None else int(turn)      # the first so many channels are turned, the rest pass
    for t in ((cos, sin) if turn else ()):
        if t is None or t.dtype != torch.float32 or t.shape != (rows, turn // 2):
            raise KernelError(f"rotate_place: {turn} turned channels need float32 tables {(rows, turn // 2)}")
    _check(library().fw_rotate_place(_p(x), _code(x.dtype), x.shape[1], x.shape[1] // heads, int(col0), _p(cos), _p(sin), _p(out),
                                     _code(out.dtype), out.shape[1], out.shape[1] // heads, int(out_col0), rows, heads, int(rot), turn,
                                     int(interleaved), _stream()))
    return out


# ---- a recurrence with a decay per key channel formed by the token ("wkv") --------------------------------------
def token_shift_mix(x: torch.Tensor, norm_weight: Optional[torch.Tensor], eps: float, one_centered: bool, mu: torch.Tensor,
                    last: torch.Tensor, row_seg: torch.Tensor, seg_row0: torch.Tensor, seg_slot: torch.Tensor, segments: int,
                    out_dtype: torch.dtype) -> torch.Tensor:
    """h = rmsnorm(x) * weight (``norm_weight`` None: h = x); returns [mixes, rows, hidden] = h + (h of the row before - h)
    * mu[s]. ``last`` float32 [slots, hidden]: the h of each request's last row so far, read for a segment's first
    row and moved on."""
    _dev(x, norm_weight, mu, last, row_seg, seg_row0, seg_slot)
    _want(x, torch.float32, "x")
    _want(mu, torch.float32, "mu")
    _want(last, torch.float32, "last")
    rows, hidden = x.shape
    if mu.dim() != 2 or mu.shape[1] != hidden or last.dim() != 2 or last.shape[1] != hidden:
        raise KernelError(f"token_shift_mix: mu {tuple(mu.shape)} / last {tuple(last.shape)} beside rows of {hidden}")
    if norm_weight is not None and (norm_weight.dtype != torch.float32 or norm_weight.shape != (hidden,)):
        raise KernelError("token_shift_mix: the norm's weight is float32 [hidden]")
    for name, t, n in (("row_seg", row_seg, rows), ("seg_row0", seg_row0, segments + 1), ("seg_slot", seg_slot, segments)):
        _want(t, torch.int32, name)
        if t.numel() < n:
            raise KernelError(f"token_shift_mix: {name} holds {t.numel()} entries, needs {n}")
    out = torch.empty((mu.shape[0], rows, hidden), dtype=out_dtype, device=x.device)
    _check(library().fw_token_shift_mix(_p(x), _p(norm_weight), float(eps), int(one_centered), _p(mu), mu.shape[0], _p(last),
                                        last.shape[0], _p(row_seg), _p(seg_row0), _p(seg_slot), _p(out), _code(out_dtype), rows,
                                        int(segments), hidden, _stream()))
    return out


def tanh_rows(x: torch.Tensor, out_dtype: torch.dtype) -> torch.Tensor:
    _dev(x)
    _want(x, torch.float32, "x")
    out = torch.empty(x.shape, dtype=out_dtype, device=x.device)
    _check(library().fw_tanh_rows(_p(x), _p(out), _code(out_dtype), int(x.numel()), _stream()))
    return out


def wkv_recurrence(r: torch.Tensor, k: torch.Tensor, v: torch.Tensor, a: torch.Tensor, w0: torch.Tensor, u: torch.Tensor,
                   state: torch.Tensor, seg_row0: torch.Tensor, seg_slot: torch.Tensor, segments: int, heads: int, dim: int,
                   chunks: Optional[tuple] = None) -> torch.Tensor:
    """Per head o_t = S^T r_t + (r_t . (u k_t)) v_t, then S <- diag(exp(-exp(a_t + w0))) S + k_t v_t^T, over each segment's rows
    in order. ``r``, ``k``, ``v`` float32 [rows, heads dim] with one row stride (views of wider rows will do), ``a``
    likewise; ``state`` float32 [slots, heads, dim, dim] is read and moved on. ``chunks``: as for ``decay_recurrence``. Returns
    float32 [rows, heads dim]."""
    _dev(w0, u, state, seg_row0, seg_slot)
    rows = r.shape[0]
    width = heads * dim
    for name, t in (("r", r), ("k", k), ("v", v), ("a", a)):
        _dev_rows(t, name)
        _want(t, torch.float32, name)
        if t.shape != (rows, width):
            raise KernelError(f"wkv_recurrence: {name} is {tuple(t.shape)}, expected {(rows, width)}")

    def stride(t):
        return t.stride(0) if rows > 1 else max(width, t.stride(0))

    if not (stride(r) == stride(k) == stride(v)):
        raise KernelError("wkv_recurrence: r, k and v have one row stride")
    for name, t in (("w0", w0), ("u", u)):
        _want(t, torch.float32, name)
        if t.numel() != width:
            raise KernelError(f"wkv_recurrence: {name} holds {t.numel()} values, expected {width}")
    _want(state, torch.float32, "state")
    if state.dim() != 4 or state.shape[1:] != (heads, dim, dim):
        raise KernelError(f"wkv_recurrence: the state is {tuple(state.shape)}, expected [slots, {heads}, {dim}, {dim}]")
    for name, t, n in (("seg_row0", seg_row0, segments + 1), ("seg_slot", seg_slot, segments)):
        _want(t, torch.int32, name)
        if t.numel() < n:
            raise KernelError(f"wkv_recurrence: {name} holds {t.numel()} entries, needs {n}")
    out = torch.empty((rows, width), dtype=torch.float32, device=r.device)
    places, count, *how = _chunks("wkv_recurrence", chunks, segments)
    if count and library().fw_wkv_chunk_plan() != DECAY_CHUNK:
        raise KernelError("the kernel library's chunks are of another length")
    workspace = torch.empty(count * width * (dim + 1), dtype=torch.float32, device=r.device) if count else None
    _check(library().fw_wkv_recurrence(_p(r), _p(k), _p(v), stride(r), _p(a), stride(a), _p(w0), _p(u), _p(state), state.shape[0], _p(out),
                                       _p(seg_row0), _p(seg_slot), rows, int(segments), heads, dim, *(_p(t) for t in places), count, *how,
                                       _p(workspace), _stream()))
    return out


# ---- a mixture of feed-forward units chosen per token ------------------------------------------------------------
MOE_SCORES = ("softmax_chosen", "softmax_all", "sigmoid")


def moe_route(logits: torch.Tensor, bias: Optional[torch.Tensor], top: int, groups: int = 1, keep: int = 1,
              score_all: bool = False, scores: Optional[str] = None, group_pair: bool = False, correction: Optional[torch.Tensor] = None,
              weight_scale: float = 1.0, normalize: bool = True):
    """(chosen int32 [rows, top], weight float32 [rows, top]): the ``top`` largest of logits + bias per row, largest
    first (ties: the lowest id), and the softmax over those alone. ``groups`` > 1: only experts of the ``keep`` groups
    (of neighbours, equal in size) whose best expert scores highest can be chosen. ``score_all``: the weights are the
    softmax over all experts at the chosen ones, divided by their sum + 1e-20. ``scores`` names the same choice
    ("softmax_chosen", "softmax_all") or "sigmoid": each expert's own sigmoid at the chosen ones, divided by their sum + 1e-20.
    ``group_pair``: groups are ranked by what their two best experts score together (not with "softmax_chosen").
    ``correction`` (float32 [experts], with "sigmoid"): the choice is by score + correction, the weights are the scores
    without it. ``weight_scale`` multiplies the weights; ``normalize`` False (with "softmax_all" and "sigmoid"): they are not
    divided by their sum. Rows of ``logits`` may lie apart."""
    scores = scores or ("softmax_all" if score_all else "softmax_chosen")
    if scores not in MOE_SCORES or (group_pair and scores == "softmax_chosen"):
        raise KernelError(f"moe_route: scores {scores!r} (known: {', '.join(MOE_SCORES)}; groups by pairs: {group_pair})")
    _dev(bias, correction)
    _dev_rows(logits, "logits")
    _want(logits, torch.float32, "logits")
    rows, experts = logits.shape
    if correction is not None and (correction.dtype != torch.float32 or correction.shape != (experts,) or scores != "sigmoid"):
        raise KernelError("moe_route: a correction is float32 [experts] and goes with sigmoid scores")
    if not normalize and scores == "softmax_chosen":
        raise KernelError("moe_route: the softmax over the chosen is a distribution over them")
    if bias is not None and (bias.dtype != torch.float32 or bias.shape != (experts,)):
        raise KernelError("moe_route: the bias is float32 [experts]")
    chosen = torch.empty((rows, top), dtype=torch.int32, device=logits.device)
    weight = torch.empty((rows, top), dtype=torch.float32, device=logits.device)
    _check(library().fw_moe_route(_p(logits), _stride(logits), _p(bias), _p(correction), _p(chosen), _p(weight), rows, experts, int(top),
                                  int(groups), int(keep), int(group_pair), MOE_SCORES.index(scores), float(weight_scale),
                                  int(normalize), _stream()))
    return chosen, weight


def moe_arrange(chosen: torch.Tensor, experts: int):
    """The pairs (row, choice) sorted by expert, an expert's pairs in their order: (expert_begin int32 [experts + 1],
    place_row int32 [pairs], pair_place int32 [rows, top])."""
    _dev(chosen)
    _want(chosen, torch.int32, "chosen")
    rows, top = chosen.shape
    expert_begin = torch.empty((experts + 1,), dtype=torch.int32, device=chosen.device)
    place_row = torch.empty((rows * top,), dtype=torch.int32, device=chosen.device)
    pair_place = torch.empty((rows, top), dtype=torch.int32, device=chosen.device)
    _check(library().fw_moe_arrange(_p(chosen), _p(expert_begin), _p(place_row), _p(pair_place), rows, int(experts), top, _stream()))
    return expert_begin, place_row, pair_place


def grouped_few_tiles(places: int, experts: int) -> int:
    """Tiles of 16 places to a wave of the grouped product whose experts' weights come in operand tiles (fw_grouped_gemm_few), 0 where the tiles
    of moe.hip and gemm_mfma_big.hip are faster (the bits are the same). By places an expert in the mean, us for both products (those tiles / one / two): 32 experts of
    1,536 features over 2,048, 4 a row, 1 / 8 / 32 / 64 / 96 / 128 rows 37 / 19 / -, 87 / 64 / -, 121 / 92 / 93, 126 / 99 / 97, 127 / 109 / 101, 128 / 143 / 108; 8 of 4,096
    over 2,048, 2 a row, 8 / 32 / 64 rows 90 / 58 / 58, 109 / 71 / 72, 110 / 89 / 74."""
    return 1 if places <= 8 * experts else 2 if places <= 16 * experts else 0


def grouped_gemm(a: torch.Tensor, place_row: Optional[torch.Tensor], w: Union[torch.Tensor, ExpertWeights], expert_begin: torch.Tensor, places: int,
                 gated: bool, out_dtype: torch.dtype, glu: Optional[tuple] = None, w_tiled: Optional[torch.Tensor] = None) -> torch.Tensor:
    """out[place] = a[place_row[place]] . w[expert of place]^T (``place_row`` None: a[place]); ``w`` [experts, N, K], or
    with ``gated`` [experts, 2 N, K] (gate rows, then up rows) and out = silu(gate) * up, or with ``glu`` = (limit, alpha,
    shift) the unit with clamped halves. ``w_tiled``: the rows of ``w`` [experts * N, K] once more in operand tiles
    (``tile_weights``), for steps of a few places an expert; an ``ExpertWeights`` holds its rows in them alone. Returns [places, N]."""
    shape = w.shape
    if isinstance(w, ExpertWeights):
        w, w_tiled = w.rows, w.tiled
    _dev(a, place_row, w, expert_begin)
    experts, n_rows, K = shape
    N = n_rows // 2 if gated else n_rows
    if a.dim() != 2 or a.shape[1] != K or (gated and n_rows % 2) or expert_begin.numel() != experts + 1:
        raise KernelError(f"grouped_gemm: a is {tuple(a.shape)}, w {tuple(shape)}, {expert_begin.numel()} expert bounds")
    _want(expert_begin, torch.int32, "expert_begin")
    if place_row is not None:
        _want(place_row, torch.int32, "place_row")
        if place_row.numel() < places:
            raise KernelError("grouped_gemm: fewer rows named than places")
    elif a.shape[0] < places:
        raise KernelError("grouped_gemm: fewer rows than places")
    out = torch.empty((places, N), dtype=out_dtype, device=a.device)
    if w is None and a.data_ptr() % 16:
        a = a.clone()
    if w_tiled is not None and a.dtype == torch.bfloat16 and out_dtype == (torch.bfloat16 if gated else torch.float32) and a.data_ptr() % 16 == 0:
        place_tiles = grouped_few_tiles(places, experts)
        if place_tiles:
            if w is not None:
                w_tiled = _tiled_for(w.view(experts * n_rows, K), w_tiled)
            _check(library().fw_grouped_gemm_few(_p(a), _p(place_row), _p(w_tiled), _p(expert_begin), _p(out), int(gated), int(places), experts, N, K, place_tiles,
                                                 *_glu(glu if gated else None), _stream()))
            return out
    held, held_code = (w_tiled, BF16_TILES) if w is None else (w, _code(w.dtype))
    _check(library().fw_grouped_gemm(_p(a), _code(a.dtype), a.shape[0], _p(place_row), _p(held), held_code, _p(expert_begin), _p(out),
                                     _code(out_dtype), int(gated), int(places), experts, N, K, *_glu(glu if gated else None), _stream()))
    return out


def moe_combine_(x: torch.Tensor, y: torch.Tensor, weight: torch.Tensor, pair_place: torch.Tensor, shared: Optional[torch.Tensor] = None,
                 gate: Optional[torch.Tensor] = None) -> torch.Tensor:
    """x[row] += sum over the row's choices, in their order, of weight[row, j] * y[pair_place[row, j]], plus with ``shared``
    [rows, hidden] and ``gate`` [rows, 1] (rows may lie apart) sigmoid(gate) * shared; float32."""
    _dev(x, y, weight, pair_place, shared)
    for name, t in (("x", x), ("y", y), ("weight", weight)):
        _want(t, torch.float32, name)
    _want(pair_place, torch.int32, "pair_place")
    rows, hidden = x.shape
    top = weight.shape[1]
    if weight.shape != (rows, top) or pair_place.shape != (rows, top) or y.shape != (rows * top, hidden):
        raise KernelError(f"moe_combine: x {tuple(x.shape)}, y {tuple(y.shape)}, weight {tuple(weight.shape)}, places {tuple(pair_place.shape)}")
    if (shared is None) != (gate is None):
        raise KernelError("moe_combine: rows to be gated and their gate come together")
    if shared is not None:
        _dev_rows(gate, "gate")
        if shared.dtype != torch.float32 or shared.shape != (rows, hidden) or gate.dtype != torch.float32 or gate.shape != (rows, 1):
            raise KernelError(f"moe_combine: shared rows {tuple(shared.shape)} and gate {tuple(gate.shape)} beside x {tuple(x.shape)}")
    _check(library().fw_moe_combine(_p(x), _p(y), _p(weight), _p(pair_place), _p(shared), _p(gate), _stride(gate) if gate is not None else 0,
                                    rows, top, hidden, _stream()))
    return x


# ---- a short causal convolution per channel, and a gated linear recurrence per channel ---------------------------------
def causal_conv(x: torch.Tensor, taps: torch.Tensor, bias: Optional[torch.Tensor], state: torch.Tensor, row_seg: torch.Tensor,
                seg_row0: torch.Tensor, seg_slot: torch.Tensor, segments: int, single_rows: bool = False,
                echo: Optional[tuple] = None, silu: bool = False, rounded: bool = False):
    """y[t, c] = sum_j taps[c, j] * x[t - L + 1 + j, c] (+ bias[c]) over the step's segments, float32. ``x`` float32
    [rows, channels] (rows may lie apart), ``taps`` [channels, L] with the last column the current token's, ``state``
    float32 [slots, channels, L - 1]: the inputs before each segment's first row, read and moved on. ``echo`` = (first
    channel, count): those channels are written once more behind the others (the output is then that much wider).
    ``single_rows``: every segment is one row. ``silu``: y passes silu. ``rounded``: y is returned twice, (float32, bfloat16)."""
    _dev(taps, bias, state, row_seg, seg_row0, seg_slot)
    _dev_rows(x, "x")
    for name, t in (("x", x), ("taps", taps), ("state", state)):
        _want(t, torch.float32, name)
    rows, channels = x.shape
    L = taps.shape[1]
    if taps.shape != (channels, L) or state.dim() != 3 or state.shape[1:] != (channels, L - 1):
        raise KernelError(f"causal_conv: x {tuple(x.shape)}, taps {tuple(taps.shape)}, state {tuple(state.shape)}")
    if bias is not None and (bias.dtype != torch.float32 or bias.shape != (channels,)):
        raise KernelError("causal_conv: the bias is float32 [channels]")
    for name, t, n in (("row_seg", row_seg, rows), ("seg_row0", seg_row0, segments + 1), ("seg_slot", seg_slot, segments)):
        _want(t, torch.int32, name)
        if t.numel() < n:
            raise KernelError(f"causal_conv: {name} holds {t.numel()} entries, needs {n}")
    first, count = echo if echo is not None else (0, 0)
    if count and not (0 <= first and first + count <= channels):
        raise KernelError(f"causal_conv: channels {first}..{first + count} of {channels}")
    out = torch.empty((rows, channels + count), dtype=torch.float32, device=x.device)
    short = torch.empty((rows, channels), dtype=torch.bfloat16, device=x.device) if rounded else None
    stride = x.stride(0) if rows > 1 else max(channels, x.stride(0))
    _check(library().fw_causal_conv(_p(x), stride, _p(taps), _p(bias), _p(state), _p(row_seg), _p(seg_row0), _p(seg_slot), _p(out),
                                    channels + count, int(first), int(count), channels, int(silu), _p(short), rows, int(segments), channels, L,
                                    state.shape[0], int(bool(single_rows)), _stream()))
    return (out, short) if rounded else out


SCAN_LONG = 256     # rows of a segment beyond which the recurrence walks it in chunks side by side


def rglru_scan(u: torch.Tensor, gates: torch.Tensor, y: torch.Tensor, r_bias: torch.Tensor, i_bias: torch.Tensor, lam: torch.Tensor,
               rate: float, state: torch.Tensor, seg_row0: torch.Tensor, seg_slot: torch.Tensor, segments: int, block_width: int,
               out_dtype: torch.dtype) -> torch.Tensor:
    """The gated linear recurrence per channel over the step's segments: r = sigmoid(g_r + r_bias), i = sigmoid(g_i +
    i_bias), a = exp(-rate r softplus(lam)), S <- a S + sqrt(1 - a^2) i u, out = S * gelu_tanh(y). ``u``, ``y`` float32
    [rows, channels] (rows may lie apart); ``gates`` float32 [rows, 2 channels], block after block [g_r of the block | g_i
    of the block]; ``state`` float32 [slots, channels], read and moved on."""
    _dev(gates, r_bias, i_bias, lam, state, seg_row0, seg_slot)
    _dev_rows(u, "u")
    _dev_rows(y, "y")
    rows, channels = u.shape
    for name, t in (("u", u), ("gates", gates), ("y", y), ("r_bias", r_bias), ("i_bias", i_bias), ("lam", lam), ("state", state)):
        _want(t, torch.float32, name)
    if y.shape != (rows, channels) or gates.shape != (rows, 2 * channels) or channels % block_width or state.dim() != 2 \
            or state.shape[1] != channels or any(t.numel() != channels for t in (r_bias, i_bias, lam)):
        raise KernelError(f"rglru_scan: u {tuple(u.shape)}, gates {tuple(gates.shape)}, y {tuple(y.shape)}, state {tuple(state.shape)}, "
                          f"blocks of {block_width}")
    for name, t, n in (("seg_row0", seg_row0, segments + 1), ("seg_slot", seg_slot, segments)):
        _want(t, torch.int32, name)
        if t.numel() < n:
            raise KernelError(f"rglru_scan: {name} holds {t.numel()} entries, needs {n}")
    out = torch.empty((rows, channels), dtype=out_dtype, device=u.device)
    # a step that may hold a long segment: the kernels walk such a one in chunks side by side and need room for it
    workspace = torch.empty((2, rows, channels), dtype=torch.float32, device=u.device) if rows > SCAN_LONG else None

    def stride(t: torch.Tensor) -> int:
        return t.stride(0) if rows > 1 else max(channels, t.stride(0))

    _check(library().fw_rglru_scan(_p(u), stride(u), _p(gates), 2 * channels, _p(y), stride(y), _p(r_bias), _p(i_bias), _p(lam),
                                   float(rate), _p(state), _p(seg_row0), _p(seg_slot), _p(out), _code(out_dtype), rows,
                                   int(segments), channels, int(block_width), state.shape[0], _p(workspace), _stream()))
    return out


# ---- a residual stream of several rows side by side ----------------------------------------------------------------
NEXT_SUM, NEXT_TANH = 1, 2
SOURCE_ROWS, SOURCE_BRANCHES, SOURCE_CHOSEN = 0, 1, 2
MAX_STREAMS = 32


def _reader(kind: int, streams: int, hidden: int, reader_in: Optional[torch.Tensor], weight: Optional[torch.Tensor],
            bias: Optional[torch.Tensor], alpha: Optional[torch.Tensor]) -> tuple:
    for name, t, shape in (("reader_in", reader_in, (streams,)), ("weight", weight, (hidden,)), ("bias", bias, (hidden,))):
        if t is not None:
            _want(t, torch.float32, name)
            if t.shape != shape:
                raise KernelError(f"streams: {name} is {tuple(t.shape)}, expected {shape}")
    if kind == NEXT_TANH and (weight is None or bias is None or alpha is None or alpha.dtype != torch.float32 or alpha.numel() != 1):
        raise KernelError("streams: the tanh norm has a weight, a bias and one float32 alpha")
    return int(kind), _p(reader_in), _p(weight), _p(bias), _p(alpha)


def stream_read(x: torch.Tensor, reader_in: Optional[torch.Tensor], out_dtype: torch.dtype, *, kind: int = NEXT_SUM,
                weight: Optional[torch.Tensor] = None, bias: Optional[torch.Tensor] = None, alpha: Optional[torch.Tensor] = None,
                row_index: Optional[torch.Tensor] = None) -> torch.Tensor:
    """u = sum_s reader_in[s] x_s of the streams ``x`` float32 [rows, streams, hidden] (``reader_in`` None: their plain sum),
    as it is (``NEXT_SUM``) or through the norm tanh(alpha u) weight + bias (``NEXT_TANH``); rows gathered through
    ``row_index`` if given."""
    _dev(x, reader_in, weight, bias, alpha, row_index)
    _want(x, torch.float32, "x")
    if x.dim() != 3 or kind not in (NEXT_SUM, NEXT_TANH):
        raise KernelError(f"stream_read: the streams are {tuple(x.shape)}, kind {kind}")
    rows, streams, hidden = x.shape
    if row_index is not None:
        _want(row_index, torch.int32, "row_index")
        rows = row_index.numel()
    out = torch.empty((rows, hidden), dtype=out_dtype, device=x.device)
    _check(library().fw_stream_read(_p(x), streams, *_reader(kind, streams, hidden, reader_in, weight, bias, alpha), _p(row_index), _p(out),
                                    _code(out_dtype), rows, hidden, _stream()))
    return out


def stream_join_(x: torch.Tensor, ls: torch.Tensor, mix: torch.Tensor, out_weight: torch.Tensor, a: torch.Tensor, *,
                 branches: Optional[tuple] = None, chosen: Optional[tuple] = None, next_kind: int = NEXT_NOTHING,
                 next_in: Optional[torch.Tensor] = None, next_weight: Optional[torch.Tensor] = None,
                 next_bias: Optional[torch.Tensor] = None, next_alpha: Optional[torch.Tensor] = None,
                 next_dtype: Optional[torch.dtype] = None) -> Optional[torch.Tensor]:
    """In place on the streams ``x`` float32 [rows, streams, hidden]: x_t <- sum_s mix[s, t] x_s + out_weight[t] * (ls * y).
    y is ``a`` [rows, hidden]; with ``branches`` = (b, weight_a, weight_b, scale_a, scale_b, eps) it is scale_a rms(a) weight_a +
    scale_b rms(b) weight_b; with ``chosen`` = (choice_weight, pair_place, b or None, gate or None) it is the sum of the rows of
    ``a`` [places, hidden] that each row chose, in order, plus sigmoid(gate) b (``gate`` float32, one number a row, rows may lie
    apart; b [rows, hidden]). ``next_kind`` NEXT_SUM or NEXT_TANH: what reads the streams next (see ``stream_read``) is formed in
    the same kernel and returned in ``next_dtype``."""
    _dev(x, ls, mix, out_weight, a, next_in, next_weight, next_bias, next_alpha)
    for name, t in (("x", x), ("ls", ls), ("mix", mix), ("out_weight", out_weight), ("a", a)):
        _want(t, torch.float32, name)
    if x.dim() != 3:
        raise KernelError(f"stream_join: the streams are {tuple(x.shape)}, expected [rows, streams, hidden]")
    rows, streams, hidden = x.shape
    if ls.shape != (hidden,) or mix.shape != (streams, streams) or out_weight.shape != (streams,) or next_kind not in (NEXT_NOTHING, NEXT_SUM, NEXT_TANH):
        raise KernelError(f"stream_join: streams {tuple(x.shape)}, scales {tuple(ls.shape)}, mix {tuple(mix.shape)}, kind {next_kind}")
    source, b, weight_a, weight_b, scale_a, scale_b, eps = SOURCE_ROWS, None, None, None, 1.0, 1.0, 0.0
    choice_weight, pair_place, top, gate = None, None, 0, None
    places = rows
    if branches is not None:
        source = SOURCE_BRANCHES
        b, weight_a, weight_b, scale_a, scale_b, eps = branches
        for name, t, shape in (("b", b, (rows, hidden)), ("weight_a", weight_a, (hidden,)), ("weight_b", weight_b, (hidden,))):
            _dev(t)
            if t is None or t.dtype != torch.float32 or t.shape != shape:
                raise KernelError(f"stream_join: {name} must be float32 {shape}")
    elif chosen is not None:
        source = SOURCE_CHOSEN
        choice_weight, pair_place, b, gate = chosen
        _dev(choice_weight, pair_place, b)
        _want(choice_weight, torch.float32, "choice_weight")
        _want(pair_place, torch.int32, "pair_place")
        top = choice_weight.shape[1]
        places = rows * top
        if choice_weight.shape != (rows, top) or pair_place.shape != (rows, top):
            raise KernelError(f"stream_join: weights {tuple(choice_weight.shape)} and places {tuple(pair_place.shape)} of {rows} rows")
        if b is not None and (b.dtype != torch.float32 or b.shape != (rows, hidden)):
            raise KernelError(f"stream_join: b is {tuple(b.shape)}, expected float32 {(rows, hidden)}")
        if gate is not None:
            _dev_rows(gate, "gate")
            if b is None or gate.dtype != torch.float32 or gate.shape != (rows, 1):
                raise KernelError(f"stream_join: a gate is one float32 number a row beside rows to gate, found {tuple(gate.shape)}")
    if a.shape != (places, hidden):
        raise KernelError(f"stream_join: a is {tuple(a.shape)}, expected {(places, hidden)}")
    out = torch.empty((rows, hidden), dtype=next_dtype or torch.float32, device=x.device) if next_kind != NEXT_NOTHING else None
    _check(library().fw_stream_join(
        _p(x), streams, _p(ls), _p(mix), _p(out_weight), source, _p(a), _p(b), _p(weight_a), _p(weight_b), float(scale_a),
        float(scale_b), float(eps), _p(choice_weight), _p(pair_place), int(top), _p(gate),
        _stride(gate) if gate is not None else 0, *_reader(next_kind, streams, hidden, next_in, next_weight, next_bias, next_alpha), _p(out),
        _code(out.dtype) if out is not None else F32, rows, hidden, _stream()))
    return out


# ---- a linear recurrence over a matrix state per head with a fixed decay -------------------------------------------------
def _segments(name: str, segments: int, seg_row0: torch.Tensor, seg_slot: torch.Tensor) -> None:
    _dev(seg_row0, seg_slot)
    for which, t, n in (("seg_row0", seg_row0, segments + 1), ("seg_slot", seg_slot, segments)):
        _want(t, torch.int32, which)
        if t.numel() < n:
            raise KernelError(f"{name}: {which} holds {t.numel()} entries, needs {n}")


MAX_DECAY_DIM = 256      # key channels of a head


def _chunks(name: str, chunks: Optional[tuple], segments: int):
    """(chunk_seg, chunk_row0, seg_chunk0, rows beyond which a segment is walked in chunks, whether every segment of the step is
    that long) -> a launch's arguments: the arrays, their number, the rows, the flag."""
    if chunks is None:
        return (None, None, None), 0, 0, 0
    chunk_seg, chunk_row0, seg_chunk0, long_rows, all_long = chunks
    _dev(chunk_seg, chunk_row0, seg_chunk0)
    count = chunk_seg.numel()
    for which, t, n in (("chunk_seg", chunk_seg, count), ("chunk_row0", chunk_row0, count), ("seg_chunk0", seg_chunk0, segments + 1)):
        _want(t, torch.int32, which)
        if t.numel() < n:
            raise KernelError(f"{name}: {which} holds {t.numel()} entries, needs {n}")
    return (chunk_seg, chunk_row0, seg_chunk0), count, int(long_rows), int(all_long)


DECAY_CHUNK = 64        # rows of a chunk, as the kernels have them


def decay_powers(decays, device) -> torch.Tensor:
    """decay^0 .. decay^chunk of every head, formed in float64: float32 [heads, chunk + 1]."""
    if library().fw_decay_chunk_rows() != DECAY_CHUNK or library().fw_scan_chunk_rows() != DECAY_CHUNK:
        raise KernelError("the kernel library's chunks are of another length")
    exponents = torch.arange(DECAY_CHUNK + 1, dtype=torch.float64)
    return torch.pow(torch.as_tensor(decays, dtype=torch.float64)[:, None], exponents[None, :]).to(dtype=torch.float32, device=device)


def decay_recurrence(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, powers: torch.Tensor, state: torch.Tensor, seg_row0: torch.Tensor,
                     seg_slot: torch.Tensor, segments: int, heads: int, dim: int, vdim: int, chunks: Optional[tuple] = None) -> torch.Tensor:
    """Per head S <- decay S + silu(k) silu(v)^T, o = S^T silu(q) over each segment's rows in order. ``q``, ``k`` float32
    [rows, heads dim] and ``v`` [rows, heads vdim] with one row stride (views of wider rows will do); ``powers``: see
    ``decay_powers``; ``state`` float32 [slots, heads, dim, vdim] is read and moved on. ``chunks`` (chunk_seg, chunk_row0, seg_chunk0,
    long_rows, whether every segment is longer than that): segments of more than long_rows rows are walked in these chunks side by side. Returns float32 [rows, heads vdim]."""
    _dev(powers, state)
    _segments("decay_recurrence", segments, seg_row0, seg_slot)
    rows = q.shape[0]
    for name, t, width in (("q", q, heads * dim), ("k", k, heads * dim), ("v", v, heads * vdim)):
        _dev_rows(t, name)
        _want(t, torch.float32, name)
        if t.shape != (rows, width):
            raise KernelError(f"decay_recurrence: {name} is {tuple(t.shape)}, expected {(rows, width)}")
    if rows > 1 and not (q.stride(0) == k.stride(0) == v.stride(0)):
        raise KernelError("decay_recurrence: q, k and v have one row stride")
    stride = max(_stride(q), _stride(k), _stride(v))
    for name, t, shape in (("powers", powers, (heads, DECAY_CHUNK + 1)), ("state", state[0], (heads, dim, vdim))):
        _want(t, torch.float32, name)
        if t.shape != shape:
            raise KernelError(f"decay_recurrence: {name} is {tuple(t.shape)}, expected {shape}")
    out = torch.empty((rows, heads * vdim), dtype=torch.float32, device=q.device)
    places, count, *how = _chunks("decay_recurrence", chunks, segments)
    workspace = torch.empty((count, heads, dim, vdim), dtype=torch.float32, device=q.device) if count else None
    _check(library().fw_decay_recurrence(_p(q), _p(k), _p(v), stride, _p(powers), _p(state), state.shape[0], _p(out), _p(seg_row0),
                                         _p(seg_slot), rows, int(segments), heads, dim, vdim, *(_p(t) for t in places), count, *how,
                                         _p(workspace), _stream()))
    return out


# ---- the selective scan ---------------------------------------------------------------------------------------------
MAX_SCAN_STATES = 128


def selective_scan(x: torch.Tensor, z: torch.Tensor, bc: torch.Tensor, gate: torch.Tensor, A2: torch.Tensor, D: torch.Tensor,
                   state: torch.Tensor, seg_row0: torch.Tensor, seg_slot: torch.Tensor, segments: int, out_dtype: torch.dtype,
                   chunks: Optional[tuple] = None) -> torch.Tensor:
    """Per channel c and state n, with dt = softplus(z): S <- 2^(dt A2[n, c]) S + dt x B[n], y = sum_n S C[n] + D x, out = y *
    silu(gate), over each segment's rows in order. ``x``, ``z``, ``gate`` float32 [rows, channels], ``bc`` float32 [rows, 2 states]
    (B, then C); rows may lie apart. ``A2`` [states, channels] and ``D`` [channels] float32; ``state`` float32 [slots, states,
    channels] is read and moved on. ``chunks``: as for ``decay_recurrence``. Returns [rows, channels] of ``out_dtype``."""
    _dev(A2, D, state)
    _segments("selective_scan", segments, seg_row0, seg_slot)
    rows, channels = x.shape
    states = A2.shape[0]
    for name, t, shape in (("x", x, (rows, channels)), ("z", z, (rows, channels)), ("bc", bc, (rows, 2 * states)), ("gate", gate, (rows, channels))):
        _dev_rows(t, name)
        _want(t, torch.float32, name)
        if t.shape != shape:
            raise KernelError(f"selective_scan: {name} is {tuple(t.shape)}, expected {shape}")
    for name, t, shape in (("A2", A2, (states, channels)), ("D", D, (channels,)), ("state", state[0], (states, channels))):
        _want(t, torch.float32, name)
        if t.shape != shape:
            raise KernelError(f"selective_scan: {name} is {tuple(t.shape)}, expected {shape}")
    out = torch.empty((rows, channels), dtype=out_dtype, device=x.device)
    places, count, *how = _chunks("selective_scan", chunks, segments)
    workspace = torch.empty((count, states + 1, channels), dtype=torch.float32, device=x.device) if count else None
    _check(library().fw_selective_scan(_p(x), _stride(x), _p(z), _stride(z), _p(bc), _stride(bc), _p(gate), _stride(gate), _p(A2), _p(D), _p(state),
                                       state.shape[0], _p(out), _code(out_dtype), _p(seg_row0), _p(seg_slot), rows, int(segments), channels,
                                       states, *(_p(t) for t in places), count, *how, _p(workspace), _stream()))
    return out


def low_rank_weights(w: torch.Tensor) -> torch.Tensor:
    """A map [channels, rank] as ``selective_scan_low_rank`` reads it: [rank, channels], or of bfloat16 [rank / 2, channels, 2]."""
    channels, rank = w.shape
    if w.dtype == torch.bfloat16 and rank % 2 == 0:
        return w.view(channels, rank // 2, 2).permute(1, 0, 2).contiguous()
    return w.to(torch.float32).t().contiguous()


def selective_scan_low_rank(x: torch.Tensor, low: torch.Tensor, w: torch.Tensor, bias: torch.Tensor, gate: torch.Tensor, A2: torch.Tensor,
                            D: torch.Tensor, state: torch.Tensor, seg_slot: torch.Tensor, out_dtype: torch.dtype) -> torch.Tensor:
    """``selective_scan`` over segments of one row each (row r is segment r), with the map in front of the step sizes: z = low[:,
    :rank] . W^T + bias. ``low`` float32 [rows, rank + 2 states] (the low part, B, C; rows may lie apart); ``w`` from
    ``low_rank_weights``."""
    _dev(A2, D, state, w, bias, seg_slot)
    _want(seg_slot, torch.int32, "seg_slot")
    rows, channels = x.shape
    states = A2.shape[0]
    rank = w.shape[0] * (2 if w.dim() == 3 else 1)
    for name, t, shape in (("x", x, (rows, channels)), ("low", low, (rows, rank + 2 * states)), ("gate", gate, (rows, channels))):
        _dev_rows(t, name)
        _want(t, torch.float32, name)
        if t.shape != shape:
            raise KernelError(f"selective_scan_low_rank: {name} is {tuple(t.shape)}, expected {shape}")
    for name, t, shape in (("A2", A2, (states, channels)), ("D", D, (channels,)), ("bias", bias, (channels,)), ("state", state[0], (states, channels))):
        _want(t, torch.float32, name)
        if t.shape != shape:
            raise KernelError(f"selective_scan_low_rank: {name} is {tuple(t.shape)}, expected {shape}")
    if w.shape != ((rank // 2, channels, 2) if w.dim() == 3 else (rank, channels)) or w.dtype != (torch.bfloat16 if w.dim() == 3 else torch.float32) \
            or seg_slot.numel() < rows:
        raise KernelError(f"selective_scan_low_rank: w is {tuple(w.shape)} {w.dtype}, {seg_slot.numel()} slots for {rows} rows")
    out = torch.empty((rows, channels), dtype=out_dtype, device=x.device)
    _check(library().fw_selective_scan_low_rank(_p(x), _stride(x), _p(low), _stride(low), rank, _p(w), _code(w.dtype), _p(bias), _p(gate),
                                                _stride(gate), _p(A2), _p(D), _p(state), state.shape[0], _p(out), _code(out_dtype),
                                                _p(seg_slot), rows, channels, states, _stream()))
    return out
