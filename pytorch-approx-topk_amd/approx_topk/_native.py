"""ctypes binding of libapprox_topk_hip.so (the C ABI in include/approx_topk_hip.h).

The library is built in-tree by ``pytorch-approx-topk_amd/build.py`` and sits
next to this file, as does ``_host.so`` (csrc/host_binding.cpp), which makes the
common calls without Python in between: contiguous rows of plain tensors.  There
is no fallback: if either cannot be loaded, every call that needs them raises.
"""
from __future__ import annotations

import ctypes
import functools
import importlib
import os
import sysconfig

import torch

INTERLEAVED, BALANCED, CEIL_CHUNK, INTERLEAVED_PADDED = 0, 1, 2, 3

DTYPE_CODE = {
    torch.float32: 0, torch.float16: 1, torch.bfloat16: 2, torch.float64: 3,
    torch.uint8: 4, torch.int8: 5, torch.int16: 6, torch.int32: 7, torch.int64: 8,
}

ABI_VERSION = 3
LIB_NAME = "libapprox_topk_hip.so"

_SIGNATURES = {
    # name: (restype, argtypes)
    "atk_version": (ctypes.c_int, []),
    "atk_strerror": (ctypes.c_char_p, [ctypes.c_int]),
    "atk_stage1_workspace_bytes": (ctypes.c_size_t, [ctypes.c_int64] * 3 + [ctypes.c_int] * 3),
    "atk_stage1": (ctypes.c_int, [ctypes.c_void_p] + [ctypes.c_int64] * 4 + [ctypes.c_int] * 3
                   + [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t,
                      ctypes.c_void_p]),
    "atk_stage1_i32": (ctypes.c_int, [ctypes.c_void_p] + [ctypes.c_int64] * 4 + [ctypes.c_int] * 3
                       + [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t,
                          ctypes.c_void_p]),
    "atk_select_workspace_bytes": (ctypes.c_size_t, [ctypes.c_int64] * 3 + [ctypes.c_int]),
    "atk_select": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_void_p] + [ctypes.c_int64] * 4
                   + [ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p,
                      ctypes.c_size_t, ctypes.c_void_p]),
    "atk_topk_workspace_bytes": (ctypes.c_size_t, [ctypes.c_int64] * 3 + [ctypes.c_int, ctypes.c_int64,
                                                                          ctypes.c_int, ctypes.c_int]),
    "atk_topk_workspace_bytes_at": (ctypes.c_size_t, [ctypes.c_void_p] + [ctypes.c_int64] * 4
                                    + [ctypes.c_int, ctypes.c_int64, ctypes.c_int, ctypes.c_int]),
    "atk_topk_workspace_bytes_used": (ctypes.c_size_t, [ctypes.c_void_p] + [ctypes.c_int64] * 4
                                      + [ctypes.c_int, ctypes.c_int64, ctypes.c_int, ctypes.c_int]),
    "atk_topk": (ctypes.c_int, [ctypes.c_void_p] + [ctypes.c_int64] * 4 + [ctypes.c_int, ctypes.c_int64,
                                                                           ctypes.c_int, ctypes.c_int]
                 + [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t,
                    ctypes.c_void_p]),
    "atk_describe": (ctypes.c_int, [ctypes.c_void_p] + [ctypes.c_int64] * 4
                     + [ctypes.c_int, ctypes.c_int64, ctypes.c_int, ctypes.c_int]
                     + [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_char_p, ctypes.c_size_t]),
    "atk_topk_noalloc": (ctypes.c_int, [ctypes.c_void_p] + [ctypes.c_int64] * 4
                         + [ctypes.c_int, ctypes.c_int64, ctypes.c_int, ctypes.c_int]
                         + [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p]),
    "atk_topk_grad": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_void_p] + [ctypes.c_int64] * 3
                      + [ctypes.c_int, ctypes.c_int64, ctypes.c_int, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p]),
    "atk_topk_i32": (ctypes.c_int, [ctypes.c_void_p] + [ctypes.c_int64] * 4 + [ctypes.c_int, ctypes.c_int64,
                                                                               ctypes.c_int, ctypes.c_int]
                     + [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t,
                        ctypes.c_void_p]),
}


_HOST_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "_host.so")


def _import_host():
    """(_host.so, None), or (None, what is wrong with it).  It is linked against torch: one that was built for
    another torch or Python is not loaded, and what needs no native code goes on without it."""
    if not os.path.exists(_HOST_PATH):
        return None, "is missing"
    built_for = f"approx_topk for torch {torch.__version__}, {sysconfig.get_config_var('SOABI')};"
    with open(_HOST_PATH, "rb") as f:
        if built_for.encode() not in f.read():
            return None, f"is not built for torch {torch.__version__} and this Python"
    try:
        return importlib.import_module("._host", __package__), None
    except ImportError as e:
        return None, f"cannot be loaded ({e})"


# (imported with the package: it registers the operators' kernels for the GPU)
host, _host_fault = _import_host()


def library_path() -> str:
    return os.environ.get("APPROX_TOPK_HIP_LIB") or os.path.join(
        os.path.dirname(os.path.abspath(__file__)), LIB_NAME)


@functools.cache
def lib() -> ctypes.CDLL:
    path = library_path()
    if not os.path.exists(path):
        raise RuntimeError(
            f"approx_topk: {path} is missing. Build it with "
            "`python pytorch-approx-topk_amd/build.py` (needs hipcc); there is no fallback path.")
    handle = ctypes.CDLL(path)
    for name, (restype, argtypes) in _SIGNATURES.items():
        fn = getattr(handle, name)
        fn.restype, fn.argtypes = restype, argtypes
    if handle.atk_version() != ABI_VERSION:
        raise RuntimeError(f"approx_topk: {path} has ABI {handle.atk_version()}, expected {ABI_VERSION}")
    if host is None:
        raise RuntimeError(
            f"approx_topk: {_HOST_PATH} {_host_fault}. Build it with `python pytorch-approx-topk_amd/build.py`; "
            "there is no fallback path.")
    host.bind({name: ctypes.cast(getattr(handle, name), ctypes.c_void_p).value for name in _SIGNATURES})
    return handle


def check(status: int) -> None:
    if status != 0:
        raise RuntimeError(lib().atk_strerror(status).decode())


def dtype_code(dtype: torch.dtype) -> int:
    try:
        return DTYPE_CODE[dtype]
    except KeyError:
        raise RuntimeError(f"approx_topk: unsupported dtype {dtype}") from None


def require_gpu(xs: torch.Tensor) -> None:
    if xs.device.type != "cuda":
        raise RuntimeError(
            f"approx_topk: expected a tensor on a GPU, got device {xs.device}; "
            "the HIP kernels have no CPU path")


def _stream(device: torch.device) -> int:
    """Raw handle of the current stream of `device` (no Python stream object is built)."""
    return torch._C._cuda_getCurrentRawStream(device.index)


class _NoGuard:
    def __enter__(self):
        return None

    def __exit__(self, *exc):
        return False


_NO_GUARD = _NoGuard()


def _on_device(device: torch.device):
    """Makes `device` current for a native call; free when it already is."""
    return _NO_GUARD if device.index == torch.cuda.current_device() else torch.cuda.device(device)


@functools.lru_cache(maxsize=4096)
def _stage1_workspace(rows: int, n: int, k0: int, j: int, layout: int, code: int) -> int:
    return lib().atk_stage1_workspace_bytes(rows, n, k0, j, layout, code)


@functools.lru_cache(maxsize=4096)
def _topk_workspace(misalign: int, rows: int, n: int, step: int, k0: int, j: int, k: int, layout: int,
                    code: int) -> int:
    # the library only looks at the address's alignment: any address with the same one stands for it
    return lib().atk_topk_workspace_bytes_used(4096 + misalign, rows, n, step, k0, j, k, layout, code)


def rows_view(xs: torch.Tensor) -> tuple[torch.Tensor, int, int, int]:
    """(tensor, rows, n, row_stride) with the top-k dim last and unit stride.

    Rows may be spaced by any uniform stride >= n (e.g. a column slice of a
    matrix); anything else is made contiguous.
    """
    n = xs.shape[-1]
    rows = xs.numel() // n if n else 0
    if xs.is_contiguous():  # without walking the strides
        return xs, rows, n, n
    if xs.ndim == 1:
        return (xs if xs.stride(0) == 1 or n <= 1 else xs.contiguous()), rows, n, n
    uniform = xs.stride(-1) == 1 or n <= 1
    step = xs.stride(-2)
    expect = step
    for d in range(xs.ndim - 2, -1, -1):
        if xs.shape[d] != 1 and xs.stride(d) != expect:
            uniform = False
        expect *= xs.shape[d]
    if not uniform or step < n:
        xs = xs.contiguous()
        step = n
    return xs, rows, n, step


def _call_constants(xs: torch.Tensor, k_out: int, two_stage: bool, index_dtype: torch.dtype):
    """(rows, n, dtype code, output shape, entry point) of a call that the native host module hands on: rows at a pitch
    of their own, copies of what has none, tensors that are more than plain ones, and a process's first call.
    (Nothing is kept by the call's arguments: 8 and 8.0 are one key, and only one of them a size.)"""
    L = lib()
    n = xs.shape[-1]
    rows = xs.numel() // n if n else 0
    narrow = index_dtype != torch.int64
    if two_stage:
        entry = L.atk_topk_i32 if narrow else L.atk_topk
    else:
        entry = L.atk_stage1_i32 if narrow else L.atk_stage1
    return rows, n, dtype_code(xs.dtype), (*xs.shape[:-1], k_out), entry


def stage1(xs: torch.Tensor, k0: int, j: int, layout: int, index_dtype: torch.dtype = torch.int64,
           want_values: bool = True) -> tuple[torch.Tensor | None, torch.Tensor]:
    """Per-bucket top-j along the last dim: (values[..., k0], indices[..., k0]).

    ``index_dtype``: torch.int64 (the operator's contract) or torch.int32.
    ``want_values=False``: only the indices are written; values is None."""
    require_gpu(xs)
    if host is not None:
        out = host.run(xs, k0, j, k0, layout, index_dtype != torch.int64, want_values, False)
        if out is not None:
            return out
    step = None
    if not xs.is_contiguous():
        xs, _, _, step = rows_view(xs)
    rows, n, code, shape, entry = _call_constants(xs, k0, False, index_dtype)
    device = xs.device
    values = torch.empty(shape, dtype=xs.dtype, device=device) if want_values else None
    indices = torch.empty(shape, dtype=index_dtype, device=device)
    with _on_device(device):
        need = _stage1_workspace(rows, n, k0, j, layout, code)
        ws = torch.empty(need, dtype=torch.uint8, device=device) if need else None
        status = entry(xs.data_ptr(), rows, n, n if step is None else step, k0, j, layout, code,
                       values.data_ptr() if want_values else None, indices.data_ptr(),
                       ws.data_ptr() if ws is not None else None, need, _stream(device))
    if status != 0:
        check(status)
    return values, indices


def select(cand_values: torch.Tensor, cand_indices: torch.Tensor, k: int,
           index_bound: int) -> tuple[torch.Tensor, torch.Tensor]:
    """Exact top-k of candidates along the last dim, in candidate order."""
    require_gpu(cand_values)
    L = lib()
    cv, ci = cand_values.contiguous(), cand_indices.contiguous()
    k0 = cv.shape[-1]
    rows = cv.numel() // k0 if k0 else 0
    code = dtype_code(cv.dtype)
    shape = list(cv.shape[:-1]) + [k]
    values = torch.empty(shape, dtype=cv.dtype, device=cv.device)
    indices = torch.empty(shape, dtype=torch.int64, device=cv.device)
    with _on_device(cv.device):
        need = L.atk_select_workspace_bytes(rows, k0, k, code)
        ws = torch.empty(need, dtype=torch.uint8, device=cv.device) if need else None
        check(L.atk_select(cv.data_ptr(), ci.data_ptr(), rows, k0, k, index_bound, code,
                           values.data_ptr(), indices.data_ptr(),
                           ws.data_ptr() if ws is not None else None, need, _stream(cv.device)))
    return values, indices


def topk(xs: torch.Tensor, k0: int, j: int, k: int, layout: int, index_dtype: torch.dtype = torch.int64,
         want_values: bool = True) -> tuple[torch.Tensor | None, torch.Tensor]:
    """Stage 1 (k0 candidates) and stage 2 (k survivors) along the last dim."""
    require_gpu(xs)
    if host is not None:
        out = host.run(xs, k0, j, k, layout, index_dtype != torch.int64, want_values, True)
        if out is not None:
            return out
    step = None
    if not xs.is_contiguous():
        xs, _, _, step = rows_view(xs)
    rows, n, code, shape, entry = _call_constants(xs, k, True, index_dtype)
    device = xs.device
    values = torch.empty(shape, dtype=xs.dtype, device=device) if want_values else None
    indices = torch.empty(shape, dtype=index_dtype, device=device)
    with _on_device(device):
        pitch = n if step is None else step
        need = _topk_workspace(xs.data_ptr() % 16, rows, n, pitch, k0, j, k, layout, code)
        ws = torch.empty(need, dtype=torch.uint8, device=device) if need else None
        status = entry(xs.data_ptr(), rows, n, pitch, k0, j, k, layout, code,
                       values.data_ptr() if want_values else None, indices.data_ptr(),
                       ws.data_ptr() if ws is not None else None, need, _stream(device))
    if status != 0:
        check(status)
    return values, indices


# Longest row topk_grad takes.
MAX_GRAD_ROW = (1 << 31) - 1


def check_grad_tensors(grad_values: torch.Tensor, indices: torch.Tensor) -> None:
    """What the gradient's kernel takes for granted: it reads as many gradients as indices, of eight bytes."""
    if (indices.dtype is not torch.int64 or grad_values.shape != indices.shape or indices.ndim == 0
            or grad_values.device != indices.device):
        raise RuntimeError(
            "topk_grad: expected int64 indices and gradients of the same shape on one device, got "
            f"{indices.dtype} {tuple(indices.shape)} on {indices.device} and {tuple(grad_values.shape)} on "
            f"{grad_values.device}")


def topk_grad(grad_values: torch.Tensor, indices: torch.Tensor, n: int, k0: int, j: int, layout: int) -> torch.Tensor:
    """The gradient of a call's values with respect to its input (top-k along the last dim of `n`
    elements), given the call's indices: zero but for the selected positions."""
    check_grad_tensors(grad_values, indices)
    require_gpu(grad_values)
    grad_values, indices = grad_values.contiguous(), indices.contiguous()
    shape = indices.shape
    grad_x = grad_values.new_empty((*shape[:-1], n))
    entries, k = indices.numel(), shape[-1]
    if entries == 0:
        return grad_x.zero_()
    device = grad_values.device
    with _on_device(device):
        status = lib().atk_topk_grad(grad_values.data_ptr(), indices.data_ptr(), entries // k, n, k0, j, k, layout,
                                     dtype_code(grad_values.dtype), grad_x.data_ptr(), _stream(device))
    if status != 0:
        check(status)
    return grad_x


def describe(xs: torch.Tensor, k0: int, j: int, k: int, layout: int = INTERLEAVED,
             values: torch.Tensor | None = None, indices: torch.Tensor | None = None) -> str:
    """The kernels a call on `xs` (top-k along the last dim) would launch, as text.

    `values` and `indices`: the buffers the call will write, checked like the call's; the plan does not
    depend on them."""
    xs, rows, n, step = rows_view(xs)
    buf = ctypes.create_string_buffer(1024)
    check(lib().atk_describe(xs.data_ptr() if xs.numel() else 4096, rows, n, step, k0, j, k, layout,
                             dtype_code(xs.dtype), values.data_ptr() if values is not None else 4096,
                             indices.data_ptr() if indices is not None else 4096, buf, len(buf)))
    return buf.value.decode()
