"""Python mirror of the reference operator interface.

Reference (paths relative to the reference repository root):
``results/naive_cycle4/include/playground/matmul.hpp:11-23``::

    template <typename DType, uint8_t Version>
    void matmul(size_t m, size_t n, size_t k, const DType* A, const DType* B, DType* C);
    #define PLAYGOUND_MATMUL_CALL(Version, m, n, k, A, B, C) \
        matmul<remove_cvref_t<decltype(*A)>, Version>(m, n, k, A, B, C)

:func:`matmul` keeps the argument order and meaning: ``m, n, k`` then row-major
``A`` (m x k), ``B`` (k x n) and the output ``C`` (m x n), which is fully
overwritten (alpha = 1, beta = 0).  As in ``PLAYGOUND_MATMUL_CALL`` the input
dtype comes from ``A``; the output dtype comes from ``C`` (fp16 as in the
reference, or fp32).  Operands are device tensors; the call is asynchronous on
the current stream (or ``stream``).  Where the reference returns void with no
error channel, this raises :class:`VkError`.

Every call goes through libvk_gemm.so; there is no other implementation.
"""
from __future__ import annotations

from . import _abi
from ._abi import DTYPE_F16, DTYPE_F32, VkError


def _torch():
    import torch  # imported lazily: the ABI layer itself does not need torch
    return torch


_DTYPE_CODES = None


def _dtype_code(t) -> int:
    global _DTYPE_CODES
    if _DTYPE_CODES is None:
        torch = _torch()
        _DTYPE_CODES = {torch.float16: DTYPE_F16, torch.float32: DTYPE_F32}
    code = _DTYPE_CODES.get(t.dtype)
    if code is None:
        raise VkError(-2, f"unsupported dtype {t.dtype}")
    return code


def _stream_handle(stream, device) -> int:
    if stream is not None:
        return stream.cuda_stream
    torch = _torch()
    raw = getattr(torch._C, "_cuda_getCurrentRawStream", None)  # no Stream object: 1.7 us less per call
    return raw(device.index) if raw is not None else torch.cuda.current_stream(device).cuda_stream


def matmul(m: int, n: int, k: int, A, B, C, version: int, stream=None) -> None:
    """C = A . B with kernel ``version`` (row-major, fp32 accumulation)."""
    if not (A.is_cuda and B.is_cuda and C.is_cuda and A.is_contiguous() and B.is_contiguous() and C.is_contiguous()):
        for name, t in (("A", A), ("B", B), ("C", C)):
            if not t.is_cuda:
                raise VkError(-5, f"{name} must be a device tensor")
            if not t.is_contiguous():
                raise VkError(-4, f"{name} must be contiguous (row-major, dense)")
    if A.numel() < m * k or B.numel() < k * n or C.numel() < m * n:
        raise VkError(-3, "operand smaller than m x k / k x n / m x n")
    in_dt = _dtype_code(A)
    if _dtype_code(B) != in_dt:
        raise VkError(-2, "A and B must have the same dtype")
    out_dt = _dtype_code(C)
    st = _abi.gemm(version, in_dt, out_dt, m, n, k, A.data_ptr(), B.data_ptr(), C.data_ptr(),
                   _stream_handle(stream, C.device))
    if st != _abi.VK_OK:
        raise VkError(st, f"matmul(version={version}, m={m}, n={n}, k={k})")


def gemm(A, B, version: int | None = None, out_dtype=None, stream=None):
    """Allocate C and run :func:`matmul`; A is (m, k), B is (k, n).  With no
    version, :func:`pick_version` chooses one for the shape and dtypes."""
    torch = _torch()
    m, k = A.shape
    k2, n = B.shape
    if k != k2:
        raise VkError(-3, f"inner dimensions differ: {k} vs {k2}")
    C = torch.empty((m, n), dtype=out_dtype or A.dtype, device=A.device)
    if version is None:
        dt = "f16" if A.dtype == torch.float16 else "f32"
        version = pick_version(m, n, k, dt, "f16" if C.dtype == torch.float16 else "f32")
    matmul(m, n, k, A, B, C, version, stream)
    return C


def versions(dtype: str = "f16", leave_one_out: bool = False) -> list:
    """The library's versions for an input dtype; the leave-one-out instances
    of version 7 (fp16 71-77, measurement only) only when asked for."""
    vs = _abi.versions(DTYPE_F16 if dtype == "f16" else DTYPE_F32)
    if dtype == "f16" and not leave_one_out:
        vs = [v for v in vs if v not in _abi.LEAVE_ONE_OUT]
    return vs


def name(version: int, dtype: str = "f16"):
    return _abi.name(version, DTYPE_F16 if dtype == "f16" else DTYPE_F32)


def query(version: int, dtype: str = "f16"):
    return _abi.query(version, DTYPE_F16 if dtype == "f16" else DTYPE_F32)


def pick_version(m: int, n: int, k: int, dtype: str = "f16", out: str | None = None) -> int:
    """The fastest version that accepts this shape with 4 KiB-aligned operands
    on the current device (an MI355X's 256 compute units with none visible);
    the rule and its measurements are vk_gemm_pick's.  The reference picks
    versions at build time only (CMakeLists.txt MATMUL_VERSION)."""
    in_dt = DTYPE_F16 if dtype == "f16" else DTYPE_F32
    out_dt = DTYPE_F16 if (out or dtype) == "f16" else DTYPE_F32
    version = _abi.pick(in_dt, out_dt, m, n, k)
    if version < 0:
        raise VkError(version, f"no {dtype} version accepts m={m}, n={n}, k={k} with {out or dtype} output")
    return version
