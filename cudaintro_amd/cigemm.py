"""ctypes binding of ``include/cigemm.h``.

Every GEMM method takes device tensors (``torch.Tensor`` on the GPU), passes their raw
pointers, sizes and strides through the C ABI and returns the output tensor.  Failures of
the library raise :class:`CigemmError` carrying the status name and the handle's message.
"""
from __future__ import annotations

import ctypes as C
import enum
import os
import subprocess

_HERE = os.path.dirname(os.path.abspath(__file__))
_LIB = os.path.join(_HERE, "libcigemm.so")
_SUITE = os.path.join(_HERE, "gemm_suite")

B_KN, B_NK = 0, 1
ACT_NONE, ACT_RELU = 0, 1
ALGO_DEFAULT, ALGO_GENERIC, ALGO_TILE, ALGO_SKINNY, ALGO_SMALL, ALGO_MFMA_ANY = -1, 0, 1, 2, 3, 4
SCALE_TENSOR, SCALE_VECTOR = 0, 1
OUT_F32, OUT_BF16 = 0, 1


class Status(enum.IntEnum):
    SUCCESS = 0
    NOT_INITIALIZED = 1
    ALLOC_FAILED = 3
    INVALID_VALUE = 7
    ARCH_MISMATCH = 8
    MAPPING_ERROR = 11
    EXECUTION_FAILED = 13
    INTERNAL_ERROR = 14
    NOT_SUPPORTED = 15
    LICENSE_ERROR = 16


class CigemmError(RuntimeError):
    def __init__(self, status: int, message: str, where: str):
        self.status = Status(status) if status in Status._value2member_map_ else status
        name = getattr(self.status, "name", str(status))
        super().__init__(f"{where}: CIGEMM_STATUS_{name}" + (f" ({message})" if message else ""))


def library_path() -> str:
    return _LIB


def suite_path() -> str:
    return _SUITE


def build_library(jobs: int = 8) -> str:
    """Compile the HIP sources in ``csrc/`` for gfx950 (works without a GPU)."""
    subprocess.run(["make", "-C", os.path.join(_HERE, "csrc"), f"-j{jobs}", "-B", "all"],
                   check=True)
    return _LIB


_lib = None

# name -> (restype, argtypes); must list every symbol include/cigemm.h declares.
_i64, _u64, _vp, _ci, _f32 = C.c_int64, C.c_uint64, C.c_void_p, C.c_int, C.c_float
SIGNATURES = {
    "cigemmCreate": (_ci, [C.POINTER(_vp)]),
    "cigemmDestroy": (_ci, [_vp]),
    "cigemmSetStream": (_ci, [_vp, _vp]),
    "cigemmGetStream": (_ci, [_vp, C.POINTER(_vp)]),
    "cigemmResetWorkspace": (_ci, [_vp]),
    "cigemmGetStatusString": (C.c_char_p, [_ci]),
    "cigemmGetLastErrorString": (C.c_char_p, [_vp]),
    "cigemmGetVersion": (_ci, []),
    "cigemmGetLastKernelName": (C.c_char_p, [_vp]),
    "cigemmGetLastPlan": (C.c_int, [_vp, C.POINTER(C.c_int), C.POINTER(C.c_int)]),
    "cigemm_matrixMulTiled": (C.c_int, [_vp, _vp, _vp, _vp, C.c_int]),
    "cigemm_matrixMulMatrixCores": (C.c_int, [_vp, _vp, _vp, _vp, C.c_int]),
    "cigemm_matrixMulMatrixCoresBfloat16": (C.c_int, [_vp, _vp, _vp, _vp, C.c_int]),
    "cigemmSetAlgo": (C.c_int, [_vp, C.c_int]),
    "cigemmGetAlgo": (C.c_int, [_vp, C.POINTER(C.c_int)]),
    "cigemm_gemm_f32": (_ci, [_vp, _i64, _i64, _i64, _vp, _i64, _vp, _i64, _vp, _i64]),
    "cigemm_gemm_f16": (_ci, [_vp, _i64, _i64, _i64, _vp, _i64, _vp, _i64, _vp, _i64]),
    "cigemm_gemm_bf16": (_ci, [_vp, _i64, _i64, _i64, _vp, _i64, _vp, _i64, _vp, _i64]),
    "cigemm_gemm_bf16_static": (_ci, [_vp, _i64, _i64, _i64, _vp, _i64, _vp, _i64, _vp, _i64,
                                      C.c_char_p, C.c_size_t]),
    "cigemm_gemm_i8_i32": (_ci, [_vp, _i64, _i64, _i64, _vp, _i64, _vp, _i64, _ci, _vp, _i64]),
    "cigemm_gemm_i8_dequant": (_ci, [_vp, _i64, _i64, _i64, _vp, _i64, _vp, _i64, _ci, _vp, _ci,
                                     _vp, _ci, _vp, _ci, _i64, _vp, _i64]),
    "cigemm_linear_f32": (_ci, [_vp, _i64, _i64, _i64, _vp, _i64, _vp, _i64, _vp, _ci, _vp, _i64]),
    "cigemm_fill_random_f32": (_ci, [_vp, _vp, _i64, _u64, _f32, _f32]),
    "cigemm_fill_random_bf16": (_ci, [_vp, _vp, _i64, _u64, _f32, _f32]),
    "cigemm_fill_random_f16": (_ci, [_vp, _vp, _i64, _u64, _f32, _f32]),
    "cigemm_fill_random_i8": (_ci, [_vp, _vp, _i64, _u64, _ci, _ci]),
    "cigemm_quantize_rows_i8": (_ci, [_vp, _i64, _i64, _vp, _i64, _vp, _i64, _vp]),
}


def load_library():
    """dlopen ``libcigemm.so`` (built in-tree) and declare the prototypes."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(_LIB):
        raise FileNotFoundError(
            f"{_LIB} is not built; run `python -c 'import __graft_entry__ as g; g.build()'` "
            "or `make -C cudaintro_amd/csrc all python`.  There is no CPU fallback.")
    lib = C.CDLL(_LIB)
    for name, (res, args) in SIGNATURES.items():
        fn = getattr(lib, name)
        fn.restype = res
        fn.argtypes = args
    _lib = lib
    return lib


def _torch():
    import torch
    return torch


_entries = None


def _native():
    """The binding of the hot calls in native code (``csrc/binding.cpp``), built beside the library."""
    _torch()  # (it is linked against torch's own libraries)
    try:
        from . import _binding
    except ImportError as e:
        raise FileNotFoundError(f"{os.path.join(_HERE, '_binding.so')} is not built or does not load ({e}); run "
                                "`python -c 'import __graft_entry__ as g; g.build()'`") from e
    return _binding


def _native_entries():
    """The attributes of a :class:`Handle` that its hot calls use: the binding's functions (``_n_``) and the
    library's entry points as addresses (``_p_``); looked up once."""
    global _entries
    if _entries is None:
        native, lib = _native(), load_library()
        _entries = {f"_n_{name}": getattr(native, name)
                    for name in ("gemm", "linear_f32", "gemm_i8_i32", "gemm_i8_dequant", "quantize_rows_i8")}
        for name in ("gemm_f32", "gemm_f16", "gemm_bf16", "linear_f32", "gemm_i8_i32", "gemm_i8_dequant",
                     "quantize_rows_i8"):
            _entries[f"_p_{name}"] = C.cast(getattr(lib, f"cigemm_{name}"), _vp).value
    return _entries


def gemm_bf16_static(A, B, out=None, stream=None):
    """``cigemm_gemm_bf16_static``: the decode-shape bf16 GEMM without a handle and without any
    allocation inside the library (``out`` is allocated here, by torch, when not given)."""
    torch = _torch()
    lib = load_library()
    assert A.dtype == torch.bfloat16 and B.dtype == torch.bfloat16
    M, K = A.shape
    K2, N = B.shape
    assert K == K2
    if out is None:
        out = torch.empty((M, N), dtype=torch.bfloat16, device=A.device)
    s = torch.cuda.current_stream() if stream is None else stream
    err = C.create_string_buffer(256)
    st = lib.cigemm_gemm_bf16_static(_vp(s.cuda_stream), M, N, K, A.data_ptr(), Handle._ld(A),
                                     B.data_ptr(), Handle._ld(B), out.data_ptr(), _out_ld(out, M, N, 2),
                                     err, len(err))
    if st != 0:
        raise CigemmError(st, err.value.decode(), "cigemm_gemm_bf16_static")
    return out


def _mat(t):
    """(rows, columns, leading dimension) of a matrix whose rows are contiguous."""
    s = t.stride()
    assert len(s) == 2
    rows, cols = t.shape
    assert cols <= 1 or s[1] == 1, "rows must be contiguous"
    return rows, cols, s[0] if rows > 1 else max(cols, s[0], 1)


def _out_ld(t, M, N, itemsize):
    """Leading dimension of an output with room for M x N elements of `itemsize` bytes."""
    rows, cols, ld = _mat(t)
    assert rows >= M and cols >= N and t.element_size() >= itemsize, "the output is too small"
    return ld


class Handle:
    """Owns one ``cigemmHandle_t`` bound to the current device and to torch's current stream."""

    def __init__(self, stream=None):
        self.lib = load_library()
        h = _vp()
        st = self.lib.cigemmCreate(C.byref(h))
        if st != 0:
            raise CigemmError(st, "", "cigemmCreate")
        self._h = h
        torch = _torch()
        self._f32, self._bf16, self._f16, self._i8 = (torch.float32, torch.bfloat16, torch.float16,
                                                      torch.int8)
        s = torch.cuda.current_stream() if stream is None else stream
        self.set_stream(s.cuda_stream)
        self._address = h.value  # the handle, for the native binding
        self.__dict__.update(_native_entries())

    # -- plumbing ---------------------------------------------------------------------------
    def close(self):
        if getattr(self, "_h", None):
            self.lib.cigemmDestroy(self._h)
            self._h = None
            self._address = 0  # (a null handle: the library answers NOT_INITIALIZED)

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        self.close()

    def _check(self, st, where):
        if st != 0:
            raise CigemmError(st, self.lib.cigemmGetLastErrorString(self._h).decode(), where)

    def set_stream(self, raw_stream: int):
        self._check(self.lib.cigemmSetStream(self._h, _vp(raw_stream)), "cigemmSetStream")

    def reset_workspace(self):
        """Zero the split-K arrival counters and exchange words (after a failure seen elsewhere)."""
        self._check(self.lib.cigemmResetWorkspace(self._h), "cigemmResetWorkspace")

    def set_algo(self, algo: int):
        """Restrict following GEMM calls to one kernel family (``ALGO_*``)."""
        self._check(self.lib.cigemmSetAlgo(self._h, algo), "cigemmSetAlgo")

    def get_algo(self) -> int:
        v = C.c_int(0)
        self._check(self.lib.cigemmGetAlgo(self._h, C.byref(v)), "cigemmGetAlgo")
        return v.value

    def algo(self, algo: int):
        """Context manager: ``with h.algo(ALGO_TILE): ...`` and back to the previous choice."""
        import contextlib

        @contextlib.contextmanager
        def scope():
            prev = self.get_algo()
            self.set_algo(algo)
            try:
                yield self
            finally:
                self.set_algo(prev)

        return scope()

    @property
    def raw(self):
        return self._h

    @property
    def last_kernel(self) -> str:
        return self.lib.cigemmGetLastKernelName(self._h).decode()

    @property
    def last_plan(self):
        """(tile rows, K ranges) of the last GEMM when the LDS-tiled kernel ran, else (0, 0)."""
        rows, splits = C.c_int(0), C.c_int(0)
        self._check(self.lib.cigemmGetLastPlan(self._h, C.byref(rows), C.byref(splits)),
                    "cigemmGetLastPlan")
        return rows.value, splits.value

    # -- GEMMs ------------------------------------------------------------------------------
    @staticmethod
    def _ld(t):
        return _mat(t)[2]

    # A small product takes as long as the host needs to issue it, so a call with its output given goes
    # through the native binding (us a call at the host's pace, in Python -> there: fp32 3 x 277 x 64
    # 5.1 -> 2.9, bf16 33 x 250 x 333 5.6 -> 3.1, quantizer and int8 product 2 x 5376 x 128 10.4 -> 5.7); what that does not
    # take (-1) and calls that allocate are done here.
    def _gemm(self, fn, name, A, B, out, out_dtype):
        M, K, lda = _mat(A)
        K2, N, ldb = _mat(B)
        assert K == K2
        if out is None:
            out = _torch().empty((M, N), dtype=out_dtype, device=A.device)
        self._check(fn(self._h, M, N, K, A.data_ptr(), lda, B.data_ptr(), ldb, out.data_ptr(),
                       _out_ld(out, M, N, A.element_size())), name)
        return out

    def gemm_f32(self, A, B, out=None):
        if out is not None:
            st = self._n_gemm(self._p_gemm_f32, self._address, 0, A, B, out)
            if st == 0:
                return out
            if st > 0:
                self._check(st, "cigemm_gemm_f32")
        f32 = self._f32
        assert A.dtype == f32 and B.dtype == f32
        return self._gemm(self.lib.cigemm_gemm_f32, "cigemm_gemm_f32", A, B, out, f32)

    def linear_f32(self, X, W, bias=None, act=ACT_NONE, out=None):
        """out = act(bias + X @ W) with W stored K x N (input-major)."""
        if out is not None:
            st = self._n_linear_f32(self._p_linear_f32, self._address, X, W, bias, act, out)
            if st == 0:
                return out
            if st > 0:
                self._check(st, "cigemm_linear_f32")
        f32 = self._f32
        assert X.dtype == f32 and W.dtype == f32
        M, K, ldx = _mat(X)
        K2, N, ldw = _mat(W)
        assert K == K2 and (bias is None or (bias.dtype == f32 and bias.numel() == N and bias.is_contiguous()))
        if out is None:
            out = _torch().empty((M, N), dtype=f32, device=X.device)
        st = self.lib.cigemm_linear_f32(self._h, M, N, K, X.data_ptr(), ldx, W.data_ptr(), ldw,
                                        bias.data_ptr() if bias is not None else None, act,
                                        out.data_ptr(), _out_ld(out, M, N, 4))
        if st:
            self._check(st, "cigemm_linear_f32")
        return out

    def gemm_f16(self, A, B, out=None):
        if out is not None:
            st = self._n_gemm(self._p_gemm_f16, self._address, 1, A, B, out)
            if st == 0:
                return out
            if st > 0:
                self._check(st, "cigemm_gemm_f16")
        f16 = self._f16
        assert A.dtype == f16 and B.dtype == f16
        return self._gemm(self.lib.cigemm_gemm_f16, "cigemm_gemm_f16", A, B, out, f16)

    # -- study kernels (TileProgramming demo) -------------------------------------------------
    def matrixMulTiled(self, A, B):
        torch = _torch()
        w = A.shape[0]
        assert A.dtype == torch.float32 and A.shape == (w, w) and B.shape == (w, w)
        assert A.is_contiguous() and B.is_contiguous()
        Cm = torch.empty((w, w), dtype=torch.float32, device=A.device)
        st = self.lib.cigemm_matrixMulTiled(self._h, Cm.data_ptr(), A.data_ptr(), B.data_ptr(), w)
        self._check(st, "cigemm_matrixMulTiled")
        return Cm

    def matrixMulMatrixCores(self, A, B):
        """A, B fp16 or bf16 square tensors; fp32 result."""
        torch = _torch()
        w = A.shape[0]
        assert A.dtype == B.dtype and A.dtype in (torch.float16, torch.bfloat16)
        assert A.shape == (w, w) and B.shape == (w, w) and A.is_contiguous() and B.is_contiguous()
        name = ("cigemm_matrixMulMatrixCores" if A.dtype == torch.float16
                else "cigemm_matrixMulMatrixCoresBfloat16")
        Cm = torch.empty((w, w), dtype=torch.float32, device=A.device)
        st = getattr(self.lib, name)(self._h, A.data_ptr(), B.data_ptr(), Cm.data_ptr(), w)
        self._check(st, name)
        return Cm

    def gemm_bf16(self, A, B, out=None):
        if out is not None:
            st = self._n_gemm(self._p_gemm_bf16, self._address, 2, A, B, out)
            if st == 0:
                return out
            if st > 0:
                self._check(st, "cigemm_gemm_bf16")
        bf16 = self._bf16
        assert A.dtype == bf16 and B.dtype == bf16
        return self._gemm(self.lib.cigemm_gemm_bf16, "cigemm_gemm_bf16", A, B, out, bf16)

    def gemm_i8_i32(self, A, B, b_layout=B_KN, out=None):
        if out is not None:
            st = self._n_gemm_i8_i32(self._p_gemm_i8_i32, self._address, A, B, b_layout, out)
            if st == 0:
                return out
            if st > 0:
                self._check(st, "cigemm_gemm_i8_i32")
        assert A.dtype == self._i8 and B.dtype == self._i8
        M, K, lda = _mat(A)
        K2, N, ldb = _mat(B)
        if b_layout == B_NK:
            K2, N = N, K2
        assert K == K2
        if out is None:
            torch = _torch()
            out = torch.empty((M, N), dtype=torch.int32, device=A.device)
        st = self.lib.cigemm_gemm_i8_i32(self._h, M, N, K, A.data_ptr(), lda, B.data_ptr(), ldb,
                                         b_layout, out.data_ptr(), _out_ld(out, M, N, 4))
        if st:
            self._check(st, "cigemm_gemm_i8_i32")
        return out

    def gemm_i8_dequant(self, A, B, scale_a, scale_b, b_layout=B_KN, out_type=OUT_F32, out=None,
                        dump_acc=False):
        """Returns ``out`` or ``(out, acc)`` when ``dump_acc``.  A scale tensor with one
        element is per-tensor, otherwise per-row (A) / per-column (B)."""
        if out is not None and not dump_acc:
            st = self._n_gemm_i8_dequant(self._p_gemm_i8_dequant, self._address, A, B, scale_a, scale_b, b_layout, out_type, out)
            if st == 0:
                return out
            if st > 0:
                self._check(st, "cigemm_gemm_i8_dequant")
        f32 = self._f32
        assert A.element_size() == 1 and B.element_size() == 1
        M, K, lda = _mat(A)
        K2, N, ldb = _mat(B)
        if b_layout == B_NK:
            K2, N = N, K2
        assert K == K2
        assert scale_a.dtype == f32 and scale_b.dtype == f32
        assert scale_a.is_contiguous() and scale_b.is_contiguous()
        na, nb = scale_a.numel(), scale_b.numel()
        assert (na == 1 or na == M) and (nb == 1 or nb == N)
        if out is None:
            out = _torch().empty((M, N), device=A.device,
                                 dtype=self._bf16 if out_type == OUT_BF16 else f32)
        acc = None
        if dump_acc:
            torch = _torch()
            acc = torch.empty((M, N), dtype=torch.int32, device=A.device)
        st = self.lib.cigemm_gemm_i8_dequant(
            self._h, M, N, K, A.data_ptr(), lda, B.data_ptr(), ldb, b_layout, scale_a.data_ptr(),
            SCALE_VECTOR if na > 1 else SCALE_TENSOR, scale_b.data_ptr(),
            SCALE_VECTOR if nb > 1 else SCALE_TENSOR, out.data_ptr(), out_type,
            _out_ld(out, M, N, 2 if out_type == OUT_BF16 else 4),
            acc.data_ptr() if dump_acc else None, N if dump_acc else 0)
        if st:
            self._check(st, "cigemm_gemm_i8_dequant")
        return (out, acc) if dump_acc else out

    # -- generators / quantizer ---------------------------------------------------------------
    def fill_random(self, out, seed, lo=-1.0, hi=1.0):
        torch = _torch()
        name = {torch.float32: "cigemm_fill_random_f32", torch.bfloat16: "cigemm_fill_random_bf16",
                torch.float16: "cigemm_fill_random_f16", torch.int8: "cigemm_fill_random_i8"}[out.dtype]
        if out.dtype == torch.int8:
            lo, hi = int(lo), int(hi)
        assert out.is_contiguous()
        self._check(getattr(self.lib, name)(self._h, out.data_ptr(), out.numel(), seed, lo, hi), name)
        return out

    def quantize_rows_i8(self, x, out=None):
        if out is not None:
            q, s = out
            st = self._n_quantize_rows_i8(self._p_quantize_rows_i8, self._address, x, q, s)
            if st == 0:
                return q, s
            if st > 0:
                self._check(st, "cigemm_quantize_rows_i8")
        assert x.dtype == self._f32 and x.dim() == 2
        rows, cols, ldx = _mat(x)
        if out is None:
            torch = _torch()
            q = torch.empty((rows, cols), dtype=torch.int8, device=x.device)
            s = torch.empty((rows,), dtype=torch.float32, device=x.device)
        else:
            q, s = out
            assert q.dtype == self._i8 and q.shape == x.shape and s.dtype == self._f32
            assert s.numel() >= rows and s.is_contiguous()
        st = self.lib.cigemm_quantize_rows_i8(self._h, rows, cols, x.data_ptr(), ldx, q.data_ptr(),
                                              _mat(q)[2], s.data_ptr())
        if st:
            self._check(st, "cigemm_quantize_rows_i8")
        return q, s
