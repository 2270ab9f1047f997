"""The native binding of the hot calls (csrc/binding.cpp) without a GPU: the entry points it is given are
Python callbacks that record their arguments, over every order and stride the Python code takes, against
what that computes; what that refuses is refused."""
import ctypes as C
import os
import subprocess
import sys

import pytest
import torch

import cudaintro_amd as ci
from cudaintro_amd import cigemm

native = cigemm._native()
HANDLE = 0x1230
CSRC = os.path.join(os.path.dirname(cigemm.__file__), "csrc")


class Entry:
    """A C function of the prototype of `name` that records its arguments and returns `status`."""

    def __init__(self, name, status=0):
        res, args = cigemm.SIGNATURES[name]
        self.calls = []

        def body(*a):
            self.calls.append(a)
            return status
        self._keep = C.CFUNCTYPE(res, *args)(body)
        self.address = C.cast(self._keep, C.c_void_p).value


def matrices(rows, cols, dtype):
    """The same matrix shape in every form: packed, a column block, a row step, one row, offset."""
    big = torch.zeros((2 * rows + 1, cols + 5), dtype=dtype)
    yield torch.zeros((rows, cols), dtype=dtype)
    yield big[:rows, 3:3 + cols]
    yield big[1:1 + 2 * rows:2, :cols]
    yield torch.zeros((1, cols), dtype=dtype).expand(rows, cols)      # every row the same one
    if cols == 1:
        yield torch.zeros((1, rows), dtype=dtype).t()                 # a single column of any stride


def expect(t):
    rows, cols, ld = cigemm._mat(t)
    return rows, cols, ld, t.data_ptr() or None


@pytest.mark.parametrize("code,dtype", [(0, torch.float32), (1, torch.float16), (2, torch.bfloat16)])
def test_gemm(code, dtype):
    fn = Entry("cigemm_gemm_f32")
    for M, K, N in ((3, 5, 7), (1, 4, 1), (4, 1, 6), (2, 0, 3), (0, 2, 2)):
        for A in matrices(M, K, dtype):
            for B in matrices(K, N, dtype):
                for out in matrices(M, N, torch.float32):
                    assert native.gemm(fn.address, HANDLE, code, A, B, out) == 0
                    (m, k, lda, a), (_, n, ldb, b), (_, _, ldc, c) = expect(A), expect(B), expect(out)
                    assert fn.calls.pop() == (HANDLE, m, n, k, a, lda, b, ldb, c, ldc)
    assert native.gemm(Entry("cigemm_gemm_f32", 13).address, HANDLE, code, A, B, out) == 13


def test_refused_as_before():
    fn = Entry("cigemm_gemm_f32")
    A, B, out = torch.zeros(3, 5), torch.zeros(5, 7), torch.zeros(3, 7)
    for bad in ((A.double(), B, out), (A, B.half(), out), (A, torch.zeros(4, 7), out), (A.t().contiguous().t(), B, out),
                (A, torch.zeros(7, 5).t(), out), (A, B, torch.zeros(7, 3).t()), (A, B, torch.zeros(21)),
                (torch.zeros(5), B, out), (torch.zeros(1, 3, 5), B, out)):
        with pytest.raises(AssertionError):
            native.gemm(fn.address, HANDLE, 0, *bad)

    class Sub(torch.Tensor):
        pass
    for odd in ((A.numpy(), B, out), (A, B.as_subclass(Sub), out), (A, B, None)):
        assert native.gemm(fn.address, HANDLE, 0, *odd) == -1      # (left to the Python code)
    assert native.gemm(fn.address, HANDLE, 0, torch.nn.Parameter(A), B, out) == 0
    with pytest.raises(TypeError):
        native.gemm(fn.address, HANDLE, 0, A, B)
    assert len(fn.calls) == 1


def test_linear_int8_quantizer():
    fn = Entry("cigemm_linear_f32")
    X, W, out = torch.zeros(3, 5), torch.zeros(5, 7), torch.zeros(3, 7)
    bias = torch.zeros(7)
    for b in (None, bias):
        assert native.linear_f32(fn.address, HANDLE, X, W, b, ci.ACT_RELU, out) == 0
        assert fn.calls.pop() == (HANDLE, 3, 7, 5, X.data_ptr(), 5, W.data_ptr(), 7, b.data_ptr() if b is not None else None,
                                  int(ci.ACT_RELU), out.data_ptr(), 7)
    for b in (torch.zeros(6), bias.double()):
        with pytest.raises(AssertionError):
            native.linear_f32(fn.address, HANDLE, X, W, b, 0, out)

    A, sa, sb = torch.zeros((3, 5), dtype=torch.int8), torch.zeros(3), torch.zeros(1)
    f32, f16 = Entry("cigemm_gemm_i8_i32"), Entry("cigemm_gemm_i8_dequant")
    for layout, B in ((ci.B_KN, torch.zeros((5, 7), dtype=torch.int8)), (ci.B_NK, torch.zeros((7, 5), dtype=torch.int8))):
        acc, y = torch.zeros((3, 7), dtype=torch.int32), torch.zeros((3, 7), dtype=torch.bfloat16)
        assert native.gemm_i8_i32(f32.address, HANDLE, A, B, layout, acc) == 0
        assert f32.calls.pop() == (HANDLE, 3, 7, 5, A.data_ptr(), 5, B.data_ptr(), B.stride(0), int(layout), acc.data_ptr(), 7)
        assert native.gemm_i8_dequant(f16.address, HANDLE, A, B, sa, sb, layout, ci.OUT_BF16, y) == 0
        assert f16.calls.pop() == (HANDLE, 3, 7, 5, A.data_ptr(), 5, B.data_ptr(), B.stride(0), int(layout), sa.data_ptr(),
                                   int(ci.SCALE_VECTOR), sb.data_ptr(), int(ci.SCALE_TENSOR), y.data_ptr(),
                                   int(ci.OUT_BF16), 7, None, 0)
        for bad in ((sa[:2], sb), (sa, torch.zeros(3)), (sa.double(), sb)):
            with pytest.raises(AssertionError):
                native.gemm_i8_dequant(f16.address, HANDLE, A, B, *bad, layout, ci.OUT_BF16, y)

    q = Entry("cigemm_quantize_rows_i8")
    x, xq, sx = torch.zeros(3, 9)[:, 2:7], torch.zeros((3, 5), dtype=torch.int8), torch.zeros(3)
    assert native.quantize_rows_i8(q.address, HANDLE, x, xq, sx) == 0
    assert q.calls.pop() == (HANDLE, 3, 5, x.data_ptr(), 9, xq.data_ptr(), 5, sx.data_ptr())
    for bad in ((x.double(), xq, sx), (x, xq[:2], sx), (x, xq.int(), sx), (x, xq, sx.double())):
        with pytest.raises(AssertionError):
            native.quantize_rows_i8(q.address, HANDLE, *bad)


def test_what_would_be_written_or_read_past_its_end_is_refused():
    """Outputs with too few rows, columns or bytes an element, scales and biases that are short or not dense; room to
    spare is taken."""
    i8 = torch.int8
    e = Entry("cigemm_gemm_f32")
    A, B = torch.zeros(3, 5), torch.zeros(5, 7)
    small = (torch.zeros(2, 7), torch.zeros(3, 6), torch.zeros(3, 14)[:, 4:10], torch.zeros((3, 7), dtype=torch.float16),
             torch.zeros(1, 21))
    for out in small:
        with pytest.raises(AssertionError):
            native.gemm(e.address, HANDLE, 0, A, B, out)
    with pytest.raises(AssertionError):
        native.gemm(e.address, HANDLE, 2, A.bfloat16(), B.bfloat16(), torch.zeros((3, 7), dtype=i8))
    for out in (torch.zeros(4, 7), torch.zeros(3, 9), torch.zeros((3, 7), dtype=torch.float64),
                torch.zeros((3, 7), dtype=torch.int32)):
        assert native.gemm(e.address, HANDLE, 0, A, B, out) == 0

    e = Entry("cigemm_linear_f32")
    for out in small:
        with pytest.raises(AssertionError):
            native.linear_f32(e.address, HANDLE, A, B, None, 0, out)
    for bias in (torch.zeros(14)[::2], torch.zeros(1).expand(7)):
        with pytest.raises(AssertionError):
            native.linear_f32(e.address, HANDLE, A, B, bias, 0, torch.zeros(3, 7))
    assert native.linear_f32(e.address, HANDLE, A, B, torch.zeros(1, 7), 0, torch.zeros(3, 7)) == 0

    qa, sa, sb = torch.zeros((3, 5), dtype=i8), torch.zeros(3), torch.zeros(7)
    e, d = Entry("cigemm_gemm_i8_i32"), Entry("cigemm_gemm_i8_dequant")
    for layout, qb in ((ci.B_KN, torch.zeros((5, 7), dtype=i8)), (ci.B_NK, torch.zeros((7, 5), dtype=i8))):
        for out in small:
            with pytest.raises(AssertionError):
                native.gemm_i8_i32(e.address, HANDLE, qa, qb, layout, out)
            with pytest.raises(AssertionError):
                native.gemm_i8_dequant(d.address, HANDLE, qa, qb, sa, sb, layout, ci.OUT_F32, out)
        y = torch.zeros((3, 7), dtype=torch.bfloat16)
        assert native.gemm_i8_dequant(d.address, HANDLE, qa, qb, sa, sb, layout, ci.OUT_BF16, y) == 0
        assert native.gemm_i8_dequant(d.address, HANDLE, qa.view(torch.uint8), qb, sa, sb, layout, ci.OUT_BF16, y) == 0
        for bad in ((qa.float(), qb, sa, sb), (qa, qb.half(), sa, sb), (qa, qb, torch.zeros(6)[::2], sb),
                    (qa, qb, sa, torch.zeros(1).expand(7))):
            with pytest.raises(AssertionError):
                native.gemm_i8_dequant(d.address, HANDLE, *bad, layout, ci.OUT_BF16, y)

    q = Entry("cigemm_quantize_rows_i8")
    for s in (torch.zeros(2), torch.zeros(6)[::2], torch.zeros(1).expand(3)):
        with pytest.raises(AssertionError):
            native.quantize_rows_i8(q.address, HANDLE, A, qa, s)
    assert native.quantize_rows_i8(q.address, HANDLE, A, qa, torch.zeros(4)) == 0


def test_refused_by_the_python_code_too():
    """The same calls where the native binding hands them back."""
    class Reached(Exception):
        pass

    class Lib:
        def __getattr__(self, name):
            def call(*a):
                raise Reached(name)
            return call
    h = object.__new__(ci.Handle)
    h.lib, h._h, h._address = Lib(), None, 0
    h._f32, h._bf16, h._f16, h._i8 = torch.float32, torch.bfloat16, torch.float16, torch.int8
    for name in cigemm._native_entries():
        setattr(h, name, (lambda *a: -1) if name.startswith("_n_") else 0)
    i8 = torch.int8
    A, B, C = torch.zeros(3, 5), torch.zeros(5, 7), torch.zeros(3, 7)
    qa, qb, sa, sb = torch.zeros((3, 5), dtype=i8), torch.zeros((5, 7), dtype=i8), torch.zeros(3), torch.zeros(7)
    taken = [lambda: h.gemm_f32(A, B, out=C), lambda: h.gemm_bf16(A.bfloat16(), B.bfloat16(), out=C),
             lambda: h.linear_f32(A, B, sb, out=torch.zeros(5, 9)), lambda: h.gemm_i8_i32(qa, qb, out=C),
             lambda: h.gemm_i8_dequant(qa, qb, sa, sb, out=C), lambda: h.quantize_rows_i8(A, out=(qa, sa))]
    refused = [lambda: h.gemm_f32(A, B, out=torch.zeros(2, 7)), lambda: h.gemm_f32(A, B, out=C.half()),
               lambda: h.gemm_f16(A.half(), B.half(), out=torch.zeros((3, 6), dtype=torch.float16)),
               lambda: h.linear_f32(A, B, torch.zeros(14)[::2], out=C), lambda: h.linear_f32(A, B, sb, out=C.half()),
               lambda: h.gemm_i8_i32(qa, qb, out=C.half()), lambda: h.gemm_i8_dequant(qa.float(), qb, sa, sb, out=C),
               lambda: h.gemm_i8_dequant(qa, qb, sa, torch.zeros(1).expand(7), out=C),
               lambda: h.gemm_i8_dequant(qa, qb, sa, sb, out=C.half()),
               lambda: h.quantize_rows_i8(A, out=(qa, torch.zeros(2)))]
    for call in taken:
        with pytest.raises(Reached):
            call()
    for call in refused:
        with pytest.raises(AssertionError):
            call()


def test_the_libraries_and_the_driver_build_without_python(tmp_path):
    """`make` asks no Python for anything; `make python` builds the module for the Python it is given."""
    plan = lambda *a: subprocess.run(["make", "-n", "-B", "-C", CSRC, *a], capture_output=True, text=True)  # noqa: E731
    asked = tmp_path / "asked"
    python = tmp_path / "python"
    python.write_text(f"#!/bin/sh\ntouch {asked}\nexec {sys.executable} \"$@\"\n")
    python.chmod(0o755)
    out = plan("all", f"PYTHON={python}")
    assert out.returncode == 0 and "gemm_suite" in out.stdout and "binding" not in out.stdout and not asked.exists()
    out = plan("python", f"PYTHON={python}")
    assert out.returncode == 0 and "binding.cpp" in out.stdout and os.path.dirname(torch.__file__) in out.stdout
    assert asked.exists() and "libcigemm" not in out.stdout
