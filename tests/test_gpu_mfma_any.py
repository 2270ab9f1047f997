"""The any-shape matrix-core kernels (CIGEMM_ALGO_MFMA_ANY: the tile kernel's any-alignment form and
the register-staged kernel, each by itself and as the library chooses): 16-bit and int8 calls with an odd N
or K, leading dimensions and pointers with no alignment beyond the element's, matrices smaller
than a tile.  int8 bit for bit against the CPU loop, 16-bit bit for bit on exact-arithmetic
inputs and within the K-scaled bound on normal ones; the padding around every operand is NaN
(127 for int8) and the output sits inside a sentinel-filled buffer."""
import re
from contextlib import contextmanager

import numpy as np
import pytest

import cudaintro_amd as ci
from cudaintro_amd import probe
from gpu_util import bits, error_bound_16

pytestmark = pytest.mark.gpu

VALS = np.array([0, 0.5, -0.5, 1, -1, 2, -2], np.float32)
SHAPES = [(1, 1, 1), (3, 5, 7), (64, 63, 64), (129, 131, 67), (300, 257, 1000), (128, 128, 33),
          (17, 1000, 129), (260, 4, 2049),
          # few tiles and a long K: run as K ranges into the workspace plus a reduction launch
          (1, 2047, 2050), (16, 1000, 4097), (130, 257, 3001)]
SPLIT = {(1, 2047, 2050), (16, 1000, 4097), (130, 257, 3001), (260, 4, 2049), (300, 257, 1000)}


def is_register_staged(name):
    return re.search(r"_mfma_any_128x128x", name) is not None


def is_tile_form(name):
    return re.search(r"_mfma_any_[0-9+]+x256x", name) is not None


def too_narrow(N, K, elem, kn):
    """Fewer than 16 bytes of K, or of the N of a K x N operand: the tile kernel's form refuses."""
    return K * elem < 16 or (kn and N * elem < 16)


@contextmanager
def choice(handle, how):
    """How the kernel is chosen: "staged", "tile" (imposed), "any" (ALGO_MFMA_ANY) or "default"."""
    if how in ("staged", "tile"):
        with probe.any_kernel(handle, probe.ANY_TILE if how == "tile" else probe.ANY_REGISTER_STAGED):
            yield
    else:
        with handle.algo(ci.ALGO_MFMA_ANY if how == "any" else ci.ALGO_DEFAULT):
            yield


CHOICES = ["staged", "tile", "any", "default"]


def check_family(how, name, N, K, elem, kn):
    if how == "staged" or too_narrow(N, K, elem, kn):
        assert is_register_staged(name), name
    elif how == "tile":
        assert is_tile_form(name), name
    else:
        assert "_mfma_any_" in name, name


def embed(torch, a, dtype, off, pad, fill):
    """`a` placed at element offset `off` of a flat buffer, rows `a.shape[1] + pad` apart."""
    r, c = a.shape
    ld = c + pad
    flat = torch.full((off + r * ld + 3,), fill, dtype=dtype, device="cuda")
    view = flat[off: off + r * ld].view(r, ld)[:, :c]
    src = torch.from_numpy(np.ascontiguousarray(a)).cuda()
    view.copy_(src.view(dtype) if src.dtype != dtype else src)
    return flat, view


@pytest.mark.parametrize("kind", ["bf16", "f16"])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_any_shape_16bit(handle, torch_gpu, oracle, rng, kind, M, N, K):
    torch = torch_gpu
    narrow = oracle.f32_to_bf16 if kind == "bf16" else oracle.f32_to_f16
    widen = oracle.bf16_to_f32 if kind == "bf16" else oracle.f16_to_f32
    tdt = torch.bfloat16 if kind == "bf16" else torch.float16
    npv = np.int16
    fn = handle.gemm_bf16 if kind == "bf16" else handle.gemm_f16
    for exact in (True, False):
        if exact:
            Af, Bf = rng.choice(VALS, size=(M, K)), rng.choice(VALS, size=(K, N))
        else:
            Af = rng.standard_normal((M, K)).astype(np.float32)
            Bf = rng.standard_normal((K, N)).astype(np.float32)
        Ab, Bb = narrow(Af), narrow(Bf)
        _, a = embed(torch, Ab.view(npv), tdt, 1, 3, float("nan"))
        _, b = embed(torch, Bb.view(npv), tdt, 3, 1, float("nan"))
        flat, out = embed(torch, np.zeros((M, N), npv), tdt, 1, 5, 0.0)
        flat.fill_(3.0)
        for how in CHOICES:
            flat.fill_(3.0)
            with choice(handle, how):
                fn(a, b, out=out)
            check_family(how, handle.last_kernel, N, K, 2, True)
            assert handle.last_kernel.endswith("_splitk") == ((M, N, K) in SPLIT), handle.last_kernel
            got = bits(torch, out)
            if exact:
                np.testing.assert_array_equal(got, narrow(oracle.gemm_f32(widen(Ab), widen(Bb))))
            else:
                ref, S = oracle.gemm_f64(widen(Ab), widen(Bb), with_abs=True)
                err = np.abs(widen(got).astype(np.float64) - ref)
                assert (err <= error_bound_16(ref, S, K, kind)).all()
            f = bits(torch, flat)
            guard = np.ones(f.shape, bool)
            for i in range(M):
                guard[1 + i * (N + 5): 1 + i * (N + 5) + N] = False
            assert (f[guard] == narrow(np.float32(3.0))).all()


@pytest.mark.parametrize("layout", [ci.B_KN, ci.B_NK])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_any_shape_int8(handle, torch_gpu, oracle, rng, layout, M, N, K):
    torch = torch_gpu
    nk = layout == ci.B_NK
    A = rng.integers(-127, 128, size=(M, K), dtype=np.int8)
    B = rng.integers(-127, 128, size=(N, K) if nk else (K, N), dtype=np.int8)
    acc_ref = oracle.gemm_i8_i32(A, B, b_is_nk=nk)
    _, a = embed(torch, A, torch.int8, 1, 3, 127)
    _, b = embed(torch, B, torch.int8, 5, 1, 127)
    flat, out = embed(torch, np.zeros((M, N), np.int32), torch.int32, 1, 3, -9)
    sa = rng.uniform(1e-3, 5e-2, M).astype(np.float32)
    sb = rng.uniform(1e-3, 5e-2, N).astype(np.float32)
    for how in CHOICES:
        flat.fill_(-9)
        with choice(handle, how):
            handle.gemm_i8_i32(a, b, layout, out=out)
            check_family(how, handle.last_kernel, N, K, 1, not nk)
            np.testing.assert_array_equal(out.cpu().numpy(), acc_ref)
            f = flat.cpu().numpy()
            guard = np.ones(f.shape, bool)
            for i in range(M):
                guard[1 + i * (N + 3): 1 + i * (N + 3) + N] = False
            assert (f[guard] == -9).all()
            for out_type, ot in (("f32", ci.OUT_F32), ("bf16", ci.OUT_BF16)):
                y, acc = handle.gemm_i8_dequant(a, b, torch.from_numpy(sa).cuda(), torch.from_numpy(sb).cuda(),
                                                layout, ot, dump_acc=True)
                # (the accumulator dump on unaligned rows is the register-staged kernel's)
                assert is_register_staged(handle.last_kernel) and "dequant" in handle.last_kernel
                np.testing.assert_array_equal(acc.cpu().numpy(), acc_ref)
                expect = oracle.dequant(acc_ref, sa, sb, out_dtype=out_type, sa_per_row=True, sb_per_col=True)
                got = bits(torch, y) if out_type == "bf16" else y.cpu().numpy()
                np.testing.assert_array_equal(got, expect)


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_any_shape_f32(handle, torch_gpu, oracle, rng, M, N, K):
    """fp32: within the scaled 1e-5 tolerance of the CPU loop on uniform inputs, bit for bit on
    exact-arithmetic inputs; with and without bias + ReLU."""
    torch = torch_gpu
    for exact in (True, False):
        if exact:
            A, B = rng.choice(VALS, size=(M, K)), rng.choice(VALS, size=(K, N))
        else:
            A = rng.uniform(-1, 1, size=(M, K)).astype(np.float32)
            B = rng.uniform(-1, 1, size=(K, N)).astype(np.float32)
        bias = rng.choice(VALS, size=N) if exact else rng.uniform(-1, 1, size=N).astype(np.float32)
        _, a = embed(torch, A, torch.float32, 1, 3, float("nan"))
        _, b = embed(torch, B, torch.float32, 3, 1, float("nan"))
        flat, out = embed(torch, np.zeros((M, N), np.float32), torch.float32, 1, 5, 0.0)
        for how in CHOICES:
            for with_bias in (False, True):
                flat.fill_(3.0)
                with choice(handle, how):
                    if with_bias:
                        handle.linear_f32(a, b, torch.from_numpy(bias).cuda(), ci.ACT_RELU, out=out)
                        cpu = oracle.linear_f32(A, B, bias, True)
                    else:
                        handle.gemm_f32(a, b, out=out)
                        cpu = oracle.gemm_f32(A, B)
                if how == "default" and "f32_mfma_any_small" in handle.last_kernel:
                    pass     # (the small kernel takes any fp32 call)
                else:
                    check_family(how, handle.last_kernel, N, K, 4, True)
                if how == "staged" and (M, N, K) in SPLIT:
                    assert handle.last_kernel.endswith("_splitk"), handle.last_kernel
                got = out.cpu().numpy()
                if exact:
                    np.testing.assert_array_equal(got, cpu)
                else:
                    plain = oracle.gemm_f32(A, B).astype(np.float64)
                    rms = float(np.sqrt(np.mean(plain ** 2)))
                    lim = 1e-5 * np.maximum(np.abs(plain), rms) + 1e-30
                    assert (np.abs(got.astype(np.float64) - cpu) <= lim).all()
                f = flat.cpu().numpy()
                guard = np.ones(f.shape, bool)
                for i in range(M):
                    guard[1 + i * (N + 5): 1 + i * (N + 5) + N] = False
                assert (f[guard] == 3.0).all()


@pytest.mark.parametrize("kind", ["bf16", "f16", "f32"])
def test_leading_dimension_beyond_the_tile_kernels_offsets(handle, torch_gpu, oracle, rng, kind):
    """256 rows of A span 2 GiB and more: the tile kernel's 32-bit row offsets do not reach, the
    call stays on the register-staged kernel without being asked to."""
    torch = torch_gpu
    M, N, K = 3, 137, 75
    A, B = rng.choice(VALS, size=(M, K)), rng.choice(VALS, size=(K, N))
    ref = oracle.gemm_f32(A, B)
    dt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[kind]
    ld = (1 << 31) // 256 // dt.itemsize + 1
    flat = torch.full((M * ld,), float("nan"), dtype=dt, device="cuda")
    a = flat.view(M, ld)[:, 1:K + 1]
    a.copy_(torch.from_numpy(A).cuda())
    _, b = embed(torch, B, torch.float32, 0, 0, float("nan"))
    with handle.algo(ci.ALGO_MFMA_ANY):     # (by itself an fp32 call this small goes to the small kernel)
        out = getattr(handle, "gemm_" + kind)(a, b.to(dt).contiguous())
    assert is_register_staged(handle.last_kernel), handle.last_kernel
    np.testing.assert_array_equal(out.float().cpu().numpy(), torch.from_numpy(ref).to(dt).float().numpy())


def test_wide_rows_of_b_leave_a_large_fp32_call_to_the_register_staged_kernel(handle, torch_gpu, oracle, rng):
    """256 rows of B span 2 GiB: not the tile kernel's; A's rows are aligned and K a multiple of 8, so
    the small kernel takes the call, but 4096 tiles of 32 x 32 are not where it is the faster."""
    torch = torch_gpu
    M, N, K = 2048, 2047, 64
    A, B = rng.choice(VALS, size=(M, K)), rng.choice(VALS, size=(K, N))
    flat = torch.full((K * ((1 << 21) + 1),), float("nan"), dtype=torch.float32, device="cuda")
    b = flat.view(K, (1 << 21) + 1)[:, :N]
    b.copy_(torch.from_numpy(B).cuda())
    out = handle.gemm_f32(torch.from_numpy(A).cuda(), b)
    assert is_register_staged(handle.last_kernel), handle.last_kernel
    np.testing.assert_array_equal(out.cpu().numpy(), oracle.gemm_f32(A, B))


def test_choice_by_shape(handle, torch_gpu):
    """Which of the kernels that take any alignment serves a call, where their times differ by a
    factor (any_plan.h): narrow outputs and short K stay off the 256-column tiles."""
    torch = torch_gpu
    def kernel_for(kind, M, N, K):
        dt = {"bf16": torch.bfloat16, "f32": torch.float32, "i8nk": torch.int8}[kind]
        a = torch.zeros((M, K), dtype=dt, device="cuda")
        if kind == "i8nk":
            handle.gemm_i8_i32(a, torch.zeros((N, K), dtype=dt, device="cuda"), ci.B_NK)
        else:
            getattr(handle, "gemm_" + kind)(a, torch.zeros((K, N), dtype=dt, device="cuda"))
        return handle.last_kernel
    assert is_tile_form(kernel_for("bf16", 4096, 4095, 1024))
    assert is_tile_form(kernel_for("f32", 2049, 2047, 1025))
    assert is_tile_form(kernel_for("i8nk", 2048, 2047, 4097))
    assert is_register_staged(kernel_for("i8nk", 4456, 7, 1575))
    assert is_register_staged(kernel_for("bf16", 33, 11, 741))
    assert is_register_staged(kernel_for("bf16", 171960, 25, 257))
    # an output layer of 10 columns keeps its 16-column form beyond one round of 256-row tiles
    assert kernel_for("f32", 65536, 10, 512) == kernel_for("f32", 70000, 10, 512) == "f32_mfma_small_16x16_ksplit4"
    assert "small" in kernel_for("f32", 1000, 3, 77)        # narrower than a 16-byte piece, K odd
    # K a multiple of 4 but not of 8, all aligned
    assert "small" in kernel_for("f32", 512, 512, 508)
    assert "_mfma_any" not in kernel_for("f32", 3837, 808, 1588)


def test_any_shape_kernel_is_the_fallback_not_the_first_choice(handle, torch_gpu):
    """Aligned shapes keep the LDS-DMA tile kernel and the small fp32 kernel."""
    torch = torch_gpu
    a = torch.zeros((256, 256), dtype=torch.bfloat16, device="cuda")
    handle.gemm_bf16(a, a)
    assert "mfma_any" not in handle.last_kernel and "_mfma_" in handle.last_kernel
    f = torch.zeros((512, 512), dtype=torch.float32, device="cuda")
    handle.gemm_f32(f, f)
    assert "mfma_any" not in handle.last_kernel
    f = torch.zeros((4096, 64), dtype=torch.float32, device="cuda")
    handle.gemm_f32(f, torch.zeros((64, 4096), dtype=torch.float32, device="cuda"))
    assert "x256x16_w" in handle.last_kernel
