"""The kernel of batches (64 or 128 rows x 64 columns, k shared out to four pairs of waves) at the sizes where it can
go wrong: M and N around its tiles, K around its 128-byte stages (less than one, as many as its ring of 6 or 8 holds
and one to either side, a last one partly filled).  Operand values are small integers and halves, so every sum is
exact in any order and the comparison is bit for bit; the padding around the operands is NaN (127 for int8), the
output sits in a sentinel-filled buffer."""
import numpy as np
import pytest

import cudaintro_amd as ci
from cudaintro_amd import probe
from gpu_util import bits
from test_gpu_mfma_any import VALS, embed

pytestmark = pytest.mark.gpu
BYTES = {"bf16": 2, "f16": 2, "i8_nk": 1}
SHAPES = [(33, 64), (63, 68), (64, 260), (65, 128), (130, 196), (257, 132), (300, 320)]


@pytest.mark.parametrize("rows", [64, 128])
@pytest.mark.parametrize("kind", list(BYTES))
def test_panel(handle, torch_gpu, oracle, rng, kind, rows):
    torch = torch_gpu
    int8 = kind.startswith("i8")
    layout = ci.B_NK
    eb = BYTES[kind]
    stage, piece = 128 // eb, 16 // eb
    host = lambda t: bits(torch, t) if t.element_size() == 2 else t.contiguous().cpu().numpy()  # noqa: E731
    for M, N in SHAPES:
        for K in (piece, stage, 2 * stage + piece, 6 * stage, 7 * stage, 8 * stage, 9 * stage + 3 * piece,
                  18 * stage - piece):
            if int8:
                A = rng.integers(-127, 128, size=(M, K), dtype=np.int8)
                B = rng.integers(-127, 128, size=(N, K), dtype=np.int8)
                ref = oracle.gemm_i8_i32(A, B, b_is_nk=True)
                dt, odt, pad = torch.int8, torch.int32, 127
            else:
                A, B = rng.choice(VALS, size=(M, K)), rng.choice(VALS, size=(K, N))
                ref = oracle.gemm_f32(A, B)
                dt = odt = {"bf16": torch.bfloat16, "f16": torch.float16}[kind]
                pad = float("nan")
                narrow = {"bf16": oracle.f32_to_bf16, "f16": oracle.f32_to_f16}[kind]
                A, B, ref = narrow(A).view(np.int16), narrow(B).view(np.int16), narrow(ref)
            _, a = embed(torch, A, dt, 0, -A.shape[1] % piece + piece, pad)
            _, b = embed(torch, B, dt, 0, -B.shape[1] % piece + piece, pad)
            po = -N % (16 // odt.itemsize) + 16 // odt.itemsize
            flat, out = embed(torch, np.zeros((M, N), np.int32).astype(np.int16 if odt.itemsize == 2 else np.int32),
                              odt, 0, po, 0)
            guard = np.ones(flat.numel(), bool)
            for i in range(M):
                guard[i * (N + po): i * (N + po) + N] = False
            probe.force_panel_rows(handle, rows)
            try:
                flat.fill_(7)
                sentinel = host(flat)[0]
                if int8:
                    handle.gemm_i8_i32(a, b, layout, out=out)
                else:
                    getattr(handle, "gemm_" + kind)(a, b, out=out)
                what = f"{handle.last_kernel} M={M} N={N} K={K}"
                assert f"panel_{rows}x64" in what and handle.last_plan == (rows, 1)
                np.testing.assert_array_equal(host(out), ref, err_msg=what)
                assert (host(flat)[guard] == sentinel).all(), what
                if int8:
                    sa = rng.uniform(1e-3, 5e-2, M).astype(np.float32)
                    sb = rng.uniform(1e-3, 5e-2, N).astype(np.float32)
                    for out_name, ot in (("f32", ci.OUT_F32), ("bf16", ci.OUT_BF16)):
                        for n_a, n_b in ((M, N), (1, 1)):
                            y = handle.gemm_i8_dequant(a, b, torch.from_numpy(sa[:n_a]).cuda(),
                                                       torch.from_numpy(sb[:n_b]).cuda(), layout, ot)
                            if N % (16 // (2 if out_name == "bf16" else 4)) == 0:   # (else rows of out are unaligned)
                                assert f"panel_{rows}x64" in handle.last_kernel, handle.last_kernel
                            np.testing.assert_array_equal(
                                host(y), oracle.dequant(ref, sa[:n_a], sb[:n_b], out_dtype=out_name,
                                                        sa_per_row=n_a > 1, sb_per_col=n_b > 1), err_msg=what)
            finally:
                probe.force_panel_rows(handle, 0)


@pytest.mark.parametrize("kind,M,N,K", [("bf16", 229, 2752, 1984), ("f16", 1097, 1664, 1664), ("i8_nk", 584, 2752, 2944),
                                        ("i8_nk", 512, 4096, 4096)])
def test_chosen(handle, torch_gpu, kind, M, N, K):
    """Calls that come here by themselves give what the tile kernel gives (values as above: bit for bit), twice."""
    torch = torch_gpu
    gen = torch.Generator(device="cuda").manual_seed(3)
    ints = lambda r, c: torch.randint(-2, 3, (r, c), generator=gen, device="cuda")  # noqa: E731
    if kind == "i8_nk":
        a, b = ints(M, K).to(torch.int8), ints(N, K).to(torch.int8)
        call = lambda: handle.gemm_i8_i32(a, b, ci.B_NK)  # noqa: E731
    else:
        dt = {"bf16": torch.bfloat16, "f16": torch.float16}[kind]
        a, b = ints(M, K).to(dt), ints(K, N).to(dt)
        call = lambda: getattr(handle, "gemm_" + kind)(a, b)  # noqa: E731
    got = call()
    assert "panel" in handle.last_kernel, handle.last_kernel
    again = call()
    probe.force_panel_rows(handle, -1)
    try:
        want = call()
    finally:
        probe.force_panel_rows(handle, 0)
    assert "panel" not in handle.last_kernel
    assert torch.equal(got, want) and torch.equal(again, want)
