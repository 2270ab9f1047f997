"""The fp32 tile kernel at the heights between multiples of 64 rows (one row of four waves, an odd number
of A instructions per wave): M around the tile and its 32-row pieces, K around the 16-float stages and
their pairs, one and several K ranges, the aligned and the any-alignment form.  Operand values are small
integers and halves, so every sum is exact and the comparison is bit for bit; the padding around the
operands is NaN, the output sits in a sentinel-filled buffer."""
import numpy as np
import pytest

import cudaintro_amd as ci
from cudaintro_amd import probe
from test_gpu_mfma_any import VALS, embed

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("aligned", [True, False])
@pytest.mark.parametrize("rows", [96, 160, 224])
def test_heights(handle, torch_gpu, oracle, rng, rows, aligned):
    torch = torch_gpu
    n = 260 if aligned else 261
    for M in (1, rows - 31, rows, rows + 1, 2 * rows + 33):
        for K in (4, 16, 32, 48, 212, 13 * 16, 400) if aligned else (5, 17, 33, 211, 401):
            A, B = rng.choice(VALS, size=(M, K)), rng.choice(VALS, size=(K, n))
            bias = rng.choice(VALS, size=n)
            off, pad = (0, 4) if aligned else (1, 3)
            _, a = embed(torch, A, torch.float32, off, pad + (-K % 4 if aligned else 0), float("nan"))
            _, b = embed(torch, B, torch.float32, off, pad, float("nan"))
            flat, out = embed(torch, np.zeros((M, n), np.float32), torch.float32, off, pad, 0)
            for ranges in (1, 3):
                probe.force_tile_plan(handle, rows, ranges)
                try:
                    with handle.algo(ci.ALGO_TILE if aligned else ci.ALGO_MFMA_ANY):
                        flat.fill_(7)
                        handle.gemm_f32(a, b, out=out)
                        what = f"{handle.last_kernel} M={M} K={K}"
                        assert f"{rows}x256x16" in handle.last_kernel, what
                        np.testing.assert_array_equal(out.cpu().numpy(), oracle.gemm_f32(A, B), err_msg=what)
                        out.fill_(7)
                        assert bool((flat == 7).all()), what
                        y = handle.linear_f32(a, b, torch.from_numpy(bias).cuda(), ci.ACT_RELU)
                        np.testing.assert_array_equal(y.cpu().numpy(), oracle.linear_f32(A, B, bias, True), err_msg=what)
                finally:
                    probe.force_tile_plan(handle, 0)


@pytest.mark.parametrize("rows", [64, 96, 256])
@pytest.mark.parametrize("kind", ["aligned", "any"])
def test_rows_that_begin_inside_a_line(handle, torch_gpu, rng, kind, rows):
    """The epilogue's two kinds of stores (tile_plan.h, store_streams): rows of C that begin with a line and
    rows that begin inside one, by the leading dimension and by the pointer, whole tiles and ragged
    ones; K ranges too (their partial sums have rows of N).  Sums are exact: bit for bit."""
    torch = torch_gpu
    for M, N in ((256, 512), (300, 512), (256, 516), (300, 516), (257, 740)):
        if kind == "any":
            N += 1
        A, B = (torch.from_numpy(rng.choice(VALS, size=s)).cuda() for s in ((M, 208), (208, N)))
        ref = (A.double() @ B.double()).float()
        for off, ld in ((0, -(-N // 32) * 32), (16, -(-N // 32) * 32), (0, -(-N // 4) * 4 + 4), (4, -(-N // 4) * 4 + 4)):
            flat = torch.empty(off + M * ld, device="cuda")
            out = flat[off:].view(M, ld)[:, :N]
            for ranges in (1, 3):
                probe.force_tile_plan(handle, rows, ranges)
                try:
                    with handle.algo(ci.ALGO_TILE if kind == "aligned" else ci.ALGO_MFMA_ANY):
                        flat.fill_(7)
                        handle.gemm_f32(A, B, out=out)
                        what = f"{handle.last_kernel} {M} {N} {off} {ld}"
                        assert f"{rows}x256x16" in handle.last_kernel, what
                        assert torch.equal(out, ref), what
                        out.fill_(7)
                        assert bool((flat == 7).all()), what
                finally:
                    probe.force_tile_plan(handle, 0)
