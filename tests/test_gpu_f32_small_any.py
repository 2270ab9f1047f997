"""The small fp32 kernel with a K that is no multiple of 8 or with unaligned rows of A: every length
of the separately multiplied end of K, all of K in it, waves without a share of K, edge tiles, both
forms of B's loads, bias + ReLU.  Operand values are small integers and halves, so every sum is
exact and the comparison is bit for bit; the padding around the operands is NaN and the output
sits in a sentinel-filled buffer."""
import numpy as np
import pytest

import cudaintro_amd as ci
from cudaintro_amd import probe
from test_gpu_mfma_any import VALS, embed

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N", [(1, 5), (33, 64), (70, 100), (65, 31)])
@pytest.mark.parametrize("a_off,b_pad", [(0, 0), (1, 0), (1, 3)])
def test_f32_small_any(handle, torch_gpu, oracle, rng, M, N, a_off, b_pad):
    torch = torch_gpu
    for K in [4, 5, 7, 8, 9, 15, 30, 33, 34, 35, 36, 37, 38, 39, 40, 129, 130, 131, 132, 133, 134, 135]:
        A, B = rng.choice(VALS, size=(M, K)), rng.choice(VALS, size=(K, N))
        bias = rng.choice(VALS, size=N)
        _, a = embed(torch, A, torch.float32, a_off, 0 if a_off == 0 else 3, float("nan"))
        _, b = embed(torch, B, torch.float32, 4, b_pad, float("nan"))
        flat, out = embed(torch, np.zeros((M, N), np.float32), torch.float32, 1, 5, 0.0)
        guard = np.ones(flat.numel(), bool)
        for i in range(M):
            guard[1 + i * (N + 5): 1 + i * (N + 5) + N] = False
        for relu in (False, True):
            def run():
                flat.fill_(3.0)
                if relu:
                    handle.linear_f32(a, b, torch.from_numpy(bias).cuda(), ci.ACT_RELU, out=out)
                else:
                    handle.gemm_f32(a, b, out=out)

            def check():
                np.testing.assert_array_equal(out.cpu().numpy(), ref, err_msg=f"K={K}")
                assert (flat.cpu().numpy()[guard] == 3.0).all()

            ref = oracle.linear_f32(A, B, bias, True) if relu else oracle.gemm_f32(A, B)
            with probe.any_kernel(handle, probe.ANY_F32_SMALL):
                run()
                assert "small_32x32" in handle.last_kernel, handle.last_kernel
                assert ("any" in handle.last_kernel) == (K % 8 != 0 or a_off != 0)
                check()
            # by itself a product of one or two stages may go to the tile kernel's any-alignment form
            run()
            assert "small" in handle.last_kernel or K < 64, handle.last_kernel
            check()
