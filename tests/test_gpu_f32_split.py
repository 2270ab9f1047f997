"""fp32 tiles on the bf16 matrix instructions (every operand as the exact sum of three bf16 numbers): each
height with one and several K ranges at the edges of tiles, stages and column pairs, operands whose second
and third parts matter, and what the three parts cannot hold (infinities, NaN, the largest and the smallest
magnitudes), which the kernel computes once more in fp32.  NaN padding around the operands, the output in
a sentinel-filled buffer."""
import re

import numpy as np
import pytest

import cudaintro_amd as ci
from cudaintro_amd import probe
from test_gpu_mfma_any import embed

pytestmark = pytest.mark.gpu

ROWS = (64, 96, 128)


@pytest.fixture(autouse=True)
def hand_back(handle):
    yield
    probe.force_f32_split(handle, 0)


def run(handle, torch, A, B, rows, ranges, off, pad, bias=None):
    """The product (or the layer with ReLU) on embedded operands; checks the guard around the output."""
    M, N = A.shape[0], B.shape[1]
    _, a = embed(torch, A, torch.float32, off, pad, float("nan"))
    _, b = embed(torch, B, torch.float32, off, pad, float("nan"))
    flat, out = embed(torch, np.zeros((M, N), np.float32), torch.float32, off, pad, 0)
    probe.force_f32_split(handle, rows, ranges)
    flat.fill_(7)
    if bias is None:
        handle.gemm_f32(a, b, out=out)
    else:
        handle.linear_f32(a, b, torch.from_numpy(bias).cuda(), ci.ACT_RELU, out=out)
    what = f"{handle.last_kernel} {M}x{N}x{A.shape[1]} ranges {ranges}"
    assert f"{rows}x256x16_w4" in handle.last_kernel and "32x32x2" not in handle.last_kernel, what
    got = out.cpu().numpy().copy()
    out.fill_(7)
    assert bool((flat == 7).all()), what
    return got, what


@pytest.mark.parametrize("rows", ROWS)
def test_exact_sums(handle, torch_gpu, rng, rows):
    """Integers of 12 bits times small ones: two parts of one operand, every sum exact."""
    for M in (1, rows - 1, rows + 33):
        for N in (2, 255, 257, 258, 300):
            for K in (17, 31, 32, 33, 48, 49, 113, 160, 400):
                wide = rng.integers(-2048, 2049, size=(M, K)).astype(np.float32)
                small = rng.integers(-2, 3, size=(K, N)).astype(np.float32)
                off, pad = (0, 4) if K % 2 == 0 else (1, 3)
                for ranges in (1, 3):
                    got, what = run(handle, torch_gpu, wide, small, rows, ranges, off, pad)
                    np.testing.assert_array_equal(got, wide.astype(np.float64) @ small, err_msg=what)
                small, wide = (rng.integers(-2, 3, size=(M, K)).astype(np.float32),
                               rng.integers(-2048, 2049, size=(K, N)).astype(np.float32))
                bias = rng.integers(-9, 9, size=N).astype(np.float32)
                got, what = run(handle, torch_gpu, small, wide, rows, 1, off, pad, bias)
                np.testing.assert_array_equal(got, np.maximum(small.astype(np.float64) @ wide + bias, 0), err_msg=what)


@pytest.mark.parametrize("rows", ROWS)
def test_one_hot_operands_select_all_24_bits(handle, torch_gpu, rng, rows):
    M, N, K = rows + 5, 267, 93
    X = rng.normal(size=(M, K)).astype(np.float32)
    take = rng.integers(0, K, size=N)
    W = np.zeros((K, N), np.float32)
    W[take, np.arange(N)] = 1
    got, what = run(handle, torch_gpu, X, W, rows, 1, 1, 3)
    np.testing.assert_array_equal(got, X[:, take], err_msg=what)
    Y = rng.normal(size=(K, N)).astype(np.float32)
    take = rng.integers(0, K, size=M)
    S = np.zeros((M, K), np.float32)
    S[np.arange(M), take] = 1
    got, what = run(handle, torch_gpu, S, Y, rows, 2, 0, 4)
    np.testing.assert_array_equal(got, Y[take], err_msg=what)


def on_fp32_instructions(handle, torch, A, B, ranges=1):
    """The same call on the tiles of v_mfma_f32_32x32x2_f32."""
    probe.force_f32_split(handle, 0)
    probe.force_tile_plan(handle, 256, ranges)
    try:
        with handle.algo(ci.ALGO_TILE):
            out = handle.gemm_f32(torch.from_numpy(A).cuda(), torch.from_numpy(B).cuda()).cpu().numpy()
            assert "32x32x2" in handle.last_kernel and handle.last_plan == (256, ranges)
    finally:
        probe.force_tile_plan(handle, 0)
    return out


def nonzeros(rng, M, K, count):
    """Rows of `count` values at random places, zero elsewhere."""
    A = np.zeros((M, K), np.float32)
    for row in A:
        row[rng.choice(K, count, replace=False)] = rng.uniform(-1, 1, count)
    return A


@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("kind", ["symmetric", "positive", "wide", "half zeros", "fifth", "8", "2", "dominating"])
def test_no_further_from_64_bits_than_the_fp32_instructions(handle, torch_gpu, rng, rows, kind):
    """The same call on the tiles of v_mfma_f32_32x32x2_f32 is the measure, error by sum of magnitudes, over
    131072 outputs; 1 % for the draw."""
    torch = torch_gpu
    M, N = 256, 512
    for K in (64, 700, 4096):
        draw = {"positive": lambda s: rng.uniform(0, 1, s),
                "wide": lambda s: rng.normal(size=s) * np.exp(3 * rng.normal(size=s))}.get(
                    kind, lambda s: rng.uniform(-1, 1, s))
        A, B = draw((M, K)).astype(np.float32), draw((K, N)).astype(np.float32)
        count = {"half zeros": K // 2, "fifth": K // 5, "8": 8, "2": 2}.get(kind)
        if count:
            A = nonzeros(rng, M, K, count)
        if kind == "dominating":
            A[:, 1:] *= np.float32(2.0 ** -14)
        ref = A.astype(np.float64) @ B.astype(np.float64)
        got, what = run(handle, torch, A, B, rows, 1, 0, 0)
        old = on_fp32_instructions(handle, torch, A, B)
        size = np.abs(A.astype(np.float64)) @ np.abs(B.astype(np.float64))
        err, err_old = np.linalg.norm((got - ref) / size), np.linalg.norm((old - ref) / size)
        assert err <= 1.01 * err_old, (what, err / err_old)


@pytest.mark.parametrize("rows", ROWS)
def test_a_lone_product_is_rounded_once(handle, torch_gpu, rng, rows):
    """Scaled permutations and diagonals of 24-bit factors.  The large part product is exact, and the sum of the seven
    smaller ones, below 2^-7 of it, is rounded seven times: 0.5 + 7 * 2^-8 units in the last place at most.
    The root mean square is that of a rounding, as the fp32 instructions', to 0.1 %."""
    torch = torch_gpu
    M, N, K = 2 * rows + 5, 512, 256
    for ranges in (1, 2):
        diagonal = np.zeros((K, N), np.float32)
        cols = rng.permutation(N)
        diagonal[np.arange(N) % K, cols] = rng.uniform(1, 4, N)
        X = rng.normal(size=(M, K)).astype(np.float32)
        for A, B in ((X, diagonal), (nonzeros(rng, M, K, 1), rng.normal(size=(K, N)).astype(np.float32))):
            got, what = run(handle, torch, A, B, rows, ranges, 1, 3)
            ref = A.astype(np.float64) @ B.astype(np.float64)          # one product of 48 bits: exact
            ulp = np.exp2(np.floor(np.log2(np.abs(ref))) - 23)
            off = np.abs(got - ref) / ulp
            old = np.abs(ref.astype(np.float32) - ref) / ulp
            assert off.max() <= 0.5 + 7 * 2.0 ** -8, (what, off.max())
            assert np.sqrt((off ** 2).mean()) <= 1.001 * np.sqrt((old ** 2).mean()), what


@pytest.mark.parametrize("rows", ROWS)
def test_tiny_values_beside_ordinary_ones_cost_nothing(handle, torch_gpu, rng, rows):
    """Values below 2^-110 that no result can show (a softmax's tail): bit for bit the product with zeros in their
    place, which a tile computed once more in fp32 is not (shown by a NaN in one row)."""
    torch = torch_gpu
    M, N, K = 2 * rows + 5, 300, 203
    X, Y = rng.normal(size=(M, K)).astype(np.float32), rng.normal(size=(K, N)).astype(np.float32)
    bias = rng.normal(size=N).astype(np.float32)
    tiny = np.array([1e-34, -1e-35, 1e-42, -1e-45], np.float32)
    for ranges, b in ((1, None), (2, None), (1, bias)):
        for where in ("A", "B"):
            A, B, zeros = X.copy(), Y.copy(), [X.copy(), Y.copy()]
            T, Z = (A, zeros[0]) if where == "A" else (B, zeros[1])
            at = rng.integers(0, T.size, 400)
            T.flat[at], Z.flat[at] = tiny[rng.integers(0, 4, 400)], 0
            got, what = run(handle, torch, A, B, rows, ranges, 1, 3, b)
            want, _ = run(handle, torch, *zeros, rows, ranges, 1, 3, b)
            np.testing.assert_array_equal(got, want, err_msg=f"{what} {where}")
    again = X.copy()
    again[3] = np.nan
    got, _ = run(handle, torch, again, Y, rows, 1, 1, 3)
    want, _ = run(handle, torch, X, Y, rows, 1, 1, 3)
    assert (got[:rows] != want[:rows]).mean() > 0.1 and (got[rows:] == want[rows:]).all()


@pytest.mark.parametrize("rows", ROWS)
def test_only_the_tile_that_loses_something_is_computed_again(handle, torch_gpu, rng, rows):
    """A row of zeros in the first tile of rows (results that any loss would be large beside), tiny values in the
    second: the first one's other rows keep their bits."""
    torch = torch_gpu
    M, N, K = 3 * rows, 260, 150
    A, B = rng.normal(size=(M, K)).astype(np.float32), rng.normal(size=(K, N)).astype(np.float32)
    A[5] = 0
    want, _ = run(handle, torch, A, B, rows, 1, 0, 4)
    A[rows:2 * rows, 7] = 1e-36
    got, what = run(handle, torch, A, B, rows, 1, 0, 4)
    np.testing.assert_array_equal(got[:rows], want[:rows], err_msg=what)
    # with a small row beside them, whose results the loss would show in: all of it, to fp32's precision
    A[rows + 9] = (rng.uniform(0.5, 1, K) * 2.0 ** -125).astype(np.float32)
    got, what = run(handle, torch, A, np.abs(B), rows, 1, 0, 4)
    ref = A.astype(np.float64) @ np.abs(B).astype(np.float64)
    np.testing.assert_allclose(got[rows + 9], ref[rows + 9], rtol=1e-5, err_msg=what)   # (2^-149 of some 2^-122)


@pytest.mark.parametrize("M,N,K", [(256, 4096, 4096), (700, 3000, 1600), (2048, 2048, 2048)])
def test_sums_get_no_longer_than_the_kernels_it_takes_the_place_of(handle, torch_gpu, M, N, K):
    """Positive operands, whose error grows with the length of a sum: the library's own choice against what serves
    the call without these tiles."""
    torch = torch_gpu
    gen = torch.Generator(device="cuda").manual_seed(5)
    for zeros in (0.0, 0.8):
        A, B = torch.rand((M, K), generator=gen, device="cuda"), torch.rand((K, N), generator=gen, device="cuda")
        A *= torch.rand((M, K), generator=gen, device="cuda") >= zeros
        ref = A.double() @ B.double()
        got = handle.gemm_f32(A, B)
        assert "x256x16_w4" in handle.last_kernel and "32x32x2" not in handle.last_kernel, handle.last_kernel
        probe.force_f32_split(handle, -1)
        old = handle.gemm_f32(A, B)
        assert "x256x16_w4" not in handle.last_kernel or "32x32x2" in handle.last_kernel
        probe.force_f32_split(handle, 0)
        assert float((got - ref).norm()) <= 1.01 * float((old - ref).norm()), zeros


@pytest.mark.parametrize("rows", ROWS)
def test_infinities_nan_and_extreme_magnitudes(handle, torch_gpu, rng, rows):
    """One value in the last row / column block of A or B, everything else ordinary: the rows and columns
    it reaches are those of float64 rounded to fp32, NaN and the sign of infinity included."""
    M, N, K = rows + 3, 270, 75
    big = np.float32(np.finfo(np.float32).max)
    for value in (np.inf, -np.inf, np.nan, big, -big, np.float32(1.2345678 * 2.0 ** -120), np.float32(2.0 ** -145)):
        for where in ("A", "B"):
            A = rng.choice([-1.0, 0.5, 1.0], size=(M, K)).astype(np.float32)
            B = rng.choice([-1.0, 0.5, 1.0], size=(K, N)).astype(np.float32)
            if abs(value) < 1:      # alone in its row (column), so that nothing larger hides it
                if where == "A":
                    A[M - 1] = 0
                else:
                    B[:, N - 1] = 0
            if where == "A":
                A[M - 1, 40] = value
            else:
                B[40, N - 1] = value
            for ranges in (1, 2):
                got, what = run(handle, torch_gpu, A, B, rows, ranges, 0, 0)
                with np.errstate(all="ignore"):
                    ref = (A.astype(np.float64) @ B.astype(np.float64)).astype(np.float32)
                np.testing.assert_allclose(got, ref, rtol=2e-6, atol=0, err_msg=f"{what} {value} in {where}")


@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("exponent", [-100, -102, -103, -106, -109, -110, -111, -118, -126, -133])
def test_lower_edge_of_the_parts(handle, torch_gpu, rng, rows, exponent):
    """Factors of 24 bits around 2^-110, whose third part is a subnormal bf16 number or lost, selected by one power of two
    of the other operand: bit for bit (2^100 scales nothing away)."""
    M, N, K = rows + 3, 259, 70
    scale = np.float32(2.0 ** 100)
    X = (rng.uniform(1, 2, size=(M, K)) * rng.choice([-1, 1], size=(M, K)) * 2.0 ** exponent).astype(np.float32)
    take = rng.integers(0, K, size=N)
    W = np.zeros((K, N), np.float32)
    W[take, np.arange(N)] = scale
    got, what = run(handle, torch_gpu, X, W, rows, 1, 1, 3)
    np.testing.assert_array_equal(got, X[:, take] * scale, err_msg=what)
    Y = (rng.uniform(1, 2, size=(K, N)) * 2.0 ** exponent).astype(np.float32)
    take = rng.integers(0, K, size=M)
    S = np.zeros((M, K), np.float32)
    S[np.arange(M), take] = -scale
    got, what = run(handle, torch_gpu, S, Y, rows, 2, 0, 4)
    np.testing.assert_array_equal(got, Y[take] * -scale, err_msg=what)


@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("exponent", [-108, -118, -122, -126, -130, -140])
def test_products_of_ordinary_values_near_the_smallest_numbers(handle, torch_gpu, rng, rows, exponent):
    """Lone products around 2^exponent, whose smaller part products are subnormal sums: as close as a product of
    ordinary size (test_a_lone_product_is_rounded_once) plus eight roundings to 2^-149."""
    M, N, K = rows + 3, 259, 70
    half = exponent // 2
    A = nonzeros(rng, M, K, 1)
    A[A != 0] = rng.uniform(1, 2, M) * 2.0 ** half
    B = (rng.uniform(1, 2, size=(K, N)) * 2.0 ** (exponent - half)).astype(np.float32)
    got, what = run(handle, torch_gpu, A, B, rows, 1, 1, 3)
    ref = A.astype(np.float64) @ B.astype(np.float64)
    ulp = np.maximum(np.exp2(np.floor(np.log2(ref)) - 23), 2.0 ** -149)
    assert (np.abs(got - ref) <= (0.5 + 7 * 2.0 ** -8) * ulp + 8 * 2.0 ** -150).all(), (what, np.max(np.abs(got - ref) / ulp))


def test_tiny_values_anywhere_are_not_lost(handle, torch_gpu, rng):
    """Rows of subnormal size times large columns: relative precision as of ordinary values."""
    M, N, K = 200, 300, 130
    A = (rng.uniform(0.5, 1, size=(M, K)) * 2.0 ** -122).astype(np.float32)
    B = (rng.uniform(0.5, 1, size=(K, N)) * 2.0 ** 100).astype(np.float32)
    ref = A.astype(np.float64) @ B.astype(np.float64)
    for rows in ROWS:
        got, what = run(handle, torch_gpu, A, B, rows, 1, 0, 0)
        np.testing.assert_allclose(got, ref, rtol=1e-6, err_msg=what)


@pytest.mark.parametrize("M,N,K", [(1454, 896, 704), (537, 2560, 640), (660, 4096, 704), (50, 16000, 8000),
                                   (20000, 512, 784)])
def test_left_to_the_kernels_that_are_faster(handle, torch_gpu, M, N, K):
    """us, there and here: 26.5 and 31.5, 25.1 and 28.9, 46.5 and 52.9; a long B on 64 rows; 115 and 119."""
    handle.gemm_f32(torch_gpu.zeros((M, K), device="cuda"), torch_gpu.zeros((K, N), device="cuda"))
    assert "x256x16_w4" not in handle.last_kernel or "32x32x2" in handle.last_kernel, handle.last_kernel


def test_default_takes_it_where_it_pays_and_graphs_replay(handle, torch_gpu, rng):
    """The library's own choice on a size of two launches, one of K ranges and two (one a layer with bias) with the
    remaining column on the kernel of small outputs, recorded and replayed with other work between."""
    torch = torch_gpu
    draw = lambda *s: torch.rand(s, device="cuda") - 0.5  # noqa: E731
    sizes = ((1300, 6000, 1500, None), (256, 4096, 4096, None), (4095, 4097, 1031, None), (4095, 4097, 1031, draw(4097)))
    plans = (r"f32_mfma_128\+64x256x16_w4\+w4_ring4_splitk", r"f32_mfma_128x256x16_w4_ring4_splitk",
             r"f32_mfma_any_128x256x16_w4_ring4\+32x32", r"f32_mfma_any_128x256x16_w4_ring4_bias_act\+32x32")
    ops = [(draw(M, K), draw(K, N), torch.empty((M, N), device="cuda"), bias) for M, N, K, bias in sizes]
    side = torch.cuda.Stream()
    h = ci.Handle(stream=side)

    def sequence():
        names = []
        for a, b, out, bias in ops:
            if bias is None:
                h.gemm_f32(a, b, out=out)
            else:
                h.linear_f32(a, b, bias, ci.ACT_RELU, out=out)
            names.append(h.last_kernel)
        return names

    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        names = sequence()
    side.synchronize()
    for name, plan in zip(names, plans):
        assert re.fullmatch(plan, name), (name, plan)
    eager = [o[2].clone() for o in ops]
    for (a, b, _, bias), got in zip(ops, eager):
        ref = a.double() @ b.double()
        bound = 1e-5 * float(ref.pow(2).mean().sqrt()) * 4
        if bias is not None:
            ref = (ref + bias).clamp_min(0)
        assert float((got - ref).abs().max()) <= bound
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        sequence()
    for _ in range(3):
        for o in ops:
            o[2].fill_(float("nan"))
        handle.gemm_f32(ops[1][0], ops[1][1])
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for o, e in zip(ops, eager):
            assert torch.equal(o[2], e)
    h.close()
