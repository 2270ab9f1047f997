"""The tile kernel at any alignment, at the sizes where it can go wrong: every tile height, K
around its 64-byte stages (all of K in the separately multiplied tail, one stage, an odd and an
even number of them, a tail of one element up to a whole stage), one and several K ranges (a last
range that is only tail among them), edge and interior tiles, every operand off by an element.
Operand values are small integers and halves, so every sum is exact and the comparison is bit for
bit; the padding around the operands is NaN (127 for int8), the output sits in a sentinel-filled
buffer."""
import re

import numpy as np
import pytest

import cudaintro_amd as ci
from cudaintro_amd import probe
from gpu_util import bits
from test_gpu_mfma_any import VALS, embed

pytestmark = pytest.mark.gpu
M, N = 300, 521
BYTES = {"bf16": 2, "f16": 2, "f32": 4, "i8_kn": 1, "i8_nk": 1}


def sizes_of_k(eb):
    stage = 64 // eb
    return [16 // eb, stage, stage + 1, 2 * stage, 2 * stage + 1, 13 * stage + 3, 25 * stage - 1]


@pytest.mark.parametrize("rows", [256, 192, 128, 64])
@pytest.mark.parametrize("kind", list(BYTES))
def test_tile_any(handle, torch_gpu, oracle, rng, kind, rows):
    torch = torch_gpu
    int8 = kind.startswith("i8")
    layout = ci.B_NK if kind == "i8_nk" else ci.B_KN
    for K in sizes_of_k(BYTES[kind]):
        if int8:
            A = rng.integers(-127, 128, size=(M, K), dtype=np.int8)
            B = rng.integers(-127, 128, size=(N, K) if layout == ci.B_NK else (K, N), dtype=np.int8)
            dt, odt, pad, ref = torch.int8, torch.int32, 127, oracle.gemm_i8_i32(A, B, b_is_nk=layout == ci.B_NK)
        else:
            A, B = rng.choice(VALS, size=(M, K)), rng.choice(VALS, size=(K, N))
            ref = oracle.gemm_f32(A, B)
            dt = odt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[kind]
            pad = float("nan")
            narrow = {"bf16": oracle.f32_to_bf16, "f16": oracle.f32_to_f16}.get(kind)
            if narrow:
                A, B, ref = narrow(A).view(np.int16), narrow(B).view(np.int16), narrow(ref)
        _, a = embed(torch, A, dt, 1, 3, pad)
        _, b = embed(torch, B, dt, 3, 1, pad)
        flat, out = embed(torch, np.zeros((M, N), np.int32).astype(np.int16 if odt.itemsize == 2 else np.int32),
                          odt, 1, 5, 0)
        guard = np.ones(flat.numel(), bool)
        for i in range(M):
            guard[1 + i * (N + 5): 1 + i * (N + 5) + N] = False
        host = lambda t: bits(torch, t) if t.element_size() == 2 else t.contiguous().cpu().numpy()  # noqa: E731
        for ranges in (1, 3):
            flat.fill_(7)
            sentinel = host(flat)[0]
            probe.force_tile_plan(handle, rows, ranges)
            try:
                with handle.algo(ci.ALGO_MFMA_ANY):
                    if int8:
                        handle.gemm_i8_i32(a, b, layout, out=out)
                    else:
                        getattr(handle, "gemm_" + kind)(a, b, out=out)
                    assert f"_mfma_any_{rows}x256" in handle.last_kernel, handle.last_kernel
                    np.testing.assert_array_equal(host(out), ref, err_msg=f"K={K} ranges={ranges}")
                    assert (host(flat)[guard] == sentinel).all()
                    if int8:
                        sa = rng.uniform(1e-3, 5e-2, M).astype(np.float32)
                        sb = rng.uniform(1e-3, 5e-2, N).astype(np.float32)
                        for name, ot in (("f32", ci.OUT_F32), ("bf16", ci.OUT_BF16)):
                            y = handle.gemm_i8_dequant(a, b, torch.from_numpy(sa).cuda(),
                                                       torch.from_numpy(sb).cuda(), layout, ot)
                            np.testing.assert_array_equal(
                                host(y), oracle.dequant(ref, sa, sb, out_dtype=name, sa_per_row=True,
                                                        sb_per_col=True))
                    elif kind == "f32":
                        bias = rng.choice(VALS, size=N)
                        y = handle.linear_f32(a, b, torch.from_numpy(bias).cuda(), ci.ACT_RELU)
                        np.testing.assert_array_equal(host(y), oracle.linear_f32(A, B, bias, True))
            finally:
                probe.force_tile_plan(handle, 0)


@pytest.mark.parametrize("kind", list(BYTES))
def test_every_width_of_the_last_piece(handle, torch_gpu, oracle, rng, kind):
    """Rows that end with 0 to 7 elements of a 16-byte piece, 16- and 32-bit outputs, the next row
    directly behind them."""
    torch = torch_gpu
    int8 = kind.startswith("i8")
    layout = ci.B_NK if kind == "i8_nk" else ci.B_KN
    m, K = 70, 75
    for n in range(264, 272):
        if int8:
            A = rng.integers(-127, 128, size=(m, K), dtype=np.int8)
            B = rng.integers(-127, 128, size=(n, K) if layout == ci.B_NK else (K, n), dtype=np.int8)
            acc = oracle.gemm_i8_i32(A, B, b_is_nk=layout == ci.B_NK)
            sa, sb = (rng.uniform(1e-3, 5e-2, k).astype(np.float32) for k in (m, n))
            a, b, da, db = (torch.from_numpy(v).cuda() for v in (A, B, sa, sb))
            with probe.any_kernel(handle, probe.ANY_TILE):
                np.testing.assert_array_equal(handle.gemm_i8_i32(a, b, layout).cpu().numpy(), acc)
                y = handle.gemm_i8_dequant(a, b, da, db, layout, ci.OUT_BF16)
            assert "_mfma_any_64x256" in handle.last_kernel, handle.last_kernel
            np.testing.assert_array_equal(bits(torch, y), oracle.dequant(acc, sa, sb, out_dtype="bf16",
                                                                         sa_per_row=True, sb_per_col=True))
            continue
        A, B = rng.choice(VALS, size=(m, K)), rng.choice(VALS, size=(K, n))
        dt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[kind]
        with probe.any_kernel(handle, probe.ANY_TILE):
            y = getattr(handle, "gemm_" + kind)(torch.from_numpy(A).cuda().to(dt), torch.from_numpy(B).cuda().to(dt))
        assert "_mfma_any_64x256" in handle.last_kernel, handle.last_kernel
        assert torch.equal(y.cpu(), torch.from_numpy(oracle.gemm_f32(A, B)).to(dt)), n


# Columns left over by the full rounds of 256-row tiles: fewer than a 16-byte piece (the second
# launch then covers columns that are narrower than one piece), one piece, more than one tile.
@pytest.mark.parametrize("rest", ["one", "piece - 1", "piece", "tile + 1"])
@pytest.mark.parametrize("kind", list(BYTES))
def test_two_launches(handle, torch_gpu, rng, kind, rest):
    """The two-launch plan on unaligned rows: 16 x 16 tiles of 256 rows, the rest of the columns as
    a second launch with its own plan (of one K range for the short K, several where the planner
    splits the long one), so that output, bias and per-column scales start at a column of their own.
    Reference: torch in 64 bits, on operands whose sums are exact in 32."""
    torch = torch_gpu
    eb = BYTES[kind]
    m = 4095
    n = 4096 + {"one": 1, "piece - 1": max(2, 16 // eb - 1), "piece": 16 // eb, "tile + 1": 257}[rest]
    int8 = eb == 1
    layout = ci.B_NK if kind == "i8_nk" else ci.B_KN
    dt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}.get(kind, torch.int8)
    odt = torch.int32 if int8 else dt
    for K in (16 // eb + 1, 1025):
        def operand(r, c, off, pad):
            src = rng.integers(-127, 128, size=(r, c), dtype=np.int8) if int8 else rng.choice(VALS, size=(r, c))
            flat = torch.full((off + r * (c + pad) + 3,), 127 if int8 else float("nan"), dtype=dt, device="cuda")
            view = flat[off: off + r * (c + pad)].view(r, c + pad)[:, :c]
            view.copy_(torch.from_numpy(src).cuda())
            return view
        a = operand(m, K, 1, 2)
        b = operand(n, K, 3, 1) if kind == "i8_nk" else operand(K, n, 3, 2)
        ref = a.double() @ (b.t() if kind == "i8_nk" else b).double().contiguous()
        flat = torch.full((1 + m * (n + 3),), 7, dtype=odt, device="cuda")
        out = flat[1:].view(m, n + 3)[:, :n]

        def check(want, name=""):
            assert re.search(r"_mfma_any_256\+\d+x256x", handle.last_kernel), handle.last_kernel
            assert torch.equal(out, want), (K, name, (out != want).nonzero()[:4].tolist())
            out.fill_(7)
            assert bool((flat == 7).all()), "a store outside the output"

        with probe.any_kernel(handle, probe.ANY_TILE):
            if not int8:
                getattr(handle, "gemm_" + kind)(a, b, out=out)
                check(ref.to(odt))
                if kind == "f32":
                    bias = torch.from_numpy(rng.choice(VALS, size=n + 1)).cuda()[1:]
                    handle.linear_f32(a, b, bias, ci.ACT_RELU, out=out)
                    check(torch.relu(ref + bias.double()).to(odt), "bias + ReLU")
            else:
                handle.gemm_i8_i32(a, b, layout, out=out)
                check(ref.to(odt))
                # scales that are powers of two: the product is exact, whatever its order
                sa = torch.from_numpy(np.ldexp(np.float32(1), rng.integers(-6, 1, size=m)).astype(np.float32)).cuda()
                sb = torch.from_numpy(np.ldexp(np.float32(1), rng.integers(-6, 1, size=n + 1)).astype(np.float32)).cuda()[1:]
                scaled = ref * sa.double()[:, None] * sb.double()[None, :]
                for ot, t in ((ci.OUT_F32, torch.float32), (ci.OUT_BF16, torch.bfloat16)):
                    flat = torch.full((1 + m * (n + 3),), 7, dtype=t, device="cuda")
                    out = flat[1:].view(m, n + 3)[:, :n]
                    handle.gemm_i8_dequant(a, b, sa, sb, layout, ot, out=out)
                    check(scaled.to(torch.float32).to(t), t)
