"""Outputs of a few columns more than full rounds of 256-row tiles: the rest runs on the kernel of small
outputs.  One column, less than a 16-byte piece, a piece, 64 columns (65 are the tile kernel's again);
aligned rows and rows off by an element; bias and per-column scales that start at a column of their own.
Reference: torch in 64 bits on operands whose sums are exact in 32; the output sits in a sentinel-filled
buffer."""
import numpy as np
import pytest

import cudaintro_amd as ci
from test_gpu_mfma_any import VALS

pytestmark = pytest.mark.gpu
BYTES = {"bf16": 2, "f16": 2, "f32": 4, "i8_kn": 1, "i8_nk": 1}


@pytest.mark.parametrize("rest", [1, 3, 16, 64, 65])
@pytest.mark.parametrize("kind", list(BYTES))
def test_rest_columns(handle, torch_gpu, rng, kind, rest):
    torch = torch_gpu
    int8 = kind.startswith("i8")
    layout = ci.B_NK if kind == "i8_nk" else ci.B_KN
    dt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}.get(kind, torch.int8)
    odt = torch.int32 if int8 else dt
    m, n = 4090, 4096 + rest
    for K, off, pad in ((8 * 128 // BYTES[kind], 0, -n % 16), (1031, 1, 3)):
        def operand(r, c):
            src = rng.integers(-127, 128, size=(r, c), dtype=np.int8) if int8 else rng.choice(VALS, size=(r, c))
            gap = -c % 16 if off == 0 else 3
            flat = torch.full((off + r * (c + gap),), 127 if int8 else float("nan"), dtype=dt, device="cuda")
            view = flat[off:].view(r, c + gap)[:, :c]
            view.copy_(torch.from_numpy(src).cuda())
            return view
        a = operand(m, K)
        b = operand(n, K) if kind == "i8_nk" else operand(K, n)
        ref = a.double() @ (b.t() if kind == "i8_nk" else b).double().contiguous()

        def run(call, dtype, want):
            flat = torch.full((off + m * (n + pad),), 7, dtype=dtype, device="cuda")
            out = flat[off:].view(m, n + pad)[:, :n]
            call(out)
            assert ("+32x" in handle.last_kernel) == (rest <= 64), handle.last_kernel
            assert torch.equal(out, want.to(dtype)), (handle.last_kernel, K)
            out.fill_(7)
            assert bool((flat == 7).all()), "a store outside the output"

        if not int8:
            run(lambda o: getattr(handle, "gemm_" + kind)(a, b, out=o), odt, ref)
            if kind == "f32":
                bias = torch.from_numpy(rng.choice(VALS, size=n)).cuda()
                run(lambda o: handle.linear_f32(a, b, bias, ci.ACT_RELU, out=o), odt, torch.relu(ref + bias.double()))
                run(lambda o: handle.linear_f32(a, b, None, ci.ACT_NONE, out=o), odt, ref)
        else:
            run(lambda o: handle.gemm_i8_i32(a, b, layout, out=o), odt, ref)
            # scales that are powers of two: the product is exact, whatever its order
            sa, sb = (torch.from_numpy(np.ldexp(np.float32(1), rng.integers(-6, 1, size=s)).astype(np.float32)).cuda()
                      for s in (m, n))
            for x, y in ((sa, sb), (sa[:1], sb[:1])):
                scaled = (ref * x.double()[:, None] * y.double()[None, :]).to(torch.float32)
                for ot, t in ((ci.OUT_F32, torch.float32), (ci.OUT_BF16, torch.bfloat16)):
                    run(lambda o: handle.gemm_i8_dequant(a, b, x, y, layout, ot, out=o), t, scaled)
