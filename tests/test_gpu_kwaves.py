"""The kernel of small outputs (32 x 64 tiles, fp32 32 x 32, k shared out to four waves, K ranges joined inside the
kernel) at the sizes where it can go wrong: M and N around its tiles, K around its 128-byte pieces (all
of K in the separately multiplied tail, fewer pieces than waves, more than its slots hold, a tail of one
element up to a whole piece, in every wave), one and several K ranges, aligned and unaligned operands.  Operand
values are small integers and halves, so every sum is exact in any order and the comparison is bit for
bit; the padding around the operands is NaN (127 for int8), the output sits in a sentinel-filled
buffer.  Every call runs twice: the second finds the workspace as the first left it."""
import numpy as np
import pytest

import cudaintro_amd as ci
from cudaintro_amd import probe
from gpu_util import bits
from test_gpu_mfma_any import VALS, embed

pytestmark = pytest.mark.gpu
BYTES = {"bf16": 2, "f16": 2, "f32": 4, "i8_kn": 1, "i8_nk": 1}
SHAPES = [  # M, N, aligned
    (33, 136, True), (129, 260, True), (200, 384, True), (65, 64, True),
    (64, 127, False), (130, 193, False), (257, 33, False),
]


def sizes_of_k(eb, aligned):
    stage, piece = 128 // eb, 16 // eb
    if aligned:
        return [piece, stage, 3 * stage, 5 * stage, 6 * stage, 15 * stage + 3 * piece]
    return [piece, stage + 1, 4 * stage + 1, 7 * stage - 1, 14 * stage]


@pytest.mark.parametrize("kind", list(BYTES))
def test_kwaves(handle, torch_gpu, oracle, rng, kind):
    torch = torch_gpu
    int8 = kind.startswith("i8")
    layout = ci.B_NK if kind == "i8_nk" else ci.B_KN
    name = "small_kwaves_32x32x32" if kind == "f32" else "kwaves_32x64"
    host = lambda t: bits(torch, t) if t.element_size() == 2 else t.contiguous().cpu().numpy()  # noqa: E731
    for M, N, aligned in SHAPES:
        for K in sizes_of_k(BYTES[kind], aligned):
            if int8:
                A = rng.integers(-127, 128, size=(M, K), dtype=np.int8)
                B = rng.integers(-127, 128, size=(N, K) if layout == ci.B_NK else (K, N), dtype=np.int8)
                ref = oracle.gemm_i8_i32(A, B, b_is_nk=layout == ci.B_NK)
                dt, odt, pad = torch.int8, torch.int32, 127
            else:
                A, B = rng.choice(VALS, size=(M, K)), rng.choice(VALS, size=(K, N))
                ref = oracle.gemm_f32(A, B)
                dt = odt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[kind]
                pad = float("nan")
                narrow = {"bf16": oracle.f32_to_bf16, "f16": oracle.f32_to_f16}.get(kind)
                if narrow:
                    A, B, ref = narrow(A).view(np.int16), narrow(B).view(np.int16), narrow(ref)
            # rows of whole 16-byte pieces at offset 0, or everything off by an element
            step = 16 // BYTES[kind]
            off, fill = (0, lambda c, e: -c % e) if aligned else (1, lambda c, e: 3)
            _, a = embed(torch, A, dt, off, fill(A.shape[1], step), pad)
            _, b = embed(torch, B, dt, off, fill(B.shape[1], step), pad)
            po = fill(N, 16 // odt.itemsize)
            flat, out = embed(torch, np.zeros((M, N), np.int32).astype(np.int16 if odt.itemsize == 2 else np.int32),
                              odt, off, po, 0)
            guard = np.ones(flat.numel(), bool)
            for i in range(M):
                guard[off + i * (N + po): off + i * (N + po) + N] = False
            for ranges in (1, 2, 3, 5):
                probe.force_kwaves_plan(handle, ranges)
                try:
                    for _ in range(2):
                        flat.fill_(7)
                        sentinel = host(flat)[0]
                        if int8:
                            handle.gemm_i8_i32(a, b, layout, out=out)
                        else:
                            getattr(handle, "gemm_" + kind)(a, b, out=out)
                        assert name in handle.last_kernel, handle.last_kernel
                        assert handle.last_plan[0] == 32    # (0: the register-loaded fp32 kernel)
                        what = f"{handle.last_kernel} {handle.last_plan} M={M} N={N} K={K}"
                        np.testing.assert_array_equal(host(out), ref, err_msg=what)
                        assert (host(flat)[guard] == sentinel).all(), what
                    if int8:
                        sa = rng.uniform(1e-3, 5e-2, M).astype(np.float32)
                        sb = rng.uniform(1e-3, 5e-2, N).astype(np.float32)
                        for out_name, ot in (("f32", ci.OUT_F32), ("bf16", ci.OUT_BF16)):
                            y = handle.gemm_i8_dequant(a, b, torch.from_numpy(sa).cuda(),
                                                       torch.from_numpy(sb).cuda(), layout, ot)
                            assert name in handle.last_kernel, handle.last_kernel
                            np.testing.assert_array_equal(
                                host(y), oracle.dequant(ref, sa, sb, out_dtype=out_name, sa_per_row=M > 1,
                                                        sb_per_col=True), err_msg=what)
                            y = handle.gemm_i8_dequant(a, b, torch.from_numpy(sa[:1]).cuda(),
                                                       torch.from_numpy(sb[:1]).cuda(), layout, ot)
                            np.testing.assert_array_equal(
                                host(y), oracle.dequant(ref, sa[:1], sb[:1], out_dtype=out_name), err_msg=what)
                    elif kind == "f32":
                        bias = rng.choice(VALS, size=N)
                        y = handle.linear_f32(a, b, torch.from_numpy(bias).cuda(), ci.ACT_RELU)
                        assert name in handle.last_kernel, handle.last_kernel
                        np.testing.assert_array_equal(host(y), oracle.linear_f32(A, B, bias, True), err_msg=what)
                finally:
                    probe.force_kwaves_plan(handle, 0)


@pytest.mark.parametrize("kind,M,N,K", [("bf16", 52, 64, 4096), ("f32", 95, 96, 4099), ("bf16", 2048, 8200, 512)])
def test_replayed_from_a_graph(torch_gpu, kind, M, N, K):
    """K ranges and a remainder of columns recorded and replayed, eager calls of another size on the same handle
    in between: every replay finds the counters at zero and gives the eager bits."""
    torch = torch_gpu
    dt = {"bf16": torch.bfloat16, "f32": torch.float32}[kind]
    gen = torch.Generator(device="cuda").manual_seed(5)
    new = lambda r, c: torch.randn((r, c), generator=gen, device="cuda").to(dt)  # noqa: E731
    a, b, a2, b2 = new(M, K), new(K, N), new(40, 2048), new(2048, 128)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side), ci.Handle() as h:
        gemm = getattr(h, "gemm_" + kind)
        want, want2 = gemm(a, b), gemm(a2, b2)
        gemm(a, b)
        if N > 256:
            assert h.last_kernel.endswith("+32x64"), h.last_kernel
        else:
            assert "kwaves" in h.last_kernel and h.last_plan[0] == 32 and h.last_plan[1] > 1, (h.last_kernel, h.last_plan)
        out = torch.zeros_like(want)
        graph = torch.cuda.CUDAGraph()
        side.synchronize()
        with torch.cuda.graph(graph, stream=side):
            gemm(a, b, out=out)
        for _ in range(4):
            out.zero_()
            graph.replay()
            assert torch.equal(gemm(a2, b2), want2)
            side.synchronize()
            assert torch.equal(out, want)


# (M, N of 16-bit and int8, N of fp32, whole pieces of k, K ranges imposed, regime): a wave has more pieces than
# slots, so that a slot is filled again while others are in flight; more workgroups than units, so that
# its one slot is; more than eight ranges, which the last workgroup adds up in groups of eight.
REGIMES = [
    (33, 136, 72, 40, 1, "ring"), (65, 200, 136, 53, 2, "ring"),
    (520, 1040, 1040, 9, 1, "one slot"), (520, 1040, 520, 22, 2, "one slot"), (545, 1100, 1100, 17, 1, "one slot"),
    (64, 136, 72, 18, 9, "ranges"), (33, 72, 40, 31, 16, "ranges"), (70, 200, 104, 45, 12, "ranges"),
]


@pytest.mark.parametrize("M,n,n32,pieces,ranges,regime", REGIMES)
@pytest.mark.parametrize("kind", list(BYTES))
def test_regimes(handle, torch_gpu, rng, kind, M, n, n32, pieces, ranges, regime):
    """Every regime is asked for by its definition (slots, pieces of a wave, ranges), with and without a tail of
    k, aligned and off by an element.  Reference: torch in 64 bits on operands whose sums are exact in 32."""
    torch = torch_gpu
    int8 = kind.startswith("i8")
    layout = ci.B_NK if kind == "i8_nk" else ci.B_KN
    dt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}.get(kind, torch.int8)
    odt = torch.int32 if int8 else dt
    units = torch.cuda.get_device_properties(0).multi_processor_count
    stage, N, tn, max_slots = 128 // BYTES[kind], n32 if kind == "f32" else n, 32 if kind == "f32" else 64, \
        4 if kind == "f32" else 3
    for tail, off in ((0, 0), (0, 1), (1, 1), (stage - 1, 1), (stage // 8, 0)):
        # (one piece less where a tail follows: `ranges` ranges of an even number of 64-byte stages)
        K = (pieces - (tail > 0)) * stage + tail

        def operand(r, c):
            src = rng.integers(-127, 128, size=(r, c), dtype=np.int8) if int8 else rng.choice(VALS, size=(r, c))
            ld = c + (-c % 16 if off == 0 else 3)
            flat = torch.full((off + r * ld,), 127 if int8 else float("nan"), dtype=dt, device="cuda")
            view = flat[off:].view(r, ld)[:, :c]
            view.copy_(torch.from_numpy(src).cuda())
            return view
        a = operand(M, K)
        b = operand(N, K) if kind == "i8_nk" else operand(K, N)
        ref = (a.double() @ (b.t() if kind == "i8_nk" else b).double().contiguous()).to(odt)
        ld = N + (-N % 16 if off == 0 else 3)
        flat = torch.empty(off + M * ld, dtype=odt, device="cuda")
        out = flat[off:].view(M, ld)[:, :N]
        probe.force_kwaves_plan(handle, ranges)
        try:
            for _ in range(2):
                flat.fill_(7)
                if int8:
                    handle.gemm_i8_i32(a, b, layout, out=out)
                else:
                    getattr(handle, "gemm_" + kind)(a, b, out=out)
                what = f"{handle.last_kernel} {handle.last_plan} {M} {N} {K}"
                assert "kwaves_32x" in handle.last_kernel and handle.last_plan[0] == 32, what
                got = handle.last_plan[1]
                workgroups = -(-M // 32) * -(-N // tn) * got
                of_a_wave = -(-(-(-K // stage) // got) // 4)
                assert {"ring": workgroups <= units and of_a_wave > max_slots,
                        "one slot": workgroups > units and of_a_wave > 1,
                        "ranges": got > 8 and got == ranges}[regime], (what, workgroups, of_a_wave)
                assert torch.equal(out, ref), what
                out.fill_(7)
                assert bool((flat == 7).all()), what
        finally:
            probe.force_kwaves_plan(handle, 0)
