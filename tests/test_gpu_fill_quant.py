"""Device generators and quantizer against the oracle, bit for bit, through the C ABI."""
import json
import os

import numpy as np
import pytest

from gpu_util import bits

pytestmark = pytest.mark.gpu
HERE = os.path.dirname(os.path.abspath(__file__))
KAT = json.load(open(os.path.join(HERE, "golden", "fill_random_kat.json")))


@pytest.mark.parametrize("count", [0, 1, 7, 255, 256, 1000003, 1 << 24])
def test_fill_f32(handle, torch_gpu, oracle, count):
    t = torch_gpu.empty(count, dtype=torch_gpu.float32, device="cuda")
    handle.fill_random(t, 0x3234)
    np.testing.assert_array_equal(t.cpu().numpy().view(np.uint32),
                                  oracle.fill_random_f32(count, 0x3234).view(np.uint32))


@pytest.mark.parametrize("dtype,seed,fn", [("bfloat16", 0x1234, "fill_random_bf16"),
                                           ("bfloat16", 0x9876, "fill_random_bf16"),
                                           ("float16", 0x2234, "fill_random_f16"),
                                           ("float16", 0x8876, "fill_random_f16")])
def test_fill_16(handle, torch_gpu, oracle, dtype, seed, fn):
    for count in (5, 4099, 1 << 24):
        t = torch_gpu.empty(count, dtype=getattr(torch_gpu, dtype), device="cuda")
        handle.fill_random(t, seed)
        np.testing.assert_array_equal(bits(torch_gpu, t), getattr(oracle, fn)(count, seed))


@pytest.mark.parametrize("seed", [0x4234, 0x6676])
def test_fill_i8(handle, torch_gpu, oracle, seed):
    for count in (3, 4097, 1 << 24):
        t = torch_gpu.empty(count, dtype=torch_gpu.int8, device="cuda")
        handle.fill_random(t, seed, -127, 127)
        np.testing.assert_array_equal(t.cpu().numpy(), oracle.fill_random_i8(count, seed))


def test_fill_golden_vectors(handle, torch_gpu):
    idx = KAT["idx"]
    n = max(idx) + 1
    for seed, vals in KAT["f32"].items():
        t = handle.fill_random(torch_gpu.empty(n, dtype=torch_gpu.float32, device="cuda"), int(seed, 16))
        assert t.cpu().numpy().view(np.uint32)[idx].tolist() == vals
    for seed, vals in KAT["bf16"].items():
        t = handle.fill_random(torch_gpu.empty(n, dtype=torch_gpu.bfloat16, device="cuda"), int(seed, 16))
        assert bits(torch_gpu, t)[idx].tolist() == vals
    for seed, vals in KAT["f16"].items():
        t = handle.fill_random(torch_gpu.empty(n, dtype=torch_gpu.float16, device="cuda"), int(seed, 16))
        assert bits(torch_gpu, t)[idx].tolist() == vals
    for seed, vals in KAT["i8"].items():
        t = handle.fill_random(torch_gpu.empty(n, dtype=torch_gpu.int8, device="cuda"), int(seed, 16), -127, 127)
        assert t.cpu().numpy()[idx].tolist() == vals


def test_fill_unaligned_and_other_range(handle, torch_gpu, oracle):
    base = torch_gpu.zeros(1000, dtype=torch_gpu.float32, device="cuda")
    handle.fill_random(base[3:903], 99, lo=0.0, hi=4.0)   # pointer 12 bytes past alignment
    got = base.cpu().numpy()
    np.testing.assert_array_equal(got[3:903], oracle.fill_random_f32(900, 99, 0.0, 4.0))
    assert (got[:3] == 0).all() and (got[903:] == 0).all()
    b = torch_gpu.zeros(1001, dtype=torch_gpu.int8, device="cuda")
    handle.fill_random(b[1:], 5, -5, 9)
    got = b.cpu().numpy()
    np.testing.assert_array_equal(got[1:], oracle.fill_random_i8(1000, 5, -5, 9))
    assert got[0] == 0


@pytest.mark.parametrize("shape", [(1, 1), (3, 5), (64, 300), (257, 4096), (2048, 4096), (7, 1028),
                                   (4, 2052), (5, 8192), (3, 16384), (2, 16388), (3, 4098)])
def test_quantize_rows(handle, torch_gpu, oracle, rng, shape):
    x = rng.normal(size=shape).astype(np.float32)
    x[0] = 0.0   # zero row
    if shape[1] >= 4:
        x[-1, :4] = [1.5, -1.5, 3.0, -3.0]
    q, s = handle.quantize_rows_i8(torch_gpu.from_numpy(x).cuda())
    qe, se = oracle.quantize_rows_i8(x)
    np.testing.assert_array_equal(s.cpu().numpy(), se)
    np.testing.assert_array_equal(q.cpu().numpy(), qe)


@pytest.mark.parametrize("pad", [4, 1])
def test_quantize_rows_of_a_wider_matrix(handle, torch_gpu, oracle, rng, pad):
    """Rows with a leading dimension above the column count: rows that stay 16-byte
    aligned and rows that do not; same bits."""
    rows, cols = 33, 1024
    wide = rng.normal(size=(rows, cols + pad)).astype(np.float32) * 3
    xd = torch_gpu.from_numpy(wide).cuda()[:, :cols]
    q, s = handle.quantize_rows_i8(xd)
    qe, se = oracle.quantize_rows_i8(np.ascontiguousarray(wide[:, :cols]))
    np.testing.assert_array_equal(s.cpu().numpy(), se)
    np.testing.assert_array_equal(q.cpu().numpy(), qe)


@pytest.mark.parametrize("shape", [(1, 1025), (300, 1027), (2, 2049), (257, 2047), (5, 4097),
                                   (300, 4099), (260, 8193), (2, 16383), (260, 16381),
                                   (2, 16385),
                                   # a wave per row, rows that leave the last workgroup part full
                                   (5, 1), (301, 3), (302, 255), (3, 256), (303, 257), (301, 510),
                                   (301, 513), (259, 1023), (258, 1024), (256, 1023)])
@pytest.mark.parametrize("scale", [1.0, 1e-36, 1e-41, 1e36])  # 127e36 is still finite
def test_quantize_rows_close_to_halves(handle, torch_gpu, oracle, rng, shape, scale):
    """Quotients on a half and one or two ulp beside it, where an estimated quotient can round to
    the other side; rows of any length, one piece or several per lane, packed and with an odd
    leading dimension; scales inside and outside the range the quotients are estimated in."""
    rows, cols = shape
    step = np.float32(scale) if scale > 1e-38 else np.float32(2.0 ** -136)  # a denormal step
    x = (rng.integers(-127, 127, size=shape).astype(np.float32) + np.float32(0.5)) * step
    ulps = rng.integers(-2, 3, size=shape)
    for _ in range(2):
        x = np.where(ulps > 0, np.nextafter(x, np.float32(np.inf)), x)
        x = np.where(ulps < 0, np.nextafter(x, np.float32(-np.inf)), x)
        ulps -= np.sign(ulps)
    x[:, -1] = 127 * step  # the row's maximum is its last, ragged element
    x = x.astype(np.float32)
    qe, se = oracle.quantize_rows_i8(x)
    xw = np.full((rows, cols + 3), np.inf, dtype=np.float32)  # the padding is not read
    xw[:, :cols] = x
    q, s = handle.quantize_rows_i8(torch_gpu.from_numpy(x).cuda())
    np.testing.assert_array_equal(s.cpu().numpy(), se)
    np.testing.assert_array_equal(q.cpu().numpy(), qe)
    qw = torch_gpu.full((rows, cols + 5), 99, dtype=torch_gpu.int8, device="cuda")
    sw = torch_gpu.empty(rows, dtype=torch_gpu.float32, device="cuda")
    handle.quantize_rows_i8(torch_gpu.from_numpy(xw).cuda()[:, :cols], out=(qw[:, :cols], sw))
    got = qw.cpu().numpy()
    np.testing.assert_array_equal(sw.cpu().numpy(), se)
    np.testing.assert_array_equal(got[:, :cols], qe)
    assert (got[:, cols:] == 99).all()
