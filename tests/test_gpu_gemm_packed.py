"""Unaligned 16-bit products of many tiles (C of 16 bits), which run on
zero-padded copies of both operands, against float64, around the line where
they start (128 tiles of 128 x 128) and at the copies' remainders."""
import numpy as np
import pytest

from oxidizedmlx_amd import abi, synth
from oxidizedmlx_amd import backend as hb
from parity import gemm_full_check
from test_gpu_gemm_wave import embed

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("hip")]

# 121 and 144 tiles; K of one partial chunk, a chunk and one more; few wide
# tiles; slices; 127 and 128 tiles of one row.
CASES = [
    (1401, 1407, 65, 1), (1409, 1411, 1, 1), (1409, 1501, 7, 1), (1500, 1409, 9, 1), (1473, 1473, 331, 1),
    (2050, 1015, 130, 1), (500, 505, 203, 9), (121, 16250, 33, 1), (121, 16377, 33, 1),
]


@pytest.mark.parametrize("m,n,k,batch", CASES)
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("dtype,shift", [("bf16", 1), ("bf16", 0), ("f16", 1)])
def test_many_tiles_unaligned(m, n, k, batch, ta, tb, dtype, shift):
    """shift 1: slices, rows and starts at odd elements, NaN between them."""
    dt = abi.BF16 if dtype == "bf16" else abi.F16
    nan16 = 0x7FC0 if dt == abi.BF16 else 0x7E00
    bits = synth.bf16_bits if dt == abi.BF16 else synth.f16_bits
    wide = synth.bf16_to_f32 if dt == abi.BF16 else lambda x: x.view(np.float16).astype(np.float32)
    x, y = synth.normal(m + k, (batch, m, k)), synth.normal(n + k + 1, (batch, k, n))
    if dtype == "f16":
        # Magnitudes from 2^-7 on: a product below 2^-14, f16's smallest normal
        # number, would round with up to 2^-25 whatever its size, which the
        # relative bound of the check does not allow for.
        x, y = (np.copysign(np.maximum(np.abs(v), 2.0 ** -7), v) for v in (x, y))
    a, b = bits(x), bits(y)
    pad_a = 1 - (m if ta else k) % 2 if shift else 0
    fa, lda, stra = embed(np.ascontiguousarray(a.transpose(0, 2, 1)) if ta else a, shift, pad_a, 3 * shift, nan16)
    fb, ldb, strb = embed(np.ascontiguousarray(b.transpose(0, 2, 1)) if tb else b, 3 * shift, 2 * shift, shift, nan16)
    da, db = hb.DeviceBuffer.from_array(fa), hb.DeviceBuffer.from_array(fb)
    ldc = n + 3
    dc = hb.DeviceBuffer.from_array(np.full((batch, m, ldc), 7, np.uint16))
    hb.gemm(dt, dt, bool(ta), bool(tb), m, n, k, da.ptr + 2 * shift, lda, db.ptr + 6 * shift, ldb, dc, ldc,
            batch=batch, stride_a=stra, stride_b=strb, stride_c=m * ldc)
    hb.synchronize()
    got = dc.download(np.uint16).reshape(batch, m, ldc)
    assert (got[:, :, n:] == 7).all()
    for i in {0, batch - 1}:
        gemm_full_check(wide(np.ascontiguousarray(got[i, :, :n])), wide(a[i]), wide(b[i]), out=dtype,
                        what=f"{m}x{n}x{k} {dtype} slice {i}")


def test_f32_result_of_packed_operands_keeps_its_k_splits():
    """Slices too long for the kernels that read unaligned 16-bit rows (4 GiB:
    1409 rows, 1.53 million elements apart) are packed with an f32 C too. 144
    tiles: K is split as it is for the same product of aligned operands, and
    the bits are that product's (its K padded with zeros)."""
    m, n, k, kp = 1409, 1408, 1023, 1024
    lda = (1 << 31) // (m - 1) + 2
    lda += 1 - lda % 2
    a, b = synth.bf16_bits(synth.normal(5, (m, k))), synth.bf16_bits(synth.normal(6, (k, n)))
    da = hb.DeviceBuffer(((m - 1) * lda + k) * 2)
    for i in range(m):
        da.upload(a[i], offset=2 * i * lda)
    db = hb.DeviceBuffer.from_array(b)
    dc = hb.DeviceBuffer(m * n * 4)
    hb.gemm(abi.BF16, abi.F32, False, False, m, n, k, da, lda, db, n, dc, n)
    hb.synchronize()
    got = dc.download(np.float32, m * n).reshape(m, n)
    da.free()
    ap, bp = np.zeros((m, kp), np.uint16), np.zeros((kp, n), np.uint16)
    ap[:, :k], bp[:k] = a, b
    da, db = hb.DeviceBuffer.from_array(ap), hb.DeviceBuffer.from_array(bp)
    hb.gemm(abi.BF16, abi.F32, False, False, m, n, kp, da, kp, db, n, dc, n)
    hb.synchronize()
    np.testing.assert_array_equal(got.view(np.uint32), dc.download(np.uint32, m * n).reshape(m, n))
    gemm_full_check(got, synth.bf16_to_f32(a), synth.bf16_to_f32(b), what="packed, f32 C")
