"""Products with K split over a workgroup's waves (kernels/gemm_wave.hip):
every tile shape, tile edges and K remainders in all four layouts, gaps
between rows and slices filled with NaN, operands at any alignment of their
elements, against float64 within the f32 summation bound."""
import numpy as np
import pytest

from oxidizedmlx_amd import abi, synth
from oxidizedmlx_amd import backend as hb
from oxidizedmlx_amd.tensor import Tensor
from parity import gemm_full_check

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("hip")]

CASES = [
    # (m, n, k, batch): 16 x 16 tiles first, then 16 x 32, 32 x 32, 32 x 64,
    # 64 x 64; the first of them (K <= 128) stay with the 4-wave kernel.
    (1, 1, 1, 1), (17, 33, 63, 1), (1, 1, 129, 1), (16, 16, 192, 1), (17, 33, 575, 1), (15, 250, 576, 1),
    (8, 64, 1025, 1), (33, 31, 217, 60), (256, 512, 512, 1),
    (300, 250, 129, 1), (5, 1000, 700, 7), (129, 1000, 197, 1), (128, 768, 768, 1),
    (640, 900, 31, 1), (65, 3071, 130, 1),
    (500, 700, 515, 1), (128, 3072, 66, 1),
    (800, 1000, 200, 1), (1000, 1023, 133, 1), (63, 65, 300, 70),
]


def embed(rows, offset, gap, slice_gap, fill=np.nan):
    """A flat array of `fill` with the batch's matrices in it: row pitch cols
    + gap, slices slice_gap apart, starting `offset` elements in."""
    b, r, c = rows.shape
    ld = c + gap
    stride = r * ld + slice_gap
    buf = np.full(offset + b * stride, fill, rows.dtype)
    for i in range(b):
        view = buf[offset + i * stride:offset + i * stride + r * ld].reshape(r, ld)
        view[:, :c] = rows[i]
    return buf, ld, stride


@pytest.mark.parametrize("m,n,k,batch", CASES)
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_tiles_remainders_and_gaps(m, n, k, batch, ta, tb):
    odd = (m + n + k) % 2
    a = synth.normal(m + k, (batch, m, k))
    b = synth.normal(n + k + 1, (batch, k, n))
    sa = np.ascontiguousarray(a.transpose(0, 2, 1)) if ta else a
    sb = np.ascontiguousarray(b.transpose(0, 2, 1)) if tb else b
    fa, lda, stra = embed(sa, 3 * odd, 5 * odd, 7 * odd)
    fb, ldb, strb = embed(sb, 1 * odd, 2 * odd, 3 * odd)
    da, db = hb.DeviceBuffer.from_array(fa), hb.DeviceBuffer.from_array(fb)
    ldc = n + 3
    c0 = np.full((batch, m, ldc), 7.0, np.float32)
    dc = hb.DeviceBuffer.from_array(c0)
    hb.gemm(abi.F32, abi.F32, bool(ta), bool(tb), m, n, k, da.ptr + 12 * odd, lda, db.ptr + 4 * odd, ldb, dc, ldc,
            batch=batch, stride_a=stra, stride_b=strb, stride_c=m * ldc)
    hb.synchronize()
    got = dc.download().reshape(batch, m, ldc)
    assert (got[:, :, n:] == 7.0).all()
    for i in {0, batch - 1}:
        gemm_full_check(got[i, :, :n], a[i], b[i], what=f"{m}x{n}x{k} slice {i} ta{ta} tb{tb}")


@pytest.mark.parametrize("rows,inputs,outputs", [(8, 768, 3072), (130, 200, 77), (512, 1024, 1024)])
def test_bias_in_the_store_is_the_separate_addition(rows, inputs, outputs):
    """A linear layer's bias added as C is stored, against the unfused graph."""
    res = []
    x, w, b = synth.normal(1, (rows, inputs)), synth.normal(2, (outputs, inputs)), synth.normal(3, (outputs,))
    for fusion in (True, False):
        st = hb.HipStream(fusion=fusion)
        t = [Tensor.from_f32(v, v.shape, st) for v in (x, w, b)]
        y = t[0].matmul(t[1].transpose())
        res.append(y.add(t[2].broadcast_to(y.shape)).to_numpy())
        st.close()
    # The unfused graph's product may be laid out differently (its transposed
    # weight is made), so the same sums may come in another order.
    exact = x.astype(np.float64) @ w.T.astype(np.float64) + b
    bound = (inputs + 1) * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w.T) + np.abs(b)) * 1.01
    for y in res:
        assert (np.abs(y - exact) <= bound).all()


CASES16 = [
    # 16 x 16, 16 x 32, 32 x 32, 32 x 64 and 64 x 64 tiles; rounds of 16-wide
    # ones for few rows; the last is past the rule.
    (1, 1, 1, 1), (17, 33, 63, 1), (15, 250, 1601, 1), (33, 31, 217, 50), (8, 4096, 1535, 1),
    (129, 500, 199, 1), (100, 1500, 65, 1), (5, 30001, 70, 1),
    (511, 512, 145, 1), (129, 257, 255, 4),
    (500, 1000, 777, 1), (1000, 1016, 528, 1), (900, 1000, 1023, 1),
]


@pytest.mark.parametrize("m,n,k,batch", CASES16)
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
def test_16_bit_tiles_remainders_and_gaps(m, n, k, batch, ta, tb, dtype):
    dt = abi.BF16 if dtype == "bf16" else abi.F16
    nan16 = 0x7FC0 if dt == abi.BF16 else 0x7E00
    bits = synth.bf16_bits if dt == abi.BF16 else synth.f16_bits
    wide = synth.bf16_to_f32 if dt == abi.BF16 else lambda x: x.view(np.float16).astype(np.float32)
    odd = (m + n + k) % 2
    a = bits(synth.normal(m + k, (batch, m, k)))
    b = bits(synth.normal(n + k + 1, (batch, k, n)))
    fa, lda, stra = embed(np.ascontiguousarray(a.transpose(0, 2, 1)) if ta else a, 3 * odd, 5 * odd, 6 * odd, nan16)
    fb, ldb, strb = embed(np.ascontiguousarray(b.transpose(0, 2, 1)) if tb else b, odd, 2 * odd, 3 * odd, nan16)
    da, db = hb.DeviceBuffer.from_array(fa), hb.DeviceBuffer.from_array(fb)
    exact = {i: (wide(a[i]), wide(b[i])) for i in {0, batch - 1}}
    for ct in (abi.F32, dt):
        ldc = n + 3
        c0 = np.full((batch, m, ldc), 7 if ct == dt else 7.0, np.uint16 if ct == dt else np.float32)
        dc = hb.DeviceBuffer.from_array(c0)
        hb.gemm(dt, ct, bool(ta), bool(tb), m, n, k, da.ptr + 6 * odd, lda, db.ptr + 2 * odd, ldb, dc, ldc,
                batch=batch, stride_a=stra, stride_b=strb, stride_c=m * ldc)
        hb.synchronize()
        got = dc.download(c0.dtype).reshape(batch, m, ldc)
        assert (got[:, :, n:] == 7).all()
        for i, (x, y) in exact.items():
            c = got[i, :, :n] if ct == abi.F32 else wide(np.ascontiguousarray(got[i, :, :n]))
            gemm_full_check(c, x, y, out="f32" if ct == abi.F32 else dtype, what=f"{m}x{n}x{k} {dtype} slice {i}")
