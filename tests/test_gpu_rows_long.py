"""Row kernels at the edges of their register-resident shapes: rows of 8 and
16 waves (up to 32768 columns), any 4-byte alignment, partial last vectors, and
special values beside them. Tolerances as in test_gpu_rows.py."""
import numpy as np
import pytest

from oxidizedmlx_amd import backend as hb
from oxidizedmlx_amd import synth
from oxidizedmlx_amd.opkind import OpKind
from parity import assert_allclose
from test_gpu_rows import oracle, run_rows

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("hip", "oracle_lib")]

EPS = 1e-5
SHAPES = [(5, 254), (3, 1021), (2, 4097), (2, 8190), (3, 8192), (2, 8195), (1, 16383), (2, 16384), (2, 16388),
          (2, 32003), (2, 32767), (1, 32768), (2, 32769)]


@pytest.mark.parametrize("rows,cols", SHAPES)
@pytest.mark.parametrize("offset", [0, 1, 3])
def test_long_and_misaligned_rows(rows, cols, offset):
    print(f"rows {rows}x{cols}+{offset}", flush=True)
    x = synth.normal(31 * rows + cols, (rows, cols), 0.5, 2.0)
    dy = synth.normal(37 * rows + cols, (rows, cols))
    what = f"{rows}x{cols}+{offset}"
    y = run_rows(hb.softmax_rows, x, offset=offset)
    assert_allclose(y, oracle(OpKind.Softmax(-1), x), 1e-6, 1e-5, f"softmax {what}")
    sm = oracle(OpKind.Softmax(-1), x)
    y = run_rows(lambda a, b, o, r, c: hb.softmax_vjp_rows(a, b, o, r, c), dy, sm, offset=offset)
    assert_allclose(y, oracle(OpKind.SoftmaxVjp(-1), dy, sm), 1e-5, 1e-4, f"softmax vjp {what}")
    for name, op, fn, vjp, vfn in (
            ("layernorm", OpKind.LayerNorm, hb.layernorm_rows, OpKind.LayerNormVjp, hb.layernorm_vjp_rows),
            ("rmsnorm", OpKind.RmsNorm, hb.rmsnorm_rows, OpKind.RmsNormVjp, hb.rmsnorm_vjp_rows)):
        y = run_rows(lambda a, o, r, c: fn(a, o, r, c, EPS), x, offset=offset)
        assert_allclose(y, oracle(op(EPS), x), 1e-6, 1e-5, f"{name} {what}")
        y = run_rows(lambda a, b, o, r, c: vfn(a, b, o, r, c, EPS), dy, x, offset=offset)
        assert_allclose(y, oracle(vjp(EPS), dy, x), 1e-5, 1e-4, f"{name} vjp {what}")


@pytest.mark.parametrize("cols", [7, 1022, 8194, 32003])
def test_special_values_beside_partial_vectors(cols):
    """Rows of -inf only, of the type's lowest value, with one +inf, one NaN,
    and with one finite value among -inf (in the partial last vector)."""
    x = synth.normal(cols, (6, cols), 0.0, 2.0)
    x[0] = -np.inf
    x[1] = np.finfo(np.float32).min
    x[2, cols // 2] = np.inf
    x[3, 0] = np.nan
    x[4] = -np.inf
    x[4, -1] = 1.0
    with np.errstate(invalid="ignore"):
        want = oracle(OpKind.Softmax(-1), x)
    y = run_rows(hb.softmax_rows, x)
    np.testing.assert_allclose(y, want, rtol=1e-5, atol=1e-7, equal_nan=True)


@pytest.mark.parametrize("cols,offset", [(4097, 0), (6000, 0), (6000, 1), (8190, 0), (8192, 0), (8195, 0), (12000, 0),
                                         (16383, 0), (16384, 3), (20001, 0), (32003, 0), (32768, 0)])
def test_softmax_of_long_rows_is_as_exact_as_expf(cols, offset):
    """Each value's relative error against float64. exp(x - m) has one unit in
    the last place of v_exp_f32 (2^-23) and, of the difference's rounding, at
    most half a last place of x (|x| < 16: 2^-21); the wave's factor as much
    again without the latter and a rounding, the product one: below 1e-6 in
    all, and 1e-7 in the root mean square (about 3.4e-8 per rounding of 2^-24,
    at most six of them). expf against the row's maximum, whose difference is
    rounded, has 2.1e-7 to 2.4e-7."""
    rows = (1 << 18) // cols
    x = synth.normal(cols + offset, (rows, cols), 0.0, 2.0)
    y = run_rows(hb.softmax_rows, x, offset=offset).astype(np.float64)
    z = np.exp(x.astype(np.float64) - x.max(1, keepdims=True))
    err = y / (z / z.sum(1, keepdims=True)) - 1
    rms, worst = np.sqrt(np.square(err).mean()), np.abs(err).max()
    print(f"softmax {rows}x{cols}+{offset}: rms {rms:.2e} max {worst:.2e}", flush=True)
    assert rms <= 1e-7 and worst <= 1e-6
