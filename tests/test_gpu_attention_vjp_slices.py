"""Gradient of fused attention for few heads (kernels/attention_bwd.hip): the
blocks of each sum sliced over workgroups, on both sides of the rule, with even
and uneven slices, against float64. The bound is the unsliced kernels' own
error on the same head (repeated until they run), which is held against the
oracle elsewhere: the slices only regroup its sums, into shorter ones."""
import math

import numpy as np
import pytest

from oxidizedmlx_amd import backend as hb
from oxidizedmlx_amd import synth
from oxidizedmlx_amd.tensor import Tensor, value_and_grad
from test_gpu_attention_vjp import f64_vjp, gpu_grads

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("hip")]


@pytest.mark.parametrize("heads,t,copies,causal", [
    (1, 192, 1, True),       # 3 blocks: unsliced
    (1, 256, 80, True),      # 4 slices of 1; 80 heads: unsliced
    (1, 256, 24, False),
    (7, 448, 40, True),      # 7 slices of 1
    (14, 512, 48, False),    # 896 pairs of blocks: 4 slices of 2
    (10, 1024, 72, True),    # 1360 pairs: 6 slices of 3, the last of 1
])
def test_slices_match_float64_as_the_whole_does(heads, t, copies, causal):
    q, k, v, do = (synth.normal(500 + t + i, (heads, t, 64)) for i in range(4))
    scale = 1.0 / math.sqrt(64)
    got = gpu_grads(q, k, v, do, scale, causal)
    whole = gpu_grads(*(np.repeat(x[:1], copies, axis=0) for x in (q, k, v, do)), scale, causal)
    for name, g, w, e in zip("qkv", got, whole, f64_vjp(q, k, v, do, scale, causal)):
        err, ref = float(np.abs(g - e).max()), float(np.abs(w[0] - e[0]).max())
        print(f"  d{name}: sliced {err:.3e}, whole {ref:.3e}", flush=True)
        assert (w == w[:1]).all()
        assert err <= 1.5 * ref + 2.0 ** -22 * float(np.abs(e).max())


def test_head_layouts_agree_sliced():
    """Heads side by side in rows and head-major: the same sums, bit for bit."""
    b, t, heads = 1, 320, 2
    q, k, v, g = (synth.normal(70 + i, (b, t, heads * 64)) for i in range(4))

    def major(a):
        return np.ascontiguousarray(a.reshape(b, t, heads, 64).transpose(0, 2, 1, 3).reshape(b * heads, t, 64))

    def run(arrs, heads_arg):
        st = hb.HipStream()
        tq, tk, tv, tg = (Tensor.from_f32_on_stream(a.reshape(-1), a.shape, st) for a in arrs)
        loss = tq.head_attention(tk, tv, 0.125, True, heads=heads_arg).mul(tg).sum_all()
        return [x.to_numpy().reshape(arrs[0].shape) for x in value_and_grad(loss, [tq, tk, tv])[1]]

    for a, e in zip(run((q, k, v, g), heads), run(tuple(major(a) for a in (q, k, v, g)), None)):
        np.testing.assert_array_equal(major(a), e)


def test_sliced_gradient_replays_from_a_graph():
    """Recorded on a stream whose workspace it is the first to need, and
    replayed between eager calls that use the same workspace."""
    h, t = 2, 512
    arrs = [synth.normal(40 + i, (h, t, 64)) for i in range(4)]
    want = gpu_grads(*arrs, 0.125, True)
    q, k, v, do = (hb.DeviceBuffer.from_array(a) for a in arrs)
    o, dq, dk, dv, *other = (hb.DeviceBuffer(arrs[0].nbytes) for _ in range(7))
    s = hb.create_stream()
    try:
        with hb.Graph(s) as g:
            hb.attention(q, k, v, o, h, t, t, 64, 0.125, True, stream=s)
            hb.attention_vjp(q, k, v, o, do, dq, dk, dv, h, t, 64, 0.125, True, stream=s)
        for _ in range(3):
            for x in (dq, dk, dv):
                x.upload(np.zeros_like(arrs[0]))
            g.launch()
            hb.synchronize(s)
            for x, w in zip((dq, dk, dv), want):
                np.testing.assert_array_equal(x.download(np.float32, w.size).reshape(w.shape), w)
            hb.attention_vjp(k, q, v, o, do, *other, h, t, 64, 0.125, True, stream=s)
            hb.synchronize(s)
        g.close()
    finally:
        hb.destroy_stream(s)
