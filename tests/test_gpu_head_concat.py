"""Multi-head attention written head by head (Narrow, Reshape, Attention per
head, Concatenate) runs as one launch on the projections; graphs that differ
from that form run node by node. Either way the values are the unfused
graph's (to the attention kernels' rounding, test_gpu_attention.py) and so is
eval_count."""
import math

import numpy as np
import pytest

from oxidizedmlx_amd import synth
from oxidizedmlx_amd.backend import HipStream
from oxidizedmlx_amd.tensor import Tensor, eval_all
from parity import assert_allclose

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("hip")]


def heads_graph(st, seq, heads, dh, variant, tk=None):
    """The per-head graph's outputs over three source tensors, each the result
    of an op."""
    tk = tk or seq
    d = heads * dh
    src = [Tensor.from_f32(synth.normal(40 + j, (t, d)), (t, d), st).neg() for j, t in enumerate((seq, tk, tk))]
    split = [x.reshape((t, heads, dh)).transpose((1, 0, 2)) for x, t in zip(src, (seq, tk, tk))]
    outs, extra = [], []
    order = range(heads)
    if variant == "order":
        order = [1, 0, *range(2, heads)]
    for i in order:
        q, k, v = (x.narrow(0, i, 1).reshape((t, dh)) for x, t in zip(split, (seq, tk, tk)))
        scale = 1.0 / math.sqrt(dh) * (2.0 if variant == "scale" and i == 1 else 1.0)
        o = q.attention(k, v, scale, not (variant == "mask" and i == 0))
        if variant == "head_asked" and i == 0:
            extra.append(o)
        if variant == "head_read" and i == 0:
            extra.append(o.neg())
        if variant == "split_read" and i == 0:
            extra.append(split[1].neg())
        outs.append(o)
    return [Tensor.cat(outs, -1 if variant == "axis" else 1)] + extra


VARIANTS = ["plain", "axis", "order", "scale", "mask", "head_asked", "head_read", "split_read"]


@pytest.mark.parametrize("variant", VARIANTS)
@pytest.mark.parametrize("seq,heads,dh,tk", [(37, 4, 32, None), (130, 3, 64, 77), (16, 2, 24, None), (520, 40, 16, None)])
def test_values_and_counts(seq, heads, dh, tk, variant):
    res = {}
    for fusion in (False, True):
        st = HipStream(fusion=fusion)
        outs = heads_graph(st, seq, heads, dh, variant, tk)
        eval_all(outs)
        launches = st.launch_count()
        res[fusion] = ([o.to_numpy() for o in outs], launches, st.eval_count())
        # A head asked for afterwards is computed then.
        late = outs[0].narrow(1, 0, dh).to_numpy()
        np.testing.assert_array_equal(late, res[fusion][0][0][:, :dh])
        st.close()
    for a, b in zip(res[True][0], res[False][0]):
        assert_allclose(a, b, 2e-6 * float(np.abs(b).max()) * 4, 1e-5, f"{variant} {seq}x{heads}x{dh}")
    assert res[True][2] == res[False][2]
    folds = variant in ("plain", "axis") and dh in (16, 32, 64, 128)
    assert (res[True][1] == 4) == folds  # three sources and the attention
