"""Large results into pageable memory (csrc/host_copy.cpp): sizes around the
line (128 KiB) and the chunks (2 MiB of the destination), destinations at any
alignment, several streams at once from several threads."""
import threading

import numpy as np
import pytest

from oxidizedmlx_amd import abi
from oxidizedmlx_amd.backend import HipStream
from oxidizedmlx_amd.opkind import OpKind, meta

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("hip")]

MIB = 1 << 18  # floats


def negated(st, n, seed):
    x = np.random.default_rng(seed).standard_normal(n, dtype=np.float32)
    node = st.add_op(OpKind.Neg, [st.add_constant(x, meta([n]))], meta([n]))
    st.eval(node)
    return x, node


@pytest.mark.parametrize("n", [(1 << 15) - 1, 1 << 15, 2 * MIB, 2 * MIB + 1, 4 * MIB - 1, 4 * MIB, 21 * MIB - 7])
@pytest.mark.parametrize("offset", [0, 1, 100003])
def test_sizes_and_alignments(n, offset):
    st = HipStream()
    x, node = negated(st, n, n + offset)
    out = np.full(offset + n + 1, 7.0, np.float32)
    abi.check(st._L.mlxhip_stream_get_buffer(st._s, node, out.ctypes.data + 4 * offset, n), st._L)
    np.testing.assert_array_equal(out[offset:offset + n], -x)
    assert (out[:offset] == 7.0).all() and out[-1] == 7.0
    st.close()


def test_threads_with_streams_of_their_own():
    bad = []

    def work(seed):
        st = HipStream(async_eval=seed % 2 == 0)
        for k in range(3):
            x, node = negated(st, 9 * MIB + seed, 10 * seed + k)
            if not np.array_equal(st.get_buffer(node), -x):
                bad.append((seed, k))
        st.close()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
