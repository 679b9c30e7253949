"""Large results into pageable memory (csrc/host_copy.cpp): sizes around the
line (128 KiB) and the chunks (2 MiB of the destination), destinations at any
alignment, several streams at once from several threads; through the pinned
slots, which a stream that stays open has earned (csrc/host_slots.hpp,
test_host_slots.py), and the runtime's way."""
import os
import subprocess
import sys
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


@pytest.fixture(scope="module")
def owner():
    """A stream that has copied 576 MiB: every slot is earned while it lives."""
    st = HipStream()
    x, node = negated(st, 64 * MIB, 1)
    for _ in range(9):
        np.testing.assert_array_equal(st.get_buffer(node), -x)
    yield st
    st.close()


@pytest.mark.parametrize("n", [(1 << 15) - 1, 1 << 15, 2 * MIB, 2 * MIB + 1, 4 * MIB - 1, 4 * MIB, 21 * MIB - 7])
@pytest.mark.parametrize("offset", [0, 1, 100003])
def test_sizes_and_alignments(owner, n, offset):
    st = HipStream()
    x, node = negated(st, n, n + offset)
    out = np.full(offset + n + 1, 7.0, np.float32)
    abi.check(st._L.mlxhip_stream_get_buffer(st._s, node, out.ctypes.data + 4 * offset, n), st._L)
    np.testing.assert_array_equal(out[offset:offset + n], -x)
    assert (out[:offset] == 7.0).all() and out[-1] == 7.0
    st.close()


def test_threads_with_streams_of_their_own(owner):
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


def test_a_first_fetch_goes_the_runtimes_way():
    """In a process of its own: the first copies have no slots yet."""
    code = """
import numpy as np
from oxidizedmlx_amd.backend import HipStream
from oxidizedmlx_amd.opkind import OpKind, meta
for n in (1 << 15, (1 << 19) + 3, 5 << 18):
    st = HipStream()
    x = np.arange(n, dtype=np.float32)
    node = st.add_op(OpKind.Neg, [st.add_constant(x, meta([n]))], meta([n]))
    st.eval(node)
    assert np.array_equal(st.get_buffer(node), -x)
    st.close()
print("ok")
"""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", code], cwd=root, capture_output=True, text=True, timeout=100)
    assert r.stdout.strip() == "ok", r.stdout + r.stderr
