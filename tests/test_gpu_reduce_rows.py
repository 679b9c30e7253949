"""Sum / Mean / Max along contiguous rows (reduce_rows_kernel) against the
oracle: the same sequential fold, so the same bits, at the edges of its
chunks (4096 elements over 4 or 16 rows) and of its row groups."""
import numpy as np
import pytest

from oracle.cpu_ref import CpuRefBackend
from oxidizedmlx_amd import backend as hb
from oxidizedmlx_amd.opkind import NodeInput, OpKind, meta

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("hip", "oracle_lib")]

SHAPES = [(1, 64), (5, 65), (4, 1023), (3, 1024), (6, 1025), (2, 3072), (7, 6148), (1, 7169),
          (4095, 64), (4096, 255), (4097, 256), (4100, 513), (4099, 1540)]


@pytest.mark.parametrize("rows,cols", SHAPES)
@pytest.mark.parametrize("kind", ["sum", "mean", "max"])
@pytest.mark.parametrize("offset", [0, 1])
def test_rows_fold_in_order(rows, cols, kind, offset):
    """offset 1: rows that start 4 bytes past a 16-byte boundary."""
    op = {"sum": OpKind.Sum, "mean": OpKind.Mean, "max": OpKind.Max}[kind](-1)
    x = np.random.default_rng(rows + cols).standard_normal((rows, cols), dtype=np.float32) * 3 + 1
    x[0, :] = -0.0
    if rows > 1:
        x[1, cols // 2] = -np.inf
    want = CpuRefBackend().eval_node(op, [NodeInput(x.reshape(-1), x.shape)], meta([rows]))
    d = hb.DeviceBuffer(x.nbytes + 16)
    d.upload(x, offset=4 * offset)
    y = hb.DeviceBuffer(4 * rows)
    hb.eval_node_dev(op, [(d.ptr + 4 * offset, x.shape)], meta([rows]), y)
    hb.synchronize()
    np.testing.assert_array_equal(y.download().view(np.uint32), np.asarray(want, np.float32).view(np.uint32))


@pytest.mark.parametrize("n", [1, 2, 63, 1025, 65535, 65536])
@pytest.mark.parametrize("kind", ["sum", "mean", "max"])
def test_whole_tensor_folds_in_order(n, kind):
    op = {"sum": OpKind.Sum, "mean": OpKind.Mean, "max": OpKind.Max}[kind](None)
    x = np.random.default_rng(n).standard_normal(n, dtype=np.float32)
    want = CpuRefBackend().eval_node(op, [NodeInput(x, x.shape)], meta([]))
    got = hb.HipBackend().eval_node(op, [NodeInput(x, x.shape)], meta([]))
    np.testing.assert_array_equal(got.view(np.uint32), np.asarray(want, np.float32).view(np.uint32))


@pytest.mark.parametrize("shape", [(2, 3), (1, 7), (1, 8), (1, 15), (1, 17), (2, 63), (1, 65), (1, 127), (1, 129), (3, 255), (1, 511),
                                   (1, 512), (2, 513), (1, 1023), (1, 1025), (3, 1537)])
@pytest.mark.parametrize("inner", [2, 15, 17, 63, 64, 65])
@pytest.mark.parametrize("kind", ["sum", "mean", "max"])
def test_columns_fold_in_order(shape, inner, kind):
    """The middle axis at the edges of the register batches (16, 64, 128) and
    of the LDS chunks (256 rows, 16 columns), rows at every alignment."""
    op = {"sum": OpKind.Sum, "mean": OpKind.Mean, "max": OpKind.Max}[kind](1)
    outer, dim = shape
    x = np.random.default_rng(dim + inner).standard_normal((outer, dim, inner), dtype=np.float32) * 3 + 1
    x[0, :, 0] = -0.0
    x[0, dim - 1, 1] = -np.inf
    want = CpuRefBackend().eval_node(op, [NodeInput(x.reshape(-1), x.shape)], meta([outer, inner]))
    d = hb.DeviceBuffer(x.nbytes + 16)
    d.upload(x, offset=4)
    y = hb.DeviceBuffer(4 * outer * inner)
    hb.eval_node_dev(op, [(d.ptr + 4, x.shape)], meta([outer, inner]), y)
    hb.synchronize()
    np.testing.assert_array_equal(y.download().view(np.uint32), np.asarray(want, np.float32).reshape(-1).view(np.uint32))
