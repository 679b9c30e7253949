"""The launches of a row operation (csrc/kernels/row_launch.hpp, plain C++,
compiled here with g++): together they cover every row once, none counts more
work-items than a dispatch can (2^32 - 1), and a causal mask is indexed right
in each. The row counts are those of buffers up to 288 GB."""
import subprocess

import pytest

from oxidizedmlx_amd import build

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "row_launch.hpp"
int main(int argc, char** argv) {
    const int64_t rows = atoll(argv[1]), cols = atoll(argv[2]);
    mlxhip::for_row_chunks(rows, cols, atoi(argv[3]), [&](int64_t r0, int64_t n, int causal) {
        std::printf("%lld %lld %d %d\n", (long long)r0, (long long)n, causal, mlxhip::row_threads(cols));
        return 0;
    });
}
"""


@pytest.fixture(scope="module")
def chunks(tmp_path_factory):
    d = tmp_path_factory.mktemp("row_launch")
    (d / "p.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", f"{build.CSRC}/kernels", "-o", str(d / "p"), str(d / "p.cpp")], check=True)

    def run(rows, cols, causal):
        out = subprocess.run([str(d / "p"), str(rows), str(cols), str(causal)], check=True, capture_output=True, text=True)
        return [tuple(map(int, line.split())) for line in out.stdout.splitlines()]

    return run


# Row counts around the launches' limits at every kernel's widths: 4194304 rows
# of more than 8192 columns (137 GB) are the case of one work-item too many.
SIZES = [(1, 1), ((1 << 22) + 1, 64), (1 << 24, 4096), ((1 << 22) + 3, 4097), (1 << 23, 8192), (1 << 22, 8193),
         ((1 << 20) - 1, 16385), ((1 << 20) + 1, 32768), (1 << 21, 32769), (7, 1 << 30)]


@pytest.mark.parametrize("rows,cols", SIZES)
@pytest.mark.parametrize("causal", [0, 1])
def test_every_row_once_within_a_dispatch(chunks, rows, cols, causal):
    got = chunks(rows, cols, causal)
    at = 0
    for r0, n, mask, threads in got:
        assert r0 == at and n > 0
        assert n * threads < 1 << 32
        # The kernel masks by its own row number: right at row 0, and without
        # a mask where a row sees every column.
        assert mask == causal if r0 == 0 else (mask == 0 and (not causal or r0 >= cols))
        at += n
    assert at == rows
    # The waves that a row takes (dispatch_rows).
    assert got[0][3] >= (256 if cols <= 4096 else 512 if cols <= 8192 else 1024 if cols <= 32768 else 256)
