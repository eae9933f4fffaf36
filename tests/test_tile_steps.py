"""Which K steps of a tile GEMM plain 16-byte loads read (csrc/tile_steps.hpp,
compiled for the host): every one of them inside the matrix, at most two left
to the guarded loads, none at all for K = 0."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "onnx-light_amd", "csrc")


@pytest.fixture(scope="module")
def plain_steps(tmp_path_factory):
    d = tmp_path_factory.mktemp("tile_steps")
    (d / "s.cpp").write_text('#include "tile_steps.hpp"\nextern "C" int plain_steps(int64_t K, int step, int rows, '
                             "int64_t pitch) { return onnxl_amd::tg::PlainSteps(K, step, rows != 0, pitch); }\n")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", CSRC, str(d / "s.cpp"), "-o",
                    str(d / "s.so")], check=True)
    f = ctypes.CDLL(str(d / "s.so")).plain_steps
    f.argtypes = [ctypes.c_int64, ctypes.c_int, ctypes.c_int, ctypes.c_int64]
    return f


@pytest.mark.parametrize("step", [64, 128])
@pytest.mark.parametrize("rows", [True, False])
def test_plain_steps_stay_inside(plain_steps, step, rows):
    for K in list(range(0, 4 * step + 3)) + [1001, 4096, 4097]:
        total = -(-K // step)
        for pitch in list(range(1, 50)) + [64, 100, 127, 128, 1001, 4096]:
            n = plain_steps(K, step, int(rows), pitch)
            assert max(0, total - 2) <= n <= total, (K, pitch, n)
            assert n * step <= K, (K, pitch, n)  # a row of A, or of a transposed B, ends there or later
            if rows and n > 0:  # the last piece of the last row that a plain step reads
                starts = np.arange(0, pitch, 16)
                assert (n * step - 1) * pitch + int(starts[-1]) + 16 <= K * pitch, (K, pitch, n)
            if K % step == 0 and (not rows or pitch % 16 == 0):
                assert n == total, (K, pitch, n)
