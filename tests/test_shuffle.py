"""The training shuffle's steps against the sequential Fisher-Yates loop: every
position of the order, with the sorted buffer short enough that lists go on to
the insertion in place (a host build of the kernels' own functions)."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
M64 = (1 << 64) - 1


def fisher_yates(n, state):
    order = list(range(n))
    for i in range(n - 1, 0, -1):
        state = (state + 0x9E3779B97F4A7C15) & M64
        z = state
        z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & M64
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & M64
        j = (z ^ (z >> 31)) % (i + 1)
        order[i], order[j] = order[j], order[i]
    return order


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("no host compiler")
    so = str(tmp_path_factory.mktemp("shuffle") / "shuffle.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-Wall", "-o", so,
                    os.path.join(HERE, "host", "shuffle_driver.cpp")], check=True)
    lib = ctypes.CDLL(so)
    lib.shuffle_host.argtypes = [ctypes.c_uint64] + [ctypes.c_int] * 3 + [ctypes.c_void_p] * 2
    return lib


@pytest.mark.parametrize("links", [0, 1, 2])
@pytest.mark.parametrize("buffer", [1, 2, 5, 24])
@pytest.mark.parametrize("n,state", [(1, 3), (2, 4), (3, 5), (7, 6), (64, 7), (1000, 8), (20011, 9), (66000, 326 ^ 0x5DEECE66D)])
def test_every_position_is_the_sequential_loops(host, n, state, buffer, links):
    order, longest = np.full(n, -1, np.int32), ctypes.c_int()
    assert host.shuffle_host(state, n, buffer, links, order.ctypes.data, ctypes.byref(longest)) == 0
    assert order.tolist() == fisher_yates(n, state)
    if n == 66000:
        assert longest.value == 26  # longer than the kernels' buffer
