"""Launch shapes of the f32-faithful matrix-core GEMV (engine_amd/csrc/f32mma_shape.hpp), on the host:
the cases of tests/test_gpu_f32mma.py take the forms their names claim on 256 CUs, and the K split
of a weight does not depend on the member count (a member's bits are the same at any batch)."""
import os
import subprocess

import pytest

from .test_gpu_f32mma import PAIR_SHAPES

HERE = os.path.dirname(os.path.abspath(__file__))
PARTIAL_BYTES = 16 << 20  # kF32MmaPartialBytes


@pytest.fixture(scope="module")
def shape(tmp_path_factory):
    exe = tmp_path_factory.mktemp("shape") / "f32mma_shape_print"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(os.path.dirname(HERE), "engine_amd", "csrc"),
                    os.path.join(HERE, "cpp", "f32mma_shape_print.cpp"), "-o", str(exe)], check=True)

    def run(t, k, n, members, cus=256):
        out = subprocess.run([str(exe)] + [str(v) for v in (t, k, n, members, cus, PARTIAL_BYTES)], check=True,
                             capture_output=True, text=True).stdout
        return tuple(int(v) for v in out.split())

    return run


@pytest.mark.parametrize("t,k,n,members", list(PAIR_SHAPES))
def test_pair_shapes(shape, t, k, n, members):
    assert shape(t, k, n, members) == PAIR_SHAPES[(t, k, n, members)]


@pytest.mark.parametrize("t,k,n", [(12, 4096, 12288), (12, 512, 48), (13, 768, 272), (14, 512, 304)])
def test_split_is_the_weights_alone(shape, t, k, n):
    assert len({shape(t, k, n, m)[1] for m in (9, 16, 17, 33, 64)}) == 1
