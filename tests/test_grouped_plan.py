"""Which kernel a grouped product runs on, by shape (moe_grouped_plan: host code, no GPU).

The figures behind each line are at the rules; here are the choices that a change of a rule must
not lose: what was measured slower on the other side."""
import ctypes

import pytest

from moe_prefetch import _lib, lib

Q4, Q6 = _lib.TYPE_Q4K, _lib.TYPE_Q6K


def plan(down, dt, T, K, E, I, host=0, shared=0):
    p = (ctypes.c_int32 * 3)()
    _lib.check(lib().moe_grouped_plan(down, dt, T, K, E, I, host, shared, p), "moe_grouped_plan")
    return tuple(p)


@pytest.mark.parametrize("T", [1, 16, 64, 200, 300, 512, 700, 1000])
@pytest.mark.parametrize("E,I", [(128, 768), (256, 512), (64, 256), (1, 768)])
def test_host_weights_take_large_chunks(E, I, T):
    """An expert in host memory is read over PCIe once per chunk, so with such weights a chunk is as
    large as a kernel has, at any number of pairs per expert and whether or not there is a slot pool
    (chunks of one tile: up to 12 % slower than passes of 32 pairs of the 64-row kernel)."""
    K = min(8, E)
    for shared in (0, 1):
        assert plan(0, Q4, T, K, E, I, 1, shared)[:2] == (128, 3)
        assert plan(1, Q4, T, K, E, I, 1, shared) == (128, 3, 4 if I == 256 or 16 < T * K <= 2 * E else 1)
        assert plan(1, Q6, T, K, E, I, 1, shared)[:2] == (128, 2)


@pytest.mark.parametrize("T,tiles", [(64, 1), (300, 1), (512, 1), (640, 3), (1000, 3), (4000, 3)])
def test_hbm_weights_take_large_chunks_from_40_pairs(T, tiles):
    """A cache whose experts are all in HBM is told apart from one that reads some over PCIe."""
    assert plan(0, Q4, T, 8, 128, 768)[:2] == (128, tiles)


def test_plan_refuses_bad_shapes():
    p = (ctypes.c_int32 * 3)()
    for bad in ((0, Q4, 0, 8, 128, 768), (0, Q4, 9000, 8, 128, 768), (0, Q4, 1, 8, 257, 768), (0, Q4, 1, 8, 128, 300),
                (1, 99, 1, 8, 128, 768)):
        assert lib().moe_grouped_plan(*bad, 0, 0, p) != 0
    assert lib().moe_grouped_plan(0, Q4, 1, 8, 128, 768, 0, 0, None) != 0
