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


# (down, type, tokens, K, experts, I) -> (rows, tiles, row tiles); the comment: what the other side costs
FEW_WORKGROUPS = [
    ((0, Q4, 16, 1, 1, 768), (64, 1, 1)),           # 15.8 us for 9.7 on tiles: a shared expert in launches of its own
    ((0, Q4, 32, 1, 1, 768), (64, 2, 1)),           # 15.9 for 12.1
    ((0, Q4, 33, 1, 1, 768), (128, 1, 1)),          # 21.3 for 15.6 in passes of 16
    ((0, Q4, 64, 2, 8, 768), (64, 2, 1)),           # 16.2 for 12.0
    ((0, Q4, 64, 8, 64, 512), (64, 1, 1)),          # 22.4 for 20.4: exactly 512 workgroups
    ((0, Q4, 96, 8, 128, 256), (64, 1, 1)),         # 22.4 for 20.4
    ((0, Q4, 128, 8, 128, 256), (128, 1, 1)),       # 23.4 for 22.4: with so many experts some have over 16 pairs
    ((1, Q4, 16, 8, 32, 768), (64, 1, 1)),          # 11.8 for 9.6
    ((1, Q6, 8, 1, 1, 768), (64, 1, 1)),            # 17.3 for 8.4 (two row tiles a workgroup: 8 workgroups)
    ((1, Q6, 24, 1, 1, 768), (64, 2, 1)),           # 17.4 for 10.0
    ((1, Q6, 64, 1, 1, 768), (128, 1, 1)),          # 23.4 for 11.2 in chunks of two tiles
    ((1, Q6, 512, 1, 1, 768), (128, 1, 1)),         # 25.1 for 12.9
    ((1, Q6, 32, 2, 8, 512), (64, 1, 1)),           # 15.2 for 7.2
    ((1, Q6, 128, 2, 16, 512), (64, 2, 1)),         # 16.1 for 11.2
    ((1, Q6, 192, 2, 8, 768), (128, 1, 1)),         # 24.4 for 12.5
    ((1, Q6, 16, 8, 256, 512), (64, 1, 1)),         # 35.6 for 31.8
    ((1, Q6, 64, 8, 64, 512), (64, 1, 1)),          # 24.7 for 22.9
]


@pytest.mark.parametrize("shape,want", FEW_WORKGROUPS)
def test_few_workgroups(shape, want):
    """Shapes that leave most of the chip idle on tiles of 128 rows take the 64-row kernels, and one
    row tile a workgroup."""
    assert plan(*shape) == want


@pytest.mark.parametrize("shape", [s for s, w in FEW_WORKGROUPS if w[0] == 64])
def test_shared_expert_beside_runs_on_tiles(shape):
    """The 64-row kernels know no shared expert beside the routed ones."""
    assert plan(*shape, 0, 1)[0] == 128


def test_plan_refuses_bad_shapes():
    p = (ctypes.c_int32 * 3)()
    for bad in ((0, Q4, 0, 8, 128, 768), (0, Q4, 9000, 8, 128, 768), (0, Q4, 1, 8, 257, 768), (0, Q4, 1, 8, 128, 300),
                (1, 99, 1, 8, 128, 768)):
        assert lib().moe_grouped_plan(*bad, 0, 0, p) != 0
    assert lib().moe_grouped_plan(0, Q4, 1, 8, 128, 768, 0, 0, None) != 0
