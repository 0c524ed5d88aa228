"""The NF4 GEMM's choice of tile and K slices (grpo_nf4_gemm_tile; host only)."""

import ctypes

import pytest


def plan(m, n, k, r, bs=64, silu=0):
    """(rows, columns, K groups, slices) of the ring kernel, None where it does not run."""
    from grpo_mi355x import _lib

    v = [ctypes.c_int(0) for _ in range(4)]
    on = _lib.library().grpo_nf4_gemm_tile(m, n, k, r, bs, silu, *(ctypes.byref(x) for x in v))
    return tuple(x.value for x in v) if on else None


# workgroups of each tile that run together on a CU, without and with LoRA
TOGETHER = {(256, 256, 1): (1, 1), (128, 128, 1): (2, 2), (64, 128, 2): (1, 1),
            (64, 64, 2): (2, 1), (128, 128, 2): (1, 1)}


@pytest.mark.parametrize("n,k", [(256, 1536), (1536, 1536), (3584, 3584), (4608, 3584),
                                 (1536, 8960), (3584, 18944), (1024, 4096)])
@pytest.mark.parametrize("r", [0, 16])
def test_slices_do_not_start_a_round_of_few_workgroups(n, k, r):
    """Tiles are dealt to the 8 XCDs of 32 CUs, ceil(tiles / 8) per slice on the fullest: K
    is not cut so that the last of those workgroups run a round of their own, less than
    half full, where one slice fewer would have needed a round less."""
    cdiv = lambda a, b: -(-a // b)
    for m in range(65, 1025, 7):
        rows, cols, groups, s = plan(m, n, k, r)
        tiles = cdiv(cdiv(m, rows) * cdiv(n, cols), 8)
        room = 32 * TOGETHER[rows, cols, groups][r > 0]
        if s > 1:
            assert cdiv(tiles * s, room) == 1 or tiles * s % room == 0 or \
                2 * (tiles * s % room) >= room, (m, rows, cols, groups, s)


def test_shapes_of_other_kernels_have_no_tile():
    assert plan(128, 256, 1536, 17) is None   # rank beyond 16
    assert plan(128, 256, 1568, 16) is None   # K % 128 != 0
    assert plan(128, 256, 1536, 16, bs=32) is None
    assert plan(128, 256, 1536, 16, silu=1) is None
    assert plan(128, 256, 1536, 0, silu=1) is not None
