"""Which grids have room for a split in the workspace (CPU: the size functions
carry the plans): short grids are split, grids that a split was measured to
slow down are not."""

import pytest

from avgen_amd import _lib


@pytest.fixture(scope="module")
def lib():
    return _lib.load()


@pytest.mark.parametrize("fp8", [0, 1])
@pytest.mark.parametrize("H,Lq,Lk,D,split", [
    (4, 4096, 4096, 128, True),      # 64 blocks of 256 rows
    (16, 2048, 20000, 128, True),    # 128: half the CUs
    (17, 2048, 10752, 128, False),   # 136 .. 256: one round on most of the CUs
    (20, 1792, 10752, 128, False),
    (17, 2048, 20000, 128, False),
    (24, 2013, 20000, 128, False),
    (32, 2048, 20000, 128, False),
    (33, 2048, 20000, 128, True),    # a second round of 8 blocks
    (4, 4096, 4096, 64, True),
])
def test_forward(lib, H, Lq, Lk, D, split, fp8):
    base = (lib.avattn_fwd_fp8_workspace_size if fp8 else lib.avattn_fwd_workspace_size)(1, H, Lk, D)
    assert (lib.avattn_fwd_split_workspace_size(1, H, H, Lq, Lk, D, fp8) > base) == split


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,H,Lq,Lk,split", [
    (1, 16, 20000, 256, True),    # 32 key blocks
    (2, 20, 20000, 256, True),    # 80
    (1, 5, 12000, 6400, False),   # 250: nearly every CU
    (1, 5, 12000, 6656, False),   # 260: more than one round
    (2, 40, 75600, 512, False),
])
def test_backward(lib, B, H, Lq, Lk, D, split):
    staged = lib.avattn_bwd_staged_workspace_size(B, H, H, Lq, Lk, D, B * H)
    assert (lib.avattn_bwd_split_workspace_size(B, H, H, Lq, Lk, D) > staged) == split
