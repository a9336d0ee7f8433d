"""Scratch sizes of 3D calls, on the CPU.  The no-allocation entry point holds a
fixed array, so a 3D call that grows its scratch refuses volumes that it took:
each size is bounded by its two parts, the transposed image and distances
(derived here) and the descriptors and exchange buffer (recorded sizes)."""
import ctypes
import pathlib

import pytest

import fastgeodis_amd as FG

LIB = ctypes.CDLL(str(pathlib.Path(FG.native_library_paths()[0])))
LIB.fg_workspace_bytes.restype = ctypes.c_size_t

# (op, C, D, H, W, requested halo): bytes beyond the voxel buffers
RECORDED = {
    (0, 1, 320, 322, 324, 0): 1746944,
    (0, 1, 16, 16, 16, 0): 40448,
    (1, 2, 97, 211, 163, 0): 1200524,
    (2, 3, 40, 64, 50, 0): 288768,
    (0, 3, 2500, 1, 400, 7): 16275200,
    (0, 1, 1, 700, 4000, 3): 45655552,
    (1, 4, 3000, 1, 5000, 30): 205824,
}


@pytest.mark.parametrize("case", sorted(RECORDED), ids=str)
def test_3d_scratch_does_not_grow(case):
    op, C, D, H, W, halo = case
    old = FG.get_tuning()
    FG.set_tuning(halo=halo)
    try:
        got = LIB.fg_workspace_bytes(op, C, D, H, W)
    finally:
        FG.set_tuning(**old)
    dists = {0: 1, 1: 2, 2: 4}[op]
    voxel_buffers = 4 * D * H * W * (C + 2 * dists - 1)
    assert got - voxel_buffers <= RECORDED[case]
