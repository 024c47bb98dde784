"""Lengths with a compile-time kernel in small grids: which kernel the planner
takes on either side of its size rule, and both against the oracle (3D round
trips of R2C and C2C types, in two memory orders).

Tolerance: 8 u log2(points of the grid) relative L2, as each axis adds a few u
per radix pass.
"""
import math

import numpy as np
import pytest

import cases as C
import emu_binding as emu
import oracle_binding as orc

# dims, axes that take the single-buffer kernel (in FP32 and FP64)
GRIDS = [
    ([48, 48, 60], (0, 1, 2)),    # no power of two, above 256 KiB
    ([96, 40, 72], (0, 1, 2)),
    ([96, 3, 5], ()),             # below: the compile-time kernel
    ([128, 128, 24], (2,)),       # powers of two above 64 points keep theirs
]


@pytest.mark.parametrize("prec", [8, 4])
@pytest.mark.parametrize("mo2", [[0, 1, 2], [1, 2, 0]])
@pytest.mark.parametrize("dims,mid", GRIDS)
def test_small_grids(dims, mid, mo2, prec):
    types = [C.R2C_D, C.CF_D, C.CF_D]
    mo1 = [0, 1, 2]
    x = C.random_input(types, dims, mo1, 7)
    x = x if prec == 8 else x.astype(np.float32)
    od = C.out_dims(types, dims)
    tol = 8 * 2.0 ** (-53 if prec == 8 else -24) * math.log2(np.prod(dims))
    ref = orc.exec3d(types, dims, mo1, mo2, x.astype(np.float64))
    got, desc = emu.exec3d([t - (prec == 4) for t in types], dims, mo1, od, mo2, x, prec)
    assert C.rel_l2(got, ref) < tol, desc
    for stage in desc.split(" | "):
        for axis in range(3):
            if f"[axis {axis}, N=" in stage and dims[axis] in (48, 60, 72, 96, 40, 24):
                assert (", mid" in stage) == (axis in mid), stage
    emu.lib().emu_set_fast(0)
    try:
        other, _ = emu.exec3d([t - (prec == 4) for t in types], dims, mo1, od, mo2, x, prec)
    finally:
        emu.lib().emu_set_fast(1)
    assert C.rel_l2(other, ref) < tol
