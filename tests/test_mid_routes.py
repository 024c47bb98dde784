"""The single-buffer mixed-radix path at the edges of its radices and routes,
against the oracle: on the CPU (the host build, every class, memory order and
precision of a case) and on the GPU.

The lengths: one radix pass (11, 16, 17), two (34, 169, 250), three (360,
1001) and four (1029), composite radices (6, 10, 12, 14, 15), primes above 16
first (17 * 7, 2 * 47), Bluestein (53 to 997), two primes above 16 (323, the
generic path); odd line counts leave partial tiles and an unpaired last real
line.  Tolerance: 8 u log2(points) relative L2 (a radix pass adds a few u of
relative error per element, log2 of the work length of them at most; the
factor covers Bluestein's two transforms and three products).
"""
import math

import numpy as np
import pytest

import cases as C
import oracle_binding as orc

# lengths that also have a compile-time kernel, which the planner leaves for
# this path by order, precision and size: run here with that kernel disabled
FIXED = [32, 48, 72, 96, 120, 144, 240, 256, 384]
LENGTHS = [11, 16, 17, 34, 119, 94, 169, 250, 360, 1001, 1029, 53, 61, 127, 131, 997, 323]
# memory orders in and out: both sides along the lines of axis 0, both
# across, and one of each
ORDERS = [([0, 1, 2], [0, 1, 2]), ([2, 0, 1], [1, 2, 0]), ([0, 1, 2], [1, 2, 0]), ([1, 2, 0], [0, 2, 1])]
KINDS = ["DCT1", "DST1", "DCT2", "DST2", "DCT3", "DST3", "DST4"]


def tol(prec, n):
    return 8 * 2.0 ** (-53 if prec == 8 else -24) * math.log2(n)


def the_cases(n, prec):
    """(types, in dims, out dims, mo1, mo2, input) of a length along axis 0, the other axes EMPTY."""
    rng = np.random.default_rng(n + prec)
    for (mo1, mo2), other in zip(ORDERS, ([5, 3], [18, 2], [7, 2], [33, 1])):
        dims = [n] + other
        half = [n // 2 + 1] + other

        def real(d):
            return rng.uniform(-1, 1, orc.storage_shape(d, mo1))

        def cplx(d):
            return real(d) + 1j * real(d)

        yield C.CF_D, dims, dims, mo1, mo2, cplx(dims)
        yield C.CB_D, dims, dims, mo1, mo2, cplx(dims)
        yield C.R2C_D, dims, half, mo1, mo2, real(dims)
        yield C.C2R_D, half, dims, mo1, mo2, cplx(half)
        if n <= 360:
            for k in KINDS:
                yield C.r2r_id(k, False, 8), dims, dims, mo1, mo2, real(dims)
            yield C.r2r_id("DST3", True, 8), dims, dims, mo1, mo2, cplx(dims)


def narrow(x, prec):
    if prec == 8:
        return x
    return x.astype(np.complex64 if np.iscomplexobj(x) else np.float32)


def wide(x):
    return x.astype(np.complex128 if np.iscomplexobj(x) else np.float64)


@pytest.mark.parametrize("prec", [8, 4])
@pytest.mark.parametrize("n", LENGTHS + FIXED)
def test_host_build(n, prec):
    import emu_binding as emu
    emu.lib().emu_set_fast(int(n not in FIXED))
    try:
        run_host_build(emu, n, prec)
    finally:
        emu.lib().emu_set_fast(1)


def run_host_build(emu, n, prec):
    for t, d1, d2, mo1, mo2, x in the_cases(n, prec):
        xi = narrow(x, prec)
        ref = orc.exec_1d(t, 0, d1, mo1, d2, mo2, wide(xi))
        got = emu.exec1d(t - (prec == 4), 0, d1, mo1, d2, mo2, xi, prec)
        assert C.rel_l2(got, ref) < tol(prec, max(n, 16)), (t, d1, mo1, mo2)


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [8, 4])
@pytest.mark.parametrize("n", LENGTHS + FIXED)
def test_gpu(n, prec):
    torch = pytest.importorskip("torch")
    import p3dfft3 as P
    P.setup()
    P.set_fast_path(n not in FIXED)
    try:
        run_gpu(torch, P, n, prec)
    finally:
        P.set_fast_path(True)


def run_gpu(torch, P, n, prec):
    pg = P.init_proc_grid((1, 1, 1))
    for t, d1, d2, mo1, mo2, x in the_cases(n, prec):
        xi = narrow(x, prec)
        print("case: route", n, prec, t, d1, mo1, mo2, flush=True)
        ref = orc.exec_1d(t, 0, d1, mo1, d2, mo2, wide(xi))
        g1 = P.init_data_grid(d1, -1, pg, (0, 1, 2), mo1)
        g2 = P.init_data_grid(d2, -1, pg, (0, 1, 2), mo2)
        h = P.plan_1Dtrans(g1, g2, t - (prec == 4), 0)
        din = torch.from_numpy(np.ascontiguousarray(xi)).cuda()
        out = narrow(np.zeros(orc.storage_shape(d2, mo2), ref.dtype), prec)
        dout = torch.from_numpy(out).cuda()
        torch.cuda.synchronize()
        P.exec_1Dtrans(h, din.data_ptr(), dout.data_ptr(), 0, prec)
        assert C.rel_l2(dout.cpu().numpy(), ref) < tol(prec, max(n, 16)), (t, d1, mo1, mo2)
