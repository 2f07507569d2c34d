"""The direct sums on the full-precision matrix cores (csrc/direct_gemm.h) at
the sizes where they can go wrong, against the FP64 probe on every pixel:
holograms one pixel off whole 128 x 64 workgroup tiles, point counts around
the K slots and the 120-point chunks, point depths that need every rank of
the RS expansion and that leave pairs to the per-pixel kernels, partial masks.

Tolerances (rel-L2 over the field), derived from the terms the sums drop:
FP64 1e-11 (at most 6e-13 of a term per pair plus the FP64 phase rounding of
~1e3 cycles), FP32 1e-5, the bars of the other direct-kernel tests; pixels
that no point's mask covers are exactly zero.
"""
import numpy as np
import pytest

from openholo_amd import capi, synth

pytestmark = pytest.mark.gpu

FP64 = capi.MODE_GPU
FP32 = capi.MODE_GPU | capi.MODE_FLOAT
LAM = 532e-9


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


def check(ctx, v, pn, pp, diff, mode, tol, **kw):
    npx = pn[0] * pn[1]
    got = capi.generate(ctx, v, pn, pp, [LAM], diff, mode, **kw)[0].ravel()
    dv = ctx.to_device(v)
    try:
        want = ctx.probe_f64(dv, len(v), capi.params(pn, pp, LAM, **kw), diff, np.arange(npx))
    finally:
        dv.free()
    assert np.array_equal(got != 0, want != 0)
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    print(f"{pn} n {len(v)} diff {diff} mode {mode}: rel-L2 {err:.2e}")
    assert err < tol


@pytest.mark.parametrize("mode,tol", [(FP64, 1e-11), (FP32, 1e-5)])
@pytest.mark.parametrize("diff", [0, 1])
@pytest.mark.parametrize("pn,n", [((1, 1), 1), ((127, 63), 2), ((128, 64), 3), ((129, 65), 5), ((257, 191), 119),
                                  ((256, 130), 120), ((130, 129), 121), ((300, 70), 363)])
def test_tile_and_point_remainders(ctx, pn, n, diff, mode, tol):
    v = synth.random_cloud(6100 + n, n, 0.6e-3, (0.2, 0.25), complex_amplitude=True)
    check(ctx, v, pn, (8e-6, 6e-6), diff, mode, tol, offset=(2, -3), use_phase=True)


# depths at 8 um pitch: every rank from 3 to 8 (FP64) and 2 to 4 (FP32), and
# pairs left to the per-pixel kernels (2-20 mm; partial masks below ~60 mm)
@pytest.mark.parametrize("mode,tol", [(FP64, 1e-11), (FP32, 1e-5)])
@pytest.mark.parametrize("diff", [0, 1])
@pytest.mark.parametrize("z", [(2e-3, 2e-2), (2e-2, 6e-2), (6e-2, 0.12), (0.12, 0.3), (0.3, 1.5)])
def test_depths(ctx, z, diff, mode, tol):
    v = synth.random_cloud(6200 + int(1e3 * z[0]), 150, 2e-3, z)
    check(ctx, v, (420, 300), (8e-6, 8e-6), diff, mode, tol)


# Fresnel near the hologram, where phases are small: the FP64 sums and the probe
# round phases of at most lambda z / (4 pitch^2) cycles (both axes at the box
# corner) to half a unit in the last place, a few times each
@pytest.mark.parametrize("pp", [8e-6, 3.74e-6])
@pytest.mark.parametrize("z", [1e-3, 3e-3, 1e-2])
def test_fresnel_fp64_phase_rounding(ctx, z, pp):
    v = synth.random_cloud(6250, 200, 200 * pp, (0.9 * z, z), complex_amplitude=True)
    check(ctx, v, (700, 500), (pp, pp), 1, FP64, 8 * np.pi * (LAM * z / (4 * pp * pp) + 1) * 2.0**-53, use_phase=True)


# one RS point at a time, where the terms dropped beside the last power of the
# expansion weigh most (6th rank, the largest tiles that the product takes), and at
# depths that take all ranks: no pixel is off by more than the tolerance of the
# expansion, 2e-13, and the rounding of the phases
@pytest.mark.parametrize("x,y,z", [(8e-5, 8.1e-4, 0.0252), (-4e-4, -8.1e-4, 0.0207), (3.5e-4, 8.8e-4, 0.0286),
                                   (-1e-4, 6.5e-4, 0.0222), (5.2e-4, -9e-4, 0.0246), (0.0, 0.0, 0.06),
                                   (1e-3, -1e-3, 0.12), (2e-3, 1e-3, 0.3), (-1e-3, 2e-3, 0.6)])
def test_rs_fp64_single_points(ctx, x, y, z):
    v = synth.random_cloud(6260, 1, 1e-3, (0.1, 0.2)).copy()
    v["pos"][0] = x, y, z
    pn, pp = (700, 500), (8e-6, 8e-6)
    got = capi.generate(ctx, v, pn, pp, [LAM], 0, FP64)[0].ravel()
    dv = ctx.to_device(v)
    try:
        want = ctx.probe_f64(dv, 1, capi.params(pn, pp, LAM), 0, np.arange(pn[0] * pn[1]))
    finally:
        dv.free()
    inside = want != 0
    assert np.array_equal(got != 0, inside)
    err = float(np.max(np.abs(got - want)[inside] / np.abs(want[inside])))
    print(f"z {z}: {err:.2e}")
    assert err < 2e-13 + 8 * np.pi * (LAM * z / (4 * pp[0] * pp[1]) + 1) * 2.0**-53


# RS points near the hologram, all left to the per-pixel FP64 terms: around the
# points listed at a time (1024 or 256), the 64 x 8 tiles (64 x 32 from 512 of them) and the
# shares of a tile (16, a server's job 4)
@pytest.mark.parametrize("pn", [(64, 8), (65, 9), (70, 13), (130, 71), (1030, 961), (1030, 960)])
@pytest.mark.parametrize("n", [1, 5, 17, 255, 257, 1023, 1025, 2100])
def test_rs_fp64_left_points(ctx, pn, n):
    pp = (8e-6, 8e-6)
    v = synth.random_cloud(6270 + n, n, 0.6 * pn[1] * pp[1], (2e-3, 8e-3))
    check(ctx, v, pn, pp, 0, FP64, 1e-11)
    one = capi.generate(ctx, v, pn, pp, [LAM], 0, FP64)[0]
    with capi.Server(0) as srv:
        status, _, field, _ = srv.wait(srv.submit(v, capi.params(pn, pp, LAM), 0, FP64, want_field=True))
    assert status == capi.OK
    assert np.array_equal(field.reshape(one.shape) != 0, one != 0)
    assert np.linalg.norm(field.reshape(one.shape) - one) <= 1e-11 * np.linalg.norm(one)


# around the 240 points that the FP64 sums list at a time, over the depths of many
# ranks (each rank's points padded in the list)
@pytest.mark.parametrize("diff", [0, 1])
@pytest.mark.parametrize("z", [(0.05, 0.06), (0.06, 1.5)])
@pytest.mark.parametrize("n", [239, 240, 241, 255, 257, 481, 721])
def test_fp64_listed_points(ctx, n, z, diff):
    v = synth.random_cloud(6290 + n, n, 1.5e-3, z, complex_amplitude=True)
    check(ctx, v, (300, 200), (8e-6, 8e-6), diff, FP64, 1e-11, use_phase=True)


# Fresnel points so far away that their phases have no digits left: finite, and as
# in the probe
@pytest.mark.parametrize("mode", [FP64, FP32])
@pytest.mark.parametrize("x,z", [(1e3, 1e6), (1e12, 1e18), (1e80, 1e90), (1e150, 1e160)])
def test_fresnel_far_points(ctx, x, z, mode):
    v = synth.random_cloud(6295, 3, 1e-3, (0.1, 0.2)).copy()
    v["pos"][1] = x, -0.5 * x, z
    pn, pp = (200, 100), (8e-6, 8e-6)
    got = capi.generate(ctx, v[1:2], pn, pp, [LAM], 1, mode)[0].ravel()
    assert np.isfinite(got).all() and (got != 0).any()
    check(ctx, v, pn, pp, 1, mode, 1e-11 if mode == FP64 else 1e-5)
