"""The direct sums where their kernels hand over, against the FP64 probe on
every pixel: FP32 sums at the edges of the 128 x 128 tiles, of the 16-point
batches, of the 30, 60 and 240-point folds and of the 480 points listed at a
time; boxes that end inside the hologram (the RS edge lines); clouds around the
work at which RS in FP32 takes the per-pixel kernel; amplitudes that a zero
factor cannot mask.

Tolerances (rel-L2 over the field): the bars of the other direct-kernel tests,
FP64 1e-11 and FP32 1e-5; the mask is exact.
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
    got = capi.generate(ctx, v, pn, pp, [LAM], diff, mode, **kw)[0].ravel()
    dv = ctx.to_device(v)
    try:
        want = ctx.probe_f64(dv, len(v), capi.params(pn, pp, LAM, **kw), diff, np.arange(pn[0] * pn[1]))
    finally:
        dv.free()
    finite = np.isfinite(want)
    assert np.array_equal(np.isfinite(got), finite)
    assert np.array_equal(got[finite] != 0, want[finite] != 0)
    err = np.linalg.norm(got[finite] - want[finite]) / np.linalg.norm(want[finite])
    print(f"{pn} n {len(v)} diff {diff} mode {mode}: rel-L2 {err:.2e}")
    assert err < tol


@pytest.mark.parametrize("diff", [0, 1])
@pytest.mark.parametrize("pn,n", [((127, 127), 15), ((128, 128), 16), ((129, 129), 17), ((257, 255), 30),
                                  ((256, 256), 31), ((130, 140), 60), ((140, 130), 61), ((100, 90), 481),
                                  ((260, 130), 2041), ((1030, 514), 3841)])
def test_fp32_tiles_and_folds(ctx, pn, n, diff):
    v = synth.random_cloud(6300 + n, n, 0.8e-3, (0.25, 0.3), complex_amplitude=True)
    check(ctx, v, pn, (8e-6, 8e-6), diff, FP32, 1e-5)


@pytest.mark.parametrize("mode,tol", [(FP64, 1e-11), (FP32, 1e-5)])
@pytest.mark.parametrize("diff", [0, 1])
@pytest.mark.parametrize("pn,n,z", [((300, 200), 1, 0.02), ((300, 200), 9, 0.03), ((700, 300), 65, 0.06),
                                    ((513, 257), 130, 0.04), ((1300, 700), 400, 0.05)])
def test_boxes_inside_the_hologram(ctx, pn, n, z, diff, mode, tol):
    v = synth.random_cloud(6400 + n, n, 0.8 * pn[1] * 8e-6, (0.9 * z, z))
    check(ctx, v, pn, (8e-6, 8e-6), diff, mode, tol)


@pytest.mark.parametrize("pn,n", [((640, 480), 325), ((640, 480), 326), ((640, 288), 100), ((641, 288), 100)])
def test_rs_fp32_per_pixel_limits(ctx, pn, n):
    v = synth.random_cloud(6500 + n, n, 2e-3, (0.1, 0.2))
    check(ctx, v, pn, (8e-6, 8e-6), 0, FP32, 1e-5)


@pytest.mark.parametrize("mode,tol", [(FP64, 1e-11), (FP32, 1e-5)])
@pytest.mark.parametrize("diff", [0, 1])
@pytest.mark.parametrize("amp", [float("inf"), float("nan"), 0.0, 1e-30])
def test_amplitudes(ctx, amp, diff, mode, tol):
    v = synth.random_cloud(6600, 40, 1.5e-3, (0.02, 0.03)).copy()
    v["color"][17] = amp
    check(ctx, v, (400, 300), (8e-6, 8e-6), diff, mode, tol)


# a phase that is not finite: NaN at the pixels of the point's mask (of the whole
# hologram where the mask covers it), as in the probe, and only there; few points
# on a large hologram take the per-pixel kernel in RS FP32, the others the matrix
# products
@pytest.mark.parametrize("mode,tol", [(FP64, 1e-11), (FP32, 1e-5)])
@pytest.mark.parametrize("diff", [0, 1])
@pytest.mark.parametrize("phase", [float("nan"), float("inf"), -float("inf")])
@pytest.mark.parametrize("pn,n,z", [((400, 300), 40, (0.02, 0.03)), ((900, 500), 40, (0.02, 0.03)),
                                    ((700, 400), 700, (0.1, 0.2)), ((700, 400), 700, (0.05, 0.06))])
def test_phases_not_finite(ctx, pn, n, z, phase, diff, mode, tol):
    v = synth.random_cloud(6650, n, 1.5e-3, z, complex_amplitude=True).copy()
    v["phase"][17] = phase
    pp = (8e-6, 8e-6)
    got = capi.generate(ctx, v, pn, pp, [LAM], diff, mode, use_phase=True)[0].ravel()
    dv = ctx.to_device(v)
    try:
        want = ctx.probe_f64(dv, len(v), capi.params(pn, pp, LAM, use_phase=True), diff, np.arange(pn[0] * pn[1]))
    finally:
        dv.free()
    finite = np.isfinite(want)
    assert not finite.all() and np.array_equal(np.isfinite(got), finite)
    assert np.linalg.norm(got[finite] - want[finite]) <= tol * np.linalg.norm(want[finite])


# clouds that Fresnel in FP32 leaves to the FP64 terms altogether (amplitudes below
# the products' range), around the points tested at a time and with some that the
# products take between them: FP64 accuracy
@pytest.mark.parametrize("n", [1, 511, 512, 513, 1100])
@pytest.mark.parametrize("mixed", [False, True])
def test_fresnel_fp32_left_points(ctx, n, mixed):
    v = synth.random_cloud(6680 + n, n, 1.5e-3, (0.02, 0.03)).copy()
    v["color"] *= 1e-38
    if mixed:
        v["color"][n // 3:n // 2] = 0.0
    check(ctx, v, (300, 200), (8e-6, 8e-6), 1, FP32, 1e-11)


# faint clouds: their products keep every part of a factor down to amplitudes (in
# the field) of 1e-30
@pytest.mark.parametrize("diff", [0, 1])
@pytest.mark.parametrize("scale", [1e-12, 1e-25, 1e-30, 1e-35, 1e-36])
def test_fp32_faint_clouds(ctx, scale, diff):
    v = synth.random_cloud(6690, 300, 1.5e-3, (0.25, 0.3)).copy()
    ref = capi.generate(ctx, v, (300, 200), (8e-6, 8e-6), [LAM], diff, FP32)[0]
    v["color"] *= scale
    got = capi.generate(ctx, v, (300, 200), (8e-6, 8e-6), [LAM], diff, FP32)[0] / scale
    # both round to FP32
    assert np.linalg.norm(got - ref) <= 2e-6 * np.linalg.norm(ref)


# Fresnel points so near that a phase runs over more than 64 cycles on 64 x 32
# pixels (boxes of at most 25 pixels here): FP64 terms in FP32 mode too
@pytest.mark.parametrize("pn,n,pp,z", [((300, 200), 300, 8e-6, (1e-3, 3e-3)), ((130, 129), 2000, 8e-6, (0.5e-3, 2e-3)),
                                       ((700, 500), 900, 3.74e-6, (0.2e-3, 0.6e-3))])
def test_fresnel_fp32_nearest_points(ctx, pn, n, pp, z):
    v = synth.random_cloud(6695 + n, n, 0.6 * pn[1] * pp, z, complex_amplitude=True)
    check(ctx, v, pn, (pp, pp), 1, FP32, 1e-11, use_phase=True)


# The FP32 sums hold FP32 factors in three BF16 parts.  What they round: phases to
# 2^-25 cycles (2e-7 rad) and sines to about 1e-7 per factor, two factors a term, and
# FP32 sums of up to 240 terms (up to 3e-7 of the sum); ranks cut at 4.5e-8: in all
# below 1e-6.  A factor without its third part is off by up to 8e-6, a rank's factor
# without its second by 3e-5 of the term.
ROUNDING = 1e-6


@pytest.mark.parametrize("pn,n,z", [((256, 256), 100, (0.1, 0.3)), ((256, 256), 2000, (0.1, 0.3)),
                                    ((640, 500), 600, (0.3, 0.6)), ((500, 300), 300, (0.02, 0.04))])
def test_fresnel_fp32_rounding(ctx, pn, n, z):
    v = synth.random_cloud(6710 + n, n, 1e-3, z, complex_amplitude=True)
    check(ctx, v, pn, (8e-6, 8e-6), 1, FP32, ROUNDING, use_phase=True)


# depths at which points near the axis of 256 x 256 pixels take rank 2, 3 and 4
# (theta = 1.83e-6 / z^3 at the far corner of a tile)
@pytest.mark.parametrize("n", [100, 700, 2000])
@pytest.mark.parametrize("z", [(0.3, 0.35), (0.08, 0.1), (0.042, 0.05)])
def test_rs_fp32_rounding(ctx, n, z):
    v = synth.random_cloud(6720 + n, n, 0.1e-3, z, complex_amplitude=True)
    check(ctx, v, (256, 256), (8e-6, 8e-6), 0, FP32, ROUNDING, use_phase=True)
