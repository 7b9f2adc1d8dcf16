"""Focus fields of few planes (tables and sums in one kernel) against the forms
with tables and per point: the same integrals summed in another order.

Tolerance: each of the two sums of n float32 products is within n 2^-24 of the
sum of the terms' magnitudes, which the field at the focus (every term in
phase) bounds."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

UNITS, LAM = (.1, .1, .1), .5


@pytest.mark.parametrize("nx,ny", [(178, 178), (182, 182), (200, 90), (512, 512)])
@pytest.mark.parametrize("nz", [2, 4, 6])
def test_few_planes_equal_the_table_form(nx, ny, nz):
    from bpm_amd.focus_fields import focus_field_debye_device as field
    for na, steps in ((.4, 200), ([.3, .5, .6, .9], 130)):
        few = field((nx, ny, nz), UNITS, LAM, na, n0=1.33, n_integration_steps=steps)
        many = field((nx, ny, 12), UNITS, LAM, na, n0=1.33, n_integration_steps=steps)
        n = (steps + 1) * (1 if na == .4 else 2)
        top = float(many[1].abs().max())
        lo = 6 - nz // 2
        for a, b in zip(few[1:], many[1:]):
            assert float((a - b[lo:lo + nz]).abs().max()) <= 2 * n * 2**-24 * top
        # I = sum of |E|^2: twice the field's bound times its largest value, three components
        assert float((few[0] - many[0][lo:lo + nz]).abs().max()) <= 3 * 4 * n * 2**-24 * top**2


@pytest.mark.parametrize("shape", [(64, 64), (65, 63), (91, 46), (300, 17)])
def test_plane_equals_the_points(shape):
    from bpm_amd.focus_fields import focus_field_debye_at, focus_field_debye_plane
    nx, ny = shape
    steps = 150
    got = focus_field_debye_plane(shape, UNITS[:2], z=.7, lam=LAM, NA=.6, n0=1.33, n_integration_steps=steps)
    x = np.linspace(-(nx // 2) * .1, (nx - nx // 2) * .1, nx, dtype=np.float32)
    y = np.linspace(-(ny // 2) * .1, (ny - ny // 2) * .1, ny, dtype=np.float32)
    yy, xx = np.meshgrid(y, x, indexing="ij")
    ref = focus_field_debye_at(xx, yy, np.full_like(xx, .7), LAM, .6, n0=1.33, n_integration_steps=steps)[1]
    zero = np.zeros(1, np.float32)
    top = abs(focus_field_debye_at(zero, zero, zero, LAM, .6, n0=1.33, n_integration_steps=steps)[1][0])
    # the axis may round a coordinate by an ulp: 2^-23 of its distance times k, on the field
    shift = 2 * np.pi * 1.33 / LAM * 2**-23 * 2 * .1 * max(shape)
    assert np.abs(got - ref).max() <= (2 * (steps + 1) * 2**-24 + 2 * shift) * top


@pytest.mark.parametrize("edge", [.05, 14., 2.**30])
def test_bessel_at_the_edges_of_its_branches(edge):
    """Within 2 ulp of 1 below 14 (float64 rounded), 8 ulp of the amplitude above."""
    from scipy.special import jv
    from bpm_amd.focus_fields import bessel_jn
    e = np.float32(edge)
    x = np.concatenate([np.nextafter(e, np.float32(0)) - np.spacing(e) * np.arange(64, dtype=np.float32),
                        e + np.spacing(e) * np.arange(64, dtype=np.float32), -e[None]]).astype(np.float32)
    ax = np.abs(x).astype(np.float64)
    bound = np.where(ax < 14, 2 * 2.**-24, 8 * 2.**-24 * np.sqrt(2 / (np.pi * ax)))
    for n in range(3):
        assert np.all(np.abs(bessel_jn(n, x).astype(np.float64) - jv(n, x.astype(np.float64))) <= bound), n
