"""Per-shot spectral stages (surface range compression, band crop and
decimation, the specular spectra) and the target lists, against the FP64
oracle at the edges of their variants: range lengths at and around the
one-pass sizes (2048 bins) and powers of two, the smallest ones, bands that
keep every frequency and only the first; target lists that come with their
counts and those that follow (16384 entries).

Tolerance: helpers.compare_traces; FP32 transforms of up to 32768 points leave
about 1e-6 of the trace, a hundredth of the bounds."""
import numpy as np
import pytest

from europaraypaths_amd import surfaces, workloads
from europaraypaths_amd._abi import ERP_RUN_DETERMINISTIC
from europaraypaths_amd.params import make_shots, parse_parameters
from oracle import oracle
from tests.helpers import compare_traces

pytestmark = pytest.mark.gpu


def scene(nr, nx=32, ny=24, ns=3, targets=3, ttype=1, rst=2940.0, band=None, **over):
    fs = 20.0
    z = surfaces.gaussian_heights(nx, ny, fs, 0.3, 60.0, 3)
    soa = surfaces.terrain_soa(nx, ny, fs, -fs * nx / 2, -fs * ny / 2, z)
    p = workloads.make_params("REASON_VHF", "planetary_ice", nr=nr, smpl=48e6, rst=rst,
                              aperture=20.0, fs=fs, ns=ns, sx0=-30.0, sdx=20.0, sy=7.0, sz=3000.0,
                              **over)
    par = parse_parameters(p)
    e = par.to_erp()
    if band is not None:
        e.B = band * 48e6
    t = np.zeros((6, targets), np.float32)
    t[0] = np.linspace(-140.0, 140.0, targets)
    t[1], t[2], t[5] = 13.0, -60.0, 1.0
    return e, soa, (t, np.full(targets, ttype, np.uint8)), make_shots(par)


def check(ctx, e, soa, tg, shots, flags=0):
    o, ov = oracle.run(e, soa, tg, shots)
    m, t = ctx.upload_mesh(soa), ctx.upload_targets(*tg)
    try:
        g, gv = ctx.run(e, m, t, shots, flags=flags)
    finally:
        m.release()
        t.release()
    np.testing.assert_array_equal(gv, ov)
    assert np.abs(o).max() > 0
    print(compare_traces(g, o), flush=True)


LENGTHS = [2, 3, 31, 64, 500, 512, 513, 1024, 2047, 2048, 2049, 4096, 5000, 20000]


@pytest.mark.parametrize("nr", LENGTHS)
def test_typed_targets_alone(gpu_ctx, nr):
    """The band crop without the echo on top of it."""
    check(gpu_ctx, *scene(nr, rst=3103.0 if nr < 4 else 3030.0 if nr < 100 else 2940.0,
                           disable_surface=True))


@pytest.mark.parametrize("nr", LENGTHS)
def test_surface_and_typed_deterministic(gpu_ctx, nr):
    check(gpu_ctx, *scene(nr, rst=2998.0 if nr < 4 else 2980.0), flags=ERP_RUN_DETERMINISTIC)


@pytest.mark.parametrize("nr", [2, 300, 2048, 2049, 6000])
def test_specular_typed(gpu_ctx, nr):
    check(gpu_ctx, *scene(nr, rst=2998.0 if nr < 4 else 2980.0, specular=True, convolution=True,
                          convolution_linear=True, rerad_funct=0))


@pytest.mark.parametrize("nr", [200, 1500, 3000])
@pytest.mark.parametrize("band", [1.0, 0.5, 0.3])
def test_bands(gpu_ctx, nr, band):
    """Every frequency, half the sample rate, and a part."""
    check(gpu_ctx, *scene(nr, band=band, disable_surface=True))


@pytest.mark.parametrize("nr", [200, 3000])
def test_first_frequency_only(gpu_ctx, nr):
    """Only the mean is kept: the deterministic run keeps the transforms here."""
    check(gpu_ctx, *scene(nr, band=0.4 / (2 * nr - 1), disable_surface=True),
          flags=ERP_RUN_DETERMINISTIC)


@pytest.mark.parametrize("targets", [1638, 1639])
def test_short_and_long_target_lists(gpu_ctx, targets):
    """10 shots: 16380 and 16390 list entries."""
    check(gpu_ctx, *scene(600, nx=12, ny=10, ns=10, targets=targets, disable_surface=True))
