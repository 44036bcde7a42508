"""The surface echo without targets (its own kernel) against the FP64 oracle
where it can go wrong: meshes that end inside a facet block, tiled and
row-ordered meshes, a range spread wider than the LDS window, facet frames
that are not orthonormal, total internal reflection, facets at a null of
their pattern, ranges on bin edges, and each option of the plain method.

Tolerance: helpers.compare_traces; the kernel's hardware sine, root and
exponential are within a few 1e-7, a thousandth of the bounds."""
import numpy as np
import pytest

from europaraypaths_amd import surfaces, workloads
from europaraypaths_amd.params import make_shots, parse_parameters
from oracle import oracle
from tests.helpers import compare_traces

pytestmark = pytest.mark.gpu


def scene(nx, ny, fs=30.0, rough=0.6, nr=512, alt=4000.0, ahead=300.0, aperture=25.0, ns=2,
          platform="REASON_VHF", **over):
    z = surfaces.gaussian_heights(nx, ny, fs, rough, 90.0, 5) if rough else np.zeros((ny, nx))
    soa = surfaces.terrain_soa(nx, ny, fs, -fs * nx / 2, -fs * ny / 2, z)
    p = workloads.make_params(platform, "planetary_ice", nr=nr, smpl=48e6, rst=alt - ahead,
                              aperture=aperture, fs=fs, ns=ns, sx0=-20.0, sdx=45.0, sy=3.0, sz=alt,
                              **over)
    par = parse_parameters(p)
    return par.to_erp(), soa, make_shots(par)


def check(ctx, e, soa, shots):
    g, gv = ctx.run(e, ctx.upload_mesh(soa), None, shots)
    o, ov = oracle.run(e, soa, None, shots)
    np.testing.assert_array_equal(gv, ov)
    assert np.abs(o).max() > 0
    compare_traces(g, o)


@pytest.mark.parametrize("nx,ny", [(1, 1), (2049, 1), (64, 32), (64, 64), (61, 67), (128, 96)])
def test_meshes(gpu_ctx, nx, ny):
    check(gpu_ctx, *scene(nx, ny))


@pytest.mark.parametrize("over", [{"lossless": True}, {"incoherent": True, "seed": 9},
                                  {"eps_1": 3.15, "eps_2": 1.0}, {"sig_1": 1e-5}])
def test_options(gpu_ctx, over):
    check(gpu_ctx, *scene(60, 50, **over))


def test_spread_wider_than_the_window(gpu_ctx):
    """One block of 2048 facets in a row: ranges over about 4000 bins."""
    check(gpu_ctx, *scene(2048, 3, fs=40.0, nr=6000, alt=3000.0, aperture=86.0, ns=1))


def test_range_window_cuts_the_echo(gpu_ctx):
    """Ranges below the first and past the last bin."""
    check(gpu_ctx, *scene(128, 96, nr=100, ahead=-40.0, aperture=40.0))


def test_general_frames(gpu_ctx):
    e, soa, shots = scene(50, 40)
    rng = np.random.default_rng(1)
    soa[6:12] += 0.05 * rng.standard_normal(soa[6:12].shape).astype(np.float32)
    check(gpu_ctx, e, soa, shots)


def test_ranges_on_bin_edges(gpu_ctx):
    """A flat mesh straight below: the nadir range lies on a bin, others
    within rounding of theirs; facets down the x axis see sin(Iph) = 0."""
    e, soa, shots = scene(65, 65, fs=20.0, rough=0.0)
    e.dr = 6.25
    shots["sx"], shots["sy"] = 10.0, 10.0
    shots["rst"] = 4000.0 - 50 * 6.25
    check(gpu_ctx, e, soa, shots)
