"""The specular method's terms, whose angles enter through sines and cosines
only, against the FP64 oracle where an angle is special: total reflection in
either direction, facets straight below the shot (no azimuth) and targets
straight below a facet, targets beside and above the facets, tilted target
normals, frames that are not orthonormal, prisms, ranges on bin edges; for
typed and type-0 targets, with and without convolution, and deterministic.

Tolerance: helpers.compare_traces; the terms' hardware sines and roots are
within a few 1e-7, a thousandth of the bounds."""
import numpy as np
import pytest

from europaraypaths_amd import surfaces, workloads
from europaraypaths_amd._abi import ERP_RUN_DETERMINISTIC, PRISM_DTYPE
from europaraypaths_amd.params import make_shots, parse_parameters, prism_alpha
from oracle import oracle
from tests.helpers import compare_traces

pytestmark = pytest.mark.gpu


def scene(ttype, convolution=True, rough=0.3, fs=20.0, nr=1024, **over):
    nx, ny = 48, 40
    z = surfaces.gaussian_heights(nx, ny, fs, rough, 60.0, 4) if rough else np.zeros((ny, nx))
    soa = surfaces.terrain_soa(nx, ny, fs, -fs * nx / 2, -fs * ny / 2, z)
    over = dict(dict(specular=True, convolution=convolution, convolution_linear=convolution,
                     rerad_funct=0), **over)
    p = workloads.make_params("REASON_VHF", "planetary_ice", nr=nr, smpl=48e6, rst=2600.0,
                              aperture=20.0, fs=fs, ns=2, sx0=-30.0, sdx=45.0, sy=7.0, sz=3000.0,
                              **over)
    par = parse_parameters(p)
    t = np.zeros((6, 3), np.float32)
    t[0], t[1], t[2] = (-80.0, 10.0, 130.0), (13.0, 5.0, -40.0), (-250.0, -300.0, -400.0)
    t[5] = 1.0
    return par, soa, (t, np.full(3, ttype, np.uint8)), make_shots(par)


def check(ctx, par, soa, tg, shots, prisms=None, flags=0):
    e = par.to_erp()
    o, ov = oracle.run(e, soa, tg, shots, prisms=prisms)
    m, t = ctx.upload_mesh(soa), ctx.upload_targets(*tg)
    try:
        g, gv = ctx.run(e, m, t, shots, prisms=prisms, flags=flags)
    finally:
        m.release()
        t.release()
    np.testing.assert_array_equal(gv, ov)
    assert np.abs(o).max() > 0
    print(compare_traces(g, o), flush=True)


KINDS = [(1, True), (0, True), (0, False)]


@pytest.mark.parametrize("ttype,conv", KINDS)
@pytest.mark.parametrize("over", [{}, {"eps_1": 3.15, "eps_2": 1.0}, {"lossless": True},
                                  {"eps_1": 1.0, "eps_2": 8.0}])
def test_media(gpu_ctx, ttype, conv, over):
    check(gpu_ctx, *scene(ttype, conv, **over))


@pytest.mark.parametrize("ttype,conv", KINDS)
def test_flat_and_straight_below(gpu_ctx, ttype, conv):
    par, soa, (t, ty), shots = scene(ttype, conv, rough=0.0)
    shots["sx"], shots["sy"] = soa[0, 500], soa[1, 500]
    shots["rst"] = 3000.0 - 50 * par.to_erp().dr
    t[0, 0], t[1, 0] = soa[0, 500], soa[1, 500]
    check(gpu_ctx, par, soa, (t, ty), shots)


@pytest.mark.parametrize("ttype,conv", KINDS)
def test_general_frames_tilted_targets_and_prisms(gpu_ctx, ttype, conv):
    par, soa, (t, ty), shots = scene(ttype, conv, sig_2=1e-3)
    soa = soa.copy()
    soa[6:12] += 0.05 * np.random.default_rng(1).standard_normal(soa[6:12].shape).astype(np.float32)
    n = np.array([0.2, -0.1, 1.0])
    t[3:6, ::2] = (n / np.linalg.norm(n)).astype(np.float32)[:, None]
    pr = np.zeros(1, PRISM_DTYPE)
    pr[0] = (prism_alpha(par, 1e-2), -200, -200, -250, 0, 200, 0)
    check(gpu_ctx, par, soa, (t, ty), shots, prisms=pr)


@pytest.mark.parametrize("ttype", [0, 1])
def test_targets_beside_and_above(gpu_ctx, ttype):
    par, soa, (t, ty), shots = scene(ttype, rough=6.0)
    t[2] = (-4.0, 3.0, -40.0)
    check(gpu_ctx, par, soa, (t, ty), shots)


@pytest.mark.parametrize("ttype", [0, 1])
def test_deterministic(gpu_ctx, ttype):
    check(gpu_ctx, *scene(ttype), flags=ERP_RUN_DETERMINISTIC)
