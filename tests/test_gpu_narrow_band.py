"""The narrow-band chain of typed targets (erp_narrow.hip) against the FP64
oracle and against the full-rate transforms, which a deterministic run keeps:
range lengths from the first the chain takes, odd and even, at and off powers
of two; bands from one frequency to the limit of the rule and past it; slices
of one and of many pairs, cut by the launches; rows wider than the target
kernel's window; the single-shot target kernel; multi-track batches that mix
plans; the allocation-free entry point.

Tolerance: helpers.compare_traces against the oracle, 1e-4 of the peak between
the chains.  The filter's stop band (180 dB) and the FP32 sums leave about 1e-6
of the trace, a hundredth of the bounds."""
import numpy as np
import pytest

from europaraypaths_amd import surfaces, workloads
from europaraypaths_amd._abi import (ERP_RUN_DETERMINISTIC, ERP_TUNE_PAIRS_PER_LAUNCH,
                                    ERP_TUNE_SINGLE_SHOT)
from europaraypaths_amd.params import make_shots, parse_parameters
from oracle import oracle
from tests.helpers import compare_traces
from tests.test_gpu_tracks import _Uploaded
from tests.test_zz_no_alloc import DevOut

pytestmark = pytest.mark.gpu


def scene(nr, band=None, nx=48, ny=40, fs=20.0, nt=(3, 2), depth=300.0, rst=2600.0, ns=3,
          aperture=20.0, sdx=25.0, **over):
    """band: the kept part of the sample rate (None: 1 of 48 MHz)."""
    z = surfaces.gaussian_heights(nx, ny, fs, 0.4, 60.0, 2)
    soa = surfaces.terrain_soa(nx, ny, fs, -fs * nx / 2, -fs * ny / 2, z)
    p = workloads.make_params("REASON_HF", "planetary_ice", nr=nr, smpl=48e6, rst=rst,
                              aperture=aperture, fs=fs, ns=ns, sx0=-40.0, sdx=sdx, sy=7.0,
                              sz=3000.0, **over)
    par = parse_parameters(p)
    e = par.to_erp()
    if band is not None:
        e.B = band * 48e6
        e.rng_res = float(e.dr) / band
    xs, ys = np.meshgrid(np.linspace(-150.0, 150.0, nt[0]), 13.0 + np.linspace(-40.0, 40.0, nt[1]))
    t = np.zeros((6, xs.size), np.float32)
    t[0], t[1], t[2], t[5] = xs.ravel(), ys.ravel(), -depth, 1.0
    return par, e, soa, (t, np.ones(xs.size, np.uint8)), make_shots(par)


def check(ctx, e, soa, tg, shots, tune=()):
    o, ov = oracle.run(e, soa, tg, shots)
    m, t = ctx.upload_mesh(soa), ctx.upload_targets(*tg)
    try:
        d, _ = ctx.run(e, m, t, shots, flags=ERP_RUN_DETERMINISTIC)
        for k, v in tune:
            ctx.set_tuning(k, v)
        g, gv = ctx.run(e, m, t, shots)
    finally:
        for k, _ in tune:
            ctx.set_tuning(k, 0)
        m.release()
        t.release()
    np.testing.assert_array_equal(gv, ov)
    assert np.abs(o).max() > 0
    print(compare_traces(g, o), flush=True)
    for a, b, c in zip(g, d, o):
        assert np.abs(a - b).max() <= 1e-4 * np.abs(c).max()


@pytest.mark.parametrize("nr", [513, 600, 1023, 1024, 2049, 4096, 6001, 16383, 16384])
def test_range_lengths(gpu_ctx, nr):
    _, e, soa, tg, shots = scene(nr, disable_surface=True)
    check(gpu_ctx, e, soa, tg, shots)


@pytest.mark.parametrize("band", [0.4 / 2047, 1 / 500, 1 / 100, 1 / 24, 0.99 / 12, 1.01 / 12])
def test_bands(gpu_ctx, band):
    """From one kept frequency to both sides of the rule (the compressed
    window is then as wide as the band asks)."""
    _, e, soa, tg, shots = scene(1024, band, disable_surface=True)
    check(gpu_ctx, e, soa, tg, shots)


@pytest.mark.parametrize("nt,tune", [((1, 1), ()), ((17, 2), ()),
                                     ((17, 4), ((ERP_TUNE_PAIRS_PER_LAUNCH, 45),)),
                                     ((9, 4), ((ERP_TUNE_SINGLE_SHOT, 1),))])
def test_slices(gpu_ctx, nt, tune):
    """Slices of one, 32 and the pairs left over; launches that cut them;
    both target kernels."""
    _, e, soa, tg, shots = scene(1500, nt=nt, disable_surface=True)
    check(gpu_ctx, e, soa, tg, shots, tune)


@pytest.mark.parametrize("rst", [2950.0, 1100.0])
def test_echo_at_the_ends_of_the_range(gpu_ctx, rst):
    """Windows at the first bins and past the last."""
    _, e, soa, tg, shots = scene(640, rst=rst, disable_surface=True)
    check(gpu_ctx, e, soa, tg, shots)


def test_rows_wider_than_the_window(gpu_ctx):
    _, e, soa, tg, shots = scene(16384, nx=300, ny=24, fs=100.0, aperture=85.0, ns=2,
                                 disable_surface=True)
    check(gpu_ctx, e, soa, tg, shots)


def test_tracks_of_several_plans(gpu_ctx):
    """One range length: two bands of the chain, a track without targets, one
    of the transforms; against the oracle."""
    tracks = []
    for k, over in enumerate(({}, {"bandwidth": 5e5}, {}, {"bandwidth": 1e7})):
        par, e, soa, tg, shots = scene(1024, nt=(5, 2 + k), ns=5 + k, **over)
        tracks.append((f"t{k}", par, soa, None if k == 2 else tg, shots))
    up = _Uploaded(gpu_ctx, tracks)
    try:
        for _ in range(2):
            got = gpu_ctx.run_tracks(up.jobs)
            for (name, par, soa, tg, shots), (g, gv) in zip(tracks, got):
                o, ov = oracle.run(par.to_erp(), soa, tg, shots)
                np.testing.assert_array_equal(gv, ov)
                print(name, compare_traces(g, o), flush=True)
    finally:
        up.release()


@pytest.mark.parametrize("nr", [1024, 16384])
def test_allocation_free(gpu_ctx, nr):
    _, e, soa, tg, shots = scene(nr, nt=(5, 3), ns=5)
    o, ov = oracle.run(e, soa, tg, shots)
    m, t = gpu_ctx.upload_mesh(soa), gpu_ctx.upload_targets(*tg)
    d = DevOut(shots.shape[0], nr)
    try:
        gpu_ctx.run_dev_noalloc(e, m, t, shots, d.out.value, d.nv.value)
        g, gv = d.read()
    finally:
        d.free()
        m.release()
        t.release()
    np.testing.assert_array_equal(gv, ov)
    compare_traces(g, o)
