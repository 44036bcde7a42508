"""Tracks without targets in a multi-track call: they run no spectral chain, so
their band neither parts them from the other tracks of their range length nor
has tables built.  Every track against the FP64 oracle."""
import ctypes

import numpy as np
import pytest

from europaraypaths_amd import surfaces, workloads
from europaraypaths_amd._abi import (ERP_RUN_DETERMINISTIC, ERP_TUNE_PAIRS_PER_LAUNCH,
                                    ERP_TUNE_TRACK_ROWS)
from europaraypaths_amd._native import Context
from europaraypaths_amd.params import make_shots, parse_parameters
from oracle import oracle
from tests.helpers import compare_traces

pytestmark = pytest.mark.gpu

MB = 1 << 20


def track(platform, nr, targets, ns=3, band=None, seed=2):
    nx, ny, fs = 32, 24, 20.0
    z = surfaces.gaussian_heights(nx, ny, fs, 0.4, 60.0, seed)
    soa = surfaces.terrain_soa(nx, ny, fs, -fs * nx / 2, -fs * ny / 2, z)
    p = workloads.make_params(platform, "planetary_ice", nr=nr, smpl=48e6, rst=2600.0,
                              aperture=20.0, fs=fs, ns=ns, sx0=-20.0, sdx=25.0, sy=7.0, sz=3000.0)
    par = parse_parameters(p)
    e = par.to_erp()
    if band is not None:
        e.B, e.rng_res = band * 48e6, float(e.dr) / band
    t = np.zeros((6, targets), np.float32)
    t[0], t[1], t[5] = np.linspace(-80.0, 80.0, targets), 13.0, 1.0
    t[2] = -300.0
    return e, soa, (t, np.ones(targets, np.uint8)) if targets else None, make_shots(par)


def run(ctx, tracks, flags=0):
    jobs = [(e, ctx.upload_mesh(soa), ctx.upload_targets(*tg) if tg else None, sh)
            for e, soa, tg, sh in tracks]
    try:
        return ctx.run_tracks(jobs, flags=flags)
    finally:
        for _, m, t, _ in jobs:
            m.release()
            if t:
                t.release()


HF, VHF = "REASON_HF", "REASON_VHF"


@pytest.mark.parametrize("kinds,batches", [
    (((HF, 0), (VHF, 0)), 1),                    # no targets at all
    (((HF, 0), (VHF, 3), (HF, 0)), 1),           # beside the transforms
    (((VHF, 0), (HF, 3), (HF, 0)), 1),           # beside the narrow-band chain
    (((VHF, 0), (HF, 2), (HF, 0), (VHF, 4)), 2),  # one batch per chain
])
@pytest.mark.parametrize("nr", [1024, 1500])
def test_batches(gpu_ctx, nr, kinds, batches):
    tracks = [track(pf, nr, n, ns=2 + k, seed=k) for k, (pf, n) in enumerate(kinds)]
    gpu_ctx.profile(True)
    got = run(gpu_ctx, tracks)
    stages = gpu_ctx.profile_read()
    gpu_ctx.profile(False)
    for (e, soa, tg, shots), (g, gv) in zip(tracks, got):
        o, ov = oracle.run(e, soa, tg, shots)
        np.testing.assert_array_equal(gv, ov)
        print(compare_traces(g, o), flush=True)
    assert stages["mask"][1] == batches
    # deterministic: the same bits as each track alone
    for t, (d, _) in zip(tracks, run(gpu_ctx, tracks, ERP_RUN_DETERMINISTIC)):
        np.testing.assert_array_equal(d, run(gpu_ctx, [t], ERP_RUN_DETERMINISTIC)[0][0])


def test_no_tables_for_tracks_without_targets():
    """Four of 45 MB each, were they built."""
    h = ctypes.CDLL("libamdhip64.so")

    def free_bytes():
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert h.hipDeviceSynchronize() == 0
        assert h.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
        return a.value

    ctx = Context(0)
    try:
        ctx.set_tuning(ERP_TUNE_PAIRS_PER_LAUNCH, 64)
        ctx.set_tuning(ERP_TUNE_TRACK_ROWS, 4)
        first = track(HF, 16384, 2)
        others = [track(HF, 16384, 0, band=1 / (24.0 + 0.25 * k)) for k in range(4)]
        run(ctx, [first] * 5)
        before = free_bytes()
        got = run(ctx, [first] + others)
        used = before - free_bytes()
        for (e, soa, tg, shots), (g, _) in zip([first] + others, got):
            compare_traces(g, oracle.run(e, soa, tg, shots)[0])
        print(used // MB, flush=True)
        assert used <= 32 * MB
    finally:
        ctx.close()
