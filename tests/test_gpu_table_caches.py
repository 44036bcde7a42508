"""The contexts' caches of device tables (range kernels, band crops, the
narrow-band chain) stay bounded however a program calls: many range lengths
through erp_run_tracks, as jobs and one by one, many receive window starts
under circular convolution; a destroyed context gives its tables back.  Traces
agree with the first pass after their tables have been dropped and built again.

Bounds: the caches keep at most 256 MB of narrow-band tables (45 MB each here),
16 circular and 64 other range kernels (0.25 MB each); a run holds the few it
reads besides.  384 MB covers that and what the work buffers grow by; the
tables of one pass would take 1080 MB."""
import ctypes
import threading

import numpy as np
import pytest

from europaraypaths_amd import surfaces, workloads
from europaraypaths_amd._abi import ERP_TUNE_PAIRS_PER_LAUNCH, ERP_TUNE_TRACK_ROWS
from europaraypaths_amd._native import Context
from europaraypaths_amd.params import make_shots, parse_parameters
from tests.helpers import compare_traces

pytestmark = pytest.mark.gpu

MB = 1 << 20
LENGTHS = [16384 - 16 * k for k in range(24)]


def free_bytes():
    h = ctypes.CDLL("libamdhip64.so")
    a, b = ctypes.c_size_t(), ctypes.c_size_t()
    assert h.hipDeviceSynchronize() == 0
    assert h.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
    return a.value


@pytest.fixture
def ctx():
    c = Context(0)
    c.set_tuning(ERP_TUNE_PAIRS_PER_LAUNCH, 64)  # small work buffers
    c.set_tuning(ERP_TUNE_TRACK_ROWS, 4)
    yield c
    c.close()


def scene(nr, **over):
    nx, ny, fs = 24, 20, 20.0
    z = surfaces.gaussian_heights(nx, ny, fs, 0.4, 60.0, 2)
    soa = surfaces.terrain_soa(nx, ny, fs, -fs * nx / 2, -fs * ny / 2, z)
    p = workloads.make_params("REASON_HF", "planetary_ice", nr=nr, smpl=48e6, rst=2600.0,
                              aperture=20.0, fs=fs, ns=2, sx0=-20.0, sdx=25.0, sy=7.0, sz=3000.0,
                              **over)
    par = parse_parameters(p)
    t = np.zeros((6, 1), np.float32)
    t[0], t[1], t[2], t[5] = 10.0, 13.0, -300.0, 1.0
    return par.to_erp(), soa, t, make_shots(par)


def jobs_of(ctx):
    """One narrow-band track per range length, 1/24 of the sample rate kept."""
    e, soa, t, shots = scene(LENGTHS[0])
    m, tg = ctx.upload_mesh(soa), ctx.upload_targets(t, np.ones(1, np.uint8))
    out = []
    for nr in LENGTHS:
        e = scene(nr)[0]
        e.B, e.rng_res = 48e6 / 24, float(e.dr) * 24
        out.append((e, m, tg, shots))
    return out


def run_all(ctx, entry, jobs):
    if entry == "tracks":
        return [g for g, _ in ctx.run_tracks(jobs)]
    if entry == "submit":
        running = [ctx.submit(*j) for j in jobs]
        return [j.wait()[0] for j in running]
    return [ctx.run(*j)[0] for j in jobs]


@pytest.mark.parametrize("entry", ["tracks", "submit", "run"])
def test_many_range_lengths(ctx, entry):
    jobs = jobs_of(ctx)
    ref = ctx.run(*jobs[0])[0]
    run_all(ctx, entry, jobs[:1] * 8)  # work buffers, slots
    before = free_bytes()
    first = run_all(ctx, entry, jobs)
    used = before - free_bytes()
    again = run_all(ctx, entry, jobs)
    print(entry, used // MB, (before - free_bytes()) // MB, flush=True)
    assert used <= 384 * MB and before - free_bytes() <= 384 * MB
    compare_traces(first[0], ref)
    for a, b in zip(first, again):
        assert np.abs(a).max() > 0
        compare_traces(b, a)


def test_many_window_starts(ctx):
    e, soa, t, shots = scene(16384, specular=True, convolution=True, convolution_linear=False,
                             rerad_funct=0)
    m, tg = ctx.upload_mesh(soa), ctx.upload_targets(t, np.zeros(1, np.uint8))
    shots = np.repeat(shots, 8)
    first = ctx.run(e, m, tg, shots)[0]
    before = free_bytes()
    for k in range(96):
        s = shots.copy()
        s["rst"] += 1.0 + 0.25 * (np.arange(16) + 16 * k)
        ctx.run(e, m, tg, s)
    used = before - free_bytes()
    print(used // MB, flush=True)
    assert used <= 64 * MB  # 1552 range kernels of 0.25 MB would take 384
    compare_traces(ctx.run(e, m, tg, shots)[0], first)


def test_a_context_gives_its_tables_back():
    def once():
        c = Context(0)
        c.set_tuning(ERP_TUNE_PAIRS_PER_LAUNCH, 64)
        for j in jobs_of(c)[:4]:
            c.run(*j)
        j = scene(16384)  # and range kernels in all their layouts, band tables
        m, tg = c.upload_mesh(j[1]), c.upload_targets(j[2], np.ones(1, np.uint8))
        e = j[0]
        for k in range(8):
            e.B, e.rng_res = 48e6 / 4, float(e.dr) * (4 + k)
            c.run(e, m, tg, j[3])
        m.release()
        tg.release()
        c.close()

    once()
    before = free_bytes()
    for _ in range(6):
        once()
    used = before - free_bytes()
    print(used // MB, flush=True)
    assert used <= 16 * MB  # 6 x 8 range kernels in three layouts would take 36


def test_dropped_beside_running_tracks(ctx):
    """Jobs drop and build tables while another thread's multi-track calls,
    which capture and replay graphs, hold some of them."""
    jobs = jobs_of(ctx)
    ref = run_all(ctx, "run", jobs)
    got, errors = [], []

    def tracks():
        try:
            for _ in range(4):
                got.append(run_all(ctx, "tracks", jobs[:6]))
        except Exception as e:  # noqa: BLE001 - reported by the main thread
            errors.append(e)

    th = threading.Thread(target=tracks)
    th.start()
    served = [run_all(ctx, "submit", jobs[k:] + jobs[:k]) for k in (0, 12)]
    th.join()
    assert not errors, errors
    for g in got:
        for a, b in zip(g, ref):
            compare_traces(a, b)
    for k, g in zip((0, 12), served):
        for a, b in zip(g, ref[k:] + ref[:k]):
            compare_traces(a, b)
