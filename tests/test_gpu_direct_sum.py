"""The direct sinc sums (specular method without convolution) against the FP64
oracle at the edges of their tiles and splits: bins around the 1024-bin tile,
term groups around 256 facets and around the groups one workgroup takes, a
range lying exactly on a bin (where the sinc is 1), no type-0 target in the
aperture, and the splits of a shot not depending on its batch.

Tolerance: every quantity per term is FP32 of about 1e-6 relative error and
the sums are FP64, so the parity bounds of helpers.compare_traces (1e-3 rad,
1e-4 relative within 40 dB, 1e-4 of the peak everywhere) hold with room."""
import numpy as np
import pytest

from europaraypaths_amd import surfaces, workloads
from europaraypaths_amd._abi import ERP_TUNE_SHOTS_PER_BATCH
from europaraypaths_amd.params import make_shots, parse_parameters
from oracle import oracle
from tests.helpers import compare_traces

pytestmark = pytest.mark.gpu


def scene(nx, ny, nr, ns, nt, rough=0.2, alt=3000.0, rst=2600.0):
    fs = 20.0
    z = surfaces.gaussian_heights(nx, ny, fs, rough, 60.0, 3) if rough else np.zeros((ny, nx))
    soa = surfaces.terrain_soa(nx, ny, fs, -fs * (nx // 2), -fs * (ny // 2), z)
    p = workloads.make_params("REASON_VHF", "planetary_ice", nr=nr, smpl=48e6, rst=rst,
                              aperture=60.0, fs=fs, ns=ns, sx0=0.0, sdx=40.0, sy=0.0, sz=alt,
                              specular=True, convolution=False, convolution_linear=False,
                              rerad_funct=0)
    par = parse_parameters(p)
    tg = None
    if nt:
        xyzn = np.zeros((6, nt), np.float32)
        xyzn[0] = np.linspace(-90.0, 90.0, nt)
        xyzn[2] = -300.0
        xyzn[5] = 1.0
        tg = (xyzn, np.zeros(nt, np.uint8))
    return par.to_erp(), soa, tg, make_shots(par)


@pytest.mark.parametrize("nx,ny,nr,ns,nt", [
    (1, 1, 2, 1, 1),        # one facet, the two bins the transforms need at least
    (16, 16, 255, 1, 1),    # 256 facets: one full term group
    (257, 1, 1023, 2, 3),   # one facet past a group; bins short of a tile
    (32, 32, 1024, 1, 1),   # four groups: one split; a full tile
    (41, 25, 1025, 1, 5),   # one facet past four groups; one bin past a tile
    (30, 27, 5000, 3, 2),   # several tiles, fewer splits
])
def test_direct_sum_edges(gpu_ctx, nx, ny, nr, ns, nt):
    e, soa, tg, shots = scene(nx, ny, nr, ns, nt)
    m, t = gpu_ctx.upload_mesh(soa), gpu_ctx.upload_targets(*tg)
    g, gv = gpu_ctx.run(e, m, t, shots)
    o, ov = oracle.run(e, soa, tg, shots)
    np.testing.assert_array_equal(gv, ov)
    compare_traces(g, o)
    g0, _ = gpu_ctx.run(e, m, None, shots)
    compare_traces(g0, oracle.run(e, soa, None, shots)[0])


def test_direct_sum_range_on_a_bin(gpu_ctx):
    """The nadir facet's range (3000 m) is bin 64's own (2600 + 64 x 6.25)."""
    e, soa, tg, shots = scene(9, 9, 200, 1, 0, rough=0.0)
    e.dr = 6.25
    g, _ = gpu_ctx.run(e, gpu_ctx.upload_mesh(soa), None, shots)
    compare_traces(g, oracle.run(e, soa, None, shots)[0])


def test_direct_sum_does_not_depend_on_the_batch(gpu_ctx):
    e, soa, tg, shots = scene(64, 50, 900, 5, 4)
    m, t = gpu_ctx.upload_mesh(soa), gpu_ctx.upload_targets(*tg)
    a, _ = gpu_ctx.run(e, m, t, shots)
    gpu_ctx.set_tuning(ERP_TUNE_SHOTS_PER_BATCH, 2)
    try:
        b, _ = gpu_ctx.run(e, m, t, shots)
    finally:
        gpu_ctx.set_tuning(ERP_TUNE_SHOTS_PER_BATCH, 0)
    np.testing.assert_array_equal(a, b)
