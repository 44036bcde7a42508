"""The rounding error of the typed targets' chains, the band crop and the
direct sinc sums against the FP64 oracle, of the trace's peak.

Tolerance 3e-6: the factors that all terms of an echo share round some eight
times in each of two legs (1e-6 at the worst), the terms of type-0 targets carry
their reradiation squared twice (another 1e-6), and five FP32 transforms of up
to 2^15 points leave about 2.3e-7 each (6e-8 sqrt(15)), 5e-7 together."""
import numpy as np
import pytest

from europaraypaths_amd import surfaces, workloads
from europaraypaths_amd._abi import ERP_RUN_DETERMINISTIC
from europaraypaths_amd.params import make_shots, parse_parameters
from oracle import oracle

pytestmark = pytest.mark.gpu

DIRECT = {"specular": True, "convolution": False, "convolution_linear": False, "rerad_funct": 0}


@pytest.mark.parametrize("flags", [0, ERP_RUN_DETERMINISTIC])
@pytest.mark.parametrize("platform,nr,ttype,over", [
    ("REASON_HF", 700, 1, {}), ("REASON_HF", 4096, 1, {}), ("REASON_HF", 16000, 1, {}),
    ("REASON_VHF", 400, 1, {}), ("REASON_VHF", 1024, 1, {}), ("REASON_VHF", 3000, 1, {}),
    ("REASON_VHF", 16384, 1, {}), ("REASON_VHF", 20000, 1, {}),
    ("REASON_VHF", 900, 0, DIRECT), ("REASON_HF", 2500, 0, DIRECT)])
def test_against_the_oracle(gpu_ctx, platform, nr, ttype, over, flags):
    nx, ny, fs = 48, 40, 20.0
    z = surfaces.gaussian_heights(nx, ny, fs, 0.3, 100.0, 5)
    soa = surfaces.terrain_soa(nx, ny, fs, -fs * nx / 2, -fs * ny / 2, z)
    if not over:
        over = {"disable_surface": True}  # the targets' echo alone
    p = workloads.make_params(platform, "planetary_ice", nr=nr, smpl=48e6, rst=2950.0,
                              aperture=12.0, fs=fs, ns=3, sx0=-30.0, sdx=25.0, sy=7.0, sz=3000.0,
                              **over)
    par = parse_parameters(p)
    e, shots = par.to_erp(), make_shots(par)
    t = np.zeros((6, 4), np.float32)
    t[0], t[1], t[5] = np.linspace(-80.0, 80.0, 4), 13.0, 1.0
    t[2] = -150.0
    tg = (t, np.full(4, ttype, np.uint8))
    m, T = gpu_ctx.upload_mesh(soa), gpu_ctx.upload_targets(*tg)
    g = gpu_ctx.run(e, m, T, shots, flags=flags)[0]
    m.release()
    T.release()
    o = oracle.run(e, soa, tg, shots)[0]
    err = (np.abs(g - o).max(1) / np.abs(o).max(1)).max()
    print("%.2e" % err, flush=True)
    assert err <= 3e-6
