"""Precision of a typed target's echo under the specular method against the
FP64 oracle, where the facets are small against the wavelength and the target
is straight below: all the sincs of a term are near 1 with small arguments, and
the terms add up coherently, so that an error common to them shows in full.

Compared is what the target adds to the trace.  Tolerance, of its peak: the
factors common to all terms round some eight times in each of the two traces
that are multiplied (1e-6 at the worst, 3e-7 as a rule), the transforms in FP32
add up to 5e-7.  Together 1.5e-6."""
import numpy as np
import pytest

from europaraypaths_amd import surfaces, workloads
from europaraypaths_amd.params import make_shots, parse_parameters
from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lossless", [False, True])
@pytest.mark.parametrize("alt,aperture", [(4000.0, 3.0), (12000.0, 1.5)])
@pytest.mark.parametrize("platform,fs", [("REASON_HF", 2.0), ("REASON_HF", 4.0),
                                         ("REASON_VHF", 2.0)])
def test_target_below_small_facets(gpu_ctx, platform, fs, alt, aperture, lossless):
    n = 61
    z = surfaces.gaussian_heights(n, n, fs, 0.01, 5 * fs, 11)
    soa = surfaces.terrain_soa(n, n, fs, -fs * n / 2, -fs * n / 2, z)
    p = workloads.make_params(platform, "planetary_ice", nr=700, smpl=48e6, rst=alt - 300.0,
                              aperture=aperture, fs=fs, ns=2, sx0=-20.0, sdx=12.0, sy=7.0, sz=alt,
                              specular=True, convolution=True, convolution_linear=True,
                              rerad_funct=0, lossless=lossless)
    par = parse_parameters(p)
    e, shots = par.to_erp(), make_shots(par)
    t = np.zeros((6, 1), np.float32)
    t[0], t[1], t[2], t[5] = 9.0, 5.0, -900.0, 1.0
    tg = (t, np.ones(1, np.uint8))
    m, T = gpu_ctx.upload_mesh(soa), gpu_ctx.upload_targets(*tg)
    g = gpu_ctx.run(e, m, T, shots)[0].astype(complex) - gpu_ctx.run(e, m, None, shots)[0]
    m.release()
    T.release()
    s = oracle.run(e, soa, None, shots)[0]
    o = oracle.run(e, soa, tg, shots)[0] - s
    # the traces' own rounding, 6e-8 of the surface echo, stays below the bound
    assert np.abs(o).max() > 0.2 * np.abs(s).max()
    err = np.abs(g - o).max() / np.abs(o).max()
    print("%.2e" % err, flush=True)
    assert err <= 1.5e-6
