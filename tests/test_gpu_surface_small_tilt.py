"""The surface echo without targets where a facet straight below the shot is
tilted by next to nothing: far out on a Gaussian hill the tangents' heights
fall through every power of ten, so that the squares of the ray's projections
on them pass the smallest normal float, and rounding leaves the sine of the
incidence angle a little above zero all the same.

Tolerance: helpers.compare_traces (no term of these scenes is special in the
exact arithmetic)."""
import numpy as np
import pytest

from europaraypaths_amd import surfaces, workloads
from europaraypaths_amd.params import make_shots, parse_parameters
from oracle import oracle
from tests.helpers import compare_traces

pytestmark = pytest.mark.gpu


def hill(n, fs, sigma, height):
    c = (np.arange(n) - n // 2) * fs
    z = height * np.exp(-(c[None, :] ** 2 + c[:, None] ** 2) / (2 * sigma ** 2))
    return surfaces.terrain_soa(n, n, fs, c[0], c[0], z)


@pytest.mark.parametrize("alt", [25000.0, 24000.0, 8191.7])
@pytest.mark.parametrize("platform", ["REASON_VHF", "REASON_HF"])
def test_facets_of_a_hill_straight_below(gpu_ctx, alt, platform):
    soa = hill(201, 20.0, 100.0, 30.0)
    # facets whose squared projections seen from straight above are 1e-46 to
    # 1e-24: below, among and above the denormal floats
    r2 = (alt * soa[8].astype(np.float64)) ** 2 + (alt * soa[11].astype(np.float64)) ** 2
    pick = []
    for lo in 10.0 ** np.arange(-46, -24, 0.5):
        k = np.flatnonzero((r2 >= lo) & (r2 < lo * 10 ** 0.5))
        pick += list(k[:: max(1, len(k) // 2)][:2])
    assert len(pick) > 32 and np.any((r2[pick] > 1.5e-45) & (r2[pick] < 1.17e-38))
    p = workloads.make_params(platform, "planetary_ice", nr=512, smpl=48e6, rst=alt - 300.0,
                              aperture=4.0, fs=20.0, ns=len(pick), sx0=0.0, sdx=1.0, sy=0.0, sz=alt)
    par = parse_parameters(p)
    shots = make_shots(par)
    shots["sx"], shots["sy"] = soa[0, pick], soa[1, pick]
    shots["sz"] = soa[2, pick].astype(np.float64) + alt
    e = par.to_erp()
    m = gpu_ctx.upload_mesh(soa)
    g, gv = gpu_ctx.run(e, m, None, shots)
    m.release()
    o, ov = oracle.run(e, soa, None, shots)
    np.testing.assert_array_equal(gv, ov)
    assert np.isfinite(g).all(), "shots without a number: %s" % np.flatnonzero(
        ~np.isfinite(g).all(1))
    print(compare_traces(g, o), flush=True)
