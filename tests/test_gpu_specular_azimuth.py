"""The specular method where a facet's tilt is next to nothing and gives a ray
its azimuth all the same: a shot or a target straight above or below a facet
far out on a Gaussian hill sees it along an axis whose projections on the
tangents are 1e-35 to 1e-9, with the azimuth of the tilt (atan2), which the
reradiation of the other leg turns on.  One facet is lit, so the echo of the
target is that facet's.

Compared is what the target adds to the trace.  Tolerance 1e-3 of its peak:
the traces are float32, 6e-8 of the surface's echo, at most 1e3 times the
target's here (asserted); a wrong azimuth changes the target's echo by tens of
percent."""
import numpy as np
import pytest

from europaraypaths_amd import surfaces, workloads
from europaraypaths_amd._abi import ERP_RUN_DETERMINISTIC
from europaraypaths_amd.params import make_shots, parse_parameters
from oracle import oracle

pytestmark = pytest.mark.gpu


def hill(n, fs, sigma, height):
    c = (np.arange(n) - n // 2) * fs
    z = height * np.exp(-(c[None, :] ** 2 + c[:, None] ** 2) / (2 * sigma ** 2))
    return surfaces.terrain_soa(n, n, fs, c[0], c[0], z)


def tilted(soa, exps):
    """Facets off the axes of the hill, one per power of ten of the tilt."""
    t = np.hypot(soa[8].astype(np.float64), soa[11].astype(np.float64))
    off = (np.abs(soa[0]) > 200.0) & (np.abs(soa[1]) > 300.0) & (soa[0] < 0.0)
    out = []
    for k in exps:
        i = np.flatnonzero(off & (t >= 10.0 ** k) & (t < 10.0 ** (k + 1)))
        assert len(i)
        out.append(i[len(i) // 3])
    return out


def one_facet(soa, i, below, ttype):
    """(parameters, mesh of facet i, target, shot): the other leg 14 degrees
    (below the shot) or 31 degrees (above the target) off the vertical."""
    alt, depth = 3000.0, 300.0
    p = workloads.make_params("REASON_VHF", "planetary_ice", nr=700, smpl=48e6, rst=alt - 200.0,
                              aperture=8.0, fs=20.0, ns=1, sx0=0.0, sdx=1.0, sy=0.0, sz=alt,
                              specular=True, convolution=True, convolution_linear=True,
                              rerad_funct=0)
    par = parse_parameters(p)
    shots = make_shots(par)
    c = soa[:3, i].astype(np.float64)
    o = np.array([0.0, 0.0, alt])
    t = np.zeros((6, 1), np.float32)
    t[:3, 0] = c + [0.0, 0.0, -depth]
    t[5] = 1.0
    if below == "shot":
        t[:2, 0] += np.float32([60.0, 45.0])
    else:
        o[:2] = 0.6 * alt * np.array([0.8, 0.6])
    for k, a in zip(("sx", "sy", "sz"), c + o):
        shots[k] = a
    up = o + [0.01 * alt, 0.0, 0.0]  # (a cosine rounded past 1 would leave the facet dark)
    for k, a in zip(("snx", "sny", "snz"), up / np.linalg.norm(up)):
        shots[k] = a
    shots["rst"] = np.linalg.norm(o) - 200.0
    # (a surface echo no stronger than the target's)
    shots["grefl_lin"] *= 1e-3 if ttype else 1.0
    return par.to_erp(), soa[:, [i]], (t, np.full(1, ttype, np.uint8)), shots


@pytest.mark.parametrize("flags", [0, ERP_RUN_DETERMINISTIC])
@pytest.mark.parametrize("ttype", [1, 0])
@pytest.mark.parametrize("below", ["shot", "target"])
def test_azimuth_of_a_tiny_tilt(gpu_ctx, below, ttype, flags):
    soa = hill(201, 20.0, 100.0, 30.0)
    bad = []
    for i in tilted(soa, range(-36, -8, 3)):
        e, mesh, tg, shots = one_facet(soa, i, below, ttype)
        m, t = gpu_ctx.upload_mesh(mesh), gpu_ctx.upload_targets(*tg)
        g = gpu_ctx.run(e, m, t, shots, flags=flags)[0].astype(complex)
        g = g - gpu_ctx.run(e, m, None, shots, flags=flags)[0]
        m.release()
        t.release()
        s = oracle.run(e, mesh, None, shots)[0]
        x = oracle.run(e, mesh, tg, shots)[0] - s
        peak = np.abs(x).max()
        assert peak > 1e-3 * np.abs(s).max() > 0
        err = np.abs(g - x).max() / peak
        print("tilt %.1e error %.1e" % (np.hypot(float(soa[8, i]), float(soa[11, i])), err),
              flush=True)
        bad += [i] if err > 1e-3 else []
    assert not bad
