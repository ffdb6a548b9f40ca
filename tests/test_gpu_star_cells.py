"""The star index of a celestial sphere against the walk of the whole catalogue: launch's star light
(which looks at the stars of a direction's cell only) equals sirius_hip_sample_starfield (which
tests every star) at the same escape directions. Both add the same stars in the same order with the
same float steps; only the direction's rounding differs (launch forms it in FP64 from the ray's
angles, as the host does here), so pixels are equal except where one ulp of a direction changes the
spread of a star they lie in: 99.9 % equal to 1e-6 relative, and the frame's sum to 1e-3.
Catalogues: point-like stars, stars at the poles and on the phi = +-pi seam, wide spreads (a
quarter of the sky), one star, and one whose index would be too large (walked)."""
import numpy as np
import pytest

from sirius_amd import abi
from sirius_amd.accelerator import default_opts, starfield_default

pytestmark = pytest.mark.gpu


def _stars(dirs, dist, mag):
    out = (abi.Star * len(dirs))()
    for i, (d, r) in enumerate(zip(dirs, dist)):
        out[i].dir[0], out[i].dir[1], out[i].dir[2] = d
        out[i].distance_pc, out[i].magnitude, out[i].color_bv, out[i].temperature_K = r, mag[i], 0.5, 6000.0
    return out


def _catalogue(kind):
    g = np.random.default_rng(11)
    c = starfield_default()
    n = {"one": 1, "too_many": 30000}.get(kind, 4096)
    z, ph = g.uniform(-1, 1, n), g.uniform(0, 2 * np.pi, n)
    if kind == "poles":
        z = np.where(np.arange(n) % 2, 1, -1) * np.sqrt(1 - g.uniform(0, 0.05, n) ** 2)
        z[:2] = (1.0, -1.0)
    if kind == "seam":
        ph = np.pi + g.uniform(-0.01, 0.01, n)
        ph[0] = np.pi
    if kind == "one":
        z, ph = np.array([0.3]), np.array([2.0])
    rho = np.sqrt(np.maximum(0, 1 - z * z))
    dist = g.uniform(10, 1000, n)
    if kind in ("wide", "too_many", "one"):
        c.aperture_mm = 300.0
        dist = np.full(n, 1.0) if kind != "one" else np.array([2.0])  # spread 0.3 rad: cut at 1.6 rad
    return c, _stars(np.stack([rho * np.cos(ph), rho * np.sin(ph), z], 1), dist, g.exponential(1.0, n)), n


@pytest.mark.parametrize("kind", ["points", "poles", "seam", "wide", "one", "too_many"])
def test_cell_index_equals_the_whole_catalogue(acc, kind):
    cfg, stars, n = _catalogue(kind)
    w, h = 161, 97
    cam = abi.camera(10.0, 60.0, 150.0, w, h, phi_deg=17.0)  # a wide view of a nearly flat sky
    m = abi.metric_mt(0.5)
    try:
        acc.set_starfield(0, cfg, stars, n)
        acc.set_starfield(1, cfg, stars, n)
        acc.initialise(w, h)
        for phi in (17.0, 197.0):
            cam.phi_obs = np.deg2rad(phi)
            for theta in (60.0, 10.0, 170.0):
                cam.theta_obs = np.deg2rad(theta)
                print(f"[case] star cells {kind} phi {phi} theta {theta}", flush=True)
                acc.launch(cam, m, default_opts(abi.PRECISION_FP32_ESCALATE))
                fb = acc.getFrameBuffer().reshape(-1, 4)[:, :3]
                rays = acc.fetch_results()
                esc = rays.cls == abi.RAY_ESCAPED
                want = np.zeros_like(fb)
                want[esc] = acc.sample_starfield(0, rays.direction()[esc].astype(np.float32))
                near = np.abs(fb - want) <= 1e-6 * np.abs(want) + 1e-30
                assert near.all(1).mean() > 0.999
                assert abs(fb.sum() - want.sum()) <= 1e-3 * want.sum() + 1e-30
        assert want.max() > 0 or kind in ("poles", "seam", "one", "points")
    finally:
        acc.set_starfield(0, None, None, 0)
        acc.set_starfield(1, None, None, 0)
