"""Star light of wide, overlapping stars against the walk of the whole catalogue: launch (from the spheres'
cell index where a catalogue has one) against sirius_hip_sample_starfield at the same escape directions.
The direction's rounding may differ by a unit in the last place, 6e-8 of a cosine: a star's spread of
sigma then differs by 6e-8 / sigma^2, up to three of its terms, below 1e-4 for the sigmas here (0.03 rad and
more), and a star at its 1e-6 cut may come or go. Cuts of 0.16, 0.24 and 0.32 rad (indexed) and 0.84 rad (walked),
uniform, about the poles and about the phi = +-pi seam."""
import numpy as np
import pytest

from sirius_amd import abi
from sirius_amd.accelerator import default_opts, starfield_default

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("place", ["uniform", "poles", "seam"])
@pytest.mark.parametrize("aperture", [30.0, 45.0, 60.0, 160.0])
@pytest.mark.parametrize("n", [3, 400, 4096])
def test_wide_stars(acc, n, aperture, place):
    g = np.random.default_rng(5)
    z, ph = g.uniform(-1, 1, n), g.uniform(-np.pi, np.pi, n)
    if place == "poles":
        z = np.where(np.arange(n) % 2, 1, -1) * np.sqrt(1 - g.uniform(0, 0.3, n) ** 2)
        z[0] = -1.0
    if place == "seam":
        ph = np.pi + g.uniform(-0.05, 0.05, n)
        ph[0] = np.pi
    rho = np.sqrt(np.maximum(0, 1 - z * z))
    dirs = np.stack([rho * np.cos(ph), rho * np.sin(ph), z], 1)
    stars, cfg = (abi.Star * n)(), starfield_default()
    cfg.aperture_mm = aperture
    for i in range(n):
        stars[i].dir[0], stars[i].dir[1], stars[i].dir[2] = dirs[i]
        stars[i].distance_pc, stars[i].magnitude, stars[i].color_bv, stars[i].temperature_K = 1.0, 0.25 * (i % 8), 0.5, 6000.0
    w, h = 121, 77
    cam, m = abi.camera(10.0, 60.0, 150.0, w, h), abi.metric_mt(0.5)
    try:
        acc.set_starfield(0, cfg, stars, n)
        acc.set_starfield(1, cfg, stars, n)
        acc.initialise(w, h)
        light = 0.0
        for phi in (0.0, 180.0):
            for theta in (90.0, 10.0, 170.0):
                cam.phi_obs, cam.theta_obs = np.deg2rad(phi), np.deg2rad(theta)
                print(f"[case] wide stars {n} aperture {aperture} {place} phi {phi} theta {theta}", flush=True)
                acc.launch(cam, m, default_opts(abi.PRECISION_FP32_ESCALATE))
                fb = acc.getFrameBuffer().reshape(-1, 4)[:, :3]
                rays = acc.fetch_results()
                esc = rays.cls == abi.RAY_ESCAPED
                want = np.zeros_like(fb)
                want[esc] = acc.sample_starfield(0, rays.direction()[esc].astype(np.float32))
                assert np.all(np.abs(fb - want) <= 1e-4 * want + 4e-6 * cfg.brightness_scale)
                assert (np.abs(fb - want) <= 1e-6 * want + 1e-30).all(1).mean() > 0.99
                light += want.sum()
        assert light > 0
    finally:
        acc.set_starfield(0, None, None, 0)
        acc.set_starfield(1, None, None, 0)
