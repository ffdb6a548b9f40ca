"""Performance cases: what users of the backend have it do, through the Python mirror of its C-ABI
(sirius_amd.accelerator.HipAccelerator).

  listed()           the named cases
  draw(rng)          one more case of the same ranges
  prepare(case, s)   what a program holds before the call: cameras and spacetimes made from the
                     seed, device result arrays, network weights, frames to encode
  run(state)         one pass, and its outputs
  work(case)         bytes and operations the pass cannot do without
  exact(case, s)     the outputs in 64 bits by plain torch, where they have such a value

Scenes follow the repository's own workloads: the Kerr a = 0.9 thin-disk view (r = 50 M, 75
degrees, 20 degree field of view, 16 spectral bins), the batch of random Kerr-Newman-de Sitter
spacetimes with volumetric emission (8 bins), the Ellis wormhole and the Alcubierre bubble seen
from r = 10, and the far-field network. A seed varies spin, inclination, distance and azimuth a
little, so every seed is another frame of about the same cost.
"""
import math
import random

import numpy as np
import torch

from sirius_amd import abi
from sirius_amd.accelerator import HipAccelerator, default_opts, starfield_default

DEV = "cuda:0"
FORMATS = {"ppm": abi.IMAGE_PPM, "ppm_srgb": abi.IMAGE_PPM_SRGB, "pfm": abi.IMAGE_PFM}


# ---- the cases --------------------------------------------------------------------------------
def listed():
    return [
        # an interactive preview: the smallest frame, results on the host
        dict(name="preview_kerr_fp32", kind="trace", spacetime="kerr", precision="fp32", emission="disk",
             integrator="dp45", width=96, height=54, cameras=1, bins=16, to="host"),
        # the headline frame, results in device arrays that the program post-processes there
        dict(name="frame_1080p_kerr_fp32", kind="trace", spacetime="kerr", precision="fp32", emission="disk",
             integrator="dp45", width=1920, height=1080, cameras=1, bins=16, to="device"),
        # the reference-contract frame in plain FP64 (audits, ground truth), odd sizes
        dict(name="frame_721p_kerr_fp64", kind="trace", spacetime="kerr", precision="fp64", emission="disk",
             integrator="dp45", width=1283, height=721, cameras=1, bins=16, to="device"),
        # a batch of cameras, each in its own spacetime, with radiative transfer along the rays
        dict(name="batch_volumetric_fp32", kind="trace", spacetime="knds", precision="fp32", emission="volumetric",
             integrator="dp45", width=256, height=256, cameras=6, bins=8, to="device"),
        # the warp bubble: FP32 with its wall crossers re-traced in FP64
        dict(name="warp_fp32", kind="trace", spacetime="warp", precision="fp32", emission="none",
             integrator="dp45", width=1024, height=1024, cameras=1, bins=0, to="device"),
        # long fixed-step integrations that conserve the constants of motion
        dict(name="symplectic_kerr_fp64", kind="trace", spacetime="kerr", precision="fp64", emission="disk",
             integrator="symplectic", width=320, height=181, cameras=1, bins=16, to="device"),
        # a rendered wormhole: two star catalogues, framebuffer to the host
        dict(name="launch_wormhole_stars", kind="launch", spacetime="wormhole", width=1024, height=1024, samples=1),
        # a final-quality frame: 2 x 2 samples per pixel, background image, framebuffer to the host
        dict(name="launch_kerr_4spp", kind="launch", spacetime="kerr", width=1280, height=720, samples=4),
        # each pixel's ray bundle (lens-map Jacobians and beams) on the host
        dict(name="bundle_kerr", kind="bundle", spacetime="kerr", width=641, height=361),
        # the far-field network: inference over a frame's candidates, and one training batch
        # (loss and every parameter's gradient)
        dict(name="network_forward", kind="forward", rows=600001),
        dict(name="network_loss_grad", kind="grad", rows=8192),
        # a frame in device memory encoded for disk (the renderer's default format; the compressed
        # formats' time is zlib's on the host)
        dict(name="image_ppm_1080p", kind="image", format="ppm", width=1920, height=1080),
    ]


def draw(rng):
    def side(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["fp32", "fp32", "fp64", "vol", "sky", "sym", "warp", "wormhole", "launch", "bundle", "forward",
                       "grad", "image"])
    t = dict(kind="trace", spacetime="kerr", precision="fp32", emission="disk", integrator="dp45", cameras=1, bins=16,
             to=rng.choice(["host", "device"]))
    if kind == "fp32":
        w = side(64, 1920)
        return dict(t, width=w, height=max(36, w * 9 // 16), bins=rng.choice([4, 8, 16]), to="device" if w > 1000 else t["to"])
    if kind == "fp64":
        return dict(t, precision="fp64", width=side(64, 1283), height=side(36, 721))
    if kind == "vol":
        s = side(48, 256)
        return dict(t, spacetime="knds", emission="volumetric", bins=rng.choice([4, 8]), width=s, height=s,
                    cameras=rng.randint(1, 6), to="device")
    if kind == "sky":  # the Kerr view without its disk: shadow and sky directions
        return dict(t, precision=rng.choice(["fp32", "fp64"]), emission="none", bins=0, width=side(64, 511), height=side(64, 383))
    if kind == "sym":
        return dict(t, precision="fp64", integrator="symplectic", width=side(64, 320), height=side(36, 181))
    if kind in ("warp", "wormhole"):
        s = side(96, 1024)
        return dict(t, spacetime=kind, emission="none", bins=0, width=s, height=s, precision=rng.choice(["fp32", "fp32", "fp64"]),
                    to="device")
    if kind == "launch":
        w = side(160, 1280)
        return dict(kind="launch", spacetime="kerr", width=w, height=w * 9 // 16, samples=rng.choice([1, 4]))
    if kind == "bundle":
        return dict(kind="bundle", spacetime="kerr", width=side(64, 641), height=side(36, 361))
    if kind == "forward":
        return dict(kind="forward", rows=side(64, 600000))
    if kind == "grad":
        return dict(kind="grad", rows=side(256, 8192))
    w = side(256, 1920)
    return dict(kind="image", format=rng.choice(list(FORMATS)), width=w, height=w * 9 // 16)


# ---- scenes -----------------------------------------------------------------------------------
def scene(case, seed):
    """(cameras, metrics) as dicts of plain numbers, from the seed alone."""
    r = random.Random(1000003 * int(seed) + 17)
    cams, metrics = [], []
    for i in range(case.get("cameras", 1)):
        s = case["spacetime"]
        c = dict(width=case["width"], height=case["height"], phi_deg=r.uniform(0.0, 360.0), yaw=0.0, metric_index=i)
        m = dict(family=s, a=0.0, Q=0.0, Lambda=0.0)
        if s == "kerr":
            m["a"] = r.uniform(0.88, 0.92)
            c.update(r_obs=r.uniform(48.0, 52.0), incl_deg=r.uniform(74.0, 76.0), fov_deg=20.0)
        elif s == "knds":
            m["a"] = r.uniform(0.0, 0.99)
            m["Q"] = r.uniform(0.0, 0.5 * math.sqrt(1.0 - m["a"] ** 2))
            m["Lambda"] = r.uniform(0.0, 1e-4)
            c.update(r_obs=r.uniform(20.0, 100.0), incl_deg=r.uniform(5.0, 89.0), fov_deg=30.0)
        elif s == "wormhole":
            m["b0"] = r.uniform(0.95, 1.05)
            c.update(r_obs=r.uniform(9.5, 10.5), incl_deg=r.uniform(85.0, 89.0), fov_deg=60.0, yaw=r.uniform(0.01, 0.05))
        else:
            m.update(v=r.uniform(0.48, 0.52), R=r.uniform(0.95, 1.05), sigma=8.0)
            c.update(r_obs=r.uniform(9.5, 10.5), incl_deg=r.uniform(58.0, 62.0), fov_deg=40.0)
        cams.append(c)
        metrics.append(m)
    return cams, metrics


def abi_scene(case, seed):
    cams, metrics = scene(case, seed)
    ac = [abi.camera(c["r_obs"], c["incl_deg"], c["fov_deg"], c["width"], c["height"], disk=(0.0, 30.0),
                     metric_index=c["metric_index"], phi_deg=c["phi_deg"], yaw=c["yaw"]) for c in cams]
    am = []
    for m in metrics:
        if m["family"] == "wormhole":
            am.append(abi.metric_mt(m["b0"]))
        elif m["family"] == "warp":
            am.append(abi.metric_warp(m["v"], m["R"], m["sigma"]))
        else:
            am.append(abi.metric_ks(1.0, m["a"], m["Q"], m["Lambda"]))
    return ac, am


def options(case):
    o = default_opts(abi.PRECISION_FP64 if case.get("precision") == "fp64" else abi.PRECISION_FP32_ESCALATE)
    o.emission = {"none": abi.EMISSION_NONE, "disk": abi.EMISSION_THIN_DISK,
                  "volumetric": abi.EMISSION_VOLUMETRIC}[case.get("emission", "disk")]
    if case.get("integrator") == "symplectic":
        o.integrator = abi.INTEGRATOR_SYMPLECTIC
        o.symplectic_h = 0.02
        o.r_escape = R_SYMPLECTIC
    o.n_bins = case.get("bins", 16)
    return o


# A fixed step of 0.02 M would take 50,000 steps to the adaptive integrator's escape radius of 1000 M;
# beyond 100 M a ray's direction has settled to 1e-4 rad.
R_SYMPLECTIC = 100.0

_ACC = {}


def accelerator(case):
    """A program keeps one accelerator for all its frames of one size, its sky installed once."""
    key = (case["kind"], case.get("spacetime"), case.get("width"), case.get("height"), case.get("samples"))
    acc = _ACC.get(key)
    if acc is None:
        acc = _ACC[key] = HipAccelerator()
        if case["kind"] == "launch":
            acc.initialise(case["width"], case["height"])
            acc.set_shading(samples_per_pixel=case["samples"])
            if case["spacetime"] == "wormhole":
                for s in (0, 1):
                    acc.set_starfield(s, starfield_default(), stars(4096, 20 + s))
            else:
                g = np.random.default_rng(3)
                acc.uploadBackground(g.integers(0, 256, (512, 1024, 4), dtype=np.uint8))
    return acc


def stars(n, seed):
    """A sphere of n stars: uniform directions, magnitudes ~ Exp(1)."""
    g = np.random.default_rng(seed)
    z, ph = g.uniform(-1, 1, n), g.uniform(0, 2 * np.pi, n)
    mag, dist, bv = g.exponential(1.0, n), g.uniform(10, 1000, n), g.uniform(-0.3, 1.7, n)
    temp = np.clip(np.where(bv > -0.1, 4600 / (0.92 + np.maximum(bv, -0.1)), 30000 + 10000 * (-bv - 0.1)), 2500, 50000)
    rho = np.sqrt(1 - z * z)
    out = (abi.Star * n)()
    for i in range(n):
        out[i].dir[0], out[i].dir[1], out[i].dir[2] = rho[i] * np.cos(ph[i]), rho[i] * np.sin(ph[i]), z[i]
        out[i].distance_pc, out[i].magnitude, out[i].color_bv, out[i].temperature_K = dist[i], mag[i], bv[i], temp[i]
    return out


# ---- the network's weights and batches ----------------------------------------------------------
def network(seed):
    """FP32 parameters, layer by layer W (out x in) then b: 5 -> 4 x 256 -> 6."""
    g = torch.Generator().manual_seed(int(seed))
    layers = []
    for i, o in ((5, 256), (256, 256), (256, 256), (256, 256), (256, 6)):
        lim = math.sqrt(6.0 / i)
        layers.append(((torch.rand(o, i, generator=g) * 2 - 1) * lim, (torch.rand(o, generator=g) * 2 - 1) * 0.1))
    return layers


def network_rows(case, seed):
    """Rays of random cameras: the network's inputs, and a training batch's targets."""
    n = case["rows"]
    g = torch.Generator(device=DEV).manual_seed(int(seed) + 1)
    u = torch.rand(n, 5, generator=g, device=DEV)
    x = torch.stack([0.99 * u[:, 0], u[:, 1], 2 * u[:, 2] - 1, 2.4 * u[:, 3] - 1.2, 2.4 * u[:, 4] - 1.2], 1).contiguous()
    cls = (torch.rand(n, generator=g, device=DEV) * 3).to(torch.int32).clamp(max=2)
    dirs = torch.randn(n, 3, generator=g, device=DEV) * 0.5
    return x, cls, dirs


# ---- prepare and run ------------------------------------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    st = dict(kind=kind, case=case)
    if kind in ("trace", "launch", "bundle"):
        st["acc"] = accelerator(case)
        st["cams"], st["metrics"] = abi_scene(case, seed)
        st["opts"] = options(case)
        if case.get("to") == "device":
            n, b = case["cameras"] * case["width"] * case["height"], max(case["bins"], 1)
            f = lambda *shape: torch.zeros(*shape, device=DEV)  # noqa: E731
            out = dict(cls=torch.zeros(n, dtype=torch.uint8, device=DEV), theta=f(n), phi=f(n), lam=f(n), disk_r=f(n),
                       redshift=f(n), intensity=f(b, n))
            st["arrays"] = out
            st["out"] = abi.RayOutput(cls=out["cls"].data_ptr(), theta=out["theta"].data_ptr(), phi=out["phi"].data_ptr(),
                                      lambda_=out["lam"].data_ptr(), disk_r=out["disk_r"].data_ptr(),
                                      redshift=out["redshift"].data_ptr(), intensity=out["intensity"].data_ptr(), on_device=1)
            torch.cuda.synchronize()
    elif kind in ("forward", "grad"):
        st["acc"] = HipAccelerator()
        st["acc"].mlp_set_params(torch.cat([t.reshape(-1) for l in network(seed) for t in l]).numpy())
        st["x"], st["cls"], st["dirs"] = network_rows(case, seed)
        st["y"] = torch.zeros(case["rows"], 6, device=DEV)
        st["g"] = torch.zeros(st["acc"].mlp_param_count(), device=DEV)
        torch.cuda.synchronize()
    else:
        st["acc"] = accelerator(case)
        st["frame"] = frame(case, seed)
        torch.cuda.synchronize()
    return st


def frame(case, seed):
    """A rendered frame in device memory: a smooth disk, sharp stars, black sky, alpha 1."""
    w, h = case["width"], case["height"]
    g = torch.Generator(device=DEV).manual_seed(int(seed) + 2)
    y, x = torch.meshgrid(torch.linspace(-1, 1, h, device=DEV), torch.linspace(-1.8, 1.8, w, device=DEV), indexing="ij")
    r = torch.sqrt(x * x + 9 * y * y) + 0.02 * torch.rand(1, generator=g, device=DEV)
    disk = torch.exp(-4 * (r - 0.9) ** 2) * (1 + 0.8 * x / (r + 0.1)) * (r > 0.35)
    col = torch.tensor([1.0, 0.72, 0.45], device=DEV)
    rgb = 3 * disk[..., None] * col + 0.002 * torch.rand(h, w, 3, generator=g, device=DEV) * (disk[..., None] > 0.01)
    sky = torch.rand(h, w, generator=g, device=DEV)
    rgb += ((sky > 0.9995).float() * sky * 5)[..., None]
    return torch.cat([rgb, torch.ones(h, w, 1, device=DEV)], 2).contiguous()


def run(st):
    kind, acc = st["kind"], st["acc"]
    if kind == "trace":
        if "out" in st:
            acc.trace_batch(st["cams"], st["metrics"], st["opts"], device_out=st["out"])
            return st["arrays"]
        rays, _ = acc.trace_batch(st["cams"], st["metrics"], st["opts"])
        return dict(cls=rays.cls, theta=rays.theta, phi=rays.phi, lam=rays.lam, disk_r=rays.disk_r, redshift=rays.redshift,
                    intensity=rays.intensity)
    if kind == "launch":
        acc.launch(st["cams"][0], st["metrics"][0], st["opts"])
        return acc.getFrameBuffer()
    if kind == "bundle":
        out = acc.trace_bundle(st["cams"], st["metrics"], st["opts"])
        return dict(cls=out["cls"], jac=out["jac"], beam=out["beam"])
    if kind == "forward":
        acc.mlp_forward(st["x"].data_ptr(), st["y"].data_ptr(), st["case"]["rows"])
        return st["y"]
    if kind == "grad":
        loss = acc.mlp_loss_grad(st["x"].data_ptr(), st["cls"].data_ptr(), st["dirs"].data_ptr(), st["case"]["rows"],
                                 st["g"].data_ptr())
        return dict(loss=loss, grad=st["g"])
    data, _ = acc.encode_image(FORMATS[st["case"]["format"]], rgba=st["frame"])
    return np.frombuffer(data, np.uint8)


# ---- work ---------------------------------------------------------------------------------------
# Step attempts per ray of the default tolerances on these scenes, and operations per attempt (six
# right-hand sides and the Dormand-Prince sums; for the symplectic integrator per step).
ATTEMPTS = {("kerr", "disk", "fp32"): 14.3, ("kerr", "disk", "fp64"): 57, ("kerr", "none", "fp32"): 22,
            ("kerr", "none", "fp64"): 400, ("knds", "volumetric", "fp32"): 95, ("warp", "none", "fp32"): 30,
            ("warp", "none", "fp64"): 520, ("wormhole", "none", "fp32"): 28, ("wormhole", "none", "fp64"): 520}
FLOPS = {"kerr": 1326.0, "knds": 1326.0, "warp": 678.0, "wormhole": 576.0}


def work(case):
    kind = case["kind"]
    if kind == "trace":
        n = case["cameras"] * case["width"] * case["height"]
        per = 1 + 5 * 4 + 4 * case["bins"]
        if case["integrator"] == "symplectic":
            return dict(bytes=n * per, flops=n * 2500 * 2184.0)
        return dict(bytes=n * per, flops=n * ATTEMPTS[case["spacetime"], case["emission"], case["precision"]] * FLOPS[case["spacetime"]])
    if kind == "launch":
        n = case["width"] * case["height"]
        em = "disk" if case["spacetime"] == "kerr" else "none"
        return dict(bytes=16 * n, flops=n * case["samples"] * ATTEMPTS[case["spacetime"], em, "fp32"] * FLOPS[case["spacetime"]])
    if kind == "bundle":
        n = case["width"] * case["height"]
        return dict(bytes=n * (1 + 16 + 12), flops=n * 14.3 * 3 * 1326.0)
    if kind == "forward":
        return dict(bytes=case["rows"] * 44 + 200454 * 4, flops=case["rows"] * 398848.0)
    if kind == "grad":
        return dict(bytes=case["rows"] * 36 + 2 * 200454 * 4, flops=case["rows"] * 3 * 398848.0)
    return dict(bytes=case["width"] * case["height"] * 19, flops=0)


# ---- the same in 64 bits --------------------------------------------------------------------------
def exact(case, seed):
    kind = case["kind"]
    if kind == "trace":
        return exact_trace(case, seed)
    if kind in ("forward", "grad"):
        return exact_network(case, seed)
    # Framebuffers are display colours (samplers of 8-bit textures and point-like stars, a colour
    # chain defined in 32 bits), image files are bytes, and a bundle's Jacobian is the derivative of
    # the traced steps themselves: none has a value apart from its definition.
    return None


def exact_network(case, seed):
    x, cls, dirs = network_rows(case, seed)
    x, dirs, cls = x.double(), dirs.double(), cls.long()
    P = [t.to(DEV).double().requires_grad_(case["kind"] == "grad") for l in network(seed) for t in l]

    def net(h):
        for i in range(5):
            h = h @ P[2 * i].T + P[2 * i + 1]
            if i < 4:
                h = torch.nn.functional.gelu(h, approximate="tanh")
        return h

    if case["kind"] == "forward":
        with torch.no_grad():
            return torch.cat([net(c) for c in x.split(65536)])
    y = net(x)
    loss = torch.nn.functional.cross_entropy(y[:, :3], cls) + \
        100.0 * (((y[:, 3:] - dirs) ** 2).sum(1) * (cls == 0)).sum() / len(x)
    g = torch.autograd.grad(loss, P)
    return dict(loss=float(loss), grad=torch.cat([t.reshape(-1) for t in g]))


class Geodesics:
    """Null geodesics of H = g^{mu nu} p_mu p_nu / 2 by Dormand-Prince 5(4) at a tight tolerance; the
    state of n rays is (6, n): position and spatial momentum; p_t is constant. Each ray has its own
    spacetime: the rows of P are a, Q^2, Lambda (Kerr-Newman-de Sitter in Kerr-Schild form), b0
    (wormhole), or v, R, sigma (warp bubble)."""

    A = ((1 / 5,), (3 / 40, 9 / 40), (44 / 45, -56 / 15, 32 / 9), (19372 / 6561, -25360 / 2187, 64448 / 6561, -212 / 729),
         (9017 / 3168, -355 / 33, 46732 / 5247, 49 / 176, -5103 / 18656), (35 / 384, 0, 500 / 1113, 125 / 192, -2187 / 6784, 11 / 84))
    E = (71 / 57600, 0, -71 / 16695, 71 / 1920, -17253 / 339200, 22 / 525, -1 / 40)

    def __init__(self, family, lam=False):
        self.f, self.lam = family, lam
        self.hole = family in ("kerr", "knds")

    def parameters(self, m, n):
        row = {"wormhole": ("b0",), "warp": ("v", "R", "sigma")}.get(self.f)
        v = [m[k] for k in row] if row else [m["a"], m["Q"] ** 2, m["Lambda"]]
        return torch.tensor(v, dtype=torch.float64, device=DEV)[:, None].expand(len(v), n)

    def radius(self, y, P):
        if self.f == "wormhole":
            return y[0].abs()
        R2 = y[0] * y[0] + y[1] * y[1] + y[2] * y[2]
        if not self.hole:
            return R2.sqrt()
        a2 = P[0] * P[0]
        w = R2 - a2
        return (0.5 * (w + (w * w + 4 * a2 * y[2] * y[2]).sqrt())).sqrt()

    def null_vector(self, y, P):
        """(H, l_x, l_y, l_z) of the Kerr-Schild form g = eta + H l l, l_t = 1."""
        r, a = self.radius(y, P), P[0]
        d = r * r + a * a
        return ((2 * r - P[1]) * r * r / (r ** 4 + a * a * y[2] ** 2), (r * y[0] + a * y[1]) / d,
                (r * y[1] - a * y[0]) / d, y[2] / r)

    def shape(self, rs, P):
        """The warp bubble's shape function and its derivative."""
        _, R, s = P
        n = 2 * torch.tanh(s * R)
        u, w = torch.tanh(s * (rs + R)), torch.tanh(s * (rs - R))
        return (u - w) / n, s * (w * w - u * u) / n

    def rhs(self, y, pt, P):
        x, z, px, py, pz = y[0], y[2], y[3], y[4], y[5]
        if self.f == "wormhole":
            r2 = x * x + P[0] * P[0]
            o = torch.zeros_like(x)
            return torch.stack([px, py / r2, o, x * (py / r2) ** 2, o, o])
        if self.f == "warp":
            rs = (y[:3] * y[:3]).sum(0).sqrt()
            f, df = self.shape(rs, P)
            u = pt + P[0] * f * px  # H = (-(p_t + v f p_x)^2 + p^2) / 2
            return torch.cat([torch.stack([px - u * P[0] * f, py, pz]), u * px * P[0] * df / rs * y[:3]])
        Y, a, Q2, L = y[1], P[0], P[1], P[2]
        a2 = a * a
        R2 = x * x + Y * Y + z * z
        w = R2 - a2
        s = (w * w + 4 * a2 * z * z).sqrt()
        r2 = 0.5 * (w + s)
        r = r2.sqrt()
        d, D = r2 + a2, r2 * r2 + a2 * z * z
        h = (2 * r - Q2) * r2 / D
        h_r, h_z = (6 * r2 - 2 * Q2 * r - 4 * h * r2 * r) / D, -2 * a2 * z * h / D
        u1, u2 = px * x + py * Y, a * (px * Y - py * x)
        lp = -pt + (r * u1 + u2) / d + pz * z / r  # l^mu p_mu, and its derivatives
        lp_r = (u1 - 2 * r * (r * u1 + u2) / d) / d - pz * z / r2
        dr = torch.stack([x * r / s, Y * r / s, z * d / (r * s)])
        dlp = lp_r * dr + torch.stack([(r * px - a * py) / d, (r * py + a * px) / d, pz / r])
        dh = h_r * dr
        dh[2] += h_z
        l = torch.stack([(r * x + a * Y) / d, (r * Y - a * x) / d, z / r])
        k = y[3:] - h * lp * l
        f = 0.5 * lp * lp * dh + h * lp * dlp
        if self.lam:  # g^{-1} of g + c e_t e_t, c = -Lambda R^2 / 3: H - c K^2 / (2 N)
            c, K = -L / 3 * R2, -pt + h * lp
            N = 1 - c * (1 + h)
            dc = -2 * L / 3 * y[:3]
            dK, dN = dh * lp + h * dlp, -dc * (1 + h) - c * dh
            k = k - c * K / N * h * l
            f = f + 0.5 * ((dc * K * K + 2 * c * K * dK) / N - c * K * K / (N * N) * dN)
        return torch.cat([k, f])

    def metric(self, x, P):
        """Covariant g at one position (tensor (3,)), as a 4 x 4 tensor; P one column."""
        g = torch.diag(torch.tensor([-1.0, 1, 1, 1], dtype=torch.float64, device=DEV))
        if self.f == "warp":
            vf = P[0, 0] * self.shape((x * x).sum().sqrt(), P[:, 0])[0]
            g[0, 0] += vf * vf
            g[0, 1] = g[1, 0] = -vf
        elif self.hole:
            h, lx, ly, lz = self.null_vector(x[:, None], P)
            l = torch.stack([torch.ones_like(lx), lx, ly, lz])[:, 0]
            g += h * l[:, None] * l
            g[0, 0] -= P[2, 0] / 3 * (x * x).sum()
        return g

    def step(self, y, pt, P, k1, h):
        k = [k1]
        for row in self.A:
            s = None
            for c, q in zip(row, k):
                if c:
                    s = c * q if s is None else s.add_(q, alpha=c)
            y1 = torch.addcmul(y, s, h)
            k.append(self.rhs(y1, pt, P))
        e = None
        for c, q in zip(self.E, k):
            if c:
                e = c * q[:3] if e is None else e.add_(q[:3], alpha=c)
        return y1, k[6], h * e


def hermite(y0, k0, y1, k1, h, t):
    a = t * t * (3 - 2 * t)
    return (1 - a) * y0 + a * y1 + h * t * (1 - t) * ((1 - t) * k0 - t * k1)


def rays_of(c, m, geo):
    """Start states (6, n), p_t and parameters of a camera's pixel centres, u_obs^t, and the camera's frame
    (e_r, e_theta, e_phi and each ray's components on it)."""
    t = lambda v: torch.tensor(v, dtype=torch.float64, device=DEV)  # noqa: E731
    th, ph = math.radians(c["incl_deg"]), math.radians(c["phi_deg"])
    er = t([math.sin(th) * math.cos(ph), math.sin(th) * math.sin(ph), math.cos(th)])
    et = t([math.cos(th) * math.cos(ph), math.cos(th) * math.sin(ph), -math.sin(th)])
    ep = t([-math.sin(ph), math.cos(ph), 0.0])
    v, u = torch.meshgrid(torch.arange(c["height"], dtype=torch.float64, device=DEV) + 0.5,
                          torch.arange(c["width"], dtype=torch.float64, device=DEV) + 0.5, indexing="ij")
    half = math.tan(math.radians(c["fov_deg"]) / 2)
    dx = (2 * u.reshape(-1) / c["width"] - 1) * c["width"] / c["height"] * half
    dy = (1 - 2 * v.reshape(-1) / c["height"]) * half
    dz = -torch.ones_like(dx)
    cy, sy = math.cos(c["yaw"]), math.sin(c["yaw"])
    dx, dz = dx * cy + dz * sy, -dx * sy + dz * cy
    n = torch.stack([dz, -dy, dx]) / (dx * dx + dy * dy + dz * dz).sqrt()  # (r, theta, phi) components
    P = geo.parameters(m, len(dx))
    if geo.f == "wormhole":
        z = torch.zeros_like(dx)
        nt = (n[1] ** 2 + n[2] ** 2).sqrt()
        l0, r = math.sqrt(c["r_obs"] ** 2 - m["b0"] ** 2), c["r_obs"]
        return torch.stack([z + l0, z, z, n[0], nt * r, z]), z - 1, P, 1.0, (er, et, ep, n)
    x = c["r_obs"] * er
    d = n[0] * er[:, None] + n[1] * et[:, None] + n[2] * ep[:, None]
    g = geo.metric(x, P[:, :1])
    A, B, C = g[0, 0], 2 * (g[0, 1:, None] * d).sum(0), (d * (g[1:, 1:] @ d)).sum(0)
    sq = (B * B - 4 * A * C).sqrt()
    kp, km = (-B + sq) / (2 * A), (-B - sq) / (2 * A)
    k0 = torch.where(kp > 0, kp, km)
    p = g @ torch.cat([k0[None], d])
    return torch.cat([x[:, None].expand(3, len(dx)), p[1:]]), p[0], P, 1 / math.sqrt(-float(g[0, 0])), (er, et, ep, n)


def isco(a):
    z1 = 1 + (1 - a * a) ** (1 / 3) * ((1 + a) ** (1 / 3) + (1 - a) ** (1 / 3))
    z2 = math.sqrt(3 * a * a + z1 * z1)
    return 3 + z2 - math.sqrt((3 - z1) * (3 + z1 + 2 * z2))


def page_thorne(a, r):
    """Page & Thorne (1974) f(r) of the thin disk, closed form."""
    x, x0, ac = r.sqrt(), math.sqrt(isco(a)), math.acos(a)
    X = [2 * math.cos((ac - math.pi) / 3), 2 * math.cos((ac + math.pi) / 3), -2 * math.cos(ac / 3)]
    s = x - x0 - 1.5 * a * (x / x0).log()
    for i in range(3):
        b, c, d = X[i], X[(i + 1) % 3], X[(i + 2) % 3]
        s = s - 3 * (b - a) ** 2 / (b * (b - c) * (b - d)) * ((x - b) / (x0 - b)).log()
    return 1.5 / (x * x * (x ** 3 - 3 * x + 2 * a)) * s


def emitter(geo, y, P, rc):
    """u^t and angular velocity of the circular emitter below each position."""
    sq = (rc - P[1]).clamp(min=0).sqrt()
    om = sq / (rc * rc + P[0] * sq)
    h, lx, ly, _ = geo.null_vector(y, P)
    lv = 1 + om * (-lx * y[1] + ly * y[0])
    vv = -1 + om * om * (y[0] ** 2 + y[1] ** 2) + h * lv * lv - P[2] / 3 * (y[:3] ** 2).sum(0)
    return torch.where(vv < 0, 1 / (-vv).clamp(min=1e-300).sqrt(), -torch.ones_like(vv)), om


def transfer(geo, y0, k0, y1, k1, h, pt, P, xk, acc, tau):
    """Radiative transfer along a step: three Gauss-Legendre nodes on its Hermite interpolant; the rows
    of P after the spacetime's are the shell's inner radius and u_obs^t."""
    r_lo, norm = P[-2], P[-1]
    for t, w in ((0.5 - math.sqrt(0.15), 5 / 18), (0.5, 8 / 18), (0.5 + math.sqrt(0.15), 5 / 18)):
        q = hermite(y0, k0, y1, k1, h, t)
        r = geo.radius(q, P)
        u, v = ((r - r_lo) / (0.1 * r_lo)).clamp(0, 1), ((50 - r) / 5.0).clamp(0, 1)
        win = u ** 3 * (u * (6 * u - 15) + 10) * v ** 3 * (v * (6 * v - 15) + 10)
        ut, om = emitter(geo, q, P, (q[0] ** 2 + q[1] ** 2 - P[0] * P[0]).clamp(min=1e-12).sqrt())
        ne, no = -ut * (pt + om * (q[0] * q[4] - q[1] * q[3])), -pt * norm
        rho = torch.where((ut > 0) & (ne > 0), torch.exp(-50 * (q[2] / r) ** 2) * win / (r * r), torch.zeros_like(r))
        ne = ne.clamp(min=1e-12)
        dt = 0.3 * rho * ne * w * h
        wt = rho * no ** 3 / ne ** 2 * w * h * torch.exp(-(tau + 0.5 * dt))
        xe = xk[:, None] * ne / no
        acc = acc + wt * xe ** 3 / torch.expm1((xe / (6 / r) ** 0.75).clamp(max=600))
        tau = tau + dt
    return acc, tau


def exact_trace(case, seed):
    """Every output array of a trace, each ray landed on its event."""
    cams, metrics = scene(case, seed)
    geo = Geodesics(case["spacetime"], any(m["Lambda"] for m in metrics))
    thin, vol, nb = case["emission"] == "disk", case["emission"] == "volumetric", max(case["bins"], 1)
    r_esc = R_SYMPLECTIC if case["integrator"] == "symplectic" else 1000.0
    parts = []
    for c in cams:
        m = metrics[c["metric_index"]]
        y, pt, P, norm, frame = rays_of(c, m, geo)
        r_in = isco(m["a"]) if geo.hole else 0.0
        r_cap = 1.01 * (1 + math.sqrt(1 - m["a"] ** 2 - m["Q"] ** 2)) if geo.hole else -1.0
        more = torch.tensor([r_in, r_cap, max(r_in, 2.0), norm], dtype=torch.float64, device=DEV)[:, None]
        parts.append((y, pt, torch.cat([P, more.expand(4, len(pt))])))
    y, pt, P = (torch.cat([p[i] for p in parts], -1) for i in range(3))
    n = len(pt)
    zero = torch.zeros(n, dtype=torch.float64, device=DEV)
    out = dict(theta=zero.clone(), phi=zero.clone(), lam=zero.clone(), disk_r=zero.clone(), redshift=zero.clone(),
               intensity=zero.repeat(nb, 1))
    xk = torch.tensor([0.1 * 100 ** ((k + 0.5) / nb) for k in range(nb)], dtype=torch.float64, device=DEV)
    f_max = 0.0
    if thin:
        a = metrics[0]["a"]
        s = torch.linspace(isco(a), 30.0, 200001, dtype=torch.float64, device=DEV)[1:]
        f_max = float((page_thorne(a, s) / s).max())
    ids = torch.arange(n, device=DEV)
    lam, h, k1 = zero.clone(), zero + 0.01, geo.rhs(y, pt, P[:-4])
    acc, tau = out["intensity"].clone() if vol else zero[None, :], zero.clone()
    for _ in range(3000):
        if not len(ids):
            break
        S = P[:-4]
        r0 = geo.radius(y, S)
        h = torch.minimum(h, 0.2 * r0 + 0.05)
        if vol:  # short steps inside the emitting layer (scale height r / 10)
            cap = torch.maximum(0.5 * (y[2].abs() - 0.3 * r0), 0.02 * r0)
            h = torch.where((r0 > 1) & (r0 < 75), torch.minimum(h, cap), h)
        y1, k7, err = geo.step(y, pt, S, k1, h)
        e = err.abs().amax(0) / (1e-11 * (1 + r0))
        ok = e <= 1
        r1 = geo.radius(y1, S)
        ends = torch.zeros(len(ids), dtype=torch.int64, device=DEV)
        if thin:
            i = torch.nonzero(ok & (y[2] * y1[2] < 0))[:, 0]
            if len(i):
                t = root(lambda q: q[2], y[:, i], k1[:, i], y1[:, i], k7[:, i], h[i])
                rc = geo.radius(hermite(y[:, i], k1[:, i], y1[:, i], k7[:, i], h[i], t), S[:, i])
                ends[i[(rc >= P[-4, i]) & (rc <= 30.0)]] = 2
        radial = y1[0] * k7[0] if geo.f == "wormhole" else (y1[:3] * k7[:3]).sum(0)
        ends = torch.where((ends == 0) & ok & (r1 < P[-3]), torch.ones_like(ends), ends)
        ends = torch.where((ends == 0) & ok & (r1 > r_esc) & (radial > 0), torch.full_like(ends, 3), ends)
        if vol:
            acc1, tau1 = transfer(geo, y, k1, y1, k7, h, pt, P, xk, acc, tau)
            acc, tau = torch.where(ok, acc1, acc), torch.where(ok, tau1, tau)
            ends = torch.where((ends == 0) & (tau > 10), torch.full_like(ends, 4), ends)
        done = torch.nonzero(ends)[:, 0]
        if len(done):
            if vol:
                out["intensity"][:, ids[done]] = acc[:, done]
            land(geo, out, ids[done], ends[done], y[:, done], pt[done], P[:, done], k1[:, done], h[done], y1[:, done],
                 k7[:, done], lam[done], r_esc, frame, xk, metrics[0]["a"], f_max)
        lam = torch.where(ok, lam + h, lam)
        h = h * (0.9 * e.clamp(min=1e-12) ** -0.2).clamp(0.2, 3)
        y, k1 = torch.where(ok, y1, y), torch.where(ok, k7, k1)
        if len(done):
            keep = torch.nonzero(ends == 0)[:, 0]
            ids, y, k1, pt, P, h, lam, tau = ids[keep], y[:, keep], k1[:, keep], pt[keep], P[:, keep], h[keep], lam[keep], tau[keep]
            acc = acc[:, keep] if vol else acc
    if case["to"] == "host":
        out = {k: v.cpu().numpy() for k, v in out.items()}
        out["intensity"] = out["intensity"][:case["bins"]]
    out["cls"] = None
    if vol:
        # a ray that ends inside the opaque layer ends with its step: no value apart from the steps
        out["lam"] = out["redshift"] = out["disk_r"] = None
    if case["integrator"] == "symplectic":
        out["lam"] = None  # an escaping ray ends with its step
    return out


def root(value, y, k1, y1, k7, h):
    """Fraction of each step where value() of its Hermite interpolant changes sign, by bisection."""
    f0 = value(y)
    a, b = torch.zeros_like(h), torch.ones_like(h)
    for _ in range(45):
        t = 0.5 * (a + b)
        same = value(hermite(y, k1, y1, k7, h, t)) * f0 > 0
        a, b = torch.where(same, t, a), torch.where(same, b, t)
    return t


def land(geo, out, ids, ends, y, pt, P, k1, h, y1, k7, lam, r_esc, frame, xk, a, f_max):
    """Lands each finished ray on its event (root on the step, then Newton with whole steps) and
    writes its outputs."""
    S, plane = P[:-4], ends == 2
    target = torch.where(ends == 1, P[-3], torch.full_like(h, r_esc))
    value = lambda q: torch.where(plane, q[2], geo.radius(q, S) - target)  # noqa: E731
    inside = plane | (value(y) * value(y1) < 0)
    t = torch.where(inside, root(value, y, k1, y1, k7, h), torch.ones_like(h))
    for _ in range(3):
        q, kq, _e = geo.step(y, pt, S, k1, t * h)
        rate = torch.where(plane, kq[2], (geo.radius(q + 1e-6 * kq, S) - geo.radius(q - 1e-6 * kq, S)) / 2e-6)
        t = torch.where(inside, t - value(q) / (rate * h), t)
    q, kq, _e = geo.step(y, pt, S, k1, t * h)
    out["lam"][ids] = lam + t * h
    esc = torch.nonzero(ends == 3)[:, 0]
    if len(esc):
        i, d = ids[esc], kq[:3, esc]
        if geo.f == "wormhole":  # from the orbital plane back to the exit side's sky
            er, et, ep, ns = frame
            e2 = (ns[1][i] * et[:, None] + ns[2][i] * ep[:, None]) / (ns[1][i] ** 2 + ns[2][i] ** 2).sqrt()
            l, psi = q[0, esc], q[1, esc]
            r = (l * l + P[0, esc] ** 2).sqrt()
            dr, dt = l / r * d[0], q[4, esc] / r
            d = dr * (psi.cos() * er[:, None] + psi.sin() * e2) + dt * (-psi.sin() * er[:, None] + psi.cos() * e2)
        out["theta"][i] = torch.acos((d[2] / d.pow(2).sum(0).sqrt()).clamp(-1, 1))
        out["phi"][i] = torch.atan2(d[1], d[0])
    hit = torch.nonzero(plane)[:, 0]
    if len(hit):
        i, s = ids[hit], q[:, hit]
        r = geo.radius(s, S[:, hit])
        ut, om = emitter(geo, s, S[:, hit], r)
        g = pt[hit] * P[-1, hit] / (ut * (pt[hit] + om * (s[0] * s[4] - s[1] * s[3])))
        tau = (page_thorne(a, r) / r / f_max).clamp(min=0) ** 0.25
        x = xk[:, None] / (g * tau).clamp(min=1e-300)
        out["disk_r"][i], out["redshift"][i] = r, g
        if len(xk) > 1:
            out["intensity"][:, i] = torch.where(tau > 0, xk[:, None] ** 3 / torch.expm1(x.clamp(max=600)), torch.zeros_like(x))
