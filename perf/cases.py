"""Performance cases: the calls a program built on this library makes, over
the sizes and options it makes them with.

listed() holds the named cases, draw() one more of the same ranges; prepare()
makes a case's inputs and buffers on the GPU, run() is one pass through the
public entry points (device pointers, queued with OPH_ASYNC where the binding
offers it), work() what a pass cannot do without and exact() its outputs in
64 bits by plain torch.

A program holds one context for its lifetime and one network per set of
weights; both are kept here for the process.  Inputs and outputs are torch
tensors whose memory is handed to the library.
"""
import math

import numpy as np
import torch

import openhologram_amd as oph
from openhologram_amd import lib, scenes

DEV = "cuda"
_KEPT = {}


def _ctx():
    if "ctx" not in _KEPT:
        _KEPT["ctx"] = oph.Context(0)
    return _KEPT["ctx"]


class _Array(lib.DeviceArray):
    """A torch tensor's memory as the array argument of a library call."""

    def __init__(self, t):
        self.t = t
        self.shape = tuple(t.shape)
        self.nbytes = t.numel() * t.element_size()
        self.ptr = t.data_ptr()

    def __del__(self):
        self.ptr = None


def _up(a):
    """A host array on the GPU."""
    return _Array(torch.from_numpy(np.ascontiguousarray(a)).to(DEV))


def _out(shape, dtype):
    return torch.zeros(shape, dtype=dtype, device=DEV)


# ---- the cases ---------------------------------------------------------------

PITCH, LAMBDA = 8e-6, 532e-9
RGB = (638e-9, 532e-9, 473e-9)
SCALE = 0.45                  # field scale a deployed correction network was trained at


def listed():
    return [
        # a small wavefront-recording-plane hologram (a preview, an icon-sized
        # object): a handful of short launches, where latency counts
        dict(name="wrp_preview", kind="wrp", n_side=256, points=500, mode=1, distance=0.02, pad=2),
        # the benchmark's WRP configuration: 100,000 points, 2048^2, 100 mm
        dict(name="wrp_100k", kind="wrp", n_side=2048, points=100_000, mode=0, distance=0.1, pad=2),
        # plain Rayleigh-Sommerfeld field, the benchmark's first configuration
        dict(name="rs_1024", kind="rs", nx=1024, ny=1024, points=1000, geometry="far", out="c64"),
        # the reference's shipped point-cloud specification: 4096 x 2160 at
        # 0.462 um, 1453 points, tilted reference wave, real fringe
        dict(name="rs_keti", kind="rs", nx=4096, ny=2160, points=1453, geometry="keti", out="fringe"),
        # reconstruction of a hologram at three depths (quality check, focus sweep)
        dict(name="refocus_1024", kind="asm", nx=1024, ny=1024, pad=2, band_limit=False),
        # the benchmark's depth-map RGB frame
        dict(name="depth_rgb_hd", kind="depth", w=1920, h=1080, Nx=4096, Ny=2048, layers=256, colors=3, lens=0.0,
             out="fringe32"),
        # an HD frame transformed unpadded with a field lens, as the
        # reference transforms its SLM grid
        dict(name="depth_lens_hd", kind="depth", w=1920, h=1080, Nx=1920, Ny=1080, layers=256, colors=1, lens=1.0,
             out="fringe32"),
        # one frame of the learned pipeline: 16-layer field, then the network
        dict(name="learned_1024", kind="learned", n=1024, layers=16, blocks=8),
        # loss and gradients of the network on a training batch
        dict(name="cnn_grad_8x128", kind="grad", batch=8, h=128, w=128, blocks=8),
        # the benchmark's Fresnel point hologram: 1e6 points on 64 planes
        dict(name="fresnel_fp16_1m", kind="fresnel", nx=4096, ny=4096, points=1_000_000, planes=64, method="fp16"),
        # the binding's default method at full single precision, a scanned
        # cloud (every point its own depth) on a panel-shaped hologram
        dict(name="fresnel_f32_cloud", kind="fresnel", nx=1280, ny=720, points=20_000, planes=0, method="valu"),
        # single-sideband encoding of a finished field for an amplitude panel
        dict(name="encode_ssb_2048", kind="encode", nx=2048, ny=2048, method="ssb", passband="left"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("wrp", "rs", "asm", "depth", "learned", "grad", "fresnel", "encode"))
    p2 = lambda lo, hi: 1 << rng.randint(lo, hi)  # noqa: E731
    if kind == "wrp":
        n = p2(8, 11)
        return dict(kind=kind, n_side=n, points=_log(rng, 200, 100_000 * (n / 2048) ** 2 + 2000), mode=rng.choice((0, 1)),
                    distance=round(rng.uniform(0.01, 0.2), 4), pad=2)
    if kind == "rs":
        nx, ny = _log(rng, 200, 4096), _log(rng, 200, 2160)
        return dict(kind=kind, nx=nx, ny=ny, points=_log(rng, 100, min(20_000, 1.3e10 / (nx * ny))),
                    geometry=rng.choice(("far", "keti")), out=rng.choice(("c64", "fringe")))
    if kind == "asm":
        pad = rng.choice((1, 2))
        return dict(kind=kind, nx=p2(8, 11), ny=p2(8, 11), pad=pad, band_limit=rng.random() < 0.5)
    if kind == "depth":
        lens = rng.choice((0.0, 1.0))
        layers = rng.choice((16, 64, 200, 256))
        colors = rng.choice((1, 3))
        out = rng.choice(("fringe32", "field"))
        if rng.random() < 0.4:
            Nx, Ny = rng.choice(((1920, 1080), (720, 540), (1080, 1920), (3840, 1080)))
            return dict(kind=kind, w=Nx, h=Ny, Nx=Nx, Ny=Ny, layers=layers, colors=colors, lens=lens, out=out)
        Nx, Ny = p2(9, 12), p2(9, 11)
        return dict(kind=kind, w=rng.randint(Nx // 3, Nx // 2), h=rng.randint(Ny // 3, Ny // 2), Nx=Nx, Ny=Ny,
                    layers=layers, colors=colors, lens=lens, out=out)
    if kind == "learned":
        return dict(kind=kind, n=p2(8, 10), layers=rng.choice((8, 16, 24)), blocks=rng.choice((4, 8)))
    if kind == "grad":
        return dict(kind=kind, batch=rng.randint(1, 12), h=rng.randint(48, 160), w=rng.randint(48, 160),
                    blocks=rng.choice((4, 8)))
    if kind == "fresnel":
        method = rng.choice(("fp16", "bf16", "fp16_split", "bf16_split", "valu"))
        nx, ny = _log(rng, 256, 4096), _log(rng, 256, 4096)
        return dict(kind=kind, nx=nx, ny=ny,
                    points=_log(rng, 1000, min(1e6, (2e11 if method == "valu" else 4e12) / (nx * ny))),
                    planes=rng.choice((0, 16, 64)), method=method)
    method = rng.choice(("ssb", "ni", "p2a", "burckhardt", "two_phase", "normalize"))
    if method == "ssb":
        return dict(kind="encode", nx=p2(8, 12), ny=p2(8, 12), method=method,
                    passband=rng.choice(("left", "right", "top", "bottom")))
    return dict(kind="encode", nx=_log(rng, 200, 4096), ny=_log(rng, 200, 4096), method=method, passband="left")


# ---- inputs (host arrays, from the seed alone) -----------------------------------

def _rs_inputs(c, seed):
    g = scenes.SplitMix64(seed)
    n = c["points"]
    if c["geometry"] == "keti":   # object coordinates; the spec scales and offsets them
        x, y, z = g.uniform(n, -0.77, 0.77), g.uniform(n, -0.77, 0.77), g.uniform(n, -0.9, 1.1)
        spec = dict(nx=c["nx"], ny=c["ny"], pitch=0.462e-6, lambda_=LAMBDA, scale=(0.05, 0.05, 0.05), offset_z=0.06,
                    tilt_deg=(22.5, 22.5))
    else:
        x, y, z = g.uniform(n, -5e-3, 5e-3), g.uniform(n, -5e-3, 5e-3), g.uniform(n, 95e-3, 105e-3)
        spec = dict(nx=c["nx"], ny=c["ny"], pitch=PITCH, lambda_=LAMBDA)
    a = g.uniform(n)
    ph = g.uniform(n, 0.0, 2 * np.pi) if c["out"] == "c64" else None
    return spec, x, y, z, a, ph


def _wrp_inputs(c, seed):
    x, y, z, a, zw = scenes.wrp_points(c["points"], seed=seed)
    s = c["n_side"] / 2048.0
    return x * s, y * s, z, a, zw


def _fresnel_inputs(c, seed):
    n = c["points"]
    if c["planes"]:
        x, y, _, z, a, ph = scenes.fresnel_points(n, planes=c["planes"], seed=seed)
    else:
        x, y, _, z, a, ph = scenes.fresnel_points(n, planes=1, seed=seed)
        z = scenes.SplitMix64(seed + (1 << 40)).uniform(n, 0.1, 0.12)
    return x, y, z, a, ph


def _field(nx, ny, seed):
    """A fully developed speckle field, complex64 on the GPU."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return torch.view_as_complex(torch.randn((ny, nx, 2), generator=g, device=DEV, dtype=torch.float32))


def _depth_inputs(c, seed):
    return scenes.depth_scene(c["w"], c["h"], seed=seed, colors=c["colors"])


def _depth_kw(c):
    """Depth range and quantisation: with the field lens the range of the
    reference's shipped configuration, requantised to the layer count."""
    near, far = (0.2, 0.7) if c["lens"] else (0.09, 0.11)
    return near, far, 1 if c["lens"] or c["layers"] != 256 else 0


def _weights(blocks):
    """A network's parameter vector at the scale training leaves it."""
    rng = np.random.default_rng(blocks)
    parts = [rng.uniform(-1, 1, 32 * 9 * 2) * math.sqrt(6 / 18), rng.normal(0, 0.02, 32)]
    for _ in range(blocks):
        for gain in (1.0, 0.2):
            parts += [rng.uniform(-1, 1, 32 * 9 * 32) * gain * math.sqrt(6 / 288), rng.normal(0, 0.02, 32)]
    parts += [rng.uniform(-1, 1, 2 * 9 * 32) * 0.2 * math.sqrt(6 / 288), rng.normal(0, 0.02, 2)]
    return np.concatenate(parts).astype(np.float32)


def _net(blocks):
    if ("net", blocks) not in _KEPT:
        net = lib.Cnn(_ctx(), blocks=blocks, channels=32, seed=1)
        net.set_params(_weights(blocks))
        _KEPT["net", blocks] = net
    return _KEPT["net", blocks]


def _grad_inputs(c, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    x = torch.randn((c["batch"], c["h"], c["w"], 2), generator=g, device=DEV)
    return x, x + 0.2 * torch.randn(x.shape, generator=g, device=DEV)


# ---- prepare and run -----------------------------------------------------------------

def prepare(case, seed):
    c = dict(case)
    ctx, kind = _ctx(), c["kind"]
    s = {"c": c, "ctx": ctx}
    if kind == "rs":
        spec, *pts = _rs_inputs(c, seed)
        s["spec"] = lib.make_spec(**spec)
        s["pts"] = [None if a is None else _up(a) for a in pts]
        s["fmt"] = lib.OUT_C64 if c["out"] == "c64" else lib.OUT_FRINGE
        s["out"] = _out((c["ny"], c["nx"]), torch.complex64 if c["out"] == "c64" else torch.float32)
    elif kind == "wrp":
        *pts, s["zw"] = _wrp_inputs(c, seed)
        s["pts"] = [_up(a) for a in pts]
        s["out"] = _out((c["n_side"], c["n_side"]), torch.complex64)
    elif kind == "fresnel":
        s["pts"] = [_up(a) for a in _fresnel_inputs(c, seed)]
        s["out"] = _out((c["ny"], c["nx"]), torch.complex64)
    elif kind == "asm":
        s["field"] = _Array(_field(c["nx"], c["ny"], seed))
        s["out"] = [_Array(_out((c["ny"], c["nx"]), torch.complex64)) for _ in range(3)]
    elif kind in ("depth", "learned"):
        if kind == "learned":
            c.update(w=c["n"], h=c["n"], Nx=2 * c["n"], Ny=2 * c["n"], colors=1, lens=0.0, out="field")
            s["net"] = _net(c["blocks"])
            s["y"] = _out((1, c["n"], c["n"], 2), torch.float32)
        s["img"], s["dep"] = (_up(a) for a in _depth_inputs(c, seed))
        s["lam"] = np.array(RGB if c["colors"] == 3 else (LAMBDA,))
        s["out"] = _out((c["colors"], c["h"], c["w"]), torch.complex64 if c["out"] == "field" else torch.float32)
    elif kind == "grad":
        s["net"] = _net(c["blocks"])
        s["x"], s["t"] = (_Array(a) for a in _grad_inputs(c, seed))
    else:
        f = _field(c["nx"], c["ny"], seed)
        if c["method"] == "normalize":
            f = f.real.contiguous()
            s["out"] = _Array(_out((c["ny"], c["nx"]), torch.uint8))
        else:
            k = {"burckhardt": 3, "two_phase": 2}.get(c["method"], 1)
            s["out"] = _out((c["ny"], k * c["nx"]), torch.float32)
        s["field"] = _Array(f)
    return s


def run(s):
    c, ctx = s["c"], s["ctx"]
    kind, out = c["kind"], s.get("out")
    if kind == "rs":
        ctx.pc_rs(s["spec"], *s["pts"], out=out.data_ptr(), fmt=s["fmt"], device=True, asynchronous=True)
        return out
    if kind == "wrp":
        ctx.wrp_hologram(c["n_side"], PITCH, LAMBDA, s["zw"], c["distance"], *s["pts"], pad=c["pad"], mode=c["mode"],
                         out=out.data_ptr(), device=True, asynchronous=True)
        return out
    if kind == "fresnel":
        ctx.fresnel(c["nx"], c["ny"], PITCH, LAMBDA, *s["pts"], method=c["method"], out=out.data_ptr(), device=True,
                    asynchronous=True)
        return out
    if kind == "asm":
        # the hologram is kept; each depth propagates a copy of it
        for o, z in zip(out, _depths()):
            ctx.copy(o, s["field"])
            ctx.asm(o, PITCH, LAMBDA, z, pad=c["pad"], band_limit=c["band_limit"], device=True, asynchronous=True)
        return [o.t for o in out]
    if kind in ("depth", "learned"):
        near, far, qm = _depth_kw(c)
        rho = (1.0 / SCALE, 0.0) if kind == "learned" else (1.0, 0.0)
        ctx.depthmap(c["w"], c["h"], c["Nx"], c["Ny"], PITCH, near, far, c["layers"], s["lam"], s["img"], s["dep"],
                     out=c["out"], quant_mode=qm, field_lens=c["lens"], rho=rho, device=True, asynchronous=True,
                     dst=out.data_ptr())
        if kind == "depth":
            return out
        s["net"].forward(out.data_ptr(), out=s["y"].data_ptr(), device=True, shape=(1, c["n"], c["n"], 2),
                         bf16_acts=True)
        return [out, s["y"]]
    if kind == "grad":
        loss, g = s["net"].gradients(s["x"], s["t"], device=True)
        return {"loss": loss, "grad": g}
    if c["method"] == "normalize":
        ctx.normalize_u8(s["field"], device=True, dst=out)
        return out.t
    ctx.encode_field(s["field"], c["method"], passband=c["passband"], device=True, out=out.data_ptr(),
                     asynchronous=True)
    return out


def _depths():
    """The quartiles of the depth range."""
    return (0.095, 0.1, 0.105)


# ---- work ------------------------------------------------------------------------------

def _fft_flops(nx, ny):
    return 5.0 * nx * ny * math.log2(nx * ny)


def work(case):
    c = dict(case)
    kind = c["kind"]
    if kind in ("rs", "fresnel"):
        pix, n = c["nx"] * c["ny"], c["points"]
        # one complex multiply-add per point and pixel
        return {"bytes": 40.0 * n + pix * (4 if c.get("out") == "fringe" else 8), "flops": 8.0 * pix * n}
    if kind == "wrp":
        n = c["n_side"]
        half = 30.0 if c["mode"] else 15.0      # mean window half-width over 1-6 mm
        return {"bytes": 32.0 * c["points"] + 8.0 * n * n,
                "flops": 8.0 * c["points"] * (2 * half) ** 2 + 2 * _fft_flops(2 * n, 2 * n)}
    if kind == "asm":
        n = c["nx"] * c["ny"]
        return {"bytes": 8.0 * n * 4, "flops": 6 * _fft_flops(c["nx"] * c["pad"], c["ny"] * c["pad"])}
    if kind in ("depth", "learned"):
        if kind == "learned":
            c.update(w=c["n"], h=c["n"], Nx=2 * c["n"], Ny=2 * c["n"], colors=1, lens=0.0)
        pix, grid = c["w"] * c["h"], c["Nx"] * c["Ny"]
        b = pix * (1.0 + c["colors"] * (1 + (8 if c.get("out", "field") == "field" else 4)))
        # a real transform and one complex multiply-add per layer, one inverse
        f = c["colors"] * (c["layers"] * (0.5 * _fft_flops(c["Nx"], c["Ny"]) + 8.0 * grid) + _fft_flops(c["Nx"], c["Ny"]))
        if kind == "learned":
            b += 8.0 * pix
            f += _conv_flops(c["blocks"]) * pix
        return {"bytes": b, "flops": f}
    if kind == "grad":
        pix = c["batch"] * c["h"] * c["w"]
        return {"bytes": 16.0 * pix + 4.0 * _weights(c["blocks"]).size, "flops": 3.0 * _conv_flops(c["blocks"]) * pix}
    pix = c["nx"] * c["ny"]
    if c["method"] == "normalize":
        return {"bytes": 5.0 * pix, "flops": 3.0 * pix}
    k = {"burckhardt": 3, "two_phase": 2}.get(c["method"], 1)
    f = 2 * 5.0 * pix * math.log2(c["nx"] if c["passband"] in ("left", "right") else c["ny"]) if c["method"] == "ssb" \
        else 20.0 * pix
    return {"bytes": pix * (8.0 + 4.0 * k), "flops": f}


def _conv_flops(blocks):
    """Per pixel."""
    return 2.0 * 9 * (2 * 32 + 2 * blocks * 32 * 32 + 32 * 2)


# ---- 64-bit values ------------------------------------------------------------------------

def _t(a):
    return torch.from_numpy(np.ascontiguousarray(a, np.float64)).to(DEV)


def _turn(t):
    """exp(2 pi i t)"""
    t = (t - torch.round(t)) * (2 * math.pi)
    return torch.complex(torch.cos(t), torch.sin(t))


def exact(case, seed):
    c = dict(case)
    with torch.no_grad():
        if c["kind"] == "rs":
            return _exact_rs(c, seed)
        if c["kind"] == "wrp":
            return _exact_wrp(c, seed)
        if c["kind"] == "fresnel":
            return _exact_fresnel(c, seed)
        if c["kind"] == "asm":
            u = _field(c["nx"], c["ny"], seed).to(torch.complex128)
            return [_asm(u, z, c["pad"], c["band_limit"]) for z in _depths()]
        if c["kind"] == "depth":
            return _exact_depth(c, seed, 1.0)
        if c["kind"] == "learned":
            c.update(w=c["n"], h=c["n"], Nx=2 * c["n"], Ny=2 * c["n"], colors=1, lens=0.0, out="field")
            u = _exact_depth(c, seed, 1.0 / SCALE)
            x = torch.view_as_real(u)
            return [u, _net64(x, torch.from_numpy(_weights(c["blocks"])).to(DEV).double(), c["blocks"])]
        if c["kind"] == "encode":
            return _exact_encode(c, seed)
    x, t = (a.double() for a in _grad_inputs(c, seed))
    p = torch.from_numpy(_weights(c["blocks"])).to(DEV).double().requires_grad_(True)
    loss = (_net64(x, p, c["blocks"]) - t).square().mean()
    loss.backward()
    return {"loss": float(loss), "grad": p.grad}


def _exact_rs(c, seed):
    spec, x, y, z, a, ph = _rs_inputs(c, seed)
    sc, nx, ny, p = spec.get("scale", (1, 1, 1)), c["nx"], c["ny"], spec["pitch"]
    X = (torch.arange(nx, device=DEV, dtype=torch.float64) + 0.5) * p - nx * p / 2
    Y = ny * p / 2 - (torch.arange(ny, device=DEV, dtype=torch.float64) + 0.5) * p
    dx2 = (X[None] - _t(x)[:, None] * sc[0]).square()          # points x columns
    dy2 = (Y[None] - _t(y)[:, None] * sc[1]).square()          # points x rows
    z2 = (_t(z) * sc[2] + spec.get("offset_z", 0.0)).square()
    t0 = _t(ph) / (2 * math.pi) if ph is not None else torch.zeros(c["points"], device=DEV, dtype=torch.float64)
    re = torch.zeros((ny, nx), device=DEV, dtype=torch.float64)
    im = torch.zeros_like(re)
    rows = max(1, (1 << 27) // nx)
    for n in range(c["points"]):
        for r in range(0, ny, rows):
            t = ((dy2[n, r:r + rows, None] + (dx2[n] + z2[n])[None]).sqrt_()).mul_(1.0 / LAMBDA).add_(t0[n])
            t.sub_(torch.round(t)).mul_(2 * math.pi)
            re[r:r + rows].add_(torch.cos(t), alpha=float(a[n]))
            im[r:r + rows].add_(torch.sin(t), alpha=float(a[n]))
    u = torch.complex(re, im)
    tilt = spec.get("tilt_deg", (0.0, 0.0))
    if tilt[0] or tilt[1]:
        sx, sy = math.sin(math.radians(tilt[0])), math.sin(math.radians(tilt[1]))
        u = u * _turn(-(X[None] * sx + Y[:, None] * sy) / LAMBDA)
    return u.real.contiguous() if c["out"] == "fringe" else u


def _exact_wrp(c, seed):
    x, y, z, a, zw = _wrp_inputs(c, seed)
    n, mode = c["n_side"], c["mode"]
    dz = zw - z
    tx, ty = (np.trunc(v / PITCH).astype(np.int64) + n // 2 for v in (x, y))
    if mode == 0:
        w = np.trunc(np.abs(dz) * math.tan(math.asin(LAMBDA / (2 * PITCH))) / PITCH).astype(np.int64)
    else:
        w = np.trunc(np.abs(LAMBDA * dz / PITCH / PITCH / 2 + 0.5)).astype(np.int64) * 2 - 1
    re = torch.zeros(n * n, device=DEV, dtype=torch.float64)
    im = torch.zeros_like(re)
    order = np.argsort(w, kind="stable")
    for lo in range(0, len(w), 2048):
        i = order[lo:lo + 2048]
        m = int(w[i].max())
        o = torch.arange(-m, m, device=DEV)
        wi, di, ai = torch.from_numpy(w[i]).to(DEV), _t(dz[i]), _t(a[i])
        col, row = torch.from_numpy(tx[i]).to(DEV)[:, None] + o, torch.from_numpy(ty[i]).to(DEV)[:, None] + o
        inx = (o >= -wi[:, None]) & (o < wi[:, None]) & (col >= 0) & (col < n)
        iny = (o >= -wi[:, None]) & (o < wi[:, None]) & (row >= 0) & (row < n)
        o2 = (o.double() * PITCH).square()
        keep = iny[:, :, None] & inx[:, None, :]
        at = (row[:, :, None] * n + col[:, None, :])[keep]
        r = torch.sign(di)[:, None, None] * (o2[None, :, None] + o2[None, None, :] + di.square()[:, None, None]).sqrt()
        v = _turn(r / LAMBDA) * (ai[:, None, None] / (r + 0.05))
        re.index_add_(0, at, v.real[keep])
        im.index_add_(0, at, v.imag[keep])
    return _asm(torch.complex(re, im).reshape(n, n), c["distance"], c["pad"], False)


def _exact_fresnel(c, seed):
    x, y, z, a, ph = (_t(v) for v in _fresnel_inputs(c, seed))
    X = (torch.arange(c["nx"], device=DEV, dtype=torch.float64) - c["nx"] // 2) * PITCH
    Y = (torch.arange(c["ny"], device=DEV, dtype=torch.float64) - c["ny"] // 2) * PITCH
    u = torch.zeros((c["ny"], c["nx"]), device=DEV, dtype=torch.complex128)
    step = 8192
    for lo in range(0, c["points"], step):
        k = slice(lo, lo + step)
        h = 1.0 / (2 * LAMBDA * z[k])
        w = _turn(z[k] / LAMBDA + ph[k] / (2 * math.pi)) * a[k]
        A = _turn((Y[:, None] - y[k][None]).square() * h[None]) * w[None]
        B = _turn((X[None, :] - x[k][:, None]).square() * h[:, None])
        u += A @ B
    return u


def _asm(u, z, pad, band):
    ny, nx = u.shape
    Nx, Ny = nx * pad, ny * pad
    ox, oy = Nx // 2 - nx // 2, Ny // 2 - ny // 2
    g = torch.zeros((Ny, Nx), device=DEV, dtype=torch.complex128)
    g[oy:oy + ny, ox:ox + nx] = u
    fx = torch.fft.fftfreq(Nx, PITCH, dtype=torch.float64, device=DEV)[None]
    fy = torch.fft.fftfreq(Ny, PITCH, dtype=torch.float64, device=DEV)[:, None]
    s = 1.0 / LAMBDA ** 2 - fx.square() - fy.square()
    H = _turn(z * s.clamp_min(0.0).sqrt()) * (s > 0)
    if band:
        # both axes' local frequency within the grid's sampling limit
        bx = fx.abs() * z * LAMBDA / (Nx * PITCH * 0.5)
        by = fy.abs() * z * LAMBDA / (Ny * PITCH * 0.5)
        q = 1.0 - LAMBDA ** 2 * (fx.square() + fy.square())
        H = H * ((bx.square() <= q) & (by.square() <= q))
    return torch.fft.ifft2(torch.fft.fft2(g) * H)[oy:oy + ny, ox:ox + nx].contiguous()


def _depth_index(dep, near, far, L, qm):
    d = dep.astype(np.int64)
    if qm == 0:
        return 256 - d
    lev = np.cumsum(np.concatenate([[near], np.full(L - 1, (far - near) / (L - 1))]))
    half = (far - near) / (L - 1) / 2.0
    dm = (1 - np.arange(256) / 255.0) * (far - near) + near
    table = np.zeros(256, np.int64)
    for i in range(L):
        table += ((dm >= lev[i] - half) & ((dm < lev[i] + half) if i < L - 1 else (dm <= lev[i] + half))) * (i + 1)
    return table[d]


def _exact_depth(c, seed, rho):
    img, dep = _depth_inputs(c, seed)
    near, far, qm = _depth_kw(c)
    w, h, Nx, Ny, L, f = c["w"], c["h"], c["Nx"], c["Ny"], c["layers"], c["lens"]
    idx = torch.from_numpy(_depth_index(dep, near, far, L, qm)).to(DEV)
    lev = np.cumsum(np.concatenate([[near], np.full(L - 1, (far - near) / (L - 1))]))
    zs = -f * lev / (lev - f) if f > 0 else lev
    sx = torch.fft.fftfreq(Nx, 1.0 / Nx, dtype=torch.float64, device=DEV)[None] / (PITCH * Nx)
    sy = (torch.fft.fftfreq(Ny, 1.0 / Ny, dtype=torch.float64, device=DEV)[:, None] + 1) / (PITCH * Ny)
    ox, oy = (Nx - w) // 2, (Ny - h) // 2
    ky = (torch.arange(Ny, device=DEV) + Ny // 2) % Ny
    lo = Ny // 2 - Ny // 4 - 1
    kept = ((ky >= lo) & (ky <= lo + Ny // 2 - 1))[:, None]
    # turns of the symmetrisation shift, per row
    shift = _turn(h / 8.0 - (torch.arange(h, device=DEV, dtype=torch.float64) + 1) / 4.0)[:, None]
    present = torch.unique(idx).tolist()
    out = []
    for k, lam in enumerate(RGB if c["colors"] == 3 else (LAMBDA,)):
        u2 = lam ** 2 * (sx.square() + sy.square())
        phi = u2 / (1.0 + (1.0 - u2).clamp_min(0.0).sqrt()) / lam     # (1 - sqrt(1 - u)) / lambda
        v = torch.from_numpy(img[k]).to(DEV).double() / 255.0
        A = torch.zeros((Ny, Nx), device=DEV, dtype=torch.complex128)
        g = torch.zeros((Ny, Nx), device=DEV, dtype=torch.float64)
        for l in present:
            if 1 <= l <= L:
                g[oy:oy + h, ox:ox + w] = v * (idx == l)
                A += torch.fft.fft2(g) * _turn(phi * float(zs[l - 1]))
        if c["out"] != "field":
            A = A * kept
        r = torch.fft.ifft2(A)[oy:oy + h, ox:ox + w] * rho
        out.append((r * shift).real if c["out"] != "field" else r)
    return torch.stack(out)


def _conv64(x, w, b):
    """3x3 convolution, NHWC, w [out][9][in]"""
    B, H, W, _ = x.shape
    xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
    y = b.expand(B, H, W, b.numel())
    for t in range(9):
        y = y + xp[:, t // 3:t // 3 + H, t % 3:t % 3 + W] @ w[:, t].transpose(0, 1).contiguous()
    return y


def _net64(x, p, blocks):
    at = 0

    def take(*shape):
        nonlocal at
        n = math.prod(shape)
        at += n
        return p[at - n:at].reshape(shape)
    h = _conv64(x, take(32, 9, 2), take(32))
    for _ in range(blocks):
        a = torch.relu(_conv64(h, take(32, 9, 32), take(32)))
        h = h + _conv64(a, take(32, 9, 32), take(32))
    return x + _conv64(h, take(2, 9, 32), take(2))


def _exact_encode(c, seed):
    if c["method"] == "normalize":
        return None
    u = _field(c["nx"], c["ny"], seed).to(torch.complex128)
    m = c["method"]
    if m == "ssb":
        A = torch.fft.fftshift(torch.fft.fft2(u))
        nx, ny = c["nx"], c["ny"]
        if c["passband"] == "left":
            A[:, nx // 2 - 1:] = 0
        elif c["passband"] == "right":
            A[:, :nx // 2] = 0
        elif c["passband"] == "top":
            A[ny // 2 - 1:] = 0
        else:
            A[:ny // 2] = 0
        r = torch.fft.ifft2(torch.fft.ifftshift(A)).real
        r = r - r.min()
        return r / r.max()
    big = u.abs().max()
    if m == "ni":
        i = (u + big).abs().square()
        return i / i.max()
    if m == "p2a":
        return u.angle() + 0.5
    am, ph = u.abs() / big, u.angle() + math.pi
    if m == "two_phase":
        d = torch.arccos(am.clamp_max(1.0))
        return torch.stack([ph + d, ph - d], -1).reshape(c["ny"], -1)
    third = 2 * math.pi / 3
    out = torch.zeros((c["ny"], c["nx"], 3), device=DEV, dtype=torch.float64)
    for k in range(3):
        q = ph - k * third
        here = (q >= 0) & (q < third)
        out[..., k] += torch.where(here, am * (torch.cos(q) + torch.sin(q) / math.sqrt(3)), 0.0)
        out[..., (k + 1) % 3] += torch.where(here, 2 * torch.sin(q) / math.sqrt(3), 0.0)
    return out.reshape(c["ny"], -1)
