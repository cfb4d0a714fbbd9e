"""The work this framework's users have it do, as cases that can be timed and checked.

A case is a dict of plain values; `kind` names the entry point:

  asm       AsmProp of one field, in place (complex64 or complex128, either direction)
  fresnel   FresnelProp of one field, loaded into the working field before the call
  grad      asm_prop of a stack of fields: forward, and backward through autograd
  plane     one step of multi-plane hologram design: loss and phase gradient
  cgh       Cgh of a point cloud (Fresnel or exact spherical r)
  wrp       WRPStep1 of a cloud, then ARSS to the hologram plane
  layered   CghLayered of a cloud (f16, bf16 or split-bf16 factors)

Lengths are in metres.  `exact` restates each operator in 64 bits with torch alone.
"""
import math

import torch

import openol_amd as ol
from openol_amd import autograd

LAM = 532e-9


def listed():
    return [
        # a small tile of a larger optical simulation: three launches, bound by latency
        dict(name="asm_256", kind="asm", ny=256, nx=256, pitch=8e-6, z=0.02, c128=False,
             bandlimit=True, adjoint=False),
        # a full-HD spatial light modulator's field, back-propagated to the object
        dict(name="asm_1080x1920", kind="asm", ny=1080, nx=1920, pitch=8e-6, z=0.1, c128=False,
             bandlimit=True, adjoint=True),
        # the Fresnel demo's field: a 4K modulator
        dict(name="fresnel_2160x3840", kind="fresnel", ny=2160, nx=3840, pitch=3.74e-6, z=0.1,
             c128=False),
        # the headline propagation
        dict(name="asm_4096", kind="asm", ny=4096, nx=4096, pitch=8e-6, z=0.1, c128=False,
             bandlimit=True, adjoint=False),
        # the plain configuration in double precision
        dict(name="asm_c128_1024", kind="asm", ny=1024, nx=1024, pitch=8e-6, z=0.1, c128=True,
             bandlimit=True, adjoint=False),
        # a training step's propagation layer: four frames forward and backward
        dict(name="grad_4x1024", kind="grad", nb=4, ny=1024, nx=1024, pitch=8e-6, z=0.1),
        # one design step of a three-plane phase-only hologram
        dict(name="plane_3x2048", kind="plane", n=2048, planes=3, pitch=8e-6, z=0.1),
        # the direct CGH configuration: spherical waves from 10,000 points
        dict(name="cgh_exact_2048", kind="cgh", n=10000, ny=2048, nx=2048, pitch=8e-6,
             exact_r=True),
        # a scanned object's point count (the larger cloud of the tests) into a full-HD hologram
        dict(name="cgh_fresnel_1080x1920", kind="cgh", n=5197, ny=1080, nx=1920, pitch=8e-6,
             exact_r=False),
        # the wavefront-recording-plane pipeline
        dict(name="wrp_arss_4096", kind="wrp", n=200000, ny=4096, nx=4096, pitch=8e-6),
        # the layered pipeline at its default precision: a million points, 64 layers
        dict(name="layered_f16_4096", kind="layered", n=1000000, layers=64, ny=4096, nx=4096,
             pitch=8e-6, precision="f16"),
        # a layered hologram for a 4K modulator where f16's error is too large
        dict(name="layered_bf16x3_2160x3840", kind="layered", n=200000, layers=32, ny=2160,
             nx=3840, pitch=8e-6, precision="bf16x3"),
    ]


# ---------------------------------------------------------------- drawn cases
def _sides(lo, hi):
    """Sides whose padded lengths factor into 2, 3, 5, 7, 11 and 13."""
    out = []
    for n in range(lo, hi + 1):
        r = n
        for p in (2, 3, 5, 7, 11, 13):
            while r % p == 0:
                r //= p
        if r == 1:
            out.append(n)
    return out


_SIDES = _sides(64, 4096)


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _side(rng, lo=64, hi=4096):
    """A supported side, uniform in its logarithm; a power of two one time in three."""
    t = _log(rng, lo, hi)
    if rng.random() < 1 / 3:
        n = 2 ** round(math.log2(t))
        return min(max(n, lo), hi)
    return min((s for s in _SIDES if lo <= s <= hi), key=lambda s: abs(s - t))


def draw(rng):
    kind = rng.choice(["asm", "asm", "fresnel", "grad", "plane", "cgh", "cgh", "wrp", "layered"])
    pitch = rng.choice([3.74e-6, 6.4e-6, 8e-6])
    if kind in ("asm", "fresnel"):
        c128 = rng.random() < 0.25
        hi = 2048 if c128 else 4096
        c = dict(kind=kind, ny=_side(rng, 64, hi), nx=_side(rng, 64, hi), pitch=pitch,
                 z=_log(rng, 0.02, 0.3), c128=c128)
        if kind == "asm":
            c.update(bandlimit=rng.random() < 0.7, adjoint=rng.random() < 0.3)
        return c
    if kind == "grad":
        return dict(kind=kind, nb=rng.randint(1, 8), ny=_side(rng, 128, 1024),
                    nx=_side(rng, 128, 1024), pitch=pitch, z=_log(rng, 0.02, 0.2))
    if kind == "plane":
        return dict(kind=kind, n=_side(rng, 128, 2048), planes=rng.randint(1, 4), pitch=8e-6,
                    z=_log(rng, 0.05, 0.2))
    if kind == "cgh":
        return dict(kind=kind, n=round(_log(rng, 284, 20000)), ny=round(_log(rng, 200, 2160)),
                    nx=round(_log(rng, 200, 2160)), pitch=pitch, exact_r=rng.random() < 0.5)
    if kind == "wrp":
        return dict(kind=kind, n=round(_log(rng, 1000, 200000)), ny=_side(rng, 256, 4096),
                    nx=_side(rng, 256, 4096), pitch=8e-6)
    precision = rng.choice(["f16", "f16", "bf16", "bf16x3"])
    return dict(kind=kind, n=round(_log(rng, 10000, 1e6 if precision != "bf16x3" else 3e5)),
                layers=rng.choice([16, 32, 64, 100]), ny=round(_log(rng, 256, 4096)),
                nx=round(_log(rng, 256, 4096)), pitch=8e-6, precision=precision)


# ---------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _rand(g, *shape, lo=0.0, hi=1.0, dtype=torch.float32):
    return torch.rand(*shape, generator=g, device="cuda", dtype=dtype) * (hi - lo) + lo


def _field(c, g, lead=()):
    """Amplitude uniform in [0, 1), phase uniform in [0, 2 pi)."""
    shape = (*lead, c["ny"], c["nx"])
    rt = torch.float64 if c.get("c128") else torch.float32
    return torch.polar(_rand(g, *shape, dtype=rt), _rand(g, *shape, hi=2 * math.pi, dtype=rt))


def _targets(c, g):
    """One target per plane: 32 Gaussians over the field, scaled to [0, 1]."""
    n = c["n"]
    i = torch.arange(n, device="cuda", dtype=torch.float64)
    out = []
    for _ in range(c["planes"]):
        cy, cx = (_rand(g, 32, hi=n, dtype=torch.float64) for _ in range(2))
        s = _rand(g, 32, lo=n / 100, hi=n / 10, dtype=torch.float64)
        a = _rand(g, 32, lo=0.5, dtype=torch.float64)
        gy = torch.exp(-((i[None] - cy[:, None]) / s[:, None]) ** 2 / 2) * a[:, None]
        gx = torch.exp(-((i[None] - cx[:, None]) / s[:, None]) ** 2 / 2)
        t = gy.T.contiguous() @ gx
        t = t - t.min()
        out.append((t / t.max()).float())
    return out


def _planes(c):
    return [c["z"] * (1.0, 1.2, 1.5, 1.7)[k] for k in range(c["planes"])]


def _cloud(c, g):
    """Host coordinates of a cloud over the hologram's aperture, as a program reads them."""
    n, p = c["n"], c["pitch"]
    zlo, zhi = (0.151, 0.155) if c["kind"] == "wrp" else (0.10, 0.20)
    x = _rand(g, n, hi=c["nx"] * p, dtype=torch.float64)
    y = _rand(g, n, hi=c["ny"] * p, dtype=torch.float64)
    z = _rand(g, n, lo=zlo, hi=zhi, dtype=torch.float64)
    a = _rand(g, n, lo=0.5)
    ph = _rand(g, n, hi=2 * math.pi)
    return [t.cpu().numpy() for t in (x, y, z, a, ph)]


def prepare(case, seed):
    c, g = case, _gen(seed)
    s = dict(c=c)
    if c["kind"] == "asm":
        s["u"] = _field(c, g)
    elif c["kind"] == "fresnel":
        s["src"] = _field(c, g)
        s["u"] = torch.empty_like(s["src"])
    elif c["kind"] == "grad":
        s["u"] = _field(c, g, (c["nb"],)).requires_grad_(True)
        s["g"] = _field(c, g, (c["nb"],))
    elif c["kind"] == "plane":
        s["phi"] = _rand(g, c["n"], c["n"], hi=2 * math.pi).requires_grad_(True)
        s["targets"], s["zs"] = _targets(c, g), _planes(c)
    else:
        x, y, z, a, ph = _cloud(c, g)
        s["obj"] = ol.Object(x, y, z) if c["kind"] == "wrp" else ol.Object(x, y, z, a, ph)
        s["U"] = torch.empty((c["ny"], c["nx"]), dtype=torch.complex64, device="cuda")
        if c["kind"] == "wrp":
            s["H"] = torch.empty_like(s["U"])
    return s


# ---------------------------------------------------------------- one pass
def run(state):
    s, c = state, state["c"]
    k, p = c["kind"], c["pitch"]
    if k == "asm":
        return ol.AsmProp(s["u"], c["ny"], c["nx"], p, p, LAM, c["z"], bandlimit=c["bandlimit"],
                          adjoint=c["adjoint"])
    if k == "fresnel":
        # FresnelProp scales by 1/M^2: each pass starts from the loaded field
        s["u"].copy_(s["src"])
        return ol.FresnelProp(s["u"], c["ny"], c["nx"], p, p, LAM, c["z"])
    if k == "grad":
        y = autograd.asm_prop(s["u"], p, p, LAM, c["z"])
        (gu,) = torch.autograd.grad(y, s["u"], s["g"])
        return y.detach(), gu
    if k == "plane":
        loss = autograd.multiplane_loss(s["phi"], s["targets"], s["zs"], p, p, LAM, norm="mean")
        (gphi,) = torch.autograd.grad(loss, s["phi"])
        return loss.detach(), gphi
    if k == "cgh":
        return ol.Cgh(s["obj"], s["U"], c["ny"], c["nx"], p, p, LAM, exact_r=c["exact_r"])
    if k == "wrp":
        ol.WRPStep1(s["obj"], s["U"], c["ny"], c["nx"], p, LAM, 0.15)
        ol.ARSSFresnelProp(s["U"], s["H"], c["ny"], c["nx"], p, p, LAM, 0.15, 0.5)
        return s["U"], s["H"]
    return ol.CghLayered(s["obj"], s["U"], c["ny"], c["nx"], p, p, LAM, c["layers"], 0.10, 0.20,
                         precision=c["precision"])


def _prop_work(ny, nx, item):
    """Field in, field out; row transforms of the stored rows, column transforms both ways."""
    return dict(bytes=2 * ny * nx * item,
                flops=5.0 * (2 * ny * 2 * nx * math.log2(2 * nx)
                             + 2 * 2 * nx * 2 * ny * math.log2(2 * ny)))


def work(case):
    c, k = case, case["kind"]
    if k in ("asm", "fresnel"):
        w = _prop_work(c["ny"], c["nx"], 16 if c["c128"] else 8)
        return dict(bytes=w["bytes"] * (2 if k == "fresnel" else 1), flops=w["flops"])
    if k == "grad":
        w = _prop_work(c["ny"], c["nx"], 8)
        return dict(bytes=2 * c["nb"] * w["bytes"], flops=2 * c["nb"] * w["flops"])
    if k == "plane":
        px, w = c["n"] ** 2, _prop_work(c["n"], c["n"], 8)
        return dict(bytes=4 * px * (2 + c["planes"]), flops=2 * c["planes"] * w["flops"])
    px = c["ny"] * c["nx"]
    if k == "cgh":
        # spherical: distance, phase and the term per point and pixel; Fresnel separates, so
        # one complex multiply-add is left
        return dict(bytes=32 * c["n"] + 8 * px, flops=c["n"] * px * (16.0 if c["exact_r"] else 8.0))
    if k == "wrp":
        # circular windows, mean area from the mean distance to the plane; ARSS after them
        w = _prop_work(c["ny"], c["nx"], 8)
        r = 0.003 / math.sqrt(4 * (c["pitch"] / LAM) ** 2 - 1) / c["pitch"]
        return dict(bytes=32 * c["n"] + 8 * px + w["bytes"],
                    flops=c["n"] * math.pi * r * r * 12.0 + w["flops"])
    return dict(bytes=32 * c["n"] + 8 * px, flops=8.0 * c["n"] * px)


# ---------------------------------------------------------------- the same in 64 bits
F64, C128 = torch.float64, torch.complex128


def _cis(cycles):
    """exp(2 pi i cycles), the integer part dropped first."""
    a = 2 * math.pi * (cycles - torch.round(cycles))
    return torch.complex(torch.cos(a), torch.sin(a))


def _arange(n, half=0):
    return torch.arange(n, device="cuda", dtype=F64) - half


def _pad(u):
    ny, nx = u.shape
    out = torch.zeros((2 * ny, 2 * nx), dtype=C128, device="cuda")
    out[ny // 2:ny // 2 + ny, nx // 2:nx // 2 + nx] = u
    return out


def _crop(u):
    ny, nx = u.shape
    return u[ny // 4:ny // 4 + ny // 2, nx // 4:nx // 4 + nx // 2]


def _asm_h(ny, nx, p, z, bandlimit, adjoint=False):
    v = (_arange(2 * ny, ny) / (2 * ny * p))[:, None]
    u = (_arange(2 * nx, nx) / (2 * nx * p))[None]
    arg = 1 / LAM ** 2 - u * u - v * v
    keep = arg >= 0
    if bandlimit:
        for f, n in ((u, nx), (v, ny)):
            lim = 1 / math.sqrt((z / (n * p)) ** 2 + 1) / LAM
            keep = keep & (f.abs() < lim)
    h = _cis(torch.sqrt(arg.clamp_min(0)) * z) * keep
    return torch.fft.ifftshift(h.conj() if adjoint else h)


def _conv(u, h):
    return _crop(torch.fft.ifft2(torch.fft.fft2(_pad(u)) * h)).contiguous()


def _asm(u, p, z, bandlimit, adjoint=False):
    return _conv(u.to(C128), _asm_h(*u.shape, p, z, bandlimit, adjoint))


def _chirp(n, p, z, q, lin=0.0):
    """exp(i pi (q x^2 + lin x) / (lambda z)) on centred coordinates."""
    x = _arange(n, n // 2) * p
    return _cis((q * x * x + lin * x) / (2 * LAM * z))


def _limit(v, p):
    """A window's half-width in pixels, kept finite where there is none."""
    return min(math.floor(v / p), 2 ** 31 - 1)


def _fresnel(u, p, z):
    ny, nx = u.shape
    hy, hx = _chirp(2 * ny, p, z, 1.0), _chirp(2 * nx, p, z, 1.0)
    sy, sx = (torch.fft.fft(torch.fft.ifftshift(h)) for h in (hy, hx))
    return _conv(u.to(C128), sy[:, None] * sx[None] / (4 * ny * nx))


def _arss(u, p, z, s):
    ny, nx = u.shape
    iy, ix = _arange(ny, ny // 2).abs()[:, None], _arange(nx, nx // 2).abs()[None]
    lim = _limit(LAM * z * 0.5 / (s * abs(s - 1) * p), p)
    pre = _chirp(ny, p, z, s * s - s)[:, None] * _chirp(nx, p, z, s * s - s)[None]
    src = u.to(C128) * pre * ((iy < lim) & (ix < lim))
    lim = _limit(LAM * z * 0.5 / (p * s), p)
    spec = [torch.fft.fft(torch.fft.ifftshift(_chirp(2 * n, p, z, s)
                                              * (_arange(2 * n, n).abs() < lim))) for n in (ny, nx)]
    m2 = 4 * ny * nx
    out = _conv(src, spec[0][:, None] * spec[1][None] / m2)
    lim = _limit(LAM * z * 0.5 / (abs(1 - s) * p), p)
    post = _chirp(ny, p, z, 1 - s)[:, None] * _chirp(nx, p, z, 1 - s)[None]
    return torch.where((iy < lim) & (ix < lim), out * post, out)


def _points(state):
    """The cloud's records as the device holds them: float amplitudes and phases."""
    r = state["obj"].host
    return [torch.from_numpy(r[k].astype("f8")).cuda() for k in ("x", "y", "z", "amp", "phase")]


def _cgh_exact(c, pts):
    x, y, z, a, ph = pts
    p, px = c["pitch"], _arange(c["nx"])[None, :] * c["pitch"]
    U = torch.zeros((c["ny"], c["nx"]), dtype=C128, device="cuda")
    rows = max(1, int(1.5e8) // (c["nx"] * 64))
    for h0 in range(0, c["ny"], rows):
        py = (_arange(c["ny"])[h0:h0 + rows] * p)[:, None]
        for j in range(0, len(x), 64):
            k = slice(j, j + 64)
            dx2 = (px - x[k, None]).square()[:, None, :]
            dy2 = (py.T - y[k, None]).square()[:, :, None]
            cyc = torch.sqrt(dx2 + dy2 + z[k, None, None].square()) / LAM
            t = cyc.sub_(torch.round(cyc)).mul_(2 * math.pi).add_(ph[k, None, None])
            re = torch.einsum("j,jhw->hw", a[k], torch.cos(t))
            im = torch.einsum("j,jhw->hw", a[k], torch.sin(t))
            U[h0:h0 + rows] += torch.complex(re, im)
    return U


def _cgh_fresnel(c, x, y, z, a, ph):
    """Separable in 64 bits: two factors per point, multiplied as matrices."""
    p = c["pitch"]
    U = torch.zeros((c["ny"], c["nx"]), dtype=C128, device="cuda")
    for j in range(0, len(x), 4096):
        k = slice(j, j + 4096)
        q = 1 / (2 * LAM * z[k])
        fy = _cis((_arange(c["ny"])[:, None] * p - y[None, k]) ** 2 * q)
        fx = _cis((_arange(c["nx"])[None] * p - x[k, None]) ** 2 * q[:, None]
                  + (ph[k] / (2 * math.pi))[:, None]) * a[k, None]
        U += fy @ fx
    return U


def _wrp(c, pts, plane):
    x, y, z = pts[:3]
    p, ny, nx = c["pitch"], c["ny"], c["nx"]
    W = (z - plane).abs() / math.sqrt(4 * (p / LAM) ** 2 - 1)
    r = int(W.max().item() / p) + 2
    o = torch.arange(-r, r + 1, device="cuda")
    U = torch.zeros(ny * nx, 2, dtype=F64, device="cuda")
    step = max(1, int(2e7) // (2 * r + 1) ** 2)
    for j in range(0, len(x), step):
        k = slice(j, j + step)
        w = torch.round(x[k] / p).long()[:, None, None] + o[None, None, :]
        h = torch.round(y[k] / p).long()[:, None, None] + o[None, :, None]
        rho = (p * w.to(F64) - x[k, None, None]) ** 2 + (p * h.to(F64) - y[k, None, None]) ** 2
        dz = (z[k] - plane)[:, None, None]
        inside = (rho < W[k, None, None] ** 2) & (w >= 0) & (w < nx) & (h >= 0) & (h < ny)
        t = _cis(rho / (2 * dz * LAM)) / dz.abs()
        at = (h * nx + w)[inside]
        U.index_add_(0, at, torch.view_as_real(t[inside]))
    return torch.view_as_complex(U).view(ny, nx)


def exact(case, seed):
    s, c = prepare(case, seed), case
    k, p = c["kind"], c["pitch"]
    if k == "asm":
        return _asm(s["u"], p, c["z"], c["bandlimit"], c["adjoint"])
    if k == "fresnel":
        return _fresnel(s["src"], p, c["z"])
    if k == "grad":
        u = s["u"].detach()
        return (torch.stack([_asm(f, p, c["z"], True) for f in u]),
                torch.stack([_asm(f, p, c["z"], True, adjoint=True) for f in s["g"]]))
    if k == "plane":
        phi = s["phi"].detach().to(F64).requires_grad_(True)
        u = torch.complex(torch.cos(phi), torch.sin(phi))
        loss = 0.0
        for t, z in zip(s["targets"], s["zs"]):
            f = _asm(u, p, z, True)
            i = f.real ** 2 + f.imag ** 2
            t = t.to(F64)
            loss = loss + ((i / i.mean() - t / t.mean()) ** 2).mean()
        (g,) = torch.autograd.grad(loss, phi)
        return loss.detach(), g
    pts = _points(s)
    if k == "cgh":
        return _cgh_exact(c, pts) if c["exact_r"] else _cgh_fresnel(c, *pts)
    if k == "wrp":
        U = _wrp(c, pts, 0.15)
        return U, _arss(U, p, 0.15, 0.5)
    x, y, z, a, ph = pts
    layer = torch.floor((z - 0.10) / (0.20 - 0.10) * c["layers"]).clamp(0, c["layers"] - 1)
    return _cgh_fresnel(c, x, y, 0.10 + (layer + 0.5) * (0.20 - 0.10) / c["layers"], a, ph)
