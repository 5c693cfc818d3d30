"""Performance cases: what users of the phasing engine run, through its public entry points.

A case is a plain dict; ``kind`` names the entry points it goes through:

``phaser``  one reconstruction through the reference's phasing API (sp_phaser_*), 2-D or 3-D:
            sp_phaser_iterate, the model read as a device array, and with ``scores`` the metrics
            that a driver reads at every output point; ``area`` adds the area shrinkwrap
``batch``   many same-shape reconstructions in one Batch, as Reconstructor.reconstruct_loop and
            the server advance them between two output points, then the models before projection
            of all of them (page-locked download); ``mixed`` gives every slot its own algorithm
            and beta, as the server does
``fft``     spx_fft_device, forward and inverse, on device arrays
``prtf``    libspimage_amd.prtf.prtf of host reconstructions (aligned against each other)

Patterns are the exact amplitudes of a textured object in an ellipse of semi-axes n / 6.4 (the
disc of the 256 x 256 workload, scaled), four pixels of beamstop, the ellipse plus 3 pixels as
support, and a start near the solution: the late phase of a reconstruction, where an iteration
does not amplify rounding differences, so results can be compared after tens of iterations.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from libspimage_amd import spimage as sp
from libspimage_amd.prtf import prtf

_DEV = torch.device("cuda")
_ALG = {"hio": sp.SpHIO, "raar": sp.SpRAAR, "er": sp.SpER}


def listed():
    return [
        # the smallest call in use: a low-resolution preview, scores read every 10 iterations;
        # two launches an iteration and two host waits a pass
        {"name": "preview_128", "kind": "phaser", "nz": 1, "ny": 128, "nx": 128, "alg": "hio", "n": 10, "scores": True},
        # the plain 1024 x 1024 HIO iteration of one reconstruction
        {"name": "hio_1024", "kind": "phaser", "nz": 1, "ny": 1024, "nx": 1024, "alg": "hio", "n": 20},
        # RAAR with the area shrinkwrap every 20 iterations, as it is run in production
        {"name": "raar_shrinkwrap_1024", "kind": "phaser", "nz": 1, "ny": 1024, "nx": 1024, "alg": "raar", "n": 20,
         "area": True, "period": 20},
        # a cropped detector: ragged mixed-radix sides and a positive real object
        {"name": "er_real_900x750", "kind": "phaser", "nz": 1, "ny": 900, "nx": 750, "alg": "er", "n": 20,
         "real": True},
        # the largest 2-D arrays: a 16-megapixel detector
        {"name": "hio_4096", "kind": "phaser", "nz": 1, "ny": 4096, "nx": 4096, "alg": "hio", "n": 4},
        # a detector crop with prime sides: any length is accepted, as by the reference's FFT
        {"name": "hio_1021x769", "kind": "phaser", "nz": 1, "ny": 769, "nx": 1021, "alg": "hio", "n": 5},
        # the 256-cubed volume: difference map
        {"name": "dm_256_cubed", "kind": "phaser", "nz": 256, "ny": 256, "nx": 256, "alg": "dm", "n": 4},
        # 256 random starts of a small pattern, shrinkwrap every 25 iterations
        {"name": "starts_128x256", "kind": "batch", "nz": 1, "ny": 128, "nx": 128, "nrec": 256, "alg": "raar",
         "n": 50, "area": True, "period": 25},
        # part of a quantum of a served class: 16 requests of 720 x 720 with their own algorithms
        {"name": "served_720x16", "kind": "batch", "nz": 1, "ny": 720, "nx": 720, "nrec": 16, "mixed": True, "n": 30},
        # part of a quantum of a served 3-D class
        {"name": "served_96_cubed_x8", "kind": "batch", "nz": 96, "ny": 96, "nx": 96, "nrec": 8, "mixed": True,
         "n": 30},
        # plain transforms of a ragged volume, both directions
        {"name": "fft_120x200x216", "kind": "fft", "nz": 120, "ny": 200, "nx": 216},
        # resolution estimate over 32 reconstructions, arrays from and to the host
        {"name": "prtf_256x32", "kind": "prtf", "nz": 1, "ny": 256, "nx": 256, "nrec": 32},
    ]


def _smooth(lo, hi, primes=(2, 3, 5)):
    def ok(n):
        for p in primes:
            while n % p == 0:
                n //= p
        return n == 1
    return [n for n in range(lo, hi + 1) if ok(n)]


def _pick(rng, lo, hi, primes=(2, 3, 5)):
    """A smooth length, spread over the logarithm of [lo, hi]."""
    t = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(_smooth(lo, hi, primes), key=lambda n: abs(math.log(n / t)))


def _side(rng, n, lo, hi, primes=(2, 3, 5)):
    """The other side of an array: equal in half of the cases, else within a factor 1.5."""
    return n if rng.random() < 0.5 else _pick(rng, max(lo, int(n / 1.5)), min(hi, int(n * 1.5)), primes)


def draw(rng):
    what = rng.choice(["small", "single", "shrinkwrap", "large", "odd", "volume", "starts", "served", "served3d",
                       "fft", "prtf"])
    if what in ("small", "single", "shrinkwrap", "large"):
        lo, hi = {"small": (64, 384), "single": (400, 1400), "shrinkwrap": (200, 1400), "large": (1500, 4096)}[what]
        nx = _pick(rng, lo, hi, (2, 3, 5, 7))
        ny = _side(rng, nx, lo, hi, (2, 3, 5, 7))
        c = {"kind": "phaser", "nz": 1, "ny": ny, "nx": nx, "alg": rng.choice(["hio", "raar", "er"]),
             "n": 4 if what == "large" else 20}
        if what == "small":
            c["scores"] = True
            c["n"] = 10
        if what == "shrinkwrap":
            c.update(alg="raar", n=20, area=True, period=20)
        elif rng.random() < 0.3:
            c["real"] = True
        return c
    if what == "odd":
        # at least one side with a prime factor above 7
        while True:
            nx, ny = (int(math.exp(rng.uniform(math.log(100), math.log(1100)))) for _ in range(2))
            if not (sp.spx_supported_length(nx) and sp.spx_supported_length(ny)) and max(nx, ny) < 4 * min(nx, ny):
                return {"kind": "phaser", "nz": 1, "ny": ny, "nx": nx, "alg": rng.choice(["hio", "raar", "er"]), "n": 5}
    if what == "volume":
        nx = _pick(rng, 64, 256)
        return {"kind": "phaser", "nz": _side(rng, nx, 64, 256), "ny": _side(rng, nx, 64, 256), "nx": nx,
                "alg": rng.choice(["dm", "hio", "er"]), "n": 4}
    if what in ("starts", "served"):
        nx = _pick(rng, 96 if what == "starts" else 128, 512 if what == "starts" else 1024)
        ny = _side(rng, nx, 96, 1024)
        most = max(2, int((4.2e6 if what == "starts" else 8.4e6) / (nx * ny)))
        c = {"kind": "batch", "nz": 1, "ny": ny, "nx": nx, "nrec": rng.randint(max(2, most // 8), min(256, most))}
        if what == "starts":
            c.update(alg="raar", n=50, area=True, period=25)
        else:
            c.update(mixed=True, n=30)
        return c
    if what == "served3d":
        n = _pick(rng, 64, 128)
        return {"kind": "batch", "nz": n, "ny": n, "nx": n, "nrec": rng.randint(2, max(2, int(7.1e6 / n ** 3))),
                "mixed": True, "n": 30}
    if what == "fft":
        if rng.random() < 0.5:
            nx = _pick(rng, 64, 256, (2, 3, 5, 7))
            return {"kind": "fft", "nz": _side(rng, nx, 64, 256, (2, 3, 5, 7)),
                    "ny": _side(rng, nx, 64, 256, (2, 3, 5, 7)), "nx": nx}
        return {"kind": "fft", "nz": 1, "ny": int(math.exp(rng.uniform(math.log(60), math.log(2000)))),
                "nx": _pick(rng, 64, 4096, (2, 3, 5, 7))}
    nx = _pick(rng, 128, 400)
    return {"kind": "prtf", "nz": 1, "ny": _side(rng, nx, 128, 400), "nx": nx, "nrec": rng.randint(4, 32)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _shape(case):
    return (case["ny"], case["nx"]) if case["nz"] == 1 else (case["nz"], case["ny"], case["nx"])


def _generator(seed):
    return torch.Generator(device=_DEV).manual_seed(int(seed) * 7919 + 17)


def _radius(shape, grow):
    """Distance from the origin (FFT order) in units of the ellipse's semi-axes + grow."""
    r2 = 0.0
    for ax, n in enumerate(shape):
        k = torch.fft.fftfreq(n, 1.0 / n, device=_DEV, dtype=torch.float64) / (n / 6.4 + grow)
        r2 = r2 + k.reshape([-1 if a == ax else 1 for a in range(len(shape))]) ** 2
    return r2.sqrt()


def _pattern(shape, gen):
    """(amplitudes f32, mask bool, support bool, start c64) on the GPU."""
    o = torch.rand(shape, generator=gen, device=_DEV, dtype=torch.float64) * (_radius(shape, 0.0) <= 1)
    amp = torch.fft.fftn(o).abs()
    o, amp = o / amp.square().mean().sqrt(), amp / amp.square().mean().sqrt()
    d2 = 0.0
    for ax, n in enumerate(shape):
        c = torch.arange(n, device=_DEV, dtype=torch.float64)
        c = torch.minimum(c, n - 1 - c)
        d2 = d2 + c.reshape([-1 if a == ax else 1 for a in range(len(shape))]) ** 2
    mask = d2 >= 16
    start = o * (1 + 0.01 * torch.randn(shape, generator=gen, device=_DEV, dtype=torch.float64))
    return (amp * mask).float(), mask, _radius(shape, 3.0) <= 1, start.to(torch.complex64)


def _patterns(case, seed):
    gen = _generator(seed)
    return [_pattern(_shape(case), gen) for _ in range(case.get("nrec", 1))]


def _area(case):
    """Area fraction of the support that the shrinkwrap keeps: the ellipse plus 2 pixels."""
    return float(np.float32(math.pi * math.prod(n / 6.4 + 2 for n in _shape(case)) / math.prod(_shape(case))))


def _slots(case):
    """Algorithm and beta of every slot of a mixed batch."""
    names = ("er", "hio", "raar")
    return [(names[r % 3], 0.9 if r % 2 else 0.8) for r in range(case["nrec"])]


def _algorithm(case, keep):
    c = sp.SpPositiveRealObject if case.get("real") else sp.SpNoConstraints
    alg = "er" if case.get("mixed") else case["alg"]
    if alg == "er":
        return sp.sp_phasing_er_alloc(c)
    beta = sp.smap([(0, 0.8 if alg == "dm" else 0.9)])
    keep.append(beta)
    if alg == "dm":
        return sp.sp_phasing_diff_map_alloc(beta, float("inf"), float("inf"), c)
    return (sp.sp_phasing_hio_alloc if alg == "hio" else sp.sp_phasing_raar_alloc)(beta, c)


def _before(case):
    """Iterations that a state has behind it: with a shrinkwrap, the update falls inside the pass."""
    return case["period"] // 2 if case.get("area") else 0


def _schedule(case, keep):
    if not case.get("area"):
        return None
    blur, area = sp.smap([(0, 2.0)]), sp.smap([(0, _area(case))])
    keep += [blur, area]
    return sp.sp_support_array_init(sp.sp_support_area_alloc(blur, area), case["period"])


class _DeviceArray:
    """complex64 device memory of a phaser's engine, for torch.as_tensor: the tensor holds this
    object, and with it the phaser whose memory it is."""

    def __init__(self, owner, address, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<c8", "data": (address, False), "version": 3}


class _Phaser:
    _free = staticmethod(sp.sp_phaser_free)

    def __init__(self, case, seed):
        self.shape, self.keep, self.images = _shape(case), [], []
        (amp, mask, support, start), = _patterns(case, seed)
        self.ph = sp.sp_phaser_alloc()
        if sp.sp_phaser_init(self.ph, _algorithm(case, self.keep), _schedule(case, self.keep), sp.SpEngineHIP) != 0:
            raise RuntimeError(sp.last_error())
        a = self._image(amp, mask)
        g = self._image(start)
        s = self._image(support.float())
        sp.sp_phaser_set_amplitudes(self.ph, a)
        if sp.sp_phaser_init_model(self.ph, g, 0) != 0 or sp.sp_phaser_init_support(self.ph, s, 0, 0.0) != 0:
            raise RuntimeError(sp.last_error())
        for im in self.images:
            sp.sp_image_free(im)
        if _before(case) and sp.sp_phaser_iterate(self.ph, _before(case)) != 0:
            raise RuntimeError(sp.last_error())

    def _image(self, data, mask=None):
        im = sp.image_from_array(data.cpu().numpy(), None if mask is None else mask.cpu().numpy())
        self.images.append(im)
        return im

    def model(self):
        g1 = C.c_void_p()
        if sp.spx_phaser_device_arrays(self.ph, C.byref(g1), None, None) != 0:
            raise RuntimeError(sp.last_error())
        return torch.as_tensor(_DeviceArray(self, g1.value, self.shape), device=_DEV)

    def __del__(self):
        self._free(self.ph)


class _HostArray(np.ndarray):
    """A view of a batch's page-locked staging memory that holds the batch."""

    owner = None


def _batch(case, seed, keep):
    shape, n = _shape(case), case["nrec"]
    b = sp.Batch(shape, n)
    pats = _patterns(case, seed)
    amp, mask, support, start = (torch.stack([p[k] for p in pats]).cpu().numpy() for k in range(4))
    b.set_data(-1, amp, mask, support)
    b.set_algorithm(_algorithm(case, keep))
    b.set_model(-1, start)
    if case.get("area"):
        b.set_support_schedule(_schedule(case, keep))
    if case.get("mixed"):
        slots = _slots(case)
        b.set_rec_algorithms([_ALG[a] for a, _ in slots], [beta for _, beta in slots])
        b.set_active([1] * n)
    if _before(case):
        b.iterate(_before(case))
    return b


def _reconstructions(case, seed):
    """Noisy shifted, reflected and phase-shifted copies of one object, and its supports."""
    gen, shape, n = _generator(seed), _shape(case), case["nrec"]
    region = _radius(shape, 0.0) <= 1
    obj = torch.complex(*(torch.rand(shape, generator=gen, device=_DEV) for _ in range(2))) * region
    host = np.random.default_rng(int(seed))
    imgs, masks = [], []
    for r in range(n):
        a = obj + 0.05 * torch.complex(*(torch.randn(shape, generator=gen, device=_DEV) for _ in range(2)))
        m = region
        if r and host.random() < 0.5:
            a = a.flip(tuple(range(len(shape))))
        sh = [int(host.integers(0, k)) for k in shape]
        dims = tuple(range(len(shape)))
        a = torch.roll(a, sh, dims) * np.exp(2j * np.pi * host.random())
        imgs.append(a.to(torch.complex64))
        masks.append(torch.roll(m, sh, dims))
    return torch.stack(imgs).cpu().numpy(), torch.stack(masks).cpu().numpy().astype(np.int32)


def prepare(case, seed):
    if case["kind"] == "phaser":
        return {"case": case, "ph": _Phaser(case, seed)}
    if case["kind"] == "batch":
        keep = []
        return {"case": case, "batch": _batch(case, seed, keep), "keep": keep}
    if case["kind"] == "fft":
        x = torch.randn(_shape(case), generator=_generator(seed), device=_DEV, dtype=torch.complex64)
        return {"case": case, "in": x, "f": torch.empty_like(x), "out": torch.empty_like(x)}
    images, masks = _reconstructions(case, seed)
    return {"case": case, "images": images, "masks": masks}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    case = state["case"]
    if case["kind"] == "phaser":
        p = state["ph"]
        if sp.sp_phaser_iterate(p.ph, case["n"]) != 0:
            raise RuntimeError(sp.last_error())
        out = {"model": p.model()}
        if case.get("scores"):
            fcfo = C.c_float()
            # of the two scores of this call FcFo is compared: near the solution E_F is a small
            # difference of large numbers, whose last digits change with any rounding
            sp.sp_phaser_efourier(p.ph, C.byref(fcfo))
            out["fcfo"] = fcfo.value
            out["support"] = sp.sp_phaser_support_fraction(p.ph)
        if case.get("area"):
            out["support"] = sp.sp_phaser_support_fraction(p.ph)
        return out
    if case["kind"] == "batch":
        b = state["batch"]
        b.iterate(case["n"])
        out = b.model_before_projection(staged=True).view(_HostArray)
        out.owner = b
        return {"before": out}
    if case["kind"] == "fft":
        z, y, x = case["nz"], case["ny"], case["nx"]
        torch.cuda.current_stream().synchronize()  # the library's stream is its own
        if sp.spx_fft_device(state["in"].data_ptr(), state["f"].data_ptr(), x, y, z, -1) != 0 or \
                sp.spx_fft_device(state["f"].data_ptr(), state["out"].data_ptr(), x, y, z, 1) != 0:
            raise RuntimeError(sp.last_error())
        return {"forward": state["f"], "inverse": state["out"]}
    return prtf(state["images"], state["masks"])


def work(case):
    """What an iteration cannot do without: the iterate, the amplitudes and the flags read, the new
    iterate written (21 bytes a pixel; the difference map carries a second array through the
    transforms, not through memory), and the transforms' 5 N log2 N operations each."""
    px = case["nz"] * case["ny"] * case["nx"] * case.get("nrec", 1)
    lg = math.log2(case["nz"] * case["ny"] * case["nx"])
    if case["kind"] == "fft":
        return {"bytes": 2 * 16 * px, "flops": 2 * 5 * px * lg}
    if case["kind"] == "prtf":
        # images and masks in; six transforms for each reconstruction
        return {"bytes": 12 * px, "flops": 6 * 5 * px * lg}
    n = case["n"]
    pairs = 2 if case.get("alg") == "dm" else 1
    return {"bytes": n * 21 * px, "flops": n * px * pairs * (10 * lg + 20)}


# ---------------------------------------------------------------------------
# the same in 64 bits, from the definitions (torch, complex128)
# ---------------------------------------------------------------------------
def _project(F, amp, mask):
    m = amp / F.abs()
    P = torch.where(torch.isfinite(m), F * torch.nan_to_num(m, posinf=0.0), amp.to(F.dtype))
    return torch.where(mask, P, F)


def _constrain(g, real):
    return torch.complex(g.real.clamp(min=0), torch.zeros_like(g.imag)) if real else g


def _step(alg, g, amp, mask, sup, beta, real):
    """(new iterate, model before projection)"""
    gp = torch.fft.ifftn(_project(torch.fft.fftn(g), amp, mask))
    if alg == "dm":
        b = float(np.float32(0.8))
        s = 0.1
        gamma1, gamma2 = -(4 + (2 + b) * s + b * s * s) / (b * (4 - s + s * s)), (3 - b) / (2 * b)
        f1 = torch.where(sup, g, -gamma1 * g)
        pf = torch.fft.ifftn(_project(torch.fft.fftn(f1), amp, mask))
        new = torch.where(sup, g + b * ((1 + gamma2) * gp - gamma2 * g), g) - b * pf
        return torch.where(sup, _constrain(new, real), new), gp
    outside = {"er": torch.zeros_like(g), "hio": g - beta * gp, "raar": beta * g + (1 - 2 * beta) * gp}[alg]
    return torch.where(sup, _constrain(gp, real), outside), gp


def _shrinkwrap(g, area, sigma):
    """Support from |g| blurred (the transfer function's frequencies are in units of 1 / nx on
    every axis) above the value of descending index N area."""
    r2 = 0.0
    for ax, n in enumerate(g.shape):
        k = torch.fft.fftfreq(n, 1.0 / n, device=_DEV, dtype=torch.float64) / g.shape[-1]
        r2 = r2 + k.reshape([-1 if a == ax else 1 for a in range(g.ndim)]) ** 2
    b = torch.fft.ifftn(torch.fft.fftn(g.abs()) * torch.exp(-2 * math.pi ** 2 * sigma ** 2 * r2)).abs()
    k = int(np.float32(g.numel()) * np.float32(area))
    return b > torch.topk(b.flatten(), k + 1).values[-1]


def _iterate(case, pat, alg, beta):
    amp, mask, sup, g = pat[0].double(), pat[1], pat[2], pat[3].to(torch.complex128)
    gp = g
    for it in range(_before(case) + case["n"]):
        if case.get("area") and it % case["period"] == case["period"] - 1:
            sup = _shrinkwrap(g, _area(case), 2.0)
        else:
            g, gp = _step(alg, g, amp, mask, sup, float(np.float32(beta)), case.get("real"))
    return g, gp, sup


def exact(case, seed):
    if case["kind"] == "fft":
        x = torch.randn(_shape(case), generator=_generator(seed), device=_DEV, dtype=torch.complex64)
        f = torch.fft.fftn(x.to(torch.complex128))
        return {"forward": f, "inverse": x.to(torch.complex128) * x.numel()}
    if case["kind"] == "prtf":
        return _exact_prtf(*_reconstructions(case, seed))
    pats = _patterns(case, seed)
    if case["kind"] == "batch":
        slots = _slots(case) if case.get("mixed") else [(case["alg"], 0.9)] * case["nrec"]
        return {"before": torch.stack([_iterate(case, p, a, b)[1] for p, (a, b) in zip(pats, slots)])}
    g, _, sup = _iterate(case, pats[0], case["alg"], 0.9)
    out = {"model": g}
    if case.get("scores"):
        F, amp = torch.fft.fftn(g).abs(), pats[0][0].double()
        mask = pats[0][1]
        out["fcfo"] = float(amp[mask].sum() / F[mask].sum())
    if case.get("scores") or case.get("area"):
        out["support"] = float(sup.double().mean())
    return out


def _exact_prtf(images, masks):
    imgs = torch.from_numpy(images).to(_DEV).to(torch.complex128)
    dims = tuple(range(imgs.ndim - 1))
    avg = imgs[0].clone()
    F = torch.fft.fftn(avg)
    total = F / F.abs()
    for a in imgs[1:]:
        A, B = torch.fft.fftn(avg.abs().to(avg.dtype)), torch.fft.fftn(a.abs().to(avg.dtype))
        corr, conv = torch.fft.ifftn(A * B.conj()).abs(), torch.fft.ifftn(A * B).abs()
        reflect = bool(conv.max() > corr.max())
        at = np.unravel_index(int((conv if reflect else corr).argmax()), corr.shape)
        if reflect:
            a, at = a.flip(dims), [k + 1 for k in at]
        a = torch.roll(a, [int(k) for k in at], dims)
        a = a * torch.exp(1j * (avg.abs() ** 2 * torch.exp(1j * (avg.angle() - a.angle()))).sum().angle())
        avg = avg + a
        F = torch.fft.fftn(a)
        total = total + F / F.abs()
    return {"prtf": torch.fft.fftshift((total / len(imgs)).abs()), "super_image": avg}
