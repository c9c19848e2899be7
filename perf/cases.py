"""Workloads of the framework, for timing and for comparing results.

Each case is one pass through public entry points as a program that generates
initial conditions calls them:

* ``run``       one box of the whole pipeline (``ICRun.execute``): noise, LPT
                sources, assembly, transforms, component fields or particles
* ``batch``     many 2LPT boxes replayed as one HIP graph (``batch.Batch``)
* ``adjoint``   the differentiable 2LPT map, forward and backward, through
                ``torch.autograd`` (``adjoint.lpt2_map``)
* ``sources``   the potentials phi2, phi3, A3 from a given phi1
                (``lpt.lpt_sources``)
* ``products``  dealiased products through ``OrszagConvolver``, the way code
                written against the reference's convolver forms the 2LPT source
* ``poisson``   a potential from a density field with ``Grid``: transform,
                inverse Laplacian, transform back
* ``noise``     NGenIC white noise of a grid (``lpt.ngenic_fill``)
* ``ppt``       the semiclassical density and velocity fields of an executed
                run (``mfic_ppt_fields``)

``exact`` restates them in 64 bits with plain torch and numpy.
"""
import ctypes
import math

import numpy as np
import torch

from monofonic_amd import BCC, F32, F64, KSPACE, RSPACE, SC, Context, Grid, _lib, lpt
from monofonic_amd.adjoint import LPT2, lpt2_map
from monofonic_amd.batch import Batch

FCC = _lib.FCC
# subgroups of 2^a 3^b: lengths every transform takes, and grids whose 3/2
# padded length is one of them too
LENGTHS = [16, 18, 24, 32, 36, 48, 64, 72, 96, 128, 144, 192, 256, 288, 384, 512, 576, 768]
CUBES = [16, 24, 32, 48, 64, 96, 128, 192, 256, 384, 512]


def _run(name, n, box, order, lattice="sc", plt=False, prec="f32", particles=False, baryons=False, z=24.0):
    c = {"kind": "run", "n": n, "box": box, "order": order, "lattice": lattice, "plt": plt, "prec": prec,
         "particles": particles, "baryons": baryons, "z": z}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the small box of the parity tests: a parameter scan or a check on a
        # laptop-sized grid, where launches and latency count
        _run("run_64_2lpt_f64", 64, 100.0, 2, prec="f64", z=49.0),
        # an ordinary box with component fields, in single precision
        _run("run_256_3lpt_f32", 256, 500.0, 3),
        # the benchmark: a production box with lattice corrections and two
        # particles per cell; the particles are handed on in 32 bits, as the
        # Gadget files hold them
        _run("run_512_3lpt_plt_bcc_f32", 512, 1000.0, 3, lattice="bcc", plt=True, particles=True),
        # a hydrodynamics box in double precision (the SWIFT files hold 64
        # bits): dark matter and baryons on a face-centred load
        _run("run_192_3lpt_fcc_gas_f64", 192, 200.0, 3, lattice="fcc", prec="f64", particles=True, baryons=True),
        # an ensemble: boxes of three sizes in one graph launch
        {"name": "batch_128_256_2lpt_f32", "kind": "batch", "n": 128, "count": 6, "box": 400.0, "prec": "f32"},
        # one step of an inference loop over the initial noise
        {"name": "adjoint_256_f32", "kind": "adjoint", "n": 256, "box": 500.0, "prec": "f32"},
        # the source block alone, in double precision
        {"name": "sources_192_f64", "kind": "sources", "n": 192, "order": 3, "box": 300.0, "prec": "f64"},
        # code written against the reference's convolver, product by product
        {"name": "products_192_f32", "kind": "products", "n": 192, "box": 300.0, "prec": "f32"},
        # a small transform pair, where launches count, and a large one on
        # axes of unequal length
        {"name": "poisson_64_f64", "kind": "poisson", "n0": 64, "n1": 64, "n2": 64, "box": 64.0, "prec": "f64"},
        {"name": "poisson_576x384x288_f32", "kind": "poisson", "n0": 576, "n1": 384, "n2": 288, "box": 100.0,
         "prec": "f32"},
        # the noise field by itself, as a constrained-noise or restart tool
        # asks for it
        {"name": "noise_256_f64", "kind": "noise", "n": 256, "prec": "f64"},
        # Eulerian output of a run for a grid-based code
        {"name": "ppt_192_f64", "kind": "ppt", "n": 192, "box": 100.0, "z": 24.0, "order": 2, "prec": "f64"},
    ]


def _log_choice(rng, sizes):
    """an entry of `sizes`, its logarithm spread evenly over their range"""
    at = math.exp(rng.uniform(math.log(sizes[0]), math.log(sizes[-1])))
    return min(sizes, key=lambda s: abs(math.log(s / at)))


def draw(rng):
    kind = rng.choice(["run", "run", "run", "batch", "adjoint", "sources", "products", "poisson", "noise", "ppt"])
    box = round(math.exp(rng.uniform(math.log(60.0), math.log(1500.0))), 2)
    prec = rng.choice(["f32", "f64"])
    if kind == "run":
        lattice = rng.choice(["sc", "sc", "bcc", "fcc"])
        particles = lattice != "sc" or rng.random() < 0.5
        baryons = particles and rng.random() < 0.25
        plt = particles and rng.random() < 0.4
        top = 512 if prec == "f32" and lattice != "fcc" and not baryons else 384 if lattice == "sc" and not baryons else 256
        n = _log_choice(rng, [s for s in CUBES if 32 <= s <= top])
        return _run(None, n, box, rng.choice([1, 2, 3, 3]), lattice, plt, prec, particles, baryons,
                    round(rng.uniform(15.0, 99.0), 2))
    if kind == "batch":
        n = _log_choice(rng, [32, 64, 128])
        return {"kind": kind, "n": n, "count": rng.randint(2, 9), "box": box, "prec": prec}
    if kind == "adjoint":
        return {"kind": kind, "n": _log_choice(rng, [s for s in CUBES if s <= 256]), "box": box, "prec": prec}
    if kind in ("sources", "products"):
        c = {"kind": kind, "n": _log_choice(rng, [s for s in CUBES if s <= (384 if kind == "sources" else 256)]),
             "box": box, "prec": prec}
        return dict(c, order=rng.choice([2, 3])) if kind == "sources" else c
    if kind == "poisson":
        most = 2 ** 27 if prec == "f32" else 2 ** 26
        while True:
            n0, n1, n2 = (_log_choice(rng, LENGTHS) for _ in range(3))
            if n0 * n1 * n2 <= most:
                return {"kind": kind, "n0": n0, "n1": n1, "n2": n2, "box": box, "prec": prec}
    if kind == "noise":
        return {"kind": kind, "n": rng.choice([n for n in LENGTHS if n <= 384]), "prec": prec}
    # FP32 phases of order 100 radians lose too much: the fields are made in FP64
    return {"kind": "ppt", "n": _log_choice(rng, [s for s in CUBES if s <= 256]), "box": box,
            "z": round(rng.uniform(15.0, 60.0), 2), "order": rng.choice([1, 2]), "prec": "f64"}


# ------------------------------------------------------------------ sizes --

def _transform_flops(points, count):
    return 2.5 * points * math.log2(points) * count


def _pipeline_flops(n, order):
    """padded transforms of the LPT sources (each Hessian and product once)"""
    per = {1: 0, 2: 6 + 1, 3: 6 + 5 + 4 + 6 + 4}[order]
    return _transform_flops((1.5 * n) ** 3, per) if per else 0.0


def work(case):
    s = 8 if case["prec"] == "f64" else 4
    kind = case["kind"]
    if kind == "poisson":
        cells = case["n0"] * case["n1"] * case["n2"]
        return {"bytes": 2.0 * cells * s, "flops": _transform_flops(cells, 2) + 6.0 * cells}
    n = case["n"]
    cells = float(n) ** 3
    if kind == "run":
        nsub = {"sc": 1, "bcc": 2, "fcc": 4}[case["lattice"]] * (2 if case["baryons"] else 1)
        out = cells * 6 * nsub * s
        return {"bytes": 4.0 * n * n + out, "flops": _pipeline_flops(n, case["order"]) + _transform_flops(cells, 6 * nsub)}
    if kind == "batch":
        bytes_, flops = 0.0, 0.0
        for i in range(case["count"]):
            m = _batch_size(n, i)
            bytes_ += 4.0 * m * m + 6.0 * m ** 3 * s
            flops += _pipeline_flops(m, 2) + _transform_flops(m ** 3, 6)
        return {"bytes": bytes_, "flops": flops}
    if kind == "adjoint":
        return {"bytes": 8.0 * cells * s, "flops": 3 * _pipeline_flops(n, 2) + _transform_flops(cells, 9)}
    if kind == "sources":
        outs = 1 if case["order"] == 2 else 5
        return {"bytes": (1.0 + outs) * cells * s, "flops": _pipeline_flops(n, case["order"])}
    if kind == "products":
        return {"bytes": 3.0 * cells * s, "flops": _transform_flops((1.5 * n) ** 3, 6 + 1 + 3)}
    if kind == "noise":
        # 202 subtractions with borrow per 12 numbers, two numbers per mode
        return {"bytes": 4.0 * n * n + cells * s, "flops": cells / 2 * 2 * 202 / 12 * 4}
    return {"bytes": (1.0 + 4.0) * cells * s, "flops": _transform_flops(cells, 2 + 2 * 2 + 2)}


# ---------------------------------------------------------------- prepare --

class _DeviceArray:
    """a device buffer of the library as an array torch can look at; keeps the
    owner of the memory alive"""

    def __init__(self, ptr, shape, double, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": tuple(shape),
                                         "typestr": "<f8" if double else "<f4", "version": 2}


def _tensor(ptr, shape, double, owner):
    return torch.as_tensor(_DeviceArray(ptr, shape, double, owner), device="cuda")


def _view(grid, owner=None):
    """the whole buffer of a grid, [n0][n1][n2 + 2]"""
    return _tensor(grid.device_ptr(), grid.shape_real, grid.prec == F64, owner or grid)


def _kview(grid, owner=None):
    v = _view(grid, owner)
    return torch.view_as_complex(v.reshape(grid.n[0], grid.n[1], grid.nc, 2))


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)


def _random_real(shape, seed):
    return torch.randn(shape, generator=_generator(seed), device="cuda", dtype=torch.float64)


def _noise_seed(seed):
    return 12345 + int(seed) % 2000000000


def _potential(n, seed):
    """a Gaussian potential with a falling spectrum and empty Nyquist planes,
    unitary half spectrum in 64 bits"""
    w = torch.fft.rfftn(_random_real((n, n, n), seed), norm="ortho")
    k2 = sum(k * k for k in _modes(n, w.device))
    phi = w * torch.where(k2 > 0, k2, torch.ones_like(k2)) ** -1.5
    return _no_nyquist(phi * (k2 > 0))


def _batch_size(n, i):
    return (n, 3 * n // 2, 2 * n)[i % 3]


def _lattice(case):
    return {"sc": SC, "bcc": BCC, "fcc": FCC}[case["lattice"]]


def prepare(case, seed):
    kind, prec = case["kind"], F64 if case["prec"] == "f64" else F32
    ctx = Context(0)
    s = {"case": case, "ctx": ctx, "prec": prec}
    if kind == "run" or kind == "ppt":
        run = kind == "run"
        cfg = lpt.ICConfig(n=case["n"], box=case["box"], zstart=case["z"], lpt_order=case["order"],
                           lattice=_lattice(case) if run else SC, plt=run and case["plt"], prec=prec,
                           seed=_noise_seed(seed), particles=run and case["particles"],
                           baryons=run and case["baryons"])
        s["run"] = lpt.ICRun(ctx, cfg)
        if not run:
            s["run"].execute()
            s["out"] = [Grid(ctx, (case["n"],) * 3, (case["box"],) * 3, prec=prec) for _ in range(4)]
    elif kind == "batch":
        boxes = [(_batch_size(case["n"], i), _noise_seed(seed * 16 + i), case["box"] * (1.0 + 0.1 * i))
                 for i in range(case["count"])]
        s["batch"] = Batch(ctx, boxes, lpt_order=2, prec=prec, zstart=24.0, tune=False)
        s["batch"].capture()
    elif kind == "adjoint":
        n = case["n"]
        s["plan"] = LPT2(ctx, n, case["box"], prec=prec, zstart=24.0)
        dtype = torch.float64 if prec == F64 else torch.float32
        s["noise"] = _random_real((n, n, n), seed).to(dtype).requires_grad_(True)
        s["cot"] = _random_real((3, n, n, n), seed + 1).to(dtype)
    elif kind == "poisson":
        shape = (case["n0"], case["n1"], case["n2"])
        side = [case["box"] * m / shape[0] for m in shape]
        s["rho"], s["phi"] = Grid(ctx, shape, side, prec=prec), Grid(ctx, shape, side, prec=prec)
        ctx.sync()
        _view(s["rho"])[:, :, :shape[2]] = _random_real(shape, seed)
    elif kind == "noise":
        s["seed"] = _noise_seed(seed)
        s["grid"] = Grid(ctx, (case["n"],) * 3, (1.0,) * 3, prec=prec)
    else:
        n = case["n"]
        grids = {"products": 3, "sources": 2 if case.get("order") == 2 else 6}[kind]
        s["grids"] = [Grid(ctx, (n,) * 3, (case["box"],) * 3, prec=prec, space=KSPACE) for _ in range(grids)]
        ctx.sync()
        _kview(s["grids"][0]).copy_(_potential(n, seed))
        if kind == "products":
            s["conv"] = lpt.OrszagConvolver(ctx, (n,) * 3, (case["box"],) * 3, prec=prec)
    torch.cuda.synchronize()
    return s


# -------------------------------------------------------------------- run --

def _particles(s, baryons):
    run, n = s["run"], s["case"]["n"]
    pos, vel, count = run.particles_device(baryons=baryons)
    out = [_tensor(p, (count, 3), True, run) for p in (pos, vel)]
    return out if s["prec"] == F64 else [t.to(torch.float32) for t in out]


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    if kind == "run":
        r, n = s["run"], case["n"]
        r.execute()
        if case["particles"]:
            return [_particles(s, False)] + ([_particles(s, True)] if case["baryons"] else [])
        return [_view(r.field(c), r)[:, :, :n] for c in range(6)]
    if kind == "batch":
        b = s["batch"]
        b.launch()
        return [[_view(r.field(c), r)[:, :, :r.cfg.n] for c in range(6)] for r in b.runs]
    if kind == "adjoint":
        x = s["noise"]
        x.grad = None
        psi = lpt2_map(x, s["plan"])
        psi.backward(s["cot"])
        return [psi.detach(), x.grad]
    if kind == "poisson":
        phi = s["phi"]
        phi.copy_from(s["rho"])
        phi.FourierTransformForward()
        phi.apply_InverseLaplacian()
        phi.FourierTransformBackward()
        return _view(phi)[:, :, :case["n2"]]
    if kind == "noise":
        lpt.ngenic_fill(s["grid"], s["seed"])
        return _kview(s["grid"])
    if kind == "sources":
        g = s["grids"]
        lpt.lpt_sources(s["ctx"], case["order"], *(g if case["order"] == 2 else (g[0], g[1], g[2], g[3:])))
        return [_kview(x) for x in g[1:]]
    if kind == "products":
        phi, phi2, cubic = s["grids"]
        conv = s["conv"]
        conv.convolve_SumOfHessians(phi, [0, 0], phi, [1, 1], [2, 2], lpt.assign_to(phi2))
        conv.convolve_Hessians(phi, [1, 1], phi, [2, 2], lpt.add_to(phi2))
        conv.convolve_Hessians(phi, [0, 1], phi, [0, 1], lpt.subtract_from(phi2))
        conv.convolve_Hessians(phi, [0, 2], phi, [0, 2], lpt.subtract_from(phi2))
        conv.convolve_Hessians(phi, [1, 2], phi, [1, 2], lpt.subtract_from(phi2))
        phi2.apply_InverseLaplacian()
        conv.convolve_Hessians(phi, [0, 0], phi, [1, 1], phi, [2, 2], lpt.assign_to(cubic))
        return [_kview(phi2), _kview(cubic)]
    hbar = ctypes.c_double()
    _lib.call("mfic_ppt_fields", s["run"].h, 1.0, *[g.h for g in s["out"]], ctypes.byref(hbar))
    return [_view(g)[:, :, :case["n"]] for g in s["out"]] + [hbar.value]


# ------------------------------------------------------------------ exact --
# 64-bit restatement of the paths in plain torch and numpy.

def _signed(n, device, gradient):
    k = torch.arange(n, device=device, dtype=torch.float64)
    k = torch.where(k > n // 2, k - n, k)
    return torch.where(k == n // 2, torch.zeros_like(k), k) if gradient else k


def _modes(n, device, gradient=False):
    """integer wave numbers of a cubic half spectrum; with `gradient`, 0 at n/2"""
    k = _signed(n, device, gradient)
    return k[:, None, None], k[None, :, None], k[None, None, : n // 2 + 1]


def _no_nyquist(f):
    n, h = f.shape[0], f.shape[0] // 2
    f = f.clone()
    f[h], f[:, h], f[:, :, n // 2] = 0, 0, 0
    return f


def _source_index(n, device):
    i = torch.arange(n, device=device)
    return torch.where(i > n // 2, i + n // 2, i)


def _pad(f):
    """unitary half spectrum of an n^3 grid -> real field on the 3/2 grid"""
    n, m = f.shape[0], 3 * f.shape[0] // 2
    at = _source_index(n, f.device)
    p = torch.zeros((m, m, m // 2 + 1), dtype=f.dtype, device=f.device)
    p[at[:, None], at[None, :], : n // 2 + 1] = f * 1.5 ** 1.5
    return torch.fft.irfftn(p, s=(m, m, m), norm="ortho")


def _unpad(x):
    n = 2 * x.shape[0] // 3
    at = _source_index(n, x.device)
    f = torch.fft.rfftn(x, norm="ortho")[at[:, None], at[None, :], : n // 2 + 1] / 1.5 ** 1.5
    return _no_nyquist(f)


def _hessians(f, box):
    g = [k * (2 * math.pi / box) for k in _modes(f.shape[0], f.device, True)]
    return [_pad(-(g[a] * g[b]) * f) for a, b in ((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2))]


def _inverse_laplacian(f, box):
    k2 = sum(k * k for k in _modes(f.shape[0], f.device)) * (2 * math.pi / box) ** 2
    out = -f / torch.where(k2 > 0, k2, torch.ones_like(k2))
    out[0, 0, 0] = 0
    return out


def _second_order(a):
    return a[0] * (a[1] + a[2]) + a[1] * a[2] - a[3] ** 2 - a[4] ** 2 - a[5] ** 2


def _exact_sources(phi1, box, order):
    a = _hessians(phi1, box)
    phi2 = _inverse_laplacian(_unpad(_second_order(a)), box)
    if order == 2:
        return [phi2]
    b = _hessians(phi2, box)
    q = [_pad(_unpad(x)) for x in (a[0] * a[1] - a[3] ** 2, a[3] * a[4], a[5] ** 2, a[4] ** 2)]
    third = (q[0] * a[2] + 2 * q[1] * a[5] - q[2] * a[0] - q[3] * a[1]
             - 5.0 / 7.0 * (a[0] * (b[1] + b[2]) + a[1] * (b[2] + b[0]) + a[2] * (b[0] + b[1]))
             + 10.0 / 7.0 * (a[3] * b[3] + a[4] * b[4] + a[5] * b[5]))
    curl = [b[3] * a[4] - b[4] * a[3] + a[5] * (b[1] - b[2]) - b[5] * (a[1] - a[2]),
            b[5] * a[3] - b[3] * a[5] + a[4] * (b[2] - b[0]) - b[4] * (a[2] - a[0]),
            b[4] * a[5] - b[5] * a[4] + a[3] * (b[0] - b[1]) - b[3] * (a[0] - a[1])]
    return [phi2] + [_inverse_laplacian(_unpad(x), box) for x in [third] + curl]


_MASK = (1 << 48) - 1


def _luxury_cycle(x, c):
    """202 subtract-with-borrow steps of RANLUX; the 12 newest words, oldest first"""
    for step in range(202):
        i = step % 12
        d = x[(i + 7) % 12] + (1 << 48) - x[i] - c
        c = 1 - (d >> 48)
        x[i] = d & _MASK
    return x[10:] + x[:10], c


def _luxury_seed(seed, zero):
    bits, x = [(seed >> b) & 1 for b in range(31)], []
    i, j = 0, 18
    for _ in range(12):
        w = zero
        for _ in range(48):
            w = 2 * w + (1 - bits[i])
            bits[i] = bits[i] ^ bits[j]
            i, j = (i + 1) % 31, (j + 1) % 31
        x.append(w)
    return x


def _seed_table(seed, n):
    x, c, at, out = _luxury_seed(seed or 1, 0), 0, 12, np.zeros((n, n), dtype=np.int64)

    def number():
        nonlocal x, c, at
        if at == 12:
            (x, c), at = _luxury_cycle(x, c), 0
        at += 1
        return int(2147483647.0 * (x[at - 1] / 281474976710656.0))

    for i in range(n // 2):
        e, f = n - 1 - i, lambda j: n - 1 - j  # noqa: E731
        for count, cell in ((i, lambda j: (i, j)), (i + 1, lambda j: (j, i)), (i, lambda j: (e, j)),
                            (i + 1, lambda j: (f(j), i)), (i, lambda j: (i, f(j))), (i + 1, lambda j: (j, e)),
                            (i, lambda j: (e, f(j))), (i + 1, lambda j: (f(j), e))):
            for j in range(count):
                out[cell(j)] = number()
    return out


def _exact_noise(n, seed, device="cuda"):
    table = torch.from_numpy(_seed_table(seed, n)).to(device)
    zero = torch.zeros_like(table)
    x, c, at = _luxury_seed(torch.where(table == 0, 1, table), zero), zero, 12

    def number():
        nonlocal x, c, at
        if at == 12:
            (x, c), at = _luxury_cycle(x, c), 0
        at += 1
        return x[at - 1].double() / 281474976710656.0

    h = n // 2
    f = torch.zeros((n, n, h + 1), dtype=torch.complex128, device=device)
    for k in range(h + 1):
        phase, ampl = number() * 2 * math.pi, number()
        f[:, :, k] = torch.polar(torch.sqrt(-torch.log(ampl)), phase)
    # kz = 0: one half plane is drawn, the other its mirror
    drawn = torch.zeros((n, n), dtype=torch.bool, device=device)
    drawn[:h], drawn[0] = True, False
    drawn[0, 1:h] = True
    plane = torch.where(drawn, f[:, :, 0], torch.zeros_like(f[:, :, 0]))
    plane[h], plane[:, h] = 0, 0
    back = -torch.arange(n, device=device) % n
    f[:, :, 0] = torch.where(plane != 0, plane, plane[back][:, back].conj())
    return _no_nyquist(f)


def _cosmology(z):
    """growth D+ and its velocity factor at z and the Eisenstein & Hu amplitude
    k^(n_s/2) T(k), normalised to sigma_8, of the default parameters"""
    p = lpt.baseline_cosmology(z)
    h, pi, c = p.H0 / 100.0, math.pi, 2.99792458e8
    sigma = pi ** 2 * 1.38064852e-23 ** 4 / 60.0 / 1.054571800e-34 ** 3 / c ** 2
    rho = 3e10 / (8 * pi * 6.6740800e-11) / 3.0857e22 ** 2
    gamma = 4 * sigma / c ** 3 * p.Tcmb ** 4 / rho / h ** 2
    radiation = gamma * (1 + p.N_ur * 7.0 / 8.0 * (4.0 / 11.0) ** (4.0 / 3.0))
    dark = 1.0 - p.Omega_m - radiation

    def hubble(a):
        return p.H0 * math.sqrt(radiation / a ** 4 + p.Omega_m / a ** 3 + dark)

    def rate(x, y):
        a = math.exp(x)
        ah = a * hubble(a)
        return y[1] / ah, -y[1] + 1.5 * p.Omega_m * p.H0 ** 2 * y[0] / (a * ah)

    def grow(y, x0, x1, steps):
        e = (x1 - x0) / steps
        for i in range(steps):
            x = x0 + i * e
            k1 = rate(x, y)
            k2 = rate(x + e / 2, [u + e / 2 * v for u, v in zip(y, k1)])
            k3 = rate(x + e / 2, [u + e / 2 * v for u, v in zip(y, k2)])
            k4 = rate(x + e, [u + e * v for u, v in zip(y, k3)])
            y = [u + e / 6 * (a + 2 * b + 2 * d + g) for u, a, b, d, g in zip(y, k1, k2, k3, k4)]
        return y

    x0, xs = math.log(1e-10), -math.log(1.0 + z)
    start = grow([1e-10, 0.0], x0, xs, 12000)
    now = grow(start, xs, 0.0, 3000)
    a = math.exp(xs)
    growth = start[0] / now[0]
    vfac = start[1] / start[0] / h  # f a H / h

    om, fb, th = p.Omega_m * h * h, p.Omega_b / p.Omega_m, p.Tcmb / 2.7
    ob = om * fb
    zeq, keq = 2.50e4 * om / th ** 4, 0.0746 * om / th ** 2
    zd = (1291 * om ** 0.251 / (1 + 0.659 * om ** 0.828)
          * (1 + 0.313 * om ** -0.419 * (1 + 0.607 * om ** 0.674) * ob ** (0.238 * om ** 0.223)))
    rd, req = 31.5 * ob / th ** 4 * (1000 / (1 + zd)), 31.5 * ob / th ** 4 * (1000 / zeq)
    sound = 2 / 3 / keq * math.sqrt(6 / req) * math.log((math.sqrt(1 + rd) + math.sqrt(rd + req)) / (1 + math.sqrt(req)))
    silk = 1.6 * ob ** 0.52 * om ** 0.73 * (1 + (10.4 * om) ** -0.95)
    ac = ((46.9 * om) ** 0.670 * (1 + (32.1 * om) ** -0.532)) ** -fb * ((12.0 * om) ** 0.424 * (1 + (45.0 * om) ** -0.582)) ** -fb ** 3
    bc = 1 / (1 + 0.944 / (1 + (458 * om) ** -0.708) * ((1 - fb) ** ((0.395 * om) ** -0.0266) - 1))
    y = zeq / (1 + zd)
    g = y * (-6 * math.sqrt(1 + y) + (2 + 3 * y) * math.log((math.sqrt(1 + y) + 1) / (math.sqrt(1 + y) - 1)))
    ab = 2.07 * keq * sound * (1 + rd) ** -0.75 * g
    node, bb = 8.41 * om ** 0.435, 0.5 + fb + (3 - 2 * fb) * math.sqrt((17.2 * om) ** 2 + 1)

    def transfer(kh):
        k = kh * h
        q, x = k / 13.41 / keq, k * sound
        lb, ln = torch.log(2.718282 + 1.8 * bc * q), torch.log(2.718282 + 1.8 * q)
        lo = 386.0 / (1 + 69.9 * q ** 1.08)
        f = 1 / (1 + (x / 5.4) ** 4)
        tc = f * lb / (lb + (14.2 + lo) * q * q) + (1 - f) * lb / (lb + (14.2 / ac + lo) * q * q)
        xt = k * sound * (1 + (node / x) ** 3) ** (-1.0 / 3.0)
        tb = torch.sin(xt) / xt * (ln / (ln + (14.2 + lo) * q * q) / (1 + (x / 5.2) ** 2)
                                   + ab / (1 + (bb / x) ** 3) * torch.exp(-(k / silk) ** 1.4))
        return fb * tb + (1 - fb) * tc

    lnk = torch.linspace(math.log(1e-4), math.log(1e4), (1 << 21) + 1, dtype=torch.float64)
    k = torch.exp(lnk)
    x = 8 * k
    w = torch.where(x < 1e-3, 1 - 0.1 * x * x, 3 * (torch.sin(x) - x * torch.cos(x)) / x ** 3)
    v = k ** (3 + p.n_s) * (w * transfer(k)) ** 2
    simpson = (v[0] + v[-1] + 4 * v[1:-1:2].sum() + 2 * v[2:-1:2].sum()) * (lnk[-1] - lnk[0]) / (len(v) - 1) / 3
    root = p.sigma_8 / math.sqrt(4 * pi * float(simpson))
    return growth, vfac, lambda kh: root * kh ** (0.5 * p.n_s) * transfer(kh)


def _linear_factor(n, box, amplitude, device="cuda"):
    """-A(k) / k^2 / volfac: phi1 per unit of white noise"""
    k2 = sum(k * k for k in _modes(n, device)) * (2 * math.pi / box) ** 2
    k2 = torch.where(k2 > 0, k2, torch.ones_like(k2))
    f = -amplitude(torch.sqrt(k2)) / k2 / (box / n / 2 / math.pi) ** 1.5
    f[0, 0, 0] = 0
    return f


def _exact_component_spectra(case, pots, growth, vfac):
    """displacement and velocity spectra (unit / L folded in) from phi1, phi2, ..."""
    n, box = case["n"], case["box"]
    g = [k * (2 * math.pi / box) for k in _modes(n, pots[0].device, True)]
    d, order = growth, case["order"]
    c = [-d, -3.0 / 7.0 * d * d, d ** 3 / 3.0]
    out = []
    for vel in (False, True):
        total = sum(c[o] * (vfac * (o + 1) if vel else 1.0) * pots[o] for o in range(order))
        for a in range(3):
            f = 1j * g[a] * total
            if order == 3:
                b, e = (a + 1) % 3, (a + 2) % 3
                f = f + d ** 3 / 7.0 * (3 * vfac if vel else 1.0) * (1j * g[b] * pots[3 + e] - 1j * g[e] * pots[3 + b])
            f = f / box
            f[0, 0, 0] = 0
            out.append(f)
    return out


def _exact_box(case, noise_seed):
    """the component fields of a run, or its particles"""
    n = case["n"]
    growth, vfac, amplitude = _cosmology(case.get("z", 24.0))
    pots = [_exact_noise(n, noise_seed) * _linear_factor(n, case["box"], amplitude)]
    if case["order"] > 1:
        pots += _exact_sources(pots[0], case["box"], case["order"])
    spectra = _exact_component_spectra(case, pots, growth, vfac)
    shape = (n, n, n)
    if not case.get("particles"):
        return [torch.fft.irfftn(f, s=shape, norm="ortho") for f in spectra]
    sub = {"sc": [(0, 0, 0)], "bcc": [(0, 0, 0), (0.5, 0.5, 0.5)],
           "fcc": [(0, 0, 0), (0, 0.5, 0.5), (0.5, 0, 0.5), (0.5, 0.5, 0)]}[case["lattice"]]
    second = (0.5, 0.5, 0.0) if case["lattice"] == "bcc" else (0.5, 0.5, 0.5)
    k = _modes(n, spectra[0].device)
    cell = torch.arange(n, device=spectra[0].device, dtype=torch.float64)
    species = []
    for base in ((0.0, 0.0, 0.0), second)[: 2 if case["baryons"] else 1]:
        pos, vel = [], []
        for w in sub:
            off = [base[a] + w[a] for a in range(3)]
            turn = torch.exp(2j * math.pi / n * sum(off[a] * k[a] for a in range(3)))
            fields = [torch.fft.irfftn(f * turn, s=shape, norm="ortho") for f in spectra]
            q = torch.meshgrid(*[(cell + off[a]) / n for a in range(3)], indexing="ij")
            pos.append(torch.stack([q[a] + fields[a] for a in range(3)], dim=-1).reshape(-1, 3))
            vel.append(torch.stack(fields[3:], dim=-1).reshape(-1, 3))
        species.append([torch.cat(pos), torch.cat(vel)])
    return species


def _exact_ppt(case, noise_seed):
    n, box = case["n"], case["box"]
    growth, vfac, amplitude = _cosmology(case["z"])
    phi1 = _exact_noise(n, noise_seed) * _linear_factor(n, box, amplitude)
    real = lambda f: torch.fft.irfftn(f, s=(n, n, n), norm="ortho")  # noqa: E731
    phi = real(phi1) * -growth
    phi2 = real(_exact_sources(phi1, box, 2)[0]) * (-3.0 / 7.0 * growth ** 2) if case["order"] > 1 else torch.zeros_like(phi)
    inner = phi[:-1]
    jump = max(float((x - inner).abs().max()) for x in
               (phi[1:], torch.roll(phi, -1, 1)[:-1], torch.roll(phi, -1, 2)[:-1]))
    hbar = jump / math.pi / growth * 1.01
    k = _signed(n, phi.device, False) * (2 * math.pi / box)
    k = [k[:, None, None], k[None, :, None], k[None, None, :]]
    psi = torch.polar(torch.ones_like(phi), (phi + phi2) / (hbar * growth))
    drift = torch.polar(torch.ones_like(phi), -0.5 * hbar * growth * sum(x * x for x in k))
    psi = torch.fft.ifftn(torch.fft.fftn(psi) * drift) * torch.polar(torch.ones_like(phi), phi2 / (hbar * growth))
    delta = psi.abs() ** 2 - 1
    spec = torch.fft.fftn(psi)
    out = [delta]
    for a in range(3):
        grad = torch.fft.ifftn(1j * k[a] * spec)
        out.append(growth * vfac / box * hbar * (psi.conj() * grad).imag / (1 + delta))
    return out + [hbar]


def exact(case, seed):
    kind = case["kind"]
    if kind == "poisson":
        shape = (case["n0"], case["n1"], case["n2"])
        f = torch.fft.rfftn(_random_real(shape, seed), norm="ortho")
        k2 = 0.0
        for a in range(3):
            k = _signed(shape[a], f.device, False) * (2 * math.pi / (case["box"] * shape[a] / shape[0]))
            k = k[: shape[a] // 2 + 1] if a == 2 else k
            k2 = k2 + (k * k).reshape([-1 if b == a else 1 for b in range(3)])
        k2[0, 0, 0] = 1.0
        f = -f / k2
        f[0, 0, 0] = 0
        return torch.fft.irfftn(f, s=shape, norm="ortho")
    if kind == "noise":
        return _exact_noise(case["n"], _noise_seed(seed))
    if kind == "run":
        # the lattice corrections' tables have no short form, and grids
        # over 256 no room beside the run's own
        return None if case["plt"] or case["n"] > 256 else _exact_box(case, _noise_seed(seed))
    if kind == "batch":
        return [_exact_box({"n": _batch_size(case["n"], i), "box": case["box"] * (1.0 + 0.1 * i), "order": 2},
                           _noise_seed(seed * 16 + i)) for i in range(case["count"])]
    if kind == "ppt":
        return _exact_ppt(case, _noise_seed(seed))
    n, box = case["n"], case["box"]
    # inputs are what the framework is given: rounded to its precision first
    given = torch.float64 if case["prec"] == "f64" else torch.float32
    if kind == "adjoint":
        growth, _, amplitude = _cosmology(24.0)
        factor = _linear_factor(n, box, amplitude)
        x = _random_real((n, n, n), seed).to(given).double().requires_grad_(True)
        cot = _random_real((3, n, n, n), seed + 1).to(given).double()
        keep = _no_nyquist(torch.ones_like(factor))
        phi1 = torch.fft.rfftn(x, norm="ortho") * keep * factor
        phi2 = _inverse_laplacian(_unpad(_second_order(_hessians(phi1, box))), box)
        total = -growth * phi1 - 3.0 / 7.0 * growth ** 2 * phi2
        g = [k * (2 * math.pi / box) for k in _modes(n, x.device, True)]
        psi = torch.stack([torch.fft.irfftn(1j * g[a] * total, s=(n, n, n), norm="ortho") for a in range(3)])
        psi.backward(cot)
        return [psi.detach(), x.grad]
    phi1 = _potential(n, seed)
    phi1 = torch.view_as_complex(torch.view_as_real(phi1).to(given).double())
    if kind == "sources":
        return _exact_sources(phi1, box, case["order"])
    a = _hessians(phi1, box)
    return [_inverse_laplacian(_unpad(_second_order(a)), box), _unpad(_pad(_unpad(a[0] * a[1])) * a[2])]
