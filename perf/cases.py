"""The workloads that the speed of this framework is measured on, through its public entry points.

A case names a call (what a program asks the framework for) and its sizes:

  thin         one Stokes I image of thin splats: thin_image (the march and the splat sums of one frame)
  image        one polarized image: polarized_image
  cube         a movie over observation times and frequencies: polarized_cube
  spacetime    the screen marched anew at a spin and inclination, and the image there: regenerate and polarized_cube,
               the step of a fit of (a, theta_o)
  gradient     the dual sweep from given image adjoints: polarized_gradient
  vis_fit      a fit iteration on visibilities: the splat constants of the current parameters, the forward pass, every
               slice's chi2 and seed, the reverse pass
  image_fit    a fit iteration on an image movie: fit.chi2_gradient
  graph_fit    the same iteration replayed as one captured graph: FitGraph.step
  visibilities the visibilities of rendered frames: visibilities

The splats are the seeded draws of kerrsplat_amd.synthetic (every seed another model), a movie's splats follow the
pattern rotation or, with knots, Keplerian orbits. precision "mixed" is the framework's FP32 transfer and dual sweep
over FP64 geodesics: what it computes are FP32 numbers, which its entry points hand back in FP64 arrays, so those
cases keep them in FP32; every other case's results stay FP64.
"""
import math

import numpy as np
import torch

import kerrsplat_amd as K
from kerrsplat_amd import synthetic as syn

FOV = 15.0               # half the screen's width [M]
NU = (230e9, 345e9, 86e9)
KNOT_TIMES = (-100.0, 0.0, 100.0, 200.0)

# defaults of a case's fields: call, model (thin, thermal, powerlaw, kappa, kappa_knots, composite), the marcher
# (recurrence: stored samples; direct: stored closed-form samples; fused: no stored samples), the precision policy, the
# screen (na x nb points, its centre `shift` M off the hole; screens: further screens in the same launch), N samples a
# ray, ns splats, nt frames x nnu frequencies, nuv baselines, nmax half orbits kept (-1: all)
DEFAULTS = dict(call="image", model="thermal", marcher="recurrence", precision="fp64", na=64, nb=64, shift=0.0, screens=0, N=256, ns=8,
                nt=1, nnu=1, nuv=0, nmax=-1, spin=0.9, theta_deg=60.0)


def _case(**fields):
    return {**DEFAULTS, **fields}


def listed():
    return [
        # the smallest call: a quick look at a thin model, marched inside the call (latency and launches)
        _case(name="thin-64-fused", call="thin", model="thin", marcher="fused", na=64, nb=64, N=512, ns=8, spin=0.94, theta_deg=17.0),
        # a small polarized image on an odd, off-centre screen, the inner loop of a sampler over few splats
        _case(name="image-50x37-6thermal", call="image", na=50, nb=37, shift=0.37, N=301, ns=6, spin=0.5),
        # an image of a cache that stores no samples, the first half orbits only (the direct image and the first ring)
        _case(name="image-96-fused-nmax", call="image", marcher="fused", na=96, nb=72, N=500, ns=16, nmax=1, spin=0.7, theta_deg=30.0),
        # a step of a fit of the spin and inclination: every ray marched anew, then the image
        _case(name="spacetime-128-32thermal", call="spacetime", na=128, nb=128, N=1024, ns=32, spin=0.5),
        # the fit step's gradient on one image, everything in FP64
        _case(name="gradient-128-32thermal", call="gradient", na=128, nb=128, N=1024, ns=32, spin=0.5),
        # the same of power-law splats on ragged sizes, two frames
        _case(name="gradient-102x67-48powerlaw", call="gradient", model="powerlaw", na=102, nb=67, shift=-0.21, N=333, ns=48, nt=2, spin=-0.6,
              theta_deg=40.0),
        # a fit iteration on the visibilities of four frames, the mixed policy
        _case(name="visfit-128-64thermal-mixed", call="vis_fit", precision="mixed", na=128, nb=128, N=1024, ns=64, nt=4, nuv=2048, spin=0.7,
              theta_deg=30.0),
        # small fit iterations, thousands of them in a fit: replayed as a captured graph
        _case(name="graphfit-64-16thermal-mixed", call="graph_fit", precision="mixed", na=64, nb=64, N=256, ns=16, nt=4, spin=0.7),
        # the large fit: kappa splats on orbits, one slice of its frames and frequencies, mixed
        _case(name="visfit-256-1024kappa-mixed", call="vis_fit", model="kappa_knots", precision="mixed", na=256, nb=256, N=1024, ns=1024,
              nuv=8192, theta_deg=163.0),
        # the same fit in FP64 on a coarser screen
        _case(name="visfit-112x96-1024kappa", call="vis_fit", model="kappa_knots", na=112, nb=96, N=512, ns=1024, nuv=4096, theta_deg=163.0),
        # a movie of mixed populations over several screens of uneven sizes in one launch, mixed
        _case(name="cube-5screens-128mixed-mixed", call="cube", model="composite", precision="mixed", na=128, nb=128, screens=4, N=512, ns=128,
              nt=4, nnu=3, theta_deg=45.0),
        # the visibilities of a movie's frames on a large screen and dense coverage
        _case(name="visibilities-512-8192uv", call="visibilities", na=512, nb=512, N=64, ns=8, nt=3, nuv=8192),
    ]


# Seconds a pass took when the ranges below were set, within a factor of a few: per ray-sample and frame, from the
# march, the per-sample work and the splats. It only bounds what draw() returns.
def _seconds(c):
    px = c["na"] * c["nb"] * (1 + 0.5 * c["screens"])
    rs = px * c["N"] * c["nt"] * c["nnu"]
    fp = 1.0 if c["precision"] == "fp64" else 0.25
    per = {"thin": 1.5, "thermal": 25.0, "powerlaw": 35.0, "composite": 45.0, "kappa": 60.0, "kappa_knots": 60.0}[c["model"]]
    adj = 3.5 if c["call"] in ("gradient", "vis_fit", "image_fit", "graph_fit") else 1.0
    t = 2e-4 + rs * 1e-12 * fp * adj * (100.0 + per * c["ns"])
    if c["marcher"] == "fused" or c["call"] == "spacetime":
        t += rs * 6e-10
    if c["nuv"]:
        t += c["nuv"] * c["na"] * c["nb"] * c["nt"] * c["nnu"] * 16 / 2e13
    return t


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: the calls as often as they are used, sizes over their logarithm, sizes that
    are no multiple of a wavefront or an anchor interval among them."""
    call = rng.choice(["thin", "image", "image", "cube", "spacetime", "gradient", "gradient", "vis_fit", "vis_fit", "image_fit", "graph_fit",
                       "visibilities"])
    c = _case(call=call)
    c["na"], c["nb"] = 2 * _log(rng, 12, 128), _log(rng, 24, 256)      # an even width keeps rays off the spin axis
    c["shift"] = round(rng.uniform(-0.5, 0.5), 3)
    c["N"] = _log(rng, 100, 1500)
    c["spin"] = round(rng.choice([1, 1, -1]) * rng.uniform(0.1, 0.97), 3)
    c["theta_deg"] = round(rng.choice([rng.uniform(15.0, 75.0), rng.uniform(110.0, 165.0)]), 2)
    c["precision"] = rng.choice(["fp64", "mixed"])
    c["marcher"] = rng.choice(["recurrence", "recurrence", "direct"])
    c["model"] = rng.choice(["thermal", "thermal", "powerlaw", "kappa", "kappa_knots", "composite"])
    c["ns"] = _log(rng, 4, 1100)
    if call == "thin":
        c["model"], c["marcher"], c["precision"] = "thin", rng.choice(["fused", "recurrence"]), "fp64"
    elif call in ("image", "cube", "spacetime"):
        if rng.random() < 0.3:
            c["marcher"], c["precision"] = "fused", "fp64"
        c["nmax"] = rng.choice([-1, -1, 1, 2])
    elif call in ("image_fit", "graph_fit") and c["model"] == "composite":
        c["model"] = "thermal"
    if call == "cube":
        c["nt"], c["nnu"], c["screens"] = rng.randint(1, 8), rng.randint(1, 3), rng.choice([0, 0, 2, 3])
    if call in ("gradient", "vis_fit", "image_fit", "graph_fit"):
        c["nt"] = rng.choice([1, 1, 2, 3, 5])
    if call == "vis_fit":
        c["nuv"] = _log(rng, 50, 8192)
    if call == "visibilities":
        c["model"], c["precision"], c["ns"], c["N"] = "thermal", "fp64", 8, 64
        c["na"], c["nb"], c["nt"], c["nuv"] = 2 * _log(rng, 16, 256), _log(rng, 32, 512), rng.randint(1, 4), _log(rng, 50, 8192)
    while _seconds(c) > 0.4:                      # no dearer than the listed ones
        k = max(("N", "ns", "nt"), key=lambda f: c[f] / {"N": 100, "ns": 16, "nt": 1.5}[f])
        c[k] = max(1, int(c[k] * 0.7))
    return c


# ---- inputs ------------------------------------------------------------------------------------------------------
def _camera(c):
    half = FOV * (c["nb"] - 1) / max(c["na"] - 1, 1)                   # square pixels
    s = c["shift"]
    cam = K.Camera((-FOV + s, FOV + s), (-half - s, half - s), (c["na"], c["nb"]))
    if not c["screens"]:
        return cam
    more = [K.Camera((-FOV, FOV), (-FOV, FOV), 2 * (c["na"] * (3 + q % 4) // 16)) for q in range(c["screens"])]
    return K.concatenate_screens(cam, *more)


def _knots(a, params, omega):
    """The centres at KNOT_TIMES on their circular orbits: (3, nknots, ns)."""
    x, y, z = params[0], params[1], params[2]
    ph = np.asarray(KNOT_TIMES)[:, None] * omega[None, :]
    return np.stack([x * np.cos(ph) - y * np.sin(ph), x * np.sin(ph) + y * np.cos(ph), np.broadcast_to(z, ph.shape)])


def _populations(c, seed):
    """[(kind, parameters, Model keywords)]: one population, or three parts of a composite."""
    a, single = c["spin"], c["nt"] == 1
    make = {"thin": syn.thin_splats, "thermal": syn.thermal_splats, "powerlaw": syn.powerlaw_splats, "kappa": syn.kappa_splats}

    def population(kind, n, s):
        P = make[kind](s, a, n) if kind == "thin" else make[kind](s, a, n, single_frame=single)
        return kind, np.asfortranarray(P), {}

    if c["model"] == "composite":
        n = [(c["ns"] + 2) // 3, (c["ns"] + 1) // 3, c["ns"] // 3]
        return [population(k, m, seed) for k, m in zip(("thermal", "powerlaw", "kappa"), n) if m > 0]
    kind, P, _ = population(c["model"].split("_")[0], c["ns"], seed)
    if c["model"] == "kappa_knots":
        return [(kind, P, {"knots": _knots(a, P, P[-1]), "knot_times": np.asarray(KNOT_TIMES)})]
    return [(kind, P, {})]


def _model(parts):
    models = [K.Model(P, kind=kind, **kw) for kind, P, kw in parts]
    return models[0] if len(models) == 1 else K.CompositeModel(*models)


_MARCHERS = {"recurrence": K.Recurrence, "direct": K.Direct, "fused": K.Fused}


def _blob(rng, cam):
    """An image-like (npix, 4) array of the size of the models' Stokes parameters: a ring and its polarization."""
    r = np.hypot(cam.alphas - rng.uniform(-1, 1), cam.betas - rng.uniform(-1, 1))
    ring = 1e-3 * np.exp(-0.5 * ((r - 5.5) / 1.5) ** 2)
    psi = np.arctan2(cam.betas, cam.alphas) + rng.uniform(0, math.pi)
    return np.stack([ring, 0.15 * ring * np.cos(2 * psi), 0.15 * ring * np.sin(2 * psi), 0.02 * ring], axis=-1)


def prepare(case, seed):
    c = {**DEFAULTS, **case}
    rng = np.random.default_rng(seed)
    cam = _camera(c)
    a, th = c["spin"], math.radians(c["theta_deg"])
    s = {"c": c, "cam": cam, "a": a, "th": th, "L": syn.length_unit(), "march": _MARCHERS[c["marcher"]]()}
    s["cache"] = cache = K.GeodesicCache(cam, c["N"], store_samples=c["marcher"] != "fused")
    K.regenerate(cache, a, th, marcher=s["march"])
    K.precision(cache, c["precision"])
    s["parts"] = _populations(c, seed)
    s["times"] = np.linspace(0.0, 10.0 * (c["nt"] - 1), c["nt"]) + rng.uniform(-5.0, 5.0)
    s["nus"] = np.asarray(NU[:c["nnu"]])
    s["psize"] = syn.pixel_size_rad(-FOV, FOV, c["na"])
    frames = c["nt"] * c["nnu"]
    shape = (c["na"], c["nb"], c["nt"], c["nnu"], 4)
    if c["call"] == "gradient":
        s["seeds"] = rng.normal(size=shape)
    if c["call"] in ("image_fit", "graph_fit"):
        blob = _blob(rng, cam)
        data = np.stack([blob * rng.uniform(0.8, 1.2) for _ in range(frames)], axis=1).reshape((c["na"], c["nb"]) + shape[2:], order="F")
        data = data + 1e-5 * rng.normal(size=shape)
        s["movie"] = K.StokesMovie(data, s["times"], s["nus"], np.full(4, 2e-5))
        if c["call"] == "graph_fit":
            s["graph"] = K.FitGraph(cache, s["times"], s["nus"], s["L"], image=(data, np.full(4, 2e-5)))
    if c["nuv"]:
        s["u"], s["v"] = syn.uv_disc(seed, c["nuv"])
        if c["call"] == "vis_fit":                 # a Gaussian source of 1 Jy, 40 uas wide, noise of 1%
            q2 = (s["u"] ** 2 + s["v"] ** 2) * (2 * math.pi * 40e-6 / 206264.8 / 2.355) ** 2
            stokes = np.array([1.0, 0.1, -0.05, 0.01])
            s["vis"] = [np.exp(-0.5 * q2)[:, None] * stokes + 0.01 * (rng.normal(size=(c["nuv"], 4)) + 1j * rng.normal(size=(c["nuv"], 4)))
                        for _ in range(frames)]
            s["sigma"] = np.full(4, 0.01)
    if c["call"] in ("cube", "spacetime", "graph_fit", "visibilities"):
        s["model"] = _model(s["parts"])
    if c["call"] == "visibilities":
        K.render_device(cache, s["model"], s["times"], s["nus"], s["L"])
    return s


def run(s):
    c, cache = s["c"], s["cache"]
    call = c["call"]
    # a program keeps the FP32 numbers of the mixed policy as such
    keep = (lambda x: x.astype(np.float32)) if c["precision"] == "mixed" else (lambda x: x)
    if call == "thin":
        return {"image": K.thin_image(cache, s["parts"][0][1], float(s["times"][0]))}
    if call == "image":                            # a new model each time, as in a sampler
        return {"image": keep(K.polarized_image(cache, _model(s["parts"]), float(s["times"][0]), float(s["nus"][0]), s["L"], nmax=c["nmax"], slab=0.5))}
    if call == "cube":
        return {"cube": keep(K.polarized_cube(cache, s["model"], s["times"], s["nus"], s["L"], nmax=c["nmax"], slab=0.5))}
    if call == "spacetime":
        K.regenerate(cache, s["a"], s["th"], marcher=s["march"])
        return {"cube": keep(K.polarized_cube(cache, s["model"], s["times"], s["nus"], s["L"], nmax=c["nmax"], slab=0.5))}
    if call == "visibilities":
        return {"vis": K.visibilities(cache, c["nt"] * c["nnu"], s["psize"], s["u"], s["v"])}
    if call == "graph_fit":
        chi, g = s["graph"].step(s["model"], s["parts"][0][1])
        return {"chi2": chi, "gradient": keep(g)}
    model = _model(s["parts"])                     # the constants of the iteration's parameters
    if call == "gradient":
        g, cube = K.polarized_gradient(cache, model, s["times"], s["nus"], s["L"], s["seeds"])
        return {"gradient": keep(g), "cube": keep(cube)}
    g = np.zeros(model.grad_shape, order="F")
    if call == "image_fit":
        chi = K.fit.chi2_gradient(g, model, s["movie"], cache, s["L"])
    else:
        K.gradient_forward(cache, model, s["times"], s["nus"], s["L"], copy=False)
        chi = sum(K.vis_chi2_seed(cache, f, s["psize"], s["u"], s["v"], vis, s["sigma"]) for f, vis in enumerate(s["vis"]))
        K.gradient_reverse(cache, model, g)
    return {"chi2": chi, "gradient": keep(g)}


# ---- what a pass cannot do without ----------------------------------------------------------------------------------
# Floating operations by the counted work of the formulas: per sample of a march 480; per step-taking sample (a third
# of them) 2000 for its geometry and Stokes step and 6000 for their adjoint; per (sample, splat) pair above the weight cutoff
# (one in twenty) the population's coefficients and their adjoint.
_PAIR = {"thin": (60, 0), "thermal": (200, 800), "powerlaw": (300, 1500), "kappa": (350, 1470), "kappa_knots": (350, 1470), "composite": (280, 1250)}


def work(case):
    c = {**DEFAULTS, **case}
    px = _camera(c).npix
    frames = c["nt"] * c["nnu"]
    rays = px * c["N"]
    rows = {"thin": 14, "thermal": 21}.get(c["model"], 22)
    call = c["call"]
    fit = call in ("gradient", "vis_fit", "image_fit", "graph_fit")
    vis_flops = 2 * (2 * c["nuv"]) * c["na"] * (4 * c["nb"]) * frames + 16 * c["nuv"] * c["nb"] * frames
    vis_bytes = 16 * c["nuv"] + 64 * c["nuv"] * frames
    image = 32 * px * frames
    if call == "visibilities":
        return {"bytes": image + vis_bytes, "flops": vis_flops}
    fwd, adj = _PAIR[c["model"]]
    flops = rays * frames * (fwd + (adj if fit else 0)) * c["ns"] / 20
    if call != "thin":
        flops += rays * frames / 3 * (8000 if fit else 2000)
    if c["marcher"] == "fused" or call == "spacetime":
        flops += rays * 480
    data = 16 * px + 8 * rows * c["ns"]                     # the screen and the parameters
    if c["marcher"] != "fused":
        data += 33 * rays                                   # t, r, theta, phi and the flags of every sample, read or written
    if call == "gradient":
        data += 2 * image + 8 * rows * c["ns"]
    elif fit:
        data += 8 * rows * c["ns"] + (vis_bytes + 96 * c["nuv"] * frames if call == "vis_fit" else image)
        flops += 2 * vis_flops
    else:
        data += image / (4 if call == "thin" else 1)
    return {"bytes": float(data), "flops": float(flops)}


# ---- the values in 64 bits ------------------------------------------------------------------------------------------
# For images of thin or thermal splats small enough to do in numpy: the geodesic equations in Mino time as regular
# polynomial ODEs (u = 1 / r and the direction n of the point on the sphere, no turning point or axis is special),
# Taylor series of order 16 from sample to sample, t and phi by Gauss-Legendre sums with the horizon's pole taken out,
# and the Stokes step as a matrix exponential.
ORDER = 16
GLX, GLW = np.polynomial.legendre.leggauss(8)


def _rf(x, y, z):
    """Carlson's R_F of complex arguments by duplication."""
    for _ in range(30):
        l = np.sqrt(x) * np.sqrt(y) + np.sqrt(y) * np.sqrt(z) + np.sqrt(z) * np.sqrt(x)
        x, y, z = (x + l) / 4, (y + l) / 4, (z + l) / 4
    return 1 / np.sqrt((x + y + z) / 3)


def _product(f, g, n):
    """Coefficient n of the product of two power series."""
    r = f[0] * g[n]
    for i in range(1, n + 1):
        r = r + f[i] * g[n - i]
    return r


def _series(u, v, n0, n1, A, kap, a):
    """The Taylor coefficients of u and of the direction (x, y, z) about a sample: u'' = U'(u) / 2 with
    U = 1 + A2 u^2 + A1 u^3 + A0 u^4, n'' = -(kap + 2 a^2 z^2) n + a^2 z e_z with kap = eta + lam^2."""
    U, D = [u, v], [[n0[q], n1[q]] for q in range(3)]
    U2, U3, Z2 = [], [], []
    for n in range(ORDER - 1):
        U2.append(_product(U, U, n))
        U3.append(_product(U2, U, n))
        Z2.append(_product(D[2], D[2], n))
        k = (n + 1) * (n + 2)
        U.append((A[0] * U[n] + 1.5 * A[1] * U2[n] + 2 * A[2] * U3[n]) / k)
        nxt = [-(kap * D[q][n] + 2 * a * a * _product(Z2, D[q], n)) / k for q in range(3)]
        nxt[2] = nxt[2] + a * a * D[2][n] / k
        for q in range(3):
            D[q].append(nxt[q])
    return U, D


def _at(f, h):
    r = f[-1]
    for x in f[-2::-1]:
        r = r * h + x
    return r


def _slope(f, h):
    return _at([i * x for i, x in enumerate(f)][1:], h)


def _rays(cam, a, th, N):
    """The samples 1..N of every ray in screen order: yields (t, r, cos theta, phi, nu_r, nu_theta, valid, dtau, lam, eta)."""
    al, be = cam.alphas, cam.betas
    st, ct = math.sin(th), math.cos(th)
    lam, eta = -al * st, (al * al - a * a) * ct * ct + be * be
    rp, rm = 1 + math.sqrt(1 - a * a), 1 - math.sqrt(1 - a * a)
    A = (a * a - lam * lam - eta, 2 * (eta + (lam - a) ** 2), -a * a * eta)
    roots = np.array([np.roots([1.0, 0.0, A[0][j], A[1][j], A[2][j]]) for j in range(len(al))]).T
    for _ in range(3):                                                  # Newton steps to full precision
        R = ((roots * roots + A[0]) * roots + A[1]) * roots + A[2]
        dR = (4 * roots * roots + 2 * A[0]) * roots + A[1]
        roots = roots - np.where(np.abs(dR) > 0, R / np.where(dR == 0, 1, dR), 0)
    real = np.abs(roots.imag) < 1e-9 * (1 + np.abs(roots))
    top = np.where(real, roots.real, -np.inf).max(axis=0)
    turns = top > rp
    end = 1 / np.where(turns, top, rp)
    X = np.sqrt((1 - roots * end).astype(complex))
    X[np.where(real, roots.real, -np.inf).argmax(axis=0)[turns], np.nonzero(turns)[0]] = 0
    W = [(X[0] * X[q] + X[r] * X[s]) / end for q, r, s in ((1, 2, 3), (2, 1, 3), (3, 1, 2))]
    fo = 2 * _rf(W[0] ** 2, W[1] ** 2, W[2] ** 2).real
    dtau = np.where(turns, 2 * fo, fo) / (N + 1)
    Pp, Pm = 2 * rp * (2 * rp - a * lam) / (rp - rm), -2 * rm * (2 * rm - a * lam) / (rp - rm)
    Qp, Qm = a * (2 * rp - a * lam) / (rp - rm), -a * (2 * rm - a * lam) / (rp - rm)
    up = 1 / rp
    kh = up / np.sqrt(np.abs(1 + up * up * (A[0] + up * (A[1] + up * A[2]))))
    u, v = np.zeros_like(al), np.ones_like(al)
    n0, n1 = [st + 0 * al, 0 * al, ct + 0 * al], [-be * ct, -al, be * st]
    t, ph, kap = 0 * al, 0 * al, eta + lam * lam
    for k in range(1, N + 1):
        U, D = _series(u, v, n0, n1, A, kap, a)
        ub, vb = _at(U, dtau), _slope(U, dtau)
        sg = np.where(_slope(U, dtau / 2) > 0, 1.0, -1.0)              # inward or outward: t + sg (r + 2 ln r) is regular
        w, f = 0 * al, 0 * al
        for x, g in zip(GLX, GLW):
            h = dtau * (1 + x) / 2
            uu, vv, cc = _at(U, h), _slope(U, h), _at(D[2], h)
            pole = np.where(turns, uu, uu - kh * vv) / (1 - rp * uu)
            inner = uu / (1 - rm * uu)
            rate = -(A[0] + uu * (A[1] + uu * A[2])) / (1 + sg * vv) * (1 + 2 * uu)
            w = w + g * (rate + 4 + Pp * pole + Pm * inner + a * a * cc * cc)
            f = f + g * (Qp * pole + Qm * inner)
        lg = np.where(turns, 0.0, -kh / rp * np.log(np.where(turns, 1.0, (1 - rp * ub) / (1 - rp * u))))
        F = lambda q: 1 / q - 2 * np.log(q)  # noqa: E731
        step = sg * F(ub) if k == 1 else sg * (F(ub) - F(u))
        t = t + w * dtau / 2 + Pp * lg - step
        m0 = [_at(D[q], dtau) for q in range(3)]
        m1 = [_slope(D[q], dtau) for q in range(3)]
        ph = ph + f * dtau / 2 + Qp * lg + np.arctan2(n0[0] * m0[1] - n0[1] * m0[0], n0[0] * m0[0] + n0[1] * m0[1])
        u, v, n0, n1 = ub, vb, m0, m1
        c = n0[2]
        # a point that a nearer part of the same polar orbit covers is not seen
        s2 = 1 - c * c
        hid = (c > abs(ct)) & (np.abs(al) >= a * np.sqrt(s2) + 2.2e-16)
        bb = np.sqrt(np.maximum((ct * ct - c * c) * (al * al - a * a * s2) / np.where(s2 > 0, -s2, -1), 0))
        ok = ~(hid & (np.abs(be) + 2.2e-16 < bb)) & (u > 0)
        before = k * dtau < fo * (1 - 1e-12)
        yield t, 1 / u, c, ph, np.where(turns, before, True), n1[2] > 0, ok, dtau, lam, eta


def _weights(P, a, t, r, c, ph):
    """The Gaussian exponent of every splat at the samples: (ns, samples)."""
    root = math.sqrt(1 - a * a)
    eps = np.finfo(float).eps
    pk = ph + a / (2 * root) * np.log(np.abs((r - 1 - root + eps) / (r - 1 + root + eps))) - np.arctan2(a, r)
    s = np.sqrt(1 - c * c)
    x, y, z = r * s * np.cos(pk), r * s * np.sin(pk), r * c
    p = P[:, :, None]
    an = p[-1] * (t - p[10])
    sp, cp = np.sin(an), np.cos(an)
    d0, d1, d2 = x - (p[0] * cp - p[1] * sp), y - (p[0] * sp + p[1] * cp), z - p[2]
    e = (d0 * cp + d1 * sp, -d0 * sp + d1 * cp, d2)
    qw, qx, qy, qz = p[6:10] / np.sqrt((p[6:10] ** 2).sum(axis=0))
    R = ((1 - 2 * (qy * qy + qz * qz), 2 * (qx * qy - qw * qz), 2 * (qx * qz + qw * qy)),
         (2 * (qx * qy + qw * qz), 1 - 2 * (qx * qx + qz * qz), 2 * (qy * qz - qw * qx)),
         (2 * (qx * qz - qw * qy), 2 * (qy * qz + qw * qx), 1 - 2 * (qx * qx + qy * qy)))
    g = ((t - p[10]) * np.exp(-p[11])) ** 2
    for b in range(3):
        g = g + ((R[0][b] * e[0] + R[1][b] * e[1] + R[2][b] * e[2]) * np.exp(-p[3 + b])) ** 2
    return g, d0 * d0 + d1 * d1 + d2 * d2


def _exact_thin(cam, c, P, a, th, t_obs):
    img = np.zeros(cam.npix)
    rp = 1 + math.sqrt(1 - a * a)
    for t, r, ct, ph, _, _, ok, dtau, lam, _ in _rays(cam, a, th, c["N"]):
        j = np.nonzero(ok & (r > rp * (1 + 1e-3)) & (r < 1e3))[0]
        g, _ = _weights(P, a, t_obs - t[j], r[j], ct[j], ph[j])
        S, D, s2 = r[j] ** 2 + (a * ct[j]) ** 2, r[j] ** 2 - 2 * r[j] + a * a, 1 - ct[j] ** 2
        Xi = (r[j] ** 2 + a * a) ** 2 - a * a * D * s2
        red = np.sqrt(D * S / Xi) / (1 - 2 * a * r[j] / Xi * lam[j])
        img[j] += red ** 2 * np.exp(P[12][:, None] - g / 2).sum(axis=0) * S * dtau[j]
    return img


ME, CL, EE, HPL = 9.1093826e-28, 2.99792458e10, 4.80320680e-10, 6.6260693e-27


def _bessel(x):
    """K0, K1 and K2 by the trapezoidal rule over exp(-x cosh s) cosh(n s)."""
    s = np.arange(0, 400) * 0.125
    with np.errstate(over="ignore", under="ignore"):
        e = np.exp(-x[:, None] * np.cosh(s)) * np.where(s == 0, 0.5, 1.0) * 0.125
    k0, k1 = e.sum(axis=1), (e * np.cosh(np.minimum(s, 40.0))).sum(axis=1)
    return k0, k1, k0 + 2 * k1 / x


def _thermal(ne, T, k, B, nu, sth, cth):
    """Dexter (2016) and Shcherbakov (2008) thermal synchrotron coefficients: jI, jQ, jV, aI, aQ, aV, rQ, rV."""
    w = 2 * np.pi * nu
    w0 = EE * B / (ME * CL) / w
    wp = 4 * np.pi * ne * EE * EE / ME / (w * w)
    x = T * np.sqrt(math.sqrt(2.0) * sth * 1e3 * w0)
    ext = (0.011 * np.exp(-x / 47.2) - 2 ** (-1 / 3) / 3 ** (23 / 6) * np.pi * 1e4 * (x + 1e-16) ** (-8 / 3)) * (0.5 + 0.5 * np.tanh(np.log(x / 120) / 0.1))
    f = 2.011 * np.exp(-x ** 1.035 / 4.7) - np.cos(x / 2) * np.exp(-x ** 1.2 / 2.73) - 0.011 * np.exp(-x / 47.2) + ext
    rQ = w / (2 * CL) * f * wp * w0 * w0 * (k[1] / k[2] + 6 * T) * sth * sth
    rV = w / CL * wp * w0 * (k[0] / k[2]) * (1 - 0.11 * np.log(1 + 0.035 * x)) * cth
    xs = nu / (3 * EE * B * sth / (4 * np.pi * ME * CL) * T * T + 1)
    y = xs ** (-1 / 3)
    e = np.exp(-1.8899 / y)
    pre = ne * EE * EE * nu / (2 * math.sqrt(3.0) * CL * T * T) * 2.5651 * e
    jI, jQ = pre * (1 + 1.92 * y + 0.9977 * y * y), pre * (1 + 0.93193 * y + 0.499873 * y * y)
    jV = 2 * ne * EE * EE * nu * cth / sth / (3 * math.sqrt(3.0) * CL * T ** 3) * (1.81384 / xs + 3.42319 * y * y + 0.0292545 / np.sqrt(xs) + 2.03773 * y) * e
    ib = np.expm1(HPL * nu / (ME * CL * CL * T)) / (2 * HPL * nu ** 3 / (CL * CL))
    return jI, jQ, jV, jI * ib, jQ * ib, jV * ib, rQ, rV


def _frame(a, r, c, lam, eta, nur, nuth, al, be, st_o, u, b):
    """1 + z, the cosine of the pitch angle and the polarization angle on the screen, for a fluid of ZAMO velocity u
    (axes r, phi, -theta) and field direction b."""
    s2 = 1 - c * c
    s = np.sqrt(s2)
    S, D = r * r + a * a * c * c, r * r - 2 * r + a * a
    Xi = (r * r + a * a) ** 2 - a * a * D * s2
    lapse, om = np.sqrt(D * S / Xi), 2 * a * r / Xi
    w = r * r + a * a - a * lam
    R = w * w - D * (eta + (lam - a) ** 2)
    Th = eta + a * a * c * c - lam * lam * c * c / s2
    pr = np.where(nur, 1, -1) * np.sqrt(np.where(R > 1e-14 * w * w, R, 0)) / D
    pt = np.where(nuth, 1, -1) * np.sqrt(np.maximum(Th, 0))
    p = (Xi / (D * S) - 2 * a * r / (D * S) * lam, D / S * pr, pt / S, 2 * a * r / (D * S) + (D - a * a * s2) / (D * S * s2) * lam)
    er, et, ep = np.sqrt(S / D), np.sqrt(S), s * np.sqrt(Xi / S)
    z0, z = lapse * p[0], (er * p[1], ep * (p[3] - om * p[0]), -et * p[2])
    g = np.sqrt(1 + u[0] ** 2 + u[1] ** 2 + u[2] ** 2)
    ud = u[0] * z[0] + u[1] * z[1] + u[2] * z[2]
    red = 1 / (g * z0 - ud)
    k = [(z[q] + u[q] * (ud / (g + 1) - z0)) * red for q in range(3)]
    cosb = k[0] * b[0] + k[1] * b[1] + k[2] * b[2]
    f = [k[1] * b[2] - k[2] * b[1], k[2] * b[0] - k[0] * b[2], k[0] * b[1] - k[1] * b[0]]
    n = np.sqrt(f[0] ** 2 + f[1] ** 2 + f[2] ** 2)
    f = [x / n for x in f]
    uf = u[0] * f[0] + u[1] * f[1] + u[2] * f[2]
    ft, fr, fth = uf / lapse, (f[0] + u[0] * uf / (g + 1)) / er, -(f[2] + u[2] * uf / (g + 1)) / et
    fp = (f[1] + u[1] * uf / (g + 1)) / ep + om * ft
    W1 = p[0] * fr - p[1] * ft + a * s2 * (p[1] * fp - p[3] * fr)
    W2 = ((r * r + a * a) * (p[3] * fth - p[2] * fp) - a * (p[0] * fth - p[2] * ft)) * s
    k1, k2 = W1 * r - W2 * a * c, -(W1 * a * c + W2 * r)
    mu = -(al + a * st_o)
    return red, cosb, np.arctan2(-(be * k2 - mu * k1), be * k1 + mu * k2)


def _exact_thermal(cam, c, P, a, th, t_obs, nu, L):
    n = cam.npix
    rp = 1 + math.sqrt(1 - a * a)
    T, B = np.exp(P[13]), np.exp(P[14])
    kb = _bessel(1 / T)
    bh = np.stack([np.sin(P[15]) * np.cos(P[16]), np.sin(P[15]) * np.sin(P[16]), np.cos(P[15])])
    tr, out = np.broadcast_to(np.eye(4), (n, 4, 4)).copy(), np.zeros((n, 4))
    cut = -2 * math.log(1e-6)
    smax = P[3:6].max(axis=0)
    for t, r, ct, ph, nur, nuth, ok, dtau, lam, eta in _rays(cam, a, th, c["N"]):
        j = np.nonzero(ok & (r > rp * (1 + 1e-3)) & (r < 100))[0]
        g, d2 = _weights(P, a, t_obs - t[j], r[j], ct[j], ph[j])
        G = np.exp(-g / 2)
        i, q = np.nonzero((G > 1e-6) & (d2 <= cut * np.exp(2 * smax)[:, None]))
        if not len(i):
            continue
        J = j[q]
        red, cosb, chi = _frame(a, r[J], ct[J], lam[J], eta[J], nur[J], nuth[J], cam.alphas[J], cam.betas[J], math.sin(th), P[17:20, i], bh[:, i])
        nf = nu / red
        cth = np.clip(cosb, -1, 1)
        jI, jQ, jV, aI, aQ, aV, rQ, rV = _thermal(np.exp(P[12][i]) * G[i, q], T[i], [k[i] for k in kb], B[i], nf, np.sqrt(1 - cth * cth), cth)
        nh = nf / 1e11
        fe = np.minimum(1, 0.99 * jI / np.hypot(jQ, jV))
        fa = np.minimum(1, 0.99 * aI / np.hypot(aQ, aV))
        c2, s2 = np.cos(2 * chi), np.sin(2 * chi)
        rows = [jI / nh ** 2, fe * jQ * c2 / nh ** 2, fe * jQ * s2 / nh ** 2, fe * jV / nh ** 2, aI * nh, fa * aQ * c2 * nh, fa * aQ * s2 * nh, fa * aV * nh,
                rQ * c2 * nh, rQ * s2 * nh, rV * nh]
        sums = np.stack([np.bincount(q, x, len(j)) for x in rows])
        at = np.unique(q)
        J, (j0, j1, j2, j3, a0, a1, a2, a3, r1, r2, r3) = j[at], sums[:, at]
        D = L / (nu / 1e11) * (r[J] ** 2 + (a * ct[J]) ** 2) * dtau[J]
        M = np.zeros((len(J), 5, 5))
        M[:, :4, :4] = -np.stack([a0, a1, a2, a3, a1, a0, r3, -r2, a2, -r3, a0, r1, a3, r2, -r1, a0], axis=-1).reshape(-1, 4, 4) * D[:, None, None]
        M[:, :4, 4] = np.stack([j0, j1, j2, j3], axis=-1) * D[:, None]
        scale = np.abs(M[:, :4, 4]).max(axis=1) + 1e-300                # the source column to order one
        M[:, :4, 4] /= scale[:, None]
        X = torch.linalg.matrix_exp(torch.from_numpy(M)).numpy()
        out[J] += np.einsum("nij,nj->ni", tr[J], X[:, :4, 4]) * scale[:, None]
        tr[J] = tr[J] @ X[:, :4, :4]
    return out * (nu / 1e11) ** 3


def exact(case, seed):
    """The image of a thin or thermal case that numpy does in some seconds. The other calls (gradients, mixed
    populations, large screens) take minutes or more written out like this; the visibilities transform frames that only
    the framework renders: None."""
    c = {**DEFAULTS, **case}
    cost = c["na"] * c["nb"] * c["N"] * (1 + c["ns"] / 8)
    if c["call"] not in ("thin", "image") or c["model"] not in ("thin", "thermal") or c["nmax"] >= 0 or cost > 6e6:
        return None
    rng = np.random.default_rng(seed)
    cam, a, th = _camera(c), c["spin"], math.radians(c["theta_deg"])
    P = _populations(c, seed)[0][1]
    t_obs = float(rng.uniform(-5.0, 5.0))                               # as prepare() draws it
    if c["call"] == "thin":
        return {"image": _exact_thin(cam, c, P, a, th, t_obs).reshape(cam.size, order="F")}
    img = _exact_thermal(cam, c, P, a, th, t_obs, NU[0], syn.length_unit())
    return {"image": img.reshape(cam.size + (4,), order="F")}
