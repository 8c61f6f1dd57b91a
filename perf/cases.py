"""The work that users of this package have it do, as a list of measurable
cases: ionization boxes of single redshifts, batches and sweeps, the steps
before and after the bubble finder, and the differentiable mode.

listed() are the cases, draw() gives more of the same ranges, prepare() makes
what a program holds before the call (device or host boxes from the seed, and
the context it keeps), run() is one pass through the public entry points,
work() the bytes and operations that no implementation can avoid, exact() the
same outputs in 64 bits from plain torch.

Inputs follow the recipe of the benchmark: a Gaussian field with P(k) ~
k^-2.5 and sigma 1.2 mapped to a lognormal density, point sources with
probability ~ (1 + delta)^2 and lognormal strengths, the emissivity scaled to
a fraction of the mean recombination rate (0.03-0.25: boxes between the first
bubbles and overlap, a mean x_HII of 0.2 to 0.9).
"""
import math

import numpy as np
import torch
import torch.utils.checkpoint

import simfast21_amd as sf

DEV = "cuda" if torch.cuda.is_available() else "cpu"
PI = 3.1415926535897932385
H0 = 3.24078e-18  # 1/s for h = 1

# sides with a register plan, and the other multiples of 8 that the finder
# takes (factors 2, 3, 5; the dilation's lanes tile the side)
PLAN = (64, 96, 128, 192, 256, 512)
COSMO = dict(hubble=0.71, omega_m=0.27, omega_b=0.046, omega_lambda=0.73)


def other_sides(lo, hi):
    out = []
    for n in range(lo, hi + 1, 8):
        m = n
        for p in (2, 3, 5):
            while m % p == 0:
                m //= p
        lanes = [q for q in range(1, 17) if n % q == 0 and n // q <= 64 and (n // q) % 8 == 0]
        if m == 1 and n not in PLAN and lanes:
            out.append(n)
    return out


def geometric(rmax, ratio, dx):
    radii, r = [], float(rmax)
    while r >= dx:
        radii.append(r)
        r *= ratio
    return radii


def ladder(case):
    """Descending radii of a finder case: R_max down to the cell size, either
    by the factor 0.9 or in `nbins` logarithmic steps (the ini's ladder)."""
    side, n = case["side"], case["n"]
    dx, rmax = side / n, case["rmax"]
    ratio = 10.0 ** (-math.log10(rmax / dx) / case["nbins"]) if case.get("nbins") else 0.9
    return geometric(rmax, ratio, dx)


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def finder(name, n, mode, side, rmax, frac, nbins=0, z=8.0, **more):
    return dict(name=name, kind="slice", n=n, mode=mode, side=side, rmax=rmax, nbins=nbins, frac=frac,
                z=z, **more)


def listed():
    return [
        # the smallest box a user runs: one redshift of a quick parameter
        # study, bound by launches and latency
        finder("slice_64", 64, "direct", 75.0, 18.75, 0.05),
        # an ordinary box in the reference's own mode (deltanl and SFRD boxes)
        finder("slice_128_sfr", 128, "sfr", 142.0, 42.6, 0.12),
        # one redshift as the drop-in program runs it: boxes in host memory
        finder("host_256_sfr", 256, "sfr", 213.0, 56.8, 0.12, host=True),
        # the headline configuration: redshift slices of 512^3, 47 radii,
        # resident in HBM, in one graph launch (the largest case)
        dict(name="batch_512", kind="batch", n=512, count=2, mode="direct", side=400.0, rmax=100.0, nbins=0,
             frac=0.05, z=8.0),
        # a small box whose side is not a power of two, with a residual
        # neutral fraction
        finder("slice_120", 120, "direct", 140.0, 35.0, 0.06, fresid=True),
        # the reference's sample ini: 600^3, 150 Mpc, h 0.71, R_max 60 Mpc in
        # 50 bins, deltanl and SFRD boxes
        finder("slice_600_sfr", 600, "sfr", 106.5, 42.6, 0.12, nbins=50, z=9.0),
        # a parameter sweep: boxes of uneven sides at one cell size in one
        # graph launch
        dict(name="sweep_64_256", kind="sweep", sides="64,128,96,256,64,192,128,96", cell=300.0 / 256, frac=0.06),
        # a training step of the differentiable mode: exact forward, relaxed
        # gradient, every output a loss can use
        dict(name="train_128", kind="train", n=128, side=200.0, rmax=60.0, nbins=0, frac=0.06, tau=0.05, pk=20),
        # brightness temperature of one redshift with the spin boxes
        dict(name="t21_256", kind="t21", n=256, side=213.0, axis=3, spin=True, z=9.0),
        # non-linear density: displacement deposit on the halo grid
        dict(name="nldensity_512", kind="nldensity", n=256, n_halo=512, side=213.0, z=9.0),
        # SFRD box of a halo catalog
        dict(name="sfrd_512", kind="sfrd", n=256, n_halo=512, side=213.0, halos=1000000, z=9.0),
        # power spectrum of a box
        dict(name="power_256", kind="power", n=256, side=300.0, pk=20),
    ]


def draw(rng):
    kind = rng.choice(["slice"] * 5 + ["sweep", "train", "t21", "nldensity", "sfrd", "power"])
    frac = round(math.exp(rng.uniform(math.log(0.03), math.log(0.25))), 4)
    cell = rng.uniform(0.4, 1.6)
    z = round(rng.uniform(6.5, 12.0), 2)

    def side_of(pool, lo, hi):
        """A side of the pool, spread evenly over the logarithm."""
        want = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        return min(pool, key=lambda n: abs(math.log(n / want)))

    if kind == "slice":
        n = side_of(sorted(PLAN + tuple(other_sides(64, 600))), 64, 600)
        mode = rng.choice(["direct", "sfr"])
        nbins = rng.choice([0, rng.randint(15, 45)])
        return dict(kind="slice", n=n, mode=mode, side=n * cell, rmax=n * cell * rng.uniform(0.15, 0.4),
                    nbins=nbins, frac=frac, z=z, host=n <= 256 and rng.random() < 0.2,
                    fresid=mode == "direct" and rng.random() < 0.3)
    if kind == "sweep":
        sides = [rng.choice([64, 80, 96, 120, 128, 160, 192, 256]) for _ in range(rng.randint(3, 10))]
        return dict(kind="sweep", sides=",".join(str(n) for n in sides), cell=cell, frac=frac)
    if kind == "train":
        n = rng.choice([64, 80, 96, 120, 128])
        return dict(kind="train", n=n, side=n * cell, rmax=n * cell * rng.uniform(0.2, 0.3), nbins=0, frac=frac,
                    tau=round(rng.uniform(0.02, 0.06), 4), pk=rng.randint(10, 24))
    if kind == "t21":
        n = side_of(sorted(PLAN + tuple(other_sides(64, 512))), 64, 512)
        return dict(kind="t21", n=n, side=n * cell, axis=rng.randint(1, 3), spin=rng.random() < 0.6, z=z)
    if kind == "power":
        n = side_of(sorted(PLAN + tuple(other_sides(64, 512))), 64, 512)
        return dict(kind="power", n=n, side=n * cell, pk=rng.randint(8, 40))
    n = rng.randint(50, 300)  # deposits take any side
    sm = rng.randint(1, 3)
    case = dict(kind=kind, n=n, n_halo=n * sm, side=n * cell, z=z)
    if kind == "sfrd":
        case["halos"] = int(10 ** rng.uniform(3.5, 6.3))
    return case


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def freq(n):
    return torch.arange(n, device=DEV, dtype=torch.int64).add(n // 2 - 1).remainder(n).sub(n // 2 - 1)


def gaussian(gen, n, slope=-2.5, sigma=1.2):
    spec = torch.fft.rfftn(torch.randn((n, n, n), generator=gen, device=DEV))
    f = freq(n).float() ** 2
    h = torch.arange(n // 2 + 1, device=DEV, dtype=torch.float32) ** 2
    k2 = f[:, None, None] + f[None, :, None] + h[None, None, :]
    spec *= torch.where(k2 > 0, k2.clamp_min(1.0) ** (slope / 4.0), torch.zeros_like(k2))
    del k2
    g = torch.fft.irfftn(spec, s=(n, n, n))
    del spec
    g = g.double()
    return ((g - g.mean()) * (sigma / g.std())).float()


def lognormal(g):
    e = torch.exp(g.double())
    return e / e.mean()


def sources(gen, delta1, count):
    """Point sources, about `count` of them, with probability ~ (1+delta)^2
    and lognormal strengths (float32)."""
    w = delta1 * delta1
    p = (w * (count / w.sum())).float()
    del w
    u = torch.rand(delta1.shape, generator=gen, device=DEV)
    hit = u < p
    del u, p
    return torch.where(hit, torch.exp(torch.randn(delta1.shape, generator=gen, device=DEV)),
                       torch.zeros((), device=DEV))


def physics(case):
    """Scalars of the SFR mode's cell pre-pass (64 bits)."""
    z, h = case["z"], COSMO["hubble"]
    e = -4.37152818e-05 * z ** 5 + 1.64394635e-03 * z ** 4 - 2.03044756e-02 * z ** 3 \
        + 7.18335221e-02 * z ** 2 - 8.85791388e-02 * z - 1.20887500e+01
    c_fres = 1.881e-7 * (1 + z) ** 3 * 4.19232273531e-13 / 10.0 ** e
    dvv = (case["side"] * 3.0857e24 / case["n"] / h / (1 + z)) ** 3
    k_rec = 1e-24 * 9.84815696 * (1 + z) ** 5.06773134 * dvv / 1e45
    qion = 10.0 ** (2.05707274e-02 * z + 5.29944413e+01) / 1e45
    k_ion = (case["side"] / case["n"]) ** 3 * qion * FESC
    return c_fres, k_rec, k_ion


FESC = 0.25


def prepass(case, a, b, c):
    """rec, ion and residual neutral fraction in 64 bits."""
    a, b = a.double(), b.double()
    if case["mode"] == "direct":
        return a, b, None if c is None else c.double()
    c_fres, k_rec, k_ion = physics(case)
    d = 1 + a
    x = (d / 1.76105133) ** 0.81722878
    r = d * c_fres
    return k_rec * (x / (1 + x)) ** 4, b * k_ion, 2 * r / (2 * r + 1 + torch.sqrt(4 * r + 1))


def finder_boxes(case, gen):
    """(a, b, c): the boxes of one redshift, float32, flat."""
    n = case["n"]
    delta1 = lognormal(gaussian(gen, n))
    count = 2.5e5 * (n / 512) ** 3 if n > 128 else 4000 * (n / 128) ** 3
    emis = sources(gen, delta1, max(count, 200))
    c = None
    if case["mode"] == "direct":
        a = (delta1 * delta1).float()
        if case.get("fresid"):
            c = (1e-4 * delta1).clamp_max(0.5).float().reshape(-1).contiguous()
        unit = float(a.double().mean())
    else:
        a = (delta1 - 1).float()
        rec, _, _ = prepass(case, a, a, None)
        unit = float(rec.mean()) / physics(case)[2]
    del delta1
    b = emis * (case["frac"] * unit / max(float(emis.double().mean()), 1e-30))
    return a.reshape(-1).contiguous(), b.reshape(-1).contiguous(), c


def sweep_cases(case):
    out = []
    for k, n in enumerate(int(v) for v in case["sides"].split(",")):
        side = n * case["cell"]
        out.append(dict(kind="slice", n=n, mode="direct", side=side, rmax=side / 4, nbins=0,
                        frac=case["frac"] * (0.85 + 0.05 * (k % 7)), z=8.0))
    return out


def train_boxes(case, gen):
    n = case["n"]
    g = gaussian(gen, n)
    delta1 = lognormal(g)
    emis = sources(gen, delta1, max(4000 * (n / 128) ** 3, 200))
    zeta = case["frac"] * float((delta1 * delta1).mean()) / float(emis.double().mean())
    return g.reshape(-1).contiguous(), emis.reshape(-1).contiguous(), zeta


def pk_weights(case, seed):
    """dL/dP_b of a loss on the binned power spectrum: order one over a
    smooth power law."""
    rng = np.random.default_rng(seed)
    n, nb = case["n"], case["pk"]
    k = 1 + (np.arange(nb) + 0.5) * (n / 2 - 1) / nb
    return rng.standard_normal(nb) * k ** 2.5 / (case["side"] ** 3 * 0.02)


def smooth_box(gen, n, amp, width=6.0):
    f = freq(n).float() / n
    h = torch.arange(n // 2 + 1, device=DEV, dtype=torch.float32) / n
    k2 = f[:, None, None] ** 2 + f[None, :, None] ** 2 + h[None, None, :] ** 2
    spec = torch.fft.rfftn(torch.randn((n, n, n), generator=gen, device=DEV)) * torch.exp(-k2 * width ** 2)
    del k2
    g = torch.fft.irfftn(spec, s=(n, n, n)).double()
    return (g * (amp / g.std())).float().reshape(-1).contiguous()


def halo_catalog(case, gen):
    """count x (mass, x, y, z): lognormal density's cells as host positions,
    in no spatial order, masses over two and a half decades."""
    m = 64
    w = lognormal(gaussian(gen, m)).reshape(-1)
    cell = torch.multinomial((w * w).float().cpu(), case["halos"], replacement=True,
                             generator=torch.Generator().manual_seed(gen.initial_seed() + 1)).to(DEV)
    u = torch.rand((case["halos"], 4), generator=gen, device=DEV, dtype=torch.float64)
    mass = 10.0 ** (8.0 + 2.5 * u[:, 0] ** 3)
    scale = case["n_halo"] / m
    pos = [((v + u[:, 1 + k]) * scale) for k, v in enumerate((cell // (m * m), cell // m % m, cell % m))]
    return torch.stack([mass] + pos, 1).float().contiguous()


def t21_boxes(case, gen):
    n = case["n"]
    delta = (lognormal(gaussian(gen, n, sigma=1.0)) - 1).float().reshape(-1).contiguous()

    def uniform(lo, hi):
        return torch.rand(n ** 3, generator=gen, device=DEV) * (hi - lo) + lo

    x = uniform(0.0, 1.0)
    spin = (uniform(0.1, 1.0), uniform(0.5, 2.0), uniform(20.0, 300.0)) if case["spin"] else (None,) * 3
    return (delta, x) + spin


def nl_boxes(case, gen):
    m = case["n_halo"]
    d0 = smooth_box(gen, m, 2.0)
    # z = 0 displacements of a few Mpc (box_len in Mpc/h, velocities in Mpc)
    return [smooth_box(gen, m, 5.0, 12.0) for _ in range(3)] + [d0]


def generator(seed):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    return gen


def boxes(case, seed):
    """The case's inputs, from the seed alone."""
    gen = generator(seed)
    kind = case["kind"]
    if kind == "slice":
        return finder_boxes(case, gen)
    if kind == "batch":
        return [finder_boxes(case, gen) for _ in range(case["count"])]
    if kind == "sweep":
        return [finder_boxes(c, gen) for c in sweep_cases(case)]
    if kind == "train":
        return train_boxes(case, gen)
    if kind == "t21":
        return t21_boxes(case, gen)
    if kind == "power":
        return (lognormal(gaussian(gen, case["n"])) - 1).float().reshape(-1).contiguous()
    if kind == "nldensity":
        return nl_boxes(case, gen)
    return halo_catalog(case, gen)


def finder_context(case):
    mode = sf.INPUT_SFR if case["mode"] == "sfr" else sf.INPUT_DIRECT
    return sf.HiiContext(case["n"], case["side"], ladder(case), mode, sf.PATH_FUSED, hubble=COSMO["hubble"],
                         fesc=FESC)


def params(case):
    return dict(COSMO, n=case["n"], n_halo=case.get("n_halo", 0), box_len=case["side"],
                vel_comp=case.get("axis", 3))


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": case, "in": boxes(case, seed)}
    torch.cuda.empty_cache()  # the contexts allocate outside torch's pool
    if kind == "slice":
        state["ctx"] = finder_context(case)
        if case.get("host"):
            state["in"] = tuple(None if v is None else v.cpu().numpy() for v in state["in"])
        else:
            state["out"] = torch.empty_like(state["in"][0])
    elif kind == "batch":
        state["ctx"] = finder_context(case)
        state["out"] = [torch.empty_like(v[0]) for v in state["in"]]
    elif kind == "sweep":
        made = {}
        for c in sweep_cases(case):
            if c["n"] not in made:
                made[c["n"]] = finder_context(c)
        state["ctx"] = [made[c["n"]] for c in sweep_cases(case)]
        state["out"] = [torch.empty_like(v[0]) for v in state["in"]]
    elif kind == "train":
        state["ctx"] = sf.HiiContext(case["n"], case["side"], ladder(case), sf.INPUT_DIRECT, sf.PATH_FUSED)
        state["weights"] = pk_weights(case, seed)
        state["out"] = [torch.empty_like(state["in"][0]) for _ in range(2)]
    elif kind in ("t21", "power"):
        # transforms only: one radius, no batch buffer
        state["ctx"] = sf.HiiContext(case["n"], case["side"], [case["side"] / case["n"]], sf.INPUT_DIRECT,
                                     sf.PATH_FUSED, radius_batch=1)
        state["out"] = torch.empty(case["n"] ** 3, device=DEV)
    else:
        state["ctx"] = sf.HiiContext(case["n"], case["side"], [], sf.INPUT_HALO, sf.PATH_DEPOSIT,
                                     n_halo=case["n_halo"])
        state["out"] = torch.empty(case["n"] ** 3, device=DEV)
        if kind == "nldensity":
            state["grid"] = torch.empty(case["n_halo"] ** 3, device=DEV)
    return state


def run(state):
    case, ctx, data = state["case"], state["ctx"], state["in"]
    kind = case["kind"]
    if kind == "slice":
        a, b, c = data
        if case.get("host"):
            return ctx.run_slice_host(a, b, c, z=case["z"])
        return ctx.run_slice(a, b, c, z=case["z"], xhii=state["out"])
    if kind == "batch":
        a, b, _ = zip(*data)
        return ctx.run_batch(a, b, z_list=[case["z"]] * len(a), out_list=state["out"])
    if kind == "sweep":
        a, b, _ = zip(*data)
        return sf.run_multi(ctx, a, b, out_list=state["out"])
    if kind == "train":
        g, emis, zeta = data
        x, mean, pk = ctx.diff_forward(g, emis, zeta, case["pk"], x_out=state["out"][0])
        grad, gz, soft_mean, soft_pk = ctx.diff_backward(g, emis, zeta, case["tau"], 1.0, state["weights"],
                                                         case["pk"], grad_out=state["out"][1])
        return {"x": x, "mean": mean, "pk": pk, "grad": grad, "dzeta": gz, "soft_mean": soft_mean,
                "soft_pk": soft_pk}
    if kind == "t21":
        return ctx.t21(params(case), case["z"], *data, out=state["out"])
    if kind == "power":
        return ctx.power_spectrum(data, case["pk"])
    if kind == "nldensity":
        return ctx.nldensity(params(case), case["z"], *data, box_halo=state["grid"], out=state["out"])
    return ctx.sfrd(data, case["z"], out=state["out"])


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def fft_flops(n):
    return 2.5 * n ** 3 * 3 * math.log2(n)  # one real 3D transform


def work(case):
    """Each input read once, each output written once; operations of the
    transforms that the algorithm names (two real ones per field, two inverse
    ones per radius)."""
    kind = case["kind"]
    if kind in ("slice", "batch"):
        n3, m = case["n"] ** 3, case.get("count", 1)
        nr = len(ladder(case))
        boxes_ = 3 + (1 if case.get("fresid") else 0)
        return {"bytes": 4.0 * n3 * boxes_ * m, "flops": m * (2 + 2 * nr) * fft_flops(case["n"])}
    if kind == "sweep":
        parts = [work(c) for c in sweep_cases(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    n3 = case["n"] ** 3
    if kind == "train":
        nr = len(ladder(case))
        # forward as above; backward: one real transform pair per radius for
        # phi, the filtered pair, the ball adjoint and the seeds
        return {"bytes": 4.0 * n3 * 4, "flops": (4 + 2 * nr + 8 * nr) * fft_flops(case["n"])}
    if kind == "t21":
        return {"bytes": 4.0 * n3 * (6 if case["spin"] else 3), "flops": 2 * fft_flops(case["n"]) + 30.0 * n3}
    if kind == "power":
        return {"bytes": 4.0 * n3, "flops": fft_flops(case["n"]) + 4.0 * n3}
    m3 = case["n_halo"] ** 3
    if kind == "nldensity":
        return {"bytes": 4.0 * (5 * m3 + n3), "flops": 40.0 * m3}
    return {"bytes": 16.0 * case["halos"] + 4.0 * n3, "flops": 60.0 * case["halos"] + 2.0 * m3}


# ---------------------------------------------------------------------------
# 64 bits, plain torch
# ---------------------------------------------------------------------------
def sq_grid(n, half=True):
    """Integer |k|^2 (or squared periodic distance) of every cell."""
    f = freq(n) ** 2
    h = torch.arange(n // 2 + 1, device=DEV, dtype=torch.int64) ** 2 if half else f
    return f[:, None, None] + f[None, :, None] + h[None, None, :]


def top_hat(n, dk, radius, k2):
    """W(|k| R), one value for each integer |k|^2."""
    x = dk * radius * torch.arange(3 * (n // 2) ** 2 + 1, device=DEV, dtype=torch.float64).sqrt()
    s = x.clamp_min(1e-30)
    w = torch.where(x < 0.03, 1.0 - x * x / 10.0, 3.0 * (torch.sin(s) - s * torch.cos(s)) / s ** 3)
    return w[k2]


def ball_bound(radius, dx):
    m = int(math.floor((radius / dx) ** 2))
    while m > 0 and not math.sqrt(m) * dx <= radius:
        m -= 1
    while math.sqrt(m + 1) * dx <= radius:
        m += 1
    return m


def own_fill(rec, ion):
    one = torch.ones_like(rec)
    q = torch.where(rec > 0, torch.minimum(ion / torch.where(rec > 0, rec, one), one), one)
    return torch.where(ion > 0, q, torch.zeros_like(rec))


def exact_slice(case, a, b, c):
    n, side = case["n"], case["side"]
    shape = (n, n, n)
    rec, ion, fres = prepass(case, a.reshape(shape), b.reshape(shape), None if c is None else c.reshape(shape))
    fr, fi = torch.fft.rfftn(rec), torch.fft.rfftn(ion)
    fill = own_fill(rec, ion)
    del rec, ion
    k2 = sq_grid(n)
    d2 = sq_grid(n, half=False)
    covered = torch.zeros(shape, dtype=torch.bool, device=DEV)
    for radius in ladder(case):
        w = top_hat(n, 2 * PI / side, radius, k2)
        r = torch.fft.irfftn(fr * w, s=shape)
        o = torch.fft.irfftn(fi * w, s=shape)
        del w
        centre = (o > 0) & ((r <= 0) | (o >= r))
        del r, o
        if bool(centre.any()):
            ball = torch.fft.rfftn((d2 <= ball_bound(radius, side / n)).double())
            covered |= torch.fft.irfftn(torch.fft.rfftn(centre.double()) * ball, s=shape) > 0.5
            del ball
    x = torch.where(covered, torch.ones_like(fill), fill)
    if fres is not None:
        x = torch.minimum(x, 1 - fres)
    return x.reshape(-1), float((1 - x).mean())


def bin_index(n, nb):
    k = sq_grid(n).double().sqrt()
    b = ((k - 1) / ((n // 2 - 1) / nb)).floor().long().clamp_max(nb - 1)
    return torch.where((k >= 1) & (k <= n // 2), b, torch.full_like(b, -1)), k


def power(field, side, nb):
    n = field.shape[0]
    spec = torch.fft.rfftn(field)
    bins, k = bin_index(n, nb)
    keep = bins >= 0
    p2, kk, bb = (spec.real ** 2 + spec.imag ** 2)[keep], k[keep], bins[keep]
    total = torch.zeros(nb, dtype=torch.float64, device=DEV)
    count = torch.bincount(bb, minlength=nb).double()
    pk = total.index_add(0, bb, p2) / count * ((side / n) ** 3 / n ** 3)
    return pk, total.index_add(0, bb, kk) / count * (2 * PI / side), count


def exact_train(case, seed):
    g, emis, zeta = train_boxes(case, generator(seed))
    n, side = case["n"], case["side"]
    shape = (n, n, n)
    cap = 20.0
    e = torch.exp(g.double())
    delta1 = (e / e.mean()).float()  # the boxes that the finder is given are single precision
    x, neutral = exact_slice(dict(case, mode="direct"), (delta1 * delta1), emis * zeta, None)
    t = (1 - x) * (e / e.mean())
    pk, _, _ = power(t.reshape(shape), side, case["pk"])
    gd = g.double().reshape(shape).requires_grad_(True)
    zd = torch.tensor(float(zeta), dtype=torch.float64, device=DEV, requires_grad=True)
    e = torch.exp(gd)
    delta = e / e.mean()
    rec, ion = delta ** 2, zd * emis.double().reshape(shape)
    fr, fi = torch.fft.rfftn(rec), torch.fft.rfftn(ion)
    rho = 1e-3 * rec.mean()
    k2, d2 = sq_grid(n), sq_grid(n, half=False)

    def bubble(fr_, fi_, rho_, w, ball):
        r = torch.fft.irfftn(fr_ * w, s=shape)
        o = torch.fft.irfftn(fi_ * w, s=shape)
        u = torch.minimum(o - r, o) / torch.maximum(r, rho_) / case["tau"]
        phi = torch.nn.functional.softplus(u) - torch.nn.functional.softplus(u - cap)
        return torch.fft.irfftn(torch.fft.rfftn(phi) * ball, s=shape)

    reach = torch.zeros(shape, dtype=torch.float64, device=DEV)
    for radius in ladder(case):
        w = top_hat(n, 2 * PI / side, radius, k2)
        ball = torch.fft.rfftn((d2 <= ball_bound(radius, side / n)).double())
        reach = reach + torch.utils.checkpoint.checkpoint(bubble, fr, fi, rho, w, ball, use_reentrant=False)
    q = own_fill(rec, ion)
    soft = q + (1 - q) * (1 - torch.exp(-reach))
    soft_pk, _, _ = power((1 - soft) * delta, side, case["pk"])
    loss = soft.mean() + (torch.from_numpy(pk_weights(case, seed)).to(DEV) * soft_pk).sum()
    loss.backward()
    return {"x": x, "mean": 1 - neutral, "pk": pk, "grad": gd.grad.reshape(-1), "dzeta": float(zd.grad),
            "soft_mean": float(soft.detach().mean()), "soft_pk": soft_pk.detach()}


def hubble(z):
    return COSMO["hubble"] * H0 * math.sqrt(COSMO["omega_m"] * (1 + z) ** 3 + COSMO["omega_lambda"])


def growth(z):
    def integral(z0):
        zs = z0 + 0.0005 + 0.001 * np.arange(100000)
        e = np.sqrt(COSMO["omega_m"] * (1 + zs) ** 3 + COSMO["omega_lambda"])
        e /= math.sqrt(COSMO["omega_m"] + COSMO["omega_lambda"])
        return float(np.sum((1 + zs) / e ** 3) * 0.001)
    return hubble(z) / hubble(0.0) * integral(z) / integral(0.0)


def exact_t21(case, seed):
    delta, x, xc, xa, tk = (None if v is None else v.double() for v in t21_boxes(case, generator(seed)))
    n, z, h = case["n"], case["z"], COSMO["hubble"]
    spec = torch.fft.rfftn(delta.reshape(n, n, n))
    f = freq(n) ** 2
    half = torch.arange(n // 2 + 1, device=DEV) ** 2
    along = {1: f[:, None, None], 2: f[None, :, None]}.get(case["axis"], half[None, None, :])
    k2 = sq_grid(n)
    spec *= torch.where(k2 > 0, along.double() / k2.clamp_min(1), torch.zeros((), dtype=torch.float64, device=DEV))
    dv = torch.fft.irfftn(spec, s=(n, n, n)).reshape(-1)
    rate = (growth(z + 5e-4) - growth(z - 5e-4)) / 1e-3 * (-hubble(z) * (1 + z))
    dv = (dv * (-rate / hubble(z) / growth(z))).clamp(-0.5, 1.0)
    c21 = 23.0 / 1000 * (0.7 / h) * (COSMO["omega_b"] * h * h / 0.02) * \
        math.sqrt((0.15 / COSMO["omega_m"] / h / h) * (1 + z) / 10)
    tcmb = 2.725 * (1 + z)
    spin, ts = 1.0, 0.0
    if case["spin"]:
        y = xa + xc
        spin = y / (1 + y) * (1 - tcmb / tk)
        ts = float((tcmb * (1 + y) / (1 + y * tcmb / tk)).mean())
    t = c21 * (1 + delta) * spin / (1 + dv) * (1 - x)
    return t, float(t.mean()), ts


def deposit(grid, pos, value, m):
    """Cloud in cell with the reference's rule for negative positions."""
    cell, far = [], []
    for p in pos:
        i = p.trunc()
        fr = p - i
        i = torch.where(fr < 0, i - 1, i)
        cell.append(i.long())
        far.append(fr.abs())
    for corner in range(8):
        at, w = None, value
        for k in range(3):
            up = corner >> k & 1
            at = (cell[k] + up).remainder(m) if at is None else at * m + (cell[k] + up).remainder(m)
            w = w * (far[k] if up else 1 - far[k])
        grid.index_add_(0, at, w)


def block_mean(grid, m, n):
    sm = int(math.floor(m / n + 0.5))
    sm -= 1 if n * sm > m else 0
    g = grid.reshape(m, m, m)[: n * sm, : n * sm, : n * sm]
    return g.reshape(n, sm, n, sm, n, sm).mean((1, 3, 5)).reshape(-1)


def exact_nldensity(case, seed):
    vx, vy, vz, d0 = nl_boxes(case, generator(seed))
    m = case["n_halo"]
    g_in = growth(300.0)
    g = growth(case["z"]) - g_in
    scale = m / case["side"] * COSMO["hubble"] * g
    grid = torch.full((m ** 3,), -1.0, dtype=torch.float64, device=DEV)
    step = max(1, (1 << 24) // (m * m)) * m * m
    for lo in range(0, m ** 3, step):  # planes at a time
        ind = torch.arange(lo, min(lo + step, m ** 3), device=DEV)
        pos = [(ind // (m * m)).double() + vx[ind].double() * scale,
               (ind // m % m).double() + vy[ind].double() * scale, (ind % m).double() + vz[ind].double() * scale]
        deposit(grid, pos, 1 + d0[ind].double() * g_in, m)
    return block_mean(grid, m, case["n"]), grid


def exact_sfrd(case, seed):
    cat = halo_catalog(case, generator(seed)).double()
    m, z = case["n_halo"], case["z"]
    qion = 10.0 ** (2.05707274e-02 * z + 5.29944413e+01)
    mass = cat[:, 0]
    rate = 1.575e39 * (1 + z) ** 2.27044695 / qion * mass * (mass / 9.367608e+07) ** 0.44 \
        * torch.exp(-(9.367608e+07 / mass) ** 3)
    grid = torch.zeros(m ** 3, dtype=torch.float64, device=DEV)
    deposit(grid, [cat[:, 1], cat[:, 2], cat[:, 3]], rate, m)
    box = block_mean(grid, m, case["n"]) / (case["side"] / m) ** 3
    return box, float(box.mean())


def exact(case, seed):
    kind = case["kind"]
    if kind == "slice":
        x, neutral = exact_slice(case, *boxes(case, seed))
        return (x.cpu().numpy() if case.get("host") else x), neutral
    if kind == "batch":
        got = [exact_slice(case, *v) for v in boxes(case, seed)]
        return [g[0] for g in got], [g[1] for g in got]
    if kind == "sweep":
        got = [exact_slice(c, *v) for c, v in zip(sweep_cases(case), boxes(case, seed))]
        return [g[0] for g in got], [g[1] for g in got]
    if kind == "train":
        return exact_train(case, seed)
    if kind == "t21":
        return exact_t21(case, seed)
    if kind == "power":
        field = boxes(case, seed).double().reshape((case["n"],) * 3)
        return tuple(v.cpu().numpy() for v in power(field, case["side"], case["pk"]))
    if kind == "nldensity":
        return exact_nldensity(case, seed)
    return exact_sfrd(case, seed)
