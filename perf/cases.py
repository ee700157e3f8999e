"""What the framework does for its users, as cases that can be timed: the
accelerated Lambda iteration on the package's own workloads, the radiation
field by itself, images, whole solves of new models, and the warm-start
network.

listed() are the cases themselves, draw() more of the same ranges, prepare()
what a program holds before a call (a context, a network and its data), run()
the call, work() the bytes and operations it cannot do without, and exact()
the same outputs in 64 bits from plain torch.
"""
import math

import numpy as np
import torch

from magritte_amd.hip import BatchContext, Context, Mlp
from magritte_amd.setup import synthetic

MAX_ITERATIONS = 100   # of a solve: far above what the listed models need


def listed():
    return [
        # the 16^3 regular grid: one radiation field whose spectrum and operator the program reads
        {"name": "field regular 16", "kind": "field", "model": "regular", "n": 16, "nside": 1, "nquads": 39,
         "precision": "fp32"},
        # the smallest model of the training distribution, solved again and again: launches and latency
        {"name": "ali envelope 10", "kind": "ali", "model": "envelope", "n": 10, "nside": 1, "nquads": 31,
         "nlev": 7, "log_n0": 15.0, "T0": 1500.0, "precision": "fp32", "iterations": MAX_ITERATIONS},
        # the at-scale envelope from LTE to convergence, the headline workload
        {"name": "ali envelope 64", "kind": "ali", "model": "envelope", "n": 64, "nside": 2, "nquads": 31,
         "nlev": 7, "log_n0": 14.0, "T0": 2500.0, "precision": "fp32", "iterations": MAX_ITERATIONS},
        # the same physics in double precision, to convergence
        {"name": "ali envelope 36 fp64", "kind": "ali", "model": "envelope", "n": 36, "nside": 2, "nquads": 31,
         "nlev": 7, "log_n0": 14.0, "T0": 2500.0, "precision": "fp64", "iterations": MAX_ITERATIONS},
        # velocity jumps of +-30 km/s: long interpolated rays, optically thick
        {"name": "ali stress 36", "kind": "ali", "model": "stress", "n": 36, "nside": 2, "nquads": 31,
         "nlev": 7, "log_n0": 17.0, "T0": 2500.0, "precision": "fp32", "iterations": MAX_ITERATIONS},
        # blended lines: a bin sees up to four lines
        {"name": "ali blended 20", "kind": "ali", "model": "blended", "n": 20, "nside": 1, "nquads": 24,
         "log_n0": 14.0, "T0": 2500.0, "precision": "fp32", "iterations": 4},
        # uneven models, 12 and 48 rays, solved together as the training set is
        {"name": "batch 24", "kind": "batch", "models": 24, "precision": "fp32", "iterations": 8},
        # the banded approximate operator (n_off_diag 2)
        {"name": "ali bands 20", "kind": "ali", "model": "bands", "n": 20, "nside": 2, "nquads": 21,
         "nlev": 5, "log_n0": 13.0, "T0": 1500.0, "precision": "fp32", "iterations": 3},
        # an image of a solved model, in the host layer's default precision
        {"name": "image envelope 36", "kind": "image", "n": 36, "nquads": 31, "ray": 7, "precision": "fp64"},
        # a new model from its arrays to its populations: upload, set-up, trace, tuning, iteration
        {"name": "solve envelope 27", "kind": "solve", "n": 27, "nside": 2, "nquads": 31, "nlev": 7,
         "log_n0": 14.5, "T0": 2000.0, "precision": "fp32"},
        # the network: one gradient of a large batch, and training from given weights
        {"name": "gradient 400000", "kind": "gradient", "rows": 400000},
        {"name": "train 262144", "kind": "train", "rows": 262144, "batch": 16384, "epochs": 4},
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["field", "ali", "ali", "ali", "ali", "batch", "image", "solve", "gradient", "train"])
    if kind == "field":
        return {"kind": "field", "model": "regular", "n": log_int(5, 24), "nside": 1, "nquads": rng.randint(9, 45),
                "precision": rng.choice(["fp32", "fp64"])}
    if kind == "batch":
        return {"kind": "batch", "models": log_int(2, 24), "precision": rng.choice(["fp32", "fp32", "fp64"]),
                "iterations": rng.randint(2, 6)}
    if kind == "image":
        return {"kind": "image", "n": log_int(8, 36), "nquads": rng.randint(12, 33), "ray": rng.randint(0, 23),
                "precision": rng.choice(["fp64", "fp32"])}
    if kind == "gradient":
        return {"kind": "gradient", "rows": log_int(1, 400000)}
    if kind == "train":
        return {"kind": "train", "rows": log_int(1000, 262144), "batch": rng.choice([1000, 4096, 16384]),
                "epochs": rng.randint(1, 3)}
    c = {"kind": kind, "nside": rng.choice([1, 2]), "nlev": rng.randint(2, 8),
         "log_n0": round(rng.uniform(14.0, 16.0), 3), "T0": round(rng.uniform(500.0, 3000.0), 1)}
    if kind == "solve":
        return dict(c, n=log_int(8, 30), nquads=rng.randint(15, 33), precision="fp32")
    c["model"] = rng.choice(["envelope", "envelope", "stress", "blended", "bands"])
    c["precision"] = rng.choice(["fp32", "fp32", "fp64"])
    top = {"envelope": 56 if c["precision"] == "fp32" else 36, "stress": 30, "blended": 20, "bands": 20}[c["model"]]
    c["n"] = log_int(8, top)
    c["nquads"] = rng.randint(12, 24) if c["model"] == "blended" else rng.randint(12, 33)
    c["iterations"] = rng.randint(1, 3)
    if c["model"] == "stress":
        c["log_n0"] = 17.0
    if c["model"] == "blended":
        del c["nlev"]
    return c


# ---- a case's inputs ---------------------------------------------------------


def models_of(case, seed):
    """The case's model, or the models of its batch, in the package's layout."""
    kind = case["kind"]
    if kind == "batch":
        # the training distribution: cells log-uniform in 1000..32768, spread by the model's place in the batch
        k = np.arange(case["models"])
        sides = np.round(10.0 * 3.2 ** ((k * 0.618034) % 1.0)).astype(int)
        rng = np.random.default_rng([seed, case["models"]])
        return [synthetic.envelope_model(n=int(n), nside=1 + i % 2, n0=10.0 ** rng.uniform(13.0, 16.0),
                                         T0=rng.uniform(500.0, 3000.0), seed=int(rng.integers(0, 2 ** 31)))
                for i, n in enumerate(sides)]
    if kind == "image":
        return [synthetic.envelope_model(n=case["n"], nquads=case["nquads"], seed=seed)]
    if case.get("model") == "regular":
        rng = np.random.default_rng([seed, case["n"]])
        m = synthetic.regular_grid_model(n=case["n"], nside=case["nside"], nquads=case["nquads"])
        m.temperature = m.temperature * rng.uniform(0.8, 1.2, m.ncells)
        m.abundance = m.abundance * rng.uniform(0.5, 2.0, m.ncells)[:, None]
        return [m]
    kw = dict(n=case["n"], nside=case["nside"], nquads=case["nquads"], seed=seed, n0=10.0 ** case["log_n0"],
              T0=case["T0"])
    if case.get("model") == "blended":
        return [synthetic.blended_model(**kw)]
    if case.get("model") == "stress":
        return [synthetic.stress_model(nlev=case["nlev"], **kw)]
    m = synthetic.envelope_model(nlev=case["nlev"], **kw)
    if case.get("model") == "bands":
        m.n_off_diag = 2
    return [m]


def training_rows(case, seed):
    """Features and targets like those of the warm start: log densities,
    temperature, velocity gradient, line intensities against B_nu, and log
    level fractions that follow a Boltzmann law with a departure."""
    n = case["rows"]
    rng = np.random.default_rng([seed, n])
    X = np.empty((n, 8), np.float32)
    X[:, 0] = rng.uniform(9.0, 16.0, n)
    X[:, 1] = rng.uniform(1.5, 3.5, n)
    X[:, 2] = X[:, 0] - 4.0
    X[:, 3] = rng.normal(-10.0, 1.0, n)
    X[:, 4:] = -np.abs(rng.normal(0.0, 0.5, (n, 4)))
    J = np.arange(7)
    Tx = 10.0 ** (X[:, 1:2] + 0.3 * np.tanh(X[:, 4:5] + 0.1 * (X[:, 0:1] - 12.0)))
    y = np.log10(2.0 * J + 1.0) - 0.4343 * 2.764 * J * (J + 1) / Tx
    y -= np.log10(np.sum(10.0 ** y, axis=1, keepdims=True))
    return X, y.astype(np.float32)


def first_weights(seed):
    rng = np.random.default_rng([seed, 8])
    sizes = {"W1": (8, 128), "W2": (128, 128), "W3": (128, 7)}
    p = {k: rng.normal(0.0, math.sqrt(2.0 / s[0]), s).astype(np.float32) for k, s in sizes.items()}
    for k, n in (("b1", 128), ("b2", 128), ("b3", 7)):
        p[k] = rng.normal(0.0, 0.05, n).astype(np.float32)
    return p


def normalisation(X, Y):
    return X.mean(0), X.std(0) + 1e-3, Y.mean(0), Y.std(0) + 1e-3


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("gradient", "train"):
        X, Y = training_rows(case, seed)
        net = Mlp(seed=0)
        norm = normalisation(X, Y)
        net.set_normalisation(*norm)
        first = first_weights(seed)
        net.set_params(first)
        return {"case": case, "net": net, "first": first, "X": X, "Y": Y}
    models = models_of(case, seed)
    if kind == "solve":
        return {"case": case, "model": models[0]}
    if kind == "batch":
        ctx = BatchContext(models).setup()
    else:
        ctx = Context(models[0]).setup()
    if kind == "image":
        ctx.compute_radiation_field("fp64")
        ctx.compute_Jeff()
        ctx.compute_level_populations_from_stateq()
        ctx.compute_spectral_discretisation_image(1.5e-5)
        ctx.compute_boundary_intensities()
    else:
        ctx.trace()
        ctx.prepare(case["precision"])
    return {"case": case, "ctx": ctx}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "gradient":
        loss, grad = state["net"].loss_grad(state["X"], state["Y"])
        return {"loss": loss, "grad": grad}
    if kind == "train":
        net = state["net"]
        net.set_params(state["first"])
        losses = net.train(state["X"], state["Y"], case["epochs"], case["batch"], 4e-3, seed=3)
        return {"losses": losses, "weights": net.params()}
    if kind == "solve":
        ctx = Context(state["model"]).setup()
        ctx.trace()
        its = ctx.compute_level_populations(True, MAX_ITERATIONS, "max", case["precision"])
        out = {"iterations": its, "populations": ctx.populations()}
        ctx.close()
        return out
    ctx = state["ctx"]
    if kind == "field":
        ctx.compute_radiation_field(case["precision"])
        return {"J": ctx.J(), "lambda": ctx.lambda_diag()}
    if kind == "image":
        I_m, I_p = ctx.compute_image(case["ray"], case["precision"])
        return {"I_m": I_m, "I_p": I_p}
    ctx.compute_LTE_level_populations()
    its = ctx.compute_level_populations(True, case["iterations"], "max", case["precision"])
    if kind == "batch":
        return {"iterations": its, "each": ctx.convergence()[0], "populations": ctx.populations()}
    return {"iterations": its, "populations": ctx.populations(), "Jeff": ctx.Jeff()}


# ---- what a pass cannot do without ---------------------------------------------

# points of a ray pair over the cells of a side (mean walk, and what the
# interpolation of velocity gradients adds), measured on the package's models
POINTS_PER_SIDE = {"regular": 1.01, "envelope": 1.49, "bands": 1.49, "blended": 1.49, "stress": 16.1}
FLOPS_PER_POINT_BIN = 28   # profile, opacity, source function and elimination step of one point and bin


def work(case):
    kind = case["kind"]
    if kind in ("gradient", "train"):
        per_row = 2 * 3 * (8 * 128 + 128 * 128 + 128 * 7) - 2 * 8 * 128
        passes = case.get("epochs", 1)
        return {"bytes": 60 * case["rows"] + 3 * 4 * 18567 * 2, "flops": float(per_row) * case["rows"] * passes}
    sizes = []
    if kind == "batch":
        # cells log-uniform in 1000..32768: mean of n^3 and n^4, half of the models with 12 rays and half with 48
        sizes = [(21, R, 6 * 31, 7, 6, "envelope") for R in (12, 48) for _ in range(max(1, case["models"] // 2))]
    elif kind == "image":
        sizes = [(case["n"], 2, 6 * case["nquads"], 7, 6, "envelope")]
    else:
        V = 2 if case.get("model") == "regular" else 7 if case.get("model") == "blended" else case["nlev"]
        L = 1 if V == 2 else 10 if case.get("model") == "blended" else V - 1
        sizes = [(case["n"], 12 * case["nside"] ** 2, L * case["nquads"], V, L, case.get("model", "envelope"))]
    # radiation fields to convergence: 2 for thermalised models, more as the density falls
    n0 = case.get("log_n0", 14.5)
    needs = 2 if n0 > 16.5 else 3 if n0 >= 15.0 else 6
    fields = {"field": 1, "image": 2}.get(kind, min(case.get("iterations", MAX_ITERATIONS), needs))
    nbytes, flops = 0.0, 0.0
    for n, R, F, V, L, model in sizes:
        N = n ** 3
        points = N * (R // 2) * POINTS_PER_SIDE[model] * n
        flops += fields * FLOPS_PER_POINT_BIN * points * F
        nbytes += N * (26 * 4 + 8 * 8 + V * 8)                         # geometry, state and starting populations
        nbytes += N * {"field": F + L, "image": 2 * F}.get(kind, V + 3 * L) * 8   # outputs
    return {"bytes": nbytes, "flops": flops}


# ---- the same in 64 bits ---------------------------------------------------------

C_LIGHT, H_PLANCK, K_BOLTZ, AMU, C2 = 2.99792458e8, 6.62607004e-34, 1.38064852e-23, 1.66053904e-27, 8.98755179e16
T_CMB = 2.72548


class Exact:
    """Radiation field, operator and populations of one model with one line
    species, every quantity a float64 tensor (geometry and lines: see Model)."""

    BLOCK = 1 << 24   # (ray, bin) values in flight

    def __init__(self, m):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        t = self.t
        self.m, self.N, self.R, self.Q = m, m.ncells, m.nrays, m.nquads
        ld = m.linedata
        self.V, self.L = ld.nlev, ld.nrad
        self.F = self.L * self.Q
        self.pos, self.vel = t(m.position), t(m.velocity)
        k = int(m.n_neighbors.max())
        table = np.full((self.N, k), -1, np.int64)
        table[np.arange(k)[None, :] < m.n_neighbors[:, None]] = m.neighbors
        self.nbr = t(table)
        self.bdy = torch.zeros(self.N, dtype=torch.bool, device=self.dev)
        self.bdy[t(m.boundary2cell_nr)] = True
        self.rays, self.w = t(m.rays), t(m.weights)
        self.anti = ((self.rays[:, None] + self.rays[None]) ** 2).sum(-1).argmin(1)
        self.order = t(np.argsort(ld.frequency, kind="stable"))
        self.freq = t(ld.frequency)
        self.line = self.freq[self.order]
        self.width = torch.sqrt(2.0 * K_BOLTZ / (AMU * C2) * ld.inverse_mass * t(m.temperature) + t(m.vturb2))
        self.dsm = m.max_width_fraction * self.width
        self.T, self.ntot = t(m.temperature), t(m.abundance[:, ld.num])
        self.roots, self.qw = t(m.roots), t(m.qweights)
        self.irad, self.jrad = t(ld.irad), t(ld.jrad)
        self.A, self.Bs, self.Ba = t(ld.A), t(ld.Bs), t(ld.Ba)

    def t(self, a):
        a = torch.from_numpy(np.ascontiguousarray(a))
        return a.to(self.dev, torch.int64 if a.dtype == torch.int32 else a.dtype)

    @staticmethod
    def dot(a, b):
        return (a[..., 0] * b[..., 0] + a[..., 1] * b[..., 1]) + a[..., 2] * b[..., 2]

    def grid(self, width=None):
        """Frequencies of every cell (ascending) and the bin of every (line, root)."""
        w = self.width[:, None, None] if width is None else torch.full((self.N, 1, 1), width, dtype=torch.float64, device=self.dev)
        nu = self.line[None, :, None] + (self.line[None, :, None] * w) * self.roots[None, None, :]
        self.nu, at = nu.reshape(self.N, -1).sort(dim=1, stable=True)
        self.bin_of = torch.argsort(at, dim=1)          # [N, L Q], running index of the sorted lines
        self.I_bdy = self.planck(self.nu, T_CMB)

    @staticmethod
    def planck(nu, T):
        return 2.0 * H_PLANCK / C2 * (nu * nu * nu) / torch.expm1(H_PLANCK / K_BOLTZ / T * nu)

    def lte(self):
        ld = self.m.linedata
        p = self.t(ld.weight) * torch.exp(-self.t(ld.energy) / (K_BOLTZ * self.T[:, None]))
        return p * (self.ntot / p.sum(1))[:, None]

    def walk(self, o, d, s=None):
        """Points of the rays from cells o along d, outwards: (first point of
        each ray, cell, shift, dZ).  s: the direction of rest-frame shifts."""
        Q = o.numel()

        def shift(c, i):
            if s is None:
                return 1.0 - self.dot(self.vel[c] - self.vel[o[i]], d[i])
            return 1.0 - self.dot(self.vel[c], s[i])

        alive = torch.arange(Q, device=self.dev)
        cur, Z = o.clone(), torch.zeros(Q, dtype=torch.float64, device=self.dev)
        sc = shift(o, alive)
        ids, cells, shifts, dZs, ns = [], [], [], [], []
        while alive.numel():
            i = alive
            nb = self.nbr[cur[i]]
            Rv = self.pos[nb] - self.pos[o[i]][:, None]
            Zn = self.dot(Rv, d[i][:, None])
            far = self.dot(Rv, Rv) - Zn * Zn
            far = torch.where((nb >= 0) & (Zn > Z[i][:, None]), far, math.inf)
            best = far.amin(1)
            first = torch.where(far == best[:, None], torch.arange(nb.shape[1], device=self.dev), nb.shape[1]).amin(1)
            on = torch.isfinite(best)
            i, first, nb, Zn = i[on], first[on], nb[on], Zn[on]
            nxt = nb.gather(1, first[:, None])[:, 0]
            dz = Zn.gather(1, first[:, None])[:, 0] - Z[i]
            Z[i] = Z[i] + dz
            sn = shift(nxt, i)
            step = sn - sc[i]
            dsm = self.dsm[o[i]]
            interp = step.abs() > dsm
            n = torch.where(interp, torch.floor(step.abs() / dsm + 1.0), 1.0).long()
            rep = torch.repeat_interleave(torch.arange(i.numel(), device=self.dev), n)
            mth = torch.arange(rep.numel(), device=self.dev) - (torch.cumsum(n, 0) - n)[rep] + 1
            nf = n.double()
            half = torch.floor(0.5 * nf).long()
            ids.append(i[rep])
            cells.append(torch.where(interp[rep] & (mth < half[rep]), cur[i][rep], nxt[rep]))
            shifts.append(torch.where(interp[rep], sc[i][rep] + mth.double() * (step / nf)[rep], sn[rep]))
            dZs.append((dz / nf)[rep])
            cur[i], sc[i] = nxt, sn
            alive = i[~self.bdy[nxt]]
        ids = torch.cat(ids)
        at = torch.argsort(ids, stable=True)
        count = torch.bincount(ids, minlength=Q)
        return (torch.cumsum(count, 0) - count, count, torch.cat(cells)[at], torch.cat(shifts)[at], torch.cat(dZs)[at])

    def lines_of(self, pop):
        """Emissivity and opacity of every (cell, sorted line)."""
        up, lo = pop[:, self.irad], pop[:, self.jrad]
        f = H_PLANCK / (4.0 * math.pi)
        return (f * self.A * up)[:, self.order], (f * (lo * self.Ba - up * self.Bs))[:, self.order]

    def source(self, cell, shift, nu_o):
        """Opacity and source function at points [E] for bins [E, F] of their origins."""
        fs = shift[:, None] * nu_o
        eta = torch.zeros_like(fs)
        chi = torch.full_like(fs, 1.0e-26)
        wmax = 11.5 * float(self.width.max())
        lo_s, hi_s = float(shift.min()) - 1e-9, float(shift.max()) + 1e-9
        for l in range(self.L):
            nl = float(self.line[l])
            cols = torch.nonzero((self.nu_min * lo_s < nl * (1.0 + wmax)) & (self.nu_max * hi_s > nl * (1.0 - wmax)))[:, 0]
            if not cols.numel():
                continue
            a, b = int(cols[0]), int(cols[-1]) + 1
            iw = 1.0 / (nl * self.width[cell])[:, None]
            x = (fs[:, a:b] - nl) * iw
            g = fs[:, a:b] * (iw / math.sqrt(math.pi)) * torch.where(x.abs() <= 11.0, torch.exp(-x * x), 0.0)
            eta[:, a:b] += self.em[cell, l][:, None] * g
            chi[:, a:b] += self.op[cell, l][:, None] * g
        return chi, eta / chi

    def far(self, pts, e, nu_o):
        """Boundary intensity entering rays e at their far ends, for bins nu_o."""
        off, count, cell, shift, _ = pts
        last = (off + count - 1)[e].clamp(min=0)
        c, f = cell[last], shift[last][:, None] * nu_o
        grid, I = self.nu[c], self.I_bdy[c]
        k = torch.searchsorted(grid, f).clamp(max=self.F - 1)
        k1 = (k - 1).clamp(min=0)
        nu1, nu2, I1, I2 = grid.gather(1, k), grid.gather(1, k1), I.gather(1, k), I.gather(1, k1)
        inner = (k > 0) & (k < self.F - 1)
        return torch.where(inner, (I2 - I1) / torch.where(inner, nu2 - nu1, 1.0) * (f - nu1) + I1, I1)

    def close(self, st, chi, S, b):
        """Close the pending rows of the elimination st with the interval b and
        make (chi, S) pending.  phi q, zeta and a of the last closed row."""
        h = 0.5 * (st["a"] + b)
        phi = h + st["pq"]
        q = 1.0 / (1.0 + b * phi)
        st["z"] = (st["S"] * h + st["z"]) * q
        st["pq"], st["a"], st["S"], st["chi"] = phi * q, b, S, chi

    def inwards(self, pts, e, nu_o, I_far, chi_o, S_o):
        """Rays e eliminated from their far ends to their origins, the origin pending."""
        off, count, cell, shift, dZ = pts
        n = count[e]
        by = torch.argsort(n, descending=True)
        e, n, nu_s = e[by], n[by], nu_o[by]
        st = {"a": torch.zeros_like(nu_s), "pq": torch.ones_like(nu_s), "z": I_far[by].clone(),
              "S": torch.zeros_like(nu_s), "chi": torch.zeros_like(nu_s)}
        dz_out = torch.zeros(e.numel(), dtype=torch.float64, device=self.dev)
        active = torch.bincount(n, minlength=1).flip(0).cumsum(0).flip(0).tolist() if n.numel() else []
        for k in range(len(active) - 1, 0, -1):
            A = active[k]          # rays with at least k points
            at = off[e[:A]] + k - 1
            chi, S = self.source(cell[at], shift[at], nu_s[:A])
            part = {x: v[:A] for x, v in st.items()}
            self.close(part, chi, S, 0.5 * (part["chi"] + chi) * dz_out[:A, None])
            for x, v in part.items():
                st[x][:A] = v
            dz_out[:A] = dZ[at]
        b = 0.5 * (st["chi"] + chi_o[by]) * dz_out[:, None]
        self.close(st, chi_o[by], S_o[by], b)
        back = torch.argsort(by)
        return {x: v[back] for x, v in st.items()}

    def outwards(self, pts, e, nu_o, st):
        """The elimination st continued along rays e to their far ends, which are left pending."""
        off, count, cell, shift, dZ = pts
        n = count[e]
        by = torch.argsort(n, descending=True)
        e, n, nu_s = e[by], n[by], nu_o[by]
        st = {x: v[by] for x, v in st.items()}
        for k in range(int(n.max()) if n.numel() else 0):
            A = int((n > k).sum())
            at = off[e[:A]] + k
            chi, S = self.source(cell[at], shift[at], nu_s[:A])
            part = {x: v[:A] for x, v in st.items()}
            self.close(part, chi, S, 0.5 * (part["chi"] + chi) * dZ[at][:, None])
            for x, v in part.items():
                st[x][:A] = v
        back = torch.argsort(by)
        return {x: v[back] for x, v in st.items()}

    def bounds_of_bins(self):
        self.nu_min, self.nu_max = self.nu.amin(0), self.nu.amax(0)

    def trace(self):
        o = torch.arange(self.N, device=self.dev).repeat_interleave(self.R)
        parts, step = [], max(1, (1 << 22) // self.R) * self.R
        for a in range(0, o.numel(), step):
            b = min(o.numel(), a + step)
            r = torch.arange(a, b, device=self.dev) % self.R
            parts.append(self.walk(o[a:b], self.rays[r]))
        base = 0
        offs = []
        for p in parts:
            offs.append(p[0] + base)
            base += p[2].numel()
        self.pts = (torch.cat(offs),) + tuple(torch.cat([p[i] for p in parts]) for i in range(1, 5))

    def field(self, pop):
        """J [N, F] and sum_r 2 w_r Lambda / chi [N, F]."""
        self.em, self.op = self.lines_of(pop)
        self.bounds_of_bins()
        J = torch.empty(self.N, self.F, dtype=torch.float64, device=self.dev)
        lam = torch.empty_like(J)
        step = max(1, self.BLOCK // (self.R * self.F))
        half = self.R // 2
        one = torch.ones(1, dtype=torch.float64, device=self.dev)
        for o0 in range(0, self.N, step):
            o = torch.arange(o0, min(self.N, o0 + step), device=self.dev)
            nu = self.nu[o]
            chi_o, S_o = self.source(o, one.expand(o.numel()), nu)
            e = (o[:, None] * self.R + torch.arange(self.R, device=self.dev)).reshape(-1)
            nu_e = nu.repeat_interleave(self.R, 0)
            far = torch.where((self.pts[1][e] > 0)[:, None], self.far(self.pts, e, nu_e),
                              self.I_bdy[o].repeat_interleave(self.R, 0))
            st = self.inwards(self.pts, e, nu_e, far, chi_o.repeat_interleave(self.R, 0),
                              S_o.repeat_interleave(self.R, 0))
            st = {k: v.reshape(o.numel(), self.R, self.F) for k, v in st.items()}
            n = self.pts[1][e].reshape(-1, self.R)
            r, a = slice(0, half), self.anti[:half]
            h = 0.5 * (st["a"][:, r] + st["a"][:, a])
            den = h + st["pq"][:, r] + st["pq"][:, a]
            u = (S_o[:, None] * h + st["z"][:, r] + st["z"][:, a]) / den
            some = ((n[:, r] + n[:, a]) > 0)[..., None]
            w = 2.0 * self.w[:half][None, :, None]
            J[o] = (w * torch.where(some, u, self.I_bdy[o][:, None])).sum(1)
            lam[o] = (w * torch.where(some, h / den, 0.0)).sum(1) / chi_o
        return J, lam

    def per_line(self, a):
        """Values [N, F] of the sorted bins as [N, transition, root]: transition
        k reads the bins of the k-th line of the sorted list, as the framework's
        spectral discretisation numbers them."""
        return a.gather(1, self.bin_of).reshape(self.N, self.L, self.Q)

    def operator(self, lam):
        """The diagonal operator; its bins are taken by their place in the sorted
        grid: bin l Q + z for root z of transition l."""
        iw = 1.0 / (self.freq[None, :] * self.width[:, None])
        nu, lam = (a.reshape(self.N, self.L, self.Q) for a in (self.nu, lam))
        x = iw[..., None] * (nu - self.freq[None, :, None])
        prof = iw[..., None] / math.sqrt(math.pi) * torch.exp(-x * x)
        return (self.A[None, :, None] * self.qw * nu * prof * lam).sum(-1)

    def rates(self, Jeff, Ls, pop):
        """Populations in statistical equilibrium."""
        ld, N, V = self.m.linedata, self.N, self.V
        M = torch.zeros(N, V, V, dtype=torch.float64, device=self.dev)
        k_IJ, k_JI = self.A + self.Bs * Jeff, self.Ba * Jeff
        opac = H_PLANCK / (4.0 * math.pi) * (pop[:, self.jrad] * self.Ba - pop[:, self.irad] * self.Bs)
        k_IJ = k_IJ - Ls * opac

        def add(i, j, down, up):   # i above j
            M[:, j, i] += down
            M[:, i, i] -= down
            M[:, i, j] += up
            M[:, j, j] -= up

        for k in range(self.L):
            add(int(ld.irad[k]), int(ld.jrad[k]), k_IJ[:, k], k_JI[:, k])
        for cp in ld.colpar:
            tab, n = self.t(cp.tmp), len(cp.tmp)
            top = torch.searchsorted(tab, self.T).clamp(max=n - 1)
            low = (top - 1).clamp(min=0)
            f = torch.where(top > 0, (self.T - tab[low]) / torch.where(top > 0, tab[top] - tab[low], 1.0), 0.0)[:, None]
            Cd, Ce = self.t(cp.Cd), self.t(cp.Ce)
            dens = self.t(self.m.abundance[:, cp.num])[:, None]
            cd, ce = ((x[low] + (x[top] - x[low]) * f) * dens for x in (Cd, Ce))
            for k in range(len(cp.icol)):
                add(int(cp.icol[k]), int(cp.jcol[k]), cd[:, k], ce[:, k])
        M[:, V - 1] = 1.0
        y = torch.zeros(N, V, dtype=torch.float64, device=self.dev)
        y[:, V - 1] = self.ntot
        return torch.linalg.solve(M, y)

    def iterate(self, iterations):
        """The accelerated Lambda iteration from LTE: its count, the populations
        and the (Jlin, Jeff, Jdif) of the last ordinary step."""
        self.grid()
        self.trace()
        pop = self.lte()
        hist, normal, its = [torch.zeros_like(pop)] * 3, 0, 0
        while its < iterations:
            its += 1
            if normal == 4:
                normal, (a, b, c) = 0, hist
                q1, q2, q3 = pop - 2 * a + b, pop - a - b + c, pop - a
                A1, A2, B2, C1, C2_ = ((x * y).sum() for x, y in ((q1, q1), (q1, q2), (q2, q2), (q1, q3), (q2, q3)))
                den = A1 * B2 - A2 * A2
                al, be = (C1 * B2 - C2_ * A2) / den, (C2_ * A1 - C1 * A2) / den
                new = (1.0 - al - be) * pop + al * a + be * b
            else:
                normal += 1
                J, lam = self.field(pop)
                Ls = self.operator(lam)
                Jlin = (self.qw * self.per_line(J)).sum(-1)
                Jdif = H_PLANCK / (4.0 * math.pi) * Ls * pop[:, self.irad]
                new = self.rates(Jlin - Jdif, Ls, pop)
            hist, old, pop = [pop] + hist[:2], pop, new
            change = 2.0 * (new - old).abs() / (new + old)
            if float(torch.where(new > 1e-10 * self.ntot[:, None], change, 0.0).max()) < self.m.pop_prec:
                break
        return its, pop, (Jlin, Jlin - Jdif, Jdif)

    def image(self, ray, width):
        """I_m and I_p of the rest-frame pair along `ray`, from the populations
        after one step from LTE."""
        self.grid()
        self.trace()
        J, lam = self.field(self.lte())
        Ls = self.operator(lam)
        pop = self.lte()
        Jlin = (self.qw * self.per_line(J)).sum(-1)
        pop = self.rates(Jlin - H_PLANCK / (4.0 * math.pi) * Ls * pop[:, self.irad], Ls, pop)
        self.em, self.op = self.lines_of(pop)
        self.grid(width)
        self.bounds_of_bins()
        out = []
        every = torch.arange(self.N, device=self.dev)
        ends = []
        for r in (int(self.anti[ray]), ray):
            d = self.rays[r].expand(self.N, 3)
            s = self.rays[r if r < self.R // 2 else int(self.anti[r])].expand(self.N, 3)
            ends.append(self.walk(every, d, s))
        step = max(1, self.BLOCK // self.F)
        for o0 in range(0, self.N, step):
            o = every[o0:o0 + step]
            nu = self.nu[o]
            chi_o, S_o = self.source(o, torch.ones(o.numel(), dtype=torch.float64, device=self.dev), nu)
            I = [torch.where((p[1][o] > 0)[:, None], self.far(p, o, nu), self.I_bdy[o]) for p in ends]
            both = []
            for x, y in ((1, 0), (0, 1)):   # towards the antipode's end (I_m), towards the ray's (I_p)
                st = self.inwards(ends[x], o, nu, I[x], chi_o, S_o)
                st = self.outwards(ends[y], o, nu, st)
                h = 0.5 * st["a"]
                u = (st["S"] * h + st["z"] + I[y]) / (h + st["pq"] + 1.0)
                none = ((ends[0][1][o] + ends[1][1][o]) == 0)[:, None]
                both.append(torch.where(none, I[y], 2.0 * u - I[y]))
            out.append(both)
        return [torch.cat([b[i] for b in out]) for i in (0, 1)]


def exact(case, seed):
    kind = case["kind"]
    if kind == "train":
        return None   # the order of the minibatches is the network's own
    if kind == "gradient":
        X, Y = training_rows(case, seed)
        return exact_gradient(first_weights(seed), X, Y, normalisation(X, Y))
    points = work(case)["flops"] / FLOPS_PER_POINT_BIN
    if points > 6e10:
        return None   # more than about 20 seconds
    models = models_of(case, seed)
    if kind == "field":
        x = Exact(models[0])
        x.grid()
        x.trace()
        J, lam = x.field(x.lte())
        return {"J": J, "lambda": x.operator(lam)}
    if kind == "image":
        I_m, I_p = Exact(models[0]).image(case["ray"], 1.5e-5)
        return {"I_m": I_m, "I_p": I_p}
    if kind == "batch":
        each = [Exact(m).iterate(case["iterations"]) for m in models]
        return {"iterations": max(e[0] for e in each), "each": torch.tensor([e[0] for e in each]),
                "populations": torch.cat([e[1] for e in each])}
    if case.get("model") == "bands":
        if case["iterations"] > 1:
            return None   # the banded operator's rate equations couple the cells
        _, _, (Jlin, _, _) = Exact(models[0]).iterate(1)
        return {"iterations": 1, "populations": None, "Jeff": [Jlin, None, None]}
    its, pop, J = Exact(models[0]).iterate(case.get("iterations", MAX_ITERATIONS))
    return {"iterations": its, "populations": pop} if kind == "solve" else {"iterations": its, "populations": pop, "Jeff": J}


def exact_gradient(first, X, Y, norm):
    xm, xs, ym, ys = (torch.from_numpy(np.asarray(v, np.float32)).double() for v in norm)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    p = {k: torch.from_numpy(v).double().to(dev).requires_grad_(True) for k, v in first.items()}
    x = ((torch.from_numpy(X).double() - xm) / xs).to(dev)
    y = ((torch.from_numpy(Y).double() - ym) / ys).to(dev)

    def gelu(z):
        return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))

    out = gelu(gelu(x @ p["W1"] + p["b1"]) @ p["W2"] + p["b2"]) @ p["W3"] + p["b3"]
    loss = ((out - y) ** 2).mean()
    loss.backward()
    return {"loss": float(loss.detach()), "grad": {k: v.grad for k, v in p.items()}}
