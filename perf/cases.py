"""What the performance of this package is measured on: the calls that a
user's program makes, from the smallest matrix-vector product to the largest
lattice, in both storage types and every kind of sector.

Each case is a dict of plain values.  Its `kind` names the call:

  hv       y = H x on device vectors (Operator.matvec), the inner product of
           every solve
  bloch    the same in a momentum sector (complex vectors as (re, im) pairs)
  step     one ietl make_step on the caller's vectors (lanczos_step_vectors),
           what the device vector space of the ietl headers calls per step
  lanczos  a device-resident recurrence: start, steps, coefficients, vectors
  solve    one sector solved (sparsediag), operator and all
  batch    many small solves submitted to one batch and run to the end
  measure  the spin sums of an eigenvector: all moments and all site pairs
  sweep    a parameter file: every (Sz, momentum) sector of a ring
"""
import ctypes
import itertools
import json
import math

import numpy as np
import torch

import alps_amd as A

GIB = 1 << 30


def listed():
    return [
        # The smallest call: a 20-site ring, where latency is all.
        {"name": "hv-ring20-f64", "kind": "hv", "lattice": "ring", "sites": 20, "n_up": 10, "dtype": "f64"},
        # A frustrated lattice of ordinary size, the default storage.
        {"name": "hv-j1j2-5x4-f64", "kind": "hv", "lattice": "j1j2", "sites": 20, "width": 4, "n_up": 10,
         "dtype": "f64"},
        # The benchmark's ring.
        {"name": "hv-ring24-f32", "kind": "hv", "lattice": "ring", "sites": 24, "n_up": 12, "dtype": "f32"},
        # Odd length, a sector off the middle, random bonds and a field.
        {"name": "hv-xxz25-f64", "kind": "hv", "lattice": "xxz", "sites": 25, "n_up": 11, "dtype": "f64"},
        # The largest: the 6x5 J1-J2 lattice, 155 million states.
        {"name": "hv-j1j2-6x5-f32", "kind": "hv", "lattice": "j1j2", "sites": 30, "width": 5, "n_up": 15,
         "dtype": "f32"},
        # A momentum sector of the ring.
        {"name": "bloch-ring24-k0-f32", "kind": "bloch", "lattice": "ring", "sites": 24, "n_up": 12, "k": 0,
         "dtype": "f32"},
        # The ietl template's step on an open random chain.
        {"name": "step-xxz21-f64", "kind": "step", "lattice": "xxz", "sites": 21, "n_up": 10, "dtype": "f64"},
        # The recurrence itself, host reads at its end only.
        {"name": "lanczos-ring24-f32", "kind": "lanczos", "lattice": "ring", "sites": 24, "n_up": 12, "steps": 32,
         "dtype": "f32"},
        # The measurements of one eigenvector: averages, correlations, structure factors.
        {"name": "measure-ring24-f64", "kind": "measure", "lattice": "ring", "sites": 24, "n_up": 12,
         "dtype": "f64"},
        # One ground state from a model to its energy.
        {"name": "solve-xxz24-f32", "kind": "solve", "lattice": "xxz", "sites": 24, "n_up": 12, "nev": 1,
         "dtype": "f32"},
        # Many small random chains at once, as a disorder average submits them.
        {"name": "batch-xxz-64-f32", "kind": "batch", "lattice": "xxz", "sites": 20, "least": 12, "count": 64,
         "dtype": "f32"},
        # The parameter file's default: every Sz and momentum of a periodic lattice.
        {"name": "sweep-ring16-f64", "kind": "sweep", "lattice": "ring", "sites": 16, "dtype": "f64"},
    ]


def draw(rng):
    kind = rng.choice(["hv", "hv", "hv", "hv", "bloch", "step", "lanczos", "measure", "solve", "batch", "sweep"])
    dtype = rng.choice(["f32", "f64"])
    c = {"kind": kind, "dtype": dtype}
    if kind in ("hv", "step", "lanczos", "measure", "solve"):
        top = {"hv": 27, "step": 25, "lanczos": 24, "measure": 23, "solve": 23}[kind]
        c["lattice"] = rng.choice(["ring", "xxz", "xxz", "j1j2"])
        if c["lattice"] == "j1j2":
            c["width"] = rng.choice([3, 4, 5])
            c["sites"] = c["width"] * rng.randint(-(-16 // c["width"]), top // c["width"])
        else:
            c["sites"] = rng.randint(20 if kind == "hv" else 12, top)
        half = c["sites"] // 2
        c["n_up"] = rng.randint(max(3, half - 4), min(c["sites"] - 3, half + 4))
        if kind == "lanczos":
            c["steps"] = rng.randint(8, 32)
        if kind == "solve":
            c["nev"] = rng.randint(1, 2)
    elif kind == "bloch":
        c["lattice"] = "ring"
        c["sites"] = rng.randint(22, 24)
        c["n_up"] = rng.randint(c["sites"] // 2 - 3, c["sites"] // 2 + 3)
        c["k"] = rng.randint(0, c["sites"] - 1)
    elif kind == "batch":
        c["lattice"] = "xxz"
        c["sites"] = rng.randint(14, 20)
        c["least"] = 12
        c["count"] = rng.randint(8, 64)
    else:
        c["lattice"] = "ring"
        c["sites"] = rng.randint(9, 15)
        c["dtype"] = "f64"
    return c


# ---------------------------------------------------------------------------
# models
# ---------------------------------------------------------------------------
def bonds_of(case, seed, sites=None):
    """(site1, site2, jz, jxy, field) of a case's model."""
    n = sites or case["sites"]
    if case["lattice"] == "ring":
        s = np.arange(n)
        return s, (s + 1) % n, np.ones(n), np.ones(n), 0.0
    if case["lattice"] == "xxz":  # random bonds, anisotropy and field; open or periodic
        rng = np.random.default_rng([seed, n])
        nb = n if rng.integers(2) else n - 1
        s = np.arange(nb)
        j = rng.uniform(0.5, 1.5, nb)
        return s, (s + 1) % n, rng.uniform(0.0, 2.0) * j, j, float(rng.uniform(0.0, 0.5))
    w = case["width"]  # j1j2: periodic square lattice, J1 = 1, J2 = 0.5
    length = n // w
    s1, s2, j = [], [], []
    for x, y in itertools.product(range(length), range(w)):
        for dx, dy, v in ((0, 1, 1.0), (1, 0, 1.0), (1, 1, 0.5), (1, -1, 0.5)):
            s1.append(x * w + y)
            s2.append((x + dx) % length * w + (y + dy) % w)
            j.append(v)
    return np.array(s1), np.array(s2), np.array(j), np.array(j), 0.0


def model_of(case, seed, sites=None, n_up=None):
    s1, s2, jz, jxy, h = bonds_of(case, seed, sites)
    return A.SpinModel(sites or case["sites"], s1, s2, jz, jxy, case["n_up"] if n_up is None else n_up, h=h)


def ring_translations(n, k):
    t = np.arange(n)
    return np.exp(2j * np.pi * k * t / n), (t[:, None] + t[None, :]) % n


def chain_sizes(case, seed):
    return np.random.default_rng([seed, 7]).integers(case["least"], case["sites"] + 1, case["count"])


class _Memory:
    """A device vector's storage as torch sees it (it keeps the vector)."""

    def __init__(self, vector):
        self.vector = vector
        self.__cuda_array_interface__ = {
            "shape": (vector.n,), "typestr": "<f4" if vector.dtype == A.F32 else "<f8",
            "data": (vector.data_ptr(), False), "strides": None, "version": 3}


def view(vector):
    return torch.as_tensor(_Memory(vector), device="cuda")


# ---------------------------------------------------------------------------
# the calls
# ---------------------------------------------------------------------------
def prepare(case, seed):
    kind, dtype = case["kind"], case["dtype"]
    s = {"kind": kind, "case": case, "seed": seed}
    if kind == "batch":
        s["models"] = [model_of(case, seed + i, int(n), (int(n) + 1) // 2)
                       for i, n in enumerate(chain_sizes(case, seed))]
        s["batch"] = A.Batch(dtype, hbm_bytes=32 * GIB)
        return s
    if kind == "sweep":
        s["text"] = ('LATTICE="chain lattice"; MODEL="spin"; local_S=1/2; L=%d; Jxy=1; Jz=%r; NUMBER_EIGENVALUES=2; '
                     'CONSERVED_QUANTUMNUMBERS="Sz"; ED_SEED=%d; {}' % (case["sites"], sweep_jz(seed), seed)).encode()
        s["json"] = ctypes.create_string_buffer(1 << 20)
        s["length"] = ctypes.c_size_t()
        return s
    s["model"] = model_of(case, seed)
    if kind == "solve":
        return s
    op = A.Operator(s["model"], ring_translations(case["sites"], case["k"]) if kind == "bloch" else None)
    s["op"] = op
    if kind == "lanczos":
        s["lz"] = A.Lanczos(op, dtype, max_steps=case["steps"])
        s["out"] = [A.Vector(op.dim, dtype) for _ in range(2)]
        s["views"] = [view(v) for v in s["out"]]
        return s
    s["x"] = A.Vector(op.dim, dtype)
    s["x"].fill_random(seed)
    if kind == "measure":
        s["i"], s["j"] = np.triu_indices(case["sites"], 1)
        return s
    s["y"] = A.Vector(op.dim, dtype)
    s["view"] = view(s["y"])
    if kind == "step":
        s["prev"] = A.Vector(op.dim, dtype)
        s["prev"].fill_random(seed + 1)
    return s


def run(s):
    kind = s["kind"]
    if kind in ("hv", "bloch"):
        s["op"].matvec(s["x"], s["y"])
        return s["view"]
    if kind == "step":
        alpha, beta = A.lanczos_step_vectors(s["op"], s["prev"], s["x"], s["y"], 0.75)
        return {"alpha": alpha, "beta": beta, "w": s["view"]}
    if kind == "lanczos":
        lz, (prev, cur) = s["lz"], s["out"]
        lz.start(s["seed"])
        lz.steps(s["case"]["steps"] - 1)
        alpha, beta = lz.coefficients()
        if A.lib().alps_ed_lanczos_vectors(lz.handle, prev.handle, cur.handle):  # into vectors that are kept
            raise RuntimeError("lanczos_vectors")
        return {"alpha": alpha, "beta": beta, "prev": s["views"][0], "cur": s["views"][1]}
    if kind == "measure":
        n2, sz, szsz = s["op"].spin_moments(s["x"])
        return {"norm2": n2, "sz": sz, "szsz": szsz, "flip": s["op"].flip_pairs(s["x"], s["i"], s["j"])}
    if kind == "solve":
        return A.sparsediag(s["model"], nev=s["case"]["nev"], seed=s["seed"], dtype=s["case"]["dtype"])["ev"]
    if kind == "batch":
        b = s["batch"]
        tickets = [b.submit(m, nev=1, seed=i) for i, m in enumerate(s["models"])]
        b.run()
        b.completed()
        return np.array([b.result(t)["ev"][0] for t in tickets])
    if A.lib().alps_ed_run_parameter_file(s["text"], s["json"], len(s["json"]), ctypes.byref(s["length"])):
        raise RuntimeError(A.lib().alps_ed_last_error().decode())
    (task,) = json.loads(s["json"].value.decode())["tasks"]
    ev = np.zeros((len(task["sectors"]), 2))
    for row, sector in zip(ev, task["sectors"]):
        row[: len(sector["eigenvalues"])] = sector["eigenvalues"]
    return ev


def sweep_jz(seed):
    return float(np.random.default_rng([seed, 11]).integers(300, 900)) / 1000


# ---------------------------------------------------------------------------
# the work that a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    es = 4 if case["dtype"] == "f32" else 8
    kind = case["kind"]
    if kind in ("batch", "sweep"):  # about 60 steps a solve: three vectors moved and one product each
        if kind == "batch":
            sizes = [(int(n), (int(n) + 1) // 2) for n in chain_sizes(case, 0)]
            dims, bonds = [math.comb(n, k) for n, k in sizes], [n for n, _ in sizes]
        else:
            n = case["sites"]
            dims, bonds = [2 ** n], [n]
        rows = 60.0 * sum(dims)
        return {"bytes": 3 * es * rows * (2 if kind == "sweep" else 1),
                "flops": 60.0 * sum(d * (2 + b) * (4 if kind == "sweep" else 1) for d, b in zip(dims, bonds))}
    n, k = case["sites"], case["n_up"]
    dim = math.comb(n, k)
    bonds = 2 * n * 2 if case["lattice"] == "j1j2" else n
    flips = bonds * 2.0 * k * (n - k) / (n * (n - 1))  # flipping bonds of a row, on average
    product = 2 * dim * (1 + flips)
    if kind == "hv":
        return {"bytes": 2 * es * dim, "flops": product}
    if kind == "bloch":
        return {"bytes": 4 * es * dim / n, "flops": 4 * product / n}
    if kind == "step":
        return {"bytes": 3 * es * dim, "flops": product + 10 * dim}
    if kind == "lanczos":
        return {"bytes": 3 * es * dim * case["steps"], "flops": (product + 10 * dim) * case["steps"]}
    if kind == "solve":  # about three steps a site
        return {"bytes": 3 * es * dim * 3 * n, "flops": (product + 10 * dim) * 3 * n}
    pairs = n * (n - 1) / 2
    return {"bytes": 2 * es * dim, "flops": dim * (2 * pairs + pairs * 2 * k * (n - k) / (n * (n - 1)))}


# ---------------------------------------------------------------------------
# what the calls return, in 64 bits
# ---------------------------------------------------------------------------
def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _uniform(seed, n, dtype):
    """Element i of the counter-based start vector: splitmix64 of seed + (i + 1) * golden gamma, on [-1, 1)."""
    def mul(z, c):  # modulo 2^64
        return z * (c - (1 << 64) if c >> 63 else c)

    def shr(z, b):
        return (z >> b) & ((1 << (64 - b)) - 1)

    z = mul(torch.arange(1, n + 1, dtype=torch.int64, device=_device()), 0x9E3779B97F4A7C15) + seed
    z = mul(z ^ shr(z, 30), 0xBF58476D1CE4E5B9)
    z = mul(z ^ shr(z, 27), 0x94D049BB133111EB)
    z = z ^ shr(z, 31)
    v = -1.0 + 2.0 * (shr(z, 11).double() * 2.0 ** -53)
    return v.float().double() if dtype == "f32" else v


class _Sector:
    """The states of a sector in ascending order, and the product with H."""

    def __init__(self, n, k, model):
        dev = _device()
        self.n, self.k = n, k
        low = min(n, 15)
        word = torch.arange(1 << max(low, n - low), device=dev)
        count = torch.zeros_like(word)
        for b in range(16):
            count += (word >> b) & 1
        self.low = low
        parts = []
        span = 1 << min(n, 24)
        for first in range(0, 1 << n, span):
            s = torch.arange(first, first + span, device=dev)
            parts.append(s[count[s & ((1 << low) - 1)] + count[s >> low] == k])
        self.states = torch.cat(parts)
        self.dim = len(self.states)
        lo = word[: 1 << low]
        order = torch.argsort(count[lo] * (1 << low) + lo)
        start = torch.cumsum(torch.bincount(count[lo], minlength=low + 1), 0)
        place = torch.empty_like(lo)
        place[order] = torch.arange(len(lo), device=dev)
        first = torch.where(count[lo] > 0, start[(count[lo] - 1).clamp(min=0)], 0)
        self.lo_rank = place - first
        self.hi_base = torch.searchsorted(self.states, torch.arange(1 << (n - low), device=dev) << low)
        s1, s2, jz, jxy, self.h = model
        self.bonds = [(n - 1 - int(a), n - 1 - int(b), float(z), float(xy)) for a, b, z, xy in zip(s1, s2, jz, jxy)]
        self.kept = None

    def rank(self, s):
        return self.hi_base[s >> self.low] + self.lo_rank[s & ((1 << self.low) - 1)]

    def diagonal(self):
        # -h Sz over all sites is the same in every state of the sector
        d = torch.full((self.dim,), -self.h * (self.k - 0.5 * self.n), dtype=torch.float64, device=self.states.device)
        for a, b, z, _ in self.bonds:
            d += (0.25 - 0.5 * (((self.states >> a) ^ (self.states >> b)) & 1).double()) * z
        return d

    def flips(self):
        for a, b, _, xy in self.bonds:
            anti = ((self.states >> a) ^ (self.states >> b)) & 1 == 1
            yield anti, torch.where(anti, self.states ^ ((1 << a) | (1 << b)), self.states), 0.5 * xy

    def keep(self):
        """Every flip's target and coefficient, kept for many products."""
        self.kept = [(self.rank(t), anti.double() * c) for anti, t, c in self.flips()] if self.dim else []
        self.diag = self.diagonal()
        return self

    def product(self, x):
        if self.kept is not None:
            y = self.diag * x
            for at, c in self.kept:
                y += c * x[at]
            return y
        y = self.diagonal() * x
        for anti, t, c in self.flips():
            y += torch.where(anti, c * x[self.rank(t)], 0.0)
        return y


def _lowest(sector, nev):
    """The lowest distinct levels of a sector: dense, or Lanczos with every vector orthogonalized twice."""
    dev = sector.states.device
    sector.keep()
    if sector.dim <= 1200:
        h = torch.zeros((sector.dim, sector.dim), dtype=torch.float64, device=dev)
        row = torch.arange(sector.dim, device=dev)
        for at, c in sector.kept:
            h.index_put_((row, at), c, accumulate=True)
        h += torch.diag(sector.diag)
        return _distinct(np.linalg.eigvalsh(h.cpu().numpy()), nev)
    most = 260
    basis = torch.zeros((most + 1, sector.dim), dtype=torch.float64, device=dev)
    v = _uniform(17, sector.dim, "f64")
    basis[0] = v / v.norm()
    alpha, beta, last = [], [], None
    for j in range(most):
        w = sector.product(basis[j])
        alpha.append(float(w @ basis[j]))
        for _ in range(2):
            w -= basis[: j + 1].T @ (basis[: j + 1] @ w)
        beta.append(float(w.norm()))
        basis[j + 1] = w / beta[-1]
        if j % 10 == 9:
            t = np.diag(alpha) + np.diag(beta[:-1], 1) + np.diag(beta[:-1], -1)
            e, z = np.linalg.eigh(t)
            if np.all(np.abs(beta[-1] * z[-1, :nev]) < 1e-9):  # a Ritz value's error is the square of that
                return e[:nev]
            last = e[:nev]
    return last


def _distinct(values, nev):
    out = []
    for v in values:
        if not out or v - out[-1] > 1e-9 * max(1.0, abs(v)):
            out.append(float(v))
        if len(out) == nev:
            break
    return np.array(out)


class _Orbits:
    """Translation orbits of a ring's states: the smallest state of each state's orbit and the first shift to it."""

    def __init__(self, sector):
        n, s = sector.n, sector.states
        self.rep, self.shift = s.clone(), torch.zeros_like(s)
        self.fixed = torch.zeros((n, sector.dim), dtype=torch.bool, device=s.device)
        for t in range(n):  # site i to i + t: bit n - 1 - i moves down by t
            moved = (s >> t) | ((s & ((1 << t) - 1)) << (n - t)) if t else s
            less = moved < self.rep
            self.rep = torch.where(less, moved, self.rep)
            self.shift = torch.where(less, t, self.shift)
            self.fixed[t] = moved == s

    def at(self, sector, k):
        """Kept representatives' ranks, every state's place among them (-1: none), phases and norms."""
        n = sector.n
        phase = torch.exp(2j * math.pi * k * torch.arange(n, device=self.rep.device).double() / n)
        reps = torch.nonzero(self.rep == sector.states)[:, 0]
        weight = (phase[:, None] * self.fixed[:, reps]).sum(0).abs().sqrt()
        kept = reps[weight >= 0.01]
        norm = weight[weight >= 0.01] / math.sqrt(n)
        place = torch.full((sector.dim,), -1, dtype=torch.int64, device=self.rep.device)
        place[kept] = torch.arange(len(kept), device=place.device)
        return kept, place[sector.rank(self.rep)], phase[self.shift], norm


def _exact_bloch(case, seed):
    sector = _Sector(case["sites"], case["n_up"], bonds_of(case, seed))
    kept, place, phase, norm = _Orbits(sector).at(sector, case["k"])
    w = torch.view_as_complex(_uniform(seed, 2 * len(kept), case["dtype"]).reshape(-1, 2))
    full = torch.where(place >= 0, phase * (norm * w)[place.clamp(min=0)], 0.0)
    y = torch.complex(sector.product(full.real), sector.product(full.imag))
    return torch.view_as_real(y[kept] / norm).reshape(-1)


def _exact_sweep(case, seed):
    n = case["sites"]
    s = np.arange(n)
    model = (s, (s + 1) % n, np.full(n, sweep_jz(seed)), np.ones(n), 0.0)
    rows = {}
    for up in range(n // 2 + 1):  # without a field, n - up has the levels of up
        sector = _Sector(n, up, model).keep()
        orbits = _Orbits(sector)
        for k in range(n // 2 + 1):  # a reflection takes k to -k
            kept, place, phase, norm = (v.cpu().numpy() for v in orbits.at(sector, k))
            h = np.zeros((len(kept), len(kept)), dtype=complex)
            h[np.arange(len(kept)), np.arange(len(kept))] = sector.diag.cpu().numpy()[kept]
            for at, c in sector.kept:
                to, c = at.cpu().numpy()[kept], c.cpu().numpy()[kept]
                sel = np.nonzero((c != 0) & (place[to] >= 0))[0]
                np.add.at(h, (sel, place[to[sel]]), c[sel] * phase[to[sel]] * norm[place[to[sel]]] / norm[sel])
            ev = _distinct(np.linalg.eigvalsh(h), 2) if len(kept) else np.zeros(0)
            for u in {up, n - up}:
                for q in {k, (n - k) % n}:
                    if len(kept):
                        rows[u, q] = np.concatenate([ev, np.zeros(2 - len(ev))])
    return np.array([rows[key] for key in sorted(rows)])


def exact(case, seed):
    kind = case["kind"]
    if not torch.cuda.is_available() and math.comb(case["sites"], case["sites"] // 2) > 3e6:
        return None
    if kind == "bloch":
        return _exact_bloch(case, seed)
    if kind == "sweep":
        return _exact_sweep(case, seed)
    if kind == "batch":
        return np.array([_lowest(_Sector(int(n), (int(n) + 1) // 2, bonds_of(case, seed + i, int(n))), 1)[0]
                         for i, n in enumerate(chain_sizes(case, seed))])
    sector = _Sector(case["sites"], case["n_up"], bonds_of(case, seed))
    if kind == "solve":
        return _lowest(sector, case["nev"])
    x = _uniform(seed, sector.dim, case["dtype"])
    if kind == "hv":
        return sector.product(x)
    if kind == "step":
        w = sector.product(x)
        alpha = w @ x
        w = w - alpha * x - 0.75 * _uniform(seed + 1, sector.dim, case["dtype"])
        return {"alpha": float(alpha), "beta": float(w.norm()), "w": w / w.norm()}
    if kind == "lanczos":
        sector.keep()
        prev, cur, alpha, beta = torch.zeros_like(x), x / x.norm(), [], [0.0]
        for _ in range(case["steps"]):
            w = sector.product(cur)
            alpha.append(float(w @ cur))
            w = w - alpha[-1] * cur - beta[-1] * prev
            beta.append(float(w.norm()))
            prev, cur = cur, w / beta[-1]
        return {"alpha": np.array(alpha), "beta": np.array(beta[1:]), "prev": prev, "cur": cur}
    n = case["sites"]  # measure
    weight = x * x
    spin = torch.stack([((sector.states >> (n - 1 - i)) & 1).double() - 0.5 for i in range(n)])
    i, j = np.triu_indices(n, 1)
    flip = []
    for a, b in zip(i.tolist(), j.tolist()):  # a down and b up, both turned
        up, down = 1 << (n - 1 - b), 1 << (n - 1 - a)
        r = torch.nonzero((sector.states & up != 0) & (sector.states & down == 0))[:, 0]
        flip.append(float(x[r] @ x[sector.rank(sector.states[r] ^ (up | down))]))
    return {"norm2": float(weight.sum()), "sz": spin @ weight, "szsz": (spin * weight) @ spin.T,
            "flip": np.array(flip)}
