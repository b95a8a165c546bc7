"""What the framework's speed is measured on.

Each case is one short run as a program makes it: Initialize, a number of D3Q27 BGK steps, then the
read-back of what the run is made for (the p, u, v, w fields on the host, with the diagnostics or the
drag where such a run reports them). The handle is the program's own and is kept between passes.

listed() holds the runs, draw() gives others of the same ranges, prepare() makes a handle whose physics
(rate, speeds, noise) come from the seed, run() makes one pass, work() says what a pass cannot do
without, and exact() computes the same fields in 64 bits with plain torch and numpy.
"""
import math

import numpy as np
import torch

from imexlb_amd import LBM, Ensemble

PI = 3.1415926  # the value of the reference's sources
ELEM = {"f64": 8, "f32": 4, "f16": 2}
NAMES = ("p", "u", "v", "w")


def _flow(name, flow, n, steps, dtype="f64", storage="pull", tau=0.0153, **more):
    nx, ny, nz = n
    c = {"flow": flow, "nx": nx, "ny": ny, "nz": nz, "steps": steps, "dtype": dtype, "storage": storage,
         "tau": tau, "calls": "step"}
    c.update(more)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # a small box stepped with the reference driver's six calls: what a call and a launch cost
        _flow("tgv 32 loop f64", "tgv", (32, 32, 32), 10, calls="loop"),
        # the Taylor-Green box at Re 100 whose 1000 steps are compared with a CPU
        _flow("tgv 64 f64 aa", "tgv", (64, 64, 64), 1000, storage="aa"),
        # an uneven small box in the compact storage: one member's size of an ensemble, run alone
        _flow("tgv 45x37x51 f16 aa", "tgv", (45, 37, 51), 501, "f16", "aa"),
        # an uneven box of ordinary size in single precision
        _flow("tgv 301x203x157 f32", "tgv", (301, 203, 157), 300, "f32"),
        # the reference's own 256^3 run: 100 steps with a report every 10
        _flow("tgv 256 report f64", "tgv", (256, 256, 256), 100, tau=0.0038, every=10),
        # the precision sweep's 512^3 box at Re 1600, in double and in the compact storage
        _flow("tgv 512 f64 aa", "tgv", (512, 512, 512), 100, storage="aa", tau=0.0076),
        _flow("tgv 512 f16 aa", "tgv", (512, 512, 512), 300, "f16", "aa", tau=0.0076),
        # the lid-driven cavity at Re 400: the 1000 steps between two comparisons of its fields
        _flow("cavity 128 f64 aa", "cavity", (128, 128, 128), 1000, storage="aa", tau=0.096),
        # the reference's own inputs with the reference's own boundaries
        _flow("cavity 100 faithful", "cavity faithful", (100, 100, 100), 200, tau=0.096),
        _flow("sphere 512x128x128 faithful", "sphere faithful", (512, 128, 128), 100, tau=0.024),
        # the channel with a ball of 40 cells in the compact storage, with its drag
        _flow("channel 512x256x256 f16", "channel", (512, 256, 256), 600, "f16", tau=0.03),
        # many small domains of uneven size stepped together
        {"name": "ensemble 15 f32", "flow": "ensemble", "edges": "32 48 64 80 96 96 80 64 48 32 96 64 80 32 48",
         "steps": 500, "dtype": "f32", "storage": "pull", "tau": 0.03},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _box(rng, cells):
    """Three edges of about `cells` cells: round ones as often as not."""
    e = cells ** (1 / 3)
    stretch = [_log(rng, 0.6, 1.6) for _ in range(3)]
    stretch = [s / (stretch[0] * stretch[1] * stretch[2]) ** (1 / 3) for s in stretch]
    if rng.random() < 0.5:
        return tuple(max(16, 8 * round(e * s / 8)) for s in stretch)
    return tuple(max(12, round(e * s)) for s in stretch)


def draw(rng):
    flow = rng.choice(["tgv", "tgv", "tgv", "cavity", "cavity faithful", "sphere faithful", "channel", "ensemble"])
    if flow == "ensemble":
        edges = [rng.choice([32, 48, 64, 80, 96]) if rng.random() < 0.7 else rng.randint(24, 96)
                 for _ in range(rng.randint(3, 15))]
        return {"flow": flow, "edges": " ".join(map(str, edges)), "steps": rng.randint(50, 600),
                "dtype": rng.choice(["f32", "f32", "f64", "f16"]), "storage": rng.choice(["pull", "pull", "aa"]),
                "tau": round(_log(rng, 0.03, 0.1), 4)}
    cells = _log(rng, 8e3, 8e7 if flow in ("tgv", "channel") else 1.7e7)
    updates = _log(rng, 1e7, 4e9)
    dtype, storage, calls, every = "f64", "pull", "step", 0
    if not flow.endswith("faithful"):
        dtype = rng.choice(["f64", "f64", "f32", "f16"])
        if flow != "channel":
            storage = rng.choice(["pull", "aa"])
    if flow == "tgv" and rng.random() < 0.25:
        calls = "loop"
    elif rng.random() < 0.2:
        every = 10
    n = _box(rng, cells)
    if flow == "sphere faithful":  # long enough for the reference's ball, centred at nx / 8
        n = (max(72, n[0], 2 * n[1]), max(24, n[1]), max(24, n[2]))
        n = (n[0], max(n[1], n[0] // 4), max(n[2], n[0] // 4))
    if flow == "channel":
        n = (max(40, 2 * n[0]), max(24, n[1]), max(24, n[2]))
    steps = int(min(1000, max(10, updates / (n[0] * n[1] * n[2]))))
    if calls == "loop":
        steps = min(steps, 100)
    # rates at which the flow stays stable: the reference's cavity walls need the most viscosity
    tau = _log(rng, *{"tgv": (0.01, 0.1), "channel": (0.01, 0.1), "cavity faithful": (0.09, 0.2)}.get(flow, (0.03, 0.1)))
    more = {"every": every} if every else {}
    return _flow(None, flow, n, steps, dtype, storage, round(tau, 4), calls=calls, **more)


def _physics(case, seed):
    """What the seed decides of a run: the rate, the speeds and the noise."""
    r = np.random.RandomState(seed % (1 << 32))
    k = {"tau": case["tau"] * (1.0 + 0.1 * r.rand()), "u0": 0.04 + 0.02 * r.rand(), "lid_u": 0.05 + 0.05 * r.rand(),
         "seed": int(r.randint(1, 1 << 30))}
    if case["flow"] == "ensemble":
        k["domains"] = []
        for i, e in enumerate(case["edges"].split()):
            k["domains"].append({"case_id": i % 2, "nx": int(e), "ny": int(e), "nz": int(e),
                                 "tau0": case["tau"] * (1.0 + r.rand()), "rho0": 1.0, "u0": 0.04 + 0.02 * r.rand(),
                                 "lid_u": 0.05 + 0.05 * r.rand()})
    return k


def _ball(case):
    """The channel's ball: 40 of 256 cells across, a quarter of the way down the channel."""
    d = min(case["ny"], case["nz"])
    return float(case["nx"] // 4), float(case["ny"] // 2), float(case["nz"] // 2), d * 20 / 256


def prepare(case, seed):
    k = _physics(case, seed)
    if case["flow"] == "ensemble":
        return {"case": case, "ensemble": Ensemble(k["domains"], dtype=case["dtype"], storage=case["storage"])}
    kind, _, faithful = case["flow"].partition(" ")
    args = {"case": {"channel": "sphere"}.get(kind, kind), "mode": "faithful" if faithful or kind == "tgv" else "config"}
    if kind == "channel":
        args["sphere"] = _ball(case)
    lbm = LBM(case["nx"], case["ny"], case["nz"], k["tau"], u0=k["u0"], lid_u=k["lid_u"], seed=k["seed"],
              dtype=case["dtype"], storage=case["storage"], **args)
    return {"case": case, "lbm": lbm}


def run(state):
    case = state["case"]
    if case["flow"] == "ensemble":
        e = state["ensemble"]
        e.Initialize()
        e.step(case["steps"])
        return {"finite": np.array(e.status()), "fields": [e.moments(d) for d in range(len(e.domains))]}
    g = state["lbm"]
    g.Initialize()
    if case["calls"] == "loop":
        g.setup_subdomain()
        for _ in range(case["steps"]):
            g.Collision()
            g.pack()
            g.exchange()
            g.unpack()
            g.Streaming()
            g.Update()
    else:
        g.step(case["steps"], case.get("every"))
    out = dict(zip(NAMES, g.moments()))
    if case["flow"] == "tgv":
        out["energy and mass"] = np.array(g.diagnostics())
    if case["flow"] == "channel":
        out["force"] = g.sphere_force()
    return out


def work(case):
    """Per cell and step the 27 populations read and written once, as they are stored; at the end (and at
    each report) four fields of 64 bits. About 350 operations for a cell's moments, equilibria and update."""
    if case["flow"] == "ensemble":
        cells = sum(int(e) ** 3 for e in case["edges"].split())
    else:
        cells = case["nx"] * case["ny"] * case["nz"]
    reports = case["steps"] // case["every"] if case.get("every") else 1
    per = 2 * 27 * ELEM[case["dtype"]] + (1 if case["flow"] in ("channel", "sphere faithful") else 0)
    return {"bytes": float(cells) * (case["steps"] * per + reports * 32), "flops": 350.0 * cells * case["steps"]}


# ---------------------------------------------------------------- the same in 64 bits

DIRS = [(x, y, z) for z in (-1, 0, 1) for y in (-1, 0, 1) for x in (-1, 0, 1)]
OPP = [DIRS.index((-x, -y, -z)) for x, y, z in DIRS]
WEIGHT = [(8 / 27, 2 / 27, 1 / 54, 1 / 216)[abs(x) + abs(y) + abs(z)] for x, y, z in DIRS]
G = 3  # ghost layers of the runs with the reference's boundaries


def _feq_matrix(device):
    """feq = matrix @ (p, u, v, w, uu, vv, ww, uv, uw, vw)."""
    rows = []
    for (x, y, z), t in zip(DIRS, WEIGHT):
        q = [4.5 * x * x - 1.5, 4.5 * y * y - 1.5, 4.5 * z * z - 1.5, 9.0 * x * y, 9.0 * x * z, 9.0 * y * z]
        rows.append([3.0 * t, 3.0 * t * x, 3.0 * t * y, 3.0 * t * z] + [t * v for v in q])
    return torch.tensor(rows, dtype=torch.float64, device=device)


class _Exact:
    """One flow in 64 bits: f[direction][z, y, x], with ghost layers where the reference has them."""

    def __init__(self, flow, n, tau, u0, lid_u, seed=0, ball=None):
        self.flow, self.n, self.den, self.u0, self.lid = flow, n, tau + 0.5, u0, lid_u
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.A = _feq_matrix(self.dev)
        self.M = torch.tensor([[1 / 3] * 27] + [[float(d[a]) for d in DIRS] for a in range(3)],
                              dtype=torch.float64, device=self.dev)
        self.g = G if flow.endswith("faithful") else 0
        nx, ny, nz = n
        kw = {"dtype": torch.float64, "device": self.dev}
        x = torch.arange(-self.g, nx + self.g, **kw).view(1, 1, -1)
        y = torch.arange(-self.g, ny + self.g, **kw).view(1, -1, 1)
        z = torch.arange(-self.g, nz + self.g, **kw).view(-1, 1, 1)
        shape = (z.numel(), y.numel(), x.numel())
        self.m = torch.zeros((4,) + shape, **kw)
        self.solid = None
        if flow == "tgv":
            a, b, c = x / nx * 2 * PI, y / ny * 2 * PI, z / nz * 2 * PI
            self.m[0] = 1 / 3 + u0 * u0 / 16 * (torch.cos(2 * a) + torch.cos(2 * b)) * (torch.cos(2 * c) + 2)
            self.m[1] = u0 * torch.sin(a) * torch.cos(b) * torch.cos(c)
            self.m[2] = -u0 * torch.cos(a) * torch.sin(b) * torch.cos(c)
        elif flow == "cavity":
            self.m[0] = 1 / 3
        elif flow == "channel":
            self.solid = (x - ball[0]) ** 2 + (y - ball[1]) ** 2 + (z - ball[2]) ** 2 <= ball[3] ** 2
            self.m[0] = 1 / 3
            self.m[1] = u0
            self.m[1].masked_fill_(self.solid, 0.0)
            self.fin = self.A[:, 0] / 3 + self.A[:, 1] * u0 + self.A[:, 4] * u0 * u0
        elif flow == "sphere faithful":
            c, r = (nx - 1) // 8, (nx - 1) / 64
            self.solid = (x - c) ** 2 + (y - c) ** 2 + (z - c) ** 2 <= r * r
            i, j, k = np.meshgrid(*(np.arange(v, dtype=np.uint64) for v in shape[::-1]), indexing="ij", sparse=True)
            at = (i * np.uint64(shape[1]) + j) * np.uint64(shape[0]) + k
            noise = torch.from_numpy((_hash(np.uint64(seed) + at * np.uint64(0x9E3779B97F4A7C15)) % np.uint64(100))
                                     .astype(np.float64).transpose(2, 1, 0).copy()).to(self.dev)
            self.profile = u0 * 4 * z * (nz - 1 - z) / (nz - 1) ** 2
            self.m[1] = (self.profile * (1 + noise * 0.001)).masked_fill(self.solid, 0.0)
        self.f = [torch.empty(shape, **kw) for _ in DIRS]
        for s in self._slabs(shape):
            for q, part in enumerate(self._feq(self.m[:, s])):
                self.f[q][s] = part
        self.bounce = []
        if flow == "channel":  # fluid cells whose link comes from the ball
            for q, d in enumerate(DIRS):
                near = torch.roll(self.solid, d[::-1], (0, 1, 2)) & ~self.solid
                self.bounce.append(near.nonzero(as_tuple=True))
        if flow == "sphere faithful":  # solid cells beside a fluid cell
            for q, (a, b, c) in enumerate(DIRS):
                near = self.solid & ~torch.roll(self.solid, (-c, -b, -a), (0, 1, 2))
                near[:G], near[-G:], near[:, :G], near[:, -G:], near[:, :, :G], near[:, :, -G:] = (False,) * 6
                self.bounce.append(near.nonzero(as_tuple=True))

    def _slabs(self, shape):
        """Slabs in z of some millions of cells."""
        step = max(1, (1 << 23) // (shape[1] * shape[2]))
        return [slice(a, min(shape[0], a + step)) for a in range(0, shape[0], step)]

    def _feq(self, m):
        b = m.reshape(4, -1)
        p, u, v, w = b
        basis = torch.stack([p, u, v, w, u * u, v * v, w * w, u * v, u * w, v * w])
        return (self.A @ basis).view((27,) + m.shape[1:])

    def _inside(self, t):
        g = self.g
        return t if g == 0 else t[..., g:-g, g:-g, g:-g]

    def collide(self):
        f, m = [self._inside(t) for t in self.f], self._inside(self.m)
        for s in self._slabs(m.shape[1:]):
            for t, feq in zip(f, self._feq(m[:, s])):
                t[s] += (feq - t[s]) / self.den

    def step(self):
        self.collide()
        if self.g:
            self._ghosts()
            self._stream_ghosts()
        else:
            self._stream()
        self._update()

    def _stream(self):
        old = self.f
        nx, ny, nz = self.n
        self.f = []
        for q, (a, b, c) in enumerate(DIRS):
            new, back = torch.roll(old[q], (c, b, a), (0, 1, 2)), old[OPP[q]]
            if self.flow == "cavity":  # halfway bounce-back; the lid moves along x at the top in z
                if a:
                    at = 0 if a > 0 else nx - 1
                    new[:, :, at] = back[:, :, at]
                if b:
                    at = 0 if b > 0 else ny - 1
                    new[:, at] = back[:, at]
                if c > 0:
                    new[0] = back[0]
                if c < 0:
                    new[-1] = back[-1] + 6 * WEIGHT[q] * a * self.lid
            elif self.flow == "channel":  # inflow equilibrium, zero-gradient outflow, y and z periodic
                if a > 0:
                    new[:, :, 0] = self.fin[q]
                if a < 0:
                    new[:, :, -1] = torch.roll(old[q][:, :, -1], (c, b), (0, 1))
                new[self.bounce[q]] = back[self.bounce[q]]
            self.f.append(new)

    def _ghosts(self):
        """The reference's own boundary order on the first ghost layer."""
        f, lens = self.f, self.f[0].shape
        lo, hi = G, [G + v for v in self.n]

        def wall(axis, plane, source, sign, step=(2, 2, 2)):
            for q, d in enumerate(DIRS):
                if d[axis] != sign:
                    continue
                dst, src = [None] * 3, [None] * 3  # z, y, x
                for o in range(3):
                    end = lens[2 - o] - G + 1
                    if o == axis:
                        dst[2 - o], src[2 - o] = plane, source
                    else:
                        dst[2 - o] = slice(G - 1, end)
                        src[2 - o] = slice(G - 1 + step[o] * d[o], end + step[o] * d[o])
                f[q][tuple(dst)] = f[OPP[q]][tuple(src)]

        if self.flow == "cavity faithful":
            for t in f:  # what the reference's halo brings with one rank
                t[:, hi[1]] = 0
                t[hi[2]] = 0
                t[:, :, lo - 1] = 0
                t[:, :, hi[0]] = 0
            wall(0, lo - 1, lo + 1, 1)
            wall(0, hi[0], hi[0] - 2, -1)
        wall(1, lo - 1, lo + 1, 1)
        wall(1, hi[1], hi[1] - 2, -1)
        wall(2, lo - 1, lo + 1, 1)
        wall(2, hi[2], hi[2] - 2, -1, (2, 1, 2) if self.flow == "cavity faithful" else (2, 2, 2))
        if self.flow == "sphere faithful":
            rz, ry = slice(G - 1, lens[0] - G + 1), slice(G - 1, lens[1] - G + 1)
            for q, (a, b, c) in enumerate(DIRS):
                if a > 0:
                    f[q][rz, ry, G - 1] = f[q][rz, ry, G]
                if a < 0:
                    f[q][rz, ry, hi[0]] = f[q][G - 1 + c:lens[0] - G + 1 + c, G - 1 + b:lens[1] - G + 1 + b, hi[0] - 1]
            for q, (a, b, c) in enumerate(DIRS):
                z, y, x = self.bounce[q]
                f[q][z, y, x] = f[OPP[q]][z + 2 * c, y + 2 * b, x + 2 * a]

    def _stream_ghosts(self):
        nx, ny, nz = self.n
        for q, (a, b, c) in enumerate(DIRS):
            self._inside(self.f[q]).copy_(self.f[q][G - c:G - c + nz, G - b:G - b + ny, G - a:G - a + nx].clone())

    def _update(self):
        f, m = [self._inside(t) for t in self.f], self._inside(self.m)
        for s in self._slabs(m.shape[1:]):
            m[:, s] = (self.M @ torch.stack([t[s] for t in f]).view(27, -1)).view(m[:, s].shape)
        if self.solid is not None:
            m.masked_fill_(self._inside(self.solid), 0.0)
        if self.flow == "cavity faithful":
            m[1, -1] = 0.1
        if self.flow == "sphere faithful":
            m[1, :, :, 0] = self.profile[G:-G, :, 0]
            m[2:, :, :, 0] = 0
            m[0, :, :, -1] = 0

    def fields(self):
        return [t.contiguous() for t in self._inside(self.m)]

    def energy_and_mass(self):
        return torch.stack([0.5 * self.m[1:].square().sum(), 3 * self.m[0].sum()])

    def force(self):
        """Twice the momentum of the populations that leave for the ball."""
        self.collide()
        out = torch.zeros(3, dtype=torch.float64, device=self.dev)
        for q, d in enumerate(DIRS):
            leaving = 2 * self.f[OPP[q]][self.bounce[q]].sum()
            out -= leaving * torch.tensor(d, dtype=torch.float64, device=self.dev)
        return out


def _hash(x):
    """The finaliser of splitmix64, on 64-bit whole numbers."""
    x = x ^ (x >> np.uint64(30))
    x = x * np.uint64(0xBF58476D1CE4E5B9)
    x = x ^ (x >> np.uint64(27))
    x = x * np.uint64(0x94D049BB133111EB)
    return x ^ (x >> np.uint64(31))


def exact(case, seed):
    k = _physics(case, seed)
    if case["flow"] == "ensemble":
        fields = []
        for d in k["domains"]:
            e = _Exact("cavity" if d["case_id"] else "tgv", (d["nx"], d["ny"], d["nz"]), d["tau0"], d["u0"], d["lid_u"])
            for _ in range(case["steps"]):
                e.step()
            fields.append(e.fields())
        return {"finite": None, "fields": fields}
    n = (case["nx"], case["ny"], case["nz"])
    if n[0] * n[1] * n[2] * case["steps"] > 2.2e10:  # 20 seconds and more
        return None
    e = _Exact(case["flow"], n, k["tau"], k["u0"], k["lid_u"], k["seed"], _ball(case) if case["flow"] == "channel" else None)
    for _ in range(case["steps"]):
        e.step()
    out = dict(zip(NAMES, e.fields()))
    if case["flow"] == "tgv":
        out["energy and mass"] = e.energy_and_mass()
    if case["flow"] == "channel":
        out["force"] = e.force()
    return out
