"""The work that users of this framework have it do, as measurable cases.

A case is a dict of plain values:

  use      "frame": one world, one step per call, then every body read back: a
           game or render loop (with "contacts": the manifolds too, as a
           contact-event or debug-overlay loop reads them);
           "batch": many worlds stepped together, "steps" steps per call, then
           every body of every world read back: environment rollouts;
           "serve": "worlds" new scenes of 16 to "n" bodies built, submitted to
           a running server for "steps" steps each, drained, read back, freed.
  scene    "pyramid" (n = rows of unit boxes), "pile" (discs and rectangles
           dropped on a ground), "world" (a pile with distance joints and
           springs), "constrained" (walls, ropes, motors and loose bodies).
  n, worlds, n_min   bodies per world: n, or U{n_min..n} when n_min > 0
  settle   untimed steps before the first pass (-1: until a dropped pile lies)
  order    "reference" or "coloured" solver order
  hash     "reference" (cell 4 m) or "tuned" (twice the largest extent)
  warm     warm-starting factor, 0 = off

Materials and sizes are those of resolve2d_amd.scenes; every step is
dt = 1/60 with 4 sub-steps and 4 iterations, as the demos call it.
"""
import ctypes
import math

import numpy as np

from resolve2d_amd import _native as N
from resolve2d_amd.engine import GpuWorld
from resolve2d_amd.scenes import DT, ITERS, SUB_STEPS
from resolve2d_amd.serve import Server
from resolve2d_amd.solver import Context

G = float(np.float32(9.81))
INF = float("inf")


def _case(name, use, scene, n, worlds=1, steps=1, settle=0, n_min=0, order="reference", hash="reference", warm=0.0,
          contacts=False):
    c = dict(use=use, scene=scene, n=n, worlds=worlds, steps=steps, settle=settle, n_min=n_min, order=order, hash=hash,
             warm=warm, contacts=contacts)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # a toy scene stepped every frame: launches and round trips are all there is
        _case("frame_pyramid_3_rows", "frame", "pyramid", 3),
        # a small scene whose contacts the caller reads every frame (impact sounds, debug overlay)
        _case("frame_contacts_10_rows", "frame", "pyramid", 10, contacts=True),
        # the 20-row pyramid: one ordinary stacked scene, bound by its chain of dependent contacts
        _case("frame_pyramid_20_rows", "frame", "pyramid", 20),
        # one level of a game: a few hundred bodies with joints and springs
        _case("frame_world_387", "frame", "world", 387),
        # a large single world in the reference's order
        _case("frame_pile_4096", "frame", "pile", 4096, settle=-1),
        # the same world with the caller's choice of the coloured order and the tuned spatial hash
        _case("frame_pile_4096_coloured", "frame", "pile", 4096, settle=-1, order="coloured", hash="tuned"),
        # ropes, motors and 65,536 bodies between walls: the largest world
        _case("frame_constrained_65536", "frame", "constrained", 65536, settle=60),
        # 1,024 ragged worlds: rollouts at the size the throughput is quoted on
        _case("batch_1024", "batch", "world", 500, worlds=1024, steps=60, settle=220, n_min=50),
        # a batch that does not fill the chip, an odd number of worlds
        _case("batch_97", "batch", "world", 500, worlds=97, steps=8, settle=220, n_min=50),
        # warm-started rollouts
        _case("batch_warm_256", "batch", "world", 500, worlds=256, steps=16, settle=220, n_min=50, warm=0.8),
        # worlds too large for one workgroup's whole step, stepped together
        _case("batch_piles_24", "batch", "pile", 3000, worlds=24, steps=8, settle=-1, n_min=1200),
        # a burst of served scenes of very different sizes, from building to reading the results
        _case("serve_40", "serve", "pile", 8192, worlds=40, steps=48, n_min=16),
    ]


def draw(rng):
    def log(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    kind = rng.choice(["pyramid", "world", "pile", "pile", "constrained", "batch", "batch", "warm", "piles", "serve"])
    if kind == "pyramid":
        return _case(None, "frame", "pyramid", rng.randint(2, 24), contacts=rng.random() < 0.3)
    if kind == "world":
        return _case(None, "frame", "world", log(16, 1000), warm=rng.choice([0.0, 0.0, 0.8]))
    if kind == "pile":
        coloured = rng.random() < 0.3
        return _case(None, "frame", "pile", log(24, 6000), settle=-1, order="coloured" if coloured else "reference",
                     hash=rng.choice(["reference", "tuned"]))
    if kind == "constrained":
        return _case(None, "frame", "constrained", log(6000, 65536), settle=60)
    if kind == "piles":
        return _case(None, "batch", "pile", log(1100, 3000), worlds=rng.randint(2, 24), steps=rng.randint(1, 8),
                     settle=-1, n_min=200)
    if kind == "serve":
        return _case(None, "serve", "pile", log(400, 8192), worlds=rng.randint(6, 40), steps=rng.randint(8, 48), n_min=16)
    return _case(None, "batch", "world", rng.randint(60, 700), worlds=log(3, 700), steps=rng.randint(1, 40), settle=220,
                 n_min=rng.randint(8, 50), warm=0.8 if kind == "warm" else 0.0)


# ------------------------------------------------------------------- scenes
def _bodies(kind, x, y, a, b, angle=None, mu=0.4, static=None):
    """A scene's bodies as arrays: kind 0 disc (radius a), 1 rectangle (a x b); density 1."""
    n = len(kind)
    f = lambda v: np.broadcast_to(np.asarray(v, np.float32), (n,)).copy()
    return dict(kind=np.asarray(kind, np.int32), x=f(x), y=f(y), a=f(a), b=f(b), angle=f(0.0 if angle is None else angle),
                mu=f(mu), static=np.zeros(n, bool) if static is None else static, joints=[], motors=[], springs=[])


def _mixed(rng, n):
    """Discs and rectangles in turn: r U[0.2, 0.6]; sides U[0.3, 1], any angle."""
    kind = np.arange(n) % 2
    a = np.where(kind == 0, rng.uniform(0.2, 0.6, n), rng.uniform(0.3, 1.0, n))
    return kind, a, np.where(kind == 0, 0.0, rng.uniform(0.3, 1.0, n)), np.where(kind == 0, 0.0, rng.uniform(0, 2 * math.pi, n))


def _on_ground(kind, x, y, a, b, angle, mu, ground):
    """The bodies with a static ground of that width in front (id 0)."""
    cat = lambda h, t: np.concatenate([[h], t])
    s = _bodies(cat(1, kind), cat(0.0, x), cat(-0.5, y), cat(ground, a), cat(1.0, b), cat(0.0, angle), mu)
    s["static"][0] = True
    return s


def _scene(case, rng, n):
    kind = case["scene"]
    if kind == "pyramid":
        rows = n
        x = np.concatenate([np.arange(rows - r) - (rows - 1 - r) / 2.0 for r in range(rows)])
        y = np.concatenate([np.full(rows - r, 0.5 + r) for r in range(rows)])
        m = len(x)
        # stacked by hand: each box a little off its place
        return _on_ground(np.ones(m), x + rng.uniform(-0.02, 0.02, m), y, np.full(m, 1.0), np.full(m, 1.0), np.zeros(m), 0.5,
                          100.0)
    if kind == "constrained":
        size = 600.0 * math.sqrt(n / 65536.0)
        ropes, links, motors = max(1, n * 100 // 65536), 20, max(1, n * 64 // 65536)
        inner, t = size / 2 - 5.0, 10.0
        wall = [(0.0, -t / 2, size + 2 * t, t), (0.0, size + t / 2, size + 2 * t, t), (-size / 2 - t / 2, size / 2, t, size),
                (size / 2 + t / 2, size / 2, t, size)]
        rx = np.repeat(rng.uniform(-inner, inner - 0.8 * links, ropes), links + 1) + 0.8 * np.tile(np.arange(links + 1), ropes)
        ry = np.repeat(rng.uniform(5.0, size - 5.0, ropes), links + 1)
        rest = n - len(rx) - motors
        k, a, b, angle = _mixed(rng, rest)
        cat = np.concatenate
        s = _bodies(cat([np.ones(4), np.zeros(len(rx) + motors), k]),
                    cat([[w[0] for w in wall], rx, rng.uniform(-inner, inner, motors + rest)]),
                    cat([[w[1] for w in wall], ry, rng.uniform(5.0, size - 5.0, motors + rest)]),
                    cat([[w[2] for w in wall], np.full(len(rx), 0.2), np.ones(motors), a]),
                    cat([[w[3] for w in wall], np.zeros(len(rx) + motors), b]),
                    cat([np.zeros(4 + len(rx) + motors), angle]))
        s["static"][:4] = True
        for r in range(ropes):
            i = 4 + r * (links + 1)
            s["joints"] += [(i + j, i + j + 1, float(s["x"][i + j + 1] - s["x"][i + j])) for j in range(links)]
        s["motors"] = [(4 + len(rx) + j, float(np.float32(rng.uniform(-5.0, 5.0)))) for j in range(motors)]
        return s
    k, a, b, angle = _mixed(rng, n)
    width = 40.0 if kind == "world" else max(8.0, 100.0 * math.sqrt(n / 4096.0))
    height = max(10.0, n * 0.12) if kind == "world" else 2.0 * width
    s = _on_ground(k, rng.uniform(-width / 2, width / 2, n), rng.uniform(1.0, 1.0 + height, n), a, b, angle, 0.4, width + 20.0)
    if kind == "world":
        for _ in range(rng.integers(0, 21) if n > 1 else 0):
            i, j = (int(v) + 1 for v in rng.choice(n, 2, replace=False))
            d = math.hypot(float(s["x"][j]) - float(s["x"][i]), float(s["y"][j]) - float(s["y"][i]))
            s["joints"].append((i, j, float(np.float32(d))))
        for _ in range(rng.integers(0, 11)):
            i = int(rng.integers(0, n)) + 1
            s["springs"].append((i, float(np.float32(rng.uniform(10.0, 100.0))), float(np.float32(0.1)), float(s["x"][i]),
                                 float(s["y"][i])))
    return s


def _scenes(case, seed):
    # a case has the same ragged sizes whatever the seed; the bodies come from the seed
    lo, size_rng, rng = case["n_min"], np.random.default_rng([case["worlds"], case["n"]]), np.random.default_rng(seed)
    if case["use"] == "serve":   # log-uniform sizes, the largest always among them
        sizes = np.exp(size_rng.uniform(math.log(lo), math.log(case["n"]), case["worlds"])).round().astype(int)
        sizes[case["worlds"] // 2] = case["n"]
    else:
        sizes = size_rng.integers(lo, case["n"] + 1, case["worlds"]) if lo else [case["n"]] * case["worlds"]
    return [_scene(case, rng, int(n)) for n in sizes]


def _build(ctx, case, s):
    """A new world holding the scene, through the bulk and joint constructors."""
    w = GpuWorld(ctx)
    w.make_gravity(G)
    z = np.zeros(len(s["kind"]), np.float32)
    w.make_bodies(s["kind"], s["x"], s["y"], z, z, s["angle"], z, s["mu"], np.zeros(len(z), np.int32), z + 1, s["a"], s["b"])
    for i in np.flatnonzero(s["static"]):
        w.set_static(int(i), True)
    for i, j, d in s["joints"]:
        w.make_joint(0, INF, -INF, 10.0, i, j, 0.0, 0.0, 0.0, 0.0, d, 0.0, 0.0)
    for i, omega in s["motors"]:
        w.make_joint(3, 50.0, -50.0, 10.0, i, 0, 0.0, 0.0, 0.0, 0.0, omega, 0.0, 0.0)
    for i, k, c, ax, ay in s["springs"]:
        w.make_spring(i, k, c, ax, ay)
    if case["hash"] == "tuned":
        loose = ~s["static"]
        rect = s["kind"][loose] == 1
        a, b, t = s["a"][loose], s["b"][loose], s["angle"][loose]
        c, sn = np.abs(np.cos(t)), np.abs(np.sin(t))
        w.set_hash(float(np.float32(2.0 * np.where(rect, np.maximum(a * c + b * sn, a * sn + b * c), 2 * a).max())), 2)
    if case["order"] == "coloured":
        w.set_schedule(1)
    if case["warm"]:
        w.set_warm_start(case["warm"])
    return w


# -------------------------------------------------------------- measured path
WORDS = ctypes.sizeof(N.BodyState) // 4
HEAD = 4   # id, type, static flag, normals: whole numbers; then floats
# two ids, normal, tangent, friction; for each of two points a flag and 12 floats
CONTACT_WORDS = ctypes.sizeof(N.ManifoldState) // 4


def _contact_rows(n):
    return 4 * n + 16


class State:
    """What a program keeps between calls: a context, its worlds (or a server
    and the scenes it is about to submit) and the buffer states are read into."""

    def __init__(self, case, seed):
        self.case = case
        self.ctx = Context(0)
        self.scenes = _scenes(case, seed)
        self.worlds, self.server = [], None
        sizes = [len(s["kind"]) for s in self.scenes]
        self.raw = np.zeros((sum(sizes), WORDS), np.uint32)
        at = np.concatenate([[0], np.cumsum(sizes)])
        body = ctypes.POINTER(N.BodyState)
        self.rows = [(ctypes.cast(self.raw.ctypes.data + int(o) * WORDS * 4, body), n) for o, n in zip(at, sizes)]
        self.count = ctypes.c_size_t()
        # room for the contacts of a stack (under 3 a body)
        self.contacts = np.zeros((_contact_rows(sizes[0]) if case["contacts"] else 0, CONTACT_WORDS), np.uint32)
        if case["use"] == "serve":
            self.server = Server(self.ctx, 64 << 30, 4096, DT, SUB_STEPS, ITERS, steps_per_tick=8)
            return
        self.worlds = [_build(self.ctx, case, s) for s in self.scenes]
        self.batch = self.ctx.prepare_batch([w.handle for w in self.worlds])
        settle = case["settle"]
        if settle < 0:   # the fall from the top of the box, and a second at rest
            top = max(float(s["y"].max()) for s in self.scenes)
            settle = int(60 * math.sqrt(2 * top / G)) + 60
        if settle:
            self.batch.process(DT, SUB_STEPS, ITERS, settle)

    def read(self):
        for w, (rows, n) in zip(self.worlds, self.rows):
            N.check(w.lib.r2d_get_bodies(w.handle, rows, n, ctypes.byref(self.count)), "r2d_get_bodies")
        return {"head": self.raw[:, :HEAD], "state": self.raw.view(np.float32)[:, HEAD:]}

    def read_contacts(self):
        w, rows = self.worlds[0], self.contacts.ctypes.data_as(ctypes.POINTER(N.ManifoldState))
        N.check(w.lib.r2d_get_manifolds(w.handle, rows, len(self.contacts), ctypes.byref(self.count)), "r2d_get_manifolds")
        self.contacts[self.count.value:] = 0
        real = self.contacts.view(np.float32)
        return {"contact_ids": self.contacts[:, :2], "contacts": real[:, 2:7],
                "points": [real[:, 8:20], real[:, 21:33]], "points_valid": [self.contacts[:, 7], self.contacts[:, 20]]}

    def __del__(self):
        try:
            self.ctx.close()
        except Exception:
            pass   # a context that never opened


def prepare(case, seed):
    return State(case, seed)


def run(state):
    case = state.case
    if case["use"] == "serve":
        state.worlds = [_build(state.ctx, case, s) for s in state.scenes]
        for w in state.worlds:
            state.server.submit(w, case["steps"])
        state.server.drain()
        state.server.completed()
        out = state.read()
        for w in state.worlds:
            w.close()
        return out
    if case["use"] == "frame":
        w = state.worlds[0]
        N.check(w.process(DT, SUB_STEPS, ITERS), "r2d_process")
    else:
        state.batch.process(DT, SUB_STEPS, ITERS, case["steps"])
    out = state.read()
    if case["contacts"]:
        out.update(state.read_contacts())
    return out


# manifolds per body of a scene at rest (falling bodies of "constrained": few)
_CONTACTS = {"pyramid": 2.3, "pile": 1.5, "world": 1.6, "constrained": 0.1}


def work(case):
    rows = case["n"]
    n = rows * (rows + 1) / 2 + 1 if case["scene"] == "pyramid" else rows
    if case["n_min"]:
        n = ((rows - case["n_min"]) / math.log(rows / case["n_min"]) if case["use"] == "serve" else
             (rows + case["n_min"]) / 2)
    bodies, steps = n * case["worlds"], case["steps"]
    # per pass: the state (21 words a body) read, what moves (13 words) written, the states read back;
    # per step: 2 points of about 60 operations for each manifold in each iteration, 200 a body
    contacts = _CONTACTS[case["scene"]] * bodies
    return {"bytes": bodies * 4 * (21 + 13 + WORDS),
            "flops": steps * (SUB_STEPS * ITERS * contacts * 120 + bodies * 200)}


# ------------------------------------------------------------ the step in 64 bits
def exact(case, seed):
    """The first pass of a fresh pyramid or jointed world, from its equations
    in Python's 64-bit numbers; None where a pass starts after many steps
    (contact dynamics multiply any rounding) or would take too long."""
    if case["use"] != "frame" or case["settle"] or case["warm"] or case["order"] != "reference":
        return None
    s = _scenes(case, seed)[0]
    if len(s["kind"]) > 2000:
        return None
    out = _Step64(s).process()
    return out if case["contacts"] else {"head": None, "state": out["state"]}


def _norm(x, y):
    d = math.sqrt(x * x + y * y)
    return (0.0, 0.0) if d < 1e-3 else (x / d, y / d)


class _Step64:
    def __init__(self, s):
        v = lambda k: [float(t) for t in s[k]]
        self.n = len(s["kind"])
        self.rect = [bool(k) for k in s["kind"]]
        self.static = [bool(t) for t in s["static"]]
        self.x, self.y, self.th, self.a, self.b, self.mu = v("x"), v("y"), v("angle"), v("a"), v("b"), v("mu")
        self.m = [a * b if r else math.pi * a * a for a, b, r in zip(self.a, self.b, self.rect)]
        self.I = [m * (a * a + b * b) / 12 if r else 0.5 * m * a * a for m, a, b, r in zip(self.m, self.a, self.b, self.rect)]
        self.px, self.py, self.L = [0.0] * self.n, [0.0] * self.n, [0.0] * self.n
        self.joints, self.springs = s["joints"], s["springs"]
        self.box = [self.extent(i) for i in range(self.n)]

    def verts(self, i, centre=True):
        c, s, hw, hh = math.cos(self.th[i]), math.sin(self.th[i]), self.a[i] / 2, self.b[i] / 2
        ox, oy = (self.x[i], self.y[i]) if centre else (0.0, 0.0)
        return [(x * c - y * s + ox, x * s + y * c + oy) for x, y in ((-hw, -hh), (-hw, hh), (hw, hh), (hw, -hh))]

    def extent(self, i):
        if not self.rect[i]:
            return (self.x[i], self.y[i], self.a[i], self.a[i])
        p = self.verts(i, False)
        return (self.x[i], self.y[i], max(q[0] for q in p), max(q[1] for q in p))

    def pairs(self):
        """Candidate pairs in the order a 4 m spatial hash of 2 n buckets finds them."""
        buckets, cells = {}, []
        for i, (x, y, w, h) in enumerate(self.box):
            mine = []
            for cy in range(math.floor((y - h) / 4), math.floor((y + h) / 4) + 1):
                for cx in range(math.floor((x - w) / 4), math.floor((x + w) / 4) + 1):
                    k = (((cx * 92837111) ^ (cy * 689287499)) & (2 ** 64 - 1)) % (2 * self.n)
                    mine.append(k)
                    buckets.setdefault(k, set()).add(i)
            cells.append(mine)
        for i in range(self.n):
            seen = set()
            for k in cells[i]:
                for j in sorted(buckets[k], reverse=True):
                    if j <= i or j in seen:
                        continue
                    seen.add(j)
                    (xa, ya, wa, ha), (xb, yb, wb, hb) = self.box[i], self.box[j]
                    if not (self.static[i] and self.static[j]) and abs(xb - xa) <= wa + wb + 0.01 and abs(yb - ya) <= ha + hb + 0.01:
                        yield i, j

    def closest(self, i, p):
        if not self.rect[i]:
            d = _norm(p[0] - self.x[i], p[1] - self.y[i])
            return (self.x[i] + d[0] * self.a[i], self.y[i] + d[1] * self.a[i])
        return min(self.verts(i), key=lambda q: (q[0] - p[0]) ** 2 + (q[1] - p[1]) ** 2)

    def normal(self, i, other, k):
        if not self.rect[i]:
            c = self.closest(other, (self.x[i], self.y[i]))
            return _norm(c[0] - self.x[i], c[1] - self.y[i]), None, None
        v = self.verts(i)
        p, q = v[k], v[(k + 1) % 4]
        d = _norm(q[0] - p[0], q[1] - p[1])
        return (-d[1], d[0]), p, q

    def span(self, i, n):
        if not self.rect[i]:
            c = self.x[i] * n[0] + self.y[i] * n[1]
            return c - self.a[i], c + self.a[i]
        d = [p[0] * n[0] + p[1] * n[1] for p in self.verts(i)]
        return min(d), max(d)

    def sat(self, first, second):
        """The reference body, its face and the normal of the least overlap; None when apart."""
        pen, best = INF, None
        near = lambda p, q: abs(p[0] - q[0]) < 1e-4 and abs(p[1] - q[1]) < 1e-4
        for ref, inc in ((first, second), (second, first)):
            dx, dy = self.x[inc] - self.x[ref], self.y[inc] - self.y[ref]
            for k in range(4 if self.rect[ref] else 1):
                n = self.normal(ref, inc, k)[0]
                flip = n[0] * dx + n[1] * dy < 0
                n = (-n[0], -n[1]) if flip else n
                (lo1, hi1), (lo2, hi2) = self.span(ref, n), self.span(inc, n)
                d = min(hi1 - lo2, hi2 - lo1)
                if d <= -0.01:
                    return None
                take = d + 1e-4 < pen
                if best and not flip and near(n, best[3]):
                    take = take or self.x[ref] * n[0] + self.y[ref] * n[1] < self.x[inc] * n[0] + self.y[inc] * n[1] - 1e-4
                if best and not flip and near(n, (-best[3][0], -best[3][1])):
                    take = take or dx * n[0] + dy * n[1] > dx * best[3][0] + dy * best[3][1] + 1e-4
                if take:
                    pen, best = d, (ref, inc, k, n)
        return best

    def points(self, ref, inc, k):
        """Contact points (on the incident body) and depths along the face normal."""
        if not self.rect[ref]:
            p = self.closest(inc, (self.x[ref], self.y[ref]))
            n = self.normal(ref, inc, k)[0]
            if n[0] * (self.x[inc] - self.x[ref]) + n[1] * (self.y[inc] - self.y[ref]) < 0:
                n = (-n[0], -n[1])
            return [(p, n[0] * (p[0] - self.x[ref]) + n[1] * (p[1] - self.y[ref]) - self.a[ref])], n
        n, ea, eb = self.normal(ref, inc, k)
        if not self.rect[inc]:
            p = (self.x[inc] - n[0] * self.a[inc], self.y[inc] - n[1] * self.a[inc])
            return [(p, (p[0] - ea[0]) * n[0] + (p[1] - ea[1]) * n[1])], n
        v = self.verts(inc)
        along = []
        for i in range(4):
            d = _norm(v[(i + 1) % 4][0] - v[i][0], v[(i + 1) % 4][1] - v[i][1])
            along.append(n[0] * -d[1] + n[1] * d[0])
        i = min(range(4), key=lambda j: along[j])
        ia, ib = v[i], v[(i + 1) % 4]
        size = math.hypot(eb[0] - ea[0], eb[1] - ea[1])
        t = ((eb[0] - ea[0]) / size, (eb[1] - ea[1]) / size)

        def clip(p, q):
            at = (p[0] - ea[0]) * t[0] + (p[1] - ea[1]) * t[1]
            if 0 < at < size:
                return p
            e = ea if at < 0.5 * size else eb
            d = (p[0] - q[0], p[1] - q[1])
            u = -(t[0] * (q[0] - e[0]) + t[1] * (q[1] - e[1])) / (t[0] * d[0] + t[1] * d[1])
            return (q[0] + d[0] * u, q[1] + d[1] * u)

        got = []
        for p, e in ((clip(ia, ib), ea), (clip(ib, ia), eb)):
            d = (p[0] - e[0]) * n[0] + (p[1] - e[1]) * n[1]
            if d < 0.01:
                got.append((p, d))
        return got, n

    def process(self):
        n, h = self.n, float(np.float32(DT)) / SUB_STEPS
        im = [0.0 if s else 1 / m for s, m in zip(self.static, self.m)]
        ii = [0.0 if s else 1 / i for s, i in zip(self.static, self.I)]
        mans = []
        for i, j in self.pairs():
            hit = self.sat(i, j)
            if not hit:
                continue
            ref, inc, k, nrm = hit
            pts = []
            got, along = self.points(ref, inc, k)
            for p, d in got:
                mid = (p[0] - along[0] * d / 2, p[1] - along[1] * d / 2)
                pts.append(dict(r1=(mid[0] - self.x[ref], mid[1] - self.y[ref]), r2=(mid[0] - self.x[inc], mid[1] - self.y[inc]),
                                pos=mid, depth=d, pn=0.0, pt=0.0))
            t = (nrm[1], -nrm[0])
            for q in pts:
                for name, ax in (("mn", nrm), ("mt", t)):
                    c1, c2 = q["r1"][0] * ax[1] - q["r1"][1] * ax[0], q["r2"][0] * ax[1] - q["r2"][1] * ax[0]
                    kk = im[ref] + im[inc] + ii[ref] * c1 * c1 + ii[inc] * c2 * c2
                    q[name] = 1 / kk if kk > 0 else 0.0
            mans.append((ref, inc, nrm, t, math.sqrt(self.mu[ref] * self.mu[inc]), pts))
        X, Y, P, Q, L = self.x, self.y, self.px, self.py, self.L
        for step in range(SUB_STEPS):
            force = [(0.0, 0.0 if s else -G * m) for s, m in zip(self.static, self.m)]
            for i, k, c, ax, ay in self.springs:
                fx, fy = force[i]
                force[i] = (fx - k * (X[i] - ax) - c * P[i] / self.m[i], fy - k * (Y[i] - ay) - c * Q[i] / self.m[i])
            self.box = [self.extent(i) for i in range(n)]
            for i in range(n):
                P[i] += force[i][0] * h
                Q[i] += force[i][1] * h
            for _ in range(ITERS):
                for i, j, want in self.joints:
                    rx, ry = P[j] * im[j] - P[i] * im[i], Q[j] * im[j] - Q[i] * im[i]
                    d = (X[j] - X[i], Y[j] - Y[i])
                    u = _norm(*d)
                    err = math.hypot(*d) - want
                    s = -(rx * u[0] + ry * u[1] + 10.0 * err / max(want, 0.001)) / (im[i] + im[j])
                    P[i] -= u[0] * s; Q[i] -= u[1] * s; P[j] += u[0] * s; Q[j] += u[1] * s
                for ref, inc, nrm, t, mu, pts in mans:
                    va, vb = (P[ref] * im[ref], Q[ref] * im[ref]), (P[inc] * im[inc], Q[inc] * im[inc])
                    wa, wb = L[ref] * ii[ref], L[inc] * ii[inc]
                    for q in pts:
                        if q["depth"] >= 0:
                            q["pn"] = q["pt"] = 0.0
                            continue
                        (ax, ay), (bx, by) = q["r1"], q["r2"]
                        dx, dy = va[0] - ay * wa - (vb[0] - by * wb), va[1] + ax * wa - (vb[1] + bx * wb)
                        pn = (dx * nrm[0] + dy * nrm[1] + 0.02 * max(0.0, -q["depth"] - 0.005) / h) * q["mn"]
                        if pn < 1e-4:
                            continue
                        new = max(0.0, q["pn"] + pn)
                        dn, q["pn"] = new - q["pn"], new
                        tangent = min(max(q["pt"] + (dx * t[0] + dy * t[1]) * q["mt"], -mu * abs(new)), mu * abs(new))
                        dt_, q["pt"] = tangent - q["pt"], tangent
                        jx, jy = nrm[0] * dn + t[0] * dt_, nrm[1] * dn + t[1] * dt_
                        if not self.static[ref]:
                            P[ref] -= jx; Q[ref] -= jy; L[ref] -= ax * jy - ay * jx
                        if not self.static[inc]:
                            P[inc] += jx; Q[inc] += jy; L[inc] += bx * jy - by * jx
            for i in range(n):
                if not self.static[i]:
                    X[i] += P[i] * h / self.m[i]
                    Y[i] += Q[i] * h / self.m[i]
                    self.th[i] += L[i] * h / self.I[i]
        z = [0.0] * n
        disc = [0.0 if r else a for a, r in zip(self.a, self.rect)]
        wide = [a if r else 0.0 for a, r in zip(self.a, self.rect)]
        high = [b if r else 0.0 for b, r in zip(self.b, self.rect)]
        box = [[e[k] for e in self.box] for k in range(4)]
        state = np.array([X, Y, P, Q, z, z, self.m, self.th, L, z, self.I, self.mu] + box + [disc, wide, high]).T
        flat, points = np.zeros((_contact_rows(n), 5)), [np.zeros((_contact_rows(n), 12)) for _ in range(2)]
        for row, (ref, inc, nrm, t, mu, pts) in enumerate(mans):
            flat[row] = [*nrm, *t, mu]
            for q, to in zip(pts, points):
                to[row] = [q["pn"], q["pt"], *q["r1"], *q["r2"], *q["pos"], q["depth"], q["depth"], q["mn"], q["mt"]]
        return {"head": None, "state": state, "contact_ids": None, "contacts": flat, "points": points, "points_valid": None}
