"""The workloads this library's speed is judged by, each through its public Python entry points.

listed() names one size of every kind of use; draw(rng) gives another size and other options of the same kinds.
prepare() makes what a simulation program has in hand before the call (particles on the device, or on the host for
the request loop, and the long-lived object it steps), run() is one call as such a program makes it, exact() the
same in 64 bits where the result is a computed number, work() what one pass must read, write and compute.

Keys, orders, trees, sorted copies of the inputs and neighbor rows are defined bit for bit, so they come back as whole
words; sums over neighbors and mass centers come back as floating-point numbers.
"""

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cornerstone-octree_amd"))

import hipcstone as hip  # noqa: E402

NEIGHBORS = 100  # mean neighbors the smoothing lengths are made for (64 for the batched clouds)
DRIFT = 1e-3  # displacement of a warm step in units of h


def listed():
    return [
        # one step of an interactive or many-small-systems program: latency and launches are all of it
        _step("step_f32_2k", 2000, ngmax=150),
        # an ordinary update of a resident cloud (the request loop's size), odd count
        _step("step_f32_150k", 150_003, ngmax=128),
        # the flagship: the 16.8 M-particle warm step, 64-bit Hilbert keys
        _step("step_f32_16m", 16_777_216, ngmax=150),
        # a first call: full build of 1 M uniform fp64 particles from unsorted input
        {"name": "build_f64_1m", "kind": "build", "n": 1_000_000, "key_bits": 64, "real_bits": 64, "bucket": 64,
         "ngmax": 150, "cloud": "uniform"},
        # an SPH step behind the one-rank Domain: sync and the search over its focus tree
        {"name": "domain_f32_4m", "kind": "domain", "n": 4_000_000, "real_bits": 32, "bucket": 64, "focus": 16,
         "ngmax": 150, "cloud": "plummer", "periodic": False},
        # the same in a periodic fp64 box (cosmology, turbulence boxes)
        {"name": "domain_f64_periodic_300k", "kind": "domain", "n": 300_001, "real_bits": 64, "bucket": 64,
         "focus": 64, "ngmax": 150, "cloud": "uniform", "periodic": True},
        # a gravity step: sync with masses and the focus tree's expansion centers
        {"name": "grav_f32_8m", "kind": "grav", "n": 8_388_608, "real_bits": 32, "bucket": 64, "focus": 16},
        # many independent clouds at once, two warm steps as one captured graph
        {"name": "batched_64_clouds", "kind": "batched", "clouds": 64, "nmin": 1000, "nmax": 1_000_000, "bucket": 128,
         "ngmax": 128},
        # a burst of requests (builds from host arrays, updates of resident clouds) through the request loop
        {"name": "served_burst", "kind": "served", "requests": 24, "nmin": 10_000, "nmax": 1_000_000, "slots": 4,
         "ngmax": 128},
        # one rank's share of a large run at its real size: build, assignment, halo discovery and gather
        {"name": "share_f64_134m", "kind": "share", "n": 134_217_728, "bucket": 128, "ranks": 8, "rank": 2},
        # an SPH-like sum over neighbors without stored rows
        {"name": "ijloop_f32_1m", "kind": "ijloop", "n": 1_000_000, "real_bits": 32, "bucket": 64, "ngmax": 200},
        # keys and the stable sort with its gather on their own, input in no order
        {"name": "sort_f32_u32_4m", "kind": "sort", "n": 4_000_037, "key_bits": 32, "real_bits": 32, "curve": 0},
    ]


def _step(name, n, **more):
    c = {"kind": "step", "n": n, "key_bits": 64, "real_bits": 32, "bucket": 64, "ngmax": 150, "cloud": "plummer"}
    return dict({"name": name} if name else {}, **dict(c, **more))


def _size(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))


def draw(rng):
    kind = rng.choice(["step", "step", "build", "build", "domain", "domain", "grav", "batched", "served", "share",
                       "ijloop", "sort"])
    if kind == "step":
        return _step(None, _size(rng, 1000, 16_000_000), key_bits=rng.choice([64, 64, 32]),
                     real_bits=rng.choice([32, 32, 64]), bucket=rng.choice([64, 64, 128, 32]),
                     ngmax=rng.choice([128, 150, 200]), cloud=rng.choice(["plummer", "uniform"]))
    if kind == "build":
        return {"kind": kind, "n": _size(rng, 1000, 8_000_000), "key_bits": rng.choice([64, 32]),
                "real_bits": rng.choice([32, 64]), "bucket": rng.choice([32, 64, 128]),
                "ngmax": rng.choice([128, 150, 200]), "cloud": rng.choice(["plummer", "uniform"])}
    if kind == "domain":
        periodic = rng.random() < 0.5
        return {"kind": kind, "n": _size(rng, 2000, 2_000_000 if periodic else 8_000_000),
                "real_bits": rng.choice([32, 64]), "bucket": 64, "focus": rng.choice([16, 32, 64]),
                "ngmax": rng.choice([128, 150]), "cloud": "uniform" if periodic else rng.choice(["plummer", "uniform"]),
                "periodic": periodic}
    if kind == "grav":
        return {"kind": kind, "n": _size(rng, 2000, 16_000_000), "real_bits": rng.choice([32, 64]), "bucket": 64,
                "focus": rng.choice([16, 32, 64])}
    if kind == "batched":
        return {"kind": kind, "clouds": rng.randrange(4, 129), "nmin": 1000, "nmax": _size(rng, 10_000, 800_000),
                "bucket": rng.choice([64, 128]), "ngmax": 128}
    if kind == "served":
        return {"kind": kind, "requests": rng.randrange(4, 33), "nmin": 10_000, "nmax": _size(rng, 20_000, 1_500_000),
                "slots": rng.choice([1, 4]), "ngmax": 128}
    if kind == "share":
        ranks = rng.choice([2, 4, 8])
        return {"kind": kind, "n": _size(rng, 100_000, 100_000_000), "bucket": rng.choice([64, 128]), "ranks": ranks,
                "rank": rng.randrange(ranks)}
    if kind == "ijloop":
        return {"kind": kind, "n": _size(rng, 5000, 4_000_000), "real_bits": rng.choice([32, 64]),
                "bucket": rng.choice([32, 64]), "ngmax": 200}
    return {"kind": kind, "n": _size(rng, 1000, 32_000_000), "key_bits": rng.choice([32, 64]),
            "real_bits": rng.choice([32, 64]), "curve": rng.choice([0, 1])}


# ---------------------------------------------------------------- device memory seen from torch


class _Memory:
    """A device range as torch takes it; whole words for everything that is compared bit for bit."""

    def __init__(self, ptr, count, typestr, owner=None):
        self.__cuda_array_interface__ = {"shape": (int(count),), "typestr": typestr, "data": (int(ptr), False),
                                         "version": 2}
        self.owner = owner


_WORDS = {1: "|u1", 4: "<i4", 8: "<i8"}


def _words(ptr, count, size, owner=None):
    return torch.as_tensor(_Memory(ptr, count, _WORDS[size], owner), device="cuda")


def _floats(ptr, count, size, owner=None):
    return torch.as_tensor(_Memory(ptr, count, "<f%d" % size, owner), device="cuda")


def _device(t):
    """A device array of the library with the values of the torch tensor t."""
    d = hip.DeviceArray(t.numel(), {torch.float32: np.float32, torch.float64: np.float64, torch.int32: np.uint32,
                                    torch.int64: np.uint64}[t.dtype])
    size = t.element_size()
    view = (_floats if t.is_floating_point() else _words)(d.ptr, d.count, size, d)
    view.copy_(t)
    torch.cuda.synchronize()
    return d


def _of(d):
    """The words of a library array."""
    return _words(d.ptr, d.count, d.dtype.itemsize, d)


def _zeros(n, dtype):
    d = hip.DeviceArray(n, dtype)
    _of(d).zero_()
    return d


class _Views:
    """torch views of the arrays a pipeline or a domain shows, made once per buffer as a program keeps them. A view
    keeps the objects that own the memory alive."""

    def __init__(self, *owners):
        self.made, self.owners = {}, owners

    def __call__(self, ptr, count, size):
        key = (ptr, count, size)
        if key not in self.made:
            if len(self.made) > 256:
                self.made.clear()
            self.made[key] = _words(ptr, count, size, self.owners)
        return self.made[key]


class _Kept:
    """A program's own copies of a tree's arrays, whose lengths change from step to step: each in a buffer with room
    to spare, zeros past what was ever written."""

    def __init__(self, room):
        self.room, self.kept = room, {}

    def __call__(self, name, view):
        if name not in self.kept:
            self.kept[name] = torch.zeros(self.room, dtype=view.dtype, device="cuda")
        self.kept[name][: view.numel()].copy_(view)
        return self.kept[name]


# ---------------------------------------------------------------- particles


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _uniform(n, g):
    return torch.rand(n, generator=g, device="cuda", dtype=torch.float64)


def _cloud(kind, n, g, target=NEIGHBORS, a=0.05):
    """x, y, z, h in float64, in no spatial order, h for about `target` neighbors within 2h; and the box limits."""
    if kind == "uniform":
        h = 0.5 * (target / (4.0 / 3.0 * math.pi * n)) ** (1.0 / 3.0)
        return [_uniform(n, g) for _ in range(3)] + [torch.full((n,), h, device="cuda", dtype=torch.float64)], (0.0, 1.0)
    # Plummer sphere of scale radius a inside r <= 1
    top = (1.0 + a * a) ** -1.5
    m = _uniform(n, g).clamp_(min=1e-12) * top
    r = a / torch.sqrt(m.pow(-2.0 / 3.0) - 1.0)
    cz = 2.0 * _uniform(n, g) - 1.0
    phi = 2.0 * math.pi * _uniform(n, g)
    s = torch.sqrt((1.0 - cz * cz).clamp_(min=0.0))
    rho = 3.0 * n / (4.0 * math.pi * a**3) * (1.0 + (r / a) ** 2) ** -2.5
    h = 0.5 * (target * 3.0 / (4.0 * math.pi * rho)) ** (1.0 / 3.0)
    return [(r * s * torch.cos(phi)).clamp_(-1, 1), (r * s * torch.sin(phi)).clamp_(-1, 1), (r * cz).clamp_(-1, 1),
            h], (-1.0, 1.0)


def _typed(arrays, real_bits):
    return [a.to(torch.float32 if real_bits == 32 else torch.float64) for a in arrays]


def _box(limits, real_bits, periodic=False):
    b = (hip.PERIODIC,) * 3 if periodic else (hip.OPEN,) * 3
    return hip.make_box(limits[0], limits[1], np.float32 if real_bits == 32 else np.float64, b)


# ---------------------------------------------------------------- one pass of each kind


def prepare(case, seed):
    return _KINDS[case["kind"]](case, seed)


def run(state):
    return state.run()


class _Pipe:
    """Warm steps of one pipeline: the particles are in the order of the step before and have moved a little, from one
    snapshot to the other and back; and full builds, whose input is in no order."""

    def __init__(self, c, seed):
        g = _generator(seed)
        n, rb = c["n"], c["real_bits"]
        raw, limits = _cloud(c["cloud"], n, g)
        self.n, self.box, self.full = n, _box(limits, rb), c["kind"] == "build"
        self.pipe = hip.Pipeline(curve=hip.HILBERT, key_bits=c["key_bits"], real_bits=rb, bucket_size=c["bucket"],
                                 ngmax=c["ngmax"])
        self.nb, self.nc = _zeros(n * c["ngmax"], np.uint32), _zeros(n, np.uint32)
        self.key, self.real, self.turn = c["key_bits"] // 8, rb // 8, 0
        self.views, self.kept = _Views(self.pipe, self.nb, self.nc), _Kept(4096 + 16 * (n // c["bucket"]))
        first = [_device(a) for a in _typed(raw, rb)]
        self.inputs = [first]
        if not self.full:
            self.pipe.sync(*first, n, self.box, full_build=True, neighbors=self.nb, counts=self.nc)
            v = self.pipe.view()
            cur = [_floats(p, n, self.real).clone() for p in (v.x, v.y, v.z, v.h)]
            moved = [(a + DRIFT * cur[3] * (2.0 * _uniform(n, g) - 1.0).to(a.dtype)).clamp_(*limits) for a in cur[:3]]
            self.inputs = [[_device(a) for a in cur], [_device(a) for a in moved + [cur[3]]]]

    def run(self):
        self.turn = (self.turn + 1) % len(self.inputs)
        self.pipe.sync(*self.inputs[self.turn], self.n, self.box, full_build=self.full, neighbors=self.nb,
                       counts=self.nc)
        v, w, n, k, r = self.pipe.view(), self.views, self.n, self.key, self.real
        return {"keys": w(v.keys, n, k), "perm": w(v.perm, n, 4),
                "particles": [w(p, n, r) for p in (v.x, v.y, v.z, v.h)],
                "num_leaves": v.num_leaves, "leaves": self.kept("leaves", w(v.leaves, v.num_leaves + 1, k)),
                "layout": self.kept("layout", w(v.layout, v.num_leaves + 1, 4)),
                "neighbors": w(self.nb.ptr, self.nb.count, 4), "neighbor_counts": w(self.nc.ptr, n, 4)}


class _Domain:
    """A step of a program that keeps its particles in the Domain's order: they move (the program's own update), are
    synchronized in place, and their neighbors are searched in the focus tree; or masses go along and the focus
    tree's expansion centers come out instead."""

    def __init__(self, c, seed):
        g = _generator(seed)
        n, rb = c["n"], c["real_bits"]
        self.grav = c["kind"] == "grav"
        raw, limits = _cloud(c.get("cloud", "plummer"), n, g)
        if self.grav:
            raw.append((0.5 + _uniform(n, g)) / n)
        self.n, self.real, self.step, self.seed = n, rb // 8, 0, int(seed)
        self.periodic = c.get("periodic", False)
        self.dtype = np.float32 if rb == 32 else np.float64
        self.box = _box(limits, rb, self.periodic)
        self.domain = hip.Domain(self.box, key_bits=64, bucket_size=c["bucket"], bucket_size_focus=c["focus"])
        self.arrays = [_device(a) for a in _typed(raw, rb)]
        self.ngmax = c.get("ngmax", 0)
        if self.grav:
            self.domain.sync_grav(*self.arrays, n)
        else:
            self.domain.sync(*self.arrays, n)
            self.nb, self.nc = _zeros(n * self.ngmax, np.uint32), _zeros(n, np.uint32)
        self.views = _Views(self.domain, self.arrays, None if self.grav else (self.nb, self.nc))
        self.kept = _Kept(16384 + 64 * (n // c["focus"]))

    def run(self):
        d, n, w = self.arrays, self.n, self.views
        hip.displace(d[0], d[1], d[2], d[3], n, DRIFT, self.seed, self.step, self.box)
        self.step += 1
        if self.grav:
            self.domain.sync_grav(*d, n)
        else:
            self.domain.sync(*d, n)
        v, r = self.domain.view(), self.real
        out = {"keys": w(v.keys, n, 8), "particles": [w(a.ptr, n, r) for a in d],
               "num_leaves": [v.num_global_leaves, v.num_leaves],
               "global_leaves": self.kept("global_leaves", w(v.global_leaves, v.num_global_leaves + 1, 8)),
               "leaves": self.kept("leaves", w(v.leaves, v.num_leaves + 1, 8)),
               "layout": self.kept("layout", w(v.layout, v.num_leaves + 1, 4))}
        if self.grav:
            centers = _floats(v.expansion_centers, 4 * v.num_nodes, r, self.domain)
            out["expansion_centers"] = self.kept("expansion_centers", centers)
            return out
        b = (hip.PERIODIC,) * 3 if self.periodic else (hip.OPEN,) * 3
        box = hip.make_box(v.box_lo[:], v.box_hi[:], self.dtype, b)
        hip.find_neighbors(d[0], d[1], d[2], d[3], 0, n, box, v.child_offsets, v.parents, v.internal_to_leaf, v.layout,
                           v.centers, v.sizes, v.num_nodes, self.ngmax, self.nb, self.nc)
        out.update(neighbors=w(self.nb.ptr, self.nb.count, 4), neighbor_counts=w(self.nc.ptr, n, 4))
        return out


def _mix(num, nmin, nmax, seed):
    """Sizes of `num` clouds, log-uniform in [nmin, nmax] (evenly spread, in an order of the seed's)."""
    order = np.random.RandomState(seed % (1 << 31)).permutation(num)
    u = (np.arange(num) + 0.5) / num
    return np.exp(math.log(nmin) + math.log(nmax / nmin) * u).astype(np.int64)[order]


class _Batched:
    """Two warm drift steps of many independent clouds as one replayed graph."""

    def __init__(self, c, seed):
        g = _generator(seed)
        sizes = _mix(c["clouds"], c["nmin"], c["nmax"], seed)
        clouds = [_cloud("uniform" if i % 2 else "plummer", int(m), g, target=64, a=0.1) for i, m in enumerate(sizes)]
        self.stream = hip.Stream()
        self.n, self.ngmax = int(sizes.sum()), c["ngmax"]
        self.batched = hip.Batched(sizes, [_box(lim, 32) for _, lim in clouds],
                                   np.full(len(sizes), c["bucket"], dtype=np.uint32), curve=hip.HILBERT,
                                   ngmax=c["ngmax"])
        arrays = [_device(torch.cat([p[k] for p, _ in clouds]).to(torch.float32)) for k in range(4)]
        self.batched.set_particles(*arrays, stream=self.stream)
        self.batched.build(stream=self.stream)
        self.views, self.kept = _Views(self.batched), _Kept(65536 + 16 * (self.n // c["bucket"]))
        v = self.batched.view(stream=self.stream)
        _words(v.neighbors, self.n * self.ngmax, 4).zero_()
        torch.cuda.synchronize()
        self.batched.capture(2, 0.1 * DRIFT, int(seed) & 0xFFFFFF, 0, self.stream)
        self.stream.sync()

    def run(self):
        self.batched.replay(self.stream)
        v, w, n = self.batched.view(stream=self.stream), self.views, self.n
        return {"keys": w(v.keys, n, 8), "perm": w(v.perm, n, 4),
                "particles": [w(p, n, 4) for p in (v.x, v.y, v.z, v.h)],
                "num_leaves": v.num_leaves, "leaves": self.kept("leaves", w(v.leaves, v.num_leaves + 1, 8)),
                "layout": self.kept("layout", w(v.layout, v.num_leaves + 1, 4)),
                "neighbors": w(v.neighbors, n * self.ngmax, 4),
                "neighbor_counts": w(v.neighbor_counts, n, 4)}


class _Served:
    """A burst of requests released at once: 30 % builds of a new cloud from host arrays, the rest updates of a
    resident one; the outputs are the requests' digests over keys, neighbor counts and rows."""

    def __init__(self, c, seed):
        g = _generator(seed)
        builds = max(1, round(0.3 * c["requests"]))
        sizes = _mix(builds, c["nmin"], c["nmax"], seed)
        rng = np.random.RandomState(seed % (1 << 31))
        clouds = []
        for m in sizes:
            arrays, _ = _cloud("plummer", int(m), g)
            clouds.append([a.to(torch.float32).cpu().numpy() for a in arrays])
        self.requests, built = [], 0
        for i in range(c["requests"]):
            build = built * c["requests"] <= i * builds and built < builds
            cloud = built if build else int(rng.randint(built))
            built += build
            x, y, z, h = clouds[cloud] if build else (None,) * 4
            self.requests.append({"id": i, "cloud": cloud, "kind": hip.SERVE_BUILD if build else hip.SERVE_UPDATE,
                                  "n": int(sizes[cloud]), "x": x, "y": y, "z": z, "h": h, "arrival_s": 0.0,
                                  "seed": int(rng.randint(1 << 30))})
        self.slots, self.ngmax = c["slots"], c["ngmax"]

    def run(self):
        res, _ = hip.serve_run(self.requests, slots=self.slots, ngmax=self.ngmax, realtime=False, digests=True)
        res = sorted(res, key=lambda r: r["id"])
        return {"digest": np.array([r["digest"] for r in res], dtype=np.uint64).view(np.int64),
                "status": np.array([r["status"] for r in res], dtype=np.int64),
                "leaves": np.array([r["num_leaves"] for r in res], dtype=np.int64)}


class _Share:
    """One rank's share of a clustered run: full build of the whole set (Morton keys), assignment, halo discovery and
    the gather of the rank's particles with its halos."""

    def __init__(self, c, seed):
        n = c["n"]
        self.n, self.ranks, self.rank = n, c["ranks"], c["rank"]
        self.inputs = [hip.DeviceArray(n, np.float64) for _ in range(4)]
        hip.gaussian_mixture(*self.inputs, n, seed=int(seed), clusters=64, background=0.2, target_neighbors=NEIGHBORS)
        self.box = hip.make_box(0.0, 1.0, np.float64)
        self.pipe = hip.Pipeline(curve=hip.MORTON, key_bits=64, real_bits=64, bucket_size=c["bucket"], ngmax=0)
        self.pipe.sync(*self.inputs, n, self.box, full_build=True)
        self.outputs = [_zeros(n, np.float64) for _ in range(4)]  # a share is never more than the whole
        self.views, self.kept = _Views(self.pipe, self.outputs), _Kept(4096 + 16 * (n // c["bucket"]))

    def run(self):
        self.pipe.sync(*self.inputs, self.n, self.box, full_build=True)
        m = self.pipe.halos(self.ranks, self.rank, self.outputs, self.n)
        v, w = self.pipe.view(), self.views
        return {"keys": w(v.keys, self.n, 8), "perm": w(v.perm, self.n, 4), "num_local": m,
                "leaves": self.kept("leaves", w(v.leaves, v.num_leaves + 1, 8)),
                "flags": self.kept("flags", w(v.halo_flags, v.num_nodes, 1)),
                "layout": self.kept("layout", w(v.local_layout, v.num_leaves + 1, 4)),
                "local": [w(a.ptr, self.n, 8) for a in self.outputs], "assigned": [v.assigned_first, v.assigned_last]}


class _IjLoop:
    """The sum over neighbors of an SPH-like interaction on a synced tree."""

    def __init__(self, c, seed):
        g = _generator(seed)
        n, rb = c["n"], c["real_bits"]
        raw, limits = _cloud("uniform", n, g)
        m = _typed([0.5 + _uniform(n, g)], rb)[0]
        self.n, self.real, self.ngmax, self.box = n, rb // 8, c["ngmax"], _box(limits, rb)
        self.pipe = hip.Pipeline(curve=hip.HILBERT, key_bits=64, real_bits=rb, bucket_size=c["bucket"], ngmax=0)
        self.pipe.sync(*[_device(a) for a in _typed(raw, rb)], n, self.box, full_build=True)
        self.v = self.pipe.view()
        perm = _words(self.v.perm, n, 4).long()
        self.m = _device(m[perm])
        dt = np.float32 if rb == 32 else np.float64
        self.outputs = [_zeros(n, np.uint32 if k == 1 else dt) for k in range(5)]
        self.out = {name: (_words if k == 1 else _floats)(d.ptr, n, d.dtype.itemsize, d)
                    for k, (name, d) in enumerate(zip(("rho", "count", "dmin", "dmax", "fx"), self.outputs))}

    def run(self):
        v = self.v
        hip.ijloop_example(v.x, v.y, v.z, v.h, self.m, 0, self.n, self.box, v.child_offsets, v.parents,
                           v.internal_to_leaf, v.layout, v.centers, v.sizes, v.num_nodes, self.ngmax, *self.outputs,
                           total_bodies=self.n)
        return self.out


class _Sort:
    """Keys of particles in no order, and their stable sort with the gather of x, y, z, h."""

    def __init__(self, c, seed):
        raw, limits = _cloud("plummer", c["n"], _generator(seed))
        n, rb, kb = c["n"], c["real_bits"], c["key_bits"]
        self.box, self.curve = _box(limits, rb), c["curve"]
        self.inputs = [_device(a) for a in _typed(raw, rb)]
        self.outputs = [hip.DeviceArray(n, self.inputs[0].dtype) for _ in range(4)]
        self.keys, self.perm = hip.DeviceArray(n, np.uint64 if kb == 64 else np.uint32), hip.DeviceArray(n, np.uint32)
        self.out = {"keys": _of(self.keys), "perm": _of(self.perm), "particles": [_of(a) for a in self.outputs]}

    def run(self):
        x, y, z, h = self.inputs
        hip.compute_sfc_keys(x, y, z, self.keys, self.box, curve=self.curve)
        hip.sort_gather(self.keys, self.perm, x, y, z, h, *self.outputs)
        return self.out


_KINDS = {"step": _Pipe, "build": _Pipe, "domain": _Domain, "grav": _Domain, "batched": _Batched, "served": _Served,
          "share": _Share, "ijloop": _IjLoop, "sort": _Sort}


# ---------------------------------------------------------------- what a pass cannot do without


def work(case):
    """Bytes: every particle coordinate read and every output written once, rows with their mean length. Flops: eight
    per stored neighbor (three differences, three products, two sums); the sum's own operations on top."""
    kind = case["kind"]
    if kind in ("batched", "served"):
        if kind == "batched":
            n = 2 * int(_mix(case["clouds"], case["nmin"], case["nmax"], 0).sum())  # two steps
            k = 64
        else:
            builds = max(1, round(0.3 * case["requests"]))
            n = int(_mix(builds, case["nmin"], case["nmax"], 0).mean() * case["requests"])
            k = NEIGHBORS
        return {"bytes": n * (32 + 8 + 4 + 4 + 4 * k), "flops": 8.0 * k * n}
    n = case["n"]
    r, key = case.get("real_bits", 64) // 8, case.get("key_bits", 64) // 8
    if kind in ("sort", "share", "grav"):
        extra = 64 * n // case["ranks"] if kind == "share" else 2 * r * n if kind == "grav" else 0
        return {"bytes": n * (8 * r + key + 4) + extra, "flops": 20.0 * n}
    if kind == "ijloop":
        return {"bytes": n * (9 * r + 4), "flops": 20.0 * NEIGHBORS * n}
    return {"bytes": n * (8 * r + key + 4 + 4 + 4 * NEIGHBORS), "flops": 8.0 * NEIGHBORS * n}


# ---------------------------------------------------------------- the computed numbers in 64 bits


def exact(case, seed):
    if case["kind"] != "ijloop" or case["n"] > 2_000_000:
        return None
    g = _generator(seed)
    n = case["n"]
    raw, _ = _cloud("uniform", n, g)
    m = 0.5 + _uniform(n, g)
    x, y, z, h = (a.double() for a in _typed(raw, case["real_bits"]))
    m = _typed([m], case["real_bits"])[0].double()
    order = torch.sort(_hilbert(x, y, z), stable=True)[1]
    p, m, h = torch.stack([x, y, z], 1)[order], m[order], h[order]
    rho, dmin, dmax, fx = _neighbor_sums(p, m, h)
    return {"rho": rho, "count": None, "dmin": dmin, "dmax": dmax, "fx": fx}


def _hilbert(x, y, z):
    """63-bit Hilbert keys of points in the unit cube: the octant's place along the curve, level by level, and the
    rotation it leaves for the levels below."""
    place = torch.tensor([0, 1, 3, 2, 7, 6, 4, 5], device=x.device)
    p = [torch.floor(a * 2097152.0).long().clamp_(max=2097151) for a in (x, y, z)]
    key = torch.zeros_like(p[0])
    for level in range(20, -1, -1):
        b = [(a >> level) & 1 for a in p]
        key = key * 8 + place[4 * b[0] + 2 * b[1] + b[2]]
        xi, yi, zi = (v.bool() for v in b)
        p[0] = p[0] ^ -(xi & (~yi | zi)).long()
        p[1] = p[1] ^ -((xi & (yi | zi)) | (yi & ~zi)).long()
        p[2] = p[2] ^ -((xi & ~yi & ~zi) | (yi & ~zi)).long()
        turn, swap = zi, ~zi & ~yi
        p = [torch.where(turn, p[1], torch.where(swap, p[2], p[0])), torch.where(turn, p[2], p[1]),
             torch.where(turn, p[0], torch.where(swap, p[0], p[2]))]
    return key


def _neighbor_sums(p, m, h):
    """Kernel sum, smallest and largest squared distance and the odd x moment over all neighbors within 2h, by cells
    of that width."""
    n = p.shape[0]
    cells = max(1, int(math.floor(1.0 / (2.0 * float(h.max())))))
    c = (p * cells).long().clamp_(0, cells - 1)
    ident = (c[:, 0] * cells + c[:, 1]) * cells + c[:, 2]
    by = torch.argsort(ident)
    start = torch.searchsorted(ident[by].contiguous(), torch.arange(cells**3 + 1, device=p.device))
    most = int((start[1:] - start[:-1]).max())
    r2 = 4.0 * h * h
    rho, fx = m.clone(), torch.zeros_like(m)
    real = torch.finfo(torch.float64)
    dmin, dmax = torch.full_like(m, real.max), torch.full_like(m, real.min)
    for o in range(27):
        q = c + torch.tensor([o // 9 - 1, o // 3 % 3 - 1, o % 3 - 1], device=p.device)
        inside = ((q >= 0) & (q < cells)).all(1)
        at = ((q[:, 0] * cells + q[:, 1]) * cells + q[:, 2]).clamp_(0, cells**3 - 1)
        lo, hi = start[at], torch.where(inside, start[at + 1], start[at])
        for k in range(most):
            j = by[(lo + k).clamp_(max=n - 1)]
            d = p - p[j]
            d2 = (d * d).sum(1)
            near = (lo + k < hi) & (d2 < r2) & (j != torch.arange(n, device=p.device))
            u = 1.0 - d2 / r2
            zero = torch.zeros_like(m)
            rho += torch.where(near, m[j] * u * u * u, zero)
            fx += torch.where(near, m[j] * d[:, 0], zero)
            dmin = torch.where(near, torch.minimum(dmin, d2), dmin)
            dmax = torch.where(near, torch.maximum(dmax, d2), dmax)
    return rho / (h * h * h), dmin, dmax, fx
