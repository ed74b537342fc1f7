"""Performance cases: the calls a program makes on this library, over the range
of sizes, point distributions, boxes and precisions it makes them with.

``listed()`` names the standing cases, ``draw(rng)`` gives one more of the same
ranges; ``prepare`` makes what a program has in hand (device inputs, the
triangulation object with its buffers), ``run`` is one pass through the public
entry points, ``work`` what such a pass cannot do without, and ``exact`` its
floating-point results in plain 64-bit tensor operations.

Kinds of case:

* ``triangulate``: ``DelaunayGPU.globalDelaunayTriangulation`` of one periodic
  set (uniform points, a jittered triangular lattice, or a square lattice off
  by rounding errors; rectangular or sheared box);
* ``batch``: the same for many uneven sets in one call;
* ``repair``: ``testAndRepairDelaunayTriangulation`` after every point moved a
  little, from the rings of the old positions;
* ``md``: ``BatchedDelaunayGPU.md_run``, the Brownian displace, test and repair
  loop on the device;
* ``voronoi``: energy of the Voronoi tessellation and its gradient.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from gpudelaunaytriangulation_amd import PREC_EXACT, PREC_FP32F, PREC_FP64
from gpudelaunaytriangulation_amd.delaunay import (BatchedDelaunayGPU, Context, DelaunayGPU,
                                                   PeriodicBoundaries)
from gpudelaunaytriangulation_amd.voronoi import voronoi_energy

PRECISION = {"fp64": PREC_FP64, "fp32f": PREC_FP32F, "exact": PREC_EXACT}
ROW3 = math.sqrt(3.0) / 2.0        # row distance of a triangular lattice
MOVE = 0.01                        # displacement per coordinate of a repair, in mean spacings
RING_SLOTS = 16                    # the class's usual first guess of the row stride
PER_SET = 15_300                   # mean points per set that leaves the smallest sets about 1,000
MD_SLOTS = 20                      # rows with room for rings that grow during the loop


def _case(kind, n, **options):
    c = dict(kind=kind, n=n, dist="uniform", precision="fp64", cell=1.0, aspect=1.0, shear=0.0,
             sets=1, steps=0)
    c.update(options)
    return c


def listed():
    cases = {
        # one small tissue or colloid simulation frame: launches and latency count
        "tri_4096": _case("triangulate", 4096),
        # an ordinary ragged set in an oblong box, at the reference's own cell size
        "tri_50021": _case("triangulate", 50021, aspect=1.7, cell=1.1),
        # the headline workload of bench.py, in the library's default precision ...
        "tri_1M": _case("triangulate", 1 << 20),
        # ... and with FP32-filtered predicates
        "tri_1M_fp32f": _case("triangulate", 1 << 20, precision="fp32f"),
        # a slightly disordered crystal: nearly cocircular points everywhere
        "lattice_1M": _case("triangulate", 1 << 20, dist="triangular"),
        # every decision exact: random input, where FP64 mostly certifies itself ...
        "exact_262k": _case("triangulate", 1 << 18, precision="exact"),
        # ... and what the mode is for, a square lattice off by rounding errors
        "exact_lattice_65k": _case("triangulate", 1 << 16, dist="square", precision="exact"),
        # a sheared (Lees-Edwards) box
        "general_1M": _case("triangulate", 1 << 20, shear=0.3125),
        # a parameter sweep: 256 independent simulations triangulated at once (the largest)
        "batch_256": _case("batch", 3_900_000, sets=256),
        # one step of a caller's own dynamics: move, then test and repair
        "repair_1M": _case("repair", 1 << 20),
        # the device-side dynamics of 64 simulations
        "md_64": _case("md", 980_000, sets=64, steps=50),
        # forces of a vertex or self-propelled Voronoi model
        "voronoi_65k": _case("voronoi", 1 << 16),
    }
    return [dict(c, name=name) for name, c in cases.items()]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["triangulate"] * 7 + ["batch", "repair", "repair", "md", "voronoi"])
    opt = dict(aspect=round(rng.uniform(1.0, 2.0), 3), cell=rng.choice([1.0, 1.0, 1.05, 1.1, 1.2]))
    precision = rng.choice(["fp64", "fp64", "fp32f"])
    if kind == "triangulate":
        form = rng.choice(["plain", "plain", "plain", "lattice", "exact", "exact_lattice", "general"])
        if form == "lattice":
            return _case(kind, size(4000, 1 << 20), dist="triangular", precision=precision)
        if form == "exact":
            return _case(kind, size(4000, 1 << 18), precision="exact", **opt)
        if form == "exact_lattice":
            return _case(kind, size(4000, 1 << 16), dist="square", precision="exact")
        if form == "general":
            return _case(kind, size(4000, 1 << 20), shear=round(rng.uniform(-0.6, 0.6), 3), **opt)
        return _case(kind, size(2000, 3_900_000), precision=precision, **opt)
    if kind == "batch":
        n = size(60_000, 3_900_000)
        return _case(kind, n, sets=rng.randint(2, max(2, n // PER_SET)), precision=precision)
    if kind == "repair":
        return _case(kind, size(4000, 1 << 20), precision=precision, **opt)
    if kind == "md":
        n = size(40_000, 980_000)
        return _case(kind, n, sets=rng.randint(1, max(1, n // PER_SET)), precision=precision,
                     steps=rng.randint(20, 50))
    return _case(kind, size(4000, 1 << 18), precision=precision, aspect=opt["aspect"])


# --- inputs -----------------------------------------------------------------

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _box(case):
    """Box matrix (lattice vectors as columns) holding the points at density 1
    (lattices: their own spacing)."""
    if case["dist"] != "uniform":
        nx, ny, h = _lattice(case)
        return (nx * h, 0.0, 0.0, ny * h * (ROW3 if case["dist"] == "triangular" else 1.0))
    ly = math.sqrt(case["n"] / case["aspect"])
    return (case["n"] / ly, case["shear"] * ly, 0.0, ly)


def _lattice(case):
    """Columns, rows and spacing: about n points, an even number of rows."""
    if case["dist"] == "triangular":
        ny = 2 * max(2, round(math.sqrt(case["n"]) / 2))
        return max(4, round(case["n"] / ny)), ny, 1.0
    nx = max(4, round(math.sqrt(case["n"])))
    return nx, nx, 0.1


def _points(case, gen):
    box = _box(case)
    if case["dist"] == "uniform":
        u = torch.rand(case["n"], 2, dtype=torch.float64, device="cuda", generator=gen)
        return torch.stack([u[:, 0] * box[0] + u[:, 1] * box[1], u[:, 1] * box[3]], 1).contiguous()
    nx, ny, h = _lattice(case)
    i = torch.arange(nx * ny, device="cuda")
    col, row = (i % nx).double(), torch.div(i, nx, rounding_mode="floor").double()
    noise = torch.randn(nx * ny, 2, dtype=torch.float64, device="cuda", generator=gen)
    if case["dist"] == "triangular":
        xy = torch.stack([col + 0.5 * (row % 2), row * ROW3], 1) + 1e-5 * noise
    else:       # centres of a square lattice, off by about the last digits written
        xy = torch.stack([(col + 0.5) * h, (row + 0.5) * h], 1) + 1e-13 * noise
    return torch.remainder(xy, torch.tensor([box[0], box[3]], dtype=torch.float64, device="cuda"))


def _cell(case):
    return case["cell"] * (0.1 if case["dist"] == "square" else 1.0)


def _boundaries(case):
    b = _box(case)
    return PeriodicBoundaries(*b) if case["shear"] else PeriodicBoundaries(b[0], b[3])


def _ring_buffers(n, slots):
    return (torch.zeros(n * slots, dtype=torch.int32, device="cuda"),
            torch.zeros(n, dtype=torch.int32, device="cuda"))


def _single(case, gen):
    pts = _points(case, gen)
    n = int(pts.shape[0])
    dg = DelaunayGPU(n, RING_SLOTS, _cell(case), _boundaries(case))
    dg.setPrecision(PRECISION[case["precision"]])
    tri, num = _ring_buffers(n, RING_SLOTS)
    return dict(case=case, dg=dg, pts=pts, tri=tri, num=num)


def _set_sizes(case):
    """Uneven set sizes, log-uniform over a factor of 64, summing to about n."""
    k = case["sets"]
    w = [math.exp(math.log(64.0) * ((0.5 + 0.618034 * s) % 1.0)) for s in range(k)]
    return [max(64, round(case["n"] * v / sum(w))) for v in w]


def _batched(case, gen, slots):
    sizes = _set_sizes(case)
    sides = [math.sqrt(s) for s in sizes]
    scale = torch.repeat_interleave(torch.tensor(sides, dtype=torch.float64, device="cuda"),
                                    torch.tensor(sizes, device="cuda"))
    pts = torch.rand(sum(sizes), 2, dtype=torch.float64, device="cuda", generator=gen)
    pts = (pts * scale[:, None]).contiguous()
    bd = BatchedDelaunayGPU(sizes, [(s, s) for s in sides], slots, case["cell"],
                            precision=PRECISION[case["precision"]])
    tri, num = _ring_buffers(bd.N, slots)
    return dict(case=case, bd=bd, pts=pts, tri=tri, num=num)


def prepare(case, seed):
    gen = _generator(seed)
    kind = case["kind"]
    if kind == "triangulate":
        return _single(case, gen)
    if kind == "batch":
        return _batched(case, gen, RING_SLOTS)
    if kind == "repair":
        st = _single(case, gen)
        st["dg"].globalDelaunayTriangulation(st["pts"], st["tri"], st["num"])
        st["tri0"], st["num0"] = st["tri"].clone(), st["num"].clone()
        move = torch.randn(st["pts"].shape, dtype=torch.float64, device="cuda", generator=gen)
        b = _box(case)
        side = torch.tensor([b[0], b[3]], dtype=torch.float64, device="cuda")
        st["moved"] = torch.remainder(st["pts"] + MOVE * move, side).contiguous()
        return st
    if kind == "md":
        st = _batched(case, gen, MD_SLOTS)
        st["bd"].globalDelaunayTriangulation(st["pts"], st["tri"], st["num"])
        st["pts0"], st["tri0"], st["num0"] = (st[k].clone() for k in ("pts", "tri", "num"))
        st["seed"] = int(seed) & 0xFFFF
        return st
    st = _single(dict(case, precision="fp64"), gen)
    st["case"] = case
    st["dg"].globalDelaunayTriangulation(st["pts"], st["tri"], st["num"])
    st["xy"] = st["pts"].clone().requires_grad_(True)
    st["ctx"] = Context(0)
    st["box"] = (_box(case)[0], _box(case)[3])
    return st


# --- one pass ---------------------------------------------------------------

def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "triangulate":
        st["dg"].globalDelaunayTriangulation(st["pts"], st["tri"], st["num"])
        return st["tri"], st["num"]
    if kind == "batch":
        st["bd"].globalDelaunayTriangulation(st["pts"], st["tri"], st["num"])
        return st["tri"], st["num"]
    if kind == "repair":
        # the rings of the old positions are kept, as by a program that may
        # reject a move
        st["tri"].copy_(st["tri0"])
        st["num"].copy_(st["num0"])
        st["dg"].testAndRepairDelaunayTriangulation(st["moved"], st["tri"], st["num"])
        return st["tri"], st["num"]
    if kind == "md":
        # each trajectory starts from the same kept state
        st["pts"].copy_(st["pts0"])
        st["tri"].copy_(st["tri0"])
        st["num"].copy_(st["num0"])
        st["bd"].md_run(st["pts"], st["tri"], st["num"], case["steps"], MOVE, seed=st["seed"])
        return st["pts"], st["tri"], st["num"]
    energy = voronoi_energy(st["xy"], st["tri"], st["num"], st["box"], a0=1.0, p0=3.8,
                            precision=PRECISION[case["precision"]], context=st["ctx"])
    (grad,) = torch.autograd.grad(energy, st["xy"])
    return energy.detach(), grad


# --- what a pass cannot do without ------------------------------------------

def work(case):
    """Per point: a position is 16 bytes, a ring 6 entries and a count (28
    bytes); of the operations, one in-circle predicate (about 17) for each of
    the 3 edges per point, and for the energy 6 circumcentres, lengths and
    their derivatives (about 60 each)."""
    n = case["n"]
    if case["kind"] in ("triangulate", "batch"):
        return {"bytes": 44.0 * n, "flops": 51.0 * n}
    if case["kind"] == "repair":       # rings copied, then read with the positions; a sixth rewritten
        return {"bytes": (28.0 + 28.0 + 28.0 + 16.0 + 28.0 / 6.0) * n, "flops": 51.0 * n}
    if case["kind"] == "md":           # per step: positions moved, rings read, a sixth rewritten
        step = 32.0 + 28.0 + 28.0 / 6.0
        return {"bytes": (88.0 + step * case["steps"]) * n, "flops": 61.0 * n * case["steps"]}
    return {"bytes": (16.0 + 28.0 + 16.0) * n, "flops": 360.0 * n}


# --- floating-point results in 64 bits --------------------------------------

def exact(case, seed):
    """Rings and counts are whole numbers, and the loop's positions follow the
    library's own noise stream: only the energy and its gradient have values
    of this kind."""
    if case["kind"] != "voronoi":
        return None
    st = prepare(case, seed)           # the inputs: positions and their ring table
    x = st["pts"].cpu()
    n = int(x.shape[0])
    rows = st["tri"].cpu().view(n, -1).long()
    cnt = st["num"].cpu().long()
    slots = int(cnt.max())
    m = torch.arange(slots)
    valid = m[None, :] < cnt[:, None]
    here = torch.where(valid, rows[:, :slots], rows[:, :1])
    after = torch.gather(rows[:, :slots], 1, torch.remainder(m[None, :] + 1, cnt[:, None]))
    after = torch.where(valid, after, rows[:, :1])
    side = torch.tensor(st["box"], dtype=torch.float64)
    xg = x.clone().requires_grad_(True)

    def displacement(j):
        d = xg[j] - xg[:, None, :]
        return d - side * torch.round(d.detach() / side)

    def cross(p, q):
        return p[..., 0] * q[..., 1] - p[..., 1] * q[..., 0]

    a, b = displacement(here), displacement(after)
    # unused slots: any proper triangle, masked out below
    a = torch.where(valid[..., None], a, torch.tensor([1.0, 0.0], dtype=torch.float64))
    b = torch.where(valid[..., None], b, torch.tensor([0.0, 1.0], dtype=torch.float64))
    an, bn = (a * a).sum(-1), (b * b).sum(-1)
    s = 0.5 / cross(a, b)
    h = torch.stack([s * (an * b[..., 1] - a[..., 1] * bn), s * (a[..., 0] * bn - an * b[..., 0])], -1)
    nxt = torch.remainder(m[None, :] + 1, cnt[:, None])
    hn = torch.gather(h, 1, nxt[..., None].expand(-1, -1, 2))
    step = torch.where(valid[..., None], hn - h, torch.ones(2, dtype=torch.float64))
    zero = torch.zeros((), dtype=torch.float64)
    area = 0.5 * torch.where(valid, cross(h, hn), zero).sum(1)
    perim = torch.where(valid, (step * step).sum(-1).sqrt(), zero).sum(1)
    energy = ((area - 1.0) ** 2 + (perim - 3.8) ** 2).sum()
    (grad,) = torch.autograd.grad(energy, xg)
    return np.array([float(energy.detach())]), grad.numpy()
