"""Performance cases of the partitioner: what its users have it do, from the
smallest meshes to the largest, through the public entry points.

A case names a mesh (its generator and sizes), the call and the call's
options.  Meshes are generated on the GPU from the seed alone: every
generator returns (vtx int64 [nel, nv], xyz float64 [nel, nv, ndim]) in the
layout parrsb_part_mesh takes, with the shapes of the repository's workloads
(jittered hex boxes, smoothly warped boxes, warped annular pipes, quad grids
with holes) and, for the connectivity, boxes graded along each axis.

Calls:
  rsb      recursive spectral bisection, device pointers (part_mesh_dev)
  rsb_host the same on host arrays (part_mesh), as a C or Fortran solver calls it
  rcb, rib the geometric partitioners alone (partitioner 1 and 2)
  conn     vertex ids from corner coordinates (parrsb_amd_conn_mesh_dev)
  quality  the figures of a finished partition (quality_dev)
"""
import math
import os
import random

import torch

import parrsb_amd as pa
from parrsb_amd import lws_train

_HEX = ((0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1))
_QUAD = ((0, 0), (1, 0), (1, 1), (0, 1))


def _case(call, mesh, nx, ny, nz=0, parts=0, bits=64, learned=False, mg=False, shuffled=False):
    """nx, ny, nz: cells per lattice direction (nz = 0: quads); parts: number
    of parts; bits: Lanczos vector precision; learned: the shipped learned
    start; mg: the MG inverse iteration instead of Lanczos; shuffled: elements
    in random order instead of lattice order."""
    return dict(call=call, mesh=mesh, nx=nx, ny=ny, nz=nz, parts=parts, bits=bits,
                learned=learned, mg=mg, shuffled=shuffled)


def listed():
    def named(name, *a, **k):
        return dict(_case(*a, **k), name=name)

    return [
        # the smallest mesh of the test suite with the default options: what a
        # user's first run and every small study costs; launches and latency
        named("hex16_f64", "rsb", "box", 16, 16, 16, parts=8),
        # an odd, ragged box into a part count that is no power of two, its
        # elements in a mesher's own order
        named("ragged_f32", "rsb", "box", 31, 22, 19, parts=23, bits=32, shuffled=True),
        # a mid-size solver start-up: host arrays, default options
        named("host_f64", "rsb_host", "warped", 64, 60, 48, parts=256),
        # a million elements, about a thousand per part: the default precision,
        # and the benchmark's settings (32-bit vectors, learned start)
        named("hex1m_f64", "rsb", "box", 128, 128, 64, parts=1024),
        named("hex1m_f32_learned", "rsb", "box", 128, 128, 64, parts=1024, bits=32, learned=True),
        # planar meshes with holes: narrow necks, components, slow convergence
        named("quads_f32", "rsb", "holes", 512, 509, parts=256, bits=32),
        # a long pipe, 2M elements: slow convergence at many levels
        named("pipe2m_f32", "rsb", "pipe", 8, 256, 1024, parts=2048, bits=32),
        # the largest mesh: its first two cuts, where one iteration streams
        # through every element
        named("warped16m_f32", "rsb", "warped", 256, 256, 256, parts=4, bits=32),
        # the multigrid solver
        named("mg_pipe", "rsb", "pipe", 4, 48, 128, parts=24, mg=True),
        # the geometric partitioner alone, a common quick choice at scale
        named("rcb1m", "rcb", "warped", 128, 128, 64, parts=1000),
        # connectivity of a mesh read from coordinates (a genmap run's first
        # step), its elements in the file's order
        named("conn1m", "conn", "graded", 127, 120, 65, shuffled=True),
        # checking a partition
        named("quality1m", "quality", "warped", 128, 128, 64, parts=1024),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    call = rng.choice(["rsb"] * 6 + ["rsb_host", "mg", "rcb", "rib", "conn", "quality"])
    mg = call == "mg"
    if mg:
        call = "rsb"
    mesh = rng.choice(["box", "warped", "pipe", "holes"])
    if call == "conn" and mesh != "holes":
        mesh = "graded"  # the search separates points axis by axis
    top = 3e4 if mg else 1.5e6 if call in ("rcb", "rib", "conn", "quality") else 1e6
    if mesh == "holes":
        top = min(top, 2.6e5)
    nel = _log(rng, 2e3, top)
    if mesh == "holes":
        a = math.exp(rng.uniform(-0.5, 0.5))
        nx, ny, nz = max(8, round(math.sqrt(nel) * a)), max(8, round(math.sqrt(nel) / a)), 0
    elif mesh == "pipe":
        nx = rng.randrange(2, 9)
        ny = max(8, round(math.sqrt(nel / nx) * math.exp(rng.uniform(-0.7, 0.0))))
        nz = max(2, round(nel / (nx * ny)))
    else:
        a, b = math.exp(rng.uniform(-0.4, 0.4)), math.exp(rng.uniform(-0.4, 0.4))
        nx, ny = max(3, round(nel ** (1 / 3) * a)), max(3, round(nel ** (1 / 3) * b))
        nz = max(3, round(nel / (nx * ny)))
    n = nx * ny * max(nz, 1)
    parts = 0 if call == "conn" else max(2, round(n / _log(rng, 100, 4000)))
    bits = rng.choice([64, 32])
    return _case(call, mesh, nx, ny, nz, parts=parts, bits=bits, mg=mg,
                 learned=call == "rsb" and bits == 32 and not mg and rng.random() < 0.4,
                 shuffled=rng.random() < 0.3 or call == "conn")


# --- meshes -----------------------------------------------------------------
def _cells(nx, ny, nz, dev):
    """Lattice index (i, j, k) of every cell, x fastest."""
    e = torch.arange(nx * ny * nz, device=dev)
    return e % nx, (e // nx) % ny, e // (nx * ny)


def _warp(u, rng, amp):
    """Per coordinate d: sum_e a_de sin(2 pi k_de u_e + phi_de), one column of
    the seeded smooth displacement of points u in [0, 1]^3."""
    for d in range(3):
        y = torch.zeros_like(u[0])
        for e in range(3):
            a, k, ph = rng.uniform(0.3 * amp, amp), rng.choice((1.0, 2.0)), rng.uniform(0, 2 * math.pi)
            y += a * torch.sin(2 * math.pi * k * u[e] + ph)
        yield y


def _mesh(case, seed, dev):
    rng = random.Random("%d" % seed)
    gen = torch.Generator(device=dev).manual_seed(seed)
    nx, ny, nz, kind = case["nx"], case["ny"], case["nz"], case["mesh"]
    if kind == "holes":
        # disks of 2 to 40 cells' radius (less on small grids) taken out until
        # 5% of the cells are gone, the last disk only as far as it takes
        m = nx + 1
        i, j, _ = _cells(nx, ny, 1, dev)
        keep = torch.ones(nx * ny, dtype=torch.bool, device=dev)
        left, top = nx * ny - nx * ny // 20, max(2.5, min(40.0, 0.08 * min(nx, ny)))
        while (over := int(keep.sum()) - left) > 0:
            r, cx, cy = rng.uniform(2.0, top), rng.uniform(0, nx), rng.uniform(0, ny)
            d = (i + 0.5 - cx) ** 2 + (j + 0.5 - cy) ** 2
            disk = torch.nonzero(keep & (d <= r * r)).flatten()
            keep[disk[torch.argsort(d[disk], stable=True)][:over]] = False
        h = 1.0 / max(nx, ny)
        i, j = i[keep], j[keep]
        vtx = torch.stack([1 + i + a + m * (j + b) for a, b in _QUAD], 1)
        xyz = torch.stack([torch.stack([(i + a) * h, (j + b) * h], 1) for a, b in _QUAD], 1).double()
    else:
        my = ny if kind == "pipe" else ny + 1  # a pipe closes around its axis
        sx, sy = nx + 1, (nx + 1) * my
        i, j, k = _cells(nx, ny, nz, dev)
        vtx = torch.stack([1 + i + a + sx * ((j + b) % my) + sy * (k + c) for a, b, c in _HEX], 1)
        del i, j, k
        v = torch.arange(sy * (nz + 1), device=dev)
        li, lj, lk = (x.double() for x in (v % sx, (v // sx) % my, v // sy))
        del v
        if kind == "pipe":
            r, th = 0.5 + 0.5 * li / nx, 2 * math.pi * lj / ny
            length = nz * 2 * math.pi * 0.75 / ny
            X = [r * torch.cos(th), r * torch.sin(th), length * lk / nz]
            u = [0.5 + 0.5 * X[0], 0.5 + 0.5 * X[1], lk / nz]
            size, amp = 2.0, 0.05
        elif kind == "graded":  # cell sizes vary along each axis by a factor of up to 3
            X = []
            for x, n in ((li, nx), (lj, ny), (lk, nz)):
                t, a = x / n, rng.uniform(0.02, 0.08)
                X.append((t + a * torch.sin(2 * math.pi * t + rng.uniform(0, 6.28))) * n / max(nx, ny, nz))
            u, amp = None, 0.0
        else:
            h = 1.0 / max(nx, ny, nz)
            X = [li * h, lj * h, lk * h]
            u = [li / nx, lj / ny, lk / nz]
            size, amp = 1.0, 0.05 if kind == "warped" else 0.0
        if amp:
            X = [x + size * y for x, y in zip(X, _warp(u, rng, amp))]
        del li, lj, lk, u
        P = torch.stack(X, 1)
        del X
        xyz = P[vtx - 1]
        del P
        if kind == "box":  # each element moved as a whole by up to a tenth of a cell
            d = torch.rand((vtx.shape[0], 1, 3), generator=gen, device=dev, dtype=torch.float64)
            xyz += (0.2 * d - 0.1) / max(nx, ny, nz)
    if case["shuffled"]:
        p = torch.randperm(vtx.shape[0], generator=gen, device=dev)
        vtx, xyz = vtx[p], xyz[p]
    else:  # lattice order, from a cell of its own on
        k = rng.randrange(vtx.shape[0])
        vtx, xyz = torch.roll(vtx, k, 0), torch.roll(xyz, k, 0)
    return vtx.contiguous(), xyz.contiguous()


def _slabs(xyz, parts, rng):
    """A finished partition's stand-in: about equal wavy bricks of the mesh."""
    c = xyz.mean(1)
    lo, hi = c.amin(0), c.amax(0)
    u = (c - lo) / (hi - lo)
    ndim = c.shape[1]
    n = max(1, round(parts ** (1.0 / ndim)))
    at = torch.zeros(c.shape[0], dtype=torch.int64, device=c.device)
    for d in range(ndim):
        w = u[:, d] + 0.02 * torch.sin(6 * u[:, (d + 1) % ndim] + rng.uniform(0, 6.28))
        at = at * n + (w * n).floor().long().clamp(0, n - 1)
    return (at % parts).int()


# --- the interface ----------------------------------------------------------
_weights = []


def _learned():
    if not _weights:
        _weights.append(lws_train.load_params(
            os.path.join(os.path.dirname(pa.__file__), "lws_weights.bin")))
    return _weights[0]


def prepare(case, seed):
    dev = torch.device("cuda")
    vtx, xyz = _mesh(case, seed, dev)
    nel, nv = vtx.shape
    s = dict(case=case, nel=nel, nv=nv, vtx=vtx, xyz=xyz)
    s["parts"] = min(case["parts"], nel)
    if case["call"] == "rsb_host":
        s["vtx"], s["xyz"] = vtx.cpu().numpy(), xyz.cpu().numpy()
    elif case["call"] == "conn":
        # corners of one vertex agree to single precision, as mesh files hold them
        gen = torch.Generator(device=dev).manual_seed(seed + 1)
        e = torch.rand(xyz.shape, generator=gen, device=dev, dtype=torch.float64) - 0.5
        s["xyz"] = xyz + 6e-8 * e
        s["out"] = torch.zeros((nel, nv), dtype=torch.int64, device=dev)
        del s["vtx"]
    elif case["call"] == "quality":
        s["part"] = _slabs(xyz, s["parts"], random.Random(seed))
        del s["xyz"]
    else:
        s["out"] = torch.zeros(nel, dtype=torch.int32, device=dev)
    s["learned"] = _learned() if case["learned"] else None
    torch.cuda.synchronize()
    return s


def run(s):
    c = s["case"]
    call, nel, nv, parts = c["call"], s["nel"], s["nv"], s["parts"]
    if call == "quality":
        return pa.quality_dev(s["part"].data_ptr(), s["vtx"].data_ptr(), nel, nv, parts)
    if call == "conn":
        rc = pa.lib().parrsb_amd_conn_mesh_dev(s["out"].data_ptr(), s["xyz"].data_ptr(), nel,
                                               3 if nv == 8 else 2, 0.2)
        if rc:
            raise pa.ParrsbError(rc, pa.last_error())
        return s["out"]
    pa.set_precision(c["bits"])
    pa.set_warm_start(s["learned"])
    if call == "rsb_host":
        return pa.part_mesh(s["vtx"], s["xyz"], nv, parts)[0]
    kind = {"rsb": 0, "rcb": 1, "rib": 2}[call]
    pa.part_mesh_dev(s["out"].data_ptr(), s["vtx"].data_ptr(), s["xyz"].data_ptr(), nel, nv, parts,
                     partitioner=kind, rsb_algo=1 if c["mg"] else 0)
    return s["out"]


def work(case):
    """Inputs read once, outputs written once; for the spectral calls one
    application of every level's Laplacian (2 operations per entry)."""
    n = case["nx"] * case["ny"] * max(case["nz"], 1)
    nv, ndim, nb = (8, 3, 26) if case["nz"] else (4, 2, 8)
    ids, crd, flops = 8 * nv * n, 8 * nv * ndim * n, 0
    if case["call"] == "conn":
        return {"bytes": crd + ids, "flops": 0}
    if case["call"] == "quality":
        return {"bytes": ids + 4 * n, "flops": 0}
    if case["call"] in ("rsb", "rsb_host"):
        flops = 2 * nb * n * max(1, math.ceil(math.log2(max(2, case["parts"]))))
    return {"bytes": ids + crd + 4 * n, "flops": flops}


def exact(case, seed):
    return None  # every output is whole numbers: part numbers, vertex ids, counts
