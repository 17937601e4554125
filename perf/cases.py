"""Performance cases of the block-stencil path, through its Python entry points.

A case is a dict of plain values.  Its "kind" is the call a program makes:

  step    one diffusion_step (Laplacian stored, FP64 norm)
  run     diffusion_run over several Euler steps, a norm per step
  weno    weno5 face states of every component
  sweep   one jacobi_sweep2 on a z-stretched grid
  solve   jacobi_solve, a fixed number of cycles
  batch   one Batch.run over uneven grids
  labs    lab_all, the ghost-extended blocks of a whole grid
  fields  grid_field_op arithmetic, grid_sums and grid_compare

"bc" is six letters, one per domain face (x low, x high, y low, ...): P
periodic, D Dirichlet, A absorbing, S / N symmetry of sign +1 / -1.

Grids live in torch tensors (Cartesian.from_tensor), inputs come from the
seed alone, and every pass runs on the default stream with the library's
built-in tiles.
"""
import ctypes
import math
import random
import types

import numpy as np
import torch

import cubismnova_amd as cnv

DEV = "cuda"
WALL = (0.5, -0.25, 0.125, -0.5, 0.25, -0.125)  # Dirichlet value of each domain face
NUDT = 0.1                                      # Euler step in units of h^2 (bench.py)
OMEGA = 2.0 / 3.0


def listed():
    return [
        # the smallest ordinary call: one step of a 64^3 grid of 16^3 blocks
        dict(name="step_64_f64", kind="step", nb="4,4,4", n="16,16,16", dtype="f64", ncomp=1, bc="PPPPPP"),
        # time stepping of a large periodic box in the fast precision
        dict(name="run_256_f32", kind="run", nb="8,8,8", n="32,32,32", dtype="f32", ncomp=1, bc="PPPPPP", steps=100,
             norms=True),
        # time stepping between walls, double precision, an odd number of steps
        dict(name="run_walls_f64", kind="run", nb="6,5,4", n="32,32,32", dtype="f64", ncomp=1, bc="DDPPAS", steps=41,
             norms=True),
        # several components on block edges that are no power of two
        dict(name="run_ragged_f32", kind="run", nb="6,4,5", n="24,24,24", dtype="f32", ncomp=3, bc="AAPPDS", steps=20,
             norms=True),
        # many small blocks, as block-adaptive applications keep them
        dict(name="run_blocks8_f64", kind="run", nb="16,16,16", n="8,8,8", dtype="f64", ncomp=1, bc="PPPPPP",
             steps=10, norms=False),
        # face states of a compressible state, the heaviest operator
        dict(name="weno5_256_f32", kind="weno", nb="8,8,8", n="32,32,32", dtype="f32", ncomp=5, bc="PPAAAA"),
        # the same on uneven blocks in double precision
        dict(name="weno5_ragged_f64", kind="weno", nb="8,6,4", n="20,12,18", dtype="f64", ncomp=2, bc="PPSSAD"),
        # the smoother of the stretched-grid Poisson solver at its full size
        dict(name="sweep_512_f32", kind="sweep", nb="8,8,8", n="64,64,64", dtype="f32", ncomp=1, bc="DDDDDD"),
        # a small Poisson solve, FP32 sweeps refined in FP64: launches count
        dict(name="solve_64_refined", kind="solve", nb="2,2,2", n="32,32,32", dtype="f64", ncomp=1, bc="DDDDDD",
             refine=True, cycles=6, sweeps=50),
        # 96 grids of uneven blocks, components, operators and walls at once
        dict(name="batch_96_f32", kind="batch", grids=96, maxb="8,8,4", salt=4),
        # ghost-extended blocks for user-written operators, corners included
        dict(name="labs_128_f64", kind="labs", nb="8,8,8", n="16,16,16", dtype="f64", ncomp=1, bc="AAPPDS", lo=-3,
             hi=4, tensorial=True, entity="cell"),
        # Runge-Kutta style field arithmetic with conservation sums
        dict(name="fields_256_f32", kind="fields", nb="4,4,4", n="64,64,64", dtype="f32", ncomp=3, entity="cell"),
    ]


EDGES = (8, 12, 16, 20, 24, 32, 40, 48, 64)


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_bc(rng, letters="DASN", periodic=0.4):
    return "".join("PP" if rng.random() < periodic else rng.choice(letters) + rng.choice(letters) for _ in range(3))


def _draw_blocks(rng, cells, edges=EDGES, cubic=0.7):
    """Block cells and block counts of a grid of about `cells` cells."""
    e = rng.choice([x for x in edges if x ** 3 <= cells] or [min(edges)])
    n = [e] * 3 if rng.random() < cubic else [max(4, e + rng.choice((-3, -2, 0, 0, 1, 4))) for _ in range(3)]
    want = max(1.0, cells / float(n[0] * n[1] * n[2]))
    nb = [max(1, int(round(want ** (1 / 3) * rng.uniform(0.7, 1.4)))) for _ in range(2)]
    nb.append(max(1, int(round(want / (nb[0] * nb[1])))))
    while nb[0] * nb[1] * nb[2] > 4 * want and max(nb) > 1:
        nb[nb.index(max(nb))] -= 1
    return ",".join(map(str, nb)), ",".join(map(str, n))


def draw(rng):
    kind = rng.choice(("step", "run", "run", "weno", "sweep", "solve", "batch", "labs", "fields"))
    dtype = rng.choice(("f32", "f64"))
    if kind == "batch":
        mb = [rng.randint(1, 6), rng.randint(1, 6), rng.randint(1, 4)]
        return dict(kind=kind, grids=_log(rng, 4, 64), maxb=",".join(map(str, mb)), salt=rng.randrange(1, 1 << 16))
    if kind in ("sweep", "solve"):
        top = 1.6e7 if kind == "sweep" else 5e5
        e = rng.choice((16, 32, 64))
        n = "%d,%d,%d" % (e, e, rng.choice((e, e, max(8, e - 4))))
        want = max(1.0, _log(rng, 2e4, top) / float(e ** 3))
        nb = [max(1, int(round(want ** (1 / 3) * rng.uniform(0.7, 1.3)))) for _ in range(3)]
        c = dict(kind=kind, nb=",".join(map(str, nb)), n=n, dtype=dtype, ncomp=1, bc=_draw_bc(rng, periodic=0.25))
        if kind == "solve":
            refine = rng.random() < 0.6
            c.update(refine=refine, dtype="f64" if refine else dtype, cycles=rng.randint(1, 6),
                     sweeps=2 * rng.randint(2, 25))
        return c
    if kind == "run":
        steps = _log(rng, 1, 60)
        nb, n = _draw_blocks(rng, _log(rng, 4e3, 6e7 / max(8, steps)))
        return dict(kind=kind, nb=nb, n=n, dtype=dtype, ncomp=rng.randint(1, 3), bc=_draw_bc(rng), steps=steps,
                    norms=rng.random() < 0.7)
    if kind == "step":
        nb, n = _draw_blocks(rng, _log(rng, 2e3, 4e6))
        return dict(kind=kind, nb=nb, n=n, dtype=dtype, ncomp=rng.randint(1, 3), bc=_draw_bc(rng))
    if kind == "weno":
        nb, n = _draw_blocks(rng, _log(rng, 4e3, 4e6))
        return dict(kind=kind, nb=nb, n=n, dtype=dtype, ncomp=rng.randint(1, 5), bc=_draw_bc(rng, "DAS"))
    entity = rng.choice(("cell", "cell", "node", "face"))
    if kind == "labs":
        nb, n = _draw_blocks(rng, _log(rng, 4e3, 2e6), edges=(8, 12, 16, 20, 24, 32))
        return dict(kind=kind, nb=nb, n=n, dtype=dtype, ncomp=1, bc=_draw_bc(rng, "DAS"), lo=-rng.randint(1, 3),
                    hi=rng.randint(2, 4), tensorial=rng.random() < 0.5, entity=entity)
    nb, n = _draw_blocks(rng, _log(rng, 4e3, 8e6))
    return dict(kind=kind, nb=nb, n=n, dtype=dtype, ncomp=rng.randint(1, 3), entity=entity)


# ------------------------------------------------------------------ layout


def _three(s):
    return tuple(int(x) for x in s.split(","))


def _torch(dtype):
    return torch.float64 if dtype == "f64" else torch.float32


def _size(dtype):
    return 8 if dtype == "f64" else 4


def _to_blocks(u, nb, n):
    """(Z, Y, X) -> (blocks, cells per block), blocks and cells x-fastest."""
    v = u.reshape(nb[2], n[2], nb[1], n[1], nb[0], n[0]).permute(0, 2, 4, 1, 3, 5)
    return v.reshape(nb[0] * nb[1] * nb[2], n[0] * n[1] * n[2])


def _stride(n, dtype):
    per = 32 // _size(dtype)
    return (n[0] * n[1] * n[2] + per - 1) // per * per


def _storage(ncomp, nb, n, dtype, entity="cell"):
    """Zeroed grid memory (slabs, blocks, stride) in the library's layout:
    blocks rounded up to 32 bytes, one more element per dimension in node and
    face grids, three slabs per component in face grids."""
    plus = 0 if entity == "cell" else 1
    stride = _stride([m + plus for m in n], dtype)
    ncomp = 3 * ncomp if entity == "face" else ncomp
    return torch.zeros((ncomp, nb[0] * nb[1] * nb[2], stride), dtype=_torch(dtype), device=DEV)


def _grid(t, nb, n, ncomp, entity="cell"):
    return cnv.Cartesian.from_tensor(t, nb, n, ncomp=ncomp, entity=entity)


class Out:
    """Grid memory of `ncomp` components, the grid over it and its cells."""

    def __init__(self, nb, n, dtype, ncomp, values=None, bc=None, wall=None):
        self.t = _storage(ncomp, nb, n, dtype)
        cells = n[0] * n[1] * n[2]
        self.cells = self.t[:, :, :cells]
        if values is not None:
            for c, v in enumerate(values):
                self.cells[c].copy_(_to_blocks(v, nb, n))
        self.g = _grid(self.t, nb, n, ncomp)
        if bc:
            _walls(self.g, bc, wall)


def _walls(g, bc, wall=None):
    for f, letter in enumerate(bc):
        d, s = f // 2, f % 2
        if letter == "D":
            g.addFaceBC(cnv.Dirichlet(d, s, (WALL if wall is None else wall)[f]))
        elif letter == "A":
            g.addFaceBC(cnv.Absorbing(d, s))
        elif letter in "SN":
            g.addFaceBC(cnv.Symmetry(d, s, 1.0 if letter == "S" else -1.0))


# ------------------------------------------------------------------ inputs


def _axes(shape):
    return [(torch.arange(m, dtype=torch.float64, device=DEV) + 0.5) / m for m in shape]


def _modes(shape, r, count=8, kmax=16):
    """Sum of Fourier modes of amplitude 1/|k| and random phase, (Z, Y, X) FP64."""
    z, y, x = _axes(shape)
    u = torch.zeros(shape, dtype=torch.float64, device=DEV)
    done = 0
    while done < count:
        k = [r.randint(-kmax, kmax) for _ in range(3)]
        m = math.sqrt(sum(v * v for v in k))
        if not 1.0 <= m <= kmax:
            continue
        a = 2 * math.pi * k[0] * x
        b = 2 * math.pi * (k[1] * y[None, :] + k[2] * z[:, None]) + r.random() * 2 * math.pi
        u += (torch.cos(b)[:, :, None] * torch.cos(a) - torch.sin(b)[:, :, None] * torch.sin(a)) / m
        done += 1
    return u


def _noise(shape, seed, scale):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.rand(shape, generator=g, dtype=torch.float64, device=DEV) * 2 - 1) * scale


def _scalar(shape, seed, c):
    r = random.Random(seed * 64 + c)
    return _modes(shape, r) + _noise(shape, seed * 64 + c, 0.1)


def _compressible(shape, seed, c):
    """Component c of (rho, rho u, rho v, rho w, E): smooth background and a
    steep planar pressure front of ratio 10."""
    r = random.Random(seed * 64)
    rho = 1.0 + 0.1 * _modes(shape, r, 4, 4)
    if c % 5 == 0:
        return rho
    vel = [0.1 * _modes(shape, r, 2, 4) for _ in range(3)]
    if c % 5 < 4:
        return rho * vel[c % 5 - 1]
    z, y, x = _axes(shape)
    nx, ny, nz = (r.uniform(0.3, 1.0) for _ in range(3))
    s = nx * (x - 0.5) + (ny * (y - 0.5))[:, None] + (nz * (z - 0.5))[:, None, None]
    p = 1.0 + 4.5 * (1.0 + torch.tanh(s * shape[0] / 2.0))
    return p / 0.4 + 0.5 * rho * (vel[0] ** 2 + vel[1] ** 2 + vel[2] ** 2)


def _zfaces(m):
    j = np.arange(m + 1, dtype=np.float64)
    return 0.5 * (1.0 + np.tanh(2.0 * (2.0 * j / m - 1.0)) / np.tanh(2.0))


def _source(shape, seed):
    """Three Gaussian sources, mean removed."""
    r = random.Random(seed)
    z, y, x = _axes(shape)
    zf = torch.from_numpy(_zfaces(shape[0])).to(DEV)
    z = 0.5 * (zf[1:] + zf[:-1])
    f = torch.zeros(shape, dtype=torch.float64, device=DEV)
    for _ in range(3):
        c = [r.uniform(0.2, 0.8) for _ in range(3)]
        gx, gy, gz = (torch.exp(-((v - m) ** 2) / (2 * 0.05 ** 2)) for v, m in zip((x, y, z), c))
        f += r.uniform(-1, 1) * gz[:, None, None] * gy[None, :, None] * gx
    return f - f.mean()


def _shape(nb, n):
    return nb[2] * n[2], nb[1] * n[1], nb[0] * n[0]


def _inputs(case, seed):
    """The global (Z, Y, X) FP64 fields of a case, rounded to its dtype."""
    nb, n = _three(case["nb"]), _three(case["n"])
    shape, T = _shape(nb, n), _torch(case["dtype"])
    make = _compressible if case["kind"] == "weno" else _scalar
    return [make(shape, seed, c).to(T) for c in range(case["ncomp"])]


def _nudt(nb, n):
    return NUDT * min(1.0 / (nb[d] * n[d]) for d in range(3)) ** 2


def _batch_specs(case):
    """Uneven grids: block counts up to maxb, edges 8 / 16 / 32, 1-3
    components, a diffusion step (ghost 1 or 3) or WENO5 (ghost 3), walls or
    periodic per axis."""
    r = random.Random(case["salt"])
    specs = []
    for _ in range(case["grids"]):
        nb = tuple(r.randint(1, m) for m in _three(case["maxb"]))
        e = r.choice((8, 16, 32))
        op = r.choice(("weno5", "diffusion"))
        specs.append(dict(nb=nb, n=(e, e, e), ncomp=r.randint(1, 3), op=op,
                          ghost=3 if op == "weno5" else r.choice((1, 3)), bc=_draw_bc(r, "DA"),
                          wall=[r.uniform(-1, 1) for _ in range(6)]))
    return specs


def _batch_fields(spec, seed, i):
    shape = _shape(spec["nb"], spec["n"])
    return [_modes(shape, random.Random((seed * 1024 + i) * 8 + c), 4, 4).float() for c in range(spec["ncomp"])]


# ------------------------------------------------------------------ prepare / run


def prepare(case, seed):
    torch.cuda.current_device()  # torch touches the GPU before the library does
    kind = case["kind"]
    if kind == "batch":
        return _prepare_batch(case, seed)
    nb, n, T, nc = _three(case["nb"]), _three(case["n"]), case["dtype"], case["ncomp"]
    st = {"kind": kind, "case": case}
    if kind in ("step", "run"):
        st["u"] = Out(nb, n, T, nc, _inputs(case, seed), case["bc"])
        st["v"] = Out(nb, n, T, nc, None, case["bc"])
        st["nudt"] = _nudt(nb, n)
        if kind == "step":
            st["lap"] = Out(nb, n, T, nc)
        count = 1 if kind == "step" else case["steps"]
        st["norms"] = torch.zeros(count, dtype=torch.float64, device=DEV)
        st["norms_ptr"] = ctypes.c_void_p(st["norms"].data_ptr())
    elif kind == "weno":
        st["u"] = Out(nb, n, T, nc, _inputs(case, seed), case["bc"])
        st["v"] = Out(nb, n, T, 6 * nc)
    elif kind in ("sweep", "solve"):
        shape = _shape(nb, n)
        src = _source(shape, seed)
        homog = [0.0] * 6
        if kind == "sweep":
            st["u"] = Out(nb, n, T, 1, [1e-3 * _scalar(shape, seed, 0)], case["bc"], homog)
            st["v"] = Out(nb, n, T, 1)
        else:
            st["u"] = Out(nb, n, T, 1, None, case["bc"], homog)
            st["work"] = Out(nb, n, "f32" if case["refine"] else T, 3 if case["refine"] else 2)
        st["f"] = Out(nb, n, T, 1, [src])
        cnv.set_zfaces(st["u"].g, _zfaces(shape[0]))
    elif kind == "labs":
        ent = case["entity"]
        t = _storage(1, nb, n, T, ent)
        t.copy_(_noise(t.shape, seed, 1.0))
        st["t"], st["g"] = t, _grid(t, nb, n, 1, ent)
        _walls(st["g"], case["bc"])
        st["stencil"] = cnv.Stencil(case["lo"], case["hi"], case["tensorial"])
        st["out"], st["bufs"] = [], []
        for s in range(t.shape[0]):
            p, _ = st["g"].lab_geometry(st["stencil"], s)
            st["out"].append(torch.zeros((nb[0] * nb[1] * nb[2], p[2], p[1], p[0]), dtype=_torch(T), device=DEV))
            st["bufs"].append(types.SimpleNamespace(ptr=ctypes.c_void_p(st["out"][-1].data_ptr())))
    else:  # fields
        ent = case["entity"]
        ts = [_storage(nc, nb, n, T, ent) for _ in range(4)]
        for i in (0, 1):
            ts[i].copy_(_noise(ts[i].shape, seed * 4 + i, 0.5) + 1.0)
        st["t"] = ts
        st["g"] = [_grid(t, nb, n, nc, ent) for t in ts]
        st["out"] = [t[:, :, :n[0] * n[1] * n[2]] if ent == "cell" else t for t in ts[2:]]
    return st


def _prepare_batch(case, seed):
    specs = _batch_specs(case)
    sizes = []
    for s in specs:
        cells = s["n"][0] ** 3 * s["nb"][0] * s["nb"][1] * s["nb"][2]
        sizes.append((cells * s["ncomp"], cells * s["ncomp"] * (6 if s["op"] == "weno5" else 1)))
    # one allocation for the inputs, one for the outputs (8^3 blocks need no padding)
    tin = torch.empty(sum(a for a, _ in sizes), dtype=torch.float32, device=DEV)
    tout = torch.zeros(sum(b for _, b in sizes), dtype=torch.float32, device=DEV)
    items, ia, ib = [], 0, 0
    for i, (s, (a, b)) in enumerate(zip(specs, sizes)):
        part = tin[ia:ia + a].view(s["ncomp"], -1)
        for c, v in enumerate(_batch_fields(s, seed, i)):
            part[c].copy_(_to_blocks(v, s["nb"], s["n"]).reshape(-1))
        gi = _grid(tin[ia:ia + a], s["nb"], s["n"], s["ncomp"])
        _walls(gi, s["bc"], s["wall"])
        go = _grid(tout[ib:ib + b], s["nb"], s["n"], s["ncomp"] * (6 if s["op"] == "weno5" else 1))
        items.append((gi, go, s["op"], s["ghost"], _nudt(s["nb"], s["n"])))
        ia, ib = ia + a, ib + b
    return {"kind": "batch", "items": items, "tin": tin, "out": tout, "batch": cnv.Batch(items)}


def run(st):
    kind = st["kind"]
    if kind == "step":
        cnv.diffusion_step(st["u"].g, st["v"].g, st["nudt"], lap=st["lap"].g, sumsq=st["norms_ptr"])
        return {"u": st["v"].cells, "lap": st["lap"].cells, "norm": st["norms"]}
    if kind == "run":
        c = st["case"]
        g = cnv.diffusion_run(st["u"].g, st["v"].g, c["steps"], st["nudt"], st["norms_ptr"] if c["norms"] else None)
        out = {"u": (st["u"] if g is st["u"].g else st["v"]).cells}
        if c["norms"]:
            out["norms"] = st["norms"]
        return out
    if kind == "weno":
        cnv.weno5(st["u"].g, st["v"].g)
        return st["v"].cells
    if kind == "sweep":
        cnv.jacobi_sweep2(st["u"].g, st["f"].g, st["v"].g, OMEGA)
        return st["v"].cells
    if kind == "solve":
        c = st["case"]
        cycles, sweeps, rel, hist = cnv.jacobi_solve(st["u"].g, st["f"].g, st["work"].g, c["refine"], c["sweeps"],
                                                     c["cycles"], OMEGA, 0.0)
        return {"u": st["u"].cells, "history": hist, "sweeps": sweeps}
    if kind == "batch":
        st["batch"].run()
        return st["out"]
    if kind == "labs":
        for s, buf in enumerate(st["bufs"]):
            st["g"].lab_all(st["stencil"], s, buf)
        return st["out"]
    u, v, w, x = st["g"]
    cnv.grid_field_op("mul", w, u, scalar=0.25)   # w = u / 4
    cnv.grid_field_op("add", w, w, v)             # w += v
    cnv.grid_field_op("div", x, w, u)             # x = w / u
    if st["case"]["entity"] != "cell":            # sums take cell grids
        return st["out"]
    return {"fields": st["out"], "sums": list(cnv.grid_sums(w)), "compare": list(cnv.grid_compare(w, v))}


# ------------------------------------------------------------------ work


def work(case):
    if case["kind"] == "batch":
        b = f = 0
        for s in _batch_specs(case):
            cells = s["ncomp"] * s["n"][0] ** 3 * s["nb"][0] * s["nb"][1] * s["nb"][2]
            b += cells * (28 if s["op"] == "weno5" else 8)
            f += cells * (180 if s["op"] == "weno5" else 15)
        return {"bytes": b, "flops": f}
    nb, n, nc, sz = _three(case["nb"]), _three(case["n"]), case["ncomp"], _size(case["dtype"])
    cells = nc * nb[0] * nb[1] * nb[2] * n[0] * n[1] * n[2]
    kind = case["kind"]
    if kind == "step":
        return {"bytes": 3 * sz * cells, "flops": 17 * cells}
    if kind == "run":  # the field in, the field out, whatever the number of steps
        return {"bytes": 2 * sz * cells, "flops": (17 if case["norms"] else 15) * cells * case["steps"]}
    if kind == "weno":
        return {"bytes": 7 * sz * cells, "flops": 180 * cells}
    if kind == "sweep":
        return {"bytes": 3 * sz * cells, "flops": 2 * 18 * cells}
    if kind == "solve":  # u in and out, f
        return {"bytes": 3 * sz * cells, "flops": 18 * cells * case["cycles"] * (case["sweeps"] + 1)}
    if kind == "labs":
        w = case["hi"] - 1 - case["lo"]
        lab = nb[0] * nb[1] * nb[2] * (n[0] + w) * (n[1] + w) * (n[2] + w)
        k = 3 if case["entity"] == "face" else 1
        return {"bytes": k * sz * (cells + lab), "flops": 0}
    k = 3 if case["entity"] == "face" else 1
    return {"bytes": 4 * k * sz * cells, "flops": 3 * k * cells}


# ------------------------------------------------------------------ exact


def _pad(u, axis, lo, hi, w, wall):
    """u with w ghost layers on both ends of an axis of a (Z, Y, X) field."""
    m = u.shape[axis]
    if lo == "P":
        i = torch.arange(-w, m + w, device=u.device) % m
        return u.index_select(axis, i)
    ends = []
    for side, letter in ((0, lo), (1, hi)):
        near = list(range(w)) if side == 0 else list(range(m - 1, m - 1 - w, -1))  # mirror of layer 1, 2, ...
        if letter == "A":
            near = [near[0]] * w
        if side == 0:
            near = near[::-1]
        e = u.index_select(axis, torch.tensor(near, device=u.device))
        ends.append(torch.full_like(e, wall[side]) if letter == "D" else -e if letter == "N" else e)
    return torch.cat((ends[0], u, ends[1]), axis)


def _shifted(u, axis, bc, w, wall):
    """The fields u[i - w] ... u[i + w] along an axis (0 = x)."""
    a = 2 - axis
    p = _pad(u, a, bc[2 * axis], bc[2 * axis + 1], w, wall[2 * axis:2 * axis + 2])
    return [p.narrow(a, k, u.shape[a]) for k in range(2 * w + 1)]


def _laplacian(u, bc, wall):
    out = 0.0
    for d in range(3):
        m, _, p = _shifted(u, d, bc, 1, wall)
        out = out + (p - 2.0 * u + m) * float(u.shape[2 - d]) ** 2
    return out


def _weno_states(u, bc, wall):
    out = []
    for d in range(3):
        a, b, c, e, f = _shifted(u, d, bc, 2, wall)
        m2 = (a * a + b * b + c * c + e * e + f * f) / 5.0 + 1e-30
        b0 = 13.0 / 12.0 * (a - 2 * b + c) ** 2 + 0.25 * (a - 4 * b + 3 * c) ** 2
        b1 = 13.0 / 12.0 * (b - 2 * c + e) ** 2 + 0.25 * (b - e) ** 2
        b2 = 13.0 / 12.0 * (c - 2 * e + f) ** 2 + 0.25 * (3 * c - 4 * e + f) ** 2
        al = [1.0 / (1e-6 + x / m2) ** 2 for x in (b0, b1, b2)]
        for lin, q in (((0.1, 0.6, 0.3), ((2 * a - 7 * b + 11 * c), (-b + 5 * c + 2 * e), (2 * c + 5 * e - f))),
                       ((0.3, 0.6, 0.1), ((-a + 5 * b + 2 * c), (2 * b + 5 * c - e), (11 * c - 7 * e + 2 * f)))):
            wt = [g * x for g, x in zip(lin, al)]
            out.append((wt[0] * q[0] + wt[1] * q[1] + wt[2] * q[2]) / (6.0 * (wt[0] + wt[1] + wt[2])))
    return out


def _metric(m):
    zf = torch.from_numpy(_zfaces(m)).to(DEV)
    dz, zc = zf[1:] - zf[:-1], 0.5 * (zf[1:] + zf[:-1])
    zg = torch.cat((2 * zf[:1] - zc[:1], zc, 2 * zf[-1:] - zc[-1:]))
    return [(1.0 / (dz * v))[:, None, None] for v in (zg[1:-1] - zg[:-2], zg[2:] - zg[1:-1])]


def _poisson(u, bc):
    wall = [0.0] * 6
    cm, cp = _metric(u.shape[0])
    out = 0.0
    for d in range(2):
        m, _, p = _shifted(u, d, bc, 1, wall)
        out = out + (p - 2.0 * u + m) * float(u.shape[2 - d]) ** 2
    m, _, p = _shifted(u, 2, bc, 1, wall)
    diag = -(2.0 * float(u.shape[2]) ** 2 + 2.0 * float(u.shape[1]) ** 2 + cm + cp)
    return out + cp * (p - u) - cm * (u - m), diag


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        parts = []
        for i, s in enumerate(_batch_specs(case)):
            for v in _batch_fields(s, seed, i):
                v = v.double()
                res = (_weno_states(v, s["bc"], s["wall"]) if s["op"] == "weno5" else
                       [v + _nudt(s["nb"], s["n"]) * _laplacian(v, s["bc"], s["wall"])])
                parts += [_to_blocks(x, s["nb"], s["n"]).reshape(-1) for x in res]
        return torch.cat(parts)
    nb, n = _three(case["nb"]), _three(case["n"])
    if kind == "labs" or (kind == "fields" and case["entity"] != "cell"):
        return None  # copies, and one rounding per element over padded blocks
    blocks = lambda fields: torch.stack([_to_blocks(x, nb, n) for x in fields])  # noqa: E731
    if kind in ("step", "run"):
        us = [u.double() for u in _inputs(case, seed)]
        nudt, norms, laps = _nudt(nb, n), [], None
        for _ in range(1 if kind == "step" else case["steps"]):
            laps = [_laplacian(u, case["bc"], WALL) for u in us]
            us = [u + nudt * x for u, x in zip(us, laps)]
            norms.append(sum((u * u).sum() for u in us))
        norms = torch.stack(norms)
        if kind == "step":
            return {"u": blocks(us), "lap": blocks(laps), "norm": norms}
        return {"u": blocks(us), "norms": norms} if case["norms"] else {"u": blocks(us)}
    if kind == "weno":
        return torch.cat([blocks(_weno_states(u.double(), case["bc"], WALL)) for u in _inputs(case, seed)])
    if kind in ("sweep", "solve"):
        shape, T = _shape(nb, n), _torch(case["dtype"])
        f = _source(shape, seed).to(T).double()
        if kind == "sweep":
            u = (1e-3 * _scalar(shape, seed, 0)).to(T).double()
            count, per = 2, 2
        else:
            u = torch.zeros(shape, dtype=torch.float64, device=DEV)
            count, per = case["cycles"] * case["sweeps"], case["sweeps"]
        hist = []
        for k in range(count):
            au, diag = _poisson(u, case["bc"])
            if k % per == 0:
                hist.append((f - au).square().sum())
            u = u + (f - au) * (OMEGA / diag)
        if kind == "sweep":
            return blocks([u])
        hist.append((f - _poisson(u, case["bc"])[0]).square().sum())
        hist = (torch.stack(hist) / f.square().sum()).sqrt().cpu().numpy()
        return {"u": blocks([u]), "history": hist, "sweeps": None}
    st = [(_noise((case["ncomp"], nb[0] * nb[1] * nb[2], _stride(n, case["dtype"])), seed * 4 + i, 0.5) + 1.0)
          .to(_torch(case["dtype"])).double()[:, :, :n[0] * n[1] * n[2]] for i in (0, 1)]
    w = 0.25 * st[0] + st[1]
    d = w[0] - st[1][0]
    return {"fields": [w, w / st[0]], "sums": [float(w[0].sum()), float(w[0].square().sum())],
            "compare": [float(d.square().sum()), float(st[1][0].square().sum()), float(d.abs().max())]}
