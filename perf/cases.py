"""Timed cases: the extractions a user of diso_amd runs, through its public entry points.

A case is one call as a program makes it: a module forward (mesh export), a forward and backward
(one step of an optimisation through the surface), a batch of grids, or a step with outputs of
fixed capacity. `path` names the entry point:

    mc        DiffMC(sdf, deform)                            -> vertices, triangles
    dmc       DiffDMC(sdf, deform, return_quads=True)        -> vertices, quads
    dmc_tri   DiffDMC(sdf, deform), the default              -> vertices, triangles
    fixed     FixedExtractor("dmc", ...)(sdf, deform)        -> vertices, quads, counts
    batch     BatchExtractor over MC and DMC grids in turn   -> (vertices, faces) per grid

`field` is the kind of sdf: smooth shapes (sphere, blobs) as a trained or analytic sdf has them,
noisy ones (box_noise, sphere_noise) as an sdf has them early in a fit, and white noise, the densest
surface a grid can hold. Sample points are linspace(-0.5, 0.5, n) per axis.
"""
import math

import torch
import torch.nn.functional as F

import diso_amd

_DTYPE = {"f32": torch.float32, "f64": torch.float64}


def _case(name, path, dims, field, **kw):
    c = {"name": name, "path": path, "X": dims[0], "Y": dims[1], "Z": dims[2], "field": field, "dtype": "f32",
         "deform": True, "backward": True, "normalize": True, "recompute": False, "iso": 0.0}
    c.update(kw)
    return c


def _batch(name, count, lo, hi, backward):
    return {"name": name, "path": "batch", "count": count, "lo": lo, "hi": hi, "dtype": "f32", "backward": backward}


def listed():
    return [
        # the smallest calls: one object of a coarse stage, bound by launches and the host
        _case("mc_sphere_64_forward", "mc", (64, 64, 64), "sphere", deform=False, backward=False),
        _case("dmc_blobs_33x28x41_step", "dmc_tri", (33, 28, 41), "blobs"),
        # the plain optimisation step at 256^3 on a noisy field, Marching Cubes and Dual Marching Cubes
        _case("mc_noisy_256_step", "mc", (256, 256, 256), "box_noise"),
        _case("dmc_noisy_256_step", "dmc", (256, 256, 256), "box_noise"),
        # the same step once the field is smooth, at odd sizes
        _case("mc_smooth_203x256x181_step", "mc", (203, 256, 181), "blobs", iso=0.03125),
        _case("dmc_smooth_160x131x193_step", "dmc_tri", (160, 131, 193), "blobs"),
        # exporting a mesh of a finished field at high resolution, in grid units
        _case("mc_smooth_384_export", "mc", (384, 384, 384), "blobs", deform=False, backward=False, normalize=False),
        # white noise: as many vertices as a grid can have
        _case("dmc_white_128x120x136_forward", "dmc_tri", (128, 120, 136), "noise", backward=False),
        # double precision, as gradient checks and geometry processing use it
        _case("mc_noisy_97x130x66_f64_step", "mc", (97, 130, 66), "box_noise", dtype="f64"),
        # a learnable 512^3 field: fixed capacities (no host synchronisation), classification recomputed
        _case("dmc_fixed_512_step", "fixed", (512, 512, 512), "sphere_noise", recompute=True),
        # uneven grids of mixed algorithm in one batch, forward and backward; and many small objects
        _batch("batch_uneven_16_step", 16, 32, 256, True),
        _batch("batch_small_32_forward", 32, 16, 64, False),
    ]


def draw(rng):
    log = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))  # noqa: E731
    kind = rng.choice(["mc", "mc", "dmc", "dmc", "dmc_tri", "dmc_tri", "fixed", "batch"])
    if kind == "batch":
        backward = rng.random() < 0.5
        hi = log(32, 224)
        return {k: v for k, v in _batch("", rng.randint(2, 16 if backward else 32), rng.randint(16, min(hi, 48)), hi,
                                        backward).items() if k != "name"}
    n = log(20, 400)
    dims = [max(8, int(n * rng.uniform(0.7, 1.25))) for _ in range(3)]
    field = rng.choice(["sphere", "blobs", "blobs", "box_noise", "box_noise", "sphere_noise", "noise"])
    dtype = "f64" if rng.random() < 0.2 and kind != "fixed" else "f32"
    most = 160 if field == "noise" else 300 if field == "box_noise" or dtype == "f64" else 450
    dims = [min(d, most) for d in dims]
    c = _case("", kind, dims, field, dtype=dtype, deform=rng.random() < 0.7, normalize=rng.random() < 0.8,
              backward=kind == "fixed" or rng.random() < 0.65, recompute=rng.random() < 0.25,
              iso=rng.choice([0.0, 0.0, 0.03125, -0.015625]))
    del c["name"]
    return c


# ---- inputs


def _grids(case):
    """The single grids of a batch: sizes from small to large, families and algorithms in turn."""
    n, lo, hi = case["count"], case["lo"], case["hi"]
    out = []
    for i in range(n):
        s = lo * (hi / lo) ** (i / max(1, n - 1))
        dims = (int(round(s)), max(8, int(s * 0.93)), int(round(s)) + (i % 3) - 1)
        c = _case("", ("mc", "dmc")[i % 2], dims, ("sphere", "blobs", "box_noise", "noise")[(i // 2) % 4],
                  backward=case["backward"])
        out.append(c)
    return out


def _device():
    return torch.device("cuda:0" if torch.cuda.is_available() else "cpu")


def _shape(case):
    """The case's shape, the same for every seed (so its outputs keep their sizes): sdf in float64."""
    dev, dims = _device(), (case["X"], case["Y"], case["Z"])
    g = torch.Generator(device=dev).manual_seed(1)
    gc = torch.Generator().manual_seed(2)

    def u(lo, hi, *shape):
        return (torch.rand(*shape, generator=gc, dtype=torch.float64) * (hi - lo) + lo).tolist()

    a = [torch.linspace(-0.5, 0.5, n, dtype=torch.float64, device=dev).view([-1 if i == k else 1 for i in range(3)])
         for k, n in enumerate(dims)]

    def d2(c):
        return (a[0] - c[0]) ** 2 + (a[1] - c[1]) ** 2 + (a[2] - c[2]) ** 2

    def noise(amp):
        return (torch.rand(dims, generator=g, device=dev, dtype=torch.float32) * 2 - 1) * amp

    kind = case["field"]
    if kind == "sphere":
        return d2((0.01, -0.02, 0.03)).sqrt() - 0.4
    if kind == "sphere_noise":
        return d2((0.0, 0.0, 0.0)).sqrt() - 0.4 + 0.01 * torch.randn(dims, generator=g, device=dev, dtype=torch.float32)
    if kind == "blobs":
        # eight Gaussian blobs, centres in [-0.3, 0.3]^3, sigma in [0.05, 0.15], minus one half
        f = torch.full(dims, -0.5, dtype=torch.float64, device=dev)
        for c, s in zip(u(-0.3, 0.3, 8, 3), u(0.05, 0.15, 8)):
            ex, ey, ez = (torch.exp(-((a[k] - c[k]) ** 2) / (2 * s * s)) for k in range(3))
            f += ex * ey * ez
        return f
    if kind == "box_noise":
        # a rounded box (half extent 0.35, radius 0.1) plus U(-0.05, 0.05)
        q = [x.abs() - 0.35 + 0.1 for x in a]
        f = sum(x.clamp_min(0) ** 2 for x in q).sqrt() - 0.1
        f += torch.maximum(torch.maximum(q[0], q[1]), q[2]).clamp_max(0)
        return f + noise(0.05)
    return noise(1.0).double()


def _field(case, seed):
    """(sdf, deform or None) of a case: the shape, mirrored along axes that the seed chooses, its
    distances to the isovalue stretched by the seed (smoothly where the field is smooth, sample by
    sample where it is noisy), and a deform of the seed's."""
    f, iso, dt = _shape(case), case["iso"], _DTYPE[case["dtype"]]
    dev, dims = f.device, f.shape
    g = torch.Generator(device=dev).manual_seed(seed)
    gc = torch.Generator().manual_seed(seed + 1)
    flips = [k for k in range(3) if float(torch.rand(1, generator=gc)) < 0.5]
    base = torch.flip(f, flips).to(dt)
    if case["field"] in ("sphere", "blobs"):
        stretch = 1.0
        for k, n in enumerate(dims):
            w, p = (torch.rand(2, generator=gc, dtype=torch.float64) * 6.28).tolist()
            x = torch.linspace(p, p + w, n, dtype=torch.float64, device=dev)
            stretch = stretch * (1.0 + 0.2 * torch.cos(x)).view([-1 if i == k else 1 for i in range(3)])
    else:
        stretch = 0.75 + 0.5 * torch.rand(dims, generator=g, device=dev, dtype=torch.float32)
    sdf = (iso + (base.double() - iso) * stretch).to(dt)
    sdf = torch.where((sdf >= iso) == (base >= iso), sdf, base).contiguous()
    deform = None
    if case["deform"]:
        amp = 0.1 if case["field"] == "sphere_noise" else 0.3
        deform = ((torch.rand((*dims, 3), generator=g, device=dev, dtype=torch.float32) * 2 - 1) * amp).to(dt)
    return sdf, deform


def _crossings(sdf, iso):
    """Grid edges that cross the surface, on the grid padded by one ring of inside samples."""
    p = F.pad((sdf >= iso).unsqueeze(0), (1,) * 6, value=True)[0]
    return sum(int((p.narrow(k, 1, p.shape[k] - 1) ^ p.narrow(k, 0, p.shape[k] - 1)).sum()) for k in range(3))


def _one(case, seed):
    sdf, deform = _field(case, seed)
    st = {"case": case, "sdf": sdf, "deform": deform, "iso": case["iso"]}
    if case["backward"]:
        # the loss's gradient at the vertices: a row for each the surface can have (a Marching Cubes
        # vertex is a crossing edge, a Dual Marching Cubes one has at least three of a cell's)
        edges = _crossings(sdf, case["iso"])
        rows = edges if case["path"] == "mc" else 4 * edges // 3 + 1
        g = torch.Generator(device=sdf.device).manual_seed(seed + 2)
        st["up"] = torch.randn((rows, 3), generator=g, device=sdf.device, dtype=torch.float32).to(sdf.dtype)
        st["edges"] = edges
        sdf.requires_grad_()
        if deform is not None:
            deform.requires_grad_()
    return st


def prepare(case, seed):
    if case["path"] == "batch":
        one = [_one(c, 1000 * seed + 10 * i) for i, c in enumerate(_grids(case))]
        return {"case": case, "grids": one, "ex": diso_amd.BatchExtractor(_DTYPE[case["dtype"]])}
    st = _one(case, seed)
    dt = _DTYPE[case["dtype"]]
    if case["path"] == "mc":
        st["ex"] = diso_amd.DiffMC(dt, recompute_backward=case["recompute"])
    elif case["path"] == "fixed":
        st["ex"] = diso_amd.FixedExtractor("dmc", dt, st["up"].shape[0], st["edges"] + 1,
                                           recompute_backward=case["recompute"])
    else:
        st["ex"] = diso_amd.DiffDMC(dt, recompute_backward=case["recompute"])
    return st


# ---- one pass


def _run_batch(st):
    case, grids = st["case"], st["grids"]
    for g in grids:
        g["sdf"].grad = None
        g["deform"].grad = None
    with torch.set_grad_enabled(case["backward"]):
        outs = st["ex"]([g["sdf"] for g in grids], [g["case"]["path"] for g in grids], [g["deform"] for g in grids],
                        return_quads=True)
    if not case["backward"]:
        return outs
    verts = [v for v, _ in outs]
    torch.autograd.backward(verts, [g["up"][:v.shape[0]] for g, v in zip(grids, verts)])
    return [(v, f, g["sdf"].grad, g["deform"].grad) for (v, f), g in zip(outs, grids)]


def run(state):
    case = state["case"]
    if case["path"] == "batch":
        return _run_batch(state)
    sdf, deform = state["sdf"], state["deform"]
    kw = {"isovalue": case["iso"], "normalize": case["normalize"]}
    if case["path"] == "dmc":
        kw["return_quads"] = True
    sdf.grad = None
    if deform is not None:
        deform.grad = None
    with torch.set_grad_enabled(case["backward"]):
        got = state["ex"](sdf, deform, **kw)
    out = {"verts": got[0], "faces": got[1]}
    if case["path"] == "fixed":  # rows past the quads are undefined
        out["faces"] = got[1][:state["edges"]]
        out["counts"] = got[2]
    if case["backward"]:
        got[0].backward(state["up"][:got[0].shape[0]])
        out["grad_sdf"] = sdf.grad
        if deform is not None:
            out["grad_deform"] = deform.grad
    return out


def _work_one(c):
    """Forward: the samples once, the deforms at the surface, the outputs. Backward: samples and
    deforms at the surface, the vertices' gradients, and the dense gradients."""
    sdf, _ = _field({**c, "deform": False}, 0)
    iso, s, n = c["iso"], sdf.element_size(), sdf.numel()
    e = _crossings(sdf, iso)
    q = (sdf >= iso)
    t = torch.zeros_like(q)  # samples at the end of a crossing edge
    for k in range(3):
        m = q.narrow(k, 1, q.shape[k] - 1) ^ q.narrow(k, 0, q.shape[k] - 1)
        t.narrow(k, 1, q.shape[k] - 1).logical_or_(m)
        t.narrow(k, 0, q.shape[k] - 1).logical_or_(m)
    t = int(t.sum())
    # vertices: one per crossing edge (Dual: about as many); triangles: about two per vertex; quads: one per edge
    faces = 4 * e if c["path"] in ("dmc", "fixed") else 3 * 2 * e
    b = s * n + 3 * s * e + 8 * faces + (3 * s * t if c["deform"] else 0)
    f = 25 * e
    if c["backward"]:
        b += s * t + 3 * s * e + s * n + ((3 * s * t + 3 * s * n) if c["deform"] else 0)
        f += 40 * e
    return b, f


def work(case):
    each = [_work_one(c) for c in (_grids(case) if case["path"] == "batch" else [case])]
    return {"bytes": sum(b for b, _ in each), "flops": sum(f for _, f in each)}


def tolerance(case):
    # About four times the distance from 64 bits, measured. Vertices: 6e-8 (half an ulp of the grid's
    # size). Sample gradients scale with an edge's length, whose endpoints (integer coordinate plus
    # deform) are rounded at the coordinate's size: 1e-6 at 41 samples a side, 8e-6 at 256, 1.6e-5 at
    # 512. In float64: 3e-16.
    if case["dtype"] == "f64":
        return {"rel": 1.2e-15}
    if not case["backward"]:
        return {"rel": 2.5e-7}
    return {"rel": 1.25e-7 * (case["hi"] if case["path"] == "batch" else max(case["X"], case["Y"], case["Z"]))}


# ---- the same in 64 bits, from the definitions

_EDGE_AT = ((0, 0, 0), (1, 0, 0), (0, 0, 1), (0, 0, 0), (0, 1, 0), (1, 1, 0), (0, 1, 1), (0, 1, 0), (0, 0, 0), (1, 0, 0),
            (1, 0, 1), (0, 0, 1))
_EDGE_AXIS = (0, 2, 0, 2, 0, 2, 0, 2, 1, 1, 1, 1)
# cell configurations whose patches are not listed by their lowest edge, with their order by it
_PATCH_ORDER = {20: (1, 0), 22: (0, 2, 1), 24: (1, 0), 28: (1, 0), 36: (1, 0), 40: (1, 0), 41: (0, 2, 1),
                44: (1, 0), 52: (1, 0), 56: (1, 0), 60: (1, 0), 88: (1, 0), 100: (1, 0),
                104: (1, 0, 2), 105: (0, 2, 1, 3), 108: (1, 0), 120: (1, 0), 148: (1, 0, 2),
                150: (0, 2, 1, 3), 152: (1, 0), 156: (1, 0), 164: (1, 0), 180: (1, 0), 219: (1, 0),
                231: (1, 0)}


def _edge_corners(e):
    a = list(_EDGE_AT[e])
    b = list(a)
    b[_EDGE_AXIS[e]] += 1
    return a[0] + 2 * a[1] + 4 * a[2], b[0] + 2 * b[1] + 4 * b[2]


def _patches(code):
    """The surface patches of a dual cell (corner i at (i & 1, i >> 1 & 1, i >> 2)): crossing edges
    joined across each face, two by two; a face with four crossings joins those at each inside
    corner. Returns the patches (lists of edges) and the only ambiguous face of a configuration with
    more inside than outside corners (2 * axis + side), which its neighbour there may invert."""
    ends = [_edge_corners(e) for e in range(12)]
    cross = [e for e in range(12) if (code >> ends[e][0] & 1) != (code >> ends[e][1] & 1)]
    group = {e: {e} for e in cross}

    def join(a, b):
        m = group[a] | group[b]
        for e in m:
            group[e] = m

    four = []
    for face in range(6):
        axis, side = face >> 1, face & 1
        on = [e for e in cross if all((c >> axis & 1) == side for c in ends[e])]
        if len(on) == 2:
            join(*on)
        elif len(on) == 4:
            four.append(face)
            for c in range(8):
                if (c >> axis & 1) == side and code >> c & 1:
                    join(*[e for e in on if c in ends[e]])
    got = sorted({tuple(sorted(m)) for m in group.values()})
    got = [got[i] for i in _PATCH_ORDER.get(code, range(len(got)))]
    return got, four[0] if len(four) == 1 and bin(code).count("1") > 4 else -1


class _Exact:
    """Vertices of one grid in 64 bits, differentiable."""

    def __init__(self, c, sdf, deform):
        self.c, self.iso, self.shape = c, c["iso"], sdf.shape
        self.sdf = sdf.detach().double().requires_grad_(c["backward"])
        self.deform = None if deform is None else deform.detach().double().requires_grad_(c["backward"])
        self.grid = F.pad(self.sdf.unsqueeze(0), (1,) * 6, value=self.iso + 1.0)[0]
        self.inside = self.grid.detach() >= self.iso
        self.dims = self.grid.shape
        self.step = (self.dims[1] * self.dims[2], self.dims[2], 1)

    def edges(self):
        """Owner index and axis of each crossing edge, in order of owner and then axis."""
        i, m = self.inside, torch.zeros((*self.dims, 3), dtype=torch.bool, device=self.grid.device)
        for k in range(3):
            n = self.dims[k] - 1
            m.narrow(k, 0, n)[..., k] = i.narrow(k, 0, n) ^ i.narrow(k, 1, n)
        self.number = None
        at = m.view(-1).nonzero()[:, 0]
        if self.c["path"] != "mc":
            self.number = torch.full((m.numel(),), -1, dtype=torch.int32, device=at.device)
            self.number[at] = torch.arange(at.numel(), dtype=torch.int32, device=at.device)
        return at // 3, at % 3

    def points(self):
        own, axis = self.edges()
        one = own + torch.tensor(self.step, device=own.device)[axis]
        flat = self.grid.reshape(-1)
        d0, d1 = flat.index_select(0, own), flat.index_select(0, one)
        t = ((self.iso - d0) / (d1 - d0)).clamp(0, 1).unsqueeze(1)

        def at(i):
            x = torch.stack([i // self.step[0], i // self.step[1] % self.dims[1], i % self.dims[2]], 1)
            p = x.double()
            if self.deform is None:
                return p
            x = x - 1
            hi = torch.tensor(self.shape, device=i.device)
            ok = ((x >= 0) & (x < hi)).all(1)
            j = torch.where(ok, (x[:, 0] * hi[1] + x[:, 1]) * hi[2] + x[:, 2], 0)
            return p + self.deform.reshape(-1, 3).index_select(0, j) * ok.unsqueeze(1)

        p0 = at(own)
        return p0 + (at(one) - p0) * t

    def codes(self):
        """Configurations of the cells (corner (0, 0, 0) at each sample but the last of a row)."""
        i, n = self.inside, [d - 1 for d in self.dims]
        code = torch.zeros(n, dtype=torch.uint8, device=i.device)
        for k in range(8):
            at = (k & 1, k >> 1 & 1, k >> 2)
            w = i[at[0]:at[0] + n[0], at[1]:at[1] + n[1], at[2]:at[2] + n[2]]
            code |= w.to(torch.uint8) << k
        return code

    def means(self, table):
        pts, code = self.points(), self.codes()
        face = torch.tensor([f for _, f in table], device=code.device)[code.long()]
        odd = face >= 0
        flip = torch.zeros_like(odd)
        for f in range(6):  # inverted when the cell across the ambiguous face is ambiguous too
            axis, n = f >> 1, code.shape[f >> 1] - 1
            me, other = (odd.narrow(axis, *x) for x in (((0, n), (1, n)) if f & 1 else ((1, n), (0, n))))
            flip.narrow(axis, *((0, n) if f & 1 else (1, n))).logical_or_(
                (face == f).narrow(axis, *((0, n) if f & 1 else (1, n))) & me & other)
        del odd, face
        code = torch.where(flip, code ^ 255, code)
        cell = ((code != 0) & (code != 255)).nonzero()
        code = code[cell[:, 0], cell[:, 1], cell[:, 2]].long()
        cell = (cell * torch.tensor(self.step, device=cell.device)).sum(1)
        count = torch.tensor([len(p) for p, _ in table], device=code.device)
        member = torch.zeros((256, 4, 12), dtype=torch.bool)
        for c, (p, _) in enumerate(table):
            for k, es in enumerate(p):
                member[c, k, list(es)] = True
        member = member.to(code.device)
        n = count[code]
        row = torch.repeat_interleave(torch.arange(code.numel(), device=code.device), n)
        patch = torch.arange(row.numel(), device=code.device) - (torch.cumsum(n, 0) - n)[row]
        code, cell, total, size = code[row], cell[row], 0.0, 0.0
        for e in range(12):
            on = member[code, patch, e]
            own = cell + sum(o * s for o, s in zip(_EDGE_AT[e], self.step))
            i = torch.where(on, self.number[3 * own + _EDGE_AXIS[e]].long(), 0)
            total = total + pts.index_select(0, i) * on.unsqueeze(1)
            size = size + on.double()
        return total / size.unsqueeze(1)

    def outputs(self, up):
        v = self.points() if self.c["path"] == "mc" else self.means([_patches(k) for k in range(256)])
        v = v - 1.0
        if self.c["normalize"]:
            v = v / (torch.tensor(self.shape, dtype=torch.float64, device=v.device) - 1)
        out = [v.detach()]
        if self.c["backward"]:
            leaves = [self.sdf] + ([] if self.deform is None else [self.deform])
            out += torch.autograd.grad(v, leaves, up[:v.shape[0]].double())
        return out


def exact(case, seed):
    if case["path"] == "batch":
        out = []
        for g in prepare(case, seed)["grids"]:
            with torch.set_grad_enabled(case["backward"]):
                r = _Exact(g["case"], g["sdf"], g["deform"]).outputs(g.get("up"))
            out.append((r[0], None, *r[1:]))
        return out
    st = _one(case, seed)
    with torch.set_grad_enabled(case["backward"]):
        r = _Exact(case, st["sdf"], st["deform"]).outputs(st.get("up"))
    out = {"verts": r[0], "faces": None}
    if case["path"] == "fixed":
        full = torch.zeros((st["up"].shape[0], 3), dtype=torch.float64, device=r[0].device)
        full[:r[0].shape[0]] = r[0]
        out["verts"], out["counts"] = full, None
    if case["backward"]:
        out["grad_sdf"] = r[1]
        if st["deform"] is not None:
            out["grad_deform"] = r[2]
    return out
