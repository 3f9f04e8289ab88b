"""Emission, gather and split at the edges of their work units (needs a GPU).

The emission works on 64 active cells at a time wherever they lie, the gather on 64 touched vertices
of a few segments, the split on 64 quads: fields and sizes at which a unit is one cell short or over,
spans more segments than a wave can look at at once, holds more edge vertices than are kept, or
straddles the grids of a batch. Faces and vertices must be bit-identical to the oracle; gradients are
compared as in test_gpu_parity.py (the same terms, at most six per vertex, in another order).
"""
import numpy as np
import pytest
import torch

import diso_amd
from oracle import oracle as O
from tests.helpers import grad_close

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TOL = {np.float32: 2e-5, np.float64: 1e-12}
TDT = {np.float32: torch.float32, np.float64: torch.float64}


def _field(kind, rng):
    if kind == "sparse":  # eight cells every eight planes: a unit's cells lie hundreds of segments apart
        f = 0.5 + rng.random((70, 9, 67))
        f[3::8, 4, 5::61] *= -1
        return f
    if kind == "checker":  # every edge crosses: 512 edge vertices in a unit
        i, j, k = np.ogrid[:6, :7, :71]
        return np.where((i + j + k) % 2, 1, -1) * (0.5 + rng.random((6, 7, 71)))
    if kind == "wall":  # a surface along z: every vertex of whole segments is touched
        return (np.arange(9)[:, None, None] - 4.3) + 0.2 * rng.random((9, 20, 190))
    n = int(kind)  # columns of alternating signs: 9 (n + 1) or so cells, around multiples of 64
    f = np.ones((2, 2, n + 2)) * (0.5 + rng.random((2, 2, n + 2)))
    f[:, :, 1:-1:2] *= -1
    return f


@pytest.mark.parametrize("algo", [O.MC, O.DMC])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("recompute", [False, True])
@pytest.mark.parametrize("kind", ["sparse", "checker", "wall", "1", "6", "7", "8", "60", "62", "64"])
def test_units_match_oracle(algo, dtype, recompute, kind):
    print(f"case algo={algo} dtype={np.dtype(dtype).name} recompute={recompute} kind={kind}", flush=True)
    rng = np.random.default_rng(11)
    sdf_np = _field(kind, rng).astype(dtype)
    def_np = (rng.random((*sdf_np.shape, 3)) * 0.6 - 0.3).astype(dtype)
    ref = O.Extractor(algo, dtype)
    rv, rf = ref.forward(sdf_np, def_np, 0.0, True, return_quads=True)
    assert not ref.empty
    sdf = torch.tensor(sdf_np, device=DEV, requires_grad=True)
    deform = torch.tensor(def_np, device=DEV, requires_grad=True)
    mod = (diso_amd.DiffMC if algo == O.MC else diso_amd.DiffDMC)(TDT[dtype], recompute_backward=recompute)
    kw = {"return_quads": True} if algo == O.DMC else {}
    verts, faces = mod(sdf, deform, 0.0, **kw)
    assert np.array_equal(faces.cpu().numpy(), rf)
    assert np.array_equal(verts.detach().cpu().numpy(), rv)
    up = rng.standard_normal(rv.shape).astype(dtype)
    verts.backward(torch.tensor(up, device=DEV))
    gs, gd = ref.backward(up)
    grad_close(sdf.grad.cpu().numpy(), gs, TOL[dtype])
    grad_close(deform.grad.cpu().numpy(), gd, TOL[dtype])


def test_batch_units_that_straddle_grids():
    """Grids of a few cells each share units with their neighbours: the same bits as one by one."""
    rng = np.random.default_rng(5)
    dims = [(2, 2, 2), (1, 2, 3), (3, 5, 4), (2, 2, 70), (5, 1, 2), (4, 4, 4), (2, 3, 2), (1, 1, 1), (6, 7, 66)]
    algos = [("mc", "dmc")[i % 3 == 1] for i in range(len(dims))]
    sdfs = [torch.tensor(rng.standard_normal(d).astype(np.float32), device=DEV, requires_grad=True) for d in dims]
    defs = [torch.tensor((rng.random((*d, 3)) * 0.6 - 0.3).astype(np.float32), device=DEV) for d in dims]
    outs = diso_amd.BatchExtractor(torch.float32)(sdfs, algos, defs, normalize=False, return_quads=True)
    torch.autograd.backward([v for v, _ in outs], [torch.ones_like(v) for v, _ in outs])
    for a, s, d, (v, f) in zip(algos, sdfs, defs, outs):
        one = s.detach().clone().requires_grad_()
        mod = diso_amd.DiffMC(torch.float32) if a == "mc" else diso_amd.DiffDMC(torch.float32)
        kw = {"return_quads": True} if a == "dmc" else {}
        w, g = mod(one, d, normalize=False, **kw)
        assert torch.equal(v, w) and torch.equal(f, g)
        if w.shape[0]:  # (an empty mesh has no gradient)
            w.backward(torch.ones_like(w))
            assert torch.equal(s.grad, one.grad)


@pytest.mark.parametrize("idx", [torch.int32, torch.int64])
@pytest.mark.parametrize("nq", [2, 63, 64, 65, 255, 257, 1025, 262_143])
def test_split_at_unit_edges(nq, idx):
    rng = np.random.default_rng(nq)
    verts = rng.standard_normal((50, 3)).astype(np.float32)
    quads = rng.integers(0, 50, (nq, 4))
    want, _, _ = O.split_quads(verts, quads)
    got = diso_amd.split_quads(torch.tensor(verts, device=DEV), torch.tensor(quads, dtype=idx, device=DEV))
    assert np.array_equal(got.cpu().numpy(), want)


@pytest.mark.parametrize("algo", [O.MC, O.DMC])
@pytest.mark.parametrize("n,units", [(20, (1, 512)), (36, (513, 1024)), (45, (1025, 4000))])
def test_units_cut_in_parts(algo, n, units):
    """White noise of which nearly every cell is active, at sizes whose units are cut in four, in two and
    not at all."""
    print(f"case parts algo={algo} n={n}", flush=True)
    rng = np.random.default_rng(13)
    sdf_np, def_np = rng.standard_normal((n, n, n)).astype(np.float32), (rng.random((n, n, n, 3)) * 0.6 - 0.3).astype(np.float32)
    ins = np.pad(sdf_np, 1, constant_values=1) >= 0
    cubes = [ins[i:n + 1 + i, j:n + 1 + j, k:n + 1 + k] for i in (0, 1) for j in (0, 1) for k in (0, 1)]
    active = int((np.any(cubes, 0) & ~np.all(cubes, 0)).sum())
    assert units[0] <= (active + 63) // 64 <= units[1]
    ref = O.Extractor(algo, np.float32)
    rv, rf = ref.forward(sdf_np, def_np, 0.0, True, return_quads=True)
    mod = (diso_amd.DiffMC if algo == O.MC else diso_amd.DiffDMC)()
    kw = {"return_quads": True} if algo == O.DMC else {}
    for _ in range(2):  # without and with a size estimate: exact and larger capacities
        v, f = mod(torch.tensor(sdf_np, device=DEV), torch.tensor(def_np, device=DEV), 0.0, **kw)
        assert np.array_equal(f.cpu().numpy(), rf) and np.array_equal(v.cpu().numpy(), rv)
