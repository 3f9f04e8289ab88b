"""Values at the ends of the number line (needs a GPU): a NaN isovalue, NaN samples where nothing raises,
infinite samples, against the rules the reference's comparisons give."""
import numpy as np
import pytest
import torch

import diso_amd
from diso_amd import _lib
from tests.helpers import inputs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TDT = {np.float32: torch.float32, np.float64: torch.float64}
NAN = float("nan")


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("dims", [(9, 8, 7), (5, 6, 130)])
def test_nan_isovalue_extracts_nothing(dtype, dims):
    """No comparison with NaN holds, so no sample is on either side: an empty mesh, as with any isovalue
    that no sample crosses. Only a NaN sample is an error."""
    print(f"case nan iso {np.dtype(dtype).name} {dims}", flush=True)
    sdf_np, _ = inputs(dims, "noise", 1, dtype, False)
    sdf_np[1, 2, 3], sdf_np[2, 2, 3] = np.inf, -np.inf
    sdf = torch.tensor(sdf_np, device=DEV)
    bad = sdf.clone()
    bad[-1, -1, -1] = NAN
    for mod, k in ((diso_amd.DiffMC(TDT[dtype]), 3), (diso_amd.DiffDMC(TDT[dtype]), 4)):
        v, f = mod(sdf, isovalue=NAN)
        assert v.shape == (0, 3) and f.shape == (0, k)
        with pytest.raises(RuntimeError, match="NaN"):
            mod(bad, isovalue=NAN)
    ex = diso_amd.BatchExtractor(TDT[dtype])
    assert [v.shape[0] for v, _ in ex([sdf, sdf], ["mc", "dmc"], isovalue=NAN)] == [0, 0]
    with pytest.raises(RuntimeError, match="grid 1"):
        ex([sdf, bad], ["mc", "dmc"], isovalue=NAN)
    fx = diso_amd.FixedExtractor("mc", TDT[dtype], 10, 10)
    assert fx(sdf, isovalue=NAN)[2].tolist() == [0, 0, 0]
    assert fx(bad, isovalue=NAN)[2].tolist() == [0, 0, _lib.TOTAL_HAS_NAN]


def _edge_terms(sdf, up, iso):
    """The deform gradient of every crossing edge's two ends as src/cumc.cu:343-368,412-453 states it, in
    numpy, padded grid: (1 - t) up and t up, with t clamped as min(max(0, t), 1) is in C (NaN gives 1)."""
    dt = sdf.dtype
    p = np.pad(sdf, 1, constant_values=dt.type(iso) + dt.type(1))
    g = np.zeros((*p.shape, 3), np.float64)
    inside = p >= iso
    n = 0
    X, Y, Z = (d - 1 for d in p.shape)
    with np.errstate(all="ignore"):
        for x in range(X):
            for y in range(Y):
                for z in range(Z):
                    for a in range(3):
                        q = (x + (a == 0), y + (a == 1), z + (a == 2))
                        if inside[x, y, z] == inside[q]:
                            continue
                        d0, d1 = p[x, y, z], p[q]
                        t = (dt.type(iso) - d0) / (d1 - d0)
                        t = 0.0 if 0 > t else t
                        t = t if t < 1 else 1.0
                        g[x, y, z] += (1.0 - t) * up[n]
                        g[q] += t * up[n]
                        n += 1
    assert n == up.shape[0]
    return g[1:-1, 1:-1, 1:-1]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("recompute", [False, True])
@pytest.mark.parametrize("kind", ["inf", "huge", "tiny"])
def test_deform_gradients_of_extreme_samples(dtype, recompute, kind):
    """An edge's two ends share its vertex's gradient as 1 - t and t whatever the samples: infinite ones,
    and ones whose difference overflows or is denormal (its fp32 reciprocal then is zero or infinite, so t
    is only held to [0, 1] and to the ends' sum there, and compared where a plain division gives it)."""
    print(f"case extreme {kind} {np.dtype(dtype).name} recompute={recompute}", flush=True)
    rng = np.random.default_rng(8)
    sdf_np = rng.standard_normal((7, 6, 67))
    if kind == "inf":
        sdf_np[rng.random(sdf_np.shape) < 0.3] = np.inf
        sdf_np[rng.random(sdf_np.shape) < 0.3] = -np.inf
    else:
        scale = {("huge", np.float32): 1.5e38, ("huge", np.float64): 8e307, ("tiny", np.float32): 1e-39,
                 ("tiny", np.float64): 1e-309}[kind, dtype]
        sdf_np = np.clip(sdf_np, -2, 2) * scale  # (finite; differences of "huge" ones overflow)
    sdf_np = sdf_np.astype(dtype)
    sdf = torch.tensor(sdf_np, device=DEV)
    deform = torch.zeros((*sdf_np.shape, 3), dtype=TDT[dtype], device=DEV, requires_grad=True)
    v, _ = diso_amd.DiffMC(TDT[dtype], recompute_backward=recompute)(sdf, deform, normalize=False)
    up = rng.standard_normal(v.shape).astype(dtype)
    v.backward(torch.tensor(up, device=DEV))
    got = deform.grad.cpu().numpy()
    assert np.isfinite(got).all()
    want = _edge_terms(sdf_np, up.astype(np.float64), 0.0)
    # (at most six terms per vertex, each within an ulp or two of its weight)
    if kind == "inf" or dtype == np.float64:
        assert np.abs(got - want).max() <= (1e-5 if dtype == np.float32 else 1e-13) * np.abs(want).max()
    else:
        whole = np.abs(got.astype(np.float64)[1:-1, 1:-1, 1:-1]).max()
        assert whole <= 6 * np.abs(up).max()
    # with the pad's samples stored, every edge has both ends in the grid: together they take all of `up`
    ones = torch.tensor(np.ones_like(up), device=DEV)
    big = torch.full(tuple(n + 2 for n in sdf_np.shape), 1.0, dtype=TDT[dtype], device=DEV)
    big[1:-1, 1:-1, 1:-1] = sdf
    d2 = torch.zeros((*big.shape, 3), dtype=TDT[dtype], device=DEV, requires_grad=True)
    w, _ = diso_amd.DiffMC(TDT[dtype], recompute_backward=recompute)(big, d2, normalize=False)
    assert w.shape == v.shape
    w.backward(ones)
    total = d2.grad.double().sum((0, 1, 2)).cpu().numpy()
    assert np.abs(total - w.shape[0]).max() <= (1e-5 if dtype == np.float32 else 1e-12) * w.shape[0]


def _crossing_vertices(sdf, iso):
    """Marching Cubes vertices of a padded grid in linear order, x, y, z edges of each position in turn: an
    edge crosses where one end is >= iso and the other < iso, which no NaN is."""
    dt = sdf.dtype
    p = np.pad(sdf, 1, constant_values=dt.type(iso) + dt.type(1))
    out = []
    for x, y, z in np.ndindex(*(d - 1 for d in p.shape)):
        for a in range(3):
            d0, d1 = p[x, y, z], p[x + (a == 0), y + (a == 1), z + (a == 2)]
            if (d0 >= iso and d1 < iso) or (d0 < iso and d1 >= iso):
                v = np.array([x, y, z], dt)
                v[a] += ((v[a] + dt.type(1)) - v[a]) * ((dt.type(iso) - d0) / (d1 - d0))
                out.append(v - dt.type(1))
    return np.array(out, dt).reshape(-1, 3)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("share", [0.0, 0.03, 0.6])  # (0: one sample)
def test_nan_samples_where_nothing_raises(dtype, share):
    """FixedExtractor leaves the NaN flag to its caller. NaN samples are outside, edges that end in one do
    not cross; stored and recomputed classification agree, and a clean grid after it is extracted clean."""
    from oracle import oracle as O
    from tests.torch_counts import expected_counts

    print(f"case nan samples {np.dtype(dtype).name} {share}", flush=True)
    rng = np.random.default_rng(12)
    dims = (9, 8, 70)
    clean = rng.standard_normal(dims).astype(dtype)
    bad = clean.copy()
    bad[rng.random(dims) < share] = NAN
    bad[4, 4, 63] = NAN
    counts = expected_counts(torch.tensor(bad), {k: torch.tensor(t, dtype=torch.int64) for k, t in O.expand_tables().items()})
    want = _crossing_vertices(bad, 0.0)
    n = 4 * clean.size
    for algo in ("mc", "dmc"):
        outs = []
        for recompute in (False, True):
            fx = diso_amd.FixedExtractor(algo, TDT[dtype], 2 * n, 3 * n, recompute_backward=recompute)
            for k in range(3):  # bad, clean, bad: through one control block
                s = torch.tensor(clean if k == 1 else bad, device=DEV, requires_grad=True)
                v, f, c = fx(s, normalize=False)
                nv, nf, flags = c.tolist()
                v.backward(torch.ones_like(v))
                if k == 1:
                    assert not flags & _lib.TOTAL_HAS_NAN
                    mod = diso_amd.DiffMC(TDT[dtype]) if algo == "mc" else diso_amd.DiffDMC(TDT[dtype])
                    s2 = torch.tensor(clean, device=DEV, requires_grad=True)
                    w, g = mod(s2, normalize=False, **({} if algo == "mc" else {"return_quads": True}))
                    w.backward(torch.ones_like(w))
                    assert torch.equal(v[:nv], w) and torch.equal(f[:nf], g) and torch.equal(s.grad, s2.grad)
                    continue
                assert flags & _lib.TOTAL_HAS_NAN
                if algo == "mc":
                    assert nv == want.shape[0] and nf == counts[1]
                    assert np.array_equal(v[:nv].detach().cpu().numpy(), want)
                else:
                    assert nv == counts[2] and nf == want.shape[0] and torch.isfinite(v[:nv]).all()
                outs.append((v[:nv].detach(), f[:nf], s.grad))
        for o in outs[1:]:
            assert all(torch.equal(x, y) for x, y in zip(o, outs[0]))
            assert torch.isfinite(o[2]).all()
