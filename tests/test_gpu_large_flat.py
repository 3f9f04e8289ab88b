"""Grids of very many segments (needs a GPU): a flat grid has one 64-position segment per row, so a
gigabyte of samples is a quarter of a billion segments. A mesh in its far corner must be the mesh of the
corner alone."""
import pytest
import torch

import diso_amd

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _corner(n0, n1, dtype=torch.float32):
    g = torch.Generator(device=DEV).manual_seed(3)
    f = torch.rand((n0, n1, 1), generator=g, device=DEV, dtype=dtype) - 0.4
    f[0], f[:, 0] = 1, 1  # no edge to the rest of the grid crosses
    return f


@pytest.mark.parametrize("algo", ["mc", "dmc"])
def test_a_quarter_of_a_billion_segments(algo):
    """Above 239 million segments the gather's single-wave blocks no longer fit one grid dimension."""
    n, c = 15500, 40
    free, _ = torch.cuda.mem_get_info()
    if free < (60 << 30):
        pytest.skip("needs 60 GiB of device memory")
    print(f"case flat {algo} {n}", flush=True)
    make = diso_amd.DiffMC if algo == "mc" else diso_amd.DiffDMC
    kw = {"normalize": False} if algo == "mc" else {"normalize": False, "return_quads": True}
    corner = _corner(c, c).requires_grad_()
    w, x = make()(corner, **kw)
    up = torch.randn_like(w)
    w.backward(up)
    sdf = torch.ones((n, n, 1), device=DEV)
    sdf[n - c:, n - c:] = corner.detach()
    sdf.requires_grad_()
    assert (n + 2) ** 2 > 239_000_000
    v, f = make()(sdf, **kw)
    assert torch.equal(f, x)
    shift = torch.tensor([n - c, n - c, 0], device=DEV)
    # (positions near n carry less of the fraction than near 0)
    assert (v - shift - w).abs().max() <= 2 * torch.finfo(torch.float32).eps * n
    v.backward(up)
    assert torch.equal(sdf.grad[n - c:, n - c:], corner.grad)
    assert not sdf.grad[: n - c].any() and not sdf.grad[n - c:, : n - c].any()
    del sdf, v, f
    torch.cuda.empty_cache()


@pytest.mark.parametrize("algo", ["mc", "dmc"])
def test_more_segments_per_count_block_than_lds_holds(algo):
    """With one count block per CU, 1.7 million segments are 6,600 a block, whose counts pass through
    device memory; with four they stay in LDS. Recount spins 0: predecessors are counted again."""
    from diso_amd import _lib, autotune

    print(f"case flat count {algo}", flush=True)
    L = _lib.lib()
    before, spins = autotune.current(), L.diso_get_param(_lib.PARAM_RECOUNT_SPINS)
    make = diso_amd.DiffMC if algo == "mc" else diso_amd.DiffDMC
    kw = {} if algo == "mc" else {"return_quads": True}
    sdf = torch.randn((1300, 1300, 3), generator=torch.Generator(device=DEV).manual_seed(4), device=DEV)
    outs = []
    try:
        for per_cu, rs in ((4, spins), (1, spins), (1, 0)):
            autotune.apply({"count_blocks_per_cu": per_cu})
            assert L.diso_set_param(_lib.PARAM_RECOUNT_SPINS, rs) == 0
            outs.append(make()(sdf, **kw))
        torch.cuda.synchronize()
    finally:
        autotune.apply(before)
        L.diso_set_param(_lib.PARAM_RECOUNT_SPINS, spins)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert 1302 * 1302 / cus > 6144
    assert outs[0][0].shape[0] > 1_000_000
    for v, f in outs[1:]:
        assert torch.equal(v, outs[0][0]) and torch.equal(f, outs[0][1])
