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
