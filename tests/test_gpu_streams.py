"""One module on several streams, and extractions from several host threads (needs a GPU). A forward
returns before its count kernel has ended, so what calls share must be ordered by more than the host."""
import threading
import time

import pytest
import torch

import diso_amd
import diso_amd._C  # noqa: F401
from diso_amd import _lib
from tests.helpers import check_against_oracle, inputs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _grids(n, dims, seed):
    return [torch.tensor(inputs(dims, "noise" if i % 2 else "noisy_box", seed + i, "float32", False)[0], device=DEV)
            for i in range(n)]


@pytest.mark.parametrize("spins", [0, None])
@pytest.mark.parametrize("algo", ["mc", "dmc"])
def test_one_module_on_alternating_streams(algo, spins):
    """Sequential calls from one thread, each on the other stream, none synchronised: each as alone.
    (With recount spins 0 a block that finds a predecessor's word missing counts that range itself.)"""
    print(f"case streams {algo} spins={spins}", flush=True)
    L = _lib.lib()
    before = L.diso_get_param(_lib.PARAM_RECOUNT_SPINS)
    make = diso_amd.DiffMC if algo == "mc" else diso_amd.DiffDMC
    kw = {} if algo == "mc" else {"return_quads": True}
    grids = _grids(4, (70, 61, 130), 40)
    want = [make()(g, **kw) for g in grids]
    for g, (v, f) in zip(grids[:2], want):
        check_against_oracle(algo, g.cpu().numpy(), None, v, f)
    mod, streams = make(), [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    got = []
    try:
        if spins is not None:
            _lib.check(L.diso_set_param(_lib.PARAM_RECOUNT_SPINS, spins), "spins")
        for k in range(60):
            with torch.cuda.stream(streams[k % 2]):
                got.append(mod(grids[k % 4], **kw))
        torch.cuda.synchronize()
    finally:
        L.diso_set_param(_lib.PARAM_RECOUNT_SPINS, before)
    for k, (v, f) in enumerate(got):
        assert torch.equal(v, want[k % 4][0]) and torch.equal(f, want[k % 4][1]), k


def test_extractions_from_several_threads():
    """Threads with a module of their own on one stream, and on one of their own each."""
    print("case threads", flush=True)
    grids = _grids(6, (40, 51, 70), 60)
    want = [diso_amd.DiffMC()(g) for g in grids]
    for own_stream in (False, True):
        torch.cuda.synchronize()
        got, errors = [None] * len(grids), []

        def work(i):
            try:
                mod = diso_amd.DiffMC()
                st = torch.cuda.Stream() if own_stream else torch.cuda.default_stream()
                with torch.cuda.stream(st):
                    for _ in range(20):
                        got[i] = mod(grids[i])
                    st.synchronize()
            except Exception as e:  # reported below
                errors.append(e)

        threads = [threading.Thread(target=work, args=(i,)) for i in range(len(grids))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not errors, errors
        for (v, f), (w, x) in zip(got, want):
            assert torch.equal(v, w) and torch.equal(f, x)


def test_a_long_wait_does_not_hold_a_core():
    """With some 300 ms of work ahead in the stream, the waiting thread's own time stays a fraction."""
    print("case long wait", flush=True)
    sdf = _grids(1, (30, 31, 32), 80)[0]
    mod = diso_amd.DiffMC()
    want = mod(sdf)  # (the next call has a size estimate)
    big = torch.ones(1 << 29, device=DEV)
    torch.cuda.synchronize()
    big.mul_(1.0)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(10):
        big.mul_(1.0)
    torch.cuda.synchronize()
    n = int(3.0 / (time.perf_counter() - t0)) + 1  # some 0.3 s of them
    for _ in range(n):
        big.mul_(1.0)
    w0, c0 = time.perf_counter(), time.thread_time()
    got = mod(sdf)
    wall, own = time.perf_counter() - w0, time.thread_time() - c0
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    assert wall > 0.1, "the work ahead was too short for this test"
    assert own < 0.3 * wall, (own, wall)


def test_forwards_take_written_totals(monkeypatch):
    """A module's first forward on a size has no estimate to emit with, and the binding classes never
    have one, but all wait for their totals as later forwards do: no copy, no stream synchronisation
    (which made them slower than before the count became two launches)."""
    print("case first forward", flush=True)
    sdf = _grids(1, (12, 13, 14), 90)[0]

    def refuse(*args):  # the pass that copies and synchronises
        raise AssertionError("diso_count called")

    monkeypatch.setattr(_lib.lib(), "diso_count", refuse)
    for algo, make, kw in (("mc", diso_amd.DiffMC, {}), ("dmc", diso_amd.DiffDMC, {"return_quads": True})):
        for recompute in (False, True):
            mod = make(recompute_backward=recompute)
            for _ in range(2):
                v, f = mod(sdf, **kw)
                check_against_oracle(algo, sdf.cpu().numpy(), None, v, f)
        empty = make()
        for _ in range(2):
            assert empty(torch.ones_like(sdf), **kw)[0].shape == (0, 3)
            assert empty(torch.ones((1, 1, 1), device=DEV), **kw)[0].shape == (0, 3)
    padded = torch.nn.functional.pad(sdf, (1,) * 6, value=1.0)
    for algo, cls in (("mc", diso_amd._C.CUMCFloat), ("dmc", diso_amd._C.CUDMCFloat)):
        v, f = cls().forward(padded, 0.0)
        w, g = (diso_amd.DiffMC()(sdf, normalize=False) if algo == "mc" else
                diso_amd.DiffDMC()(sdf, normalize=False, return_quads=True))
        assert torch.equal(v - 1, w) and torch.equal(f.long(), g)


@pytest.mark.parametrize("known", [False, True])
def test_a_capture_refuses_to_wait(known):
    """A module's forward waits for its totals, so it is refused while its stream is captured, at once and
    before anything is recorded; the module works on afterwards."""
    print(f"case capture known={known}", flush=True)
    sdf = _grids(1, (20, 21, 22), 95)[0]
    want = diso_amd.DiffDMC()(sdf, return_quads=True)
    mod = diso_amd.DiffDMC()
    if known:
        mod(sdf, return_quads=True)
    torch.cuda.synchronize()
    x = torch.ones(8, device=DEV)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        x.add_(1)
        with pytest.raises(RuntimeError, match="captured"):
            mod(sdf, return_quads=True)
    graph.replay()
    torch.cuda.synchronize()
    assert (x == 2).all()
    for stream in (torch.cuda.default_stream(), torch.cuda.Stream()):
        with torch.cuda.stream(stream):
            v, f = mod(sdf, return_quads=True)
            stream.synchronize()
        assert torch.equal(v, want[0]) and torch.equal(f, want[1])
