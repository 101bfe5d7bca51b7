"""A new context whose first calls run on a stream of the caller's own while
the default stream is busy: the context's scratch is cleared in order with the
work that uses it, so the results are those of a quiet device."""
import numpy as np
import pytest
import torch

from gpu_helpers import bits_equal, describe_diff, to_dev, to_host

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mp():
    from advectionhpctester_amd import mpdata
    return mpdata


def _case(dims, seed):
    from advectionhpctester_amd.testdata import random_case
    return {k: to_dev(v) for k, v in random_case(*dims, seed=seed, cmax=0.25).items()}


def _keep_default_stream_busy(products):
    """Some milliseconds of work on the default stream, queued and not waited
    for."""
    a = torch.ones(4096, 4096, device="cuda:0")
    for _ in range(products):
        a = torch.mm(a, a) * 1e-4
    return a


@pytest.mark.parametrize("variant", ["gauge", "standard"])
def test_first_time_loop_on_a_side_stream(mp, variant):
    """The loop's second field is allocated by its first call.  Several new
    contexts, with the default stream's work ending while they step."""
    dims, nt = (96, 64, 24, 1), 200
    t = _case(dims, 5)
    f = [t[k] for k in ("u1", "u2", "u3", "rhr", "h", "bcx", "bcy")]
    kw = dict(variant=mp.GAUGE if variant == "gauge" else mp.STANDARD)
    want = t["x"].clone()
    with mp.Domain(*dims) as d:
        d.timeloop(nt, want, *f, **kw)
    want = to_host(want)
    for q in range(6):
        x = t["x"].clone()
        torch.cuda.synchronize()
        side = torch.cuda.Stream()
        print(f"first loop on a side stream {variant} {q}", flush=True)
        busy = _keep_default_stream_busy(1 + q)
        with mp.Domain(*dims) as d:
            with torch.cuda.stream(side):
                d.timeloop(nt, x, *f, **kw)
            side.synchronize()
            torch.cuda.synchronize()
        del busy
        got = to_host(x)
        assert bits_equal(got, want), describe_diff(got, want)


@pytest.mark.parametrize("variant", ["gauge", "standard"])
def test_tape_recorded_on_a_side_stream(mp, variant):
    """Slots reserved while the default stream is busy, recorded on another
    stream, read after the default stream has drained."""
    dims = (40, 30, 20, 1)
    t = _case(dims, 7)
    f = [t[k] for k in ("u1", "u2", "u3", "rhr", "h")]
    v = mp.GAUGE if variant == "gauge" else mp.STANDARD
    seed = torch.ones_like(t["x"])
    res = []
    for quiet in (True, False):
        out = torch.zeros_like(t["x"])
        xbar = torch.zeros_like(t["x"])
        mp.interior(xbar).copy_(mp.interior(seed))
        ub = [torch.zeros_like(t[k]) for k in ("u1", "u2", "u3")]
        torch.cuda.synchronize()
        side = torch.cuda.Stream()
        print(f"tape on a side stream {variant} quiet={quiet}", flush=True)
        busy = None if quiet else _keep_default_stream_busy(8)
        with mp.Domain(*dims) as d:
            d.adj_reserve(1)
            with torch.cuda.stream(side):
                d.adj_record(0, t["x"], out, *f, t["bcx"], t["bcy"], variant=v)
            side.synchronize()
            torch.cuda.synchronize()
            with torch.cuda.stream(side):
                d.adj_step(0, *f, xbar, *ub)
            side.synchronize()
            torch.cuda.synchronize()
        del busy
        res.append([to_host(a) for a in (xbar, *ub)])
    # the reverse kernels add with atomics, in any order: sums of a dozen
    # terms of one magnitude, far below 1e-12 of the largest
    for a, b in zip(*res):
        assert np.abs(b).max() > 0
        assert float(np.abs(a - b).max()) <= 1e-12 * float(np.abs(b).max()), describe_diff(a, b)


def test_first_density_call_on_a_side_stream(mp):
    """The velocities of the whole density step are predicted into arrays that
    its first call allocates."""
    from advectionhpctester_amd.testdata import density_case
    dims = (48, 40, 24, 1)
    f = density_case(*dims, seed=3, cmax=0.5, dtype=np.float64)
    names = ("ox", "oy", "oz", "u", "v", "w", "u1", "u2", "u3", "x_in", "x_incomp", "h", "rhoadv",
             "rhr", "pexe", "pexr1", "pexr2", "bcx", "bcy")
    res = []
    for q in range(5):  # the first on a quiet default stream
        g = {k: to_dev(f[k]) for k in names}
        pol = dict(nsubsteps=1, nsubsteps_o=1, dtn=f["dt"], dtnold=f["dt"])
        torch.cuda.synchronize()
        side = torch.cuda.Stream()
        print(f"first density call on a side stream {q}", flush=True)
        busy = _keep_default_stream_busy(q) if q else None
        with mp.Domain(*dims) as d:
            with torch.cuda.stream(side):
                for _ in range(20):
                    d.rho_gauge_gpubc(pol, *[g[k] for k in names], f["dxi"], f["dyi"], f["dzi"],
                                      f["dt"])
            side.synchronize()
            torch.cuda.synchronize()
        del busy
        res.append({k: to_host(g[k]) for k in names})
    for r in res[1:]:
        for k in names:
            assert bits_equal(r[k], res[0][k]), k + ": " + describe_diff(r[k], res[0][k])


def test_first_call_under_capture(mp):
    """A context's first call captured into a graph (relaxed mode, which lets
    it allocate): the scratch is cleared outside the graph, and every replay
    gives the eager result."""
    dims = (48, 40, 16, 1)
    t = _case(dims, 9)
    f = [t[k] for k in ("u1", "u2", "u3", "rhr", "h", "bcx", "bcy")]
    want = t["x"].clone()
    with mp.Domain(*dims) as d:
        d.timeloop(3, want, *f)
    want = to_host(want)
    with mp.Domain(*dims) as d:
        x = t["x"].clone()
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        print("first call under capture", flush=True)
        with torch.cuda.graph(g, capture_error_mode="relaxed"):
            d.timeloop(3, x, *f)
        for _ in range(3):
            x.copy_(t["x"])
            torch.cuda.synchronize()
            g.replay()
            got = to_host(x)
            assert bits_equal(got, want), describe_diff(got, want)
            other = t["x"] * 2.0  # eager work between the replays
            d.timeloop(2, other, *f)
            torch.cuda.synchronize()
        del g
