"""Every build of the fused kernels on both of its tilings (32x32 and 32x16
lanes), which the tiling rule picks between by size, and every mode of the
launch plan with more tiles than workgroups: whole tiles, then runs or chunks
of the tiles that remain."""
import numpy as np
import pytest
import torch

from gpu_helpers import bits_equal, describe_diff, interior, to_dev, to_host

pytestmark = pytest.mark.gpu

DTYPES = [(torch.float64, np.float64), (torch.float32, np.float32)]
KEYS = ("u1", "u2", "u3", "rhr", "h", "bcx", "bcy")
DIMS = (70, 45, 30, 1)
NSTEPS = 20


@pytest.fixture(scope="module")
def mp():
    from advectionhpctester_amd import mpdata
    return mpdata


@pytest.fixture(params=["0", "1"])
def cfg(request, monkeypatch):
    monkeypatch.setenv("MPDATA_FUSED_CFG", request.param)
    return request.param


def _case(dims, seed, npdt=np.float64, positive=True, cmax=0.4):
    from advectionhpctester_amd.testdata import random_case
    return random_case(*dims, seed=seed, dtype=npdt, positive=positive, cmax=cmax)


def _rel(a, b):
    return float(np.abs(a.astype(np.float64) - b).max() / np.abs(b).max())


def _oracle_steps(orc, variant, iters, nonos, c, ibc, dims, nsteps=NSTEPS):
    x = c["x"].copy()
    for _ in range(nsteps):
        orc.step(variant, iters, nonos, x, *[c[k] for k in KEYS], ibc, dims)
    return x


# FP64: the fast builds' tolerance against the exact step; FP32: the rounding
# of single precision over the steps (20 steps of some 10 roundings of 6e-8)
FAST_TOL = {torch.float64: 1e-12, torch.float32: 1e-5}


@pytest.mark.parametrize("tdt", [torch.float64, torch.float32])
@pytest.mark.parametrize("ibc,nonos", [((0, 0, 0), 1), ((0, 0, 0), 0), ((1, 1, 1), 1),
                                       ((1, 1, 1), 0), ((1, 0, 1), 1), ((1, 0, 1), 0)])
def test_fast_standard(mp, orc64, cfg, tdt, ibc, nonos):
    c = _case(DIMS, 3 + nonos + sum(ibc), positive=False)
    want = _oracle_steps(orc64, mp.STANDARD, 2, nonos, c, ibc, DIMS)
    with mp.Domain(*DIMS, ibc=ibc, dtype=tdt) as d:
        d.set_path(mp.PATH_FAST)
        t = {k: to_dev(v, tdt) for k, v in c.items()}
        print(f"fast standard cfg {cfg} {tdt} ibc={ibc} nonos={nonos}", flush=True)
        d.timeloop(NSTEPS, t["x"], *[t[k] for k in KEYS], variant=mp.STANDARD, iters=2, nonos=nonos)
        got = to_host(t["x"])
    err = _rel(interior(got), interior(want))
    print(f"  max normwise relative error {err:.3e}", flush=True)
    assert err <= FAST_TOL[tdt], err


@pytest.mark.parametrize("tdt", [torch.float64, torch.float32])
@pytest.mark.parametrize("iters,nsteps", [(2, NSTEPS), (3, 1)])
def test_fast_gauge(mp, orc64, cfg, tdt, iters, nsteps):
    """Three iterations over one step: on random fields the third pass
    amplifies a rounding from step to step (the oracle's own FP32 steps are
    1.1e-4 from its FP64 ones after 20, 2e-7 after two)."""
    c = _case(DIMS, 11)
    want = _oracle_steps(orc64, mp.GAUGE, iters, 1, c, (0, 0, 0), DIMS, nsteps)
    with mp.Domain(*DIMS, dtype=tdt) as d:
        d.set_path(mp.PATH_FAST)
        t = {k: to_dev(v, tdt) for k, v in c.items()}
        print(f"fast gauge cfg {cfg} {tdt} iters {iters}", flush=True)
        d.timeloop(nsteps, t["x"], *[t[k] for k in KEYS], variant=mp.GAUGE, iters=iters)
        got = to_host(t["x"])
    err = _rel(interior(got), interior(want))
    print(f"  max normwise relative error {err:.3e}", flush=True)
    assert err <= FAST_TOL[tdt], err


@pytest.mark.parametrize("tdt,npdt", DTYPES)
@pytest.mark.parametrize("ibc", [(0, 0, 0), (1, 0, 1), (1, 1, 1)])
@pytest.mark.parametrize("nonos", [1, 0])
def test_exact_standard(mp, cfg, tdt, npdt, ibc, nonos):
    """The stage kernels' bits, in both precisions."""
    c = _case(DIMS, 17 + sum(ibc), npdt, positive=False)
    with mp.Domain(*DIMS, ibc=ibc, dtype=tdt) as d:
        t = {k: to_dev(v) for k, v in c.items()}
        a = t["x"].clone()
        b = torch.full_like(a, float("nan"))
        f = [t[k] for k in KEYS]
        print(f"exact standard cfg {cfg} {tdt} ibc={ibc} nonos={nonos}", flush=True)
        d.set_path(mp.PATH_STAGES)
        d.step(a, *f, variant=mp.STANDARD, nonos=nonos)
        d.set_path(mp.PATH_FUSED)
        d.step_oop(t["x"], b, *f, variant=mp.STANDARD, nonos=nonos)
        a, b = to_host(a), to_host(b)
    assert bits_equal(a, b), describe_diff(a, b)


DENSITY = ("u1", "u2", "u3", "x_in", "x_incomp", "h", "rhoadv", "rhr", "pexe", "pexr1", "pexr2",
           "bcx", "bcy")


def _density(mp, dims, path, tdt=torch.float64, seed=7):
    """One call of the density step after its predictor; every array."""
    from advectionhpctester_amd.testdata import density_case
    f = density_case(*dims, seed=seed, cmax=0.5, dtype=np.float64)
    g = {k: to_dev(f[k], tdt) for k in DENSITY}
    with mp.Domain(*dims, dtype=tdt) as d:
        d.set_path(path)
        print(f"density {dims} {tdt} path {path}", flush=True)
        d.rho_gauge_core(*[g[k] for k in DENSITY])
        return {k: to_host(v) for k, v in g.items()}


@pytest.mark.parametrize("tdt", [torch.float64, torch.float32])
def test_fast_density(mp, cfg, tdt):
    """Against the stage kernels' step in FP64 (one step: single precision's
    rounding is some 10 roundings of 6e-8 of the largest value)."""
    want = _density(mp, DIMS, mp.PATH_STAGES)
    got = _density(mp, DIMS, mp.PATH_FAST, tdt)
    for k in DENSITY:
        scale = float(np.abs(want[k]).max())
        err = float(np.abs(got[k].astype(np.float64) - want[k]).max()) / (scale or 1.0)
        assert err <= (1e-12 if tdt == torch.float64 else 2e-6), f"{k}: {err:.3e}"


# 289 tiles of 32x32 and 663 of 32x16 for 256 CUs: one and two rounds of whole
# tiles, then runs (40 planes) or chunks (6)
MANY = [(450, 460, 40), (450, 460, 6)]


@pytest.mark.parametrize("size", MANY)
def test_density_whole_tiles_then_runs(mp, size):
    dims = size + (1,)
    want = _density(mp, dims, mp.PATH_STAGES)
    got = _density(mp, dims, mp.PATH_FUSED)
    for k in DENSITY:
        assert bits_equal(got[k], want[k]), f"{k}: " + describe_diff(got[k], want[k])


@pytest.mark.parametrize("size", MANY)
@pytest.mark.parametrize("variant,iters,ibc", [("gauge", 3, (0, 0, 0)), ("standard", 2, (1, 0, 1)),
                                               ("standard", 2, (1, 1, 1))])
def test_passes_and_periodic_whole_tiles_then_runs(mp, size, variant, iters, ibc):
    dims = size + (1,)
    c = _case(dims, 5)
    kw = dict(variant=mp.GAUGE if variant == "gauge" else mp.STANDARD, iters=iters)
    with mp.Domain(*dims, ibc=ibc) as d:
        t = {k: to_dev(v) for k, v in c.items()}
        a = t["x"].clone()
        b = torch.full_like(a, float("nan"))
        f = [t[k] for k in KEYS]
        print(f"many tiles {variant} iters {iters} {size} ibc={ibc}", flush=True)
        d.set_path(mp.PATH_STAGES)
        d.step(a, *f, **kw)
        d.set_path(mp.PATH_FUSED)
        d.step_oop(t["x"], b, *f, **kw)
        a, b = to_host(a), to_host(b)
    assert bits_equal(a, b), describe_diff(a, b)


@pytest.mark.parametrize("size", MANY)
@pytest.mark.parametrize("variant", ["gauge", "standard"])
def test_recorded_step_whole_tiles_then_runs(mp, size, variant):
    """The recorded step's output and, through the reverse step, its tape."""
    dims = size + (1,)
    c = _case(dims, 5)
    v = mp.GAUGE if variant == "gauge" else mp.STANDARD
    res = {}
    for path in (mp.PATH_STAGES, mp.PATH_AUTO):
        with mp.Domain(*dims) as d:
            d.set_path(path)
            t = {k: to_dev(a) for k, a in c.items()}
            f = [t[k] for k in KEYS[:5]]
            out = torch.zeros_like(t["x"])
            xbar = torch.zeros_like(t["x"])
            mp.interior(xbar).copy_(mp.interior(t["x"]))
            ub = [torch.zeros_like(t[k]) for k in KEYS[:3]]
            print(f"recorded step {variant} {size} path {path}", flush=True)
            d.adj_reserve(1)
            d.adj_record(0, t["x"], out, *f, t["bcx"], t["bcy"], variant=v)
            d.adj_step(0, *f, xbar, *ub)
            res[path] = [interior(to_host(out))] + [to_host(a) for a in (mp.interior(xbar), *ub)]
    a, b = res[mp.PATH_STAGES], res[mp.PATH_AUTO]
    assert bits_equal(a[0], b[0]), describe_diff(a[0], b[0])
    # the same tape: the reverse sums differ in the order of their atomics
    for p, q in zip(a[1:], b[1:]):
        assert float(np.abs(p - q).max()) <= 1e-13 * float(np.abs(p).max()), describe_diff(p, q)
