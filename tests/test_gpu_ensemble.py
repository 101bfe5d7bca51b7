"""Batched ensembles: members of different shapes advanced by one persistent
launch per step (and by one HIP graph per time loop) give the same bits as
the single-domain fused step on each member, for every tile configuration
and k-chunk length, in FP64 and FP32."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(24, 40, 16), (48, 32, 20), (33, 17, 9), (64, 64, 12), (16, 16, 40), (40, 24, 30)]


@pytest.fixture(scope="module")
def mpd():
    from advectionhpctester_amd import mpdata
    return mpdata


def _members(dtype, shapes=SHAPES, seed0=100):
    from advectionhpctester_amd import testdata
    return [testdata.ensemble_member(*s, seed=seed0 + q, dtype=dtype, device="cuda:0")
            for q, s in enumerate(shapes)]


def _reference_steps(mpd, shapes, members, xs, nsteps, dtype):
    """nsteps single-domain fused steps per member, from xs."""
    out = []
    for s, m, x in zip(shapes, members, xs):
        with mpd.Domain(*s, dtype=dtype) as d:
            d.set_path(mpd.PATH_FUSED)
            a, b = x.clone(), torch.empty_like(x)
            for _ in range(nsteps):
                d.step_oop(a, b, m["u1"], m["u2"], m["u3"], m["rhr"], m["h"], m["bcx"], m["bcy"])
                a, b = b, a
            out.append(a)
    torch.cuda.synchronize()
    return out


def _ensemble(mpd, shapes, members, dtype):
    ens = mpd.Ensemble(shapes, dtype=dtype)
    xa = [m["x"].clone() for m in members]
    xb = [torch.zeros_like(m["x"]) for m in members]
    ens.set_fields(xa, xb, *[[m[k] for m in members] for k in
                             ("u1", "u2", "u3", "rhr", "h", "bcx", "bcy")])
    return ens, xa, xb


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_batched_step_every_tiling(mpd, dtype):
    members = _members(dtype)
    want = _reference_steps(mpd, SHAPES, members, [m["x"] for m in members], 1, dtype)
    ens, xa, xb = _ensemble(mpd, SHAPES, members, dtype)
    with ens:
        for cfg in range(len(mpd.Ensemble.configs())):
            for clen in (7, 64):
                print(f"ensemble {dtype} cfg {cfg} clen {clen}", flush=True)
                ens.set_tiling(cfg, clen)
                for t in xb:
                    t.zero_()
                ens.step(0)
                torch.cuda.synchronize()
                for q, (got, w) in enumerate(zip(xb, want)):
                    assert torch.equal(got, w), f"cfg {cfg} clen {clen} member {q} {SHAPES[q]}"


def test_graph_time_loop_replays(mpd):
    """A 6-step loop captured once and replayed three times, with eager work
    between the replays (resetting and perturbing the start fields); every
    replay equals the single-domain steps."""
    dtype = torch.float64
    members = _members(dtype, seed0=300)
    ens, xa, xb = _ensemble(mpd, SHAPES, members, dtype)
    x0 = [t.clone() for t in xa]
    with ens:
        for rep in range(3):
            print(f"graph replay {rep}", flush=True)
            start = [t.clone() for t in x0]
            if rep == 2:
                for t in start:
                    t.mul_(0.5).add_(0.25)
            for a, s in zip(xa, start):
                a.copy_(s)
            for t in xb:
                t.fill_(-1.0)
            torch.cuda.synchronize()
            ens.run(6, graph=True)
            torch.cuda.synchronize()
            want = _reference_steps(mpd, SHAPES, members, start, 6, dtype)
            for q, (got, w) in enumerate(zip(xa, want)):  # 6 steps: result in xa
                assert torch.equal(got, w), f"replay {rep} member {q}"
        # the same loop without the graph
        for a, s in zip(xa, x0):
            a.copy_(s)
        ens.run(5, graph=False)
        torch.cuda.synchronize()
        want = _reference_steps(mpd, SHAPES, members, x0, 5, dtype)
        for q, (got, w) in enumerate(zip(xb, want)):  # 5 steps: result in xb
            assert torch.equal(got, w), f"eager member {q}"


def test_autotune_keeps_results(mpd):
    dtype = torch.float64
    members = _members(dtype, seed0=500)
    want = _reference_steps(mpd, SHAPES, members, [m["x"] for m in members], 1, dtype)
    ens, xa, xb = _ensemble(mpd, SHAPES, members, dtype)
    with ens:
        cfg, clen, ms = ens.autotune(trial_steps=2)
        print(f"autotune: cfg {cfg} ({mpd.Ensemble.configs()[cfg]}), clen {clen}, {ms:.3f} ms",
              flush=True)
        assert 0 <= cfg < len(mpd.Ensemble.configs()) and clen >= 1 and ms > 0
        assert ens.info()[1:] == (cfg, clen)
        # xa untouched by the trials
        for a, m in zip(xa, members):
            assert torch.equal(a, m["x"])
        ens.step(0)
        torch.cuda.synchronize()
        for q, (got, w) in enumerate(zip(xb, want)):
            assert torch.equal(got, w), f"member {q}"
    # the tuned choice is reused for an ensemble of the same shapes
    with mpd.Ensemble(SHAPES, dtype=dtype) as e2:
        assert e2.info()[1:] == (cfg, clen)


# Members drawn by the batched-ensemble workload's rules (each axis from
# 32..256 in steps of 16, no two axes equal, Gaussian blob of radius 4-16
# cells, solid-body rotation about a random axis at max Courant 0.3-0.8),
# small enough for the CPU oracle to advance in a fraction of a second.
C4_SMALL = [(48, 80, 32), (96, 32, 64), (32, 112, 48), (80, 48, 32), (64, 32, 96)]


def _np(t):
    return t.detach().cpu().numpy().copy()


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_batched_equals_oracle_every_tiling(mpd, dtype):
    """Three batched steps from the same start, for every tile configuration
    and two k-chunk lengths, equal three oracle steps on every member bit for
    bit over the whole array (halos included)."""
    import numpy as np
    from gpu_helpers import bits_equal, describe_diff
    from oracle import Oracle
    npdt = np.float64 if dtype == torch.float64 else np.float32
    orc = Oracle(npdt)
    members = _members(dtype, shapes=C4_SMALL, seed0=700)
    want = []
    for s, m in zip(C4_SMALL, members):
        a = {k: _np(v) for k, v in m.items()}
        x = a["x"]
        for _ in range(3):
            orc.step(1, 2, 1, x, a["u1"], a["u2"], a["u3"], a["rhr"], a["h"], a["bcx"], a["bcy"],
                     (0, 0, 0), s + (1,))
        want.append(x)
    ens, xa, xb = _ensemble(mpd, C4_SMALL, members, dtype)
    x0 = [t.clone() for t in xa]
    with ens:
        for cfg in range(len(mpd.Ensemble.configs())):
            for clen in (9, 64):
                print(f"ensemble vs oracle {dtype} cfg {cfg} clen {clen}", flush=True)
                ens.set_tiling(cfg, clen)
                for a, s in zip(xa, x0):
                    a.copy_(s)
                for t in xb:
                    t.fill_(float("nan"))
                ens.run(3, graph=False)
                torch.cuda.synchronize()
                for q, (got, w) in enumerate(zip(xb, want)):  # 3 steps: result in xb
                    g = _np(got)
                    assert bits_equal(g, w), f"cfg {cfg} clen {clen} member {q} {C4_SMALL[q]}: " \
                        + describe_diff(g, w)


def test_c4_workload_graph_equals_eager_and_oracle(mpd):
    """The full batched-ensemble workload (64 members, seed 4, axes from
    32..256, FP64 gauge MPDATA with the limiter), autotuned, 100 steps as one
    HIP graph: equal bit for bit to the same 100 steps launched eagerly, and
    on the two smallest members to 100 oracle steps; no NaN or Inf; the
    fields stay non-negative everywhere and below their initial maximum away
    from the two lid planes (the mirrored z flux at the lids lets the lid
    planes accumulate where the rotation crosses them)."""
    import numpy as np
    from gpu_helpers import bits_equal, describe_diff
    from oracle import Oracle
    from advectionhpctester_amd import testdata
    dev = torch.device("cuda:0")
    shapes = testdata.ensemble_shapes(64, 4)
    members = [testdata.ensemble_member(*sh, seed=1000 + q, device=dev)
               for q, sh in enumerate(shapes)]
    x0 = [m["x"].clone() for m in members]
    xmax0 = [float(t.max()) for t in x0]
    ens, xa, xb = _ensemble(mpd, shapes, members, torch.float64)
    with ens:
        cfg, clen, ms = ens.autotune(trial_steps=2)
        print(f"c4 autotune: cfg {cfg} clen {clen} {ms:.3f} ms/step", flush=True)
        for a, s in zip(xa, x0):
            a.copy_(s)
        ens.run(100, graph=True)
        torch.cuda.synchronize()
        graph = [t.clone() for t in xa]  # 100 steps: result in xa
        print("c4 graph run done", flush=True)
        for a, s in zip(xa, x0):
            a.copy_(s)
        ens.run(100, graph=False)
        torch.cuda.synchronize()
        print("c4 eager run done", flush=True)
        for q, (g, e) in enumerate(zip(graph, xa)):
            assert torch.equal(g, e), f"member {q} {shapes[q]}: graph != eager"
    for q, (t, sh) in enumerate(zip(graph, shapes)):
        inner = t[1:-1, 1:-1, 1:-1]
        assert bool(torch.isfinite(inner).all()), f"member {q}: non-finite values"
        assert float(inner.min()) >= 0.0, f"member {q}: min {float(inner.min())}"
        away = inner[1:-1]
        assert float(away.max()) <= xmax0[q], f"member {q}: max {float(away.max())} > {xmax0[q]}"
    small = sorted(range(len(shapes)), key=lambda q: shapes[q][0] * shapes[q][1] * shapes[q][2])[:2]
    orc = Oracle(np.float64)
    for q in small:
        a = {k: _np(v) for k, v in members[q].items()}
        x = _np(x0[q])
        print(f"c4 oracle member {q} {shapes[q]} 100 steps", flush=True)
        for _ in range(100):
            orc.step(1, 2, 1, x, a["u1"], a["u2"], a["u3"], a["rhr"], a["h"], a["bcx"], a["bcy"],
                     (0, 0, 0), shapes[q] + (1,))
        g = _np(graph[q])
        assert bits_equal(g, x), f"member {q} {shapes[q]}: " + describe_diff(g, x)


@pytest.mark.parametrize("shapes", [[(8, 8, 4), (12, 9, 5)],
                                    [(8, 8, 4)] * 3 + [(40, 24, 30), (16, 16, 40)]])
def test_dynamic_scheduling_small_and_repeated(mpd, shapes):
    """Work items are taken from per-XCD counters that the last workgroup of
    each XCD resets: a batch with fewer work items than XCDs (one run for
    the whole grid), and a mixed batch stepped eagerly five times in a row
    and as a graph replayed twice, give the single-domain steps each time
    (a counter left unreset would skip items and leave stale outputs)."""
    dtype = torch.float64
    members = _members(dtype, shapes=shapes, seed0=500)
    ens, xa, xb = _ensemble(mpd, shapes, members, dtype)
    with ens:
        for cfg, clen in ((5, 64), (1, 8)):
            ens.set_tiling(cfg, clen)
            for q, m in enumerate(members):
                xa[q].copy_(m["x"])
            print(f"dynamic scheduling {shapes} cfg {cfg} clen {clen}: eager", flush=True)
            for n in range(5):
                ens.step(n & 1)
            got = [(xb if 5 & 1 else xa)[q].clone() for q in range(len(shapes))]
            want = _reference_steps(mpd, shapes, members, [m["x"] for m in members], 5, dtype)
            for q, (g_, w_) in enumerate(zip(got, want)):
                assert torch.equal(g_, w_), f"eager, cfg {cfg} clen {clen} member {q}"
            want2 = _reference_steps(mpd, shapes, members, [m["x"] for m in members], 2, dtype)
            for rep in range(2):
                print(f"dynamic scheduling {shapes} cfg {cfg}: graph replay {rep}", flush=True)
                for q, m in enumerate(members):
                    xa[q].copy_(m["x"])
                ens.run(2, graph=True)
                torch.cuda.synchronize()
                for q, w_ in enumerate(want2):
                    assert torch.equal(xa[q], w_), f"replay {rep}, cfg {cfg} member {q}"


def test_fast_build_equals_fast_single_domain_steps(mpd):
    """The batch on the fast build (mpdata_ens_set_path(MPDATA_PATH_FAST))
    gives the bits of single-domain steps on the fast build, every tiling,
    over three steps, and stays within 1e-12 of the exact batch."""
    dtype = torch.float64
    members = _members(dtype, seed0=700)
    nsteps = 3
    want = []
    for s, m in zip(SHAPES, members):
        with mpd.Domain(*s, dtype=dtype) as d:
            d.set_path(mpd.PATH_FAST)
            a, b = m["x"].clone(), torch.empty_like(m["x"])
            for _ in range(nsteps):
                d.step_oop(a, b, m["u1"], m["u2"], m["u3"], m["rhr"], m["h"], m["bcx"], m["bcy"])
                a, b = b, a
            want.append(a)
    exact = _reference_steps(mpd, SHAPES, members, [m["x"] for m in members], nsteps, dtype)
    ens, xa, xb = _ensemble(mpd, SHAPES, members, dtype)
    with ens:
        ens.set_path(mpd.PATH_FAST)
        for cfg in range(len(mpd.Ensemble.configs())):
            print(f"fast ensemble cfg {cfg}", flush=True)
            ens.set_tiling(cfg, 16)
            for q, m in enumerate(members):
                xa[q].copy_(m["x"])
            ens.run(nsteps, graph=False)
            torch.cuda.synchronize()
            got = xb if nsteps & 1 else xa
            for q, (g_, w_, e_) in enumerate(zip(got, want, exact)):
                assert torch.equal(g_, w_), f"cfg {cfg} member {q} {SHAPES[q]}"
                i = (slice(1, -1),) * 3
                err = float((g_[i] - e_[i]).abs().max() / e_[i].abs().max())
                assert err <= 1e-12, f"cfg {cfg} member {q}: {err:.2e} from the exact build"
        with pytest.raises(mpd.MpdataError):
            ens.set_path(mpd.PATH_STAGES)


def test_many_members_with_halos(mpd):
    """More members than the launch has blocks for their halos, and one whose
    halo is many blocks' work: every cell of every member."""
    dtype = torch.float64
    shapes = [(5 + q % 7, 4 + q % 5, 3 + q % 3) for q in range(330)] + [(300, 120, 4)]
    members = _members(dtype, shapes, seed0=900)
    want = _reference_steps(mpd, shapes, members, [m["x"] for m in members], 1, dtype)
    ens, xa, xb = _ensemble(mpd, shapes, members, dtype)
    with ens:
        for cfg in (1, 5):
            print(f"331 members cfg {cfg}", flush=True)
            ens.set_tiling(cfg, 64)
            for t in xb:
                t.fill_(-1.0)
            ens.step(0)
            torch.cuda.synchronize()
            for q, (got, w) in enumerate(zip(xb, want)):
                assert torch.equal(got, w), f"cfg {cfg} member {q} {shapes[q]}"


def test_halo_cost_of_many_small_members(mpd):
    """1000 members of one tile each take about as long as 250 members of four
    tiles each (as many work items and interior cells, the same kernel): their
    halos are copied by all the blocks, not one member after the other."""
    dtype = torch.float64
    ms = {}
    for n, s in ((1000, (20, 20, 10)), (250, (40, 40, 10))):
        members = _members(dtype, [s], seed0=7) * n
        ens = mpd.Ensemble([s] * n, dtype=dtype)
        xb = [torch.zeros_like(m["x"]) for m in members]
        ens.set_fields([m["x"] for m in members], xb, *[[m[k] for m in members] for k in
                       ("u1", "u2", "u3", "rhr", "h", "bcx", "bcy")])
        with ens:
            ens.set_tiling(5, 64)
            best = []
            for _ in range(5):
                a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
                ens.step(0)
                a.record()
                for _ in range(20):
                    ens.step(0)
                b.record()
                b.synchronize()
                best.append(a.elapsed_time(b) / 20)
            ms[n] = min(best)
    print(f"1000 small members {ms[1000]:.3f} ms, 250 larger ones {ms[250]:.3f} ms", flush=True)
    assert ms[1000] < 1.6 * ms[250], ms


def test_fast_build_no_slower_on_any_tiling(mpd):
    """The fast build of the batched step, whose divisions are cheaper, is no
    slower than the exactly rounded one on any tile configuration (a
    configuration whose registers leave one workgroup on a CU where two fit
    is)."""
    shapes = [(96 + 32 * (q % 4), 80 + 24 * (q % 5), 48 + 16 * (q % 3)) for q in range(24)]
    members = _members(torch.float64, shapes, seed0=40)
    ens, xa, xb = _ensemble(mpd, shapes, members, torch.float64)
    with ens:
        for cfg, name in enumerate(mpd.Ensemble.configs()):
            ms = {}
            for _ in range(4):  # in turn
                for path in (mpd.PATH_FUSED, mpd.PATH_FAST):
                    ens.set_path(path)
                    ens.set_tiling(cfg, 64)
                    a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
                    ens.step(0)
                    a.record()
                    for _ in range(5):
                        ens.step(0)
                    b.record()
                    b.synchronize()
                    ms.setdefault(path, []).append(a.elapsed_time(b) / 5)
            exact, fast = min(ms[mpd.PATH_FUSED]), min(ms[mpd.PATH_FAST])
            print(f"{name}: exact {exact:.3f} fast {fast:.3f} ms", flush=True)
            assert fast < exact, (name, fast, exact)


def test_halo_cost_beside_a_large_member(mpd):
    """One large member and 1000 of one tile each in one ensemble take about as
    long as the two ensembles one after the other: a small member's halo is one
    share of the copy, whatever the largest member's is."""
    dtype = torch.float64
    small, large = (20, 20, 10), (512, 512, 64)
    ms = {}
    for name, shapes in (("small", [small] * 1000), ("large", [large]),
                         ("both", [large] + [small] * 1000)):
        made = {s: _members(dtype, [s], seed0=7)[0] for s in set(shapes)}
        members = [made[s] for s in shapes]
        ens = mpd.Ensemble(shapes, dtype=dtype)
        xb = [torch.zeros_like(m["x"]) for m in members]
        ens.set_fields([m["x"] for m in members], xb, *[[m[k] for m in members] for k in
                       ("u1", "u2", "u3", "rhr", "h", "bcx", "bcy")])
        with ens:
            ens.set_tiling(5, 64)
            best = []
            for _ in range(5):
                a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
                ens.step(0)
                a.record()
                for _ in range(20):
                    ens.step(0)
                b.record()
                b.synchronize()
                best.append(a.elapsed_time(b) / 20)
            ms[name] = min(best)
    print(f"1000 small and a large member: {ms}", flush=True)
    assert ms["both"] < 1.2 * (ms["small"] + ms["large"]), ms
