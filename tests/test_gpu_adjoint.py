"""Tangent-linear and adjoint MPDATA on the GPU.

* The tangent-linear step (stage kernels on dual numbers) keeps the plain
  step's values bit for bit and its tangent equals torch forward-mode
  differentiation of the CPU reference (oracle/mpdata_torch.py).
* The adjoint kernels give the CPU reference's autograd gradient (x0 and
  the three face velocities) and pass the dot-product test against the
  tangent-linear step.
* The autograd Function with checkpoints (128x128x64, 50 steps, checkpoints
  every 10) agrees with central finite differences along 16 seeded
  directions and with itself under other checkpoint spacings; its cost is
  reported against one plain forward.
"""
import time

import numpy as np
import pytest
import torch

from gpu_helpers import bits_equal, to_dev, to_host

pytestmark = pytest.mark.gpu

I = (slice(1, -1),) * 3


@pytest.fixture(scope="module")
def mpd():
    from advectionhpctester_amd import mpdata
    return mpdata


def _case(dims, seed, positive=True):
    from advectionhpctester_amd import testdata
    return testdata.random_case(*dims, seed=seed, positive=positive, cmax=0.25)


def _zero_halo(a):
    b = np.zeros_like(a)
    b[I] = a[I]
    return b


@pytest.mark.parametrize("variant,iters,nonos", [(2, 2, 1), (1, 2, 1), (1, 3, 1), (2, 2, 0)])
def test_tl_value_is_the_step(mpd, variant, iters, nonos):
    dims = (21, 13, 9, 1)
    c = _case(dims, 11)
    d = {k: to_dev(v) for k, v in c.items()}
    rng = np.random.default_rng(1)
    dx = to_dev(rng.standard_normal(c["x"].shape))
    du = [to_dev(rng.standard_normal(c[k].shape)) for k in ("u1", "u2", "u3")]
    print(f"tl value variant {variant} iters {iters} nonos {nonos}", flush=True)
    with mpd.Domain(*dims) as dom:
        dom.set_path(mpd.PATH_STAGES)
        xs = d["x"].clone()
        dom.step(xs, d["u1"], d["u2"], d["u3"], d["rhr"], d["h"], d["bcx"], d["bcy"],
                 variant=variant, iters=iters, nonos=nonos)
        xt = d["x"].clone()
        dom.tl_step(xt, dx, d["u1"], d["u2"], d["u3"], *du, d["rhr"], d["h"], d["bcx"], d["bcy"],
                    variant=variant, iters=iters, nonos=nonos)
        assert bits_equal(to_host(xt)[I], to_host(xs)[I])


def test_tl_tangent_matches_reference_jvp(mpd):
    import mpdata_torch
    dims = (17, 14, 8, 1)
    c = _case(dims, 12)
    rng = np.random.default_rng(2)
    dxn = _zero_halo(rng.standard_normal(c["x"].shape))
    dun = [rng.standard_normal(c[k].shape) for k in ("u1", "u2", "u3")]
    t = {k: torch.from_numpy(v.copy()) for k, v in c.items()}

    def f(x, u1, u2, u3):
        return mpdata_torch.step(x, u1, u2, u3, t["rhr"], t["h"], t["bcx"], t["bcy"])

    _, jv = torch.autograd.functional.jvp(
        f, (t["x"], t["u1"], t["u2"], t["u3"]),
        (torch.from_numpy(dxn), *[torch.from_numpy(v) for v in dun]))
    d = {k: to_dev(v) for k, v in c.items()}
    with mpd.Domain(*dims) as dom:
        x = d["x"].clone()
        dx = to_dev(dxn)
        dom.tl_step(x, dx, d["u1"], d["u2"], d["u3"], *[to_dev(v) for v in dun], d["rhr"], d["h"],
                    d["bcx"], d["bcy"], variant=mpd.STANDARD, iters=2, nonos=1)
        got = to_host(dx)[I]
    want = jv.numpy()[I]
    err = np.abs(got - want).max() / np.abs(want).max()
    print(f"TL vs reference jvp: max rel {err:.2e}", flush=True)
    assert err < 1e-13


def _adjoint_chain(mpd, dom, d, nsteps, xbar_host):
    """Records nsteps steps from d['x'], runs the adjoints back; returns the
    gradients (x0, u1, u2, u3) as numpy."""
    dom.adj_reserve(nsteps)
    a, b = d["x"].clone(), torch.empty_like(d["x"])
    for n in range(nsteps):
        dom.adj_record(n, a, b, d["u1"], d["u2"], d["u3"], d["rhr"], d["h"], d["bcx"], d["bcy"])
        a, b = b, a
    xbar = to_dev(xbar_host)
    ub = [torch.zeros_like(d[k]) for k in ("u1", "u2", "u3")]
    for n in reversed(range(nsteps)):
        dom.adj_step(n, d["u1"], d["u2"], d["u3"], d["rhr"], d["h"], xbar, *ub)
    return [to_host(xbar)] + [to_host(u) for u in ub], to_host(a)


@pytest.mark.parametrize("dims,seed,positive", [((20, 16, 12, 1), 21, True),
                                                ((13, 18, 7, 1), 22, False)])
def test_adjoint_matches_reference_gradient(mpd, dims, seed, positive):
    import mpdata_torch
    nsteps = 3
    c = _case(dims, seed, positive)
    rng = np.random.default_rng(seed)
    obs = rng.uniform(-1, 2, c["x"].shape)
    t = {k: torch.from_numpy(v.copy()) for k, v in c.items()}
    leaves = [t[k].clone().requires_grad_(True) for k in ("x", "u1", "u2", "u3")]
    y = leaves[0]
    for _ in range(nsteps):
        y = mpdata_torch.step(y, *leaves[1:], t["rhr"], t["h"], t["bcx"], t["bcy"])
    r = (y - torch.from_numpy(obs))[I]
    (0.5 * (r * r).sum()).backward()
    want = [leaf.grad.numpy() for leaf in leaves]
    d = {k: to_dev(v) for k, v in c.items()}
    with mpd.Domain(*dims) as dom:
        xT = y.detach().numpy()
        got, xg = _adjoint_chain(mpd, dom, d, nsteps, _zero_halo(xT - obs))
    assert bits_equal(xg[I], xT[I])
    for name, g_, w_ in zip(("x", "u1", "u2", "u3"), got, want):
        sl = I if name == "x" else (slice(None),) * 3
        err = np.abs(g_[sl] - w_[sl]).max() / np.abs(w_[sl]).max()
        print(f"adjoint vs reference gradient {name}: max rel {err:.2e}", flush=True)
        assert err < 1e-12, name


@pytest.mark.parametrize("dims,seed,positive,chunk", [((20, 16, 12, 1), 31, True, None),
                                                      ((13, 18, 7, 1), 32, False, None),
                                                      ((61, 37, 11, 1), 33, False, "3"),
                                                      ((61, 37, 11, 1), 34, True, "7")])
def test_fused_tape_equals_stage_tape(mpd, dims, seed, positive, chunk, monkeypatch):
    """The fused recording (the fused standard step writing the tape, the
    default path) and the per-stage recording give the same step and the
    same gradients: every tape value the adjoint kernels read is the same.
    The adjoint sums scattered contributions with atomics, whose order may
    differ between runs, so the gradients agree to rounding."""
    if chunk is not None:
        monkeypatch.setenv("MPDATA_FUSED_CHUNK", chunk)
    nsteps = 3
    c = _case(dims, seed, positive)
    rng = np.random.default_rng(seed)
    xbar = _zero_halo(rng.uniform(-1, 1, c["x"].shape))
    d = {k: to_dev(v) for k, v in c.items()}
    res = {}
    for name, path in (("stages", mpd.PATH_STAGES), ("fused", mpd.PATH_AUTO)):
        with mpd.Domain(*dims) as dom:
            dom.set_path(path)
            print(f"tape {name} dims={dims} chunk={chunk}", flush=True)
            res[name] = _adjoint_chain(mpd, dom, d, nsteps, xbar)
    (gs, xs), (gf, xf) = res["stages"], res["fused"]
    assert bits_equal(xs[I], xf[I])
    for name, a_, b_ in zip(("x", "u1", "u2", "u3"), gs, gf):
        sl = I if name == "x" else (slice(None),) * 3
        err = np.abs(a_[sl] - b_[sl]).max() / np.abs(a_[sl]).max()
        print(f"fused vs stage tape, gradient {name}: max rel {err:.2e}", flush=True)
        assert err < 1e-13, name


@pytest.mark.parametrize("nsteps", [1, 5])
def test_dot_product(mpd, nsteps):
    """<TL(dx, du), ybar> = <dx, xbar> + <du, ubar>."""
    dims = (24, 20, 10, 1)
    c = _case(dims, 31)
    d = {k: to_dev(v) for k, v in c.items()}
    rng = np.random.default_rng(7)
    dxn = _zero_halo(rng.standard_normal(c["x"].shape))
    dun = [rng.standard_normal(c[k].shape) for k in ("u1", "u2", "u3")]
    ybar = _zero_halo(rng.standard_normal(c["x"].shape))
    with mpd.Domain(*dims) as dom:
        x, dx = d["x"].clone(), to_dev(dxn)
        du = [to_dev(v) for v in dun]
        for _ in range(nsteps):
            dom.tl_step(x, dx, d["u1"], d["u2"], d["u3"], *du, d["rhr"], d["h"], d["bcx"],
                        d["bcy"], variant=mpd.STANDARD, iters=2, nonos=1)
        lhs = float((to_host(dx)[I] * ybar[I]).sum())
        grads, _ = _adjoint_chain(mpd, dom, d, nsteps, ybar)
    rhs = float((dxn[I] * grads[0][I]).sum()) + sum(float((a * b).sum())
                                                    for a, b in zip(dun, grads[1:]))
    rel = abs(lhs - rhs) / abs(lhs)
    print(f"dot product, {nsteps} steps: <TL,y>={lhs:.15e} <x,AD>={rhs:.15e} rel {rel:.1e}",
          flush=True)
    assert rel <= 1e-12


def test_dot_product_full_size(mpd):
    """The dot-product test on the adjoint workload's grid (128x128x64, the
    deformational flow and field of the gradient problem, 3 steps): the
    tangent-linear and adjoint steps agree over 1e6 cells and 3.2e6 faces."""
    from advectionhpctester_amd import testdata
    c = testdata.adjoint_case(128, 128, 64, nsteps=3)
    f = c.pop("factors")
    c.pop("obs")
    for k in ("u1", "u2", "u3"):
        c[k] = c[k] * f[0]
    nsteps = 3
    d = {k: to_dev(v) for k, v in c.items()}
    rng = np.random.default_rng(17)
    dxn = _zero_halo(rng.standard_normal(c["x"].shape))
    dun = [rng.standard_normal(c[k].shape) for k in ("u1", "u2", "u3")]
    ybar = _zero_halo(rng.standard_normal(c["x"].shape))
    with mpd.Domain(128, 128, 64) as dom:
        x, dx = d["x"].clone(), to_dev(dxn)
        du = [to_dev(v) for v in dun]
        print("dot product at 128x128x64, 3 steps", flush=True)
        for _ in range(nsteps):
            dom.tl_step(x, dx, d["u1"], d["u2"], d["u3"], *du, d["rhr"], d["h"], d["bcx"],
                        d["bcy"], variant=mpd.STANDARD, iters=2, nonos=1)
        lhs = float((to_host(dx)[I] * ybar[I]).sum())
        grads, _ = _adjoint_chain(mpd, dom, d, nsteps, ybar)
    rhs = float((dxn[I] * grads[0][I]).sum()) + sum(float((a * b).sum())
                                                    for a, b in zip(dun, grads[1:]))
    rel = abs(lhs - rhs) / abs(lhs)
    print(f"dot product at 128x128x64: <TL,y>={lhs:.15e} <x,AD>={rhs:.15e} rel {rel:.1e}",
          flush=True)
    assert rel <= 1e-12


def _torch_J(c, nsteps, factors, obs):
    """J = 0.5 |x_T - obs|^2 through the CPU reference and its autograd
    gradient with respect to (x0, u1, u2, u3)."""
    import mpdata_torch
    t = {k: torch.from_numpy(np.ascontiguousarray(v)) for k, v in c.items()}
    leaves = [t[k].clone().requires_grad_(True) for k in ("x", "u1", "u2", "u3")]
    y = leaves[0]
    for n in range(nsteps):
        f = factors[n]
        y = mpdata_torch.step(y, leaves[1] * f, leaves[2] * f, leaves[3] * f, t["rhr"], t["h"],
                              t["bcx"], t["bcy"])
    r = (y - torch.from_numpy(obs))[I]
    (0.5 * (r * r).sum()).backward()
    return [leaf.grad.numpy() for leaf in leaves]


def _gpu_grad(mpd, c, nsteps, factors, obs, ckpt):
    from advectionhpctester_amd import adjoint
    d = {k: to_dev(v) for k, v in c.items()}
    dims = tuple(s - 2 for s in c["x"].shape[::-1]) + (1,)
    with mpd.Domain(*dims) as dom:
        leaves = [d[k].clone().requires_grad_(True) for k in ("x", "u1", "u2", "u3")]
        xT = adjoint.advect(*leaves, dom, d["rhr"], d["h"], d["bcx"], d["bcy"], nsteps,
                            ckpt=ckpt, factors=factors)
        r = mpd.interior(xT - to_dev(obs))
        (0.5 * (r * r).sum()).backward()
        return [to_host(leaf.grad) for leaf in leaves]


def test_gradient_of_deformational_case_matches_reference(mpd):
    """The gradient test problem at 32x32x16, 10 steps, time-varying flow,
    checkpoints every 4 steps: the checkpointed GPU adjoint equals the CPU
    reference's autograd gradient."""
    from advectionhpctester_amd import testdata
    c = testdata.adjoint_case(32, 32, 16, nsteps=10, period=40)
    f = c.pop("factors")
    obs = c.pop("obs")
    want = _torch_J(c, 10, f, obs)
    got = _gpu_grad(mpd, c, 10, f, obs, ckpt=4)
    for name, g_, w_ in zip(("x", "u1", "u2", "u3"), got, want):
        sl = I if name == "x" else (slice(None),) * 3
        err = np.abs(g_[sl] - w_[sl]).max() / np.abs(w_[sl]).max()
        print(f"checkpointed adjoint vs reference, {name}: max rel {err:.2e}", flush=True)
        assert err < 1e-11, name


def test_finite_differences_away_from_switches(mpd):
    """Central differences (eps = 1e-6) along 16 seeded directions supported
    away from the walls and lids, on data whose branches (donor signs,
    limiter selections) have margins far above the perturbation: the
    directional derivative of J over 3 steps equals the adjoint's."""
    from advectionhpctester_amd import adjoint, testdata
    c = testdata.switch_free_case(32, 28, 32)
    rng = np.random.default_rng(3)
    obs = to_dev(rng.uniform(0.5, 2.0, c["x"].shape))
    d = {k: to_dev(v) for k, v in c.items()}
    rest = (d["rhr"], d["h"], d["bcx"], d["bcy"])
    box = (slice(12, 22), slice(9, 20), slice(10, 23))
    with mpd.Domain(32, 28, 32) as dom:

        def J(x0, u1, u2, u3):
            xT = adjoint.advect(x0, u1, u2, u3, dom, *rest, 3, ckpt=2)
            r = mpd.interior(xT - obs)
            return 0.5 * (r * r).sum()

        leaves = [d[k].clone().requires_grad_(True) for k in ("x", "u1", "u2", "u3")]
        J(*leaves).backward()
        grads = [leaf.grad.detach() for leaf in leaves]
        errs = []
        with torch.no_grad():
            for q in range(16):
                dirs = []
                for p, g0 in enumerate(grads):
                    v = torch.zeros_like(g0)
                    if p == 0 or q % 2:     # odd q: velocities too
                        v[box] = to_dev(rng.standard_normal(v[box].shape))
                    dirs.append(v)
                e = 1e-6
                fd = (float(J(*[a + e * v for a, v in zip(leaves, dirs)])) -
                      float(J(*[a - e * v for a, v in zip(leaves, dirs)]))) / (2 * e)
                ad = sum(float((g0 * v).sum()) for g0, v in zip(grads, dirs))
                scale = sum(float(g0.norm() * v.norm()) for g0, v in zip(grads, dirs))
                errs.append(abs(fd - ad) / max(abs(ad), 1e-2 * scale))
                print(f"direction {q}: fd {fd:.12e} ad {ad:.12e} rel {errs[-1]:.1e}", flush=True)
    assert max(errs) < 1e-6


def test_checkpointed_gradient_128x128x64(mpd):
    """The gradient problem at full size: 128x128x64, 50 steps of the
    deformational flow, checkpoints every 10 steps.  Other checkpoint
    spacings give the same gradient; central differences along 16 seeded
    directions (eps = 1e-6) are reported (on this problem they cross limiter
    switches); the cost of forward + backward is reported against one plain
    forward."""
    from advectionhpctester_amd import adjoint, testdata
    c = testdata.adjoint_case(128, 128, 64, nsteps=50)
    f = c.pop("factors")
    obs = to_dev(c.pop("obs"))
    d = {k: to_dev(v) for k, v in c.items()}
    rest = (d["rhr"], d["h"], d["bcx"], d["bcy"])
    nsteps = 50
    with mpd.Domain(128, 128, 64) as dom:

        def J(x0, u1, u2, u3, ckpt=10):
            xT = adjoint.advect(x0, u1, u2, u3, dom, *rest, nsteps, ckpt=ckpt, factors=f)
            r = mpd.interior(xT - obs)
            return 0.5 * (r * r).sum()

        leaves = [d[k].clone().requires_grad_(True) for k in ("x", "u1", "u2", "u3")]
        print("checkpointed gradient, 50 steps at 128x128x64", flush=True)
        J(*leaves).backward()
        grads = [leaf.grad.detach().clone() for leaf in leaves]
        for ck in (7, 50):
            lv = [d[k].clone().requires_grad_(True) for k in ("x", "u1", "u2", "u3")]
            J(*lv, ckpt=ck).backward()
            for g0, leaf in zip(grads, lv):
                assert torch.allclose(leaf.grad, g0, rtol=1e-12, atol=1e-14 * float(g0.abs().max()))
        gen = torch.Generator(device="cuda:0").manual_seed(5)
        errs = []
        with torch.no_grad():
            for q in range(16):
                dirs = []
                for p, g0 in enumerate(grads):
                    v = torch.randn(g0.shape, generator=gen, device="cuda:0", dtype=torch.float64)
                    if p == 0:
                        w = torch.zeros_like(v)
                        mpd.interior(w).copy_(mpd.interior(v))
                        v = w
                    elif q % 2 == 0:
                        v = torch.zeros_like(v)
                    dirs.append(v)
                e = 1e-6
                fd = (float(J(*[a + e * v for a, v in zip(leaves, dirs)])) -
                      float(J(*[a - e * v for a, v in zip(leaves, dirs)]))) / (2 * e)
                ad = sum(float((g0 * v).sum()) for g0, v in zip(grads, dirs))
                errs.append(abs(fd - ad) / abs(ad))
        errs = np.array(errs)
        print(f"finite differences across switches (16 directions): median rel "
              f"{np.median(errs):.2e}, max rel {errs.max():.2e}", flush=True)
        assert np.median(errs) < 0.1
        # cost: forward + backward with checkpoints against one plain forward
        x = d["x"].clone()
        vel = [[d[k] * f[n] for k in ("u1", "u2", "u3")] for n in range(nsteps)]
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for n in range(nsteps):
            dom.step(x, *vel[n], *rest, variant=mpd.STANDARD, iters=2, nonos=1)
        torch.cuda.synchronize()
        t_fwd = time.perf_counter() - t0
        lv = [d[k].clone().requires_grad_(True) for k in ("x", "u1", "u2", "u3")]
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        J(*lv).backward()
        torch.cuda.synchronize()
        t_fb = time.perf_counter() - t0
        print(f"cost: forward {t_fwd * 1e3:.1f} ms, forward+backward {t_fb * 1e3:.1f} ms, "
              f"ratio {t_fb / t_fwd:.2f}", flush=True)


def test_tape_replaced_between_forward_and_backward(mpd):
    """The forward records the last checkpoint segment for the backward; a
    recording on the same domain in between replaces that tape, and the
    backward then recomputes the segment: same gradient either way."""
    from advectionhpctester_amd import adjoint
    dims = (24, 20, 10, 1)
    c = _case(dims, 41, False)
    d = {k: to_dev(v) for k, v in c.items()}
    rest = (d["rhr"], d["h"], d["bcx"], d["bcy"])
    obs = to_dev(np.random.default_rng(41).uniform(-1, 2, c["x"].shape))
    grads = []
    with mpd.Domain(*dims) as dom:
        xp = d["x"].clone()
        for _ in range(7):
            dom.step(xp, d["u1"], d["u2"], d["u3"], *rest, variant=mpd.STANDARD)
        for replace in (False, True):
            leaves = [d[k].clone().requires_grad_(True) for k in ("x", "u1", "u2", "u3")]
            xT = adjoint.advect(*leaves, dom, *rest, 7, ckpt=3)
            # the taped forward (its last steps recorded) gives the plain
            # steps' whole array, halo included
            assert bits_equal(to_host(xT.detach()), to_host(xp))
            if replace:
                print("tape replaced before the backward", flush=True)
                dom.adj_record(0, d["x"], torch.empty_like(d["x"]), d["u1"], d["u2"], d["u3"],
                               *rest)
            r = mpd.interior(xT - obs)
            (0.5 * (r * r).sum()).backward()
            grads.append([leaf.grad.detach().clone() for leaf in leaves])
    for g0, g1 in zip(*grads):
        assert torch.allclose(g1, g0, rtol=1e-12, atol=1e-14 * float(g0.abs().max()))


@pytest.mark.parametrize("dims", [(130, 66, 68, 1), (128, 128, 68, 1)])
def test_dot_product_block_counts(mpd, dims):
    """The dot-product test on grids of 867 and 1088 blocks of the reverse
    pseudo-velocity kernel (between three and four a CU of 256, and more)."""
    c = _case(dims, 41)
    d = {k: to_dev(v) for k, v in c.items()}
    rng = np.random.default_rng(19)
    dxn = _zero_halo(rng.standard_normal(c["x"].shape))
    dun = [rng.standard_normal(c[k].shape) for k in ("u1", "u2", "u3")]
    ybar = _zero_halo(rng.standard_normal(c["x"].shape))
    with mpd.Domain(*dims) as dom:
        x, dx = d["x"].clone(), to_dev(dxn)
        du = [to_dev(v) for v in dun]
        print(f"dot product at {dims}", flush=True)
        dom.tl_step(x, dx, d["u1"], d["u2"], d["u3"], *du, d["rhr"], d["h"], d["bcx"], d["bcy"],
                    variant=mpd.STANDARD, iters=2, nonos=1)
        tl = to_host(dx)[I]
        grads, _ = _adjoint_chain(mpd, dom, d, 1, ybar)
    lhs = float((tl * ybar[I]).sum())
    rhs = float((dxn[I] * grads[0][I]).sum()) + sum(float((a * b).sum())
                                                    for a, b in zip(dun, grads[1:]))
    # rounding of sums of N products: some eps * sqrt(N) of the norms' product,
    # over N (1e6) independent terms; 1e-13 of it is a thousand times that
    scale = float(np.linalg.norm(tl) * np.linalg.norm(ybar[I]))
    print(f"  <TL,y>={lhs:.15e} <x,AD>={rhs:.15e} difference / norms {abs(lhs - rhs) / scale:.1e}",
          flush=True)
    assert abs(lhs - rhs) <= 1e-13 * scale
