"""One RK3 step whose substeps the right-hand-side kernels apply themselves, in
every kernel organisation that does so and in those that do not, against the
oracle's right-hand sides and substeps: the same additions and products in the
same order, so every value is equal."""
import numpy as np
import pytest
import torch

import oracle_lib as ol
from spectre_amd import _Pybindings as pyb, dg, workloads as wl
from spectre_amd._lib import SYSTEMS

pytestmark = pytest.mark.gpu

DT = 0.004


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float64)).cuda()


def host(t):
    return t.cpu().numpy()


def check(domain, system, rhs, u, params, inv):
    l0 = rhs(u)
    u1 = ol.rk3_substep(0, DT, u, u, l0)
    u2 = ol.rk3_substep(1, DT, u, u1, rhs(u1))
    end = ol.rk3_substep(2, DT, u, u2, rhs(u2))
    d_p, d_i = dev(params), dev(inv)
    args = domain.handle, SYSTEMS[system], DT
    for complete in (True, False):  # with the stage inputs kept
        d_u = dev(u)
        s1, s2, work, out = (torch.empty_like(d_u) for _ in range(4))
        pyb.rk3_step(*args, d_u, d_p, d_i, s1, s2, work, out if complete else None)
        assert np.array_equal(host(s1), u1) and np.array_equal(host(s2), u2)
        assert np.array_equal(host(d_u), u)
        if complete:
            assert np.array_equal(host(out), end)
    d_u = dev(u)  # in place, with one stage array and the work array
    pyb.rk3_step(*args, d_u, d_p, d_i, s1, work, work, d_u)
    assert np.array_equal(host(d_u), end)


@pytest.mark.parametrize("n", [2, 6, 10])
@pytest.mark.parametrize("kernel", ["fused", "composite"])
def test_scalar_wave_step(n, kernel):
    print(f"rk3 step scalar wave {n} {kernel}", flush=True)
    brick, u, g2, inv = wl.scalar_wave_plane_wave_3d(seed=2, elements=(2, 1, 3), extents=(n, n, n))
    domain = dg.Domain.from_brick(brick)
    domain.set_kernel("scalar_wave", kernel)
    check(domain, "scalar_wave", lambda v: ol.sw_rhs(brick.extents, brick.neighbors, v, g2, inv),
          u, g2, inv)


@pytest.mark.parametrize("n", [2, 6])
@pytest.mark.parametrize("kernel", ["fused", "composite", "auto"])
def test_gh_step(n, kernel):
    print(f"rk3 step gh {n} {kernel}", flush=True)
    brick, u, ga, inv = wl.gh_kerr_schild_brick(seed=5, elements=(2, 1, 2), extents=(n, n, n))
    domain = dg.Domain.from_brick(brick)
    domain.set_kernel("gh", kernel)
    check(domain, "gh", lambda v: ol.gh_rhs(brick.extents, brick.neighbors, v, ga, inv), u, ga, inv)


@pytest.mark.parametrize("kernel", ["auto", "mixed_batched"])
def test_mixed_steps(kernel):
    print(f"rk3 step mixed {kernel}", flush=True)
    brick, u, g2, inv = wl.scalar_wave_plane_wave_mixed(seed=3, elements=(2, 1, 2))
    domain = dg.MixedDomain.from_brick(brick)
    domain.set_kernel("scalar_wave", kernel)
    check(domain, "scalar_wave",
          lambda v: ol.sw_rhs_mixed(brick.extents, brick.neighbors, v, g2, inv), u, g2, inv)
    brick, u, ga, inv = wl.gh_kerr_schild_mixed(seed=4, elements=(1, 2, 1), lowest=3, highest=10)
    domain = dg.MixedDomain.from_brick(brick)
    domain.set_kernel("gh", kernel)
    check(domain, "gh", lambda v: ol.gh_rhs_mixed(brick.extents, brick.neighbors, v, ga, inv),
          u, ga, inv)


# steps of elements whose kernels need more than the default LDS, out of a graph
@pytest.mark.parametrize("extents", [(13, 13, 13), (14, 14, 14)])
def test_gh_stepper_large_elements(extents):
    print(f"rk3 stepper gh {extents}", flush=True)
    brick, u, ga, inv = wl.gh_kerr_schild_brick(seed=5, elements=(1, 1, 2), extents=extents)
    rhs = lambda v: ol.gh_rhs(brick.extents, brick.neighbors, v, ga, inv)
    u1 = ol.rk3_substep(0, DT, u, u, rhs(u))
    u2 = ol.rk3_substep(1, DT, u, u1, rhs(u1))
    end = ol.rk3_substep(2, DT, u, u2, rhs(u2))
    d_u, d_ga, d_inv = dev(u), dev(ga), dev(inv)
    stepper = dg.Rk3Stepper(dg.Domain.from_brick(brick), "gh", d_u, d_ga, d_inv)
    for _ in range(3):
        d_u.copy_(dev(u))
        stepper.step(DT)
        torch.cuda.synchronize()
        assert np.array_equal(host(d_u), end)
    stepper.close()


def step_adjoint(adjoint, lam3):
    """mu of one transposed step; adjoint(k, lam) = A^T lam at stage input k."""
    lam = (2.0 / 3.0) * (lam3 + DT * adjoint(2, lam3))
    mu = (1.0 / 3.0) * lam3 + 0.75 * lam
    lam = 0.25 * (lam + DT * adjoint(1, lam))
    return mu + (lam + DT * adjoint(0, lam))


def run_adjoint(domain, system, states, params, inv, lam3):
    d_lam3 = dev(lam3)
    a, lam, mu = (torch.full_like(d_lam3, float("nan")) for _ in range(3))
    s = [None if t is None else dev(t) for t in states]
    pyb.rk3_step_adjoint(domain.handle, SYSTEMS[system], DT, *s, dev(params), dev(inv), d_lam3, a,
                         lam, mu)
    assert np.array_equal(host(d_lam3), lam3)
    return host(mu)


@pytest.mark.parametrize("n", [2, 6, 10])
def test_scalar_wave_step_adjoint(n):
    print(f"rk3 step adjoint scalar wave {n}", flush=True)
    brick, u, g2, inv = wl.scalar_wave_plane_wave_3d(seed=2, elements=(2, 1, 3), extents=(n, n, n))
    lam3 = np.random.default_rng(3).standard_normal(u.shape)
    ref = step_adjoint(lambda k, lam: ol.sw_rhs_adjoint(brick.extents, brick.neighbors, lam, g2,
                                                        inv), lam3)
    got = run_adjoint(dg.Domain.from_brick(brick), "scalar_wave", [None] * 3, g2, inv, lam3)
    assert np.array_equal(got, ref)


# the GH kernels add the adjoint's terms in another order than the tape, to
# 1e-12 of the largest value per right-hand side; the three of a step add up,
# each with a factor dt times an adjoint of norm ~ 1 / dt
GH_TOL = 3e-12


@pytest.mark.parametrize("extents", [(2, 2, 2), (8, 9, 9), (10, 9, 9)])
def test_gh_step_adjoint(extents):
    print(f"rk3 step adjoint gh {extents}", flush=True)
    brick, u, ga, inv, _ = wl.gh_adjoint_workload(seed=1, elements=(1, 1, 2), extents=extents,
                                                  noise=1e-3)
    rng = np.random.default_rng(4)
    states = [u * (1.0 + 1e-3 * rng.standard_normal(u.shape)) for _ in range(3)]
    lam3 = rng.standard_normal(u.shape)
    ref = step_adjoint(lambda k, lam: ol.gh_rhs_vjp(brick.extents, brick.neighbors, states[k], ga,
                                                    inv, lam), lam3)
    got = run_adjoint(dg.Domain.from_brick(brick), "gh", states, ga, inv, lam3)
    assert np.max(np.abs(got - ref)) <= GH_TOL * np.max(np.abs(ref))


def test_gh_step_adjoint_mixed():
    print("rk3 step adjoint gh mixed", flush=True)
    brick, u, ga, inv, _ = wl.gh_adjoint_workload_mixed(seed=5, elements=(1, 2, 1), lowest=3,
                                                        highest=10, noise=1e-3)
    rng = np.random.default_rng(4)
    states = [u * (1.0 + 1e-3 * rng.standard_normal(u.shape)) for _ in range(3)]
    lam3 = rng.standard_normal(u.shape)
    ref = step_adjoint(lambda k, lam: ol.gh_rhs_mixed_vjp(brick.extents, brick.neighbors,
                                                          states[k], ga, inv, lam), lam3)
    got = run_adjoint(dg.MixedDomain.from_brick(brick), "gh", states, ga, inv, lam3)
    assert np.max(np.abs(got - ref)) <= GH_TOL * np.max(np.abs(ref))
