"""The kernels of the GH adjoint at the edges of their routes, against
the oracle's reverse-mode tape: elements whose 15 derivative adjoints per point
leave two workgroups per CU or one (8 x 9 x 9, 10 x 9 x 9), the largest whose fit
the LDS and ones beyond (11 x 12 x 10, 12 x 11 x 11), elements whose five fields
exceed it (16^3), the smallest and flat
ones, several point rounds per thread, and ragged elements of both size
classes, whose mortars reach the largest LDS (extents 12 and 13)."""
import numpy as np
import pytest
import torch

import oracle_lib as ol
from spectre_amd import dg, workloads as wl

pytestmark = pytest.mark.gpu

# the tape and the kernels add the same terms in different orders: some 3e3
# products per point and 3 N sums, rounding 1e-16 each, cancelling at most to
# the largest value by a factor of ten
TOL = 1e-12


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float64)).cuda()


def check(domain, u, gammas, inv, gbar, ref):
    got = domain.gh_rhs_adjoint(dev(u), dev(gammas), dev(inv), dev(gbar)).cpu().numpy()
    err = float(np.max(np.abs(got - ref)) / np.max(np.abs(ref)))
    print(f"max-norm relative error {err:.3e}", flush=True)
    assert err <= TOL


@pytest.mark.parametrize("elements,extents", [((2, 1, 2), (2, 2, 2)), ((1, 2, 1), (20, 2, 3)),
                                              ((1, 2, 1), (8, 9, 9)), ((1, 1, 2), (10, 9, 9)),
                                              ((1, 1, 1), (11, 12, 10)), ((1, 1, 1), (16, 16, 16)),
                                              ((1, 1, 1), (12, 11, 11))])
def test_gh_adjoint_volume_edges(elements, extents):
    print(f"gh adjoint {elements} x {extents}", flush=True)
    brick, u, gammas, inv, _ = wl.gh_adjoint_workload(seed=1, elements=elements, extents=extents,
                                                      noise=1e-3)
    rng = np.random.default_rng(2)
    inv = inv + 1e-2 * rng.standard_normal(inv.shape)
    gammas = gammas + 0.1 * rng.standard_normal(gammas.shape)
    gbar = rng.standard_normal(u.shape)
    ref = ol.gh_rhs_vjp(brick.extents, brick.neighbors, u, gammas, inv, gbar)
    check(dg.Domain.from_brick(brick), u, gammas, inv, gbar, ref)


# elements whose fields are staged one at a time, a workgroup per 512 points: the
# smallest of them, with a last chunk that is nearly full, and one that is not
@pytest.mark.parametrize("extents", [(17, 16, 15), (20, 18, 12)])
def test_gh_adjoint_volume_chunks(extents):
    print(f"gh adjoint chunks {extents}", flush=True)
    brick, u, gammas, inv, _ = wl.gh_adjoint_workload(seed=3, elements=(1, 1, 1), extents=extents,
                                                      noise=1e-3)
    gbar = np.random.default_rng(5).standard_normal(u.shape)
    ref = ol.gh_rhs_vjp(brick.extents, brick.neighbors, u, gammas, inv, gbar)
    check(dg.Domain.from_brick(brick), u, gammas, inv, gbar, ref)


@pytest.mark.parametrize("elements,lowest,highest", [((1, 1, 2), 2, 4), ((1, 2, 1), 8, 11),
                                                     ((1, 1, 2), 12, 13)])
def test_gh_adjoint_volume_ragged_edges(elements, lowest, highest):
    print(f"gh adjoint ragged {elements} {lowest}..{highest}", flush=True)
    brick, u, gammas, inv, _ = wl.gh_adjoint_workload_mixed(seed=5, elements=elements,
                                                            lowest=lowest, highest=highest,
                                                            noise=1e-3)
    rng = np.random.default_rng(3)
    gammas = gammas + 0.1 * rng.standard_normal(gammas.shape)
    gbar = rng.standard_normal(u.shape)
    ref = ol.gh_rhs_mixed_vjp(brick.extents, brick.neighbors, u, gammas, inv, gbar)
    check(dg.MixedDomain.from_brick(brick), u, gammas, inv, gbar, ref)
