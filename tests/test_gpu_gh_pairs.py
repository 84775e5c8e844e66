"""The GH RHS in two kernels (point state, then one workgroup per element and
symmetric pair) at the edges of its range, bit for bit against the oracle,
and its choice in place of the fused kernel."""
import numpy as np
import pytest
import torch

import oracle_lib as ol
from spectre_amd import dg, workloads as wl

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float64)).cuda()


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


# smallest extents, flat and long ones, the largest that fit the LDS (14^3)
# and the first that does not (15^3, the one-component-at-a-time kernels)
@pytest.mark.parametrize("elements,extents", [((2, 1, 2), (2, 2, 2)), ((1, 2, 2), (2, 3, 2)),
                                              ((2, 2, 1), (20, 2, 9)), ((1, 3, 1), (5, 13, 11)),
                                              ((1, 1, 2), (14, 14, 14)),
                                              ((1, 1, 2), (15, 15, 15))])
def test_gh_rhs_pairs_edges(elements, extents):
    print(f"gh pairs {elements} x {extents}", flush=True)
    brick, u, gammas, inv = wl.gh_kerr_schild_brick(seed=3, elements=elements, extents=extents,
                                                    noise=1e-3)
    inv = inv + 1e-2 * np.random.default_rng(1).standard_normal(inv.shape)
    ref = ol.gh_rhs(brick.extents, brick.neighbors, u, gammas, inv)
    domain = dg.Domain.from_brick(brick)
    domain.set_kernel("gh", "composite")
    assert np.array_equal(host(domain.gh_rhs(dev(u), dev(gammas), dev(inv))), ref)


# both sides of each line in the choice of threads: 256 and 768 points, 256
# workgroups, and rounds that 192 or 256 threads fill better
@pytest.mark.parametrize("elements,extents", [((1, 2, 1), (8, 8, 4)), ((1, 2, 1), (7, 7, 6)),
                                              ((3, 3, 3), (7, 7, 6)), ((3, 3, 3), (7, 8, 7)),
                                              ((1, 2, 1), (12, 8, 8)), ((3, 3, 3), (12, 8, 8)),
                                              ((1, 1, 2), (11, 10, 7)), ((1, 1, 2), (10, 9, 9))])
def test_gh_rhs_pairs_threads(elements, extents):
    print(f"gh pairs threads {elements} x {extents}", flush=True)
    brick, u, gammas, inv = wl.gh_kerr_schild_brick(seed=4, elements=elements, extents=extents,
                                                    noise=1e-3)
    ref = ol.gh_rhs(brick.extents, brick.neighbors, u, gammas, inv)
    domain = dg.Domain.from_brick(brick)
    domain.set_kernel("gh", "composite")
    assert np.array_equal(host(domain.gh_rhs(dev(u), dev(gammas), dev(inv))), ref)


@pytest.mark.parametrize("extents", [(2, 2, 2), (4, 6, 3), (7, 7, 7)])
def test_gh_rhs_dirichlet_pairs(extents):
    print(f"gh pairs dirichlet {extents}", flush=True)
    brick, u, gammas, inv, ghost = wl.gh_kerr_schild_dirichlet(seed=2, elements=(2, 1, 3),
                                                               extents=extents)
    ref = ol.gh_rhs_dirichlet(brick.extents, brick.neighbors, u, gammas, inv, ghost)
    domain = dg.Domain.from_brick(brick)
    domain.set_kernel("gh", "composite")
    got = host(domain.gh_rhs_dirichlet(dev(u), dev(gammas), dev(inv), dev(ghost)))
    assert np.array_equal(got, ref)


# one element count on each side of the line for every N, against the fused kernel
@pytest.mark.parametrize("n,few,many", [(3, (4, 4, 4), (8, 8, 9)), (4, (4, 4, 4), (8, 8, 10)),
                                        (5, (4, 4, 4), (8, 8, 8)), (6, (4, 4, 4), (4, 8, 8)),
                                        (8, (4, 4, 4), (4, 8, 8))])
def test_gh_auto_choice_matches_fused(n, few, many):
    for elements, kernel in ((few, "composite"), (many, "fused")):
        print(f"gh auto {elements} x {n}^3", flush=True)
        brick, u, gammas, inv = wl.gh_kerr_schild_brick(seed=5, elements=elements,
                                                        extents=(n, n, n))
        domain = dg.Domain.from_brick(brick)
        assert domain.kernel("gh") == kernel
        args = dev(u), dev(gammas), dev(inv)
        got = host(domain.gh_rhs(*args))
        domain.set_kernel("gh", "fused")
        assert np.array_equal(got, host(domain.gh_rhs(*args)))


def test_gh_auto_choice_in_a_graph():
    """A call recorded into a graph needs no work arrays: the first call on a
    fresh domain is the captured one, and every replay is right beside eager
    calls that use the work arrays."""
    brick, u, gammas, inv = wl.gh_kerr_schild_brick(seed=6, elements=(2, 2, 2), extents=(6, 6, 6))
    domain = dg.Domain.from_brick(brick)
    u, gammas, inv = dev(u), dev(gammas), dev(inv)
    out = torch.empty_like(u)
    dg.Domain.from_brick(brick).gh_rhs(u, gammas, inv)  # tables are on the device
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        domain.gh_rhs(u, gammas, inv, out)
    for k in range(3):
        u.mul_(1.0 + 1e-3 * k)
        out.zero_()
        graph.replay()
        eager = domain.gh_rhs(u, gammas, inv)
        assert np.array_equal(host(out), host(eager))


# the choice at the element counts where it changes, by rounds of workgroups on
# 256 compute units; 7^3 always takes the pair kernels
@pytest.mark.parametrize("n,pairs,fused", [(3, (428, 1025), (429, 1024)),
                                           (4, (488, 1025), (489, 1024)),
                                           (5, (270, 513), (271, 512)),
                                           (6, (129, 257, 348), (130, 256, 349)),
                                           (7, (1, 255, 256, 257, 600), ()),
                                           (8, (155, 257, 349), (156, 256, 350))])
def test_gh_auto_choice_lines(n, pairs, fused):
    brick, u, gammas, inv = wl.gh_kerr_schild_brick(seed=7, elements=(1, 1, 1),
                                                    extents=(n, n, n), noise=1e-3)
    arrays = [dev(a) for a in (u, gammas, inv)]
    for counts, kernel in ((pairs, "composite"), (fused, "fused")):
        for count in counts:
            print(f"gh auto {count} x {n}^3", flush=True)
            args = [a.repeat(count, 1, 1) for a in arrays]
            args[0] = args[0] * (1.0 + 1e-3 * torch.sin(torch.arange(
                count, dtype=torch.float64, device="cuda")))[:, None, None]
            domain = dg.Domain((n, n, n), wl.periodic_neighbors((count, 1, 1)))
            assert domain.kernel("gh") == kernel
            got = domain.gh_rhs(*args)
            domain.set_kernel("gh", "fused" if kernel == "composite" else "composite")
            assert torch.equal(got, domain.gh_rhs(*args))
