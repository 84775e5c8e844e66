"""Domains of so many small elements that one launch with a workgroup per element
(or mortar) and symmetric pair has 2^32 threads or more: against kernel
organisations with a workgroup per element, bit for bit."""
import numpy as np
import pytest
import torch

from spectre_amd import dg, workloads as wl

pytestmark = pytest.mark.gpu


def state(points, mixed):
    """One Kerr-Schild point on every point of 2^3 elements, with a factor that
    differs from point to point: [E][nc][8], flat where mixed."""
    _, u, gammas, inv = wl.gh_kerr_schild_brick(seed=1, elements=(1, 1, 1), extents=(2, 2, 2))
    e = points // 8
    factor = 1.0 + 1e-3 * torch.cos(torch.arange(points, dtype=torch.float64,
                                                 device="cuda")).reshape(e, 1, 8)
    fill = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda().expand(e, -1, -1)
    u, gammas, inv = fill(u) * factor, fill(gammas).contiguous(), fill(inv).contiguous()
    return [t.reshape(-1) for t in (u, gammas, inv)] if mixed else [u, gammas, inv]


def test_gh_pairs_of_seven_million_elements():
    print("7 million uniform elements", flush=True)
    elements = (190, 192, 192)  # 10 workgroups of 64 threads each: 4.48e9 threads
    count = int(np.prod(elements))
    u, gammas, inv = state(8 * count, False)
    domain = dg.Domain((2, 2, 2), wl.periodic_neighbors(elements))
    domain.set_kernel("gh", "fused")
    ref = domain.gh_rhs(u, gammas, inv)
    domain.set_kernel("gh", "composite")
    got = domain.gh_rhs(u, gammas, inv, torch.zeros_like(u))
    assert torch.equal(got, ref)


def test_gh_mortars_of_a_million_elements():
    print("760 thousand ragged elements", flush=True)
    elements = (95, 80, 100)  # 3 mortars each, 10 workgroups of 192 threads: 4.38e9 threads
    count = int(np.prod(elements))
    u, gammas, inv = state(8 * count, True)
    domain = dg.MixedDomain(np.full((count, 3), 2, dtype=np.int32),
                            wl.periodic_neighbors(elements))
    domain.set_kernel("gh", "mixed_batched")
    ref = domain.gh_rhs(u, gammas, inv)
    domain.set_kernel("gh", "mortar")
    got = domain.gh_rhs(u, gammas, inv, torch.zeros_like(u))
    assert torch.equal(got, ref)


@pytest.mark.parametrize("layout,elements", [("uniform", (152, 152, 152)), ("mixed", (95, 80, 100))])
def test_gh_adjoint_of_many_elements(layout, elements):
    """Equal elements: every element's adjoint is that of one element alone."""
    print(f"adjoint of many elements, {layout}", flush=True)
    count = int(np.prod(elements))
    mixed = layout == "mixed"
    rng = np.random.default_rng(2)
    _, u, gammas, inv = wl.gh_kerr_schild_brick(seed=1, elements=(1, 1, 1), extents=(2, 2, 2),
                                                noise=1e-3)
    arrays = [torch.from_numpy(np.ascontiguousarray(a)).cuda()
              for a in (u, gammas, inv, rng.standard_normal(u.shape))]

    def adjoint(elements, e):
        neighbors = wl.periodic_neighbors(elements)
        domain = (dg.MixedDomain(np.full((e, 3), 2, dtype=np.int32), neighbors) if mixed else
                  dg.Domain((2, 2, 2), neighbors))
        full = [a.expand(e, -1, -1).contiguous() for a in arrays]
        full = [a.reshape(-1) for a in full] if mixed else full
        return domain.gh_rhs_adjoint(*full, torch.zeros_like(full[0])).reshape(e, 50, 8)

    one = adjoint((1, 1, 1), 1)
    assert torch.equal(adjoint(elements, count), one.expand(count, -1, -1))
