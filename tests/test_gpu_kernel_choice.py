"""The kernel that a call runs where the library, not the caller, made the
choice: the same results with and without room for work arrays, inside and
outside of a captured graph."""
import numpy as np
import pytest
import torch

from spectre_amd import dg, workloads as wl

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float64)).cuda()


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


def gh_case(elements, n, seed=6):
    brick, u, gammas, inv = wl.gh_kerr_schild_brick(seed=seed, elements=elements,
                                                    extents=(n, n, n))
    return brick, dev(u), dev(gammas), dev(inv)


def replay_against_eager(domain, u, gammas, inv):
    """The domain's next call recorded on a stream that it has not seen."""
    out = torch.empty_like(u)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        domain.gh_rhs(u, gammas, inv, out)
    for k in range(3):
        u.mul_(1.0 + 1e-3 * k)
        out.zero_()
        graph.replay()
        assert np.array_equal(host(out), host(domain.gh_rhs(u, gammas, inv)))


def test_autotuned_choice_in_a_graph():
    """The autotuner takes the pair kernels for few small elements; a call
    recorded on a new stream still allocates nothing."""
    print("autotuned capture", flush=True)
    brick, u, gammas, inv = gh_case((2, 2, 2), 6)
    domain = dg.Domain.from_brick(brick)
    kernel, _ = domain.autotune("gh", u, gammas, inv, torch.empty_like(u))
    assert kernel == "composite" and domain.kernel("gh") == "composite"
    replay_against_eager(domain, u, gammas, inv)


def test_autotuned_choice_without_work_arrays():
    """343 elements of 7^3 would need a work array above the fixed one."""
    print("autotuned noalloc", flush=True)
    brick, u, gammas, inv = gh_case((7, 7, 7), 7)
    domain = dg.Domain.from_brick(brick)
    domain.autotune("gh", u, gammas, inv, torch.empty_like(u))
    assert domain.kernel("gh") == "composite"
    got = domain.gh_rhs_noalloc(u, gammas, inv, torch.empty_like(u))
    assert np.array_equal(host(got), host(domain.gh_rhs(u, gammas, inv)))


@pytest.mark.parametrize("choice", ["auto", "autotuned", "fused", "composite"])
def test_twin_has_the_same_choice(choice):
    """A twin is chosen for like its domain: pinned only where that is."""
    print(f"twin of {choice}", flush=True)
    brick, u, gammas, inv = gh_case((2, 2, 2), 6)
    domain = dg.Domain.from_brick(brick)
    if choice == "autotuned":
        domain.autotune("gh", u, gammas, inv, torch.empty_like(u))
    else:
        domain.set_kernel("gh", choice)
    domain.set_threads("gh", 512)
    twin = domain.twin()
    assert twin.kernel("gh") == domain.kernel("gh") and twin.threads("gh") == 512
    if choice != "composite":  # pinned, it needs its work array before a capture
        replay_against_eager(twin, u, gammas, inv)
    other = dg.Domain((5, 5, 5), brick.neighbors)
    with pytest.raises(dg.SpectreAmdError, match="different"):
        dg.check(dg.lib().sxd_domain_copy_choices(other.handle, domain.handle))
