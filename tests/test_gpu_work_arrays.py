"""Work arrays that pass from one domain to the next, and calls of several host
threads on one stream, which share them."""
import threading
import time

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


def test_domains_after_a_domain_of_nans():
    """What a destroyed domain leaves in its work arrays does not reach the next
    domain's results: RHS and adjoint, uniform and mixed p, of the same and of a
    smaller size."""
    print("work arrays of a destroyed domain", flush=True)
    rng = np.random.default_rng(1)
    dg.lib().sxd_release_cached_memory()
    for mixed in (False, True):
        first = True
        for seed, highest in ((1, 7), (1, 7), (2, 6)):
            if mixed:
                brick, u, gammas, inv = wl.gh_kerr_schild_mixed(seed, (2, 2, 1), 5, highest)
                domain = dg.MixedDomain.from_brick(brick)
                rhs, vjp = ol.gh_rhs_mixed, ol.gh_rhs_mixed_vjp
            else:
                brick, u, gammas, inv = wl.gh_kerr_schild_brick(seed, (2, 2, 1), (5, highest, 5))
                domain = dg.Domain.from_brick(brick)
                rhs, vjp = ol.gh_rhs, ol.gh_rhs_vjp
            gbar = rng.standard_normal(u.shape)
            if first:  # fills the arrays with NaN, then leaves them
                u, gbar = np.full_like(u, np.nan), np.full_like(gbar, np.nan)
            args = dev(u), dev(gammas), dev(inv)
            got, adj = host(domain.gh_rhs(*args)), host(domain.gh_rhs_adjoint(*args, dev(gbar)))
            domain.close()
            if first:
                first = False
                continue
            assert np.array_equal(got, rhs(brick.extents, brick.neighbors, u, gammas, inv))
            ref = vjp(brick.extents, brick.neighbors, u, gammas, inv, gbar)
            assert np.max(np.abs(adj - ref)) <= 1e-12 * np.max(np.abs(ref))


def test_kept_memory_is_given_back():
    print("kept memory", flush=True)
    brick, u, gammas, inv = wl.gh_kerr_schild_brick(seed=3, elements=(6, 6, 6), extents=(7, 7, 7))
    args = dev(u), dev(gammas), dev(inv)
    for _ in range(12):  # 27 MB each
        domain = dg.Domain.from_brick(brick)
        domain.gh_rhs(*args)
        domain.close()
    domains = [dg.Domain.from_brick(brick) for _ in range(14)]
    for domain in domains:
        domain.gh_rhs(*args)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]

    def freed(bytes_):
        """Whether so much more is free, the driver being given 10 seconds."""
        for _ in range(100):
            if torch.cuda.mem_get_info()[0] >= before + bytes_:
                return True
            time.sleep(0.1)
        return False

    for domain in domains:
        domain.close()
    assert freed(14 * 27e6 - (256 << 20) - 14e6)
    dg.lib().sxd_release_cached_memory()
    assert freed(14 * 26e6)


def test_two_threads_on_one_stream():
    """Calls of two host threads on one stream with different states: the pair
    kernels' work array is not written by one between the kernels of the other."""
    print("two threads on one stream", flush=True)
    brick, u, gammas, inv = wl.gh_kerr_schild_brick(seed=3, elements=(2, 2, 2), extents=(7, 7, 7),
                                                    noise=1e-3)
    d_g, d_i = dev(gammas), dev(inv)
    domain = dg.Domain.from_brick(brick)
    domain.set_kernel("gh", "composite")
    states = [dev(u), dev(u * (1.0 + 1e-2 * np.random.default_rng(4).random(u.shape)))]
    refs = [domain.gh_rhs(s, d_g, d_i).clone() for s in states]
    outs = [[torch.empty_like(states[k]) for _ in range(100)] for k in range(2)]
    torch.cuda.synchronize()
    start = threading.Barrier(2)

    def work(k):
        start.wait(30)
        for out in outs[k]:
            domain.gh_rhs(states[k], d_g, d_i, out)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    torch.cuda.synchronize()
    for k in range(2):
        assert all(torch.equal(out, refs[k]) for out in outs[k])
