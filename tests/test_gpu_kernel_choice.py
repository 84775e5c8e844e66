"""The kernel that a call runs where the library, not the caller, made the
choice: the same results with and without room for work arrays, inside and
outside of a captured graph."""
import contextlib
import ctypes
import gc
import threading

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


@pytest.mark.parametrize("layout", ["composite", "mixed"])
def test_noalloc_takes_what_fits_its_array(layout):
    """343 elements of 7^3 (117,649 points): 45 (composite) and 35 (mixed)
    doubles per point fit 16 Mi, 150 do not."""
    print(f"noalloc {layout}", flush=True)
    brick, u, gammas, inv = gh_case((7, 7, 7), 7)
    if layout == "mixed":
        domain = dg.MixedDomain(np.tile(brick.extents, (343, 1)), brick.neighbors)
        u, gammas, inv = (t.reshape(-1) for t in (u, gammas, inv))
    else:
        domain = dg.Domain.from_brick(brick)
        domain.set_kernel("gh", "composite")
    got = domain.gh_rhs_noalloc(u, gammas, inv, torch.full_like(u, float("nan")))
    assert np.array_equal(host(got), host(domain.gh_rhs(u, gammas, inv)))


def call_ms(call, calls=20):
    call()
    begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    begin.record()
    for _ in range(calls):
        call()
    end.record()
    end.synchronize()
    return begin.elapsed_time(end) / calls


@pytest.mark.parametrize("system", ["scalar_wave", "gh"])
def test_autotuned_threads(system):
    """The autotuner takes the mortar kernels, which choose their own threads; the
    threads it keeps are the ones that suit the kernels with face passes."""
    print(f"autotuned threads {system}", flush=True)
    make = (wl.scalar_wave_plane_wave_mixed if system == "scalar_wave" else
            wl.gh_kerr_schild_mixed)
    brick, u, params, inv = make(seed=1, elements=(4, 4, 4), lowest=4, highest=12)
    u, params, inv = dev(u), dev(params), dev(inv)
    out = torch.empty_like(u)
    domain = dg.MixedDomain.from_brick(brick)
    kernel, _ = domain.autotune(system, u, params, inv, out, repetitions=20)
    assert kernel == "mortar"
    kept = domain.threads(system)
    domain.set_kernel(system, "mixed_batched")
    rhs = domain.scalar_wave_rhs if system == "scalar_wave" else domain.gh_rhs
    times = {}
    for threads in (64, 128, 256):
        domain.set_threads(system, threads)
        times[threads] = call_ms(lambda: rhs(u, params, inv, out))
    print(f"kept {kept}: {times}", flush=True)
    assert times[kept] <= 1.1 * min(times.values())


def test_autotuner_leaves_threads_that_no_kernel_takes():
    print("autotuned threads on a mortar domain", flush=True)
    brick, u, params, inv = wl.gh_mortar_workload(seed=1, base=(2, 2, 2), refine={0: (0, 1)})
    u, params, inv = dev(u), dev(params), dev(inv)
    domain = dg.MortarDomain.from_brick(brick)
    for threads in (64, 256):
        domain.set_threads("gh", threads)
        domain.autotune("gh", u, params, inv, torch.empty_like(u))
        assert domain.threads("gh") == threads


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


def test_first_rhs_in_a_graph_after_other_calls():
    """A stream that has run the adjoint or a condition that needs work arrays
    may record its first RHS."""
    print("first rhs in a graph", flush=True)
    brick, u, gammas, inv = gh_case((1, 2, 1), 12)
    stream = torch.cuda.Stream()
    for other in ("adjoint", "bjorhus"):
        domain = dg.Domain.from_brick(brick)
        out = torch.empty_like(u)
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            if other == "adjoint":
                domain.gh_rhs_adjoint(u, gammas, inv, u, out)
            else:
                domain.gh_rhs_bjorhus(u, gammas, inv, dev(brick.coordinates()), out)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            domain.gh_rhs(u, gammas, inv, out)
        ref = host(dg.Domain.from_brick(brick).gh_rhs(u, gammas, inv))
        for _ in range(3):
            out.zero_()
            graph.replay()
            assert np.array_equal(host(out), ref)


def test_first_rhs_beside_a_capture():
    """A thread's first RHS leaves another thread's capture valid."""
    print("first rhs beside a capture", flush=True)
    brick, u, gammas, inv = gh_case((2, 2, 2), 6)
    ref = host(dg.Domain.from_brick(brick).gh_rhs(u, gammas, inv))
    domain, got = dg.Domain.from_brick(brick), torch.empty_like(u)
    x = torch.ones(8, device="cuda")
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    torch.cuda.synchronize()
    done = []

    def call():
        with torch.cuda.stream(stream):
            domain.gh_rhs(u, gammas, inv, got)
        done.append(True)

    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        x.add_(1.0)
        thread = threading.Thread(target=call)
        thread.start()
        thread.join(60)
    assert done == [True]
    graph.replay()
    assert np.array_equal(host(got), ref) and host(x)[0] == 2.0


def test_rhs_on_the_null_stream_beside_a_capture():
    """The capture of a stream that synchronises with the null stream does not
    fail a call on the null stream."""
    print("null stream beside a capture", flush=True)
    hip = ctypes.CDLL("libamdhip64.so")
    brick, u, gammas, inv = gh_case((2, 2, 2), 6)
    domain = dg.Domain.from_brick(brick)
    ref = host(dg.Domain.from_brick(brick).gh_rhs(u, gammas, inv))
    got = torch.empty_like(u)
    assert torch.cuda.current_stream().cuda_stream == 0
    torch.cuda.synchronize()
    stream, graph = ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipStreamCreate(ctypes.byref(stream)) == 0
    assert hip.hipStreamBeginCapture(stream, 2) == 0  # hipStreamCaptureModeRelaxed
    try:
        domain.gh_rhs(u, gammas, inv, got)
    finally:
        assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
        hip.hipGraphDestroy(graph)
        hip.hipStreamDestroy(stream)
    assert np.array_equal(host(got), ref)


@contextlib.contextmanager
def only_free(free_bytes):
    """Hold all but free_bytes (and at most 64 MiB more) of the device's memory."""
    gc.collect()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    dg.lib().sxd_release_cached_memory()
    room = torch.empty(free_bytes, dtype=torch.uint8, device="cuda")
    held = []
    try:
        for size in (16 << 30, 1 << 30, 64 << 20):
            with contextlib.suppress(torch.OutOfMemoryError):
                while True:
                    held.append(torch.empty(size, dtype=torch.uint8, device="cuda"))
        del room
        torch.cuda.empty_cache()
        yield
    finally:
        torch.cuda.synchronize()
        held.clear()
        torch.cuda.empty_cache()


def test_no_room_for_work_arrays():
    """8000 elements of 7^3: a field takes 1.1 GB, the pair kernels' work array
    1.0 GB.  With room for the fields but not for it, a stepper, a step and an
    RHS run the fused kernel; pinned pair kernels report the missing memory."""
    print("no room for work arrays", flush=True)
    _, u, gammas, inv = gh_case((1, 1, 1), 7)
    elements = (20, 20, 20)
    u, gammas, inv = (t.repeat(8000, 1, 1).contiguous() for t in (u, gammas, inv))
    field = u.numel() * 8
    create = lambda kernel: (d := dg.Domain((7, 7, 7), wl.periodic_neighbors(elements)),
                             d.set_kernel("gh", kernel))[0]
    start, out = u.clone(), torch.empty_like(u)
    stepper = dg.Rk3Stepper(create("fused"), "gh", u, gammas, inv)
    stepper.step(1e-4)
    stepper.close()
    after, rhs = u.clone(), create("fused").gh_rhs(u, gammas, inv)
    u.copy_(start)
    assert create("auto").kernel("gh") == "composite"
    with only_free(2 * field + (550 << 20)):
        with pytest.raises(dg.SpectreAmdError, match="work arrays"):
            dg.Rk3Stepper(create("composite"), "gh", u, gammas, inv)
        stepper = dg.Rk3Stepper(create("auto"), "gh", u, gammas, inv)
        stepper.step(1e-4)
        with pytest.raises(dg.SpectreAmdError, match="work arrays"):
            create("composite").gh_rhs(u, gammas, inv, out)
        create("auto").gh_rhs(u, gammas, inv, out)
        torch.cuda.synchronize()
        stepper.close()
    assert torch.equal(u, after) and torch.equal(out, rhs)
