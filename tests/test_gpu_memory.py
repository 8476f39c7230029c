"""Memory that outlives a call: one scratch buffer per stream and context, and
the cache of the solve's buffers.  What is checked is what can go wrong:
calls on two streams at once, a buffer that has to grow under work in flight,
captured calls replayed beside eager ones, factors kept across a later
factorization, the bound of what stays allocated."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
SEED = 42


def _residual_case(ctx, n, seed):
    import torch
    d = torch.empty(n, dtype=torch.float64, device="cuda")
    ctx.gen_diag(n, seed, 0, n, d)
    x = torch.from_numpy(np.random.default_rng(seed).standard_normal(n)).cuda()
    y = torch.zeros(n, dtype=torch.float64, device="cuda")
    ctx.otf_gemv(n, seed, d, 1.0, x, y)
    torch.cuda.synchronize()
    return d, x, y


def test_two_streams_do_not_share_scratch(ctx):
    import torch
    sizes = [(3000, 1), (2000, 2)]
    cases = [(n, s) + _residual_case(ctx, n, s) for n, s in sizes]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    outs = [[], []]
    for _ in range(20):
        for k, (n, s, d, x, _) in enumerate(cases):
            with torch.cuda.stream(streams[k]):
                y = torch.zeros(n, dtype=torch.float64, device="cuda")
                ctx.otf_gemv(n, s, d, 1.0, x, y)
                outs[k].append(y)
    torch.cuda.synchronize()
    for k, case in enumerate(cases):
        for y in outs[k]:
            assert torch.equal(y, case[4])


def test_scratch_grows_under_work_in_flight(ctx):
    import torch
    cases = [(n, 7) + _residual_case(ctx, n, 7) for n in (500, 3000, 9000, 20000)]
    st = torch.cuda.Stream()
    outs = []
    with torch.cuda.stream(st):
        for n, s, d, x, _ in cases:
            y = torch.zeros(n, dtype=torch.float64, device="cuda")
            ctx.otf_gemv(n, s, d, 1.0, x, y)
            outs.append(y)
    torch.cuda.synchronize()
    for y, case in zip(outs, cases):
        assert torch.equal(y, case[4])


def test_captured_calls_have_scratch_of_their_own(ctx):
    import torch
    n = 3000
    d, x, want = _residual_case(ctx, n, 3)
    d2, x2, want2 = _residual_case(ctx, n, 4)
    y, y2 = torch.empty_like(want), torch.empty_like(want)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y.zero_()
        ctx.otf_gemv(n, 3, d, 1.0, x, y)
    for _ in range(4):
        y.fill_(9.0)
        g.replay()
        y2.zero_()
        ctx.otf_gemv(n, 4, d2, 1.0, x2, y2)
        torch.cuda.synchronize()
        assert torch.equal(y, want) and torch.equal(y2, want2)


def test_kept_factors_survive_a_factorization(ctx):
    import torch
    n, b = 2048, 512
    ctx.solve(n, b, fmt="e4m3", keep_factors=True)
    lu = ctx.solution_factors(n)
    x = ctx.solution_x(n)
    A = torch.from_numpy(np.random.default_rng(1).uniform(-0.5, 0.5, (n, n)).astype(np.float32)).cuda()
    A.diagonal().fill_(n)
    ctx.factor(n, b, A, n, fmt="e4m3")
    assert np.array_equal(ctx.solution_factors(n), lu)
    assert np.array_equal(ctx.solution_x(n), x)
    ctx.release()
    import hplai
    with pytest.raises(hplai.HplaiError):
        ctx.solution_x(n)


def test_what_stays_allocated_is_bounded(ctx):
    """A sixth of the device at most is kept between solves, whatever ran."""
    import torch
    torch.cuda.empty_cache()
    total = torch.cuda.mem_get_info()[1]
    for n, fmt in ((65536, "f16"), (98304, "e4m3"), (32768, "e4m3")):
        free0 = torch.cuda.mem_get_info()[0]
        r = ctx.solve(n, 512, fmt=fmt, outer=16)
        assert r["converged"]
        ctx.release()
        assert torch.cuda.mem_get_info()[0] >= min(free0, total) - total // 6 - (1 << 30)
    assert total - torch.cuda.mem_get_info()[0] <= total // 6 + (8 << 30)


def test_large_scratch_takes_what_the_cache_holds(ctx):
    """A call whose scratch is allocated in stream order (3.2 GB of partial
    sums), with the device full but for 2 GB and the solve's idle buffers."""
    import torch
    n = 900000
    torch.cuda.empty_cache()
    d, x, want = _residual_case(ctx, n, 5)
    ctx.solve(65536, 512, fmt="e4m3", outer=16)            # 18 GB of buffers, kept idle
    torch.cuda.synchronize()
    y = torch.zeros_like(want)
    hog = torch.empty(torch.cuda.mem_get_info()[0] - (2 << 30), dtype=torch.uint8, device="cuda")
    try:
        assert torch.cuda.mem_get_info()[0] < 3 << 30
        ctx.otf_gemv(n, 5, d, 1.0, x, y)
        torch.cuda.synchronize()
    finally:
        del hog
        torch.cuda.empty_cache()
    assert torch.equal(y, want)


def test_trim_gives_everything_back(ctx):
    """After a trim the device has what it had before: for another allocator
    (torch's here) that cannot reach the library's idle memory."""
    import torch
    n = 20000
    d, x, want = _residual_case(ctx, n, 6)
    torch.cuda.empty_cache()
    ctx.trim()
    free0 = torch.cuda.mem_get_info()[0]
    r = ctx.solve(65536, 512, fmt="e4m3", outer=16, keep_factors=True)
    sol = ctx.solution_x(65536)
    y = torch.zeros_like(want)
    ctx.otf_gemv(n, 6, d, 1.0, x, y)
    ctx.trim()
    assert torch.equal(y, want)
    assert np.array_equal(ctx.solution_x(65536), sol)      # kept until they are released
    ctx.release()
    assert torch.cuda.mem_get_info()[0] < free0 - (15 << 30)   # A, 16 GiB, is idle now
    ctx.trim()
    torch.cuda.empty_cache()
    assert torch.cuda.mem_get_info()[0] >= free0 - (64 << 20)
    assert ctx.solve(65536, 512, fmt="e4m3", outer=16)["checksum"] == r["checksum"]


def _busy(stream, ms=300):
    """A spinning kernel of about `ms` on the stream, and an event behind it."""
    import torch
    with torch.cuda.stream(stream):
        torch.cuda._sleep(1000)                              # loaded before it is timed
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        torch.cuda._sleep(1 << 20)
        b.record()
    stream.synchronize()
    with torch.cuda.stream(stream):
        torch.cuda._sleep(int((1 << 20) * ms / max(a.elapsed_time(b), 1e-3)))
        done = torch.cuda.Event()
        done.record()
    return done


def test_a_growing_buffer_does_not_wait_for_its_stream():
    import hplai
    import torch
    cases = [(n, 7) + _residual_case(hplai.Context(0), n, 7) for n in (500, 3000, 9000, 30000)]
    c = hplai.Context(0)
    for first in (1, 0):                                     # once with the kernels loaded
        st = torch.cuda.Stream()
        outs = []
        done = _busy(st)
        with torch.cuda.stream(st):
            for n, s, d, x, _ in cases:
                y = torch.zeros(n, dtype=torch.float64, device="cuda")
                c.otf_gemv(n, s, d, 1.0, x, y)
                outs.append(y)
        waited = done.query()
        st.synchronize()
        for y, case in zip(outs, cases):
            assert torch.equal(y, case[4])
        assert first or not waited
    c.close()


def test_streams_past_the_bound_do_not_wait():
    """Three streams with buffers of 512 MiB: the third's call does not wait for
    the other two, whose buffers stay theirs."""
    import hplai
    import torch
    c = hplai.Context(0)
    n, m, k = 4096, 4096, 1 << 15                            # (n + m) k 2 bytes: 512 MiB
    g = torch.Generator(device="cuda").manual_seed(1)
    a = torch.rand(k, n, generator=g, device="cuda").half()
    b = torch.rand(m, k, generator=g, device="cuda").half()
    want = torch.zeros(m, n, device="cuda")
    c.gemmschur_f16(n, m, k, a, n, b, k, want, n)
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(3)]
    outs = [torch.zeros(m, n, device="cuda") for _ in range(3)]
    torch.cuda.synchronize()
    done = [_busy(st, 500) for st in streams]
    for st, out in zip(streams, outs):
        c.gemmschur_f16(n, m, k, a, n, b, k, out, n, stream=st)
    assert not any(e.query() for e in done)
    torch.cuda.synchronize()
    for out in outs:
        assert torch.equal(out, want)
    c.close()


def test_first_call_on_a_stream_beside_another_streams_capture():
    """While a stream of the thread is captured (global mode), a call on another
    stream may not use what such a capture forbids."""
    import hplai
    import torch
    c = hplai.Context(0)
    n = 3000
    d, x, want = _residual_case(c, n, 3)
    y, z = torch.zeros_like(want), torch.zeros_like(want)
    other = torch.cuda.Stream()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, capture_error_mode="global"):
        z.add_(1.0)
        c.otf_gemv(n, 3, d, 1.0, x, y, stream=other)
    other.synchronize()
    assert torch.equal(y, want)
    for k in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert (z == k + 1).all()
    c.close()
