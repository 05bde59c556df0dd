"""Serving loop on the GPU: continuous batching, admission by device memory, failure handling.

Each request's result is the same alone (hexo_price) and in the mix (served in whatever batch it
landed in), bit for bit: its tiles, reduction order and RNG stream depend only on the request.
"""
import dataclasses

import numpy as np
import pytest

import hestonexotics_amd as H
import time
from hestonexotics_amd import workloads as W

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)


def small_trace(n=40, seed=3):
    reqs, arr = W.c4(rate=400.0, duration_s=n / 400.0 * 1.2, seed=seed, path_scale=0.005)
    reqs = reqs[:n]
    arr = arr[:n]
    # every kernel class in the stream: some requests with the martingale correction, some with
    # the control-variate and geometric blocks, one in FP64
    for i, r in enumerate(reqs):
        if i % 5 == 1:
            r.flags |= H.MARTINGALE
        if i % 7 == 2 and r.payoffs & H.ASIAN:
            r.payoffs |= H.ASIAN_GEO_CV | H.GEO_ASIAN
    if len(reqs) > 3:
        reqs[3].precision = H.FP64
    return reqs, arr


def test_served_equals_alone(ctx):
    reqs, arr = small_trace()
    say("gpu serving: trace of", len(reqs), "requests")
    ctx.server_start(streams=3)
    try:
        rc, p, s, infos = ctx.run_trace(reqs, arr)
        st = ctx.server_stats()
    finally:
        ctx.server_stop()
    assert rc == 0, rc
    assert st["completed"] == len(reqs)
    o = 0
    for r, inf in zip(reqs, infos):
        p1, s1 = ctx.price(r)
        n = r.n_outputs
        np.testing.assert_array_equal(p[o:o + n], p1)
        np.testing.assert_array_equal(s[o:o + n], s1)
        assert inf["status"] == 0 and inf["done_s"] >= inf["launch_s"] >= inf["admit_s"] >= inf["arrival_s"]
        o += n
    say("  batches:", st["batches"], "max batch:", max(i["batch_size"] for i in infos))


def test_submit_wait_poll_cancel(ctx):
    reqs, _ = small_trace(8, seed=5)
    ctx.server_start(streams=1)
    try:
        tickets = [ctx.submit(r) for r in reqs]
        # the last tickets are likely still queued behind the first batch; cancel one if so
        cancelled = None
        for t in reversed(tickets):
            try:
                ctx.cancel(t)
                cancelled = t
                break
            except H.HexoError:
                continue
        # a NaN timeout is refused and leaves the ticket; one beyond the clock's range waits forever
        with pytest.raises(H.HexoError, match="NaN"):
            ctx.wait(tickets[0], reqs[0].n_outputs, timeout_s=float("nan"))
        for i, (r, t) in enumerate(zip(reqs, tickets)):
            if t == cancelled:
                with pytest.raises(H.HexoError):
                    ctx.wait(t, r.n_outputs)
                continue
            p, s, info = ctx.wait(t, r.n_outputs, timeout_s=1e300 if i == 0 else 60.0)
            p1, _ = ctx.price(r)
            np.testing.assert_array_equal(p, p1)
        with pytest.raises(H.HexoError):
            ctx.poll(10**9)
    finally:
        ctx.server_stop()


def test_admission_refused_by_budget(ctx):
    big = W.c1(n_paths=5_000_000, precision=H.FP32)
    big.strikes = [list(np.linspace(50, 150, 400))]
    ctx.server_start(memory_budget_bytes=1 << 20, streams=1)
    try:
        with pytest.raises(H.HexoError) as e:
            ctx.submit(big)
        assert e.value.code == -5  # HEXO_ERR_ADMISSION
        small = W.c1(n_paths=1000, precision=H.FP32)
        t = ctx.submit(small)
        p, s, _ = ctx.wait(t, small.n_outputs, timeout_s=60.0)
        assert np.isfinite(p).all()
    finally:
        ctx.server_stop()


def test_malformed_request_rejected(ctx):
    bad = W.c1(n_paths=1000)
    bad.steps = 0
    ctx.server_start(streams=1)
    try:
        with pytest.raises(H.HexoError) as e:
            ctx.submit(bad)
        assert e.value.code == -1
    finally:
        ctx.server_stop()


def test_injected_launch_failure_is_reported_and_server_recovers(ctx):
    reqs, _ = small_trace(4, seed=9)
    ctx.server_start(streams=1, max_batch=1)
    try:
        ctx.inject_fault(0, 1)
        tickets = [ctx.submit(r) for r in reqs]
        codes = []
        for r, t in zip(reqs, tickets):
            try:
                ctx.wait(t, r.n_outputs, timeout_s=60.0)
                codes.append(0)
            except H.HexoError as e:
                codes.append(e.code)
        assert codes[0] == -10 and all(c == 0 for c in codes[1:]), codes
    finally:
        ctx.server_stop()


def test_stop_while_clients_submit_and_wait(ctx):
    """hexo_server_stop while four threads submit and wait (ctypes releases the GIL, so the calls
    overlap): every call returns a status, each collected result equals the request priced alone,
    and calls after the stop report that the server is not running."""
    import dataclasses
    import threading
    import time
    say("gpu serving stop under concurrent clients")
    base = W.c1(n_paths=2000)
    ref, _ = ctx.price(base)
    ctx.server_start(streams=2)
    stop = threading.Event()
    results = []
    lock = threading.Lock()

    def client():
        req = dataclasses.replace(base)  # each thread keeps its own argument arrays alive
        while not stop.is_set():
            try:
                t = ctx.submit(req)
            except H.HexoError as e:
                with lock:
                    results.append(("submit", e.code, None))
                if e.code == -9:  # HEXO_ERR_STATE: the server has stopped
                    return
                continue
            try:
                p, _, _ = ctx.wait(t, req.n_outputs)
                with lock:
                    results.append(("wait", 0, bool(np.array_equal(p, ref))))
            except H.HexoError as e:
                with lock:
                    results.append(("wait", e.code, None))

    threads = [threading.Thread(target=client) for _ in range(4)]
    for th in threads:
        th.start()
    time.sleep(0.5)
    ctx.server_stop()
    stop.set()
    for th in threads:
        th.join(timeout=60)
    assert not any(th.is_alive() for th in threads)
    done = [r for r in results if r[0] == "wait" and r[1] == 0]
    say(f"  {len(done)} results collected, {len(results) - len(done)} calls refused")
    assert done and all(r[2] for r in done)
    assert all(r[1] in (0, -9) for r in results), sorted(set(r[1] for r in results))
    with pytest.raises(H.HexoError):
        ctx.submit(base)


def test_small_requests_pass_a_large_one(ctx):
    """A large request (8e9 path-steps, about 18 ms alone) submitted first runs in a batch of its
    own on part of the GPU; tiny requests submitted right after it run beside it and finish first
    (sharing its batch, they would finish with it). Results equal the requests priced alone."""
    say("gpu serving: small requests pass a large one")
    big = H.Request(v0=0.04, theta=0.04, rho=-0.7, kappa=2.0, sigma=0.3, S0=100.0, expiries=[2.0],
                    strikes=[[100.0]], steps=4000, n_paths=2_000_000, seed=3, precision=H.FP32)
    tiny = [dataclasses.replace(big, steps=10, n_paths=640, seed=10 + i) for i in range(6)]
    ctx.server_start(streams=2)
    try:
        tb = ctx.submit(big)
        tt = [ctx.submit(r) for r in tiny]
        out_t = [ctx.wait(t, r.n_outputs) for t, r in zip(tt, tiny)]
        p_big, _, info_big = ctx.wait(tb, big.n_outputs)
    finally:
        ctx.server_stop()
    done_tiny = max(i["done_s"] for _, _, i in out_t)
    say(f"  large done after {1e3 * (info_big['done_s'] - info_big['arrival_s']):.1f} ms, tiny after "
        f"{1e3 * (done_tiny - info_big['arrival_s']):.1f} ms; large batch size {info_big['batch_size']}")
    assert info_big["batch_size"] == 1
    assert done_tiny < info_big["done_s"]
    for r, (p, _, _) in zip(tiny, out_t):
        np.testing.assert_array_equal(p, ctx.price(r)[0])
    np.testing.assert_array_equal(p_big, ctx.price(big)[0])


@pytest.mark.parametrize("flags", [0, H.MARTINGALE])
@pytest.mark.parametrize("params", [dict(kappa=2.0, sigma=0.3), dict(kappa=0.5, sigma=0.9)])
def test_small_requests_pass_a_large_martingale_one(ctx, flags, params):
    """As above for a large request with the martingale step, whose kernel holds 4 waves per SIMD: tiny
    requests (of both FP32 steps) run beside it from the start, not when its grid drains at the end."""
    say("gpu serving: small requests pass a large martingale one", flags, params)
    big = H.Request(v0=0.04, theta=0.04, rho=-0.7, S0=100.0, expiries=[2.0], strikes=[[100.0]], steps=4000,
                    n_paths=2_000_000, seed=3, flags=H.MARTINGALE, precision=H.FP32, **params)
    tiny = [dataclasses.replace(big, steps=10, n_paths=640, seed=10 + i, flags=flags) for i in range(6)]
    ctx.server_start(streams=2)
    try:
        tb = ctx.submit(big)
        tt = [ctx.submit(r) for r in tiny]
        out_t = [ctx.wait(t, r.n_outputs) for t, r in zip(tt, tiny)]
        _, _, info_big = ctx.wait(tb, big.n_outputs)
    finally:
        ctx.server_stop()
    done_tiny = max(i["done_s"] for _, _, i in out_t) - info_big["arrival_s"]
    done_big = info_big["done_s"] - info_big["arrival_s"]
    say(f"  large done after {1e3 * done_big:.1f} ms, tiny after {1e3 * done_tiny:.1f} ms")
    assert done_tiny < 0.5 * done_big
    for r, (p, _, _) in zip(tiny, out_t):
        np.testing.assert_array_equal(p, ctx.price(r)[0])


def test_cancel_of_a_ticket_that_does_not_fit_yet(ctx):
    """A request that finds the arena's free space in two pieces goes back to the queue until a batch
    completes; a cancel that arrives while its batch is being tried takes effect. The arena: 24 MB of
    a finished request, 16 MB of a running one, 24 MB free, a request of 32 MB waiting."""
    def req(tiles, steps, n_strikes=100, **kw):
        return H.Request(v0=0.04, theta=0.04, rho=-0.7, kappa=2.0, sigma=0.3, S0=100.0, expiries=[1.0],
                         strikes=[list(np.linspace(70.0, 130.0, n_strikes))], steps=steps, n_paths=64 * tiles,
                         payoffs=H.ASIAN, **kw)
    first = req(15_000, 1000, seed=1, precision=H.FP32)       # about 2 ms, in the arena's first 24 MB
    running = req(10_000, 100_000, seed=2, precision=H.FP64)  # about half a second, behind it
    waiting = req(20_000, 2, seed=3, precision=H.FP32)
    say("gpu serving: cancel while a batch is tried")
    ctx.server_start(memory_budget_bytes=64_500_000, streams=3)
    try:
        tf, tr = ctx.submit(first), ctx.submit(running)
        ctx.wait(tf, first.n_outputs)
        for _ in range(20):
            t = ctx.submit(waiting)
            time.sleep(0.002)
            ctx.cancel(t)
            with pytest.raises(H.HexoError) as e:
                ctx.wait(t, waiting.n_outputs)
            assert e.value.code == -7  # HEXO_ERR_CANCELLED
        assert not ctx.poll(tr), "the running request ended before the cancels"
        assert ctx.server_stats()["cancelled"] == 20
        ctx.wait(tr, running.n_outputs)
    finally:
        ctx.server_stop()
