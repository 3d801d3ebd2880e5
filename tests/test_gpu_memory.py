"""Kept device workspaces and the pinned read-back (ngi_mem): films of every
size come back whole, one call's leftovers never show in the next, and
threads may render at once.
"""
import ctypes
import os
import threading
import time

import numpy as np
import pytest

import nanogi_amd as ngi
import oracle

pytestmark = pytest.mark.gpu


def _params(renderer, w, h, spp=1, **kw):
    return ngi.default_params(renderer=renderer, width=w, height=h, sampling=ngi.SAMPLING_PER_PIXEL, spp=spp, max_num_vertices=5,
                              rr_depth=3, seed=11, **kw)


# The read-back goes in slots of 1 MiB (43,690.7 pixels) through a ring of 16.
@pytest.mark.parametrize("w,h", [(1, 1), (257, 170), (43691, 1), (1024, 700)])
@pytest.mark.parametrize("precision", [ngi.PRECISION_FP32_FP64ACC, ngi.PRECISION_FP32_ALL])
def test_film_sizes_against_oracle(w, h, precision):
    s = ngi.Scene.generate(ngi.GEN_CORNELL, 1, 1.0)
    p = _params("ptdirect", w, h, precision=precision)
    film, st = ngi.render(s, p)
    ref = oracle.render(s, p)
    assert st["samples"] == w * h
    rel = np.abs(film - ref).max(axis=2) / (np.abs(ref).max(axis=2) + 1e-3)
    assert (rel < 2e-4).mean() >= 0.97


def test_variance_is_that_of_the_batches():
    s = ngi.Scene.generate(ngi.GEN_CORNELL, 1, 1.0)
    p = _params("pt", 300, 260)
    batches = []
    for k in range(3):
        se = ngi.Session(s, p)
        if k:
            se.render(k)        # samples 0..k-1, then the batch's own
        before = se.film() * k
        se.render(1)
        batches.append(se.film() * (k + 1) - before)
        se.close()
    se = ngi.Session(s, p)
    for _ in range(3):
        se.render_batch(1)
    film, var = se.film(variance=True)
    b = np.stack(batches)
    # FP64 sums of FP32 contributions: differences of films cost about 1e-15 of the largest value.
    tol = 1e-12 * max(1.0, np.abs(b).max()) ** 2
    assert np.abs(film - b.mean(axis=0)).max() <= tol
    assert np.abs(var - b.var(axis=0, ddof=1) / 3).max() <= tol


def test_leftovers_of_other_calls_do_not_show():
    a = ngi.Scene.generate(ngi.GEN_CORNELL, 1, 1.0)
    b = ngi.Scene.generate(ngi.GEN_NAVE, 2, 1.0)   # large enough for the 512-record shadow rings
    jobs = []
    for scene in (a, b):
        for renderer in ("pt", "ptdirect", "ltdirect", "bdpt"):
            for w, h, spp in ((96, 64, 2), (31, 17, 1)):
                jobs.append((scene, _params(renderer, w, h, spp)))
        jobs.append((scene, _params("ptdirect", 64, 48, 2, engine=ngi.ENGINE_WAVEFRONT)))
    first = [ngi.render(s, p)[0] for s, p in jobs]
    for i in np.random.default_rng(0).permutation(len(jobs)):
        again = ngi.render(*jobs[i])[0]
        assert np.abs(again - first[i]).max() <= 1e-9 * max(1.0, np.abs(first[i]).max())
    g = np.random.default_rng(1).normal(size=(48, 64, 3))
    p = _params("ptdirect", 64, 48, 4)
    gR, gL, _ = ngi.render_adjoint(a, p, g)
    ngi.render(b, _params("pt", 200, 100))
    gR2, gL2, _ = ngi.render_adjoint(a, p, g)
    assert np.allclose(gR, gR2, rtol=1e-9, atol=1e-12) and np.allclose(gL, gL2, rtol=1e-9, atol=1e-12)


def test_threads_render_at_once():
    sizes = [(40, 30), (300, 200), (640, 480), (17, 9)]
    scenes = [ngi.Scene.generate(ngi.GEN_BATCH_ROOM, 20 + i, 1.0, 200) for i in range(4)]
    params = [_params("ptdirect", w, h, 2) for w, h in sizes]
    rays = ngi.make_rays(np.full((50, 3), 0.5), np.random.default_rng(3).normal(size=(50, 3)))
    want = [(ngi.render(s, p)[0], s.trace(rays)) for s, p in zip(scenes, params)]
    bad = []

    def work(i):
        for _ in range(6):
            film = ngi.render(scenes[i], params[i])[0]
            hits = scenes[i].trace(rays)
            if np.abs(film - want[i][0]).max() > 1e-9 * np.abs(want[i][0]).max() or not np.array_equal(hits, want[i][1]):
                bad.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_results_without_pinned_memory(monkeypatch):
    """Where no host memory can be pinned (NGI_PINNED=0), films, variances,
    statistics and hits come back all the same, bit for bit."""
    s = ngi.Scene.generate(ngi.GEN_CORNELL, 1, 1.0)
    rays = ngi.make_rays(np.full((70000, 3), 0.5), np.random.default_rng(3).normal(size=(70000, 3)))
    sessions = []
    for precision in (ngi.PRECISION_FP32_FP64ACC, ngi.PRECISION_FP32_ALL):
        se = ngi.Session(s, _params("ptdirect", 300, 200, precision=precision))
        for _ in range(3):
            se.render_batch(1)
        sessions.append(se)
    b = ngi.Batch([s], [_params("ptdirect", 300, 200)], ngi.batch_opts(block_size=128, blocks_per_cu=2))
    b.render(0)
    b.sync()

    def results():
        out = [b.film(0)]
        for se in sessions:
            st = se.stats()
            out += [*se.film(variance=True), np.array([st["samples"], st["extension_rays"], st["shadow_rays"]])]
        for n in (50, 70000):   # hits of more than 1 MiB among them
            out.append(s.trace(rays[:n]).view(np.uint32))
        return out

    want = results()
    monkeypatch.setenv("NGI_PINNED", "0")
    for x, y in zip(want, results()):
        assert np.abs(x).max() > 0 and np.array_equal(x, y)
    film, st = ngi.render(s, _params("ptdirect", 300, 200))
    assert st["samples"] == 60000 and np.abs(film - want[0]).max() <= 1e-9 * np.abs(film).max()
    b.close()
    for se in sessions:
        se.close()


def test_no_thread_waits_for_anothers_render():
    """A small query behind a long render on its scene's stream keeps no other
    thread's statistics and films waiting."""
    rays = ngi.make_rays(np.full((50, 3), 0.5), np.random.default_rng(3).normal(size=(50, 3)))
    scenes = [ngi.Scene.generate(ngi.GEN_CORNELL, 1, 1.0) for _ in range(5)]
    sessions = [ngi.Session(s, _params("pt", 64, 64)) for s in scenes[1:]]
    for s, se in zip(scenes[1:], sessions):
        s.trace(rays)
        se.render(1)
        se.film()
    long = _params("ptdirect", 256, 256)
    long.paths_in_flight = 256   # one block: about a second, and room for the others' kernels
    ends = {}

    def query():
        scenes[0].trace(rays)
        ends["query"] = time.perf_counter()

    def read(i):
        sessions[i].stats()
        sessions[i].film()
        scenes[1 + i].trace(rays)
        ends[i] = time.perf_counter()

    se = ngi.Session(scenes[0], long)
    se.render(1)
    se.sync()
    spp = 4
    while True:   # as many samples as take half a second
        t0 = time.perf_counter()
        se.render(spp)
        se.sync()
        if time.perf_counter() - t0 > 0.5:
            break
        spp *= 2
    start = time.perf_counter()
    se.render(spp)
    threads = [threading.Thread(target=query)]
    threads[0].start()
    time.sleep(0.1)   # the query has been enqueued
    threads += [threading.Thread(target=read, args=(i,)) for i in range(4)]
    for t in threads[1:]:
        t.start()
    for t in threads:
        t.join()
    se.close()
    # Streams may share a hardware queue with the long render: not all four.
    assert min(ends[i] for i in range(4)) < start + 0.75 * (ends["query"] - start)
    for x in sessions:
        x.close()


def test_one_scene_after_another_costs_no_fresh_pages():
    """A film of 34 MB comes back as fast from the only scene of the process,
    made anew each time, as beside a scene that stays."""
    p = _params("pt", 1400, 1000)

    def upper_quartile(times=16):
        took = []
        for i in range(times):
            s = ngi.Scene.generate(ngi.GEN_CORNELL, 1 + i, 1.4)
            se = ngi.Session(s, p)
            se.render(1)
            se.sync()
            t0 = time.perf_counter()
            se.film()
            took.append(time.perf_counter() - t0)
            se.close()
            s.close()
        return sorted(took)[times * 3 // 4]

    for attempt in range(2):   # the machine may be busy; with fresh pages 2.5 times, with kept ones at most 1.3
        alone = upper_quartile()
        keeper = ngi.Scene.generate(ngi.GEN_CORNELL, 1, 1.0)
        ngi.render(keeper, p)
        beside = upper_quartile()
        keeper.close()
        if alone < 1.7 * beside:
            return
    assert alone < 1.7 * beside


def test_kept_workspaces_follow_the_sessions_in_use():
    """After a session of another size has filled the kept workspaces, those of
    the sessions in use replace them: the second one allocates nothing.  What is
    kept stays within its bound."""
    scene = ngi.Scene.generate(ngi.GEN_CORNELL, 1, 1.0)
    hip = ctypes.CDLL("libamdhip64.so.7", mode=os.RTLD_NOLOAD)   # the runtime that the library uses

    def free():
        left, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(left), ctypes.byref(total)) == 0
        return left.value

    def session(w, h):
        se = ngi.Session(scene, _params("pt", w, h))
        for _ in range(2):
            se.render_batch(1)
        se.sync()
        return se

    session(64, 64).close()   # what the first render allocates once
    before = free()
    session(3600, 2400).close()     # four films of 207 MB
    for _ in range(2):
        session(1500, 1000).close()   # four of 36 MB
        session(800, 500).close()     # four of 9.6 MB
        assert before - free() <= 512 << 20
    for w, h in ((1500, 1000), (800, 500)):
        idle = free()
        se = session(w, h)
        assert free() == idle
        se.close()
    scene.close()
    assert free() >= before


@pytest.mark.parametrize("precision", [ngi.PRECISION_FP32_FP64ACC, ngi.PRECISION_FP32_ALL])
@pytest.mark.parametrize("pixels", [682, 683, 1365, 1366, 10922, 10923, 43690, 43691, 349525, 349526])
def test_films_are_the_same_by_either_way_back(monkeypatch, pixels, precision):
    """Films around the sizes at which their way back changes (16 and 256 KiB, 1
    and 4 MiB of pixels) have the bits of the runtime's copy, scaled."""
    s = ngi.Scene.generate(ngi.GEN_CORNELL, 1, 1.0)
    se = ngi.Session(s, _params("pt", pixels, 1, precision=precision))
    se.render(3)
    film = se.film()
    monkeypatch.setenv("NGI_PINNED", "0")
    assert film.max() > 0 and np.array_equal(film, se.film())
    se.close()


@pytest.mark.parametrize("n", [1365, 1366, 98304, 98305, 150000, 600000])
def test_hits_are_the_same_by_either_way_back(monkeypatch, n):
    """Hits around the sizes at which their way back changes (rays in mapped
    memory, 1.5 MiB of hits) and well above them: each way, the same bits."""
    s = ngi.Scene.generate(ngi.GEN_BATCH_ROOM, 1, 1.0, 500)
    rays = ngi.make_rays(np.full((n, 3), 0.5), np.random.default_rng(n).normal(size=(n, 3)))
    hits = s.trace(rays)
    monkeypatch.setenv("NGI_PINNED", "0")
    assert (hits["tri"] != ngi.MISS).any() and np.array_equal(hits.view(np.uint32), s.trace(rays).view(np.uint32))
