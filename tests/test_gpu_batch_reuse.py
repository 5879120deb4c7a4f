"""A batch and a context used on after a call that failed, that was empty or
that was unusually large: what a call leaves behind must not reach the next.
And a server's first requests, which find its buffers as it was made."""
import ctypes as C
import threading

import numpy as np
import pytest

import cases
from part_conc_spt_abc_amd import _abi
from part_conc_spt_abc_amd.gpu import Context, Server
from part_conc_spt_abc_amd.model import prior_record, proposals_array

pytestmark = pytest.mark.gpu


def population(n_pop, log10c):
    rng = np.random.default_rng(n_pop)
    theta = np.vstack([rng.uniform(0.5, 2.5, (2, n_pop)), np.full((2, n_pop), log10c), np.full((1, n_pop), 2.0)])
    return theta, np.cumsum(np.full(n_pop, 1.0 / n_pop)), np.array([0.1, 0.1, 0.0, 0.0, 0.1])


def simulate(ctx, props, f, n, seed):
    dist, tracks = np.empty(len(props)), np.empty(len(props), np.uint32)
    p = lambda a: a.ctypes.data_as(C.c_void_p)  # noqa: E731
    arr = proposals_array(props)
    _abi.check(ctx.lib.pcs_simulate(ctx.h, C.cast(arr, C.c_void_p), len(props), p(f), p(n), len(f), seed,
                                    _abi.PCS_MODE_BATCHED, p(dist), None, p(tracks)), "pcs_simulate")
    return dist, tracks


def test_propose_after_a_failed_propose(gpu_lib):
    """A batch whose graph is captured; a proposal step of more trials that is
    refused after the buffers have grown (more than 2^32 tiles); then the same
    number of trials, which need no larger arena. Its graph is a new one."""
    model = cases.headline_model(n_k=60, n_de=40)
    obs = np.zeros((60, 40), np.uint32)
    obs[4, 7] = 3
    few, many = 400, 20000
    with Context(model, obs) as ctx:
        b = ctx.batch()
        b.propose(prior_record(model, (0.1, 5.0), (8.0, 10.0), (0.5, 4.0)), *population(50, 9.7), few,
                  np.full((few, 1), 300, np.uint32), 3)
        for seed in (1, 2, 3):  # direct, captured, replayed
            b.run(seed)
            b.read()
        assert b.arena()[0] > 0
        frames = np.full((many, 1), 12, np.uint32)
        with pytest.raises(_abi.PcsError, match="more than 2\\^32 - 1") as e:
            b.propose(prior_record(model, (0.1, 5.0), (8.0, 12.83), (0.5, 4.0)), *population(50, 12.82), many, frames, 4)
        assert e.value.code == _abi.PCS_EINVAL
        with pytest.raises(_abi.PcsError):
            b.run(5)
        pr = prior_record(model, (0.1, 5.0), (5.0, 10.0), (0.5, 4.0))
        c = ctx.batch()
        got = []
        for q in (b, c):
            q.propose(pr, *population(50, 7.0), many, frames, 6)
            for seed in (7, 8):
                q.run(seed)
                _, tracks, _ = q.read()
                got.append((tracks, q.read_exact()))
        assert int(got[0][0].sum()) > 0
        assert all(np.array_equal(x, y) for k in (0, 1) for x, y in zip(got[k], got[k + 2]))
        c.close()
        b.close()


def test_overlapping_one_shot_calls(gpu_lib):
    """Calls of pcs_simulate that overlap on one context: each has a batch of
    its own, the kept one goes to one of them only."""
    model = cases.headline_model(n_k=60, n_de=40)
    obs = np.zeros((60, 40), np.uint32)
    obs[4, 7] = 3
    loads = [cases.draw_proposals(model, k, np.random.default_rng(k), frames_choices=(30, 90), c_range=(5e7, 3e9))
             for k in (1, 2, 7, 40, 3, 90)]
    with Context(model, obs) as ctx:
        want = [simulate(ctx, *w, 5) for w in loads]
        wrong = []

        def calls(i):
            try:
                for k in range(30):
                    j = (i + k) % len(loads)
                    d, t = simulate(ctx, *loads[j], 5)
                    if not (np.array_equal(d, want[j][0]) and np.array_equal(t, want[j][1])):
                        wrong.append((i, k))
            except Exception as e:
                wrong.append((i, e))

        threads = [threading.Thread(target=calls, args=(i,)) for i in range(6)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not wrong, wrong


def test_no_simulations(gpu_lib):
    """A batch of no simulations runs and is read in every form, before the
    batch has held any and after."""
    model = cases.headline_model(n_k=60, n_de=40)
    empty = ([], np.empty(0, np.uint32), np.empty(0, np.uint32))
    some = cases.draw_proposals(model, 3, np.random.default_rng(1), frames_choices=(30,), c_range=(5e8, 3e9))
    with Context(model) as ctx:
        b = ctx.batch()
        for load in (empty, some, empty):
            b.load(*load)
            for mode in range(4):
                b.run(3, mode)
                dist, tracks, H = b.read(hist=True)
                assert len(dist) == len(tracks) == len(H) == len(b.read_exact()) == len(load[0])
                assert b.overflow_reruns() == 0 and (not len(tracks) or tracks.sum() > 0)
        b.close()


def free_bytes():
    free, total = C.c_size_t(0), C.c_size_t(0)
    assert C.CDLL("libamdhip64.so.7").hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("particles,videos", [(0, 1 << 24), (1, 1 << 21)])
def test_large_one_shot_leaves_no_buffers(gpu_lib, particles, videos):
    """A call of one simulation with very many videos, empty or not: what the
    context keeps of it stays within what pcs_abi.h states (a quarter is left
    for the allocator)."""
    model = cases.headline_model(n_k=60, n_de=40)
    p, _, _ = cases.fixed_proposal(model, [1], [2])
    with Context(model) as ctx:
        small = np.ones(1, np.uint32)
        simulate(ctx, [p], small, small, 1)
        before = free_bytes()
        p.n_videos = videos
        simulate(ctx, [p], np.full(videos, 2, np.uint32), np.full(videos, particles, np.uint32), 1)
        assert before - free_bytes() <= 1.25 * (64 << 20)
        p.n_videos = 1
        simulate(ctx, [p], small, small, 1)


@pytest.mark.parametrize("device_loop", [False, True])
def test_first_requests_of_a_server(gpu_lib, device_loop):
    model = cases.headline_model(n_k=60, n_de=40)
    obs = np.zeros((60, 40), np.uint32)
    obs[4, 7] = 3
    props, f, n = cases.draw_proposals(model, 9, np.random.default_rng(2), frames_choices=(30, 90), c_range=(5e7, 3e9))
    with Context(model, obs) as ctx:
        b = ctx.batch()
        b.load(props, f, n)
        b.run(5)
        _, tracks, _ = b.read()
        exact = b.read_exact()
        b.close()
    for p in props:
        p.first_video = 0
    for _ in range(4):
        srv = Server(arena_bytes=1 << 24, max_inflight=16, max_videos=1, device_loop=device_loop)
        sid = srv.add_system(model, obs)
        for i, p in enumerate(props):
            assert srv.submit(i, sid, p, f[i:i + 1], n[i:i + 1], 5)
        got = {}
        for _ in range(20000):
            got.update((c.tag, (c.status, int(c.tracks), int(c.exact))) for c in srv.poll(64, wait_us=1000))
            if len(got) == len(props):
                break
        srv.close()
        assert [got.get(i) for i in range(len(props))] == [(0, int(t), int(x)) for t, x in zip(tracks, exact)]
