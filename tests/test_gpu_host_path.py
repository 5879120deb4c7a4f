"""Host side of small calls: results in pinned host memory or, above 4,096
simulations, on the device; pcs_simulate's kept batch over calls of changing
size, form and record capacity; the first (direct) and later (graph) runs of a
plan; dense histograms smaller and larger than their staging."""
import ctypes as C

import numpy as np
import pytest

import cases
from part_conc_spt_abc_amd import _abi
from part_conc_spt_abc_amd.gpu import Context
from part_conc_spt_abc_amd.model import proposals_array

pytestmark = pytest.mark.gpu


def workload(model, n, seed=1):
    rng = np.random.default_rng(seed)
    return cases.draw_proposals(model, n, rng, frames_choices=(40, 77), c_range=(5e6, 5e8))


def simulate(ctx, props, f, n, seed, mode, hist=False):
    m, k = ctx.model, len(props)
    dist, tracks = np.empty(k), np.empty(k, np.uint32)
    H = np.empty((k, m.n_k, m.n_de), np.uint32) if hist else None
    p = lambda a: None if a is None else a.ctypes.data_as(C.c_void_p)  # noqa: E731
    _abi.check(ctx.lib.pcs_simulate(ctx.h, C.cast(proposals_array(props), C.c_void_p), k, p(f), p(n), len(f), seed, mode,
                                    p(dist), p(H), p(tracks)), "pcs_simulate")
    return dist, tracks, H


@pytest.mark.parametrize("n", [1, 4096, 4097])
def test_results_on_either_side(gpu_lib, n):
    model = cases.headline_model(n_k=100, n_de=64)
    obs = np.zeros((100, 64), np.uint32)
    obs[3, 5] = 9
    props, f, parts = workload(model, n)
    with Context(model, obs) as ctx:
        b = ctx.batch()
        b.load(props, f, parts)
        runs = []
        for seed in (7, 8, 7):  # direct, captured, replayed
            b.run(seed)
            dist, tracks, _ = b.read()
            runs.append((dist, tracks, b.read_exact()))
        assert all(np.array_equal(x, y) for x, y in zip(runs[0], runs[2]))
        if n > 1:
            assert not np.array_equal(runs[0][1], runs[1][1])
        k = min(n, 33)  # the same simulations in a small batch
        s = ctx.batch()
        s.load(props[:k], f[:k], parts[:k])
        s.run(7)
        dist, tracks, _ = s.read()
        assert np.array_equal(dist, runs[0][0][:k]) and np.array_equal(tracks, runs[0][1][:k])
        assert np.array_equal(s.read_exact(), runs[0][2][:k])
        s.close()
        b.close()


def test_simulate_keeps_nothing_between_calls(gpu_lib):
    model = cases.headline_model(n_k=100, n_de=64)
    big = workload(model, 300)
    with Context(model) as ctx:
        b = ctx.batch()
        b.load(*big)
        b.run(3)
        dist, tracks, H = b.read(hist=True)
        b.close()
        for k, mode, hist, factor in [(300, 1, True, 0.5), (1, 0, False, 0.5), (5, 1, True, 1e-4), (300, 3, False, 0.5),
                                      (2, 1, False, 0.5), (0, 1, False, 0.5), (7, 1, True, 0.5)]:
            ctx.set_record_capacity_factor(factor)
            d, t, h = simulate(ctx, big[0][:k], big[1][:k], big[2][:k], 3, mode, hist)
            assert np.array_equal(d, dist[:k]) and np.array_equal(t, tracks[:k]), (k, mode)
            assert h is None or np.array_equal(h, H[:k]), (k, mode)
        with pytest.raises(_abi.PcsError):
            simulate(ctx, big[0][:1], big[1][:1], big[2][:1], 3, 99)
        d, t, _ = simulate(ctx, big[0][:2], big[1][:2], big[2][:2], 3, 1)
        assert np.array_equal(d, dist[:2]) and np.array_equal(t, tracks[:2])


@pytest.mark.parametrize("n_k,n_de,n", [(3, 1, 3), (1000, 500, 9), (2500, 4096, 2)])
def test_histograms_through_staging(gpu_lib, n_k, n_de, n):
    model = cases.headline_model(n_k=n_k, n_de=n_de)
    props, f, parts = workload(model, n)
    parts[:] = np.maximum(parts, 300)
    with Context(model) as ctx:
        b = ctx.batch()
        b.load(props, f, parts)
        b.run(5)
        _, tracks, H = b.read(hist=True)
        _, _, H2 = b.read(hist=True)
        assert np.array_equal(H.reshape(n, -1).sum(1), tracks) and np.array_equal(H, H2)
        small = cases.headline_model(n_k=n_k, n_de=n_de)
        with Context(small) as c2:
            for i in range(n):
                p = cases.PCS.pcs_proposal.from_buffer_copy(props[i])
                p.first_video = 0
                _, t, h = simulate(c2, [p], f[i:i + 1], parts[i:i + 1], 5, 0, True)
                assert t[0] == tracks[i] and np.array_equal(h[0], H[i])
        b.close()


@pytest.mark.parametrize("ppl", [1, 2])
def test_longest_videos_first(gpu_lib, ppl):
    """Videos of different lengths are taken longest first in the batched form;
    each simulation's result is its own (plain form, videos as given)."""
    model = cases.headline_model(n_k=100, n_de=64)
    rng = np.random.default_rng(4)
    props, f, parts = cases.draw_proposals(model, 90, rng, frames_choices=(2, 17, 40, 41, 77), videos=3,
                                           c_range=(5e6, 3e9))
    parts[4] = parts[100] = 0
    with Context(model) as ctx:
        ctx.set_tuning(particles_per_lane=ppl)
        b = ctx.batch()
        for frames in (f, np.full_like(f, 50), f[::-1].copy()):
            b.load(props, frames, parts)
            got = []
            for mode in (1, 1, 0, 3, 2):
                b.run(3, mode)
                _, tracks, _ = b.read()
                got.append((tracks, b.read_exact()))
            assert all(np.array_equal(x, got[0][0]) and np.array_equal(y, got[0][1]) for x, y in got[1:])
        b.close()
