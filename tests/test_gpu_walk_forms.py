"""The forms of the walk against each other and the oracle, each at a number of
tiles that reaches it: a workgroup a tile (up to 6.75 tiles a CU, 3.75 with
Gaussian detection) and a wave a tile above, and in batches planned on the
device."""
import numpy as np
import pytest

import cases
import oracle_lib as O
from part_conc_spt_abc_amd import _abi
from part_conc_spt_abc_amd.gpu import Context
from part_conc_spt_abc_amd.model import prior_record

pytestmark = pytest.mark.gpu

CLASSES = {
    "slab": {},
    "slab, walls": dict(z_boundary=_abi.PCS_Z_REFLECT),
    "gauss": dict(detect_model=_abi.PCS_DETECT_GAUSS_Z, detect_sigma=1.5),
    "gauss, walls": dict(detect_model=_abi.PCS_DETECT_GAUSS_Z, detect_sigma=1.5, z_boundary=_abi.PCS_Z_REFLECT),
}


@pytest.mark.parametrize("ppl", [1, 2])
@pytest.mark.parametrize("cls", list(CLASSES))
def test_plain_launches_of_proposed_trials(gpu_lib, cls, ppl):
    """Proposed trials in the batched form (the device's plan) and one by one
    (the host has fetched it), with slices that fit and slices that overflow."""
    model = cases.headline_model(n_k=140, n_de=64, Lz=15.0, **CLASSES[cls])
    rng = np.random.default_rng(2)
    theta = np.vstack([rng.uniform(0.5, 2.5, (2, 20)), rng.uniform(7.5, 9.0, (2, 20)), np.full((1, 20), 8.0)])
    pr = prior_record(model, (0.1, 5.0), (6.5, 9.5), (0.5, 14.0))
    frames = rng.integers(2, 140, (37, 3)).astype(np.uint32)
    with Context(model) as ctx:
        ctx.set_tuning(particles_per_lane=ppl)
        got = []
        for factor in (0.5, 1e-4):
            ctx.set_record_capacity_factor(factor)
            b = ctx.batch()
            b.propose(pr, theta, np.cumsum(np.full(20, 0.05)), np.full(5, 0.1), 37, frames, seed=5)
            for mode in (_abi.PCS_MODE_BATCHED, _abi.PCS_MODE_PLAIN, _abi.PCS_MODE_PLAIN_STREAMS):
                b.run(9, mode)
                _, tracks, H = b.read(hist=True)
                got.append((tracks, H, b.read_exact()))
                assert (b.overflow_reruns() > 0) == (factor < 0.1)
            b.close()
    assert int(got[0][0].sum()) > 1000
    assert all(np.array_equal(x, y) for g in got[1:] for x, y in zip(g, got[0]))


@pytest.mark.parametrize("cls", ["slab", "gauss, walls"])
def test_autotune_on_few_tiles(gpu_lib, cls):
    """Few tiles are walked by a workgroup each, whatever the shape: tuning on
    them leaves the shape alone (one wave a group is none of the candidates)."""
    model = cases.headline_model(n_k=140, n_de=64, Lz=15.0, **CLASSES[cls])
    p, f, n = cases.fixed_proposal(model, [1000], [500])
    with Context(model) as ctx:
        ctx.set_tuning(particles_per_lane=2, waves_per_group=1, groups_per_cu=7, stage_records=128)
        best, ms = ctx.autotune([p], f, n)
        assert best == ctx.get_tuning() == dict(particles_per_lane=1, waves_per_group=1, groups_per_cu=7, stage_records=128)
        assert ms > 0.0


def many_tiles(frames, sims=34):
    """Simulations of 4,000 particles (63 tiles each: 2,142 tiles, more than
    are walked by workgroups), some smaller."""
    rng = np.random.default_rng(7)
    parts = rng.integers(3970, 4030, sims).astype(np.uint32)
    parts[1], parts[2], parts[3] = 0, 1, 65
    f = rng.choice(frames, sims).astype(np.uint32)
    props = []
    for i in range(sims):
        p, _, _ = cases.fixed_proposal(cases.headline_model(), [1], [1], sim_id=i, az=(12.0,))
        p.first_video = i
        props.append(p)
    return props, f, parts


def check_waves(model, load, tunings, seed=9):
    """The batched histograms of each tuning against the oracle's for some
    simulations, and against the plain form's (few tiles each) for all."""
    props, f, parts = load
    some = (1, 2, 3, 4, len(props) - 1)
    osys = O.system_from_abi(model.to_abi())
    want = {i: O.simulate_f32(osys, O.OracleProposal(props[i], f[i:i + 1], parts[i:i + 1]), seed)[0] for i in some}
    with Context(model) as ctx:
        b = ctx.batch()
        b.load(*load)
        b.run(seed, _abi.PCS_MODE_PLAIN)
        plain = b.read(hist=True)[2]
        for t in tunings:
            ctx.set_tuning(**t)
            b.run(seed, _abi.PCS_MODE_BATCHED_DIRECT)
            H = b.read(hist=True)[2]
            for i in some:
                assert np.array_equal(H[i], want[i]), f"{t}: simulation {i}"
            assert np.array_equal(H, plain), t
        b.close()


@pytest.mark.parametrize("kmin", [2, 3, 31, 32, 33, 47])
@pytest.mark.parametrize("cls", list(CLASSES))
def test_wave_walk_classes(gpu_lib, cls, kmin):
    model = cases.headline_model(n_k=140, n_de=64, kmin=kmin, Lz=15.0, **CLASSES[cls])
    check_waves(model, many_tiles([1, 5, 34, 97, 130]), [{}])


@pytest.mark.parametrize("cls", ["slab", "gauss, walls"])
def test_wave_walk_tunings(gpu_lib, cls):
    """Waves a group, groups a CU and record stages, at one particle a lane:
    kmin 2 and a wide window fill the stage often."""
    model = cases.headline_model(n_k=140, n_de=64, kmin=2, Lz=15.0, **CLASSES[cls])
    check_waves(model, many_tiles([60, 61]), [dict(waves_per_group=w, groups_per_cu=g, stage_records=s)
                                              for w, g in ((1, 4), (2, 16), (4, 1), (4, 8)) for s in (128, 256, 512)])


@pytest.mark.parametrize("cls", list(CLASSES))
def test_wave_walk_of_one_simulation(gpu_lib, cls):
    """The plain form above the few-tiles line: 1,900 tiles of one simulation."""
    model = cases.headline_model(n_k=140, n_de=64, Lz=15.0, **CLASSES[cls])
    p, f, n = cases.fixed_proposal(model, [121537, 63], [21, 40], az=(12.0,))
    H, _, _ = O.simulate_f32(O.system_from_abi(model.to_abi()), O.OracleProposal(p, f, n), 4)
    with Context(model) as ctx:
        b = ctx.batch()
        b.load([p], f, n)
        for mode in (_abi.PCS_MODE_PLAIN, _abi.PCS_MODE_BATCHED):
            b.run(4, mode)
            assert np.array_equal(b.read(hist=True)[2][0], H)
        b.close()
