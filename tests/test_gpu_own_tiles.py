"""Batched walk: the waves of the resident workgroups have a first tile of
their own and take the ones after from a counter. Fewer tiles than waves, as
many, a few more, many more; more workgroups than run at once; videos of one
length and of several, against the plain form of the same simulations."""
import numpy as np
import pytest

import cases
from part_conc_spt_abc_amd import _abi
from part_conc_spt_abc_amd.gpu import Context

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("ppl,wpg,groups", [(1, 1, 1), (1, 4, 8), (1, 4, 16), (2, 1, 1), (2, 2, 3), (2, 4, 16)])
@pytest.mark.parametrize("tiles", [1, 255, 256, 257, 3700, 20000])
def test_own_tiles(gpu_lib, tiles, ppl, wpg, groups, mixed):
    model = cases.headline_model(n_k=60, n_de=64, kmin=2)
    n = min(tiles, 25)
    props = []
    for i in range(n):
        p, _, _ = cases.fixed_proposal(model, [1], [10], sim_id=i, az=(12.0,))
        p.first_video = i
        props.append(p)
    f = (6 + 5 * (np.arange(n) % 4) if mixed else np.full(n, 10)).astype(np.uint32)
    share = np.full(n, tiles // n) + (np.arange(n) < tiles % n)
    parts = (share * 64 * ppl - np.arange(n) % (64 * ppl)).astype(np.uint32)
    got = []
    with Context(model) as ctx:
        ctx.set_tuning(particles_per_lane=ppl, waves_per_group=wpg, groups_per_cu=groups)
        b = ctx.batch()
        b.load(props, f, parts)
        for mode in (_abi.PCS_MODE_PLAIN, _abi.PCS_MODE_BATCHED, _abi.PCS_MODE_BATCHED):
            b.run(3, mode)
            _, tracks, _ = b.read()
            got.append((tracks, b.read_exact()))
        b.close()
    assert all(np.array_equal(t, got[0][0]) and np.array_equal(x, got[0][1]) for t, x in got[1:])
