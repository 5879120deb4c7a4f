"""The rows of a distance are shared out over a simulation's waves, the rows
that only the observed table holds among them: a wave that swept all 4,000 of
them alone would take 0.73 to 0.83 ms (0.2 us a row); all waves take 0.05 to
0.17. And over a simulation's workgroups: past 2,048 records or with 129 observed
rows, up to which one takes it alone."""
import numpy as np
import pytest

import cases
import oracle_lib as O
from part_conc_spt_abc_amd import _abi
from part_conc_spt_abc_amd.gpu import Context

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_sims", [1, 200, 300])
def test_observed_rows_are_shared_out(gpu_lib, n_sims):
    model = cases.headline_model(n_k=4000, n_de=64)
    obs = np.zeros((4000, 64), np.uint32)
    obs[::3, ::5] = 1
    props = []
    for i in range(n_sims):
        p, f, n = cases.fixed_proposal(model, [40], [60], sim_id=i)
        p.first_video = i
        props.append(p)
    with Context(model, obs) as ctx:
        b = ctx.batch()
        b.load(props, np.full(n_sims, 60, np.uint32), np.full(n_sims, 40, np.uint32))
        ms = []
        for _ in range(6):
            b.run(5, _abi.PCS_MODE_BATCHED_DIRECT)
            b.read()
            ms.append(b.timing()[2])
        exact = b.read_exact()
        b.close()
    osys = O.system_from_abi(model.to_abi())
    for i in {0, n_sims - 1}:
        H, _, _ = O.simulate_f32(osys, O.OracleProposal(props[i], f, n), 5)
        assert int(exact[i]) == O.distance(H, obs, 0)[0]
    print(f"{n_sims} simulations: {1e3 * min(ms):.1f} us", flush=True)
    assert min(ms) < 0.3


@pytest.mark.parametrize("deep", [1, 128, 129])
@pytest.mark.parametrize("n_sims", [1, 3, 60, 128, 129])
def test_one_workgroup_or_several(gpu_lib, n_sims, deep):
    """16, 4, 2 and 1 workgroups a simulation, record counts on both sides of
    2,048, the same batch twice (the tickets are zero again)."""
    model = cases.headline_model(n_k=300, n_de=200)
    obs = np.zeros((300, 200), np.uint32)
    obs[:deep, ::9] = 2
    parts = np.linspace(1250, 1500, n_sims).astype(np.uint32) if n_sims > 3 else np.array([9, 1300, 1450], np.uint32)[-n_sims:]
    if n_sims > 3:
        parts[:3] = 0, 1, 9
    props = []
    for i in range(n_sims):
        p, _, _ = cases.fixed_proposal(model, [1], [500], sim_id=i)
        p.first_video = i
        props.append(p)
    with Context(model, obs) as ctx:
        b = ctx.batch()
        b.load(props, np.full(n_sims, 500, np.uint32), parts)
        got = []
        for mode in (_abi.PCS_MODE_BATCHED, _abi.PCS_MODE_BATCHED, _abi.PCS_MODE_PLAIN_STREAMS):
            b.run(5, mode)
            _, tracks, H = b.read(hist=True)
            got.append(b.read_exact())
        b.close()
    want = [O.distance(H[i], obs, 0)[0] for i in range(n_sims)]
    assert n_sims == 1 or int(tracks.min()) <= 2048 < int(tracks.max())
    assert all([int(x) for x in g] == want for g in got)
