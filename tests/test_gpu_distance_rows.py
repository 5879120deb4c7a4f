"""The rows of a distance are shared out over a simulation's waves, the rows
that only the observed table holds among them: a wave that swept all 4,000 of
them alone would take 0.73 to 0.83 ms (0.2 us a row); all waves take 0.05 to
0.17."""
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
