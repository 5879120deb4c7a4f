"""The distance of few simulations, whose rows are split over waves and, for
less than one simulation a CU, over workgroups: column counts at the edges of
the lanes' widths, observed histograms that are empty, end before or after the
simulated rows, or hold counts past 2^20 (the 128-bit sums), both distances,
and numbers of simulations on each side of the dispatch's lines, all against
the oracle (integers, so equal)."""
import numpy as np
import pytest

import cases
import oracle_lib as O
from part_conc_spt_abc_amd import _abi
from part_conc_spt_abc_amd.gpu import Context

pytestmark = pytest.mark.gpu


def observed(kind, n_k, n_de, rng):
    H = np.zeros((n_k, n_de), np.uint32)
    if kind == "short":
        H[min(4, n_k - 1), rng.integers(0, n_de, 50)] += 1
    elif kind == "deep":
        for r in range(0, n_k, 3):
            H[r, rng.integers(0, n_de, 8)] += 2
    elif kind == "huge":
        H[min(2, n_k - 1), n_de // 2] = 3_000_000_000
        H[n_k - 1, n_de - 1] = 7
    return H


@pytest.mark.parametrize("n_sims", [1, 7, 257, 1025])
@pytest.mark.parametrize("n_k,n_de,obs,kind", [
    (300, 1, "deep", 0), (300, 255, "none", 0), (7, 256, "short", 1), (300, 257, "deep", 1), (1000, 500, "short", 0),
    (300, 512, "huge", 0), (300, 513, "huge", 1), (1000, 1000, "deep", 0), (300, 1024, "none", 1), (300, 1025, "deep", 0)])
def test_split_distance(gpu_lib, n_k, n_de, obs, kind, n_sims):
    model = cases.headline_model(n_k=n_k, n_de=n_de, dist_kind=kind)
    rng = np.random.default_rng([n_k, n_de, n_sims])
    H0 = observed(obs, n_k, n_de, rng)
    # no records, under a quad of them, a few, and (alone) past 16 parts' registers
    parts = rng.integers(0, 60, n_sims).astype(np.uint32)
    parts[0] = 6000 if n_sims <= 7 else 900
    if n_sims > 1:
        parts[1], parts[-1] = 0, 1
    props = []
    for i in range(n_sims):
        p, _, _ = cases.fixed_proposal(model, [int(parts[i])], [300], sim_id=i)
        p.first_video = i
        props.append(p)
    with Context(model, H0) as ctx:
        b = ctx.batch()
        b.load(props, np.full(n_sims, 300, np.uint32), parts)
        for mode in (_abi.PCS_MODE_BATCHED, _abi.PCS_MODE_PLAIN_STREAMS)[: 2 if n_sims <= 7 else 1]:
            b.run(5, mode)
            _, tracks, _ = b.read()
            exact = b.read_exact()
            some = range(n_sims) if n_sims <= 7 else [0, 1, n_sims // 2, n_sims - 1]
            if mode == _abi.PCS_MODE_BATCHED:
                want = {}
                osys = O.system_from_abi(model.to_abi())
                for i in some:
                    Ho, _, _ = O.simulate_f32(osys, O.OracleProposal(props[i], np.array([300], np.uint32), parts[i:i + 1]), 5)
                    want[i] = (int(Ho.sum()), O.distance(Ho, H0, kind)[0])
            for i in some:
                assert (int(tracks[i]), int(exact[i])) == want[i], f"simulation {i}, mode {mode}"
        b.close()
