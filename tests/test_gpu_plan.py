"""The device plan of proposed trials on both sides of its dispatch (one
workgroup, or block sums, scan and tables over many) and at the edges of its
blocks of 1,024: a proposed batch gives what the same records give when loaded
from the host. Cumulative weights of a resident population at the edges of the
tiles of 2,048: the proposals equal those from numpy's cumsum."""
import numpy as np
import pytest

import cases
from part_conc_spt_abc_amd.gpu import Context
from part_conc_spt_abc_amd.model import prior_record

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,J,n_pop", [(1, 1, 1), (1024, 3, 15), (1025, 3, 16), (2048, 2, 17), (2049, 1, 2047),
                                       (3071, 2, 2048), (700, 25, 2049), (5000, 1, 6145)])
def test_device_plan(gpu_lib, n, J, n_pop):
    model = cases.headline_model(n_k=60, n_de=40)
    rng = np.random.default_rng([n, J, n_pop])
    theta = np.vstack([rng.uniform(0.5, 2.5, (2, n_pop)), rng.uniform(6.6, 7.4, (2, n_pop)), np.full((1, n_pop), 2.0)])
    w = rng.gamma(1.0, 1.0, n_pop)
    w /= w.sum()
    tau = np.sqrt(2.0 * theta.var(axis=1))
    prior = prior_record(model, (0.1, 5.0), (6.5, 7.5), (0.5, 4.0))
    frames = rng.integers(2, 60, (n, J)).astype(np.uint32)
    obs = np.zeros((60, 40), np.uint32)
    obs[4, 7] = 3
    with Context(model, obs) as ctx:
        b = ctx.batch()
        b.set_population(theta, w)
        new = b.propose(prior, None, None, tau, n, frames, seed=11)
        props, parts = b.read_proposals()
        host = b.propose(prior, theta, np.cumsum(w), tau, n, frames, seed=11)
        assert np.array_equal(new, host)
        b.run(12)
        dist, tracks, _ = b.read()
        exact = b.read_exact()
        assert b.overflow_reruns() == 0
        s = ctx.batch()
        s.load(props, frames.ravel(), parts)
        assert s.arena()[0] == b.arena()[0]
        s.run(12)
        d2, t2, _ = s.read()
        assert np.array_equal(tracks, t2) and np.array_equal(exact, s.read_exact()) and np.array_equal(dist, d2)
        assert int(tracks.sum()) > 0 or n < 10
        s.close()
        b.close()
