"""The batched walk decides Gaussian-z detection by the hardware's exponential
and, next to the bound, by the exact form; the walks of few tiles by the exact
form alone. The same simulations in both: one after another (few tiles each)
and batched (more tiles than are walked by groups)."""
import numpy as np
import pytest

import cases
from part_conc_spt_abc_amd import _abi
from part_conc_spt_abc_amd.gpu import Context

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("walls", [False, True])
@pytest.mark.parametrize("sigma", [0.05, 1.5, 40.0])
def test_gauss_bound(gpu_lib, sigma, walls):
    kw = dict(z_boundary=_abi.PCS_Z_REFLECT) if walls else {}
    model = cases.headline_model(n_k=100, n_de=64, kmin=2, Lz=15.0, detect_model=_abi.PCS_DETECT_GAUSS_Z,
                                 detect_sigma=sigma, **kw)
    n = 220
    props = []
    for i in range(n):
        p, _, _ = cases.fixed_proposal(model, [1000], [40], sim_id=i, az=(12.0,))
        p.first_video = i
        props.append(p)
    f, parts = np.full(n, 40, np.uint32), np.full(n, 1000, np.uint32)
    got = []
    with Context(model) as ctx:
        assert n * 16 > 11 * 256  # tiles: more than are walked by groups
        b = ctx.batch()
        b.load(props, f, parts)
        for mode in (_abi.PCS_MODE_BATCHED, _abi.PCS_MODE_PLAIN):
            b.run(7, mode)
            _, tracks, H = b.read(hist=True)
            got.append((tracks, H))
        b.close()
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
