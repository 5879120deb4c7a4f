"""Few tiles are walked by a workgroup each (producers, movers, a tracker): at
the edges of its rounds of 32 frames and chunks of 4, of a tile's 64
particles, and of the tracker's 32-bit run test (kmin), in every model class,
with more tiles than workgroups, in the batched and the plain form. The
oracle's histograms are integers, so equal."""
import numpy as np
import pytest

import cases
import oracle_lib as O
from part_conc_spt_abc_amd import _abi
from part_conc_spt_abc_amd.gpu import Context

pytestmark = pytest.mark.gpu

CLASSES = {
    "slab": {},
    "slab, walls": dict(z_boundary=_abi.PCS_Z_REFLECT),
    "gauss": dict(detect_model=_abi.PCS_DETECT_GAUSS_Z, detect_sigma=1.5),
    "gauss, walls": dict(detect_model=_abi.PCS_DETECT_GAUSS_Z, detect_sigma=1.5, z_boundary=_abi.PCS_Z_REFLECT),
}


def check(model, frames, parts, modes, seed=9):
    """One simulation a video; its histogram against the oracle's."""
    props = []
    for i, (f, n) in enumerate(zip(frames, parts)):
        p, _, _ = cases.fixed_proposal(model, [n], [f], sim_id=i, az=(12.0,))
        p.first_video = i
        props.append(p)
    f, n = np.array(frames, np.uint32), np.array(parts, np.uint32)
    osys = O.system_from_abi(model.to_abi())
    want = [O.simulate_f32(osys, O.OracleProposal(p, f[i:i + 1], n[i:i + 1]), seed)[0] for i, p in enumerate(props)]
    with Context(model) as ctx:
        b = ctx.batch()
        b.load(props, f, n)
        for mode in modes:
            b.run(seed, mode)
            _, _, H = b.read(hist=True)
            for i in range(len(props)):
                assert np.array_equal(H[i], want[i]), f"mode {mode}: {frames[i]} frames, {parts[i]} particles"
        b.close()


@pytest.mark.parametrize("kmin", [2, 3, 31, 32, 33, 47])
@pytest.mark.parametrize("cls", list(CLASSES))
def test_group_walk_edges(gpu_lib, cls, kmin):
    model = cases.headline_model(n_k=140, n_de=64, kmin=kmin, Lz=15.0, **CLASSES[cls])
    frames = [1, 2, 4, 5, 6, 31, 32, 33, 34, 36, 64, 65, 66, 97, 98, 130]
    parts = [200, 1, 63, 64, 65, 127, 128, 129, 300, 64, 190, 65, 500, 64, 700, 257]
    check(model, frames, parts, (_abi.PCS_MODE_BATCHED, _abi.PCS_MODE_PLAIN_STREAMS))


@pytest.mark.parametrize("cls", list(CLASSES))
def test_more_tiles_than_groups(gpu_lib, cls):
    model = cases.headline_model(n_k=140, n_de=64, Lz=15.0, **CLASSES[cls])
    rng = np.random.default_rng(3)
    check(model, rng.integers(1, 80, 40), rng.integers(900, 1500, 40), (_abi.PCS_MODE_BATCHED,))
