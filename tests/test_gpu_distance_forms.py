"""The forms of the distance over large record slices at up to 1,024 columns:
the block form (more than four simulations a CU: 1,024) with its records held
in registers or read twice and its bins in LDS or HBM, and the split form by 16
and by 8 waves past what their LDS holds (at most 32,768 bins a workgroup). The
large simulations' histograms come from a batch of their own (several
workgroups each); their distances in each form equal the oracle's."""
import numpy as np
import pytest

import cases
import oracle_lib as O
from part_conc_spt_abc_amd import _abi
from part_conc_spt_abc_amd.gpu import Context

pytestmark = pytest.mark.gpu

FRAMES = 1000


def padded(model, parts, total):
    """Simulations of the given particle counts, then small ones up to `total`."""
    parts = np.concatenate([parts, np.arange(total - len(parts)) % 3]).astype(np.uint32)
    props = []
    for i in range(total):
        p, _, _ = cases.fixed_proposal(model, [1], [FRAMES], sim_id=100 + i)
        p.first_video = i
        props.append(p)
    f = np.full(total, FRAMES, np.uint32)
    f[len(props) // 2:] = 30
    return props, f, parts


def check(model, obs, parts, total, dist_kind=0):
    k = len(parts)
    props, f, n = padded(model, parts, total)
    f[:k] = FRAMES
    with Context(model, obs) as ctx:
        s = ctx.batch()
        s.load(props[:k], f[:k], n[:k])
        s.run(41)
        _, tracks, H = s.read(hist=True)
        s.close()
        b = ctx.batch()
        b.load(props, f, n)
        for seed in (41, 41):
            b.run(seed)
            t = b.read()[1]
            exact = b.read_exact()
            assert np.array_equal(t[:k], tracks)
            for i in range(k):
                want = O.distance(H[i], obs, dist_kind)[0]
                assert int(exact[i]) == want, f"simulation {i} of {total} ({tracks[i]} records)"
        b.close()
    return tracks


def observed(model):
    p, f, n = cases.fixed_proposal(model, [1500], [FRAMES], sim_id=0xFFFFFFF0)
    return O.simulate_f32(O.system_from_abi(model.to_abi()), O.OracleProposal(p, f, n), 0)[0]


# Record counts of the block form: LDS-sorted; held in registers with the bins
# in LDS or HBM; past the registers (read twice), also with bins in HBM.
BANDS = [(1, 4096), (7300, 8192), (8193, 16384), (16385, 10 ** 9)]


@pytest.mark.parametrize("n_k,n_de,kind", [(500, 200, 0), (500, 256, 1), (1000, 500, 0), (1000, 1000, 0)])
def test_block_form(gpu_lib, n_k, n_de, kind):
    model = cases.headline_model(n_k=n_k, n_de=n_de, dist_kind=kind)
    parts = np.concatenate([np.linspace(0, 14000, 25), np.linspace(2400, 2800, 9)])
    tracks = check(model, observed(model), parts, 1100, kind)
    assert tracks.min() == 0
    for lo, hi in BANDS:
        assert ((tracks >= lo) & (tracks <= hi)).any(), (lo, hi)


@pytest.mark.parametrize("total", [129, 256, 257])
@pytest.mark.parametrize("n_k,n_de,kind", [(500, 256, 0), (1000, 500, 1), (1000, 1000, 0)])
def test_split_form_past_its_lds(gpu_lib, n_k, n_de, kind, total):
    model = cases.headline_model(n_k=n_k, n_de=n_de, dist_kind=kind)
    tracks = check(model, observed(model), np.array([14000, 0, 17000, 1, 5000, 11000]), total, kind)
    assert int(tracks[0]) > 40000 and int(tracks[2]) > 40000
