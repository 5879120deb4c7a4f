"""pmc-standard weights at the edges of the kernel sums' split: blocks of 256
new members, chunks of 32 to 4,096 old ones with and without a remainder, few
and many chunk sums, each parameter count's own kernel and the general one,
against the formula in extended precision."""
import numpy as np
import pytest

from part_conc_spt_abc_amd.gpu import pmc_weights

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -52


@pytest.mark.parametrize("P", [1, 2, 3, 4, 5, 6, 7, 8, 9, 24])
@pytest.mark.parametrize("n_new,n_old", [(1, 1), (2, 31), (127, 33), (255, 4), (256, 5), (257, 64), (300, 129),
                                         (513, 8195), (40, 33333)])
def test_pmc_sums(gpu_lib, P, n_new, n_old):
    rng = np.random.default_rng(n_new + 7 * P)
    old = rng.random((P, n_old))
    tau = rng.uniform(0.2, 2.0, P)
    new = old[:, rng.integers(0, n_old, n_new)] + 0.7 * tau[:, None] * rng.standard_normal((P, n_new))
    w = rng.random(n_old) + 0.01
    got = pmc_weights(new, old, w, tau)
    d = (new / tau[:, None]).astype(np.longdouble)[:, :, None] - (old / tau[:, None]).astype(np.longdouble)[:, None, :]
    h = 0.5 * (d * d).sum(axis=0)
    k = np.exp(-h) * w.astype(np.longdouble)
    want = 1.0 / k.sum(axis=1)
    want /= want.sum()
    # a term: 3 ulp of the exponential and P + 2 roundings of s, in the exponent;
    # the sums: at most chunk + chunks roundings (128 + 512 at these sizes) and,
    # to normalise, n_new (at most 513)
    tol = EPS * (3.0 + (P + 2) * float(((h * k).sum(axis=1) / k.sum(axis=1)).max()) + 640 + 513)
    assert np.all(np.abs(got / want - 1.0) <= tol)


def test_far_members_keep_underflowing(gpu_lib):
    """Kernel terms past the smallest double are 0: the member's weight
    overflows, as in the plain formula."""
    rng = np.random.default_rng(1)
    old = rng.random((2, 700))
    new = np.concatenate([rng.random((2, 9)), [[60.0, np.inf], [0.5, 0.0]]], axis=1)
    got = pmc_weights(new, old, np.full(700, 1 / 700), np.ones(2))
    assert np.all(got[:9] == 0.0) and np.all(np.isnan(got[9:]))
