"""Window chains whose pair slots exceed what a group holds at a time (4 GiB): the
chains of a group then run in batches that share the slots."""
import numpy as np
import pytest

from pimc import _capi as A
from pimc.potentials import GaussianPair, NoPotential
from pimc.system import chain_desc

pytestmark = pytest.mark.gpu


def desc(N):
    return chain_desc(NoPotential(), dim=2, M=64, N=N, L=15.0, beta=1.0, lam=0.5, pair=GaussianPair(1.0, 0.5), ell=2, r_a=2.0,
                      com_step=0.5)


def paths(N, seed):
    rng = np.random.default_rng(seed)
    r = rng.uniform(-15.0, 15.0, size=(N, 2, 1)) + rng.normal(0, 0.1, size=(N, 2, 64))
    return (r + 15.0) % 30.0 - 15.0


def sample(sizes, keep):
    opt = A.Options()
    opt.precision, opt.sweeps_per_launch, opt.seed = A.FP32, 2, 3
    ctx = A.Context([desc(n) for n in sizes], opt)
    for c, n in enumerate(sizes):
        ctx.set_paths(c, paths(n, c))
    ctx.run(2, measure=False)
    ctx.run(2, measure=True)
    return [(ctx.get_paths(c), ctx.estimates(c).Epair, list(ctx.counters(c))) for c in keep]


def test_chains_in_batches_sample_as_without():
    """128 chains of N = 900, M = 64, ell = 2 (32 staging windows): 78 MB of pair
    slots each, two groups of 64 on two streams, so 55 chains and then 9 in each
    group.  The first and last chain of both batches of both groups sample bit for
    bit as in a context where the others are too small to share anything: a
    chain's draws are keyed by its index, and no other chain's size is part of its
    sums."""
    N, keep = 900, (0, 54, 55, 63, 64, 118, 119, 127)
    batched = sample([N] * 128, keep)
    alone = sample([N if c in keep else 2 for c in range(128)], keep)
    for c, (r, e, n), (r0, e0, n0) in zip(keep, batched, alone):
        assert np.array_equal(r, r0), c
        assert e == e0 and n == n0, c
