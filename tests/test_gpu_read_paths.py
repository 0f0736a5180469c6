"""Paths read back are the paths that were set, in both device layouts, around the
size where the rows are turned on the device and around its 32 x 64 tiles, and
in several pieces of the pinned buffer (4 MiB)."""
import numpy as np
import pytest

from pimc import _capi as A
from pimc.potentials import GaussianPair, HarmonicTrap
from pimc.system import chain_desc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [A.FP64, A.FP32])
@pytest.mark.parametrize("dim,N,M", [(2, 1, 4), (2, 3, 33), (2, 32, 64), (2, 33, 64), (1, 65, 63), (1, 64, 65), (2, 16, 129),
                                     (2, 300, 127), (1, 3000, 300), (2, 4097, 130)])
def test_paths_come_back_as_set(precision, dim, N, M):
    rng = np.random.default_rng(N + M)
    out = []
    for pair in (None, GaussianPair(1.0, 0.5)):
        if pair is not None and N > 2000:
            continue
        d = chain_desc(HarmonicTrap(1.0), dim=dim, M=M, N=N, L=40.0, beta=1.0, lam=0.5, pair=pair, ell=4, r_a=8.0)
        opt = A.Options()
        opt.precision, opt.sweeps_per_launch, opt.seed = precision, 1, 3
        ctx = A.Context([d], opt)
        r = rng.uniform(-39.0, 39.0, size=(N, dim, M))
        ctx.set_paths(0, r)
        out.append(np.array_equal(ctx.get_paths(0), r if precision == A.FP64 else r.astype(np.float32).astype(np.float64)))
    assert all(out) and out
