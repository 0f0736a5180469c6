"""Whole chains without a pair action (k_sweep_ideal) against the oracle, FP64, at
the sizes where the kernel can go wrong: more swap tries than one batch of
draws, one and two particles, windows that reach across the ring's end,
staging lengths that do not divide M (a last segment of one link too), rings
longer than a wave and than 512 slices, and chains too large for its LDS beside
them."""
import numpy as np
import pytest

from pimc.potentials import HarmonicTrap, NoPotential, SquareLattice
from pimc.system import chain_desc
from test_gpu_random_configs import run_and_check

pytestmark = pytest.mark.gpu


def chain(N, M, ell, swaps, swap_m, rule=0, pot=None, every=(1, 1, 1), seed=0):
    rng = np.random.default_rng(100 * N + M + seed)
    L = 3.0
    d = chain_desc(pot or HarmonicTrap(1.0), dim=2, M=M, N=N, L=L, beta=1.5, lam=0.5, ell=ell, com_step=0.5, swaps=swaps,
                   swap_m=swap_m, swap_rule=rule, staging_every=every[0], com_every=every[1], swap_every=every[2])
    r = rng.uniform(-L, L, size=(N, 2, 1)).repeat(M, axis=2) + rng.normal(0, 0.1, size=(N, 2, M))
    return d, (r + L) % (2 * L) - L, "none", every


@pytest.mark.parametrize("N,M,ell,swaps,swap_m,rule", [
    (1, 16, 8, 3, 8, 0), (2, 4, 2, 1, 2, 0), (2, 65, 8, 16, 64, 0), (7, 33, 8, 17, 9, 0), (10, 64, 8, 33, 8, 1),
    (3, 513, 32, 2, 40, 0), (65, 16, 5, 20, 15, 0), (5, 40, 7, 15, 2, 1)])
def test_swap_chains_match_oracle(N, M, ell, swaps, swap_m, rule):
    run_and_check([chain(N, M, ell, swaps, swap_m, rule)], 11 + N, 3)


def test_chains_of_both_kernels_in_one_context():
    """A chain whose path does not fit LDS (N M = 4 480 beads in FP64) stays on
    k_sweep_whole beside those of k_sweep_ideal; move weights on some."""
    run_and_check([chain(70, 64, 8, 4, 8), chain(4, 24, 6, 18, 10, pot=SquareLattice(2.0, 1.0), every=(2, 1, 3)),
                   chain(6, 12, 5, 5, 11, pot=NoPotential(), every=(1, 3, 1))], 5, 3)
