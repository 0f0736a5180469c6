"""Contexts whose whole chains are spread over k_sweep_whole, k_sweep_ideal and
k_sweep_allpairs, which then run beside each other on two streams."""
import numpy as np
import pytest

from pimc import _capi as A
from pimc.potentials import GaussianPair, HarmonicTrap
from pimc.system import chain_desc
from test_gpu_random_configs import run_and_check

pytestmark = pytest.mark.gpu
PAIR = GaussianPair(1.0, 0.5)


def chain(kind, N, M, ell=6):
    """ideal: swap moves; pairs: small Gaussian-pair chain; dropped: the same with its
    pair action left out of the acceptance (whole-chain kernel); swapped: pair action and swaps
    (whole-chain kernel); window: N > 96; tile: neither pairs nor swaps."""
    more = {"ideal": dict(swaps=3, swap_m=5), "pairs": dict(pair=PAIR), "dropped": dict(pair=PAIR, pair_in_accept=False),
            "swapped": dict(pair=PAIR, swaps=2, swap_m=4), "window": dict(pair=PAIR), "tile": {}}[kind]
    rng = np.random.default_rng(100 * N + M)
    L = 4.0
    d = chain_desc(HarmonicTrap(0.5), dim=2, M=M, N=N, L=L, beta=1.5, lam=0.5, ell=ell, r_a=2 * L / 4, com_step=0.5, **more)
    r = rng.uniform(-L, L, size=(N, 2, 1)).repeat(M, axis=2) + rng.normal(0, 0.1, size=(N, 2, M))
    return d, (r + L) % (2 * L) - L, "gauss" if "pair" in more else "none", (1, 1, 1)


MIXES = [("ideal", "dropped"), ("pairs", "swapped"), ("ideal", "pairs", "dropped", "window", "tile", "swapped")]
SIZES = {"ideal": (5, 20), "pairs": (9, 33), "dropped": (12, 18), "window": (100, 12), "tile": (3, 40), "swapped": (7, 26)}


def chains_of(mix):
    return [chain(k, *SIZES[k]) for k in mix]


@pytest.mark.parametrize("mix", MIXES)
def test_mixed_whole_chains_match_oracle_fp64(mix):
    run_and_check(chains_of(mix), 91, 3)


@pytest.mark.parametrize("measure_kernel", [1, 2])
@pytest.mark.parametrize("mix", MIXES + [("ideal", "pairs")])
def test_mixed_whole_chains_graph_replays_equal_eager(mix, measure_kernel):
    """Graph replays (which hold the fork and the join) equal eager launches bit
    for bit: paths, permutations, counters and estimator blocks, replay after
    replay, thermalising and measuring, with estimators in the sweep kernels
    and in kernels of their own."""
    chains, ctxs = chains_of(mix), []
    for g in (0, 1):
        opt = A.Options()
        opt.precision, opt.sweeps_per_launch, opt.seed, opt.use_graph, opt.measure_kernel = A.FP32, 3, 9, g, measure_kernel
        ctx = A.Context([d for d, _, _, _ in chains], opt)
        for c, (_, r, _, _) in enumerate(chains):
            ctx.set_paths(c, r)
        ctxs.append(ctx)
    for rep in range(4):
        for ctx in ctxs:
            ctx.run(9, measure=rep % 2 == 1)
        for c, (d, _, _, _) in enumerate(chains):
            assert np.array_equal(ctxs[0].get_paths(c), ctxs[1].get_paths(c)), (rep, c)
            assert np.array_equal(ctxs[0].counters(c), ctxs[1].counters(c)), (rep, c)
            if d.swaps:
                assert np.array_equal(ctxs[0].get_next(c), ctxs[1].get_next(c)), (rep, c)
    for c in range(len(chains)):
        assert all(np.array_equal(x, y) for x, y in zip(ctxs[0].blocks(c), ctxs[1].blocks(c))), c
