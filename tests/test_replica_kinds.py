"""The kinds of replicas of a launch: binder counts and twisting chains, several of a kind."""
import copy
from types import SimpleNamespace

import numpy as np
import pytest

from chromo_amd import _lib as L
from chromo_amd import workloads as W


def _chains(kinds):
    return [SimpleNamespace(B=b, twist=t) for b, t in kinds]


@pytest.mark.parametrize("kinds,mask", [([(2, False)], 0x4), ([(2, False)] * 3, 0x4), ([(1, True)], 0x202),
                                        ([(1, True)] * 2, 0x202), ([(3, True)] * 5, 0x808),
                                        ([(1, False), (1, True), (4, True), (4, True), (2, False)], 0x1216)])
def test_kinds_mask(kinds, mask):
    from chromo_amd.engine import kinds_mask
    assert kinds_mask(_chains(kinds)) == mask


@pytest.mark.gpu
def test_several_twisting_chains_of_one_kind():
    """Two twisting chains with the same binder count, beside a plain one, run as they do
    alone, bit for bit."""
    from chromo_amd.engine import DeviceReplicas
    print("several twisting chains", flush=True)
    systems = [W.make_twist_system(300, 2, 8, seed=40), W.make_system(350, 2, 8, seed=41),
               W.make_twist_system(260, 2, 8, seed=42)]

    def make(idx):
        return DeviceReplicas([systems[i].chain for i in idx], [systems[i].field for i in idx],
                              [copy.deepcopy(systems[i].ctrls) for i in idx], rng_mode=L.RNG_PHILOX,
                              seeds=[7] * len(idx), streams=idx)
    together = make([0, 1, 2])
    together.run(3)
    for i in range(3):
        alone = make([i])
        alone.run(3)
        for a, b in zip(together.positions(i), alone.positions(0)):
            assert np.array_equal(a, b), i
        assert np.array_equal(together.rng_words(i), alone.rng_words(0))
        assert np.array_equal(together.density_of(i), alone.density_of(0))
    assert np.all(together.counter_array()[:, L.CNT_PROPOSALS] > 3 * 100)
