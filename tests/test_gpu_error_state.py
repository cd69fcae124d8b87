"""What a replica that stops with an error leaves behind: the speculative kernel's chain,
densities, streams, controllers, counters and log are those of the one-at-a-time kernel,
whatever was drawn ahead of the failing proposal."""
import copy

import numpy as np
import pytest

from chromo_amd import _lib as L
from chromo_amd import workloads as W

pytestmark = pytest.mark.gpu


def _system(kind, i):
    s = W.make_system(500, 1 + i % 4, 8, seed=300 + i, chi=0.4, per_cycle=(7, 5, 9, 4, 6))
    for c in s.ctrls:
        if kind == "draw" and c.move == L.END_PIVOT:
            c.amp_bead, c.bead_lo, c.controlled = 0, 0, 0        # a draw that no number satisfies
        if kind == "arena" and c.move == L.SLIDE:
            c.amp_bead, c.bead_lo, c.controlled = 200, 200, 0    # windows past the arena now and then
    return s


@pytest.mark.parametrize("mode", [L.RNG_PHILOX, L.RNG_GLIBC])
@pytest.mark.parametrize("kind,error", [("draw", 5), ("arena", 2)])
def test_state_after_an_error(kind, error, mode):
    import torch

    from chromo_amd.engine import DeviceReplicas
    print("error state", kind, mode, flush=True)
    systems = [_system(kind, i) for i in range(4)]

    def run(waves):
        dr = DeviceReplicas([s.chain for s in systems], [s.field for s in systems],
                            [copy.deepcopy(s.ctrls) for s in systems], rng_mode=mode, seeds=[5, 6, 7, 8],
                            streams=[0, 1, 2, 3], caps=[(40, 40)] * 4, log_cap=4000)
        dr.np_seed([9, 10, 11, 12])
        dr.run(30, waves=waves, sync=False)
        torch.cuda.synchronize()
        return dr
    one, two = run(1), run(2)
    a, b = one.counter_array(), two.counter_array()
    assert np.all(a[:, L.CNT_ERROR] == error)
    for w in (L.CNT_ERROR, L.CNT_PROPOSALS, L.CNT_ACCEPTED, L.CNT_SUM_N, L.CNT_SUM_BINS, L.CNT_BYTES, L.CNT_LOGGED):
        assert np.array_equal(a[:, w], b[:, w]), w
    for i in range(4):
        for x, y in zip(one.positions(i), two.positions(i)):
            assert np.array_equal(x, y), i
        assert np.array_equal(one.binder_states(i), two.binder_states(i))
        assert np.array_equal(one.density_of(i), two.density_of(i))
        assert np.array_equal(one.rng_words(i), two.rng_words(i)), i
        assert one.controllers(i) == two.controllers(i)
        assert np.array_equal(one.logs(i), two.logs(i))
