"""The speculative kernel's order of slots: controller blocks of one proposal, a single
controller, controllers without proposals, and slots given back to the one-at-a-time
path while later ones are in flight.

The one-wavefront kernel, two and four wavefronts have to give the same chains bit for
bit, the random streams' final positions included.
"""
import copy

import numpy as np
import pytest

from chromo_amd import _lib as L
from chromo_amd import workloads as W

pytestmark = pytest.mark.gpu

CASES = {
    "ones": dict(per_cycle=(1, 1, 1, 1, 1)),
    "mixed": dict(per_cycle=(3, 1, 9, 2, 5)),
    "single": dict(per_cycle=(11, 1, 1, 1, 1), only=L.CRANK_SHAFT),
    "pair": dict(per_cycle=(1, 1, 2, 1, 4), only=(L.CRANK_SHAFT, L.CHANGE_BINDING_STATE)),
    # 4 nm voxels: long windows touch more voxels than a block holds
    "overflow": dict(per_cycle=(7, 2, 7, 2, 3), voxel=4.0, grid=40, amp=150),
    # whole-chain windows among the short ones
    "short chain": dict(per_cycle=(6, 3, 6, 3, 3), N=12, amp=12),
}


@pytest.mark.parametrize("mode", [L.RNG_PHILOX, L.RNG_GLIBC])
@pytest.mark.parametrize("kind", list(CASES))
def test_slot_order(kind, mode):
    import torch

    from chromo_amd.engine import DeviceReplicas
    k = CASES[kind]
    print("slot order", kind, mode, flush=True)
    units = torch.cuda.get_device_properties(0).multi_processor_count
    kw = {"voxel": k["voxel"]} if "voxel" in k else {}
    systems = []
    for i in range(4):
        s = W.make_system(k.get("N", 400 + 37 * i), 1 + i, k.get("grid", 6), seed=900 + i, chi=0.4,
                          per_cycle=k["per_cycle"], **kw)
        s.field.vf_limit = 1e9
        only = k.get("only")
        for c in s.ctrls:
            if only is not None and c.move not in (only if isinstance(only, tuple) else (only,)):
                c.on = 0
            if "amp" in k and c.move in (L.CRANK_SHAFT, L.SLIDE, L.END_PIVOT):
                c.amp_bead = min(k["amp"], int(c.bead_hi))
                c.bead_lo = c.bead_hi
        systems.append(s)

    def make(idx):
        dr = DeviceReplicas([systems[i % 4].chain for i in idx], [systems[i % 4].field for i in idx],
                            [copy.deepcopy(systems[i % 4].ctrls) for i in idx], rng_mode=mode,
                            seeds=[5 + i for i in idx], streams=list(idx))
        dr.np_seed([9 + i for i in idx])
        return dr
    steps = 5
    one, four = make(range(8)), make(range(8))
    one.run(steps, waves=1)
    four.run(steps, waves=2)
    many = make(range(units + 1))
    many.run(steps, waves=2)
    for other in (four, many):
        for i in range(8):
            for a, b in zip(one.positions(i), other.positions(i)):
                assert np.array_equal(a, b), i
            assert np.array_equal(one.binder_states(i), other.binder_states(i))
            assert np.array_equal(one.density_of(i), other.density_of(i))
            assert np.array_equal(one.rng_words(i), other.rng_words(i))
            assert one.controllers(i) == other.controllers(i)
    ca, cb = one.counter_array(), four.counter_array()
    for w in (L.CNT_PROPOSALS, L.CNT_ACCEPTED, L.CNT_SUM_N, L.CNT_SUM_BINS, L.CNT_BYTES):
        assert np.array_equal(ca[:, w], cb[:, w]), w


@pytest.mark.parametrize("mode", [L.RNG_PHILOX, L.RNG_GLIBC])
@pytest.mark.parametrize("kind", ["mixed", "overflow", "short chain", "twist"])
def test_one_proposal_launches(kind, mode):
    """One launch per proposal draws the usual proposals at once and the others word by
    word: the persistent kernel's chains for every binder count."""
    from chromo_amd.engine import DeviceReplicas
    k = CASES["mixed" if kind == "twist" else kind]
    print("one-proposal launches", kind, mode, flush=True)
    kw = {"voxel": k["voxel"]} if "voxel" in k else {}
    for B in (1, 2, 3, 4):
        build = W.make_twist_system if kind == "twist" else W.make_system
        s = build(k.get("N", 300), B, k.get("grid", 6), seed=950 + B, chi=0.4, per_cycle=k["per_cycle"], **kw)
        s.field.vf_limit = 1e9
        for c in s.ctrls:
            if "amp" in k and c.move in (L.CRANK_SHAFT, L.SLIDE, L.END_PIVOT):
                c.amp_bead = min(k["amp"], int(c.bead_hi))
                c.bead_lo = c.bead_hi

        def make():
            dr = DeviceReplicas([s.chain], [s.field], [copy.deepcopy(s.ctrls)], rng_mode=mode, seeds=[3], streams=[1])
            dr.np_seed([4])
            return dr
        a, b = make(), make()
        a.run(4, waves=1)
        b.run_plain(4)
        for x, y in zip(a.positions(0), b.positions(0)):
            assert np.array_equal(x, y), B
        assert np.array_equal(a.binder_states(0), b.binder_states(0))
        assert np.array_equal(a.density_of(0), b.density_of(0))
        assert np.array_equal(a.rng_words(0), b.rng_words(0))
        assert a.controllers(0) == b.controllers(0)
