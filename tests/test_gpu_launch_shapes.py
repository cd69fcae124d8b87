"""Every shape of the Monte Carlo kernels on one set of replicas, and the evaluator at
the edges of its 32-bead chunks.

* The one-wavefront kernel, the speculative kernel with two wavefronts (more replicas
  than compute units) and with four (fewer) give the same chains bit for bit, for every
  binder count and both random streams.
* Windows of 1 to 150 beads against the oracle, for every binder count, with and without
  sub-bin weights, and for a twisting chain; whole-chain windows on a short chain.

Bar: states, decisions, windows and voxel counts equal, dE within 1e-9 kT or 1e-12
relative, positions within 1e-9 nm.
"""
import copy

import numpy as np
import pytest

from chromo_amd import _lib as L
from chromo_amd import workloads as W

pytestmark = pytest.mark.gpu


def _dev(systems, **kw):
    from chromo_amd.engine import DeviceReplicas
    return DeviceReplicas([s.chain for s in systems], [s.field for s in systems],
                          [copy.deepcopy(s.ctrls) for s in systems], **kw)


def _wide_windows(s, amp=150):
    for c in s.ctrls:
        if c.move in (L.CRANK_SHAFT, L.SLIDE, L.END_PIVOT):
            c.amp_bead = min(amp, int(c.bead_hi))
            c.bead_lo = c.bead_hi
    return s


@pytest.mark.parametrize("mode", [L.RNG_PHILOX, L.RNG_GLIBC])
def test_shapes_identical(mode):
    import torch
    units = torch.cuda.get_device_properties(0).multi_processor_count
    n = units + 7
    print("launch shapes", mode, n, flush=True)
    systems = [W.make_system(150 + 13 * (i % 29), 1 + i % 4, 5 + i % 6, seed=400 + i, chi=0.5, cross_eps=-0.3 * (i % 2))
               for i in range(n)]
    for i, s in enumerate(systems):
        if i % 3:
            _wide_windows(s)

    def make(idx):
        dr = _dev([systems[i] for i in idx], rng_mode=mode, seeds=[5 + i for i in idx],
                  streams=list(idx))
        dr.np_seed([9 + i for i in idx])
        return dr
    one, two = make(range(n)), make(range(n))
    one.run(2, waves=1)
    two.run(2, waves=2)
    for name in ("pos", "states", "density", "rng", "ctrl"):
        assert torch.equal(getattr(one, name), getattr(two, name)), name
    some = list(range(0, n, 11))
    four = make(some)
    four.run(2, waves=2)
    for k, i in enumerate(some):
        for a, b in zip(one.positions(i), four.positions(k)):
            assert np.array_equal(a, b), i
        assert np.array_equal(one.binder_states(i), four.binder_states(k))
        assert np.array_equal(one.density_of(i), four.density_of(k))
        assert np.array_equal(one.rng_words(i), four.rng_words(k))
        assert one.controllers(i) == four.controllers(k)


@pytest.mark.parametrize("B,waves,kind", [(1, 1, ""), (2, 1, "fast"), (3, 1, ""), (4, 1, ""), (1, 2, "fast"), (2, 2, ""),
                                          (3, 2, ""), (4, 2, ""), (1, 2, "twist"), (4, 2, "twist"), (2, 2, "short")])
def test_chunk_edges(oracle, B, waves, kind):
    print("chunk edges", B, waves, kind, flush=True)
    make = W.make_twist_system if kind == "twist" else W.make_system
    N = 90 if kind == "short" else 1300
    s = _wide_windows(make(N, B, 7 if kind == "short" else 15, seed=80 + B, chi=0.4, cross_eps=-0.2 if B > 1 else 0.0,
                           per_cycle=(40, 6, 40, 10, 10)))
    if kind == "fast":
        s.field.fast_field, s.field.n_points = True, 200
    o = oracle.OracleSim(s.chain, s.field, rng_mode=0, seed=3, stream=0)
    o.np_seed(17)
    lo = o.mc_sim(4, copy.deepcopy(s.ctrls), max_logs=10 ** 5)
    dr = _dev([s], rng_mode=0, seeds=[3], log_cap=len(lo) + 10)
    dr.np_seed([17])
    dr.run(4, waves=waves)
    lg = dr.logs(0)
    assert len(lg) == len(lo)
    for f in ("move", "n", "ind0", "indf", "n_bins", "accepted"):
        assert np.array_equal(lg[f], lo[f]), f
    for f in ("dE_poly", "dE_field"):
        a, b = lg[f], lo[f]
        assert np.all(np.abs(a - b) <= 1e-9 + 1e-12 * np.maximum(np.abs(a), np.abs(b))), f
    r, _, _ = dr.positions(0)
    ro, _, _, sto = o.state()
    assert np.max(np.abs(r - ro)) < 1e-9 and np.array_equal(dr.binder_states(0), sto)
    n = lo["n"]
    assert (n <= 32).any() and ((n > 32) & (n <= 64)).any()
    if kind != "short":
        assert ((n > 64) & (n <= 96)).any() and (n > 96).any()
