"""The energy adjoint at weights that lie halfway between two values of a fixed-point word:
coordinates that are multiples of a power of two, with a voxel side that is one.  Against
the FP64 transcription, with the bonds' energy off so that the field's gradient shows.

Tolerance: a field term is a sum of fewer than 10 products with weights exact to 2^-60 and
one rounding each (2^-53), a voxel sum has 512 terms: below 1e-13 of the largest value.  A
weight off by one in a 28-bit word would be off by 3.7e-9."""
import numpy as np
import pytest
import torch

from chromo_amd import workloads as W
from test_gpu_adjoint import torch_energy

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [28, 30, 32])
def test_ties_among_the_weights(bits):
    from chromo_amd.energy import EnergyModel, energy
    print("adjoint ties", bits, flush=True)
    N, B, n, side = 300, 3, 8, 32.0
    s = W.make_system(N, B, n, seed=bits, eps=[-4.0, -2.5, -3.0], mu=[-0.4, 0.3, -1.0], cross_eps=0.6, chi=1.3)
    rs = np.random.RandomState(bits)
    s.chain.states = rs.randint(0, 4, size=(N, B))
    s.chain.F = np.concatenate([s.chain.F, s.chain.F[:, :, -1:]], axis=2)[:, :, :4]
    s.chain.bonds = np.zeros_like(s.chain.bonds)
    f = s.field
    f.x_width = f.y_width = f.z_width = side * n
    f.vf_limit = 1e9
    # two axes on voxel centres, the third an odd multiple of half a unit of the word away
    q = rs.randint(0, n, size=(N, 3)).astype(np.float64)
    odd = 2.0 * np.concatenate([[0, 1, 2 ** bits - 1, 2 ** (bits - 1)], rs.randint(0, 2 ** 28, size=N - 4)]) + 1
    q[np.arange(N), rs.randint(0, 3, size=N)] += odd * 2.0 ** -(bits + 1)
    r = torch.tensor(q * side - side * n / 2 + side / 2, dtype=torch.float64)
    assert np.array_equal((r.numpy() + side * n / 2 - side / 2) / side, q)     # no coordinate was rounded
    model = EnergyModel(s.chain, s.field, s.binders)
    th = torch.tensor(model.theta0, dtype=torch.float64)
    E, gr, gt = energy(model, r.cuda(), th.cuda())
    rt, tht = r.clone().requires_grad_(True), th.clone().requires_grad_(True)
    Et, _, _, _ = torch_energy(s, rt, tht)
    Et.backward()
    assert np.allclose(gt.cpu().numpy(), tht.grad.numpy(), rtol=1e-12, atol=0)
    assert np.max(np.abs(gr.cpu().numpy() - rt.grad.numpy())) <= 1e-12 * float(rt.grad.abs().max())
