"""Energy and gradients of condensed chains, whose tiles have long lists and are split into
parts: axes that are halved and axes too short for it, a tile that wraps onto itself, more
beads near a part, and in its cells, than it notes down at once, long lists beside short
ones; and a chain too short to be split.  Against the FP64 transcription; twice the same
bits; the energy alone as with gradients.

Tolerances: a voxel's density is a sum of up to 10^4 terms, in the transcription one after
the other (10^4 2^-53, 1e-12, at worst); the energies add up such voxels' terms, and a
gradient is a difference of interpolated values up to some 10 times its largest size."""
import numpy as np
import pytest
import torch

from chromo_amd import workloads as W
from test_gpu_adjoint import torch_energy

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,B,N,side", [((4, 4, 4), 4, 34000, 4), ((3, 8, 5), 3, 36000, 3), ((1, 2, 12), 2, 33000, 4),
                                        ((16, 17, 24), 2, 50000, 10), ((8, 8, 8), 4, 40000, 8),
                                        ((31, 7, 23), 1, 60000, 7), ((40, 33, 25), 4, 45000, 12),
                                        ((24, 24, 24), 3, 9000, 7)])
def test_condensed(n, B, N, side):
    from chromo_amd.energy import EnergyModel, energy
    print("adjoint, condensed", n, B, N, side, flush=True)
    s = W.make_system(N, B, 8, seed=sum(n) + B, eps=[-4.0, -2.5, -3.0, -1.5][:B], mu=[-0.4, 0.3, -1.0, 0.2][:B],
                      cross_eps=0.6, chi=1.3)
    rs = np.random.RandomState(N)
    s.chain.states = rs.randint(0, 4, size=(N, B))
    s.chain.F = np.concatenate([s.chain.F, s.chain.F[:, :, -1:]], axis=2)[:, :, :4]
    # the walk folded into a cube of `side` voxels across a periodic corner of the box
    w = 30.0 * side
    r = np.mod(s.chain.r, 2 * w)
    s.chain.r = np.where(r > w, 2 * w - r, r) + 15.0 * np.array(n) - w / 3
    f = s.field
    f.nx, f.ny, f.nz = n
    f.x_width, f.y_width, f.z_width = 30.0 * n[0], 30.0 * n[1], 30.0 * n[2]
    f.vf_limit = 1e9
    model = EnergyModel(s.chain, f, s.binders)
    r = torch.tensor(s.chain.r, dtype=torch.float64, device="cuda")
    th = torch.tensor(model.theta0, dtype=torch.float64, device="cuda")
    E, gr, gt = energy(model, r, th)
    for a, b in zip((E, gr, gt), energy(model, r, th)):
        assert torch.equal(a, b)
    assert torch.equal(energy(model, r, th, grad=False)[0], E)
    rt = r.cpu().requires_grad_(True)
    tht = th.cpu().requires_grad_(True)
    Et, el, fi, bi = torch_energy(s, rt, tht)
    Et.backward()
    g = rt.grad.numpy()
    assert np.allclose(E.cpu().numpy(), [Et.item(), el.item(), fi.item(), bi.item()], rtol=1e-10, atol=1e-9)
    assert np.max(np.abs(gr.cpu().numpy() - g)) <= 1e-10 * np.max(np.abs(g))
    assert np.allclose(gt.cpu().numpy(), tht.grad.numpy(), rtol=1e-10, atol=1e-9)
