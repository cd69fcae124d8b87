"""Energy and gradients on grids at the edges of the tile kernel (tiles of at most 8
voxels per axis): axes of one voxel, of one tile that wraps onto itself, of two tiles
that are each other's neighbours on both sides, ragged last tiles, and more beads in a
tile than it notes down.  Against the FP64 PyTorch transcription; the caller's-workspace
entry point against the allocating one, bit for bit."""
import ctypes

import numpy as np
import pytest
import torch

from chromo_amd import _lib as L
from chromo_amd import workloads as W
from test_gpu_adjoint import torch_energy

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,B,N", [((1, 1, 1), 1, 40), ((1, 9, 16), 2, 300), ((2, 3, 8), 3, 500), ((8, 8, 8), 4, 3000),
                                   ((9, 10, 15), 4, 700), ((16, 17, 8), 2, 900), ((23, 7, 31), 1, 5000),
                                   ((64, 2, 1), 3, 257), ((33, 40, 25), 4, 2)])
def test_tile_edges(n, B, N):
    from chromo_amd.energy import EnergyModel
    from chromo_amd.engine import _current_stream
    print("adjoint tiles", n, B, N, flush=True)
    s = W.make_system(N, B, 8, seed=sum(n) + B, eps=[-4.0, -2.5, -3.0, -1.5][:B], mu=[-0.4, 0.3, -1.0, 0.2][:B],
                      cross_eps=0.6, chi=1.3)
    s.chain.states = np.random.RandomState(N).randint(0, 4, size=(N, B))
    s.chain.F = np.concatenate([s.chain.F, s.chain.F[:, :, -1:]], axis=2)[:, :, :4]
    f = s.field
    f.nx, f.ny, f.nz = n
    f.x_width, f.y_width, f.z_width = 30.0 * n[0], 30.0 * n[1], 30.0 * n[2]
    f.vf_limit = 1e9
    model = EnergyModel(s.chain, f, s.binders)
    r = torch.tensor(s.chain.r, dtype=torch.float64, device="cuda")
    th = torch.tensor(model.theta0, dtype=torch.float64, device="cuda")

    def call(ws):
        E = torch.zeros(4, dtype=torch.float64, device="cuda")
        gr, gt = torch.full_like(r, float("nan")), torch.full_like(th, float("nan"))
        args = [ctypes.byref(model.m), r.data_ptr(), th.data_ptr(), E.data_ptr(), gr.data_ptr(), gt.data_ptr()]
        if ws:
            nb = model.lib.chromo_energy_adjoint_bytes(ctypes.byref(model.m))
            buf = torch.full((nb,), 0x5A, dtype=torch.uint8, device="cuda")
            L.check(model.lib.chromo_energy_adjoint_ws(*args, buf.data_ptr(), nb, _current_stream()))
            assert model.lib.chromo_energy_adjoint_ws(*args, buf.data_ptr(), nb - 1, _current_stream()) == -1
        else:
            L.check(model.lib.chromo_energy_adjoint(*args, _current_stream()))
        torch.cuda.synchronize()
        return E, gr, gt
    E, gr, gt = call(False)
    for a, b in zip((E, gr, gt), call(True)):
        assert torch.equal(a, b)
    rt = r.cpu().requires_grad_(True)
    tht = th.cpu().requires_grad_(True)
    Et, el, fi, bi = torch_energy(s, rt, tht)
    Et.backward()
    assert np.allclose(E.cpu().numpy(), [Et.item(), el.item(), fi.item(), bi.item()], rtol=1e-11, atol=1e-9)
    assert np.allclose(gr.cpu().numpy(), rt.grad.numpy(), rtol=1e-9, atol=1e-9)
    assert np.allclose(gt.cpu().numpy(), tht.grad.numpy(), rtol=1e-10, atol=1e-9)
