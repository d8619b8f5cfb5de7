"""dL/dK gradients of plates with frames of their own (adjoint.hip, blocks read
through their records) against the oracle's reference gradients, at the edges
of the kernel's 16-element blocks: full masks (turned vaults), partial ones
(vaults along the axes); and the 16-byte
gather against one load per value, bitwise."""

import numpy as np
import pytest

from finite_element_method_amd import FEM, PLATE
from tests import adjoint_ref as ar
from tests.test_gpu_plate_frames import _turn, _vault

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("nx,ny,turned", [(1, 1, True), (5, 3, True), (4, 4, True), (17, 1, True), (1, 2, False),
                                          (5, 3, False), (8, 2, False)])
def test_shell_backward_matches_reference(gpu, nx, ny, turned):
    """Tolerances: 1e-10 for the exact splits (E, t, k), 1e-7 for the finite
    differences (nu, coordinates), as for the flat plates."""
    mesh = _vault(nx, ny, 3 * nx + ny, turn=_turn() if turned else None)
    print("case", nx, ny, turned, flush=True)
    m = FEM.from_mesh(mesh)
    rp, ci, _ = m.stiffness_csr()
    g = np.random.default_rng(nx + 7 * ny).normal(size=len(ci))
    gd = torch.tensor(g, dtype=torch.float64, device="cuda")
    grads, dxyz = m.backward(gd)
    gp = grads[PLATE].cpu().numpy()
    eg = ar.ElementGrad(mesh, rp, ci, g)
    ref = np.array([ar.plate_param_grads(mesh, e, eg.block(PLATE, e)) for e in range(mesh.n_elements)])
    for i, tol in ((0, 1e-10), (1, 1e-7), (2, 1e-10), (3, 1e-10)):
        assert ar.rel_err(gp[:, i], ref[:, i]) < tol, (i, ar.rel_err(gp[:, i], ref[:, i]))
    refx = ar.node_coord_grads(mesh, PLATE, eg, 1e-4 / max(nx, ny))
    assert ar.rel_err(dxyz.cpu().numpy(), refx) < 1e-7, ar.rel_err(dxyz.cpu().numpy(), refx)
    m.set_option("wide_loads", 0)
    narrow, nxyz = m.backward(gd)
    assert torch.equal(narrow[PLATE].view(torch.int64), grads[PLATE].view(torch.int64))
    assert torch.equal(nxyz.view(torch.int64), dxyz.view(torch.int64))
