"""The backward's block records are made by the first backward, not by compliance
calls, which do not read them; either order of the calls gives the same bits."""

import numpy as np
import pytest

from finite_element_method_amd import FEM, meshgen
from tests.test_gpu_plate_frames import _turn, _vault

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _grown(call):
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    out = call()
    torch.cuda.synchronize()
    return out, before - torch.cuda.mem_get_info()[0]


def _bits(out):
    return [t.view(torch.int64) for t in list(out[0].values()) + ([] if out[1] is None else [out[1]])]


@pytest.mark.parametrize("kind", ["shell", "frame"])
def test_compliance_makes_no_records(gpu, kind):
    mesh = _vault(420, 310, 3, _turn()) if kind == "shell" else meshgen.beam_frame(36, 35, 34, seed=4)
    xyz = kind == "shell"
    record = 32 * (16 if kind == "shell" else 4) * mesh.n_elements
    print("case", kind, mesh.n_elements, record, flush=True)
    models = [FEM.from_mesh(mesh) for _ in range(2)]
    for m in models:
        m.build_pattern()
    nnz = models[0].csr_info()[1]
    g = torch.randn(nnz, dtype=torch.float64, device="cuda")
    u = torch.randn(6 * mesh.n_nodes, dtype=torch.float64, device="cuda")
    for m in models:  # the outputs' memory is torch's by then
        [torch.empty((mesh.n_elements, 11), dtype=torch.float64, device="cuda") for _ in range(4)]
    first, maps = _grown(lambda: models[0].compliance_sensitivity(u, xyz=xyz))
    second, records = _grown(lambda: models[0].backward(g, xyz=xyz))
    _, both = _grown(lambda: models[1].backward(g, xyz=xyz))
    print("device bytes", maps, records, both, flush=True)
    slack = 8 << 20  # the allocator's pages
    assert records >= record - slack and maps <= both - record + slack
    assert all(torch.equal(a, b) for a, b in zip(_bits(second), _bits(models[1].backward(g, xyz=xyz))))
    assert all(torch.equal(a, b) for a, b in zip(_bits(first), _bits(models[1].compliance_sensitivity(u, xyz=xyz))))
