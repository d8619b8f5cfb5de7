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


@pytest.mark.parametrize("kind", ["shell", "frame", "plate"])
def test_first_backward_in_a_capture(gpu, kind):
    """After a compliance call the first backward may be captured: it makes no
    records then (nothing is allocated), and its replays have the eager call's bits."""
    mesh = {"shell": lambda: _vault(11, 6, 3, _turn()), "frame": lambda: meshgen.beam_frame(5, 4, 3, seed=4),
            "plate": lambda: meshgen.plate_grid(9, 5, seed=5)}[kind]()
    xyz = kind != "frame"
    m = FEM.from_mesh(mesh)
    m.build_pattern()
    g = torch.randn(m.csr_info()[1], dtype=torch.float64, device="cuda")
    u = torch.randn(6 * mesh.n_nodes, dtype=torch.float64, device="cuda")
    m.compliance_sensitivity(u, xyz=xyz)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = m.backward(g, xyz=xyz)
    for _ in range(3):
        g.copy_(torch.randn_like(g))
        graph.replay()
        torch.cuda.synchronize()
        replayed = [t.clone() for t in _bits(out)]
        assert all(torch.equal(a, b) for a, b in zip(replayed, _bits(m.backward(g, xyz=xyz))))


@pytest.mark.parametrize("kind,size", [("shell", (1, 1)), ("shell", (5, 3)), ("shell", (17, 4)), ("vault", (5, 3)),
                                       ("vault", (8, 2)), ("frame", (2, 1, 1)), ("frame", (5, 4, 3)),
                                       ("frame", (9, 7, 8))])
def test_without_records(gpu, kind, size):
    """Blocks through the pattern's arrays (full and partial masks): the bits of those through the records."""
    mesh = meshgen.beam_frame(*size, seed=6) if kind == "frame" else _vault(*size, 7, _turn() if kind == "shell" else None)
    xyz = kind != "frame"
    print("case", kind, size, flush=True)
    m = FEM.from_mesh(mesh)
    m.build_pattern()
    g = torch.randn(m.csr_info()[1], dtype=torch.float64, device="cuda")
    want = _bits(m.backward(g, xyz=xyz))
    m.set_option("adjoint_records", 0)
    assert all(torch.equal(a, b) for a, b in zip(_bits(m.backward(g, xyz=xyz)), want))
