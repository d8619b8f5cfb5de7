"""fem_update_* against work on several streams and in captured graphs, for every
value path: assemblies on two streams after an update, a captured assembly
replayed after updates, a capture as the first call after an update."""

import numpy as np
import pytest

from finite_element_method_amd import BEAM, DeviceError, FEM, PLATE, TRUSS, meshgen
from tests.test_gpu_bar_records import _chain, _load
from tests.test_gpu_plate_frames import _turn, _vault

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _cuda(a):
    return torch.tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda")


class _Meshed:
    """A mesh of one element type; variant k has other sizes and coordinates."""

    def __init__(self, mesh, etype, column, one_material=False):
        self.mesh, self.etype, self.column = mesh, etype, column
        if one_material:
            mesh.props[:, [0, 1, 3]] = mesh.props[0, [0, 1, 3]]

    def data(self, k):
        m = self.mesh
        props = m.props.copy()
        props[:, self.column] *= np.random.default_rng(k).uniform(0.7, 1.4, len(props))
        return m.xyz * (1.0 + 0.25 * k), {self.etype: props}

    def model(self, k):
        m, (xyz, props) = self.mesh, self.data(k)
        return FEM.from_mesh(meshgen.Mesh(m.kind, m.node_numbers, xyz, m.numbers, m.conn, props[self.etype]))


class _Braced:
    """A chain of beams braced by trusses."""

    def __init__(self, n):
        self.chain = _chain(n, n, False, True)

    def data(self, k):
        xyz, conn, props, braces = self.chain
        props = props.copy()
        props[:, 2] *= np.random.default_rng(k).uniform(0.7, 1.4, len(props))
        return xyz * (1.0 + 0.25 * k), {BEAM: props}

    def model(self, k):
        xyz, conn, props, braces = self.chain
        x, p = self.data(k)
        return _load(FEM.create(1e-4, 1e-12, len(xyz)), x, conn, p[BEAM], braces)


CASES = {
    "lattice": lambda: _Meshed(meshgen.truss_lattice(9, seed=1), TRUSS, 1),
    "frame": lambda: _Meshed(meshgen.beam_frame(6, 7, 5, seed=2), BEAM, 2),
    "braced_chain": lambda: _Braced(90),
    "shell": lambda: _Meshed(_vault(19, 14, 3, _turn()), PLATE, 2),
    "plate": lambda: _Meshed(meshgen.plate_grid(23, 17, seed=4), PLATE, 2),
    "plate_materials": lambda: _Meshed(_materials(meshgen.plate_grid(23, 17, seed=5)), PLATE, 2),
}


class _Mixing(_Meshed):
    """Plates of one material in even variants, another in each, and of several in odd ones."""

    def data(self, k):
        xyz, props = super().data(k)
        props[PLATE][:, [0, 1]] *= [1.0 + 0.5 * k, 1.0 + 0.1 * k]
        if k % 2:
            props[PLATE][3::5, 0] *= 1.5
        return xyz, props


def _materials(mesh):
    mesh.props[:, 0] *= np.random.default_rng(6).uniform(0.5, 2.0, mesh.n_elements)
    return mesh


def _case(name):
    return CASES[name]() if name in CASES else _Mixing(meshgen.plate_grid(23, 17, seed=7), PLATE, 2)


def _update(m, case, k, stream=None):
    xyz, props = case.data(k)
    for t, p in props.items():
        m.update_params(t, _cuda(p), stream=stream)
    m.update_nodes(_cuda(xyz), stream=stream)


def _want(case, k):
    return torch.tensor(case.model(k).stiffness_csr()[2], device="cuda")


def _same(a, b):
    return torch.equal(a.view(torch.int64), b.view(torch.int64))


@pytest.mark.parametrize("name", sorted(CASES) + ["plate_mixing"])
def test_two_streams_after_an_update(gpu, name):
    """The update has finished when it returns: assemblies on any stream see it."""
    case = _case(name)
    print("case", name, flush=True)
    m = case.model(0)
    m.stiffness_csr()
    streams = [torch.cuda.Stream() for _ in range(3)]
    out = [torch.empty(m.csr_info()[1], dtype=torch.float64, device="cuda") for _ in streams]
    torch.cuda.synchronize()
    for k in (1, 2, 3):
        _update(m, case, k, stream=streams[k % 3])
        for s, o in zip(streams, out):
            m.assemble_into(o, stream=s)
        torch.cuda.synchronize()
        want = _want(case, k)
        assert all(_same(o, want) for o in out), k


@pytest.mark.parametrize("name", sorted(CASES) + ["plate_mixing"])
def test_captured_assembly_after_updates(gpu, name):
    """A captured assembly replays with the values of the last update; a capture as
    the first call after an update leaves the eager calls as they are."""
    case = _case(name)
    print("case", name, flush=True)
    m = case.model(0)
    m.stiffness_csr()
    m.set_option("time_assembly", 0)
    eager, out = (torch.zeros(m.csr_info()[1], dtype=torch.float64, device="cuda") for _ in range(2))
    _update(m, case, 1)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        m.assemble_into(out, stream=torch.cuda.current_stream())
    m.assemble_into(eager)
    torch.cuda.synchronize()
    assert _same(eager, _want(case, 1))
    for k in (1, 2, 3, 4):
        _update(m, case, k)
        graph.replay()
        torch.cuda.synchronize()
        want = _want(case, k)
        assert _same(out, want), k
        m.assemble_into(eager)
        torch.cuda.synchronize()
        assert _same(eager, want), k


def _keep_busy(stream, room):
    """Queues some hundred milliseconds of copies on `stream`; the event after them."""
    with torch.cuda.stream(stream):
        for _ in range(120):
            room.mul_(1.0)
        return stream.record_event()


def test_update_does_not_wait_for_other_work(gpu):
    """An update waits for its own model's work, not for what other programs of the
    process have queued.  Streams may share a hardware queue, in whose order
    they then run: one of several streams has to be passed."""
    case = CASES["lattice"]()
    m = case.model(0)
    m.stiffness_csr()
    mine = torch.cuda.Stream()
    out = torch.empty(m.csr_info()[1], dtype=torch.float64, device="cuda")
    _update(m, case, 1, stream=mine)
    xyz, props = case.data(2)
    xyz, props = _cuda(xyz), _cuda(props[TRUSS])
    room = torch.ones(1 << 29, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    passed = []
    for _ in range(3):
        other = torch.cuda.Stream()
        m.assemble_into(out, stream=mine)
        end = _keep_busy(other, room)
        m.update_params(TRUSS, props, stream=mine)
        m.update_nodes(xyz, stream=mine)
        passed.append(not end.query())
        torch.cuda.synchronize()
    print("passed", passed, flush=True)
    assert any(passed)


@pytest.mark.parametrize("name", ["lattice", "frame", "shell", "plate"])
def test_update_waits_for_its_own_model(gpu, name):
    """An assembly still queued on another stream, eager or as a captured graph's
    replay, has the values of before the update."""
    case = CASES[name]()
    print("case", name, flush=True)
    m = case.model(0)
    m.stiffness_csr()
    m.set_option("time_assembly", 0)
    mine, other = torch.cuda.Stream(), torch.cuda.Stream()
    out, replayed = (torch.zeros(m.csr_info()[1], dtype=torch.float64, device="cuda") for _ in range(2))
    room = torch.ones(1 << 28, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    for k in (1, 2):
        _keep_busy(other, room)
        m.assemble_into(out, stream=other)
        _update(m, case, k, stream=mine)
        torch.cuda.synchronize()
        assert _same(out, _want(case, k - 1)), k
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        m.assemble_into(replayed, stream=torch.cuda.current_stream())
    for k in (3, 4):
        _keep_busy(other, room)
        with torch.cuda.stream(other):
            graph.replay()
        _update(m, case, k, stream=mine)
        torch.cuda.synchronize()
        assert _same(replayed, _want(case, k - 1)), k


@pytest.mark.parametrize("name", ["frame", "shell", "plate"])
def test_update_in_a_capture_is_refused(gpu, name):
    """It changes nothing: the capture goes on, and the model is as it was, its
    pattern included, until the next update."""
    case = CASES[name]()
    print("case", name, flush=True)
    m = case.model(0)
    m.stiffness_csr()
    m.set_option("time_assembly", 0)
    xyz, props = case.data(1)
    xyz, props = _cuda(xyz), {t: _cuda(p) for t, p in props.items()}
    eager, out = (torch.zeros(m.csr_info()[1], dtype=torch.float64, device="cuda") for _ in range(2))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        with pytest.raises(DeviceError, match="captured"):
            m.update_nodes(xyz)
        for t, p in props.items():
            with pytest.raises(DeviceError, match="captured"):
                m.update_params(t, p)
        m.assemble_into(out, stream=torch.cuda.current_stream())
    want = _want(case, 0)
    for _ in range(2):
        graph.replay()
        m.assemble_into(eager)
        torch.cuda.synchronize()
        assert _same(out, want) and _same(eager, want)
    _update(m, case, 1)
    graph.replay()
    m.assemble_into(eager)
    torch.cuda.synchronize()
    want = _want(case, 1)
    assert _same(out, want) and _same(eager, want)


@pytest.mark.parametrize("name", ["lattice", "shell", "plate"])
def test_update_waits_for_its_values(gpu, name):
    """Values made on torch's current stream, as the last of much other work, and
    the copy that a transposed tensor needs: the update's own stream waits for both."""
    case = CASES[name]()
    print("case", name, flush=True)
    m = case.model(0)
    m.stiffness_csr()
    maker, mine = torch.cuda.Stream(), torch.cuda.Stream()
    out = torch.zeros(m.csr_info()[1], dtype=torch.float64, device="cuda")
    room = torch.ones(1 << 28, dtype=torch.float64, device="cuda")
    for k, stream in ((1, mine), (2, None), (3, mine.cuda_stream), (4, 0)):
        xyz, props = case.data(k)
        xyz, props = _cuda(xyz), {t: _cuda(p.T) for t, p in props.items()}
        torch.cuda.synchronize()
        _keep_busy(maker, room)
        with torch.cuda.stream(maker):
            made = {t: p * 1.0 for t, p in props.items()}
            for t, p in made.items():
                m.update_params(t, p.t(), stream=stream)
            _keep_busy(maker, room)
            m.update_nodes(xyz * 1.0, stream=stream)
        m.assemble_into(out)
        torch.cuda.synchronize()
        assert _same(out, _want(case, k)), k
