"""fem_assemble_into takes an array of doubles: one that starts at an odd multiple
of 8 bytes gets the values of an aligned one, and nothing beside it is written
(frames, frames with trusses, shells, flat plates, the contribution path)."""

import numpy as np
import pytest

from finite_element_method_amd import FEM, meshgen
from tests.test_gpu_bar_records import _chain, _load
from tests.test_gpu_plate_frames import _tilted_fan, _turn, _vault

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _braced(n):
    data = _chain(n, n, False, True)
    return _load(FEM.create(1e-4, 1e-12, n), *data)


MODELS = {
    "beam": lambda: FEM.from_mesh(meshgen.beam_frame(2, 1, 1, seed=1)),
    "frame": lambda: FEM.from_mesh(meshgen.beam_frame(5, 6, 7, seed=2)),
    "braced_41": lambda: _braced(41),
    "braced_90": lambda: _braced(90),
    "shell": lambda: FEM.from_mesh(_vault(13, 9, 7, _turn())),
    "plate": lambda: FEM.from_mesh(meshgen.plate_grid(13, 9, seed=3)),
    "fan": lambda: FEM.from_mesh(_tilted_fan(9)),
}


@pytest.mark.parametrize("name", sorted(MODELS))
def test_any_place(gpu, name):
    m = MODELS[name]()
    want = m.stiffness_csr()[2]
    print("case", name, len(want), m.assembly_path(), flush=True)
    for first in (0, 1, 2, 3):
        room = torch.full((len(want) + 5,), 7.0, dtype=torch.float64, device="cuda")
        m.assemble_into(room[first:first + len(want)])
        torch.cuda.synchronize()
        got = room.cpu().numpy()
        assert np.array_equal(got[first:first + len(want)].view(np.uint64), want.view(np.uint64))
        assert np.all(got[:first] == 7.0) and np.all(got[first + len(want):] == 7.0)
