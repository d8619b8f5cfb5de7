"""fem_solve_pcg's kernels for small and middle systems (one workgroup for all
updates, two launches per update) have the bits of the four-launch loop: u_a, r_r,
the update count and the stop, at the sizes where the rule changes and where
their rounds end, for solves cut after 0, 1, 2, 7 and 40 updates and to the end."""

import numpy as np
import pytest

from finite_element_method_amd import meshgen
from tests.test_gpu_solve_small import _clamped

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pre", ["jacobi", "block_jacobi"])
@pytest.mark.parametrize("n_aa", [1, 24, 63, 64, 65, 256, 257, 1024, 1025, 2047, 2048, 2049, 2305, 30001, 65535, 65536,
                                  65537])
def test_same_bits(gpu, n_aa, pre):
    mesh = meshgen.plate_grid(108, 104, seed=n_aa) if n_aa > 3000 else meshgen.beam_frame(8, 8, 8, seed=n_aa)
    m = _clamped(mesh, (0, 1, 2, 3, 4, 5), n_aa, seed=n_aa)
    print("case", n_aa, pre, flush=True)
    assert m.separate()[0] == n_aa
    for updates in (0, 1, 2, 7, 40, 6000 if n_aa < 3000 else 100):
        got = []
        for plain in (0, 1):
            m.set_option("pcg_plain", plain)
            got.append(m.solve_pcg(pre, updates))
        (ua, rr, it, conv), (ua2, rr2, it2, conv2) = got
        assert it == it2 and conv == conv2, (updates, it, it2)
        assert np.array_equal(ua.view(np.uint64), ua2.view(np.uint64)), updates
        assert np.array_equal(rr.view(np.uint64), rr2.view(np.uint64)), updates
