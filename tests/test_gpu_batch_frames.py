"""Batch groups of plates in frames of their own have one launch shape: the
tuner has nothing to time there and reports no block size; the group that is summed through
contributions keeps its own."""

import os

import pytest

from finite_element_method_amd import FEM, FEMBatch
from tests.test_gpu_plate_frames import _tilted_fan, _turn, _vault

pytestmark = pytest.mark.gpu


def test_no_block_size_for_plate_frames(gpu, monkeypatch):
    monkeypatch.setitem(os.environ, "FEM_AMD_TUNE_CACHE", "")
    batch = FEMBatch([FEM.from_mesh(m) for m in (_vault(13, 9, 7, _turn()), _vault(7, 6, 6), _tilted_fan(9))])
    groups = batch.autotune().split("; ")
    print(groups, flush=True)
    assert groups[0] == "group 0: generic" and groups[1].startswith("group 1: generic block=")
