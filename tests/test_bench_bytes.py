"""The bytes bench.py's roofline figures count: those of the kernels that run."""
import pytest

import bench


def test_bytes_of_a_stage_on_box_elements():
    # per node 32*Ns + Naux*8, per element (2d+1)*8 + 2d*4
    assert bench.box_bytes_per_stage(3, 5, 4096, 5, 4) == 4096 * (125 * 192 + 80)
    assert bench.box_bytes_per_stage(2, 4, 1, 4, 0) == 16 * 128 + 56


@pytest.mark.gpu
def test_the_headline_kernel_reads_no_geometry_arrays():
    _, dg, _, _ = bench.bubble_setup(4, 4)
    naux = dg.auxstate.shape[0]
    assert bench.stage_bytes(dg, naux) == bench.box_bytes_per_stage(3, 5, 64, 5, naux)
