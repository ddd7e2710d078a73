"""The convolution kernel's set-up: the octant of displacements and its mirror
images against the oracle's full loop, and the two ways a spectrum is built
(all components at once, or one at a time beyond 2 GiB) against each other.

Tolerances: the FP64 kernel 1e-12 of its largest value (384 charges summed in
FP64 in another order); fields 5e-6 of the largest (FP32 transforms of different
padded lengths, a few 1e-7 x log2 P)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P", [(1, 2, 2), (1, 6, 10), (2, 4, 8), (4, 5, 6), (3, 8, 7), (6, 4, 130)])
def test_mirrored_kernel_vs_oracle(mm, orc, P):
    cell = (1.0, 1.5, 0.75)
    lib = mm.load()
    out = np.empty((6,) + P, np.float64)
    Pa, ca = np.array(P, np.int32), np.array(cell, np.float64)
    lib.mm_demag_kernel(Pa.ctypes.data, ca.ctypes.data, 0, 8, out.ctypes.data)
    ref = np.asarray(orc.facekernel6(P, cell)).reshape(out.shape)
    assert np.abs(out - ref).max() < 1e-12 * np.abs(ref).max()


def test_spectrum_built_by_component_equals_all_at_once(mm):
    """The kernel depends on the displacement only: a magnetised corner of a
    grid whose set-up goes one component at a time (padded 96 x 512 x 768, 3.4
    GiB of complex components) has the field of that corner alone."""
    big, small = (40, 256, 300), (4, 9, 20)
    rng = np.random.default_rng(3)
    mb = np.zeros((3,) + big, np.float32)
    ms = rng.standard_normal((3,) + small).astype(np.float32)
    mb[:, :small[0], :small[1], :small[2]] = ms
    h = []
    for size, m in ((big, mb), (small, ms)):
        s = mm.workloads.make_sim(dict(size=size, cellsize=(4e-9, 3e-9, 5e-9), msat=8e5, aexch=1.3e-11, alpha=0.1,
                                       solver="rk4", dt=1e-14, m0=m))
        h.append(s.heff(m)[:, :small[0], :small[1], :small[2]])
        s.free()
    assert np.abs(h[0] - h[1]).max() < 5e-6 * np.abs(h[1]).max()
