"""Scans of 47 slices keep their intensity: the sum over every detected angle against the float64 oracle, where errors of
the transforms' constants add up slice by slice.

A slice multiplies a wave by two float32 factors, t and the propagator, each off by 2^-24 at most: both off by all of it
the same way in every slice move the intensity by 4 * 2^-24 = 2.4e-7 a slice, 1.12e-5 over 47 slices.
"""
import numpy as np
import pytest

from oracle import oracle as O

import simulatokit_amd as sk
from simulatokit_amd.workloads import SRTIO3_A, srtio3

pytestmark = pytest.mark.gpu

SLICES = 47  # 24 cells of SrTiO3, 2 A each
BOUND = 4 * 2.0 ** -24 * SLICES


@pytest.fixture(scope="module", autouse=True)
def device():
    if not sk.hip_is_available():
        pytest.fail("no HIP device: " + sk._native.last_error())


def errors(nx, ny, options):
    """(total - exact) / exact of every option's scan"""
    st = srtio3(max(1, round(nx / 64)), max(1, round(ny / 64)), 24)
    pot = sk.Potential(st, nx, ny, slice_thickness=2.0)
    assert pot.slice_count == SLICES
    probe = sk.Probe(sk.ElectronBeam(200e3), pot.grid, sk.Aperture(20.0))
    positions = [[0.4, 0.9], [2.1, 0.3]]
    prepared = pot.prepare(probe.beam)
    V, _ = O.potential(nx, ny, st.numbers, st.positions, st.box, pot.slice_thicknesses)
    want = O.stem_scan([V], [pot.slice_thicknesses], (st.box[0], st.box[1]), 200e3, 20.0, positions,
                       [O.det_pixelated("cutoff")])[0]
    want = np.asarray(want).reshape(len(positions), -1).sum(1)
    out = []
    for o in options:
        got = sk.STEM.scan(probe, [prepared], positions, [sk.PixelatedDetector("cutoff")], o)[0].values
        out.append(np.asarray(got).reshape(len(positions), -1).sum(1) / want - 1)
        print(nx, ny, o.fast_path, out[-1], flush=True)
    prepared.release()
    return out


@pytest.mark.parametrize("nx,ny", [(67, 67), (124, 124), (131, 97), (257, 211)])
def test_bluestein_scans_keep_their_intensity(nx, ny):
    for e in errors(nx, ny, [sk.ExecutionOptions()]):
        assert np.abs(e).max() <= BOUND


@pytest.mark.parametrize("nx,ny", [(198, 198), (486, 486)])
def test_both_paths_of_smooth_scans_keep_their_intensity(nx, ny):
    """The generic passes have other constants than the two-stage ones: each path's propagators correct its own."""
    for e in errors(nx, ny, [sk.ExecutionOptions(), sk.ExecutionOptions(fast_path=False)]):
        assert np.abs(e).max() <= BOUND
