"""Waves given in real space enter the Bluestein passes through the band's convolution: plane waves and waves with every
frequency, singly and several in one launch, at the edges of the convolutions' ranges and past the full-width ones' (865
and above), against the float64 oracle and the generic passes.

Two slices in float32 come to about 1e-6 of the largest value: 1e-5 holds them.
"""
import numpy as np
import pytest

from oracle import oracle as O
from tests.conftest import rel_max

import simulatokit_amd as sk
from simulatokit_amd.workloads import srtio3

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    if not sk.hip_is_available():
        pytest.fail("no HIP device: " + sk._native.last_error())


@pytest.mark.parametrize("nx,ny", [(67, 67), (66, 68), (97, 134), (512, 257), (130, 346), (67, 509), (600, 614), (68, 865),
                                   (70, 1037)])
def test_waves_enter_as_the_oracle(nx, ny):
    st = srtio3(max(1, round(nx / 64)), max(1, round(ny / 64)), 1)
    pot = sk.Potential(st, nx, ny, slice_thickness=2.0)
    beam = sk.ElectronBeam(200e3)
    prepared = pot.prepare(beam)
    rng = np.random.default_rng(nx + ny)
    fields = [np.ones((nx, ny), complex)] + [rng.normal(size=(nx, ny)) + 1j * rng.normal(size=(nx, ny)) for _ in range(2)]
    waves = [sk.Waves(f, pot.grid, beam) for f in fields]
    V, _ = O.potential(nx, ny, st.numbers, st.positions, st.box, pot.slice_thicknesses)
    batch = sk.Multislice.run_batch(waves, prepared)
    for w, f, b in zip(waves, fields, batch):
        want = O.multislice(V, pot.slice_thicknesses, (st.box[0], st.box[1]), 200e3, f)[0]
        one = sk.Multislice.run(w, prepared)[0]
        generic = sk.Multislice.run(w, prepared, options=sk.ExecutionOptions(fast_path=False))[0]
        assert rel_max(one.field, want) <= 1e-5
        assert rel_max(one.field, generic.field) <= 1e-5
        assert np.array_equal(one.field, b.field)
    prepared.release()
