"""Launches of many positions, where a block runs one unit after another: the same bits as launches of a few positions, on
the two-stage and the Bluestein passes, and no slower a position than launches whose waves the last-level cache holds.
"""
import numpy as np
import pytest

import simulatokit_amd as sk
from simulatokit_amd.workloads import SRTIO3_A, srtio3

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    if not sk.hip_is_available():
        pytest.fail("no HIP device: " + sk._native.last_error())


def scan_of(nx, ny):
    st = srtio3(max(1, round(nx / 64)), max(1, round(ny / 64)), 2)
    pot = sk.Potential(st, nx, ny, slice_thickness=2.0)
    probe = sk.Probe(sk.ElectronBeam(200e3), pot.grid, sk.Aperture(20.0))
    return probe, pot.prepare(probe.beam)


# positions that leave the last block and its last unit partly empty
@pytest.mark.parametrize("nx,ny,npos", [(67, 67, 6007), (97, 131, 3001), (239, 239, 2003), (347, 131, 1501),
                                        (509, 509, 1003), (613, 67, 1201), (65, 65, 6007), (96, 225, 2999),
                                        (600, 130, 1511), (1000, 66, 1201)])
def test_large_launches_give_the_bits_of_small_ones(nx, ny, npos):
    probe, prepared = scan_of(nx, ny)
    positions = np.random.default_rng(nx).uniform(0, SRTIO3_A, (npos, 2))
    dets = [sk.AnnularDetector(20, 60), sk.CenterOfMassDetector("cutoff", "mrad"), sk.SegmentedDetector(2, 4, 0, 30, 0.1)]
    large = sk.STEM.scan(probe, [prepared], positions, dets, sk.ExecutionOptions(batch=npos, tile=npos))
    sample = np.unique(np.r_[0:5, npos // 2:npos // 2 + 3, npos - 6:npos])
    small = sk.STEM.scan(probe, [prepared], positions[sample], dets, sk.ExecutionOptions(batch=3))
    for a, b in zip(large, small):
        values = np.asarray(a.values).reshape(npos, -1)[sample]
        assert np.array_equal(values, np.asarray(b.values).reshape(len(sample), -1))
    prepared.release()


@pytest.mark.parametrize("n,cached,large", [(149, 1024, 4096), (239, 539, 4096)])
def test_large_launches_cost_no_more_a_position(n, cached, large):
    """A pass reads and writes 16 bytes a compact value: at 239 x 239 0.6 MB a position, 0.15 us at 4 TB/s from HBM, half
    of what its arithmetic takes, so loads in flight together hide it. A fifth more a position is what they may cost."""
    probe, prepared = scan_of(n, n)
    positions = np.random.default_rng(n).uniform(0, SRTIO3_A, (large, 2))

    def per_position(count):
        options, best = sk.ExecutionOptions(batch=count, tile=count), np.inf
        for k in range(6):
            sk.set_timing(k > 0)
            try:
                sk.STEM.scan(probe, [prepared], positions[:count], [sk.AnnularDetector(20, 60)], options)
            finally:
                sk.set_timing(False)
            if k > 0:
                tm = sk.last_timing()
                best = min(best, (tm["row_ms"] + tm["col_ms"]) / count)
        return best

    assert per_position(large) <= 1.2 * per_position(cached)
    prepared.release()


@pytest.mark.parametrize("nx,ny", [(131, 131), (600, 97), (96, 225)])
def test_graph_replays_give_the_same_bits(nx, ny):
    # 11 positions in batches of 4: the second full batch replays the graph that was captured beside the first
    probe, prepared = scan_of(nx, ny)
    positions = np.random.default_rng(ny).uniform(0, SRTIO3_A, (11, 2))
    dets = [sk.AnnularDetector(20, 60), sk.CenterOfMassDetector("cutoff", "mrad"), sk.PixelatedDetector("cutoff")]
    eager = sk.STEM.scan(probe, [prepared], positions, dets, sk.ExecutionOptions(batch=4))
    for _ in range(2):
        replayed = sk.STEM.scan(probe, [prepared], positions, dets, sk.ExecutionOptions(batch=4, use_graph=True))
        for a, b in zip(eager, replayed):
            assert np.array_equal(np.asarray(a.values), np.asarray(b.values))
    prepared.release()
