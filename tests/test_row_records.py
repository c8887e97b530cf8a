"""Time series of p and u written by the x passes (binary masks recording
nothing else) against the point kernel (the same masks with p_max asked for as
well): the same values bit for bit, on masks with empty rows, several points a
row, a single point, an odd number of rows, and a late first record."""

import numpy as np
import pytest

SHAPES = [(30,), (24, 15), (64, 9), (16, 10, 9)]


def _run(shape, mask, record, start):
    import kwhip
    rng = np.random.default_rng(4)
    kg = kwhip.kWaveGrid(*sum(([n, 1e-4] for n in shape), []))
    kg.setTime(14, 2e-8)
    med = {"sound_speed": 1500 + 50 * rng.random(shape), "density": 1000 + 50 * rng.random(shape)}
    if len(shape) == 2:
        med.update(alpha_coeff=0.75, alpha_power=1.5)
    fn = (kwhip.kspaceFirstOrder1D, kwhip.kspaceFirstOrder2D, kwhip.kspaceFirstOrder3D)[len(shape) - 1]
    return fn(kg, med, {"p0": rng.random(shape)},
              {"mask": mask, "record": record, "record_start_index": start}, PMLSize=2, Smooth=False)


def _masks(shape):
    rng = np.random.default_rng(9)
    sparse = rng.random(shape) < 0.05
    sparse.flat[0] = True
    one = np.zeros(shape, dtype=bool)
    one.flat[-1] = True
    return [sparse, rng.random(shape) < 0.6, one]


def _check(shape):
    for start in (1, 5):
        for mask in _masks(shape):
            rows = _run(shape, mask, ["p", "u"], start)
            points = _run(shape, mask, ["p", "u", "p_max"], start)
            for k in rows:
                assert rows[k].shape[1] == 15 - start
                assert np.array_equal(rows[k], points[k]), (shape, start, k)


@pytest.mark.parametrize("shape", SHAPES)
def test_row_records_emu(shape):
    from kwhip import _abi
    with _abi._backend_override("emu"):
        _check(shape)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES + [(128, 128), (64, 64, 64)])
def test_row_records_hip(shape, hip_lib):
    _check(shape)
