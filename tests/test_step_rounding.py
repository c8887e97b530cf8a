"""kappa takes up what single precision loses of the time step and of a
uniform sound speed and density.  A simulation changed to a time step while
its fields are still zero runs on as one created with that step does: the same
records bit for bit."""

import ctypes as C

import numpy as np
import pytest


def _record(shape, density, dt_first, dt, quiet=4, steps=12):
    import kwhip
    from kwhip import _abi
    rng = np.random.default_rng(5)
    kg = kwhip.kWaveGrid(*sum(([n, 1e-4] for n in shape), []))
    kg.setTime(steps, dt_first)
    src = rng.random(shape) < 0.1
    p = np.zeros((1, steps))
    p[0, quiet:] = rng.standard_normal(steps - quiet)
    sim = kwhip.Simulation(kg, {"sound_speed": 1500.00011, "density": density},
                           {"p_mask": src, "p": p, "p_mode": "dirichlet"},
                           {"mask": np.ones(shape), "record": ["p", "u"]}, len(shape), PMLSize=3,
                           Smooth=False)
    if dt_first != dt:
        sim.step(2)
        _abi.call(sim.lib.kw_sim_change_dt, sim.h, C.c_double(dt_first), C.c_double(dt))
    sim.step(steps - sim.steps_done)
    out = {k: np.array(v) for k, v in sim.read().items()}
    sim.close()
    return out


def _check(shape, uniform):
    density = 1000.3 if uniform else 1000 + 50 * np.random.default_rng(6).random(shape)
    for dt in (1.7e-8, 1.8000000001e-8, 2.3e-8):
        created = _record(shape, density, dt, dt)
        changed = _record(shape, density, 1.9e-8, dt)
        for k in created:
            assert np.max(np.abs(created[k])) > 0
            assert np.array_equal(created[k], changed[k]), (shape, uniform, dt, k)


@pytest.mark.parametrize("uniform", [True, False])
@pytest.mark.parametrize("shape", [(40,), (24, 15)])
def test_changed_step_emu(shape, uniform):
    from kwhip import _abi
    with _abi._backend_override("emu"):
        _check(shape, uniform)


@pytest.mark.gpu
@pytest.mark.parametrize("uniform", [True, False])
@pytest.mark.parametrize("shape", [(40,), (64, 45), (20, 18, 15)])
def test_changed_step_hip(shape, uniform, hip_lib):
    _check(shape, uniform)
