"""Time series of p and u of axisymmetric simulations: the records that the x
passes write against the point kernel's (the same points with p_max asked for
as well), bit for bit.  A nonlinear step rewrites the mirrored copies of the
expanded grid after its x passes, and a kw_problem may name points there."""

import numpy as np
import pytest

import as_cases as ac
import cases


def _record(lib, name, record, copy):
    import kwhip
    from kwhip import _abi, solver
    cs = ac.case(name, Nt=14)
    kg = kwhip.kWaveGrid(cs["Nx"], cs["dx"], cs["Ny"], cs["dx"])
    kg.setTime(cs["Nt"], cs["dt"])
    opts = solver._parse_options((), dict(PMLSize=cs["pml"], Smooth=cs["smooth"]))
    pp = solver._prepare_as(kg, dict(cs["medium"]), dict(cs["source"]),
                            {"mask": cs["sensor"]["mask"], "record": record}, opts)
    at = np.ctypeslib.as_array(pp.prob.sensor_mask_index, (int(pp.prob.sensor_num_points),))
    pp.prob.sensor_mask_index = _abi.uptr(pp.hold(at + np.uint64(copy * cs["Nx"] * cs["Ny"])))
    return cases.run_entry(lib, "kw_run", pp)


def _check(lib, name, copy):
    rows = _record(lib, name, ["p", "u"], copy)
    points = _record(lib, name, ["p", "u", "p_max"], copy)
    for k in rows:
        assert np.max(np.abs(points[k])) > 0
        assert np.array_equal(rows[k], points[k]), (name, copy, k)


CASES = [(n, c) for n in ("homogeneous", "nonlinear", "source_stokes_nonlinear") for c in (0, 1, 3)]


@pytest.mark.parametrize("name,copy", CASES)
def test_as_row_records_emu(name, copy):
    from kwhip import _abi
    with _abi._backend_override("emu"):
        _check(_abi.load("emu"), name, copy)


@pytest.mark.gpu
@pytest.mark.parametrize("name,copy", CASES)
def test_as_row_records_hip(name, copy, hip_lib):
    _check(hip_lib, name, copy)
