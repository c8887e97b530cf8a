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


# a source, a medium and a record that each take another way through the
# passes that write the rows
FORMS = [("p additive", "lossless", ["p", "u"]), ("p dirichlet", "stokes", ["p", "u"]),
         ("p additive-no-correction", "absorbing", ["p"]), ("p each additive", "nonlinear", ["p", "u"]),
         ("u additive", "stokes", ["u"]), ("u dirichlet", "absorbing", ["p", "u"]),
         ("u additive-no-correction", "nonlinear", ["u"]), ("u each additive", "lossless", ["p", "u"])]


def _inputs(shape, source, medium):
    import kwhip
    rng = np.random.default_rng(11)
    kg = kwhip.kWaveGrid(*sum(([n, 1e-4] for n in shape), []))
    kg.setTime(12, 1.5e-8)
    med = {"sound_speed": 1500 + 50 * rng.random(shape), "density": 1000 + 50 * rng.random(shape)}
    if medium == "stokes":
        med.update(alpha_coeff=0.75, alpha_power=2.0, alpha_mode="stokes")
    elif medium != "lossless":
        med.update(alpha_coeff=0.75, alpha_power=1.5)
    if medium == "nonlinear":
        med["BonA"] = 6.0
    at = rng.random(shape) < 0.1
    field, *each, mode = source.split(" ")
    # eight steps of source, four without
    sig = rng.standard_normal((int(at.sum()) if each else 1, 8))
    src = {"p_mask": at, "p": sig, "p_mode": mode} if field == "p" else \
        {"u_mask": at, "ux": 1e-6 * sig, "u_mode": mode}
    return kg, med, src, rng.random(shape) < 0.3


def _forms(shape, source, medium, record):
    import kwhip
    kg, med, src, mask = _inputs(shape, source, medium)
    fn = (kwhip.kspaceFirstOrder2D, kwhip.kspaceFirstOrder3D)[len(shape) - 2]
    rows, points = (fn(kg, med, src, {"mask": mask, "record": r}, PMLSize=2, Smooth=False)
                    for r in (record, record + [record[0] + "_max"]))
    for k in rows:
        assert np.max(np.abs(points[k])) > 0
        assert np.array_equal(rows[k], points[k]), (shape, source, medium, k)


def _group(shapes):
    """Members of one engine group, of uneven sizes."""
    import kwhip
    got = []
    for more in ([], ["p_max"]):
        with kwhip.Engine() as eng:
            tickets = []
            for shape in shapes:
                kg, med, src, mask = _inputs(shape, "p dirichlet", "lossless")
                tickets.append(eng.submit(kg, med, src, {"mask": mask, "record": ["p", "u"] + more},
                                          len(shape), PMLSize=2, Smooth=False))
            got.append([eng.wait(t) for t in tickets])
    for shape, rows, points in zip(shapes, *got):
        for k in rows:
            assert np.max(np.abs(points[k])) > 0
            assert np.array_equal(rows[k], points[k]), (shape, k)


# 81 points along x in 3-D: p keeps the point kernel there
@pytest.mark.parametrize("source,medium,record", FORMS)
@pytest.mark.parametrize("shape", [(24, 15), (10, 9, 8), (81, 4, 5)])
def test_row_record_forms_emu(shape, source, medium, record):
    from kwhip import _abi
    with _abi._backend_override("emu"):
        _forms(shape, source, medium, record)


@pytest.mark.gpu
@pytest.mark.parametrize("source,medium,record", FORMS)
@pytest.mark.parametrize("shape", [(24, 15), (128, 100), (16, 10, 9), (81, 32, 20), (64, 64, 64)])
def test_row_record_forms_hip(shape, source, medium, record, hip_lib):
    _forms(shape, source, medium, record)


def test_row_records_group_emu():
    from kwhip import _abi
    with _abi._backend_override("emu"):
        _group([(24, 15), (18, 22), (40,)])


@pytest.mark.gpu
@pytest.mark.parametrize("shapes", [[(24, 15), (130, 64), (77, 91), (40,)], [(128, 128)] * 3,
                                    [(16, 10, 9), (64, 22, 30), (31, 12, 40)]])
def test_row_records_group_hip(shapes, hip_lib):
    _group(shapes)
