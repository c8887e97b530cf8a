"""kw_run_noalloc on the CPU lane emulator (no GPU): the simulation's
buffers come from the library's scratch block, the outputs equal kw_run's
bit for bit, a second, smaller call after a first one still does, and a
problem larger than the scratch block is refused with KW_ENOMEM."""

import numpy as np
import pytest

import cases


@pytest.fixture(scope="module")
def emu_lib():
    from kwhip import _abi
    return _abi.load("emu")


def test_noalloc_equals_kw_run_on_emulator(emu_lib):
    for cs in (cases.case("psrc_many", 2), cases.case("p0_lossless", 2, (24, 20))):
        pp = cases.prepared(cs)
        want = cases.run_entry(emu_lib, "kw_run", pp)
        got = cases.run_entry(emu_lib, "kw_run_noalloc", pp)
        assert set(got) == set(want)
        for k in want:
            assert np.array_equal(np.asarray(got[k]), np.asarray(want[k])), (cs["shape"], k)


def test_noalloc_refuses_oversize_on_emulator(emu_lib):
    from kwhip import _abi
    N = 192
    cs = {"dim": 3, "shape": (N, N, N), "dx": 1e-4, "Nt": 2, "dt": 2e-8,
          "medium": {"sound_speed": 1500.0, "density": 1000.0},
          "source": {"p0": np.zeros((N, N, N))},
          "sensor": {"mask": np.ones((N, N, N)), "record": ["p_final"]},
          "opts": {"PMLSize": 10, "Smooth": False}}
    pp = cases.prepared(cs)
    with pytest.raises(_abi.KWError) as ei:
        cases.run_entry(emu_lib, "kw_run_noalloc", pp)
    assert ei.value.code == _abi.KW_ENOMEM
    assert "scratch" in str(ei.value)


def test_noalloc_takes_records_up_to_the_scratch(emu_lib):
    """Sensor points in ascending order, whose records take a table of rows,
    fit the scratch block as long as the same points in another order do.
    Source series (all but the first unused) fill the block to the last few
    bytes."""
    from kwhip import _abi
    mask = np.zeros((8, 1024))
    mask[3, ::5] = 1
    cs = {"dim": 2, "shape": (8, 1024), "dx": 1e-4, "Nt": 2, "dt": 2e-8,
          "medium": {"sound_speed": 1500.0, "density": 1000.0},
          "source": {"p_mask": mask, "p": np.ones((1, 2)), "p_mode": "dirichlet"},
          "sensor": {"mask": mask, "record": ["p"]},
          "opts": {"PMLSize": 2, "Smooth": False}}
    pp = cases.prepared(cs)
    n = int(pp.prob.sensor_num_points)
    up = np.ctypeslib.as_array(pp.prob.sensor_mask_index, (n,)).copy()
    down = np.ascontiguousarray(up[::-1])
    signals, first = np.ones(34 << 20), np.ones(n, dtype=np.uint64)
    pp.prob.p_source.input = _abi.dptr(signals)
    pp.prob.p_source.sig_index = _abi.uptr(first)

    def run(series, idx):
        pp.prob.p_source.num_series = series
        pp.prob.sensor_mask_index = _abi.uptr(idx)
        try:
            return np.asarray(cases.run_entry(emu_lib, "kw_run_noalloc", pp)["p"])
        except _abi.KWError as e:
            assert e.code == _abi.KW_ENOMEM
            return None

    fits, over = 15 << 20, 17 << 20
    assert run(over, down) is None
    while over - fits > 1:
        mid = (fits + over) // 2
        if run(mid, down) is None:
            over = mid
        else:
            fits = mid
    want = run(fits, down)
    got = run(fits, up)
    assert got is not None and np.array_equal(got, want[::-1])
