"""Operators and medium maps built on the device (grids of 2^16 cells and
more) against the host's: kw_run builds them on the device, kw_run_noalloc,
which may not allocate a chunk, on the host.  Both evaluate in double
precision and round once, so an entry differs at most in its last single
bit, and a few steps at most to 1e-6 of the largest value.  The staggered
column-major layout of a density map is checked against NumPy bit for bit."""

import itertools

import numpy as np
import pytest

import cases

KINDS = ["power", "no_dispersion", "no_absorption", "stokes", "alpha_map", "lossless_ragged"]


def _case(kind, shape):
    rng = np.random.default_rng(len(kind))
    med = {"sound_speed": 1500 + 50 * rng.random(shape), "density": 1000 + 50 * rng.random(shape)}
    if kind != "lossless_ragged":
        med.update(alpha_coeff=0.75, alpha_power=1.5, BonA=6 + rng.random(shape))
    if kind in ("no_dispersion", "no_absorption", "stokes"):
        med["alpha_mode"] = kind
    if kind == "alpha_map":
        med["alpha_coeff"] = 0.5 + rng.random(shape)
    src = np.zeros(shape)
    src[tuple(n // 2 for n in shape)] = 1
    return {"dim": len(shape), "shape": shape, "dx": 1e-4, "Nt": 5, "dt": 1.5e-8, "medium": med,
            "source": {"p_mask": src, "p": np.array([[1.0, -2.0, 1.5, 0.5, -1.0]]), "p_mode": "additive"},
            "sensor": {"mask": np.ones(shape), "record": ["p_final", "p_max", "u_final"]},
            "opts": {"PMLSize": 6, "Smooth": False}}


def _check(lib, kind):
    shape = (49, 37, 41) if kind == "lossless_ragged" else (256, 300)
    pp = cases.prepared(_case(kind, shape))
    dev = cases.run_entry(lib, "kw_run", pp)
    host = cases.run_entry(lib, "kw_run_noalloc", pp)
    for k in host:
        g, w = np.asarray(dev[k], dtype=np.float64), np.asarray(host[k], dtype=np.float64)
        assert np.max(np.abs(w)) > 0 and np.max(np.abs(g - w)) <= 1e-6 * np.max(np.abs(w)), (kind, k)


@pytest.mark.parametrize("kind", KINDS)
def test_device_setup_emu(kind):
    from kwhip import _abi
    with _abi._backend_override("emu"):
        _check(_abi.load("emu"), kind)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", KINDS)
def test_device_setup_hip(kind, hip_lib):
    _check(hip_lib, kind)


@pytest.mark.parametrize("order", ["C", "F"])
@pytest.mark.parametrize("shape", [(70001,), (300, 257), (67, 33, 41), (5, 4, 3)])
def test_layout(shape, order):
    from kwhip import _abi
    a = np.asarray(np.random.default_rng(1).random(shape), order=order)
    with _abi._backend_override("emu"):
        flat, sg = _abi.fortran_staggered(a)
        assert np.array_equal(_abi.fortran_flat(a), a.ravel(order="F"))
    assert np.array_equal(flat, a.ravel(order="F"))
    for ax in range(a.ndim):
        m = np.moveaxis(a, ax, 0)
        want = m.copy()
        want[:-1] = m[:-1] + 0.5 * (m[1:] - m[:-1])
        assert np.array_equal(sg[ax], np.moveaxis(want, 0, ax).ravel(order="F"))


def _views(shape):
    """Grids in the orders that a program's arrays come in, other than C and F."""
    rng = np.random.default_rng(2)
    n = len(shape)
    wide = rng.random(tuple(k + 5 for k in shape))
    yield "slice", wide[tuple(slice(2, k + 2) for k in shape)]
    yield "slice_f", np.asfortranarray(wide)[tuple(slice(2, k + 2) for k in shape)]
    yield "step", rng.random(shape[:-1] + (2 * shape[-1],))[..., ::2]
    yield "reversed", rng.random(shape)[tuple(slice(None, None, -1) for _ in shape)]
    yield "one_plane", np.broadcast_to(rng.random(shape[:-1] + (1,)), shape)
    for p in itertools.permutations(range(n)):
        if list(p) not in (list(range(n)), list(range(n))[::-1]):
            yield f"axes{p}", rng.random([shape[i] for i in p]).transpose(np.argsort(p))
    yield "single", rng.random(shape).astype(np.float32)[:, ::-1]
    raw = np.zeros(8 * int(np.prod(shape)) + 1, dtype=np.uint8)[1:].view(np.float64).reshape(shape)
    raw[...] = rng.random(shape)
    yield "unaligned", raw


@pytest.mark.parametrize("shape", [(300, 257), (67, 33, 41), (33, 1, 2000), (1, 70, 1000)])
def test_layout_of_views(shape, monkeypatch):
    """Large grids in any order take the threaded transpose and give NumPy's
    column-major flattening and the same staggered copies."""
    from kwhip import _abi
    calls = []
    inner = _abi._layout
    monkeypatch.setattr(_abi, "_layout", lambda *a: (calls.append(1), inner(*a))[1])
    for name, a in _views(shape):
        calls.clear()
        with _abi._backend_override("emu"):
            got = _abi.fortran_flat(a)
            assert calls or a.flags.f_contiguous, name
            flat, sg = _abi.fortran_staggered(a)
        assert np.array_equal(got, a.ravel(order="F")), name
        assert np.array_equal(flat, a.ravel(order="F")), name
        d = a.astype(np.float64)
        for ax in range(a.ndim):
            m = np.moveaxis(d, ax, 0)
            want = m.copy()
            want[:-1] = m[:-1] + 0.5 * (m[1:] - m[:-1])
            assert np.array_equal(sg[ax], np.moveaxis(want, 0, ax).ravel(order="F")), (name, ax)


def test_flattening_takes_more_axes():
    from kwhip import _abi
    a = np.random.default_rng(3).random((300, 257, 1, 1))
    with _abi._backend_override("emu"):
        assert np.array_equal(_abi.fortran_flat(a), a.ravel(order="F"))
