"""Field downloads above the size from which several threads share the chunks, with
a remainder in every field's last chunk: after an idle stream, behind steps that are
still queued, and from several callers at once. A field fetched alone takes the path
of one thread, so the two paths check each other; a fresh lattice's saved
macroscopics are its initial fields rounded to the compute type."""
import threading

import numpy as np
import pytest

from helpers import base_cfg

pytestmark = pytest.mark.gpu
KEYS = ("rho", "ux", "uy", "uz")
LARGE = [((211, 203, 201), "single"), ((173, 163, 151), "double")]          # 138 and 136 MB in four fields


def make(size, precision):
    import vlbm
    nx, ny, nz = size
    lat = vlbm.Lattice(base_cfg(NX=nx, NY=ny, NZ=nz, precision=precision, builder="taylorGreenVortex").to_desc())
    rng = np.random.default_rng(nx)
    want = {k: 0.01 * rng.random((nz, ny, nx)) + (k == "rho") for k in KEYS}
    lat.init(*want.values())
    if precision == "single":
        want = {k: v.astype(np.float32).astype(np.float64) for k, v in want.items()}
    return lat, want


def one_field(lat, k):
    """Field k alone, into memory that held something else."""
    from vlbm._capi import check, lib
    import ctypes as C
    out = np.full(lat.shape, np.nan)
    p = out.ctypes.data_as(C.POINTER(C.c_double))
    check(lib.vlbm_macroscopics(lat._h, *[p if k == n else None for n in KEYS], None))
    return out


@pytest.mark.parametrize("size,precision", LARGE)
def test_values(size, precision):
    print(f"\n[gpu-case] threaded download {size} {precision}", flush=True)
    lat, want = make(size, precision)
    got = lat.macroscopics()
    for k in KEYS:
        assert np.array_equal(got[k], want[k]), k
    lat.step(12, save_last=True)
    busy = lat.macroscopics()
    idle = lat.macroscopics()
    for k in KEYS:
        assert np.array_equal(busy[k], idle[k]), k
        assert np.array_equal(busy[k], one_field(lat, k)), k
    assert not np.array_equal(busy["ux"], want["ux"])
    lat.close()


def test_callers_at_once():
    print("\n[gpu-case] threaded downloads from four callers, two lattices", flush=True)
    made = [make(*c) for c in LARGE]
    same = []

    def download(lat, want):
        got = lat.macroscopics()
        same.append(all(np.array_equal(got[k], want[k]) for k in KEYS))

    threads = [threading.Thread(target=download, args=made[i % 2]) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert same == [True] * 4
    for lat, _ in made:
        lat.close()


def test_fields_of_a_refused_call():
    """A Newtonian fluid has no omega: the call fails, with the other fields in place."""
    import ctypes as C
    from vlbm._capi import lib
    lat, want = make((9, 8, 7), "double")
    out = {k: np.full(lat.shape, np.nan) for k in KEYS + ("omega",)}
    rc = lib.vlbm_macroscopics(lat._h, *[out[k].ctypes.data_as(C.POINTER(C.c_double)) for k in KEYS + ("omega",)])
    assert rc != 0 and np.isnan(out["omega"]).all()
    for k in KEYS:
        assert np.array_equal(out[k], want[k]), k
    lat.close()
