"""Field downloads around their chunk and thread limits: less than a chunk,
several chunks with a remainder on one thread, and enough for several threads,
from one caller and from several at once. The saved macroscopics of a fresh
lattice are its initial fields rounded to the compute type, so the values are
known exactly."""
import threading

import numpy as np
import pytest

from helpers import base_cfg

pytestmark = pytest.mark.gpu


def make(size, precision):
    import vlbm
    nx, ny, nz = size
    lat = vlbm.Lattice(base_cfg(NX=nx, NY=ny, NZ=nz, precision=precision, builder="taylorGreenVortex").to_desc())
    rng = np.random.default_rng(nx)
    want = dict(zip(("rho", "ux", "uy", "uz"), rng.random((4, nz, ny, nx))))
    lat.init(*want.values())
    if precision == "single":
        want = {k: v.astype(np.float32).astype(np.float64) for k, v in want.items()}
    return lat, want


@pytest.mark.parametrize("size,precision", [((7, 5, 3), "double"), ((131, 101, 13), "single"), ((97, 71, 33), "double"),
                                            ((333, 211, 17), "single"), ((211, 111, 31), "double")])
def test_values(size, precision):
    print(f"\n[gpu-case] download {size} {precision}", flush=True)
    lat, want = make(size, precision)
    for _ in range(2):
        got = lat.macroscopics()
        for k in want:
            assert np.array_equal(got[k], want[k]), k
    lat.close()


def test_callers_at_once():
    print("\n[gpu-case] downloads from four threads, two lattices", flush=True)
    made = [make((333, 211, 17), "single"), make((131, 101, 13), "double")]
    same = []

    def download(lat, want):
        got = lat.macroscopics()
        same.append(all(np.array_equal(got[k], want[k]) for k in want))

    threads = [threading.Thread(target=download, args=made[i % 2]) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert same == [True] * 4
    for lat, _ in made:
        lat.close()
