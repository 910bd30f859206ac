"""Spreading of FP32 forces through LDS slabs of each sphere's box: 8 slabs, a
few, and one (many spheres), clear of each other, overlapping, at walls and
across periodic ends. The oracle is the FP64 fluid, whose forces spread point by
point through global atomics. Per stage and iteration an FP32 force carries the
rounding of about 20 operations on the velocities, so over 3 iterations and 2
steps the force fields agree within 2 * 3 * 20 eps, 1.5e-5, of their norm."""
import numpy as np
import pytest

from helpers import base_cfg, rel_l2

pytestmark = pytest.mark.gpu


def force(precision, size, centres, radius):
    import vlbm
    from vlbm import _capi
    nx, ny, nz = size
    lat = vlbm.Lattice(base_cfg(precision=precision, NX=nx, NY=ny, NZ=nz, tau=0.8, FX=1e-5,
                                builder="parallelPlatesBounceBack_Y").to_desc())
    rng = np.random.default_rng(4)
    u = 0.02 * (rng.random((3, nz, ny, nx)) - 0.5)
    lat.init(None, u[0], u[1], u[2])
    n = 150
    lat.ibm_enable(_capi.default_ibm_desc(max_iterations=3, periodic_x=1, periodic_y=0, periodic_z=1,
                                          max_spheres=len(centres), max_nodes=n * len(centres)))
    for c in centres:
        lat.ibm_add_sphere(c, vel=(0.01, 0, 0.005), radius=radius, density=2.0, mesh=_capi.MESH_FIBONACCI, n_fibonacci=n)
    lat.step(2)
    lat.ibm_status()
    f = lat.ibm_force()
    lat.close()
    return f - np.array([1e-5, 0, 0])[:, None, None, None]


def grid(n, size, pitch):
    m = [max(1, (s - 2) // pitch) for s in size]
    return [np.array([k % m[0], k // m[0] % m[1], k // (m[0] * m[1]) % m[2]]) * pitch + 4.3 for k in range(n)]


@pytest.mark.parametrize("count,size,pitch", [(1, (24, 24, 24), 9), (2, (20, 20, 20), 6), (40, (60, 50, 40), 10), (150, (70, 60, 60), 10)])
def test_force_field(count, size, pitch):
    print(f"\n[gpu-case] slabs: {count} spheres in {size}", flush=True)
    centres = grid(count, size, pitch)
    a, b = force("single", size, centres, 3.0), force("double", size, centres, 3.0)
    assert np.linalg.norm(b) > 0
    assert rel_l2(a, b) <= 1.5e-5
