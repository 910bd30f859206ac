"""Spreading of FP32 forces through LDS slabs: spheres with more nodes than a batch
of the kernel, slab counts that leave the last slab with fewer planes (8 slabs of
3 planes and 5 slabs of 5 planes of a box of 22), and nodes with area whose stencils
leave the box in each direction, which the first slab alone adds. The oracle is the
FP64 fluid, whose forces spread point by point through global atomics. Per stage and
iteration an FP32 force carries the rounding of about 20 operations on the
velocities, so over 3 iterations and 2 steps the force fields agree within
2 * 3 * 20 eps, 1.5e-5, of their norm."""
import numpy as np
import pytest

from helpers import base_cfg, rel_l2

pytestmark = pytest.mark.gpu


def force(precision, size, add):
    import vlbm
    from vlbm import _capi
    nx, ny, nz = size
    lat = vlbm.Lattice(base_cfg(precision=precision, NX=nx, NY=ny, NZ=nz, tau=0.8, FX=1e-5,
                                builder="parallelPlatesBounceBack_Y").to_desc())
    rng = np.random.default_rng(4)
    u = 0.02 * (rng.random((3, nz, ny, nx)) - 0.5)
    lat.init(None, u[0], u[1], u[2])
    lat.ibm_enable(_capi.default_ibm_desc(max_iterations=3, periodic_x=1, periodic_y=0, periodic_z=1, max_spheres=64,
                                          max_nodes=64 * 804))
    add(lat, _capi)
    lat.step(2)
    lat.ibm_status()
    f = lat.ibm_force()
    lat.close()
    return f - np.array([1e-5, 0, 0])[:, None, None, None]


def agree(size, add):
    a, b = force("single", size, add), force("double", size, add)
    assert np.linalg.norm(b) > 0
    assert rel_l2(a, b) <= 1.5e-5


@pytest.mark.parametrize("count,size", [(1, (30, 30, 30)), (48, (86, 86, 66))])
def test_many_nodes_and_a_short_last_slab(count, size):
    print(f"\n[gpu-case] spreading of {count} spheres of radius 8", flush=True)
    centres = [np.array([k % 4, k // 4 % 4, k // 16]) * 21.0 + 12.3 for k in range(count)]

    def add(lat, capi):
        for c in centres:
            lat.ibm_add_sphere(c, vel=(0.01, 0, 0.005), radius=8.0, density=2.0, mesh=capi.MESH_FIBONACCI, n_fibonacci=804)

    agree(size, add)


@pytest.mark.parametrize("count", [1, 4])
def test_nodes_outside_the_box(count):
    """Radius 3: the box spans 5 nodes below and 6 above the centre's node. The added
    nodes reach across its faces (5.4 and 6.2 away) and lie outside (9)."""
    print(f"\n[gpu-case] spreading of {count} spheres with nodes outside their box", flush=True)
    rng = np.random.default_rng(1)
    d = rng.normal(size=(60, 3))
    surface = 3.0 * d / np.linalg.norm(d, axis=1)[:, None]
    away = []
    for axis in range(3):
        for offset in (-9.0, -6.2, -5.4, 5.4, 6.2, 9.0):
            away.append([0.3, 0.2, 0.1])
            away[-1][axis] = offset
    area = np.full(60 + len(away), 4 * np.pi * 9 / 60)

    def add(lat, capi):
        for k in range(count):
            c = np.array([12.3, 14.2, 13.4]) + 13.0 * np.array([k % 2, 0, k // 2])
            lat.ibm_add_particle(c, (0.01, 0, 0.005), (0, 0, 0.001), 3.0, 2.0, True, np.vstack([surface, away]) + c, area)

    agree((40, 30, 40), add)
