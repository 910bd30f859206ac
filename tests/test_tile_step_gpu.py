"""The coefficient layout's tile step at the sizes where it can go wrong: one
node, ragged tiles in x and y, one wave more or less than a tile row, z chunks of
one and two planes, every boundary scheme it applies, both velocity sets and
precisions, with and without the immersed boundary force.

The oracle is the population layout, one thread per node, on the same initial
state. Both evaluate the same step; they differ in the order of about 100
rounded operations a step, each on values of the size of the fields, so after n
steps the fields agree within 100 n eps of their largest value."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
STEPS = 4

BOX = {
    "periodic": dict(builder="taylorGreenVortex"),
    "duct": dict(builder="squareDuctBounceBack"),
    "closed": dict(builder="closedBoxBounceBack"),
    "zouhe": dict(builder="squareDuctZouHe", uz_bc=[0, 0.01, 0, 0, 0, 0, 0, 0]),
    "lid": dict(builder="lidDrivenBounceBack"),
    "free_slip": dict(builder="parallelPlatesBounceBackFreeSlip"),
}
RHEOLOGY = {
    "newtonian": dict(non_newtonian_model=None),
    "bingham": dict(non_newtonian_model="BINGHAM", yield_stress=1e-5),
    "power_law": dict(non_newtonian_model="POWERLAW", n_index=0.6, k_consistency=0.05, tau_clamp=[0.51, 2.0]),
}


def run(layout, size, precision, vel_set, ibm, steps, **kw):
    import vlbm
    from vlbm import _capi
    from vlbm.config import SimConfig
    nx, ny, nz = size
    cfg = SimConfig(precision=precision, NX=nx, NY=ny, NZ=nz, tau=0.8, vel_set=vel_set, use_ibm=False, sim_id=0,
                    path_save="x", steps=1, macr_save=0, data_report=0, FX=1e-5, FZ=2e-5, layout=layout, **kw)
    lat = vlbm.Lattice(cfg.to_desc())
    rng = np.random.default_rng(nx + 7 * ny + 31 * nz)
    u = 0.02 * (rng.random((3, nz, ny, nx)) - 0.5)
    lat.init(1 + 0.01 * (rng.random((nz, ny, nx)) - 0.5), u[0], u[1], u[2])
    if ibm:
        lat.ibm_enable(_capi.default_ibm_desc(max_iterations=2, periodic_x=0, periodic_y=0, periodic_z=1))
        lat.ibm_add_sphere([nx / 2, ny / 2, nz / 2], vel=(0, 0, 0.01), radius=2.0, density=2.0)
    lat.step(steps, save_last=True)
    m = lat.macroscopics()
    assert lat.layout == layout
    used = (vlbm.build_map(lat.desc) >> 21) & 1 == 1
    lat.close()
    return m, used


def compare(size, precision, vel_set="D3Q19", ibm=False, steps=STEPS, **kw):
    print(f"\n[gpu-case] tile step {size} {precision} {vel_set} ibm={ibm} {kw}", flush=True)
    a, used = run("populations", size, precision, vel_set, ibm, steps, **kw)
    b, _ = run("moments", size, precision, vel_set, ibm, steps, **kw)
    tol = 100 * steps * np.finfo(np.float64 if precision == "double" else np.float32).eps
    u = max(np.abs(a[k][used]).max() for k in ("ux", "uy", "uz"))
    assert np.isfinite(u)
    scale = max(u, np.abs(a["rho"][used] - 1).max())
    for k in a:
        assert np.abs(a[k] - b[k])[used].max() <= tol * scale, k


@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("size", [(1, 1, 1), (3, 2, 2), (63, 7, 3), (64, 8, 1), (65, 9, 2), (130, 12, 5), (64, 16, 70)])
def test_sizes(size, precision):
    compare(size, precision, **BOX["periodic"], **RHEOLOGY["bingham"])
    compare(size, precision, **BOX["duct"], **RHEOLOGY["newtonian"])


@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("rheology", list(RHEOLOGY))
@pytest.mark.parametrize("name", list(BOX))
def test_boundary_schemes(name, rheology, precision):
    for vel_set in ("D3Q19", "D3Q27"):
        if vel_set == "D3Q27" and name in ("zouhe", "lid"):
            continue
        compare((70, 18, 9), precision, vel_set, **BOX[name], **RHEOLOGY[rheology])


@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("builder", ["circularDuctInterpBounceBack", "annularDuctInterpBounceBack"])
@pytest.mark.parametrize("vel_set", ["D3Q19", "D3Q27"])
def test_node_maps(vel_set, builder, precision):
    for rheology in RHEOLOGY.values():
        for n in (24, 33, 70):
            compare((n, n, 9), precision, vel_set, builder=builder, **rheology)
            compare((n, n, 9), precision, vel_set, builder=builder, outer_rotation=1e-3, inner_rotation=5e-4, **rheology)


@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("vel_set", ["D3Q19", "D3Q27"])
@pytest.mark.parametrize("builder", ["closedBoxBounceBack", "circularDuctInterpBounceBack"])
def test_immersed_boundary_force(builder, vel_set, precision):
    for rheology in RHEOLOGY.values():
        compare((24, 24, 20), precision, vel_set, ibm=True, builder=builder, **rheology)


@pytest.mark.parametrize("size,precision", [((70, 66, 60), "single"), ((66, 50, 50), "double")])
def test_population_step_through_the_caches(size, precision):
    """Lattices from 40 MB (two of 19 planes) on store through the caches and run every other step from the last
    block to the first; the block counts here are no multiples of 8, so some blocks stay where they are."""
    compare(size, precision, **BOX["duct"], **RHEOLOGY["bingham"])
    compare(size, precision, ibm=True, **BOX["closed"], **RHEOLOGY["newtonian"])
