"""Macroscopics of a coefficient lattice without a step (vlbm_compute_macroscopics)
against those the next step saves: both rebuild the same populations from the same
coefficients, the one from global memory (in groups or one by one, by velocity set
and precision), the other through the tile exchange, and sum them in the same order
of about 100 operations. So they agree within 100 eps of the largest value."""
import numpy as np
import pytest

from helpers import base_cfg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("vel_set", ["D3Q19", "D3Q27"])
@pytest.mark.parametrize("builder", ["closedBoxBounceBack", "parallelPlatesBounceBackFreeSlip", "circularDuctInterpBounceBack"])
def test_macroscopics_of_the_next_step(builder, vel_set, precision):
    import vlbm
    for size in ((1, 1, 1), (3, 3, 2), (33, 33, 7), (65, 65, 3)):
        if "Duct" in builder and size[0] < 12:
            continue
        print(f"\n[gpu-case] macroscopics {builder} {vel_set} {precision} {size}", flush=True)
        nx, ny, nz = size
        lat = vlbm.Lattice(base_cfg(precision=precision, vel_set=vel_set, NX=nx, NY=ny, NZ=nz, tau=0.8, FX=1e-5, layout="moments",
                                    builder=builder, non_newtonian_model="BINGHAM", yield_stress=1e-5).to_desc())
        rng = np.random.default_rng(nx)
        u = 0.02 * (rng.random((3, nz, ny, nx)) - 0.5)
        lat.init(None, u[0], u[1], u[2])
        lat.step(3)
        lat.compute_macroscopics()
        a = lat.macroscopics()
        lat.step(1, save_last=True)
        b = lat.macroscopics()
        assert lat.layout == "moments"
        used = (vlbm.build_map(lat.desc) >> 21) & 1 == 1
        lat.close()
        tol = 100 * np.finfo(np.float64 if precision == "double" else np.float32).eps
        assert np.abs(a["rho"] - b["rho"])[used].max() <= tol
        scale = max(np.abs(b[k][used]).max() for k in ("ux", "uy", "uz"))
        for k in ("ux", "uy", "uz"):
            assert np.abs(a[k] - b[k])[used].max() <= tol * max(scale, 0.01), k
