"""Births of full updates (slots handed from cells to particles) against the checker, and against the stage-by-stage
path (slots searched in the particle-order ends) where masses are out of range."""
import numpy as np
import pytest

from dogm_ctypes import DOGM, MEAS_CELL_DTYPE
from oracle_ctypes import OracleDOGM
from parity_util import assert_grid_equal, assert_particles_equal, small_params

pytestmark = pytest.mark.gpu

SEED = 31


def _grid(gs, kind, rng):
    m = np.zeros(gs * gs, MEAS_CELL_DTYPE)
    m["likelihood"] = 1.0
    m["p_A"] = rng.random(gs * gs)
    occ = m["occ_mass"]
    if kind == "one_cell":      # every slot in one cell: records of whole blocks
        occ[rng.integers(gs * gs)] = 0.7
    elif kind == "last_cell":
        occ[-1] = 0.7
    elif kind == "few":
        occ[rng.integers(0, gs * gs, 5)] = 0.6
    elif kind == "all":
        occ[:] = rng.uniform(0.01, 0.5, gs * gs)
    elif kind == "sparse":
        occ[:] = np.where(rng.random(gs * gs) < 0.02, 0.5, 0.0)
    else:
        assert kind == "none"   # no mass at all: an equal split, then unchanged empties
    return m


# B around the 64-slot blocks; grids around the 256-cell units and 1024-cell tiles.
@pytest.mark.parametrize("gs,b", [(1, 1), (3, 64), (16, 65), (17, 63), (32, 1000), (33, 128), (70, 5000)])
def test_full_births_match_checker(gs, b):
    p = small_params(gs=gs, res=0.5, n=500, b=b)
    rng = np.random.default_rng(gs + b)
    with DOGM(p, seed=SEED) as gpu:
        orc = OracleDOGM(p, seed=SEED)
        for f, kind in enumerate(["few", "one_cell", "none", "none", "sparse", "all", "one_cell", "last_cell", "few"]):
            m = _grid(gs, kind, rng)
            gpu.update_grid(m, 0.0, 0.0, 0.0, 0.1)
            orc.update_grid(m, 0.0, 0.0, 0.0, 0.1)
            assert_grid_equal(f"{kind} frame {f}", gpu.get_grid_cells(), orc.get_grid_cells())
            assert_particles_equal(f"{kind} frame {f}", gpu.get_birth_particles(), orc.get_birth_particles())
        orc.close()


@pytest.mark.parametrize("bad", [-3.0, np.nan, np.inf, 1e30])
def test_masses_out_of_range_match_stage_path(bad):
    """Free masses far outside [0, 1] make born masses negative, NaN or huge."""
    gs, b = 40, 900
    p = small_params(gs=gs, res=0.5, n=4000, b=b)
    rng = np.random.default_rng(8)
    with DOGM(p, seed=SEED) as full, DOGM(p, seed=SEED) as staged:
        for f in range(4):
            m = _grid(gs, "sparse", rng)
            if f == 2:
                m["free_mass"][:: 13] = bad
            full.update_grid(m, 0.0, 0.0, 0.0, 0.1)
            staged.update_measurement_grid(m)
            staged.update_pose(0.0, 0.0, 0.0)
            staged.particle_prediction(0.1)
            staged.particle_assignment()
            staged.grid_cell_occupancy_update(0.1)
            staged.update_persistent_particles()
            staged.initialize_new_particles()
            staged.statistical_moments()
            staged.resampling()
            a, c = full.get_grid_cells(), staged.get_grid_cells()
            for name in ("new_born_occ_mass", "w_A", "w_UA", "occ_mass"):
                np.testing.assert_array_equal(a[name].view(np.uint32), c[name].view(np.uint32), err_msg=f"{name} {f}")
            assert_particles_equal(f"frame {f}", full.get_birth_particles(), staged.get_birth_particles())
