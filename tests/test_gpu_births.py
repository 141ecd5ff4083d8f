"""Births of full updates (slots handed from cells to particles) against the checker, and against the stage-by-stage
path (slots searched in the particle-order ends) where masses are out of range."""
import numpy as np
import pytest

from dogm_ctypes import DOGM, MEAS_CELL_DTYPE, Batch
from oracle_ctypes import OracleDOGM
from parity_util import assert_grid_equal, assert_int_equal, assert_particles_equal, assert_vehicle_equal, small_params

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


WIDE_UNITS = 4096  # cell units per launch above which a wave takes a unit, four cells per lane


@pytest.mark.parametrize("bad", [None, -3.0, np.nan, 1e30])
def test_wide_form_matches_narrow(bad):
    """Launches of many cells (a wave per unit) against plain handles of the same vehicles (a workgroup per unit), on
    sides that leave 1 to 4 cells of a lane, of a mark's 64 and of the last unit, with many slots in one cell, no mass
    and masses out of range.  Every other step holds the small vehicles alone, in the narrow form: each form reads the
    marks that the other left."""
    sizes = [(1, 1), (3, 64), (16, 65), (17, 63), (32, 1000), (33, 128), (46, 2049), (61, 700), (70, 5000)]
    ps = [small_params(gs=gs, res=0.5, n=400 + gs, b=b) for gs, b in sizes]
    filler = small_params(gs=90, res=0.5, n=64, b=16)  # 31.6 units
    rng = np.random.default_rng(77)
    with Batch() as batch:
        batch.set_lanes(1)  # one launch for all vehicles
        ids = [batch.add_vehicle(p, SEED, k) for k, p in enumerate(ps)]
        rest = [batch.add_vehicle(filler, SEED, 100 + k) for k in range(130)]
        assert len(rest) * 32 > WIDE_UNITS
        assert sum(-(-gs * gs // 256) for gs, _ in sizes) < WIDE_UNITS // 4
        plain = [DOGM(p, seed=SEED, instance=k) for k, p in enumerate(ps)]
        empty = _grid(90, "few", rng)
        kinds = ["few", "one_cell", "one_cell", "none", "sparse", "sparse", "all", "few", "one_cell", "last_cell", "none"]
        for f, kind in enumerate(kinds):
            ms = [_grid(gs, kind, rng) for gs, _ in sizes]
            if bad is not None and f in (4, 7):
                for m in ms:
                    m["free_mass"][:: 13] = bad
            use = ids + (rest if f % 2 == 0 else [])
            batch.update(use, ms + [empty] * (len(use) - len(ids)), [(0.0, 0.0, 0.0)] * len(use), 0.1)
            for k, g in enumerate(plain):
                tag = f"{kind} frame {f} side {sizes[k][0]}"
                g.update_grid(ms[k], 0.0, 0.0, 0.0, 0.1)
                assert_grid_equal(tag, batch.get_grid_cells(ids[k]), g.get_grid_cells())
                assert_int_equal(tag, batch.get_resampled_indices(ids[k]), g.get_resampled_indices())
        for k, g in enumerate(plain):
            assert_vehicle_equal(f"side {sizes[k][0]}", batch.get_particles(ids[k]), g.get_particles(),
                                 batch.get_grid_cells(ids[k]), g.get_grid_cells())
            g.close()


def test_one_grid_in_the_wide_form():
    """One grid of more than 4096 units whose last unit is one cell, against the checker."""
    gs, b = 1025, 30_000
    assert -(-gs * gs // 256) > WIDE_UNITS and gs * gs % 256 == 1
    p = small_params(gs=gs, res=0.5, n=2000, b=b)
    rng = np.random.default_rng(5)
    with DOGM(p, seed=SEED) as gpu:
        orc = OracleDOGM(p, seed=SEED)
        for f, kind in enumerate(["sparse", "last_cell", "none", "few"]):
            m = _grid(gs, kind, rng)
            gpu.update_grid(m, 0.0, 0.0, 0.0, 0.1)
            orc.update_grid(m, 0.0, 0.0, 0.0, 0.1)
            assert_grid_equal(f"{kind} frame {f}", gpu.get_grid_cells(), orc.get_grid_cells())
            assert_particles_equal(f"{kind} frame {f}", gpu.get_birth_particles(), orc.get_birth_particles())
        orc.close()
