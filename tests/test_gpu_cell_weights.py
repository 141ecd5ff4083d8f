"""Full updates from uniform weights (per-cell weights) against the checker and against the general path, which a
vehicle takes once its weights have been written, bit for bit."""
import numpy as np
import pytest

from dogm_ctypes import DOGM, Batch, MEAS_CELL_DTYPE
from oracle_ctypes import OracleDOGM
from parity_util import assert_grid_equal, assert_state_equal, assert_vehicle_equal, small_params

pytestmark = pytest.mark.gpu

SEED = 91


def _grid(gs, rng, special=False):
    """Random masses, likelihoods and association probabilities on every cell."""
    m = np.zeros(gs * gs, MEAS_CELL_DTYPE)
    m["free_mass"] = rng.uniform(0.0, 0.5, gs * gs)
    m["occ_mass"] = np.where(rng.random(gs * gs) < 0.3, rng.uniform(0.0, 0.5, gs * gs), 0.0)
    m["likelihood"] = rng.uniform(0.1, 3.0, gs * gs)
    m["p_A"] = rng.random(gs * gs)
    if special:
        m["likelihood"][:: 3] = 0.0
        m["likelihood"][1:: 7] = np.float32(1e-38)
        m["likelihood"][2:: 11] = -0.5
        m["p_A"][:: 5] = 0.0
    return m


# Jumps of several grid sides clamp every particle to border cells; small grids are all border.
@pytest.mark.parametrize("gs,n,b", [(1, 5, 2), (2, 255, 0), (4, 1023, 10), (5, 1024, 64), (17, 1025, 100),
                                    (33, 7000, 700), (64, 40000, 4000)])
@pytest.mark.parametrize("ego", ["reference", "metric"])
def test_full_updates_match_checker(gs, n, b, ego):
    p = small_params(gs=gs, res=0.5, n=n, b=b)
    rng = np.random.default_rng(gs * n)
    poses = [(0.0, 0.0, 0.0), (0.6, -0.7, 0.1), (0.7, 4.0 * gs, 0.2), (1.5, 4.0 * gs, 0.3), (1.5, 4.0 * gs, 0.3)]
    with DOGM(p, seed=SEED, instance=3) as gpu:
        orc = OracleDOGM(p, seed=SEED, instance=3)
        gpu.set_ego_mode(ego)
        orc.set_ego_mode(ego)
        for f, pose in enumerate(poses):
            m = _grid(gs, rng, special=f == 3)
            gpu.update_grid(m, *pose, 0.1)
            orc.update_grid(m, *pose, 0.1)
            # read particles only at the end: the frames before read the resampled sets through the ancestors
            assert_state_equal(f"{ego} {gs} frame {f}", gpu, orc, ancestors=True, particles=f == len(poses) - 1)
        orc.close()


@pytest.mark.parametrize("special", [None, np.inf, np.nan])
def test_matches_general_path(special):
    """Two handles in the same state, one with its (unchanged) weights written back: the general path."""
    gs, n, b = 40, 30000, 3000
    p = small_params(gs=gs, res=0.5, n=n, b=b)
    rng = np.random.default_rng(12)
    with DOGM(p, seed=SEED) as cells, DOGM(p, seed=SEED) as general:
        for f in range(4):
            m = _grid(gs, rng)
            if special is not None and f == 2:
                m["likelihood"][:: 9] = special
            pose = (0.9 * f, 30.0 if f == 3 else 0.0, 0.0)
            if f:
                general.set_particles(weight=general.get_particles()["weight"])
            for g in (cells, general):
                g.update_grid(m, *pose, 0.1)
            assert_vehicle_equal(f"frame {f}", cells.get_particles(), general.get_particles(),
                                 cells.get_grid_cells(), general.get_grid_cells())
            a, c = cells.get_weight_array().view(np.uint32), general.get_weight_array().view(np.uint32)
            np.testing.assert_array_equal(a, c)
            np.testing.assert_array_equal(cells.get_resampled_indices(), general.get_resampled_indices())


def test_stage_calls_after_full_updates():
    """The stage methods find what they read (masked cell indices, weights) after updates that left per-cell weights."""
    p = small_params(gs=48, res=0.5, n=9000, b=900)
    rng = np.random.default_rng(3)
    with DOGM(p, seed=SEED) as gpu:
        orc = OracleDOGM(p, seed=SEED)
        for f in range(4):
            m = _grid(48, rng)
            pose = (1.1 * f, -20.0 if f == 1 else 0.0, 0.0)
            for o in (gpu, orc):
                if f % 2 == 0:
                    o.update_grid(m, *pose, 0.1)
                    continue
                o.update_measurement_grid(m)
                o.update_pose(*pose)
                o.particle_prediction(0.1)
                o.particle_assignment()
                o.grid_cell_occupancy_update(0.1)
                o.update_persistent_particles()
                o.initialize_new_particles()
                o.statistical_moments()
                o.resampling()
            assert_state_equal(f"frame {f}", gpu, orc, ancestors=True, particles=f == 3)
        orc.close()


@pytest.mark.parametrize("gs,n", [(1, 63), (5, 257), (33, 1000), (64, 700)])
def test_single_stages_after_full_updates(gs, n):
    """An occupancy update on its own, straight after full updates, reads the sums that both paths leave per cell: the
    cells the resampling emptied have no particles to sum.  Without births the resampled sets stay sorted, and in one
    reduction tile no cell's particles are cut, so what the stage sums does not depend on the bounds of the last sort."""
    p = small_params(gs=gs, res=0.5, n=n, b=0)
    rng = np.random.default_rng(gs)
    with DOGM(p, seed=SEED) as cells, DOGM(p, seed=SEED) as general:
        for f in range(5):
            m = _grid(gs, rng)
            m["likelihood"] = rng.choice([0.05, 5.0], gs * gs)  # cells lose all their particles
            if f:
                general.set_particles(weight=general.get_particles()["weight"])
            for g in (cells, general):
                g.update_grid(m, 0.4 * f, 3.0 * gs if f == 3 else 0.0, 0.0, 0.1)
                if f % 2:
                    continue
                if f == 4:
                    g.update_pose(0.4 * f + 1.1, 0.0, 0.0)  # moves the cells' particle ranges as well
                g.grid_cell_occupancy_update(0.1)
                g.resampling()
            assert_vehicle_equal(f"frame {f}", cells.get_particles(), general.get_particles(),
                                 cells.get_grid_cells(), general.get_grid_cells())
            a, c = cells.get_born_masses().view(np.uint32), general.get_born_masses().view(np.uint32)
            np.testing.assert_array_equal(a, c)


def test_batch_with_a_late_vehicle():
    """A vehicle that initialises its particles beside vehicles that read resampled sets, in the same launches.  Batches
    run full updates only and nothing writes their weights, so every vehicle of a batched step has per-cell weights."""
    ps = [small_params(gs=g, res=0.5, n=n, b=n // 10) for g, n in ((40, 9000), (24, 5000), (64, 20000))]
    rng = np.random.default_rng(5)
    with Batch() as batch:
        ids = [batch.add_vehicle(p, SEED, k) for k, p in enumerate(ps)]
        plain = [DOGM(p, seed=SEED, instance=k) for k, p in enumerate(ps)]
        for f in range(3):
            ms = [_grid(int(g.grid_size), rng) for g in plain]
            pose = (0.8 * f, 0.0, 0.0)
            # join one vehicle late: its first update initialises beside the others' resampled sets
            use = [0, 1, 2] if f else [0, 2]
            batch.update([ids[k] for k in use], [ms[k] for k in use], [pose] * len(use), 0.1)
            for k in use:
                plain[k].update_grid(ms[k], *pose, 0.1)
                assert_grid_equal(f"frame {f} vehicle {k}", batch.get_grid_cells(ids[k]), plain[k].get_grid_cells())
        for k, g in enumerate(plain):
            assert_vehicle_equal(f"vehicle {k}", batch.get_particles(ids[k]), g.get_particles(),
                                 batch.get_grid_cells(ids[k]), g.get_grid_cells())
            g.close()
