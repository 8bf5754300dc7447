"""The parity scenes with one agent per lane.  In the default launch shape a
plain step of a small crowd takes 16 lanes per agent, so the scenes of the
other files, which set no shape, reach k_row_step; here every simulator they
make starts in another shape, and they run the kernels that larger crowds and
other shapes take: the seeded k-nearest walk, the main ORCA pass inside and
behind it and with 16 agents per wavefront, the overflow pass (one agent per
wavefront, and per lane when its queue is longer than the grid: the scene of
6,000 agents between pillars asserts more than 1,024 queued), its tile for
long obstacle lists and the 3D-LP queue."""
import pytest

import test_gpu_collisions as collisions
import test_gpu_knn_seeds as seeds
import test_gpu_knn_walk as walk
import test_gpu_parity_scenes as scenes
import test_gpu_parity_small as small
from ecmgenerator_amd.simulator import Simulator

pytestmark = pytest.mark.gpu


@pytest.fixture(params=[(64, 2), (256, 1), (16, 2), (128, 4)], ids=str)
def lanes(request, monkeypatch):
    create = Simulator.__init__

    def init(self, *args, **kwargs):
        create(self, *args, **kwargs)
        self.set_tuning(knn_block=request.param[0], orca_obst_slots=request.param[1])
    monkeypatch.setattr(Simulator, "__init__", init)


@pytest.mark.parametrize("cell", [0.5, 1.5, 40.0])
def test_lattice_ties(lanes, cell):
    walk.test_lattice_ties(cell)


SCENES = [walk.test_lattice_moving_to_border, walk.test_sparse_far_neighbours,
          seeds.test_reused_slots_and_destroyed_neighbours, seeds.test_snapshot_from_another_time,
          seeds.test_slots_reused_across_environments, seeds.test_spawn_remove_respawn_between_steps,
          collisions.test_zero_w_colliding_pair_gives_the_reference_nan,
          collisions.test_coincident_pair_is_invisible_to_itself, collisions.test_corridor_parallel_walls,
          small.test_parity_reference_literal_params, small.test_parity_dense_crowd,
          small.test_parity_pillar_forest_obstacle_overflow, small.test_parity_pillar_forest_long_overflow_queue,
          small.test_parity_obstacle_buckets_longer_than_64_edges, scenes.test_c0_full_parity,
          scenes.test_c0_reference_literal_parity]


@pytest.mark.parametrize("scene", SCENES, ids=lambda f: f.__name__[5:])
def test_scene(lanes, scene):
    scene()
