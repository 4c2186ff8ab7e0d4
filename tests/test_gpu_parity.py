"""HIP path against the oracle, bit-exact (GPU)."""
import numpy as np
import pytest

import oracle
from tests._compare import compare_results
from voxvizthesis_amd import scenes
from voxvizthesis_amd._lib import VOX_OPT_MIP_CHAIN
from voxvizthesis_amd.voxelizer import voxelize_scene

pytestmark = pytest.mark.gpu


def _check(scene, chain=False, levels=True):
    print(f"[parity] {scene.name} chain={chain} T={scene.ntri}", flush=True)
    ref = oracle.run(scene, flags=oracle.REF_MIP_CHAIN if chain else 0, keep_mips=levels)
    vz = voxelize_scene(scene, options=VOX_OPT_MIP_CHAIN if chain else 0)
    try:
        assert vz.status == ref.status
        res = vz.result()
        gl = [vz.level(k) for k in range(ref.levels)] if levels else None
        errs = compare_results(res, ref, ref_mips=ref.mips, gpu_levels=gl)
        assert not errs, "\n".join(errs[:20])
    finally:
        vz.close()
    return ref


def test_two_triangles():
    ref = _check(scenes.scene_two_triangles())
    assert int(np.unpackbits(ref.occupancy.view(np.uint8)).sum()) > 0


def test_small_terrain():
    _check(scenes.scene_small_terrain())


def test_small_terrain_mip_chain():
    _check(scenes.scene_small_terrain(), chain=True)


def test_mixed_groups():
    _check(scenes.scene_mixed())


def test_mixed_groups_b4():
    _check(scenes.scene_mixed(seed=9, N=64, B=4))


def test_mixed_groups_rocks_first():
    # the first group is no terrain: every level-0 voxel no group reaches is zero
    _check(scenes.scene_mixed(seed=5, order="rocks_first"))


def test_mixed_groups_two_terrains():
    # a second terrain fills over voxels that the first fill and the rocks hold
    _check(scenes.scene_mixed(seed=6, order="two_terrains"))


def test_more_groups_than_one_binning_launch_holds():
    # setup and scatter take at most 8 groups per launch: 11 groups with
    # triangles (10 inside the grid) need two launches of each, and the
    # terrain's fill runs in the second
    _check(scenes.scene_many_groups())


def test_big_and_small_triangles_binned():
    # boxes of 18^3 tiles walk their bins; the small ones are listed as pairs
    _check(scenes.scene_big_triangles())


def test_type_x_split_miss():
    # N=256, B=4: the leaf typing launch split leaves x = N + extra (the +1
    # border of the last node column) unexamined.
    _check(scenes.scene_terrain_n(128, 256, 4), levels=False)


def test_brick_sizes_not_powers_of_two():
    # (B + 2)^3 odd (B = 3, 5): the brick gather writes single words; B = 6
    # writes 16-byte runs of a region that starts mid-tile
    for N, B in ((48, 3), (80, 5), (96, 6)):
        _check(scenes.scene_terrain_n(64, N, B))


def test_full_octree_generator_256():
    # the headline workload's own generator (fBm terrain + 2,000 rocks, 16^3
    # bricks) at a size the oracle runs in seconds: 256^3, depths 0-4
    _check(scenes.scene_full_octree(cells=256, N=256, B=16))


def test_full_octree_generator_512():
    # the same at 512^3 (depths 0-5, 526 K triangles), every level compared
    _check(scenes.scene_full_octree(cells=512, N=512, B=16))


def test_reference_default_brick_edge_30():
    # main.cu's default brick edge of 30 (32^3 stored bricks), N / B = 8
    _check(scenes.scene_terrain_n(120, 240, 30))


def test_brick_wider_than_the_gather_tile_table():
    # B = 64: a stored brick of 66^3 spans 9 tiles per axis, more than the
    # brick gather stages in LDS (6), so it reads the tile map directly
    _check(scenes.scene_terrain_n(64, 128, 64))


# bricks of one wave's batch (10 voxels an axis), one voxel more, the largest
# whose tiles are staged (39) and the next, which reads the maps per voxel
@pytest.mark.parametrize("N,B", [(32, 8), (36, 9), (78, 39), (80, 40)])
def test_brick_sizes_at_the_gather_s_edges(N, B):
    _check(scenes.scene_mixed(seed=21, N=N, B=B))


# bricks that reach 6 or 7 tiles an axis by where they start (some staged, some
# read from the maps, in one launch), the widest of them, the next, which
# always reach 7, and bricks that are flat on one axis
@pytest.mark.parametrize("N,B", [((176,) * 3, (44,) * 3), ((184,) * 3, (46,) * 3),
                                 ((188,) * 3, (47,) * 3), ((320, 320, 32), (80, 80, 8))], ids=str)
def test_bricks_staged_by_the_tiles_they_reach(N, B):
    cube = scenes.scene_mixed(seed=22, N=max(N), B=max(B))
    _check(scenes.Scene(meshes=cube.meshes, N=N, B=B, name=f"staged_{B[0]}_{B[2]}",
                        p=cube.p, delta=cube.delta))
