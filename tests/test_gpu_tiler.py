"""Tiler on the GPU: the device triangle-to-tile assignment equals the
tiler oracle's (sets per tile, and the z extents), and a tiled terrain +
rocks scene produces one octree per non-empty tile whose files load the way
the reference's reader loads them, listed in root.gvp."""
import os

import numpy as np
import pytest

import oracle
from oracle import tiler as ot
from voxvizthesis_amd import scenes
from voxvizthesis_amd.tiler import PagedOctTreeGenerator, TileAssignment

pytestmark = pytest.mark.gpu


def test_device_assignment_matches_oracle():
    sc = scenes.scene_full_octree(cells=64, N=64, B=8, n_rocks=60)
    gen = PagedOctTreeGenerator(sc.meshes, voxel_size=1.0 / 256, N=64, B=8)
    g = gen.grid()
    print(f"[tiler] grid {gen.dim} triangles {gen.verts.shape[0]}", flush=True)
    a = TileAssignment(gen.verts, g)
    ref = ot.assign(gen.verts, tuple(g.origin), tuple(g.size), tuple(g.border), tuple(g.dim))
    n = g.dim[0] * g.dim[1]
    assert gen.dim == (4, 4)
    for t in range(n):
        got = a.tile(t).tolist()
        assert got == ref.get(t, []), f"tile {t}"
        if got:
            z = gen.verts.reshape(-1, 3, 3)[got][:, :, 2]
            assert a.zmin[t] == z.min() and a.zmax[t] == z.max()
    # the border duplicates triangles into neighbours
    assert a.tris.size > gen.verts.shape[0]


def test_tiled_generation_writes_loadable_trees(tmp_path):
    sc = scenes.scene_full_octree(cells=64, N=64, B=8, n_rocks=40)
    gen = PagedOctTreeGenerator(sc.meshes, voxel_size=1.0 / 128, N=64, B=8)
    res = gen.generate(str(tmp_path))
    print(f"[tiler] {len(res)} trees", flush=True)
    assert len(res) >= 4 and all(st in (1, -1) for (_, _, _, st, _) in res)
    root = (tmp_path / "root.gvp").read_text().splitlines()
    listed = [l for l in root if "<OctTree " in l]
    ok = [r for r in res if r[3] == 1]
    assert len(listed) == len(ok) and len(ok) > 0
    for (x, y, z, st, ntri) in ok:
        d = os.path.join(str(tmp_path), f"grid_{x}_{y}_{z}")
        p = oracle.pool_load(d, slots=(8, 8, 8))
        assert p.blocks >= 1


def _soup(ntri, seed, dim, spread):
    """Triangles over a dim[0] x dim[1] tile grid of unit tiles: most within
    a tile or across an edge, one in eight with edges of `spread` tiles."""
    rng = np.random.default_rng(seed)
    c = rng.uniform(-0.5, 1.0, (ntri, 1, 3)) + rng.uniform(0, 1, (ntri, 1, 3)) * (dim[0], dim[1], 1)
    e = np.where(rng.random((ntri, 1, 1)) < 0.125, spread, 0.2)
    return (c + rng.normal(size=(ntri, 3, 3)) * e).astype(np.float32)


# counts around a group of 64, a workgroup's run and two of them; grids of one
# tile, ragged ones, the largest whose counters fit LDS (1024 tiles) and the
# next (sorted instead)
@pytest.mark.parametrize("ntri,dim,spread", [
    (1, (1, 1), 0.2), (63, (3, 1), 1.0), (64, (1, 5), 1.0), (65, (7, 5), 2.0), (256, (4, 4), 9.0),
    (257, (31, 33), 3.0), (700, (32, 32), 40.0), (700, (33, 32), 40.0), (3001, (5, 3), 1.0)])
def test_device_assignment_sizes(ntri, dim, spread):
    from voxvizthesis_amd import _lib
    verts = _soup(ntri, ntri, dim, spread)
    g = _lib.VoxTileGrid()
    g.origin[:], g.size[:], g.border[:], g.dim[:] = (0.0, 0.0), (1.0, 1.0), (0.1, 0.1), dim
    print(f"[tiler] {ntri} triangles on {dim}", flush=True)
    a = TileAssignment(verts, g)
    ref = ot.assign(verts, (0.0, 0.0), (1.0, 1.0), (0.1, 0.1), dim)
    assert a.start[0] == 0 and a.start[-1] == a.tris.size == sum(map(len, ref.values()))
    for t in range(dim[0] * dim[1]):
        want = ref.get(t, [])
        assert a.tile(t).tolist() == want, f"tile {t}"
        z = verts[want][:, :, 2]
        if want:
            assert a.zmin[t] == z.min() and a.zmax[t] == z.max(), f"tile {t}"
        else:
            assert np.isnan(a.zmin[t]) and np.isnan(a.zmax[t]), f"tile {t}"


# waves of few boxes (triangles sorted along rows of tiles) and of many (in no
# order), boxes of a tile or two and boxes over much of the grid, counted in LDS
# and in memory; grids at the 32 tiles from which the lists are written by a lane
# per tile, and of one and several rows in its 64
@pytest.mark.parametrize("dim", [(1, 1), (6, 4), (31, 1), (8, 4), (13, 5), (65, 2), (32, 32),
                                 (1024, 1), (40, 40), (3, 700)])
@pytest.mark.parametrize("rows", [True, False])
@pytest.mark.parametrize("spread", [0.2, 12.0])
def test_device_assignment_orders(dim, rows, spread):
    from voxvizthesis_amd import _lib
    verts = _soup(1500, 7, dim, spread)
    if rows:
        c = np.floor(verts.mean(1))
        verts = np.ascontiguousarray(verts[np.lexsort((c[:, 0], c[:, 1]))])
    g = _lib.VoxTileGrid()
    g.origin[:], g.size[:], g.border[:], g.dim[:] = (0.0, 0.0), (1.0, 1.0), (0.1, 0.1), dim
    print(f"[tiler] {dim} rows={rows} spread={spread}", flush=True)
    a = TileAssignment(verts, g)
    ref = ot.assign(verts, (0.0, 0.0), (1.0, 1.0), (0.1, 0.1), dim)
    assert a.start[-1] == a.tris.size == sum(map(len, ref.values()))
    for t in range(dim[0] * dim[1]):
        want = ref.get(t, [])
        assert a.tile(t).tolist() == want, f"tile {t}"
        if want:
            z = verts[want][:, :, 2]
            assert a.zmin[t] == z.min() and a.zmax[t] == z.max(), f"tile {t}"
