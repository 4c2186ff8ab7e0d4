"""Tile maps of levels of more than 512 x 1024 tiles (GPU), whose workgroups
take four rows of 1024: a 2048 x 2048 x 512 grid in 64 x 64 x 16 bricks has
5 M tiles on level 0 and 627 K, no whole number of workgroups, on level 1.  The
triangles lie inside one voxel each, so the occupied voxels, the active tiles of
every level and the voxels of level 1 follow from their positions alone."""
import numpy as np
import pytest

from voxvizthesis_amd import scenes
from voxvizthesis_amd._lib import VOX_OPT_MIP_CHAIN
from voxvizthesis_amd.voxelizer import voxelize_scene

pytestmark = pytest.mark.gpu

N, B, LEVELS, EXTRA = (2048, 2048, 512), (64, 64, 16), 6, 16
S = tuple(n + 4 * EXTRA for n in N)


def _voxels():
    """A row of voxels through every tile along x, the corners, the voxels of
    tiles at the ends of rows of 1024 and of workgroups of 4096, and others."""
    rng = np.random.default_rng(4)
    tg = [s // 8 for s in S]
    ends = np.concatenate([k * np.arange(1, 30) + o for k in (1024, 4096) for o in (-1, 0)])
    ends = np.concatenate([ends, [0, tg[0] * tg[1] * tg[2] - 1]])
    tiles = np.stack([ends % tg[0], ends // tg[0] % tg[1], ends // (tg[0] * tg[1])], 1)
    row = np.stack([np.arange(3, S[0], 8), np.full(tg[0], 1003), np.full(tg[0], 301)], 1)
    corners = np.array(np.meshgrid(*[(0, s - 1) for s in S])).reshape(3, -1).T
    v = np.concatenate([8 * tiles + rng.integers(0, 8, tiles.shape), row, corners,
                        rng.integers(0, S, (300, 3))])
    return np.unique(v, axis=0)


def _scene(vox, terrain):
    tri = np.array([[-0.2, -0.2, 0.0], [0.2, -0.2, 0.1], [0.0, 0.2, -0.1]])
    m = scenes.Mesh((vox[:, None] - EXTRA + 0.5 + tri).astype(np.float32))
    if terrain:
        m.uvs = np.full((len(vox), 3, 2), 0.5, np.float32)
        m.image, m.is_terrain = np.full((1, 4, 4), 255, np.uint8), True
    return scenes.Scene(meshes=[m], N=N, B=B, delta=(1.0,) * 3, name="voxels")


@pytest.mark.parametrize("terrain", [False, True])
def test_maps_of_four_rows_follow_from_the_voxels(terrain):
    vox = _voxels()
    vz = voxelize_scene(_scene(vox, terrain), options=VOX_OPT_MIP_CHAIN)
    try:
        print(f"[tilemaps] {len(vox)} voxels terrain={terrain}", flush=True)
        t = vox >> 3
        if terrain:   # the fill reaches three tiles down
            t = np.concatenate([t - (0, 0, q) for q in range(4)])
            t = t[t[:, 2] >= 0]
        st = vz.stats()
        for k in range(LEVELS):
            dims = np.array([s >> k for s in S])
            t = np.unique(t[(t < (dims + 7) // 8).all(1)], axis=0)
            assert st.active_tiles[k] == len(t), f"level {k}"
            t = t >> 1
        r = vz.raw_result()
        occ = vz._d2h(r.occupancy, r.occupancy_words, np.uint32)
        w = np.flatnonzero(occ)
        bits = np.unpackbits(occ[w].view(np.uint8), bitorder="little").reshape(-1, 32)
        a, b = np.nonzero(bits)
        assert np.array_equal(np.sort(w[a] * 32 + b),
                              np.sort((vox[:, 2] * S[1] + vox[:, 1]) * S[0] + vox[:, 0]))
        if terrain:
            return
        # level 1, the bricks one depth above the leaves
        d, e = LEVELS - 2, [x + 2 for x in B]
        R = 1 << d
        node = vz._d2h(r.brick_node[d], r.bricks[d], np.uint32).astype(np.int64)
        col = vz._d2h(r.brick_colors[d], r.bricks[d] * e[0] * e[1] * e[2], np.uint32)
        col = col.reshape(-1, e[2], e[1], e[0])
        v1 = np.unique(vox >> 1, axis=0)
        assert len(node) > 100
        for n, c in zip(node, col):
            lo = np.array([n % R, n // R % R, n // (R * R)]) * B + (EXTRA >> 1) - 1
            q = v1[((v1 >= lo) & (v1 < lo + e)).all(1)] - lo
            want = np.zeros_like(c, bool)
            want[q[:, 2], q[:, 1], q[:, 0]] = True
            assert np.array_equal(c != 0, want), f"node {n}"
    finally:
        vz.close()
