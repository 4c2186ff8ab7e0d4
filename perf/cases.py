"""What a program does with this framework, as cases that can be timed and compared.

Kinds of case, each through the entry points a program calls:

* ``voxelize``: the reference's call sequence on a handle whose triangles
  are uploaded -- ``computeEdgesFaceNormalsAndBounds`` then
  ``generateVoxelsAndOctTree`` -- with the whole device-resident result
  (occupancy bitmap, node arrays, bricks, block-compressed bricks) as output;
* ``cast``: one camera frame ray cast through a voxelized octree whose bricks
  are resident (a still camera, or one that moves little between frames);
* ``serve``: a few frames of a camera that moves, each cast and then served,
  through a brick pool too small for the tree (uploads and evictions);
* ``tiles``: one front-to-back frame over several octrees that share a pool,
  as a pager draws its visible tiles;
* ``terrain``: the height range and the triangles, normals and texture
  coordinates of one window of a resident height grid, which a pager builds
  before it voxelizes a tile;
* ``tiler``: the triangles of a resident scene assigned to a grid of tiles.

All results are bytes, whole numbers, or floats that every correct build
computes in one stated order, so they are compared exactly.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from voxvizthesis_amd import _lib, scenes
from voxvizthesis_amd.gvpool import BrickPool, OctTree
from voxvizthesis_amd.gvserve import (BrickServer, RayCaster, camera, raycast_front_to_back,
                                      raycast_params)
from voxvizthesis_amd.terrain import DeviceTerrain
from voxvizthesis_amd.voxelizer import Voxelizer

FOV_Y = 60.0


# --- cases -------------------------------------------------------------------

def _vox(name, scene, N, B, cells=0, rocks=0, tris=0, chunk=0, chain=False, compressed=False):
    return {"name": name, "kind": "voxelize", "scene": scene, "N": N, "B": B, "cells": cells,
            "rocks": rocks, "tris": tris, "chunk": chunk, "chain": chain,
            "compressed": compressed}


def listed():
    return [
        # the smallest call there is (two triangles, the reference's own
        # little test grid): launches, host round trips and empty levels
        _vox("voxelize_64_two_triangles", "two", 64, 8),
        # the small terrain workload: one textured terrain group with fill
        _vox("voxelize_128_terrain", "terrain", 128, 8, cells=128),
        # several groups of every kind (textured and plain, with and without
        # vertex normals, wrap / mirror addressing) in a grid and bricks that
        # are no multiples of a tile, a mip chain level by level
        _vox("voxelize_224_mixed_ragged", "mixed", 224, 7, cells=112, chain=True),
        # a plain random soup with vertex normals, the size of the batched
        # workload's middle: every tile a little filled, many tiles, no fill
        _vox("voxelize_512_soup", "soup", 512, 8, tris=199999),
        # the headline workload: terrain and rocks, 1024^3, 16^3 bricks
        _vox("voxelize_1024_terrain_rocks", "terrain", 1024, 16, cells=1024, rocks=2000),
        # the same in the reference's default chunks of 256^3
        _vox("voxelize_1024_chunks_256", "terrain", 1024, 16, cells=1024, rocks=2000, chunk=256),
        # block-compressed output (BC3 / BC1) beside the plain bricks
        _vox("voxelize_512_compressed", "terrain", 512, 16, cells=512, rocks=500,
             compressed=True),
        # one 1080p frame over the headline octree, all bricks resident
        {"name": "cast_1080p_1024", "kind": "cast", "N": 1024, "B": 16, "cells": 1024,
         "rocks": 2000, "W": 1920, "H": 1080, "wide": False},
        # four 720p frames of a moving camera through a pool that evicts
        {"name": "serve_720p_evicting", "kind": "serve", "N": 512, "B": 8, "cells": 512,
         "rocks": 500, "W": 1280, "H": 720, "slots": 4096, "frames": 4, "wide": True},
        # a pager's front-to-back frame over four tiles, an odd viewport
        {"name": "cast_tiles_front_to_back", "kind": "tiles", "N": 512, "B": 16, "cells": 512,
         "tiles": 2, "W": 1283, "H": 717},
        # one tile's window of a terrain, ragged
        {"name": "terrain_tile_1023x1021", "kind": "terrain", "cells": 2048, "cw": 1023,
         "ch": 1021},
        # 2.1 M triangles onto a grid of tiles with borders
        {"name": "tiler_2m_triangles", "kind": "tiler", "cells": 1024, "rocks": 2000, "N": 256,
         "B": 16, "vox": 1024},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["voxelize"] * 5 + ["cast", "cast", "serve", "tiles", "terrain", "tiler"])
    if kind == "terrain":
        cw, ch = _log(rng, 16, 1023), _log(rng, 16, 1021)
        return {"kind": kind, "cells": max(cw, ch) + rng.randint(4, 900), "cw": cw, "ch": ch}
    if kind == "tiler":
        cells = _log(rng, 32, 1000)
        return {"kind": kind, "cells": cells, "rocks": rng.randint(0, 1500),
                "N": rng.choice([64, 128, 256]), "B": 16, "vox": _log(rng, 128, 1024)}
    if kind in ("cast", "serve", "tiles"):
        B = rng.choice([8, 12, 16])
        N = B << rng.randint(3, 5 if B > 8 or kind != "cast" else 6)
        case = {"kind": kind, "N": N, "B": B, "cells": max(32, min(512, N)),
                "W": _log(rng, 65, 1920), "H": _log(rng, 65, 1080)}
        if kind == "tiles":
            case.update(tiles=2, N=min(N, 256), cells=min(case["cells"], 256),
                        W=min(case["W"], 1283), H=min(case["H"], 717))
            case["N"] = B << (3 if B == 16 else 4)
            return case
        case["rocks"] = rng.randint(0, 400)
        case["wide"] = rng.random() < 0.5
        if kind == "serve":
            case.update(W=min(case["W"], 1280), H=min(case["H"], 720), frames=4,
                        slots=_log(rng, 600, 4096))
        return case
    scene = rng.choice(["terrain", "terrain", "mixed", "soup"])
    B = rng.choice([4, 5, 6, 7, 8, 10, 12, 16])
    levels = rng.randint(2, 6)
    while (B << levels) > (1024 if scene == "terrain" else 512) or (B << levels) < 16:
        levels += 1 if (B << levels) < 16 else -1
    N = B << levels
    # a chunk is a multiple of 2^levels below the voxel space
    chunk = 0
    if rng.random() < 0.25 and (N // 4) % (1 << levels) == 0:
        chunk = N // 4
    return {"kind": "voxelize", "scene": scene, "N": N, "B": B,
            "cells": _log(rng, 24, max(32, min(1024, N))) if scene != "soup" else 0,
            "rocks": rng.randint(0, 1500) if scene == "terrain" else 0,
            "tris": _log(rng, 300, 199999) if scene == "soup" else 0, "chunk": chunk,
            "chain": rng.random() < 0.3, "compressed": rng.random() < 0.2}


# --- tensors over the library's device memory ----------------------------------

class _Hold:
    """Objects of the library, closed in the order given once neither the
    state nor a tensor over their memory is left."""

    def __init__(self, *objects):
        self.objects = objects

    def __del__(self):
        for o in self.objects:
            o.close()


class _Span:
    """n values at a device address that hold owns, as torch reads them
    without a copy (the tensor keeps this object, and so the owner)."""

    def __init__(self, hold, ptr, n, typestr):
        self.hold = hold
        self.__cuda_array_interface__ = {"shape": (int(n),), "typestr": typestr,
                                         "data": (int(ptr), False), "version": 2}


def _tensor(hold, ptr, n, typestr="<i4"):
    if not n:
        return torch.empty(0, dtype={"<i4": torch.int32, "<f4": torch.float32,
                                     "|u1": torch.uint8}[typestr], device="cuda")
    return torch.as_tensor(_Span(hold, ptr, n, typestr), device="cuda")


def _views(hold, r: _lib.VoxResult, z: _lib.VoxCompressed | None):
    """The result's arrays: occupancy, then per depth types, constant
    colours, brick indices, brick nodes and bricks (and their blocks)."""
    bvox = (r.brick_dim[0] + 2) * (r.brick_dim[1] + 2) * (r.brick_dim[2] + 2)
    out = [_tensor(hold, r.occupancy, r.occupancy_words)]
    for d in range(r.levels):
        n, nb = r.nodes[d], r.bricks[d]
        out += [_tensor(hold, r.types[d], n, "|u1"), _tensor(hold, r.const_colors[d], n),
                _tensor(hold, r.brick_index[d], n), _tensor(hold, r.brick_node[d], nb),
                _tensor(hold, r.brick_colors[d], nb * bvox),
                _tensor(hold, r.brick_normals[d], nb * bvox)]
        if z is not None:
            k = z.bricks[d] * z.blocks_per_brick
            out += [_tensor(hold, z.colors[d], 16 * k, "|u1"),
                    _tensor(hold, z.normals[d], 8 * k, "|u1")]
    return out


# --- scenes ----------------------------------------------------------------------
#
# Where the outputs' sizes follow from the geometry (bricks, tile lists, node
# textures), a case's geometry is its own and the seed gives what lies on it:
# the texture's colours, the vertex normals, where the triangle list starts,
# the camera's path.  Alphas stay, so the same voxels are empty.

GEOMETRY = 2


def _ramp(seed):
    """The height ramp with every texel's colour moved by the seed."""
    img = scenes.height_ramp_texture(256).astype(np.int64)
    img[..., :3] += np.random.default_rng(seed).integers(-30, 31, img[..., :3].shape)
    return np.clip(img, 0, 255).astype(np.uint8)


def _vary(m, seed):
    """A host mesh with the seed's colours and vertex normals."""
    rng = np.random.default_rng(seed)
    if m.is_terrain:
        m.image = _ramp(seed)
    elif m.image is not None:
        m.image[..., :3] = rng.integers(1, 256, m.image[..., :3].shape)
    if m.vnormals is not None:
        n = m.vnormals + rng.normal(scale=0.1, size=m.vnormals.shape)
        m.vnormals = (n / np.linalg.norm(n, axis=-1, keepdims=True)).astype(np.float32)
    return m


def _add_terrain(vz, t: DeviceTerrain, window, seed):
    """A window of the terrain as a textured terrain group, built on the
    device; the arrays are returned and kept with the handle."""
    x0, y0, cw, ch = window
    bufs = t.tile(x0, y0, cw, ch)
    lo, hi = t.range(x0, y0, cw + 1, ch + 1)
    step = t.extent / t.cells
    n = 2 * cw * ch
    hold = _Hold(*bufs)
    turn = 2 * int(np.random.default_rng(seed).integers(0, cw * ch))
    v, vn, uv = (torch.roll(_tensor(hold, b.ptr, n * k, "<f4"), turn * k)
                 for b, k in zip(bufs, (9, 9, 6)))
    image = torch.from_numpy(_ramp(seed)).cuda()
    torch.cuda.synchronize()
    g = _lib.VoxGroup()
    g.verts, g.vnormals, g.uvs = v.data_ptr(), vn.data_ptr(), uv.data_ptr()
    g.ntri = n
    g.bbox_min[:] = [x0 * step, y0 * step, lo]
    g.bbox_max[:] = [(x0 + cw) * step, (y0 + ch) * step, hi]
    g.is_terrain = 1
    g.rgba8 = image.data_ptr()
    g.width, g.height, g.addr0, g.addr1 = 256, 1, 1, 1
    if not vz._L.vox_add_group_device(vz._h, C.byref(g)):
        raise RuntimeError(vz.getErrorMessage())
    return v, vn, uv, image


def _voxelizer(N, B, chunk=0, options=0, p=(0.0, 0.0, 0.0), delta=None):
    vz = Voxelizer((N,) * 3, (B,) * 3, (chunk,) * 3 if chunk else None, options=options)
    d = np.float32(1.0) / np.float32(N) if delta is None else delta
    if not (vz.initCuda() and vz.allocateVoxelMemory() and vz.setVoxelizationParams(p, (d,) * 3)):
        raise RuntimeError(vz.getErrorMessage())
    return vz


def _rocks(count, geometry):
    return scenes.rocks_on_terrain(scenes.terrain_height_fn(geometry), count, geometry + 1)


def _terrain_scene(case, seed, geometry, chunk=0, options=0):
    """A handle with terrain (and rocks) added, and what it reads from."""
    t = DeviceTerrain(case["cells"], 1.0, geometry)
    vz = _voxelizer(case["N"], case["B"], chunk, options)
    keep = _add_terrain(vz, t, (0, 0, case["cells"], case["cells"]), seed)
    if case.get("rocks"):
        vz.addMesh(_rocks(case["rocks"], geometry))
    return vz, keep


def _host_scene(case):
    """The meshes of the scenes that are built on the host."""
    N, cells, g = case["N"], case["cells"], GEOMETRY
    if case["scene"] == "two":
        m = scenes.scene_two_triangles().meshes[0]
        m.vnormals = np.tile(np.float32([0.0, 0.6, 0.8]), (2, 3, 1))
        return [m]
    if case["scene"] == "soup":
        return [scenes.random_soup(case["tris"], g, N, vertex_normals=True)]
    return [scenes.heightfield_terrain(cells, g),
            scenes.rocks_on_terrain(scenes.terrain_height_fn(g), 40, g + 1, rmin=0.01, rmax=0.06),
            scenes.random_soup(6 * cells, g + 2, N, textured=True, uv_mode="random",
                               vertex_normals=True, translucent=True, addr=(0, 2)),
            scenes.random_soup(4 * cells, g + 3, N, vertex_normals=True)]


def _upload(vz):
    if not vz.allocateTriangleMemory():
        raise RuntimeError(vz.getErrorMessage())


def _generate(vz, compressed=False):
    if not vz.computeEdgesFaceNormalsAndBounds() or \
            not vz.generateVoxelsAndOctTree(None, True, compressed):
        raise RuntimeError(vz.getErrorMessage())


def _tree(case, seed, geometry, slots):
    """A voxelized terrain, its pool (slots bricks) and its octree."""
    vz, keep = _terrain_scene(case, seed, geometry)
    _upload(vz)
    del keep
    _generate(vz)
    vz.releaseWorkMemory()
    if case["wide"]:
        pool = BrickPool((case["B"],) * 3, wide_slots=slots, normals=False)
    else:
        k = 1
        while k ** 3 < slots:
            k += 1
        pool = BrickPool((case["B"],) * 3, (k,) * 3)
    return vz, pool, OctTree(pool, vz)


def _settle(step, limit=200):
    """Frames of a still camera until no brick is missing any more."""
    for _ in range(limit):
        st = step()
        if st.pending == 0 and st.last_uploads == 0:
            return
    raise RuntimeError("the brick pool did not settle")


def _frame_tensors(hold, rc):
    v = rc.view()
    n = v.width * v.height
    return [_tensor(hold, v.rgba, n), _tensor(hold, v.rgba_f32, 4 * n, "<f4"),
            _tensor(hold, v.usage, 12 * n)]


# --- prepare ------------------------------------------------------------------------

def _prepare_voxelize(case, seed):
    options = _lib.VOX_OPT_MIP_CHAIN if case["chain"] else 0
    keep = []
    if case["scene"] == "terrain":
        vz, keep = _terrain_scene(case, seed, GEOMETRY, case["chunk"], options)
    else:
        vz = _voxelizer(case["N"], case["B"], case["chunk"], options,
                        delta=1.0 if case["scene"] == "two" else None)
        for k, m in enumerate(_host_scene(case)):
            vz.addMesh(_vary(m, seed + k))
    _upload(vz)
    return {"hold": _Hold(vz), "vz": vz, "keep": keep, "compressed": case["compressed"],
            "seen": None, "out": None}


def _prepare_cast(case, seed):
    vz, pool, tree = _tree(case, seed, seed, 5 * (case["N"] // case["B"]) ** 2 + 512)
    rc = RayCaster(tree, case["W"], case["H"])
    pos, look, up = scenes.flythrough(seed=seed, frames=64, terrain_seed=seed)[20]
    cam = camera(pos, look, up, FOV_Y, case["W"], case["H"])
    prm = raycast_params((0.0,) * 3, (1.0,) * 3, jitter_seed=5)
    srv = BrickServer(tree)

    def step():
        rc.frame(cam, prm, wait=False)
        return srv.frame(rc)

    _settle(step)
    srv.close()
    hold = _Hold(rc, tree, pool, vz)
    return {"hold": hold, "rc": rc, "cam": cam, "prm": prm, "out": _frame_tensors(hold, rc)}


def _prepare_serve(case, seed):
    vz, pool, tree = _tree(case, seed, GEOMETRY, case["slots"])
    rc = RayCaster(tree, case["W"], case["H"])
    srv = BrickServer(tree)
    path = scenes.flythrough(seed=seed, frames=60, terrain_seed=GEOMETRY)
    prm = raycast_params((0.0,) * 3, (1.0,) * 3, jitter_seed=5)
    cams = [camera(*path[10 + 3 * f], FOV_Y, case["W"], case["H"], f)
            for f in range(case["frames"])]
    for cam in cams + cams:          # the flight's first laps fill the pool
        rc.frame(cam, prm, wait=False)
        srv.frame(rc, wait=False)
    srv.stats()
    v = tree.view()
    ns, sn, nt, nsl = C.c_void_p(), C.c_void_p(), C.c_uint64(), C.c_uint32()
    srv._L.vox_server_state(srv._h, C.byref(ns), C.byref(sn), C.byref(nt), C.byref(nsl))
    texels = v.node_dim[0] * v.node_dim[1] * v.node_dim[2]
    hold = _Hold(srv, rc, tree, pool, vz)
    out = _frame_tensors(hold, rc) + [_tensor(hold, v.nodes, 2 * texels),
                                      _tensor(hold, ns.value, nt.value),
                                      _tensor(hold, sn.value, nsl.value)]
    return {"hold": hold, "rc": rc, "srv": srv, "cams": cams, "prm": prm, "out": out}


def _prepare_tiles(case, seed):
    """tiles^2 unit tiles of one terrain, each voxelized to its own octree."""
    k, N, B, cells = case["tiles"], case["N"], case["B"], case["cells"]
    E = float(k)
    z0 = 0.5 * E - 0.5
    t = DeviceTerrain(k * cells, E, seed)
    margin = ((N // B) >> 1) * cells // N + 2        # cells the voxel border reaches
    boxes, vzs = [], []
    for j in range(k):
        for i in range(k):
            vz = _voxelizer(N, B, p=(float(i), float(j), z0))
            x0, y0 = max(0, i * cells - margin), max(0, j * cells - margin)
            x1 = min(k * cells, (i + 1) * cells + 3 * margin)
            y1 = min(k * cells, (j + 1) * cells + 3 * margin)
            keep = _add_terrain(vz, t, (x0, y0, x1 - x0, y1 - y0), seed)
            _upload(vz)
            _generate(vz)
            vz.releaseWorkMemory()
            del keep
            vzs.append(vz)
            boxes.append(((float(i), float(j), z0), (i + 1.0, j + 1.0, z0 + 1.0)))
    pool = BrickPool((B,) * 3, wide_slots=k * k * (8 * (N // B) ** 2 + 64), normals=False)
    trees = [OctTree(pool, vz, root_brick=False) for vz in vzs]
    texels = max(int(np.prod(tr.get3DTextureDimensions())) for tr in trees)
    srv = BrickServer.shared(pool, len(trees), texels)
    for tr in trees:
        srv.attach(tr)
    pos, look, up = scenes.flythrough(seed=seed, frames=64, extent=E,
                                      height_fn=scenes.terrain_height_fn(seed, E))[20]
    # nearest column first: the order every ray meets the boxes in
    col = [math.floor(float(pos[a])) for a in range(2)]
    order = sorted(range(k * k), key=lambda q: abs(q % k - col[0]) + abs(q // k - col[1]))
    rcs = [RayCaster(trees[q], case["W"], case["H"]) for q in order]
    prms = [raycast_params(*boxes[q], jitter_seed=5) for q in order]
    cam = camera(pos, look, up, FOV_Y, case["W"], case["H"])
    n = case["W"] * case["H"]
    frame = torch.zeros(4 * n, dtype=torch.float32, device="cuda")
    trans = torch.zeros(n, dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    s = {"hold": _Hold(*rcs, *trees, pool, *vzs), "rcs": rcs, "prms": prms, "cam": cam,
         "frame": frame, "trans": trans}

    def step():
        _cast_tiles(s)
        return srv.frame(rcs)

    _settle(step)
    srv.close()
    return s


def _cast_tiles(s):
    raycast_front_to_back(s["rcs"], s["cam"], s["prms"], s["frame"].data_ptr(), 1.0 / 255.0,
                          s["trans"].data_ptr())


def _heights(cells, seed):
    """A rough surface over the unit square: octaves of smoothly interpolated
    random values, (cells + 1)^2 float32, by torch alone."""
    g = torch.Generator().manual_seed(int(seed))
    n1 = cells + 1
    h = torch.zeros(1, 1, n1, n1, dtype=torch.float64, device="cuda")
    for o in range(6):
        k = (4 << o) + 1
        v = torch.rand(1, 1, k, k, generator=g, dtype=torch.float64).cuda() - 0.5
        h += torch.nn.functional.interpolate(v, size=(n1, n1), mode="bicubic",
                                             align_corners=True) * (0.4 * 0.5 ** o)
    return (0.5 + 0.5 * h[0, 0]).float().contiguous()


def _window(case, seed):
    r = np.random.default_rng(seed)
    return (int(r.integers(0, case["cells"] - case["cw"] + 1)),
            int(r.integers(0, case["cells"] - case["ch"] + 1)))


def _prepare_terrain(case, seed):
    nt = 2 * case["cw"] * case["ch"]
    x0, y0 = _window(case, seed)
    s = {"L": _lib.load(), "H": _heights(case["cells"], seed), "n1": case["cells"] + 1, "x0": x0,
         "y0": y0, "cw": case["cw"], "ch": case["ch"],
         "out": [torch.empty(k * nt, dtype=torch.float32, device="cuda") for k in (9, 9, 6)]}
    torch.cuda.synchronize()
    return s


def _prepare_tiler(case, seed):
    t = DeviceTerrain(case["cells"], 1.0, GEOMETRY)
    bufs = t.tile(0, 0, case["cells"], case["cells"])
    n = 9 * 2 * case["cells"] ** 2
    turn = 18 * int(np.random.default_rng(seed).integers(0, case["cells"] ** 2))
    verts = torch.roll(_tensor(_Hold(*bufs, t), bufs[0].ptr, n, "<f4"), turn)
    if case["rocks"]:
        r = torch.from_numpy(_rocks(case["rocks"], GEOMETRY).verts.reshape(-1)).cuda()
        verts = torch.cat([verts, r])
    torch.cuda.synchronize()
    vs = 1.0 / case["vox"]
    g = _lib.VoxTileGrid()
    xy = verts.view(-1, 3)[:, :2]
    lo, hi = xy.amin(0).tolist(), xy.amax(0).tolist()
    for a in range(2):
        g.origin[a] = lo[a]
        g.size[a] = vs * case["N"]
        g.border[a] = vs * ((case["N"] // case["B"]) >> 1)
        g.dim[a] = max(1, math.ceil((hi[a] - lo[a]) / g.size[a]))
    tiler = _Tiler()
    return {"hold": _Hold(tiler), "tiler": tiler, "verts": verts, "grid": g, "seen": None,
            "out": None}


class _Tiler:
    def __init__(self):
        self.L = _lib.load()
        self.h = self.L.vox_tiler_create()

    def close(self):
        self.L.vox_tiler_destroy(self.h)


_PREPARE = {"voxelize": _prepare_voxelize, "cast": _prepare_cast, "serve": _prepare_serve,
            "tiles": _prepare_tiles, "terrain": _prepare_terrain, "tiler": _prepare_tiler}


def prepare(case, seed):
    # seeds of the generators are kept small and apart (rocks and soups use
    # the next few)
    s = _PREPARE[case["kind"]](case, 8 * (int(seed) % 100003))
    s["kind"] = case["kind"]
    return s


# --- run ------------------------------------------------------------------------------

def _run_voxelize(s):
    vz = s["vz"]
    _generate(vz, s["compressed"])
    r = vz.raw_result()
    z = None
    if s["compressed"]:
        z = _lib.VoxCompressed()
        vz._L.vox_get_compressed(vz._h, C.byref(z))
    # the views are made again only when an address or a count has changed
    now = (bytes(r), bytes(z) if z is not None else b"")
    if s["seen"] != now:
        s["seen"], s["out"] = now, _views(s["hold"], r, z)
    return s["out"]


def _run_cast(s):
    s["rc"].frame(s["cam"], s["prm"], wait=False)
    return s["out"]


def _run_serve(s):
    for cam in s["cams"]:
        s["rc"].frame(cam, s["prm"], wait=False)
        s["srv"].frame(s["rc"], wait=False)
    return s["out"]


def _run_tiles(s):
    _cast_tiles(s)
    return [s["frame"], s["trans"]]


def _run_terrain(s):
    L, mm = s["L"], (C.c_float * 2)()
    H, o = s["H"].data_ptr(), s["out"]
    if not L.vox_terrain_range(H, s["n1"], s["x0"], s["y0"], s["cw"] + 1, s["ch"] + 1, mm) or \
            not L.vox_terrain_tile(H, s["n1"], 1.0, s["x0"], s["y0"], s["cw"], s["ch"], mm[0],
                                   mm[1], 256, o[0].data_ptr(), o[1].data_ptr(), o[2].data_ptr()):
        raise RuntimeError(L.vox_terrain_get_error().decode())
    return [float(mm[0]), float(mm[1])] + o


def _run_tiler(s):
    L, h, v = s["tiler"].L, s["tiler"].h, s["verts"]
    if not L.vox_tiler_assign(h, v.data_ptr(), v.numel() // 9, 1, C.byref(s["grid"])):
        raise RuntimeError(L.vox_tiler_get_error(h).decode())
    r = _lib.VoxTileLists()
    L.vox_tiler_get(h, C.byref(r))
    now = bytes(r)
    if s["seen"] != now:
        s["seen"] = now
        k = s["hold"]
        s["out"] = [_tensor(k, r.tile_start, r.ntiles + 1), _tensor(k, r.tile_tris, r.pairs),
                    _tensor(k, r.tile_zmin, r.ntiles, "<f4"),
                    _tensor(k, r.tile_zmax, r.ntiles, "<f4")]
    return s["out"]


_RUN = {"voxelize": _run_voxelize, "cast": _run_cast, "serve": _run_serve, "tiles": _run_tiles,
        "terrain": _run_terrain, "tiler": _run_tiler}


def run(state):
    return _RUN[state["kind"]](state)


# --- work, tolerance, exact ---------------------------------------------------------------

def _bricks(case, per=3.6):
    """About how many bricks an octree over a surface has: per R^2 at a depth
    of R nodes an axis (a terrain measures 3.4 to 3.8), all nodes at most."""
    n, R = 0.0, case["N"] // case["B"]
    while R >= 1:
        n += min(R ** 3, per * R * R)
        R //= 2
    return n


def _soup_bricks(case):
    n, R = 0.0, case["N"] // case["B"]
    while R >= 1:
        n += R ** 3 * (1.0 - math.exp(-case["tris"] * 2.0 / R ** 3))
        R //= 2
    return n


def work(case):
    kind = case["kind"]
    if kind == "voxelize":
        R = case["N"] // case["B"]
        S = case["N"] + 4 * (R >> 1)
        terrain = 2 * case["cells"] ** 2
        plain = case["tris"] + 80 * case["rocks"] + (2 if case["scene"] == "two" else 0)
        if case["scene"] == "mixed":
            plain += 3200 + 10 * case["cells"]
        # vertices, vertex normals and texture coordinates in; bitmap, node
        # arrays and bricks (colour and normal) out
        bricks = _soup_bricks(case) if case["scene"] == "soup" else \
            4.0 if case["scene"] == "two" else _bricks(case)
        brick = 8 * (case["B"] + 2) ** 3
        out = S ** 3 / 8 + 9 * R ** 3 * 8 / 7 + bricks * brick
        if case["compressed"]:
            out += bricks * 24 * math.ceil((case["B"] + 2) / 4) ** 2 * (case["B"] + 2)
        # about 20 overlap tests of 40 operations a triangle
        return {"bytes": 96 * terrain + 36 * plain + out, "flops": 800 * (terrain + plain)}
    if kind in ("cast", "serve", "tiles"):
        # each frame writes its images and usage lists (68 B a pixel; 20 B
        # front to back), and a ray takes about 60 trilinear samples of 70
        # operations
        n = case["W"] * case["H"] * case.get("frames", 1)
        return {"bytes": n * (20 if kind == "tiles" else 68), "flops": n * 60 * 70}
    if kind == "terrain":
        cells = case["cw"] * case["ch"]
        return {"bytes": 2 * 4 * cells + 2 * 96 * cells, "flops": 120 * cells}
    T = 2 * case["cells"] ** 2 + 80 * case["rocks"]
    return {"bytes": (36 + 5) * T, "flops": 30 * T}


def tolerance(case):
    return "exact"


def exact(case, seed):
    """Only the terrain window computes numbers that 64 bits give better: the
    others give bytes and whole numbers, minima and maxima of their inputs,
    or (ray casts) follow the fp32 decisions of a stated order, without which
    a ray samples another level of the octree."""
    if case["kind"] != "terrain":
        return None
    seed = 8 * (int(seed) % 100003)
    x0, y0 = _window(case, seed)
    cw, ch, n1 = case["cw"], case["ch"], case["cells"] + 1
    H = _heights(case["cells"], seed).double()
    step = 1.0 / (n1 - 1)
    lo = float(H[y0:y0 + ch + 1, x0:x0 + cw + 1].min())
    hi = float(H[y0:y0 + ch + 1, x0:x0 + cw + 1].max())
    P = torch.nn.functional.pad(H[None, None], (1, 1, 1, 1), mode="replicate")[0, 0]
    dx = (P[1:-1, 2:] - P[1:-1, :-2]) / (2.0 * step)
    dy = (P[2:, 1:-1] - P[:-2, 1:-1]) / (2.0 * step)
    n = torch.stack([-dx, -dy, torch.ones_like(dx)], -1)
    n = n / n.norm(dim=-1, keepdim=True)
    a = torch.arange(n1, dtype=torch.float64, device="cuda") * step
    p = torch.stack([a[None, :].expand(n1, n1), a[:, None].expand(n1, n1), H], -1)

    def soup(q):
        q = q[y0:y0 + ch + 1, x0:x0 + cw + 1]
        v00, v10, v11, v01 = q[:-1, :-1], q[:-1, 1:], q[1:, 1:], q[1:, :-1]
        return torch.stack([v00, v10, v11, v00, v11, v01], 2).reshape(-1)

    verts = soup(p)
    t = (verts.view(-1, 3, 3)[:, :, 2].mean(1) - lo) / max(hi - lo, 1e-12)
    u = ((t * 256).floor().clamp(0, 255) + 0.5) / 256
    uv = torch.stack([u, torch.full_like(u, 0.5)], -1)[:, None].expand(-1, 3, 2)
    return [lo, hi, verts, soup(n), uv.reshape(-1)]
