"""Triangles of many tiles, whose tiles the scatter shares out over its
workgroup: counts around the rounds of 256, the unit of 512 and the list's
512 entries (the last with units grown by a target of 2,112 tiles), against
the oracle bit for bit."""
import numpy as np
import pytest
import torch  # noqa: F401

from rsr_amd import scenes

pytestmark = pytest.mark.gpu


def _walls(n, width, height):
    """n upright quads one behind the other, each about 300 tiles of 32 px."""
    sc = scenes.scene_clip_floor(width, height, 2)
    z = -3.0 - 0.01 * np.arange(n)
    q = np.array([(-1.6, -0.9), (1.6, -0.9), (1.6, 0.9), (-1.6, 0.9)], np.float32)
    pos = np.concatenate([np.tile(q, (n, 1)), np.repeat(z, 4)[:, None]], 1).astype(np.float32)
    nrm = np.tile(np.array([[0, 0, 1]], np.float32), (4 * n, 1))
    uv = np.tile(np.array([(0, 0), (1, 0), (1, 1), (0, 1)], np.float32), (n, 1))
    idx = (np.arange(n)[:, None] * 4 + np.array([0, 1, 2, 0, 2, 3])).reshape(-1).astype(np.uint16)
    sc.meshes = [scenes.Mesh(scenes._mesh_buffers(pos, nrm, uv), idx)]
    sc.view = scenes.look_at((0, 0, 0), (0, 0, -1), (0, 1, 0))
    sc.tile_blocks, sc.cull, sc.name = (4, 4), False, f"walls{n}_{width}x{height}_tile32"
    return sc


def test_tiles_of_8_pixels():
    # 32,400 tiles: the unit's tile window leaves no room for its list
    import oracle_backend
    from rsr_amd import rgl
    from test_parity_gpu import _compare
    sc = _walls(3, 1920, 1080)
    sc.tile_blocks, sc.name = (1, 1), "walls3_1920x1080_tile8"
    _compare(sc.name, oracle_backend.render(sc, threads=8), rgl.render(sc))


@pytest.mark.parametrize("n,width,height", [(1, 333, 211), (128, 640, 360), (129, 640, 360), (300, 640, 360),
                                            (256, 2048, 1056), (300, 2048, 1056)])
def test_walls(n, width, height):
    import oracle_backend
    from rsr_amd import rgl
    from test_parity_gpu import _compare
    sc = _walls(n, width, height)
    ref = oracle_backend.render(sc, threads=8)
    # the first frame may report a full list: render() draws it again
    _compare(sc.name, ref, rgl.render(sc))


@pytest.mark.parametrize("n,width,height,blocks,cull", [(1, 64, 40, (8, 8), False), (7, 131, 77, (5, 3), False), (63, 200, 120, (3, 8), True),
                                                        (1025, 120, 72, (4, 4), False), (2050, 97, 61, (8, 8), True)])
def test_triangles_around_the_camera(n, width, height, blocks, cull):
    # triangles that cross several clipping planes (polygons of three to eight
    # vertices, parts left of and above the frame), tiles that are no power of
    # two, more triangles than the clipping launch has waves
    import oracle_backend
    from rsr_amd import rgl
    from test_parity_gpu import _compare
    sc = scenes.scene_clip_floor(width, height, 2)
    rng = np.random.RandomState(n)
    pos = rng.uniform(-4, 4, (3 * n, 3)).astype(np.float32)
    nrm = np.tile(np.array([[0, 0, 1]], np.float32), (3 * n, 1))
    uv = rng.uniform(-1, 2, (3 * n, 2)).astype(np.float32)
    sc.meshes = [scenes.Mesh(scenes._mesh_buffers(pos, nrm, uv), np.arange(3 * n, dtype=np.uint16))]
    sc.tile_blocks, sc.cull, sc.name = blocks, cull, f"around{n}_{width}x{height}"
    ref = oracle_backend.render(sc, threads=8)
    assert n == 1 or ref[3]["clipped"] > n // 2
    _compare(sc.name, ref, rgl.render(sc))
