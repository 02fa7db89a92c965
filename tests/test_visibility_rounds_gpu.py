"""The visibility pass at the edges of its rounds of 256 records, of the
passes of 2,048 records whose boxes it tests and of the windows of 2,048
quads, and shading at the ends of the range of its corrected reciprocals,
against the oracle bit for bit."""
import numpy as np
import pytest
import torch  # noqa: F401

from rsr_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,width,height,segment", [(1, 33, 17, 512), (127, 64, 64, 512), (128, 61, 35, 512), (129, 64, 64, 512),
                                                    (257, 64, 64, 512), (1024, 64, 40, 4096), (1025, 64, 40, 4096), (1153, 50, 64, 4096)])
def test_record_counts(n, width, height, segment):
    # one tile of 2 n records, in one segment or several
    import oracle_backend
    from rsr_amd import rgl
    from test_parity_gpu import _compare
    from test_shared_tiles_gpu import _walls
    sc = _walls(n, width, height)
    sc.tile_blocks, sc.name = (8, 8), f"rounds_{sc.name}_{segment}"
    g = rgl.GPU(0)
    g.set_raster_params(segment, 0)
    _compare(sc.name, oracle_backend.render(sc, threads=8), rgl.render(sc, gpu=g))
    g.close()


@pytest.mark.parametrize("scale", [0.0, 1e-22, 2.0 ** -51, 2.0 ** -50, 1e18, 3e19])
def test_normals_at_the_ends_of_the_range(scale):
    # squared lengths of 0, 1e-44 (subnormal), 2^-102 within a factor of two
    # either way, 1e36 and infinity
    import oracle_backend
    from rsr_amd import rgl
    from test_parity_gpu import _compare
    sc = scenes.scene_icospheres(160, 90, instances=24)
    for k in (3, 4, 5):
        sc.meshes[0].buffers[k] = (sc.meshes[0].buffers[k] * np.float32(scale)).astype(np.float32)
    sc.name = f"normals_{scale:g}"
    _compare(sc.name, oracle_backend.render(sc, threads=8), rgl.render(sc))


@pytest.mark.parametrize("x,y,w,h,width,height,blocks", [(5, 3, 21, 19, 40, 40, (8, 8)), (1, 0, 62, 64, 64, 64, (8, 8)),
                                                         (33, 31, 7, 9, 64, 64, (8, 8)), (9, 11, 60, 37, 121, 71, (5, 3))])
def test_scissored_tiles_of_many_pairs(x, y, w, h, width, height, blocks):
    # the pair boxes are the tile's; the scissor rectangle comes with the setup
    import inorder_scenes as S
    from oracle_backend import render_calls as oracle_calls
    from rsr_amd import rgl
    sc = S.scene_scissor(x, y, w, h, width, height, blocks, name=f"scissor_{x}_{y}_{w}_{h}_{width}x{height}")
    ref, rst = oracle_calls(sc, threads=8)
    out, gst = rgl.render_calls(sc)
    assert rst["fragments"] == gst["fragments"]
    for k, (r, g) in enumerate(zip(ref, out)):
        assert np.array_equal(r.view(np.uint32), g.view(np.uint32)), f"{sc.name} output {k}"
