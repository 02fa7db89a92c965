"""A binning unit's tile window at the ends of what a workgroup's LDS holds:
the largest windows draw as the oracle does, and larger ones are refused
before any of the frame's kernels runs, the recorder still usable after."""
import pytest
import torch

from rsr_amd import scenes

pytestmark = pytest.mark.gpu


def _tile8(width, height, blend=False):
    from test_shared_tiles_gpu import _walls
    sc = _walls(3, width, height)
    sc.tile_blocks, sc.blend, sc.name = (1, 1), blend, f"walls3_{width}x{height}_tile8"
    return sc


# 39,900 tiles; 40,000; 40,300 (the window's 161,200 bytes beside the scatter's 2,608)
@pytest.mark.parametrize("width,height,blend", [(2128, 1200, False), (2000, 1280, True), (1240, 2080, False)])
def test_largest_windows(width, height, blend):
    import oracle_backend
    from rsr_amd import rgl
    from test_parity_gpu import _compare
    sc = _tile8(width, height, blend)
    _compare(sc.name, oracle_backend.render(sc, threads=8), rgl.render(sc))


# 40,320 tiles; 40,800; 41,216
@pytest.mark.parametrize("width,height", [(2016, 1280), (2040, 1280), (2048, 1288)])
def test_larger_windows_are_refused(width, height):
    import oracle_backend
    from rsr_amd import rgl
    from test_parity_gpu import _compare
    g = rgl.GPU(0)
    sc = _tile8(width, height)
    ds = rgl.DeviceScene(sc, "cuda:0", True)
    ds.record(g)
    stream = torch.cuda.current_stream().cuda_stream
    for graph in (False, True):
        g.set_graph(graph)
        with pytest.raises(rgl.RglError, match=r"too many tiles.*\(-4\)"):
            g.run(stream)
    g.set_graph(False)
    small = scenes.scene_sphere_ground(160, 96)
    _compare(small.name, oracle_backend.render(small, threads=8), rgl.render(small, gpu=g))
    g.close()
