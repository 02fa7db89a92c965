"""The texture preparation's separate entry points (decode, power-of-two
resample, mip chain), called one after the other, against the one that does
all three: the same texture, bit for bit."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("h,w,pm", [(1, 1, False), (2, 2, True), (5, 17, True), (64, 64, False), (60, 100, False), (65, 128, True),
                                    (777, 1000, True), (1024, 1024, False)])
def test_steps_equal_the_one_pass(h, w, pm):
    from rsr_amd import rgl
    L = rgl.lib()
    s = torch.cuda.current_stream().cuda_stream
    rgba8 = torch.from_numpy(np.random.default_rng(3 * h + w).integers(0, 256, (h, w, 4), dtype=np.uint8)).to(DEV)
    want, dim = rgl.texture_from_rgba8(rgba8, premultiply=pm)
    base, _ = rgl.texture_from_rgba8(rgba8, premultiply=pm, mip=False)
    f = torch.empty((h, w, 4), dtype=torch.float32, device=DEV)
    assert L.rgl_texture_from_rgba8(rgba8.data_ptr(), w, h, int(pm), f.data_ptr(), s) == 0
    sq = f
    if (w, h) != (dim, dim):
        sq = torch.empty((dim, dim, 4), dtype=torch.float32, device=DEV)
        assert L.rgl_texture_pow2(f.data_ptr(), w, h, sq.data_ptr(), dim, s) == 0
    assert torch.equal(sq.view(torch.int32), base.view(torch.int32))
    out = torch.zeros((2 * dim, dim, 4), dtype=torch.float32, device=DEV)
    out[:dim] = sq
    assert L.rgl_texture_mipmap(out.data_ptr(), dim, s) == 0
    assert torch.equal(out.view(torch.int32), want.view(torch.int32))
