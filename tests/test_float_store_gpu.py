"""GPU parity of the float colour stores (full, downsampled, quad canvas)
under each colour attachment and of the Kawase blur pass: bit for bit
against the oracle."""
import numpy as np
import pytest
import torch

import float_store_scenes as F
from test_inorder_gpu import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("build", F.ALL, ids=lambda f: f().name)
def test_float_store_scene_matches_oracle(build):
    ref, rst, gst = _check(build())
    assert rst["fragments"] > 1000


@pytest.mark.parametrize("h,w", [(360, 640), (23, 37), (7, 5)])
def test_kawase_passes_match_oracle(h, w):
    from oracle_backend import lib as olib
    from rsr_amd import rgl
    L = olib()
    rng = np.random.default_rng(h * 1000 + w)
    img = rng.uniform(0, 1, (h, w, 4)).astype(np.float32)
    src = torch.from_numpy(img).cuda()
    cur = img
    for d in (0, 1, 2, 2, 3):   # a glow chain's distances
        print(f"[kawase {w}x{h} d={d}]", flush=True)
        dst = torch.full_like(src, float("nan"))
        rgl.kawase_blur(src, dst, d)
        torch.cuda.synchronize()
        want = np.full_like(cur, np.nan)
        L.rglo_kawase_blur(np.ascontiguousarray(cur).ctypes.data, want.ctypes.data, w, h, w, w, d)
        got = dst.cpu().numpy()
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), d
        src, cur = dst, want


@pytest.mark.parametrize("h,w", [(1, 1), (16, 32), (17, 33), (47, 65)])
@pytest.mark.parametrize("d", [0, 1, 4, 5, 6, 40])
def test_kawase_tiles_match_oracle(h, w, d):
    # tiles of 32 x 16 pixels up to d = 5, a thread per pixel beyond; rows
    # wider than the canvas; infinities and NaN where they land
    from oracle_backend import lib as olib
    from rsr_amd import rgl
    rng = np.random.default_rng(100 * h + d)
    img = rng.uniform(-1, 1, (h, w, 4)).astype(np.float32)
    img[h // 2, w // 2] = (np.inf, -0.0, 3e38, 1e-45)
    wide = torch.full((h, w + 3, 4), 7.0, device="cuda")
    src, dst = wide.clone(), wide.clone()
    src[:, :w] = torch.from_numpy(img).cuda()
    rgl.kawase_blur(src[:, :w], dst[:, :w], d)
    torch.cuda.synchronize()
    want = np.full_like(img, 5.0)
    olib().rglo_kawase_blur(img.ctypes.data, want.ctypes.data, w, h, w, w, d)
    got = dst.cpu().numpy()
    assert np.array_equal(got[:, :w].view(np.uint32), want.view(np.uint32))
    assert (got[:, w:] == 7.0).all()
