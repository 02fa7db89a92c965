"""Batches of 4 Mi pixels and more, where tiles without records get no keys
and resolve to the clear values: every post program, both encodings, clear
values of their own, stores left out, outputs and rows that take no 16-byte
stores, tiles that are no power of two and frames drawn in order beside them.
Every frame is drawn twice, its geometry moved in between, against the oracle
bit for bit: the first frame's keys would show where the second has none."""
import numpy as np
import pytest
import torch

from rsr_amd import scenes

import inorder_scenes as S

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
CLEAR = (0.35, 2.5, -0.25)


def _frame(width, height, name, post=scenes.PGM_DEFAULT_POST, gamma=True, tile_blocks=(8, 8), inorder=False, eye=0.0, stores=(0, 1, 2),
           exposure=0.4):
    sc, pro, _ = S.base(width, height, tile_blocks, name=f"{name}_{width}x{height}_t{tile_blocks[0] * 8}x{tile_blocks[1] * 8}")
    sc.arrays["exposure"] = np.array([exposure] + [0.0] * 31, np.float32)
    pro = [("clear_color", *CLEAR) if c[0] == "clear_color" else ("clear_depth", 2.25) if c[0] == "clear_depth" else
           ("view_matrix", scenes.look_at((eye, 2.0, 30.0), (eye, 0.75, 0), (0, 1, 0))) if c[0] == "view_matrix" else c for c in pro]
    # a far, small sphere: most tiles are empty
    body = ([("enable", scenes.GL_BLEND)] if inorder else []) + S.lambert(sc) + S.draw(sc, "sphere")
    store = [("use_program", post)] + ([("alloc_uniforms", "@exposure")] if post == scenes.PGM_EXPOSURE_POST else [])
    store += [c for k, c in enumerate([("store_color_tc", ("out", 0), gamma), ("store_depth", ("out", 1)),
                                       ("store_primitive_id", ("out", 2))]) if k in stores]
    sc.calls = pro + [("clear", S.CB | S.DB)] + body + store
    sc.outputs = S.OUT3
    return sc


def _record(g, sc, dev, outs):
    ptr_of = {id(sc.arrays[k]): t.data_ptr() for k, t in dev.items()}
    scenes.render_calls(g, sc, [o.data_ptr() for o in outs], ptr=lambda a: ptr_of[id(a)])


def _check_batch(make, offsets):
    """Frames make(eye)[k], their outputs offsets[k] words past an aligned
    address, in one batch, with two eyes one after the other."""
    from oracle_backend import render_calls as oracle_calls
    from rsr_amd import rgl
    stream = torch.cuda.current_stream().cuda_stream
    recs = [rgl.GPU(0) for _ in offsets]
    ex = rgl.GPU(0)
    for eye in (-4.0, 5.0):
        scs = make(eye)
        assert sum(sc.width * sc.height for sc in scs) >= 4 << 20
        outs, keep = [], []
        for g, sc, off in zip(recs, scs, offsets):
            n = sc.width * sc.height
            host = [scenes.output_array(k, sc.width, sc.height).view(np.uint32) for k in sc.outputs]
            o = [torch.zeros(n + off, dtype=torch.int32, device=DEV)[off:] for _ in host]
            for t, h in zip(o, host):
                t.copy_(torch.from_numpy(h.view(np.int32).reshape(-1)))
            keep.append({k: torch.from_numpy(np.ascontiguousarray(a)).to(DEV) for k, a in sc.arrays.items()})
            _record(g, sc, keep[-1], o)
            outs.append(o)
        ex.run_batch_and_wait(recs, stream)
        for sc, o in zip(scs, outs):
            ref, rst = oracle_calls(sc, threads=8)
            assert rst["fragments"] > 100
            for k, (r, t) in enumerate(zip(ref, o)):
                got = t.cpu().numpy().view(np.uint32).reshape(r.shape)
                bad = np.argwhere(r.view(np.uint32) != got)
                assert bad.size == 0, f"{sc.name} eye {eye} output {k} differs at {bad[:4].tolist()}"
    ex.close()
    for g in recs:
        g.close()


def test_posts_and_encodings():
    P = scenes
    _check_batch(lambda eye: [_frame(1280, 720, "default", P.PGM_DEFAULT_POST, True, eye=eye),
                              _frame(1280, 720, "default_linear", P.PGM_DEFAULT_POST, False, eye=eye),
                              _frame(1280, 720, "exposure", P.PGM_EXPOSURE_POST, True, eye=eye),
                              _frame(1280, 720, "exposure_linear", P.PGM_EXPOSURE_POST, False, eye=eye, exposure=-3.0),
                              _frame(1280, 720, "iq", P.PGM_IQ_POST, True, eye=eye)], [0] * 5)


def test_rows_outputs_and_stores():
    _check_batch(lambda eye: [_frame(1281, 721, "odd", eye=eye), _frame(1278, 719, "even", gamma=False, eye=eye),
                              _frame(1280, 720, "offset", eye=eye), _frame(1280, 720, "no_depth", eye=eye, stores=(0, 2)),
                              _frame(1284, 720, "depth_only", eye=eye, stores=(1,))], [0, 0, 1, 2, 0])


def test_mixed_tiles_and_paths():
    _check_batch(lambda eye: [_frame(1280, 720, "t64", eye=eye), _frame(1280, 720, "t40x24", eye=eye, tile_blocks=(5, 3)),
                              _frame(1280, 720, "blended", eye=eye, inorder=True), _frame(1283, 717, "t16", eye=eye, tile_blocks=(2, 2)),
                              _frame(1280, 720, "t8", eye=eye, tile_blocks=(1, 1)),
                              _frame(640, 360, "t32x64", eye=eye, tile_blocks=(4, 8))], [0, 0, 0, 0, 0, 0])


def test_one_frame_alone():
    # a single frame's resolve grid is two-dimensional
    _check_batch(lambda eye: [_frame(2560, 1640, "alone", scenes.PGM_EXPOSURE_POST, False, eye=eye)], [0])
    _check_batch(lambda eye: [_frame(2563, 1641, "alone", eye=eye)], [3])
