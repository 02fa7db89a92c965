"""The recorder's gl_ methods, made once per name, call the library of the
object they are called on, as the methods made per call did."""
import types

import numpy as np
import pytest


def _recorder(tag, log):
    from rsr_amd import rgl
    g = rgl.GPU.__new__(rgl.GPU)
    g.h, g._keep = None, []
    g.L = types.SimpleNamespace(rgl_gl_clear=lambda h, bits: log.append((tag, bits)) or 0,
                                rgl_gl_view_matrix=lambda h, p: log.append((tag, type(p).__name__)) or 0,
                                rgl_gl_cull_face=lambda h, v: -1,
                                rgl_gpu_last_error=lambda h: tag.encode())
    return g


def test_each_object_calls_its_own_library():
    from rsr_amd import rgl
    log = []
    a, b = _recorder("a", log), _recorder("b", log)
    for g in (a, b, a):
        g.gl_clear(3)
        g.gl_clear(True)
        g.gl_view_matrix(np.eye(4))
    assert log == [(t, x) for t in "aba" for x in (3, 1, "int")]
    for g, tag in ((a, "a"), (b, "b")):
        with pytest.raises(rgl.RglError, match=f"^{tag} "):
            g.gl_cull_face(1)
        with pytest.raises(AttributeError):
            g.gl_no_such_call
