"""rhip_draw_noalloc (the draw whose arena is the library's static scratch)
against rhip_draw, through the C-ABI: identical outputs on two no-allocation
calls in a row, the second with a smaller input, and a clear refusal of a
draw that does not fit the scratch."""
import ctypes

import numpy as np
import pytest

from softglrender_amd import _lib, scenes
from softglrender_amd import stream as S
from softglrender_amd.renderer import RendererHIP
from softglrender_amd.replay import replay

pytestmark = pytest.mark.gpu


def _run(renderer, sc, no_alloc):
    renderer.no_alloc = no_alloc
    try:
        outs, _ = replay(renderer, sc.stream.bytes(), layouts=sc.meta.get("layouts"))
    finally:
        renderer.no_alloc = False
    return outs


def _assert_identical(got, want, label):
    assert len(got) == len(want), label
    for i, (g, w) in enumerate(zip(got, want)):
        assert g.shape == w.shape, (label, i, g.shape, w.shape)
        bad = int((g.view(np.uint8) != w.view(np.uint8)).sum())
        assert bad == 0, f"{label}: output {i} differs in {bad} bytes"


def test_no_alloc_draw_equals_draw_on_two_calls(renderer):
    # first a 640x480 4x-MSAA frame of 4,096 triangles, then a smaller 160x120
    # frame whose triangles clip: the second runs on what the first left behind
    big = scenes.scene_c1(msaa=True, read_msaa=True)
    small = scenes.scene_variant("msaa_clip")
    print("[gpu] no-alloc: reference draws", flush=True)
    want_big = _run(renderer, big, False)
    want_small = _run(renderer, small, False)
    print("[gpu] no-alloc: c1_msaa through rhip_draw_noalloc", flush=True)
    got_big = _run(renderer, big, True)
    print("[gpu] no-alloc: msaa_clip through rhip_draw_noalloc", flush=True)
    got_small = _run(renderer, small, True)
    _assert_identical(got_big, want_big, "c1_msaa")
    _assert_identical(got_small, want_small, "msaa_clip")
    assert int((want_big[0][..., 3] > 0).sum()) > 60000


def test_no_alloc_draw_refuses_what_does_not_fit(renderer):
    # a 1080p 4x-MSAA target needs 66 MB of fragment jobs alone, beyond the 64 MiB scratch
    sc = scenes.scene_c1(width=1920, height=1080, msaa=True, lon=8, lat=4)
    assert _lib.load().rhip_draw_noalloc_capacity() == 64 << 20
    with pytest.raises(_lib.RhipError) as e:
        _run(renderer, sc, True)
    assert e.value.code == -3 and "scratch" in str(e.value)


def _triangles(count, floats, size=64):
    """`count` times one triangle of vertices of `floats` floats, base colour shader, opaque."""
    st = S.Stream()
    v = np.zeros((3, floats), np.float32)
    v[:, :3] = [[-0.5, -0.5, 0.5], [0.5, -0.5, 0.5], [0, 0.5, 0.5]]
    st.vao(1, v, np.tile(np.arange(3, dtype=np.int32), count))
    st.texture(2, size, size, usage=S.USAGE_COLOR)
    st.tex_init(2)
    st.texture(3, size, size, format=S.FMT_FLOAT32, usage=S.USAGE_DEPTH)
    st.tex_init(3)
    st.fbo(1, color=2, depth=3)
    st.frame()
    st.begin(1, True, True, (0, 0, 0, 0), 1.0)
    st.viewport(0, 0, size, size)
    st.draw(1, S.SHADING_BASIC, 0, scenes._common_states(S.DEPTH_LESS), S.uniforms_model(np.eye(4), np.eye(4)),
            bytes(S.SCENE_BYTES), S.uniforms_material(0, 0, 0, 1.0, 0.5, (1, 1, 1, 1)))
    st.end()
    st.read(2)
    return scenes.Scene("triangles", st, size, size, False, {})


@pytest.mark.parametrize("floats,most", [(4, 42128), (16, 30935)])
def test_no_alloc_limit_is_where_it_was(renderer, floats, most):
    print(f"[gpu] no-alloc limit, {floats} floats a vertex", flush=True)
    got = _run(renderer, _triangles(most, floats), True)
    _assert_identical(got, _run(renderer, _triangles(1, floats), False), "one triangle many times")
    with pytest.raises(_lib.RhipError) as e:
        _run(renderer, _triangles(most + 1, floats), True)
    assert e.value.code == -3 and "scratch" in str(e.value)


def _free_memory():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert _lib.load().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0  # librhip's own HIP runtime
    return free.value


def test_draw_memory_does_not_depend_on_the_vertex_size():
    """What a draw takes besides its buffers: no stage keeps raw vertices, so 64-byte vertices need no more than
    16-byte ones (their 12 clip vertices a triangle would be 230 MB of 400,000 triangles, and a quarter for growth)."""
    count, used = 400_000, []
    for floats in (4, 16):
        print(f"[gpu] memory of a draw, {floats} floats a vertex", flush=True)
        r = RendererHIP(0)
        r.create()
        replay(r, _triangles(1, floats).stream.bytes())
        before = _free_memory()
        outs, _ = replay(r, _triangles(count, floats).stream.bytes())
        used.append(before - _free_memory())
        assert outs[0].any()
        r.destroy()
    assert used[0] > 200 << 20, used
    assert abs(used[1] - used[0]) < 64 << 20, used
