"""Clipping at the sizes where the clip stage changes shape: one triangle, a full and an overfull workgroup (16 triangles
at a time), as many as share the binning's pass over the originals and one more (a sixth of a pass: 42 and 43 of 256),
thousands; opaque (two-phase raster), blended without depth writes (listed) and with them (ordered, where the
fans' order shows). Identical to the checker."""
import numpy as np
import pytest

import oracle
from softglrender_amd import scenes
from softglrender_amd import stream as S
from softglrender_amd.replay import replay, replay_batched, run_reads

from .util import assert_identical

pytestmark = pytest.mark.gpu


def _scene(n, mode, msaa, seed):
    rng = np.random.default_rng(seed)
    # every triangle has a vertex outside one or more planes; some leave the frustum altogether
    v = np.zeros((3 * n, 8), np.float32)
    p = rng.uniform(-1.6, 1.6, (n, 3, 3))
    p[:, 0, :2] = rng.uniform(-0.9, 0.9, (n, 2))
    k = rng.integers(0, 3, n)
    p[np.arange(n), 1, k] = rng.choice([-2.5, 2.5], n)
    p[:, :, 2] *= 0.7
    v[:, 0:3] = p.reshape(-1, 3)
    v[:, 4:8] = rng.uniform(0, 1, (3 * n, 4))
    st = S.Stream()
    st.vao(1, v, np.arange(3 * n, dtype=np.int32))
    st.texture(2, 90, 70, usage=S.USAGE_COLOR, msaa=msaa)
    st.tex_init(2)
    st.texture(3, 90, 70, format=S.FMT_FLOAT32, usage=S.USAGE_DEPTH, msaa=msaa)
    st.tex_init(3)
    st.fbo(1, color=2, depth=3)
    st.frame()
    st.begin(1, True, True, (0.1, 0.2, 0.3, 1.0), 1.0)
    st.viewport(0, 0, 90, 70)
    rs = S.RenderStates(depth_test=True, depth_func=S.DEPTH_LESS, blend=mode != "opaque", depth_mask=mode != "listed")
    rs.set_blend_factor(S.BF_SRC_ALPHA, S.BF_ONE_MINUS_SRC_ALPHA)
    st.draw(1, S.SHADING_VERTEX_COLOR, 0, rs, S.uniforms_model(np.eye(4), np.eye(4)), bytes(64), bytes(48))
    st.end()
    st.read(2)
    st.read(3, which=1 if msaa else 0)
    return scenes.Scene(f"clip {n} {mode}", st, 90, 70, msaa)


@pytest.mark.parametrize("mode", ["opaque", "listed", "ordered"])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 42, 43, 257, 3000])
def test_clipped_triangles_match_checker(renderer, n, mode):
    print(f"[gpu] clip {n} {mode}", flush=True)
    sc = _scene(n, mode, n % 2 == 0, 5 + n)
    got, _ = replay(renderer, sc.stream.bytes())
    out, _ = oracle.cpu_ref_replay(sc.stream.bytes(), sc.stream.output_bytes(), exact_math=False)
    assert_identical(got, sc.stream.split_outputs(out), sc.name)


def test_clipped_triangles_in_a_batch_match_checker(renderer):
    """Views of 1 to 3,000 triangles that clip, each into its own targets, replayed twice."""
    print("[gpu] clip, batched", flush=True)
    sizes = (1, 17, 42, 43, 300, 3000)
    st = S.Stream()
    for k, n in enumerate(sizes):
        rng = np.random.default_rng(50 + n)
        v = np.zeros((3 * n, 8), np.float32)
        p = rng.uniform(-1.6, 1.6, (n, 3, 3))
        p[:, 0, :2] = rng.uniform(-0.9, 0.9, (n, 2))
        p[:, 1, 0] = 2.5
        p[:, :, 2] *= 0.7
        v[:, 0:3] = p.reshape(-1, 3)
        v[:, 4:8] = rng.uniform(0, 1, (3 * n, 4))
        st.vao(1 + k, v, np.arange(3 * n, dtype=np.int32))
        st.texture(10 + 2 * k, 90, 70, usage=S.USAGE_COLOR)
        st.tex_init(10 + 2 * k)
        st.texture(11 + 2 * k, 90, 70, format=S.FMT_FLOAT32, usage=S.USAGE_DEPTH)
        st.tex_init(11 + 2 * k)
        st.fbo(1 + k, color=10 + 2 * k, depth=11 + 2 * k)
    st.frame()
    for k in range(len(sizes)):
        st.begin(1 + k, True, True, (0.1, 0.2, 0.3, 1.0), 1.0)
        st.viewport(0, 0, 90, 70)
        st.draw(1 + k, S.SHADING_VERTEX_COLOR, 0, scenes._common_states(S.DEPTH_LESS),
                S.uniforms_model(np.eye(4), np.eye(4)), bytes(64), bytes(48))
        st.end()
    for k in range(len(sizes)):
        st.read(10 + 2 * k)
        st.read(11 + 2 * k)
    out, _ = oracle.cpu_ref_replay(st.bytes(), st.output_bytes(), exact_math=False)
    want = st.split_outputs(out)
    rp, b, reads = replay_batched(renderer, st.bytes())
    for _ in range(2):
        b.run()
        assert_identical(run_reads(rp, reads), want, "clipped batch")
    b.destroy()
