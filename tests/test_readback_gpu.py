"""Read-back of images: every layout and size on either side of the read's pieces (1 MiB, a ring of 16, helper threads
above 2 MiB) gives back the bytes that were uploaded."""
import threading

import numpy as np
import pytest

from softglrender_amd import stream as S
from softglrender_amd.renderer import RendererHIP, TextureDesc

pytestmark = pytest.mark.gpu


def _image(w, h, seed):
    return np.random.default_rng(seed).integers(0, 256, (h, w, 4), dtype=np.uint8)


def _texture(r, img, layout):
    t = r.createTexture(TextureDesc(width=img.shape[1], height=img.shape[0], usage=S.USAGE_SAMPLER | S.USAGE_UPLOAD,
                                    layout=layout))
    t.setImageData([img])
    return t


@pytest.mark.parametrize("layout", [0, 1, 2])
@pytest.mark.parametrize("size", [(1, 1), (37, 51), (512, 512), (513, 513), (1024, 601), (2600, 1700)])
def test_read_returns_upload(renderer, size, layout):
    print(f"[gpu] read {size} layout {layout}", flush=True)
    img = _image(*size, 3)
    t = _texture(renderer, img, layout)
    for _ in range(2):
        assert np.array_equal(t.readImage(), img)


def test_reads_from_several_threads():
    """Three devices read images of 34 pieces at once: one has the helper threads, the others copy on their own, and all
    walk their ring twice."""
    print("[gpu] concurrent reads", flush=True)
    bad = []

    def work(k):
        r = RendererHIP(0)
        r.create()
        img = _image(2600, 3400 + k, k)
        t = _texture(r, img, 0)
        for _ in range(6):
            if not np.array_equal(t.readImage(), img):
                bad.append(k)
        del t
        r.destroy()

    threads = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
