"""Renders on a card with little memory left, and what a scene gives back:
the samples a render keeps before they go to the film (csrc/batch.hip) are
optional, and up to 2 GB of them outlive the render. Whatever is launched here
has at least half a GB of the card free (the runtime backs the private memory
of a traversal kernel with 160 MB when it first runs on a queue)."""
import contextlib

import pytest

from lm_amd import scenes
from lm_amd.renderer import GpuScene

pytestmark = pytest.mark.gpu

SAMPLES = 1 << 27     # of a render: 2 GiB kept
KEPT = 16 * SAMPLES
GIB = 1 << 30
SMALL = (512, 512)    # a pool of 2^21 path slots: 0.46 GB
LARGE = (4096, 2048)  # one-sample passes take 1.7 GB


def _scene(size):
    w, h = size
    room = scenes.box_room(open_front=False)
    prim = scenes.Primitive(room, scenes.Material(scenes.MAT_DIFFUSE, (0.5, 0.6, 0.7)), Ke=(1.0, 0.5, 0.25))
    cam = scenes.Camera((0, 0, 0.5), (0, 0, -1), (0, 1, 0), 60.0, w / h)
    return GpuScene(scenes.Scene([prim], cam, None, w, h).flatten(), width=4)


def _film(size, device):
    import torch
    return torch.zeros((size[1], size[0], 3), dtype=torch.float64, device=device)


def _free():
    import torch
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    return torch.cuda.mem_get_info()[0]


@contextlib.contextmanager
def _left(room):
    """The card's free memory taken but for `room` bytes and some 200 MB."""
    import torch
    hold = []
    try:
        while True:
            over = _free() - room
            if over < (20 << 20):
                break
            hold.append(torch.empty(min(over, 16 * GIB) & -(1 << 21), dtype=torch.uint8, device='cuda'))
        yield
    finally:
        hold.clear()
        torch.cuda.empty_cache()


def _render(sc, spp, film):
    film.zero_()
    return sc.render_raw(spp=spp, max_verts=4, seed=11, film_sum=film)[2]


def test_render_without_room_for_its_samples(device):
    """Room for the kept samples or for the path pool, not for both: the pool
    comes first and finished samples are added to the film one by one. The sum
    of the same non-negative terms in another order differs by their number
    times 2^-53 of itself at most, on each side."""
    spp = SAMPLES // (SMALL[0] * SMALL[1])
    film = _film(SMALL, device)
    st = _render(_scene(SMALL), spp, film)
    ref = film.clone()
    sc = _scene(SMALL)
    with _left(KEPT + (50 << 20)):
        st1 = _render(sc, spp, film)
    assert st1['extension_rays'] == st['extension_rays'] and st1['shadow_rays'] == st['shadow_rays']
    assert ((film - ref).abs() <= 4 * spp * 2.0 ** -53 * ref).all()


@pytest.mark.parametrize('call', ['pt', 'bdpt'])
def test_kept_samples_give_way(device, call):
    """A scene that holds the samples of a long render, and no memory left for
    the buffers of the next call: the samples are given back for them."""
    film = _film(LARGE, device)
    npix = LARGE[0] * LARGE[1]

    def go(sc):
        film.zero_()
        if call == 'bdpt':
            sc.render_bdpt(num_samples=1 << 18, max_verts=3, seed=3, film=film)
        else:
            sc.render_raw(spp=1, max_verts=4, seed=3, film_sum=film)
        return film

    ref = go(_scene(LARGE)).clone()
    sc = _scene(LARGE)
    _render(sc, SAMPLES // npix, film)
    with _left(500 << 20):
        got = go(sc)
    # FP64 sums of a few FP32 terms, in another order
    assert ((got - ref).abs() <= 1e-12 * ref).all()


def test_short_render_gives_kept_samples_back(device):
    """A render of few samples keeps no buffer made for many."""
    film = _film(SMALL, device)
    sc = _scene(SMALL)
    _render(sc, SAMPLES // (SMALL[0] * SMALL[1]), film)
    before = _free()
    _render(sc, 8, film)
    assert _free() - before > KEPT * 3 // 4
