"""Renders and builds on a card with little memory left, and what their
objects give back. The samples a render keeps before they go to the film
(csrc/batch.hip) are optional, and up to 2 GB of them outlive the render; an
object that is built again keeps its workspace, up to 2 GiB, and arrays of up to
twice the size (csrc/accel.hip). Whatever is launched here has at least half a
GB of the card free (the runtime backs the private memory of a traversal kernel
with 160 MB when it first runs on a queue)."""
import contextlib

import pytest

from lm_amd import scenes
from lm_amd.accel import Accel
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


def _triangles(n, device, seed):
    import torch
    g = torch.Generator(device=device).manual_seed(seed)
    c = torch.rand(n, 1, 3, generator=g, device=device) * 10
    v = torch.rand(n, 3, 3, generator=g, device=device)
    return v.sub_(0.5).mul_(10 / n ** (1 / 3)).add_(c).view(n, 9)


def _rays(v, device):
    """Rays at the centroids of some of the triangles, from outside."""
    import torch
    c = v[:: v.shape[0] // 1000].view(-1, 3, 3).mean(1)
    o = torch.tensor([5.0, 5.0, 40.0], device=device).expand_as(c)
    d = torch.nn.functional.normalize(c - o, dim=1)
    r = torch.empty(c.shape[0], 8, device=device)
    r[:, 0:3], r[:, 3], r[:, 4:7], r[:, 7] = o, 1e-3, d, 1e10
    return r


def _taken(before):
    return before - _free()


def test_build_workspace_given_back(device):
    """One build on an object that holds a deserialized tree is its first:
    what it holds afterwards is what any object holds after its first build.
    (The workspace of 1M triangles is 176 MB.)"""
    v = _triangles(1000000, device, 1)
    start = _free()
    a = Accel(4)
    a.build(v)
    first = _taken(start)
    blob = a.serialize()
    del a
    start = _free()
    b = Accel(4)
    b.deserialize(blob)
    b.build(v)
    assert abs(_taken(start) - first) < (32 << 20)


def test_build_workspace_kept_is_bounded(device):
    """Built again, an object keeps a workspace of up to 2 GiB: 176 MB for 1M
    triangles, none for 13M (2.3 GB)."""
    for n, kept in ((1000000, True), (13000000, False)):
        v = _triangles(n, device, 2)
        start = _free()
        a = Accel(4)
        a.build(v)
        first = _taken(start)
        a.build(v)
        more = _taken(start) - first
        assert more > (150 << 20) if kept else more < (64 << 20)
        del a


def test_build_frees_what_it_keeps_for_want_of_memory(device):
    """A tree of 24M triangles holds 5 GB of arrays, which a build of 14M
    reuses beside a workspace of 2.5 GB; with 1.2 GB left it can only start
    anew (5.5 GB)."""
    import torch
    big = _triangles(24000000, device, 3)
    small = big[:14000000]
    a = Accel(4)
    a.build(big)
    with _left(1000 << 20):
        a.build(small)
    assert a.info()['num_tris'] == small.shape[0]
    fresh = Accel(4)
    fresh.build(small)
    rays = _rays(small, device)
    hits = []
    for acc in (a, fresh):
        hits.append(torch.zeros((rays.shape[0], 4), dtype=torch.float32, device=device))
        acc.intersect_device(rays, hits[-1])
    assert torch.equal(hits[0].view(torch.int32), hits[1].view(torch.int32))
    assert (hits[0][:, 0].view(torch.int32) >= 0).all()
