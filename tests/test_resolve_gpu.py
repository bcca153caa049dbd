"""Finished samples of a single scene's render, kept by work item and
resolved into the film at the end of a run (csrc/batch.hip, k_b_resolve), or
added to the film as they finish when a guide trains over more samples than a
run keeps (renders without room for their samples: test_memory_gpu.py)."""
import numpy as np
import pytest

from lm_amd import scenes
from lm_amd.guide import Guide
from lm_amd.renderer import GpuScene

pytestmark = pytest.mark.gpu

KEPT = 1 << 27   # samples kept per run (LMGPU_REGEN_SAMPLES)


def _room(w, h):
    room = scenes.box_room(open_front=False)
    prim = scenes.Primitive(room, scenes.Material(scenes.MAT_DIFFUSE, (0.5, 0.6, 0.7)), Ke=(1.0, 0.5, 0.25))
    cam = scenes.Camera((0, 0, 0.5), (0, 0, -1), (0, 1, 0), 60.0, w / h)
    return GpuScene(scenes.Scene([prim], cam, None, w, h).flatten(), width=4)


@pytest.mark.parametrize('w,h,spp,parts', [(7, 5, 3, [1, 2]), (61, 43, 9, [2, 2, 5]), (300, 200, 16, [15, 1]),
                                           # more samples than one run keeps (128 per pixel): two runs of
                                           # 97, and runs of 86, 86 and 85 against 100 and runs of 79 and 78
                                           (1024, 1024, 194, [100, 94]), (1024, 1024, 257, [100, 157])])
@pytest.mark.parametrize('sumsq', [True, False])
def test_samples_resolve_to_their_sum(device, w, h, spp, parts, sumsq):
    """One render equals the sum of renders of its parts (the same samples),
    added to what the film held. All terms are non-negative, so a sum of spp
    of them in any order is within spp * 2^-53 of itself, relatively."""
    import torch
    assert (w * h * spp > KEPT) == (w == 1024)
    sc = _room(w, h)
    films = []
    for split in ([spp], parts):
        s = torch.full((h, w, 3), 0.5, dtype=torch.float64, device='cuda')
        q = torch.full((h, w, 3), 0.25, dtype=torch.float64, device='cuda') if sumsq else None
        at = 3
        rays = 0
        for k in split:
            st = sc.render_raw(spp=k, max_verts=4, seed=11, sample_offset=at, film_sum=s, film_sumsq=q)[2]
            at += k
            rays += st['extension_rays'] + st['shadow_rays']
        films.append((s.cpu().numpy(), q.cpu().numpy() if sumsq else None, rays))
    (s0, q0, r0), (s1, q1, r1) = films
    tol = 4 * spp * 2.0 ** -53
    assert r0 == r1
    assert s0.min() > 0.5
    np.testing.assert_allclose(s0, s1, rtol=tol, atol=0)
    if sumsq:
        np.testing.assert_allclose(q0, q1, rtol=tol, atol=0)
        # squares of the same samples: n * sum of squares >= square of the sum
        assert (spp * (q0 - 0.25) >= (s0 - 0.5) ** 2 * (1 - 1e-12)).all()


@pytest.mark.parametrize('spp', [128, 129])
def test_training_guide_around_the_kept_samples(device, spp):
    """A guide that trains over as many samples as one run keeps (resolved at
    its end) and over more (added to the film as they finish): the closed
    room's E[L] = Ke sum_k rho^k, within 5 standard errors."""
    import torch
    w = h = 1024
    assert (w * h * spp > KEPT) == (spp == 129)
    sc = _room(w, h)
    lo, hi = sc.bounds()
    s = torch.zeros((h, w, 3), dtype=torch.float64, device='cuda')
    q = torch.zeros_like(s)
    verts = 4
    st = sc.render_raw(spp=spp, max_verts=verts, seed=11, film_sum=s, film_sumsq=q,
                       guide=Guide(lo - 1e-3, hi + 1e-3, seed=2), guide_opts=dict(steps_per_pass=1, batch=4096))[2]
    n = w * h * spp
    assert st['samples'] == n and st['guide_records'] > 0
    for c, (rho, ke) in enumerate(((0.5, 1.0), (0.6, 0.5), (0.7, 0.25))):
        mean = float(s[..., c].sum()) / n
        var = float(q[..., c].sum()) / n - mean ** 2
        assert abs(mean - ke * sum(rho ** k for k in range(verts - 1))) < 5 * (var / n) ** 0.5
