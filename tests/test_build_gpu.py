"""Device BVH build: the refit's blocks, the collapse's levels and the
quantised copy at the edges of their tiles (csrc/accel.hip)."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SPAN = 1024   # leaves per refit block (kRefitSmall)
LARGE = 400000   # from here on, blocks of 4096 leaves (kRefitLargeFrom)


def _mesh(n, kind):
    rng = np.random.default_rng(n)
    c = rng.random((n, 1, 3)) * 10
    v = (c + (rng.random((n, 3, 3)) - 0.5) * (10 / n ** (1 / 3))).astype(np.float32).reshape(n, 9)
    if kind == 'equal':      # one Morton code for half of them: long chains of ties
        v[: n // 2] = v[0]
    elif kind == 'line':     # deep, uneven trees
        v = np.float32(v * 0.01 + np.exp2(-30 * rng.random((n, 1))))
    return np.ascontiguousarray(v, np.float32)


def _arrays(blob, width):
    b = np.frombuffer(blob, np.uint8)
    nt, nn, leaves = np.frombuffer(b[24:48].tobytes(), np.int64)
    nodes = b[128:128 + nn * 32 * width].view(np.float32).reshape(nn, 8, width)
    tris = b[128 + nn * 32 * width:].view(np.float32).reshape(nt, 3, 4)
    return nodes, tris, int(leaves)


@pytest.mark.parametrize('n,kind', [(1, ''), (2, ''), (SPAN - 1, ''), (SPAN, ''), (SPAN + 1, ''), (SPAN + 2, 'equal'),
                                    (2 * SPAN + 1, 'line'), (5 * SPAN, 'equal'), (40 * SPAN + 3, ''),
                                    (70 * SPAN + 511, 'line'), (LARGE - 1, 'line'), (LARGE, 'equal'),
                                    (LARGE + 4096 - LARGE % 4096 + 1, '')])
@pytest.mark.parametrize('width,collapse,builder', [(2, 0, 1), (4, 0, 1), (8, 0, 1), (4, 1, 1), (8, 0, 0)])
def test_built_bounds_and_counts(n, kind, width, collapse, builder):
    """Every child box is the exact FP32 bound of the triangles below it (a
    minimum and a maximum round nothing: no tolerance), every triangle is in
    one leaf, and the counts and the depth are those of the tree."""
    from lm_amd.accel import Accel
    verts = _mesh(n, kind)
    acc = Accel(width, collapse=collapse, builder=builder)
    acc.build(verts)
    info = acc.info()
    nodes, tris, leaves = _arrays(acc.serialize(), width)
    child = nodes[:, 6].view(np.int32)
    count = nodes[:, 7].view(np.int32)
    order = tris[:, 0, 3].copy().view(np.int32)
    assert np.array_equal(np.sort(order), np.arange(n))
    assert np.array_equal(tris[:, :, :3].reshape(n, 9), verts[order])
    assert len(nodes) == info['num_nodes'] and leaves == info['num_leaves'] == int((count > 0).sum())
    lo, hi = tris[:, :, :3].min(1), tris[:, :, :3].max(1)
    seen = np.zeros(n, np.int32)
    box = np.empty((len(nodes), 2, 3), np.float32)
    levels = [np.zeros(1, np.int64)]
    while True:
        below = child[levels[-1]][count[levels[-1]] == 0].astype(np.int64)
        if len(below) == 0:
            break
        levels.append(below)
    assert len(levels) == info['depth']
    assert np.array_equal(np.sort(np.concatenate(levels)), np.arange(len(nodes)))
    for level in reversed(levels):
        got_lo, got_hi = nodes[level, :3].transpose(0, 2, 1), nodes[level, 3:6].transpose(0, 2, 1)   # [node, child, axis]
        ch, ct = child[level], count[level]
        want = np.empty((2,) + got_lo.shape, np.float32)
        want[0], want[1] = np.inf, -np.inf
        inner = ct == 0
        want[0][inner], want[1][inner] = box[ch[inner], 0], box[ch[inner], 1]
        for k in range(ct.max()):
            m = ct > k
            at = ch[m] + k
            want[0][m] = np.minimum(want[0][m], lo[at])
            want[1][m] = np.maximum(want[1][m], hi[at])
            np.add.at(seen, at, 1)
        used = ct >= 0
        assert np.array_equal(got_lo[used], want[0][used]) and np.array_equal(got_hi[used], want[1][used])
        box[level, 0], box[level, 1] = want[0].min(1), want[1].max(1)
    assert (seen == 1).all()
    # the same triangles again, and half of them, into the same object
    acc.build(verts)
    assert acc.info()['num_nodes'] == len(nodes)
    half = max(1, n // 2)
    acc.build(verts[:half])
    assert acc.info()['num_tris'] == half
    assert np.array_equal(np.sort(_arrays(acc.serialize(), width)[1][:, 0, 3].copy().view(np.int32)), np.arange(half))


def _quantised(nodes, width):
    """QNode<width> words of WNode<width> arrays ([n, 8, width] float32; csrc/bvh.h, quantise_node). Sums of a plane
    number times a power of two and an FP32 origin are exact in FP64, so their FP32 rounding is the fma's."""
    n = len(nodes)
    count, child = nodes[:, 7].view(np.int32).astype(np.int64), nodes[:, 6].view(np.int32).astype(np.int64)
    present = count >= 0
    out = np.zeros((n, 4 * width), np.uint32)
    for a in range(3):
        lo, hi = nodes[:, a].astype(np.float64), nodes[:, 3 + a].astype(np.float64)
        mn = np.where(present, lo, np.inf).min(1)
        mx = np.where(present, hi, -np.inf).max(1)
        m, k = np.frexp((mx - mn) / 255.0)
        e = np.where(mx > mn, np.maximum(np.where(m == 0.5, k - 1, k), -126), -126)
        plane = lambda q, e: (q * np.exp2(e.astype(np.float64)) + mn).astype(np.float32)   # noqa: E731
        while True:
            grow = (plane(255.0, e) < mx) & (e < 127)
            if not grow.any():
                break
            e = e + grow
        out[:, a] = mn.astype(np.float32).view(np.uint32)
        out[:, 3] |= (e & 0xff).astype(np.uint32) << np.uint32(8 * a)
        for c in range(width):
            step = np.exp2(e.astype(np.float64))
            ql = np.clip(np.floor((lo[:, c] - mn) / step), 0, 255)
            qh = np.clip(np.ceil((hi[:, c] - mn) / step), 0, 255)
            while True:
                down = (plane(ql, e) > lo[:, c]) & (ql > 0) & present[:, c]
                up = (plane(qh, e) < hi[:, c]) & (qh < 255) & present[:, c]
                if not (down.any() or up.any()):
                    break
                ql, qh = ql - down, qh + up
            at, sh = 4 + a * (width // 4) + c // 4, np.uint32(8 * (c % 4))
            out[:, at] |= np.where(present[:, c], ql, 0).astype(np.uint32) << sh
            out[:, at + 3 * (width // 4)] |= np.where(present[:, c], qh, 0).astype(np.uint32) << sh
    leaf = -((child << 4) | count) - 1
    ent = np.where(count < 0, -1, np.where(count == 0, child, leaf))
    first = 4 + 6 * (width // 4)
    out[:, first:first + width] = ent.astype(np.int32).view(np.uint32)
    return out, first + width


@pytest.mark.parametrize('width', [4, 8])
@pytest.mark.parametrize('n', [1, 15, 16, 17, 63, 64, 65, 1000])
def test_quantised_copy(device, width, n):
    """k_quantise, word for word, at node counts around its waves (16 nodes)
    and blocks (64): partly empty nodes, flat boxes, several scales."""
    import torch
    from lm_amd import _lib
    rng = np.random.default_rng([n, width])
    nodes = np.empty((n, 8, width), np.float32)
    extent = 10.0 ** rng.uniform(-5, 3, (n, 1, 1))
    lo = (rng.uniform(-1, 1, (n, 3, 1)) * 10 + rng.random((n, 3, width)) * extent).astype(np.float32)
    flat = rng.random((n, 3, width)) < 0.1
    hi = np.maximum(lo, (lo + rng.random((n, 3, width)) * extent * ~flat).astype(np.float32))
    used = np.arange(width) < rng.integers(1, width + 1, (n, 1))
    nodes[:, :3] = np.where(used[:, None], lo, np.float32(1e30))
    nodes[:, 3:6] = np.where(used[:, None], hi, np.float32(-1e30))
    nodes[:, 6] = np.where(used, rng.integers(0, 1 << 20, (n, width)), 0).astype(np.int32).view(np.float32)
    nodes[:, 7] = np.where(used, rng.integers(0, 16, (n, width)), -1).astype(np.int32).view(np.float32)
    words, held = _quantised(nodes, width)
    src = torch.from_numpy(nodes.view(np.int32).copy()).to(device)
    dst = torch.full((n + 1, 4 * width), 77, dtype=torch.int32, device=device)
    # lmgpu::quantise_nodes(int, const float4*, float4*, int64_t, hipStream_t)
    fn = getattr(_lib.lib(), '_ZN5lmgpu14quantise_nodesEiPK15HIP_vector_typeIfLj4EEPS1_lP12ihipStream_t')
    fn.argtypes = [ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int64, ctypes.c_void_p]
    fn.restype = ctypes.c_int
    torch.cuda.synchronize()
    assert fn(width, src.data_ptr(), dst.data_ptr(), n, None) == 0
    torch.cuda.synchronize()
    got = dst.cpu().numpy().view(np.uint32)
    assert np.array_equal(got[:n, :held], words[:, :held])
    assert (got[n] == 77).all()
