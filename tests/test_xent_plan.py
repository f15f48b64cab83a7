"""How the fused cross-entropy cuts its work (msd_xent_plan) and the memory it asks for (CPU): the caller's
chunk bounds the workspace, whatever the library widens it to."""
import ctypes
import random

import pytest

from transformer_amd import _lib


def _up(x, m):
    return -(-x // m) * m


def plan(n, V, d, chunk):
    out = (ctypes.c_int32 * 8)()
    _lib.check(_lib.lib().msd_xent_plan(n, V, d, chunk, out), "msd_xent_plan")
    return list(out)


def scratch(n, V, d, chunk):
    """(bytes of the probability block and grad_h's partials, the room they are promised to keep to)."""
    cols, chunks, forward, _, _, _, splits, _ = plan(n, V, d, chunk)
    Np, Vp = _up(n, 256), _up(V, 256)
    c0 = min(_up(max(chunk, 1), 256), Vp)
    total = _lib.lib().msd_xent_workspace_bytes(n, V, d, chunk)
    partials = _up(Vp // forward * Np * 8, 256) + 2 * _up(4 * Np, 256)
    assert total >= partials + 2 * Np * cols + 4 * splits * n * d
    room = min(8, c0 // 128) * 2 * Np * c0 + 2 * (Vp + Np) * d + 4 * Np * d
    return total - partials, max(64 << 20, room)


CHUNKS = (1, 256, 384, 1000, 4096, 8192, 10 ** 6)


def test_the_chunk_bounds_the_workspace():
    r = random.Random(2)
    shapes = [(4096, 32000, 1024), (509, 32000, 768), (32768, 32000, 512), (20000, 7000, 128), (1, 77, 128)]
    shapes += [(int(2 ** r.uniform(0, 15)), int(2 ** r.uniform(1, 16)), 128 * r.randint(1, 16)) for _ in range(400)]
    for n, V, d in shapes:
        for chunk in CHUNKS:
            used, room = scratch(n, V, d, chunk)
            assert used <= room + 512, (n, V, d, chunk, used, room)


def test_a_small_chunk_holds_less_than_a_large_one():
    """4096 rows of the 306M output layer: a caller who needs the memory gets it back."""
    sizes = [_lib.lib().msd_xent_workspace_bytes(4096, 32000, 1024, c) for c in (256, 1024, 4096)]
    assert sizes[0] < 100e6 and sizes == sorted(sizes) and sizes[0] < sizes[2] / 3


@pytest.mark.parametrize("n,V,d", [(4096, 32000, 1024), (300, 1000, 256), (20000, 7000, 128), (65, 257, 128)])
def test_chunks_cover_the_vocabulary(n, V, d):
    for chunk in CHUNKS:
        cols, chunks, *tiles, first, last = plan(n, V, d, chunk)
        assert cols % 256 == 0 and (chunks - 1) * cols < V <= chunks * cols
        assert set(tiles) <= {128, 256} and 1 <= last <= first
