"""Fused cross-entropy forward and backward on the GPU (msd_xent_forward / msd_xent_backward)
against the f64 oracle of model.py:281-361.

Inputs are bf16 (h like a final-norm output, weight like the tied embedding), so the oracle's
f64 arithmetic on the same values is the exact answer.  Tolerances: the loss to 1e-5 relative
(f32 sums of exact bf16 products); the gradients are bf16 outputs formed from a bf16 softmax
block, so each element within 2e-2 relative plus 2e-3 of the largest magnitude, and the whole
tensor within 5e-3 relative (Frobenius).
"""
import ctypes

import numpy as np
import pytest
import torch

from oracle import xent as ox
from transformer_amd import _lib
from transformer_amd.xent import fused_cross_entropy, fused_output_and_loss

pytestmark = pytest.mark.gpu


def _inputs(N, V, d, seed, h_scale=1.0):
    g = torch.Generator().manual_seed(seed)
    h = (torch.randn(N, d, generator=g) * h_scale).to(torch.bfloat16)
    w = (torch.randn(V, d, generator=g) * 0.02).to(torch.bfloat16)
    t = torch.randint(0, V, (N,), generator=g)
    return h, w, t


def _run(h, w, t, chunk, g=1.0):
    hd = h.cuda().requires_grad_()
    wd = w.cuda().requires_grad_()
    loss = fused_cross_entropy(hd, wd, t.cuda(), chunk)
    gh, gw = torch.autograd.grad(loss * g, (hd, wd))
    torch.cuda.synchronize()
    return float(loss), gh.float().cpu().numpy(), gw.float().cpu().numpy()


def _check(got, ref, what):
    err = np.abs(got - ref)
    tol = 2e-2 * np.abs(ref) + 2e-3 * np.abs(ref).max()
    assert np.all(err <= tol), (what, float(err.max()), float(np.abs(ref).max()))
    rel = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    assert rel < 5e-3, (what, rel)
    return rel


def _against_oracle(N, V, d, chunk, seed, h_scale=1.0, g=1.0):
    h, w, t = _inputs(N, V, d, seed, h_scale)
    loss, gh, gw = _run(h, w, t, chunk, g)
    hn, wn, tn = h.float().numpy(), w.float().numpy(), t.numpy()
    rloss = ox.chunked_ce_fwd(hn, wn, tn, 4096)
    rgh, rgw = ox.fused_ce_bwd(hn, wn, tn, g, 4096)
    assert abs(loss - rloss) <= 1e-5 * abs(rloss), (loss, rloss)
    r1 = _check(gh, rgh, "grad_h")
    r2 = _check(gw, rgw, "grad_weight")
    print(f"N={N} V={V} d={d} chunk={chunk}: loss {loss:.6f} (oracle {rloss:.6f}), "
          f"grad_h rel {r1:.2e}, grad_weight rel {r2:.2e}")


def _plan(N, V, d, chunk):
    """msd_xent_plan: ids per chunk, chunks, tiles of (forward, logits, grad_weight, grad_h), K splits of
    grad_h in the first and the last chunk."""
    out = (ctypes.c_int32 * 8)()
    _lib.check(_lib.lib().msd_xent_plan(N, V, d, chunk, out), "msd_xent_plan")
    return tuple(out)


def test_ragged_shapes_and_chunks():
    """Rows and vocabulary not multiples of the tiles; a single row."""
    _against_oracle(300, 1000, 256, 384, seed=1)
    _against_oracle(1, 77, 128, 4096, seed=2, g=0.5)


@pytest.mark.parametrize("N,V,d,chunk,plan", [
    # one row, one id past a tile; token padding to 64
    (65, 257, 128, 100, (512, 1, 128, 128, 128, 128, 1, 1)),
    # grad_h split over K with a short last split
    (129, 4001, 384, 1000, (4096, 1, 128, 128, 128, 128, 8, 8)),
    (1023, 16500, 256, 4096, (16640, 1, 128, 128, 128, 128, 29, 29)),
    # 256-tiles for the logits and grad_weight, ragged in tokens and vocabulary
    (1000, 13800, 1024, 4096, (13824, 1, 256, 256, 256, 128, 8, 8)),
    # two chunks, the last one short and with fewer splits
    (3158, 7206, 128, 100, (3840, 2, 128, 128, 128, 128, 7, 6)),
    # three chunks with 256-tiles for the logits and grad_h, one split fewer in the last
    (10506, 3087, 256, 256, (1280, 3, 128, 256, 128, 256, 2, 1)),
    # four chunks, 256-tiles for grad_h with a half-empty last column tile
    (4352, 30000, 640, 1000, (7680, 4, 256, 256, 128, 256, 5, 5)),
    (20000, 7000, 128, 256, (1024, 7, 256, 128, 128, 128, 2, 2)),
])
def test_tile_sizes_splits_and_chunks(N, V, d, chunk, plan):
    """Each tile size of each product, at ragged edges, over one and several chunks (tolerances as above)."""
    assert _plan(N, V, d, chunk) == plan
    _against_oracle(N, V, d, chunk, seed=8)


def test_peaked_logits():
    """Large logits (h scaled by 40: logit spread ~ 15): the logsumexp stays finite and exact."""
    _against_oracle(513, 3000, 384, 1024, seed=3, h_scale=40.0)


def test_306m_output_layer_4096_rows():
    """The 306M model's output layer on 4096 rows (N = 4096, V = 32000, d = 1024), chunk 4096."""
    _against_oracle(4096, 32000, 1024, 4096, seed=4)


def test_chunk_size_changes_only_the_grad_h_summation():
    """grad_weight and the loss are bitwise independent of the chunk size (every element is formed
    the same way); grad_h sums the chunks in f32 and agrees to rounding."""
    N, V, d, chunks = 8100, 8003, 128, (256, 1000, 100000)
    assert [_plan(N, V, d, c)[1] for c in chunks] == [3, 2, 1]
    h, w, t = _inputs(N, V, d, seed=5)
    a, b, c = (_run(h, w, t, c) for c in chunks)
    assert a[0] == b[0] == c[0]
    assert np.array_equal(a[2], b[2]) and np.array_equal(b[2], c[2])
    np.testing.assert_allclose(a[1], c[1], rtol=1e-2, atol=1e-3 * np.abs(c[1]).max())


def test_deterministic_and_3d_wrapper():
    h, w, t = _inputs(2 * 96, 2048, 128, seed=6)
    a = _run(h, w, t, 512)
    b = _run(h, w, t, 512)
    assert a[0] == b[0] and np.array_equal(a[1], b[1]) and np.array_equal(a[2], b[2])
    hd = h.cuda().reshape(2, 96, 128).requires_grad_()
    wd = w.cuda().requires_grad_()
    loss = fused_output_and_loss(hd, wd, t.cuda().reshape(2, 96), 512)
    gh, gw = torch.autograd.grad(loss, (hd, wd))
    assert float(loss) == a[0]
    assert np.array_equal(gh.reshape(-1, 128).float().cpu().numpy(), a[1])
    assert np.array_equal(gw.float().cpu().numpy(), a[2])


def test_operands_off_a_16_byte_boundary():
    """Slices of a flat buffer at any offset give the bits of aligned tensors."""
    h, w, t = _inputs(130, 700, 256, seed=9)
    want = _run(h, w, t, 512)
    for off in (1, 4):
        flat = torch.empty(off + h.numel() + w.numel(), dtype=torch.bfloat16, device="cuda")
        hd = flat[off:off + h.numel()].view_as(h).copy_(h.cuda()).requires_grad_()
        wd = flat[off + h.numel():].view_as(w).copy_(w.cuda()).requires_grad_()
        assert hd.data_ptr() % 16 and wd.data_ptr() % 16
        loss = fused_cross_entropy(hd, wd, t.cuda(), 512)
        gh, gw = torch.autograd.grad(loss, (hd, wd))
        assert float(loss) == want[0]
        assert np.array_equal(gh.float().cpu().numpy(), want[1]) and np.array_equal(gw.float().cpu().numpy(), want[2])


def _loss_and_grads(x, check):
    h, w, t = x
    loss = fused_cross_entropy(h, w, t, 512, check_targets=check)
    return (loss.detach(), *torch.autograd.grad(loss, (h, w)))


def _several_inputs(n):
    out = []
    for i in range(n):
        h, w, t = _inputs(200, 9000, 256, seed=20 + i)
        out.append((h.cuda().requires_grad_(), w.cuda().requires_grad_(), t.cuda()))
    return out


@pytest.mark.parametrize("check", [True, False])
def test_calls_on_several_streams_do_not_share_scratch(check):
    """Losses of one shape issued on two streams, nothing waited for between them: each has the bits of
    the same call alone."""
    xs = _several_inputs(2)
    alone = [_loss_and_grads(x, check) for x in xs]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in xs]
    for s in streams:
        s.wait_stream(torch.cuda.current_stream())
    got = [[] for _ in xs]
    for _ in range(8):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                got[i].append(_loss_and_grads(xs[i], check))
    torch.cuda.synchronize()
    for i, runs in enumerate(got):
        for r in runs:
            assert all(torch.equal(a, b) for a, b in zip(r, alone[i]))


def test_calls_from_several_threads_do_not_share_scratch():
    """The same from two host threads on one stream, whose launches interleave."""
    import threading
    xs = _several_inputs(2)
    alone = [_loss_and_grads(x, False) for x in xs]
    torch.cuda.synchronize()
    got, errors = [[] for _ in xs], []

    def work(i):
        try:
            for _ in range(8):
                got[i].append(_loss_and_grads(xs[i], False))
        except Exception as e:   # reported by the test's own thread
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(xs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors, errors
    for i, runs in enumerate(got):
        assert len(runs) == 8
        for r in runs:
            assert all(torch.equal(a, b) for a, b in zip(r, alone[i]))


def test_bad_targets_and_arguments():
    h, w, t = _inputs(64, 500, 128, seed=7)
    for bad in (500, -1, 2 ** 32 + 5, -2 ** 32 + 5):   # the last two are valid in their low 32 bits
        t[3] = bad
        with pytest.raises(ValueError, match="target"):
            fused_cross_entropy(h.cuda(), w.cuda(), t.cuda(), 256)
        unchecked = fused_cross_entropy(h.cuda(), w.cuda(), t.cuda(), 256, check_targets=False)
        t[3] = 0
        assert torch.equal(unchecked, fused_cross_entropy(h.cuda(), w.cuda(), t.cuda(), 256)), "not used as 0"
    assert torch.equal(unchecked, fused_cross_entropy(h.cuda(), w.cuda(), t.cuda().to(torch.int16), 256))
    with pytest.raises(ValueError):
        fused_cross_entropy(h.cuda().float(), w.cuda(), t.cuda(), 256)      # f32 h
    with pytest.raises(ValueError):
        fused_cross_entropy(h.cuda()[:, :100].contiguous(), w.cuda()[:, :100].contiguous(), t.cuda(), 256)
