"""The workspace queries of the multi-row passes (CPU): a workspace sized for n rows takes every smaller
pass, so the size never falls as the rows grow (the split-K partials alone do: a pass of fewer rows
splits K more)."""
import ctypes

import pytest

from transformer_amd import _lib
from transformer_amd.configs import M306, TINY


def _cfg(d, heads, kv, ff, ctx, layers=2, vocab=32000):
    return dict(vocab_size=vocab, d_model=d, n_heads=heads, n_kv_heads=kv, n_layers=layers, d_head=64, d_ff=ff,
                context_len=ctx)


CONFIGS = {"tiny": TINY, "306m": M306, "d512": _cfg(512, 8, 8, 1408, 256), "d768": _cfg(768, 12, 4, 2048, 512),
           "d64": _cfg(64, 1, 1, 96, 1024), "wide_ff": _cfg(320, 5, 5, 8192, 700), "long": _cfg(256, 4, 1, 704, 40000)}


@pytest.mark.parametrize("name", CONFIGS)
def test_workspace_sizes_never_fall_with_the_rows(name):
    L, c = _lib.lib(), CONFIGS[name]
    cfg = _lib.MsdConfig.from_dict(c)
    for query, most in ((L.msd_prefill_workspace_bytes, min(c["context_len"], 1100)),
                        (L.msd_verify_workspace_bytes, min(c["context_len"], 300)),
                        (L.msd_batch_workspace_bytes, 1024)):
        sizes = [query(ctypes.byref(cfg), n) for n in range(1, most + 1)]
        assert sizes[0] > 0
        falls = [n + 2 for n in range(most - 1) if sizes[n + 1] < sizes[n]]
        assert not falls, (name, falls)
    at = [L.msd_prefill_workspace_bytes(ctypes.byref(cfg), n) for n in range(1100, c["context_len"] + 1, 97)]
    assert at == sorted(at)
