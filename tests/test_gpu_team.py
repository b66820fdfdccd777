"""Decode attention at every head_dim with an instantiated split kernel other
than 64, 128 and 256 (which test_gpu_attention.py covers): head_dim 32 on the
one-wave kernel, 80 to 224 on the team kernel, whose waves share a chunk's
rows, score chains, query rows and channels in uneven parts there."""
import numpy as np
import pytest

import kvexp_amd
from conftest import bits_equal, say
from kvdata import random_kv
from test_gpu_attention import ORDER, _block_modes, _escape_heavy_kv, _mixed_block_kv, max_rel_err, run_gpu

pytestmark = pytest.mark.gpu

DIMS = [(d, b) for d in (32, 80, 96, 112, 160, 192, 224) for b in ("scalar", "avx512") if b == "scalar" or d % 32 == 0]


@pytest.mark.parametrize("dim,backend", DIMS)
def test_team_dims_against_oracle(ctx, oracle, dim, backend):
    """XKV == raw == oracle, bit for bit (the outputs are the reference's for
    the same split, so no tolerance): every query-row count, lengths at the
    edges of a chunk, a wave's rows and a block, raw, 2-bit and 4-bit blocks
    side by side, blocks that start 2 bytes past a multiple of 4 (an odd
    number of escapes before them), and more escapes in a chunk than its first
    window of records holds."""
    rng = np.random.default_rng(500 + dim)
    modes, odd = set(), False
    cases = [(1, 128, 1, 1), (2, 128, 31, 1), (3, 64, 33, 1), (4, 128, 129, 2), (5, 255, 700, 3), (6, 100, 641, 4),
             (7, 128, 1280, 5), (8, 64, 64, 1), (12, 128, 511, 2)]
    for trial, (n_q, block, seq, splits) in enumerate(cases):
        heads = []
        for h in range(3):
            n = seq + h * 5
            if trial % 3 == 0:
                k, v = (_mixed_block_kv(rng, n, dim, block, kinds) for kinds in
                        (("coded", "raw", "narrow"), ("raw", "coded", "coded", "narrow")))
            else:
                k = _escape_heavy_kv(rng, n, dim, (0.3, 0.004, 0.0)[h], narrow=trial % 2 == 0)
                v = _escape_heavy_kv(rng, n, dim, (0.003, 0.2, 0.01)[h])
            heads.append(dict(k=k, v=v, seq=n, splits=splits, block=block))
            for x in (k, v):
                blob = oracle.encode(x, n, dim, block)
                modes |= _block_modes(oracle, blob, dim, n)
                odd |= bool(np.any(np.asarray(oracle.block_index(blob, dim, n)[0]) % 4 == 2))
        q = random_kv(rng, len(heads) * n_q, dim, spread_lo=-1, spread_hi=1)
        say("team dims", backend, dim, trial, dict(n_q=n_q, block=block, seq=seq, splits=splits))
        want = oracle.attention_heads(backend, q, [dict(k=h["k"], v=h["v"], seq=h["seq"], threads=h["splits"])
                                                   for h in heads], n_q=n_q, dim=dim, split=block)
        raw = run_gpu(ctx, ORDER[backend], q, heads, n_q, dim, block, False)
        xkv = run_gpu(ctx, ORDER[backend], q, heads, n_q, dim, block, True)
        assert bits_equal(raw, want), (trial, max_rel_err(raw, want))
        assert bits_equal(xkv, want), (trial, max_rel_err(xkv, want))
    assert modes == {0, 2, 4} and odd


@pytest.mark.parametrize("dim", [80, 96, 160, 224])
def test_team_three_bit_blocks(ctx, oracle, dim):
    """3-bit blocks (the format extension) at sizes whose code rows are not
    whole dwords: XKV equals the oracle over the decoded tokens."""
    rng = np.random.default_rng(60 + dim)
    n_q, block, seq = 4, 128, 1003
    k, v = _escape_heavy_kv(rng, seq, dim, 0.02), _escape_heavy_kv(rng, seq, dim, 0.001)
    q = random_kv(rng, n_q, dim, spread_lo=-1, spread_hi=1)
    want = oracle.attention("scalar", q, k, v, n_q=n_q, dim=dim, seq=seq, threads=2, split=block)
    ctx.set_encoder_modes(kvexp_amd.MODE_3BIT)
    try:
        got = run_gpu(ctx, 0, q, [dict(k=k, v=v, seq=seq, splits=2)], n_q, dim, block, True)
    finally:
        ctx.set_encoder_modes(kvexp_amd.MODES_REFERENCE)
    assert bits_equal(got, want), max_rel_err(got, want)
