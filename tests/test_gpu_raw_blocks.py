"""AVX-512 BF16 order over raw blocks of a container: the scores' flush test
reads the raw rows, so chunks on both sides of the exponent bound, and the rows
past a chunk's end that must not count, against the oracle bit for bit."""
import numpy as np
import pytest

from conftest import bits_equal, say
from kvdata import random_kv
from test_gpu_attention import run_gpu

pytestmark = pytest.mark.gpu


def raw_rows(rng, seq, dim, low_blocks, block):
    """BF16 rows whose exponents spread over 40 binades (their blocks encode
    raw), one element of each block in `low_blocks` far below the others; the
    exponent bound lies between (queries near 1: E_k >= 142 - E_q)."""
    e = rng.integers(100, 140, size=(seq, dim))
    bits = (rng.integers(0, 2, size=(seq, dim)) << 15) | (e << 7) | rng.integers(0, 128, size=(seq, dim))
    for b in range((seq + block - 1) // block):
        lo, hi = b * block, min(seq, (b + 1) * block)
        if b in low_blocks:
            bits[rng.integers(lo, hi), rng.integers(0, dim)] = rng.choice([3, 2 << 7, 5 << 7, 0x8000 | 9])
    return bits.astype(np.uint16)


@pytest.mark.parametrize("dim,block", [(32, 128), (32, 40), (64, 128), (96, 128), (96, 33), (128, 128), (160, 100),
                                       (192, 128), (224, 64), (256, 128)])
def test_raw_blocks_both_sides_of_the_bound(ctx, oracle, dim, block):
    rng = np.random.default_rng(4100 + dim + block)
    for n_q in (1, 2, 4, 5, 8):
        heads = []
        for seq in (block - 1, 3 * block, 5 * block + 7):
            n_blocks = (seq + block - 1) // block
            k = raw_rows(rng, seq, dim, set(rng.integers(0, n_blocks, size=n_blocks // 2)), block)
            blob = oracle.encode(k.reshape(-1), seq, dim, block)
            assert blob[0] == 0  # raw
            heads.append(dict(k=k.reshape(-1), v=random_kv(rng, seq, dim, sigma=0.5), seq=seq,
                              splits=int(rng.integers(1, 4)), block=block))
        q = random_kv(rng, len(heads) * n_q, dim, spread_lo=-16, spread_hi=-14)
        say("raw blocks", dim, block, n_q)
        want = oracle.attention_heads("avx512", q, [dict(k=h["k"], v=h["v"], seq=h["seq"], threads=h["splits"])
                                                    for h in heads], n_q=n_q, dim=dim, split=block)
        assert bits_equal(run_gpu(ctx, 1, q, heads, n_q, dim, block, True), want), n_q
