"""Paths of the split kernels that random scores do not reach at every head_dim:
chosen moves of the running maxima, mixed and 3-bit blocks, the AVX-512 order's
flush bound, log-sum-exp, plain rows at any 2-byte address and containers that
end with their last code byte. Bodies shared with the tests at head_dim 64, 128
and 256 (test_gpu_attention.py, test_gpu_3bit.py)."""
import numpy as np
import pytest

import test_gpu_3bit as three_bit
import test_gpu_attention as attention
from conftest import bits_equal, say, to_dev
from kvdata import random_kv
from test_gpu_3bit import ctx3  # noqa: F401
from test_gpu_attention import ORDER, max_rel_err, run_gpu

pytestmark = pytest.mark.gpu

DIMS = (32, 80, 96, 112, 160, 192, 224)
DIMS_DP = tuple(d for d in DIMS if d % 32 == 0)
BOTH = [(d, b) for d in DIMS for b in ("scalar", "avx512") if b == "scalar" or d % 32 == 0]
ALL_BOTH = BOTH + [(d, b) for d in (64, 128, 256) for b in ("scalar", "avx512")]


@pytest.mark.parametrize("dim,backend", BOTH)
def test_chosen_moves(ctx, oracle, dim, backend):
    attention.test_wave_fold_chosen_moves(ctx, oracle, dim, backend)


@pytest.mark.parametrize("dim", DIMS)
def test_mixed_raw_and_coded_blocks(ctx, oracle, dim):
    attention.test_wave_kernel_mixed_raw_and_coded_blocks(ctx, oracle, dim)


@pytest.mark.parametrize("dim", DIMS_DP)
def test_dpbf16_flush_guard(ctx, oracle, dim):
    attention.test_wave_dpbf16_flush_guard(ctx, oracle, dim)


@pytest.mark.parametrize("dim,backend", BOTH)
def test_3bit_blocks(ctx3, oracle, dim, backend):  # noqa: F811
    three_bit.test_3bit_attention(ctx3, oracle, dim, backend)


@pytest.mark.parametrize("dim", DIMS_DP + (256,))
def test_3bit_dpbf16_flush_guard(ctx3, oracle, dim):  # noqa: F811
    three_bit.test_3bit_dpbf16_flush_guard(ctx3, oracle, dim)


@pytest.mark.parametrize("dim,backend", ALL_BOTH)
def test_lse(ctx, oracle, dim, backend):
    """Log-sum-exp of one split (written by the split kernel) and of several (by
    the merge): the outputs the oracle's bits, lse = m + log l within the
    device logarithm's rounding (2 ulp of about 8: 1e-6)."""
    rng = np.random.default_rng(31 + dim)
    for n_q, seq, splits in ((1, 77, 1), (2, 700, 4), (5, 300, 1), (8, 901, 7), (11, 260, 2)):
        heads = [dict(k=random_kv(rng, seq + h, dim), v=random_kv(rng, seq + h, dim), seq=seq + h, splits=splits)
                 for h in range(3)]
        q = random_kv(rng, 3 * n_q, dim, spread_lo=-4, spread_hi=-2)
        say("lse", dim, backend, n_q, seq, splits)
        want, lse_want = oracle.attention_heads(backend, q, [dict(k=h["k"], v=h["v"], seq=h["seq"], threads=splits)
                                                             for h in heads], n_q=n_q, dim=dim, split=128, with_lse=True)
        for xkv in (False, True):
            got, lse = run_gpu(ctx, ORDER[backend], q, heads, n_q, dim, 128, xkv, with_lse=True)
            assert bits_equal(got, want), (n_q, xkv, max_rel_err(got, want))
            assert np.allclose(lse, lse_want, rtol=1e-6, atol=1e-6), (n_q, xkv)


@pytest.mark.parametrize("dim,backend", ALL_BOTH)
def test_plain_rows_at_two_byte_addresses(ctx, oracle, dim, backend):
    """Plain K, V and queries that start 2, 6 and 14 bytes past 16-byte
    boundaries (rows are read 16 bytes at a time)."""
    import torch

    rng = np.random.default_rng(17 + dim)

    def at(x, elements):
        buf = torch.zeros(x.size + 16, dtype=torch.int16, device="cuda:0")
        buf[elements:elements + x.size] = to_dev(x, torch.int16)
        out = buf[elements:elements + x.size]
        assert out.data_ptr() % 16 == 2 * elements % 16
        return out

    for n_q, seq, splits in ((1, 1, 1), (3, 65, 1), (8, 500, 3)):
        k, v = random_kv(rng, seq, dim), random_kv(rng, seq, dim)
        q = random_kv(rng, n_q, dim, spread_lo=-4, spread_hi=-2)
        say("two-byte rows", dim, backend, n_q, seq)
        want = oracle.attention(backend, q, k, v, n_q=n_q, dim=dim, seq=seq, threads=splits, split=128)
        for a, b, c in ((1, 3, 7), (7, 1, 3)):
            plan = ctx.plan([dict(k=at(k, a), v=at(v, b), seq=seq, splits=splits)], n_q, dim, 128, ORDER[backend])
            got = plan.run(at(q, c), check_errors=True).cpu().numpy()
            plan.close()
            assert bits_equal(got, want), (n_q, max_rel_err(got, want))


@pytest.mark.parametrize("dim,backend", ALL_BOTH)
@pytest.mark.parametrize("width", [14, 3])
def test_container_ends_with_its_codes(ctx, oracle, dim, backend, width):
    """The last block a whole chunk of coded rows, without escapes, two bytes
    past a multiple of 4 (one escape in the block before it), in a buffer that
    holds nothing after it."""
    import torch

    rng = np.random.default_rng(dim + width)
    seq, n_q = 192, 5

    def rows():
        e = rng.integers(118 - width, 118, (seq, dim))
        e[:2] = [[118 - width], [117]]  # every channel spans the codes' width
        e[128:130] = [[118 - width], [117]]
        e[5, 7] = 60
        return (rng.integers(0, 2, (seq, dim)) << 15 | e << 7 | rng.integers(0, 128, (seq, dim))).astype(np.uint16)

    k, v = rows().reshape(-1), rows().reshape(-1)
    heads = []
    for x in (k, v):
        blob = oracle.encode(x, seq, dim, 128)
        off, _ = oracle.block_index(blob, dim, seq)
        assert off[1] % 4 == 2 and blob[off[1]] in (2, 4) and blob[off[1] + 2] == 0 and off[2] == blob.size
        heads.append(ctx.upload(blob, dim, seq, 128))
    q = random_kv(rng, n_q, dim, spread_lo=-1, spread_hi=1)
    say("container's end", dim, backend, width)
    want = oracle.attention(backend, q, k, v, n_q=n_q, dim=dim, seq=seq, threads=2, split=128)
    plan = ctx.plan([dict(kx=heads[0], vx=heads[1], seq=seq, splits=2)], n_q, dim, 128, ORDER[backend])
    got = plan.run(to_dev(q, torch.int16), check_errors=True).cpu().numpy()
    plan.close()
    assert bits_equal(got, want), max_rel_err(got, want)
