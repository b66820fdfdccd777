"""Appends the one-pass encoder does not take (a source or tail that is not
16-byte aligned, head_dims that are no multiple of 8): one-token and
multi-block appends, single and batched with aligned ones, against the oracle's
containers, indexes and the rows kept for the next append."""
import numpy as np
import pytest

import kvexp_amd
from conftest import say, to_dev
from test_gpu_3bit import M3, _kv3
from test_gpu_codec import _kinds

pytestmark = pytest.mark.gpu


def _off_by(x, elements):
    """x on the device, `elements` BF16 past a 16-byte boundary."""
    import torch

    buf = torch.zeros(x.size + 16, dtype=torch.int16, device="cuda:0")
    buf[elements:elements + x.size] = to_dev(x, torch.int16)
    out = buf[elements:elements + x.size]
    assert out.data_ptr() % 16 == 2 * elements % 16
    return out


def _check(oracle, c, kv, pos, modes, where):
    dim, block = c.dim, c.block
    want = oracle.encode(kv[: pos * dim], pos, dim, block, modes=modes)
    n = c.size()
    assert n == want.size, where
    assert np.array_equal(c.blob[:n].cpu().numpy(), want), where
    off, first = oracle.block_index(want, dim, pos)
    assert np.array_equal(c.view().offsets.cpu().numpy(), off), where
    assert np.array_equal(c.view().first.cpu().numpy(), first), where
    rest = pos % block
    kept = c.tail[: rest * dim].cpu().numpy().view(np.uint16)
    assert np.array_equal(kept, kv[(pos - rest) * dim: pos * dim]), where


def _data(rng, total, dim, kind, modes):
    half = total // 2
    if modes == M3:
        return np.concatenate([_kv3(rng, half, dim, 0.01 * kind), _kinds(rng, total - half, dim, kind)])
    return np.concatenate([_kinds(rng, half, dim, kind), _kinds(rng, total - half, dim, (kind + 1) % 4)])


@pytest.mark.parametrize("modes", [kvexp_amd.MODES_REFERENCE, M3])
@pytest.mark.parametrize("dim,block", [(36, 100), (64, 128), (64, 1), (72, 33), (128, 128), (200, 255), (256, 128), (256, 255)])
def test_unaligned_appends(ctx, oracle, dim, block, modes):
    """One container grown by sources 2, 8 and 14 bytes off alignment."""
    rng = np.random.default_rng(dim * 300 + block)
    total = 3 * block + 41
    kv = _data(rng, total, dim, 1, modes)
    ctx.set_encoder_modes(modes)
    try:
        c = ctx.cache(dim, total, block)
        pos = 0
        for step, n in enumerate([1, 2, block, 1, 1, 2 * block + 3, 5, 1, 7, 1] * 4):
            n = min(n, total - pos)
            if n == 0:
                break
            c.append(_off_by(kv[pos * dim:(pos + n) * dim], (1, 4, 7)[step % 3]), n)
            pos += n
            say("unaligned append", dim, block, modes, step, pos)
            _check(oracle, c, kv, pos, modes, (step, pos))
    finally:
        ctx.set_encoder_modes(kvexp_amd.MODES_REFERENCE)


@pytest.mark.parametrize("modes", [kvexp_amd.MODES_REFERENCE, M3])
@pytest.mark.parametrize("dim,block", [(36, 128), (64, 128), (128, 100), (256, 128)])
def test_unaligned_append_batches(ctx, oracle, dim, block, modes):
    """Batches of containers in different states, aligned and unaligned sources
    side by side: one token each (one workgroup per container), then several
    blocks in some (every block finds its container)."""
    rng = np.random.default_rng(dim * 301 + block)
    start = [0, 1, block - 1, block, block + 1, 2 * block + 5, 0, 3]
    total = 5 * block + 60
    data = [_data(rng, total, dim, i % 4, modes) for i in range(len(start))]
    ctx.set_encoder_modes(modes)
    try:
        caches = [ctx.cache(dim, total, block) for _ in start]
        for c, d, st in zip(caches, data, start):
            if st:
                c.append(_off_by(d[: st * dim], 0), st)
        pos = list(start)
        rounds = [[1] * len(start), [0, 3, 1, block, 2 * block + 1, 0, block + 7, 1], [1] * len(start),
                  [2 * block, 1, 0, 5, 1, block - 2, 1, 2 * block + 9], [1, 0, 1, 1, 0, 1, 1, 1]]
        for rnd, sizes in enumerate(rounds):
            toks = [_off_by(d[p * dim:(p + max(n, 1)) * dim], (0, 1, 0, 5)[i % 4])
                    for i, (d, p, n) in enumerate(zip(data, pos, sizes))]
            ctx.append_batch(caches, toks, sizes, check_errors=True)
            for i, (c, d) in enumerate(zip(caches, data)):
                pos[i] += sizes[i]
                say("unaligned batch", dim, block, modes, rnd, i, pos[i])
                if pos[i]:
                    _check(oracle, c, d, pos[i], modes, (rnd, i))
    finally:
        ctx.set_encoder_modes(kvexp_amd.MODES_REFERENCE)
