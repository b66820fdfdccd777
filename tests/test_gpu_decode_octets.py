"""Block decode at head_dims that are multiples of 8 (decode_octets_kernel):
segments of 16,384 elements, a quarter of their octets per wave, escape ranks
across lanes, steps, waves and segments."""
import numpy as np
import pytest

import kvexp_amd
from conftest import say, to_dev
from test_gpu_attention import _escape_heavy_kv, _mixed_block_kv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,block", [(8, 1), (8, 255), (24, 100), (64, 128), (72, 33), (128, 128), (128, 255), (136, 240),
                                       (256, 65), (256, 255)])
def test_decode_octets_edges(ctx, oracle, dim, block):
    """Whole and cut-short decodes (the last octet inside a wave step, a wave,
    a segment) equal the tokens bit for bit, with escapes at rates of 0 to
    30 %, raw blocks between coded ones, and 3-bit blocks."""
    import torch

    rng = np.random.default_rng(dim * 1000 + block)
    seq = 3 * block + block // 2 + 1
    sets = [_escape_heavy_kv(rng, seq, dim, frac, narrow) for frac, narrow in ((0.3, False), (0.004, True), (0.0, False))]
    sets.append(_mixed_block_kv(rng, seq, dim, block, ("coded", "raw", "narrow")))
    for i, kv in enumerate(sets):
        for modes in (kvexp_amd.MODES_REFERENCE, kvexp_amd.MODES_REFERENCE | kvexp_amd.MODE_3BIT):
            ctx.set_encoder_modes(modes)
            try:
                enc = ctx.encode(to_dev(kv, torch.int16), seq, dim, block)
            finally:
                ctx.set_encoder_modes(kvexp_amd.MODES_REFERENCE)
            say("decode octets", dim, block, i, modes)
            for n in sorted({seq, seq - 1, block + 1, max(1, block // 3), 1}):
                out = torch.full((seq * dim,), 0x5A5A, dtype=torch.int16, device="cuda:0")
                got = ctx.decode(enc, n, out).cpu().numpy().view(np.uint16)
                assert np.array_equal(got, kv[: n * dim]), (i, modes, n)
                assert bool((out[n * dim:] == 0x5A5A).all())  # nothing past the tokens asked for


@pytest.mark.parametrize("dim,block", [(8, 16), (16, 16), (64, 16), (64, 32), (64, 33), (64, 64), (64, 65), (64, 129),
                                       (72, 28), (72, 29), (72, 57), (72, 114)])
def test_decode_octets_small_blocks(ctx, oracle, dim, block):
    """Blocks at the edges of the shorter segments (256, 512 and 1,024 octets)
    and of a wave and less."""
    test_decode_octets_edges(ctx, oracle, dim, block)


def test_checked_decode_refuses_a_short_index(ctx):
    """More tokens than the index covers: refused, and nothing is written."""
    import torch

    kv = torch.zeros(200 * 64, dtype=torch.int16, device="cuda:0")
    enc = ctx.encode(kv, 200, 64, 128)
    out = torch.full((300 * 64,), 7, dtype=torch.int16, device="cuda:0")
    with pytest.raises(kvexp_amd.KvexpHipError, match="xkv decode ran out of blocks"):
        ctx.decode(enc, 300, out)
    assert bool((out == 7).all())
    ctx.decode(enc, 200, out)  # the status word is clear again
