"""The one-pass encoder on blocks of more than 16,384 elements (workgroups of
512 and 1,024 threads), against the oracle's encode_bf16 and the three-launch
encoder (unaligned sources)."""
import ctypes as C

import numpy as np
import pytest

import kvexp_amd
from conftest import say, to_dev
from test_gpu_encode_fused import _data, _encode_unaligned

pytestmark = pytest.mark.gpu

# (dim, block, tokens): just above 16,384 elements, 32,768, just above it, and the format's most (65,280)
SHAPES = [(72, 228, 1000), (136, 121, 1234), (160, 128, 3001), (192, 128, 128), (256, 65, 4000), (256, 128, 10001),
          (256, 129, 300), (232, 255, 2000), (256, 255, 5100)]


@pytest.mark.parametrize("modes", [kvexp_amd.MODES_REFERENCE, kvexp_amd.MODES_REFERENCE | kvexp_amd.MODE_3BIT])
def test_large_blocks(ctx, oracle, modes):
    """Encode, and prefill appends from empty and partial containers: the
    bytes, the index and the kept tail of encode_bf16."""
    import torch

    rng = np.random.default_rng(77)
    ctx.set_encoder_modes(modes)
    try:
        for i, (dim, block, seq) in enumerate(SHAPES):
            say("large blocks", modes, dict(dim=dim, block=block, seq=seq))
            kv = _data(rng, seq, dim, ("outliers", "specials", "wide")[i % 3])
            want = oracle.encode(kv, seq, dim, block, modes=modes)
            off, first = oracle.block_index(want, dim, seq)
            enc = ctx.encode(to_dev(kv, torch.int16), seq, dim, block)
            assert np.array_equal(enc.blob[: enc.nbytes].cpu().numpy(), want), (dim, block)
            assert np.array_equal(enc.offsets.cpu().numpy(), off) and np.array_equal(enc.first.cpu().numpy(), first)
            blob, uoff, _ = _encode_unaligned(ctx, kv, seq, dim, block)
            assert np.array_equal(blob, want) and np.array_equal(uoff, off), (dim, block)
            cuts = [c for c in (0, 1, block - 1, block, seq // 2) if c < seq]
            caches = [ctx.cache(dim, seq + 1, block) for _ in cuts]
            for c, n in zip(caches, cuts):
                if n:
                    c.append(to_dev(kv[: n * dim], torch.int16), n)
            ctx.append_batch(caches, [to_dev(kv[n * dim:], torch.int16) for n in cuts], [seq - n for n in cuts],
                             check_errors=True)
            for c, n in zip(caches, cuts):
                assert c.size() == want.size and np.array_equal(c.blob[: want.size].cpu().numpy(), want), (dim, block, n)
                assert np.array_equal(c.view().offsets.cpu().numpy(), off)
                rest = seq % block
                tail = c.tail[: rest * dim].cpu().numpy().view(np.uint16)
                assert np.array_equal(tail, kv[(seq - rest) * dim:]), (dim, block, n)
    finally:
        ctx.set_encoder_modes(kvexp_amd.MODES_REFERENCE)


def test_noalloc_large_blocks(ctx, oracle):
    """The no-allocation entry on such blocks: the same bytes, and refused
    beyond the three-launch encoder's scratch as its rule says."""
    import torch

    rng = np.random.default_rng(5)
    dim, block, seq = 256, 128, 128 * 40 + 7
    kv = _data(rng, seq, dim, "outliers")
    want = oracle.encode(kv, seq, dim, block)
    src = to_dev(kv, torch.int16)
    nb = (seq + block - 1) // block
    out = torch.zeros(kvexp_amd.encode_bound(seq, dim, block), dtype=torch.uint8, device="cuda:0")
    offs = torch.zeros(nb + 1, dtype=torch.int64, device="cuda:0")
    first = torch.zeros(nb + 1, dtype=torch.int32, device="cuda:0")
    st = torch.zeros(1, dtype=torch.int32, device="cuda:0")
    lib, s = kvexp_amd.lib(), torch.cuda.current_stream().cuda_stream

    def call(n):
        return lib.kvexp_hip_encode_noalloc(ctx.h, src.data_ptr(), n, dim, block, out.data_ptr(), C.c_size_t(1 << 40),
                                            offs.data_ptr(), first.data_ptr(), st.data_ptr(), s)

    for _ in range(2):
        out.zero_()
        assert call(seq) == 0
        assert np.array_equal(out[: want.size].cpu().numpy(), want) and int(st.item()) == 0
    # 4 MiB of scratch hold about 5,350 blocks of head_dim 256 (16 + 768 bytes each); refused before any launch
    assert call(128 * 5400) == 6
