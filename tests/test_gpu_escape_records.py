"""A plan's escape records (built with the plan, and rewritten for the last
block by plan updates): attention over containers whose blocks hold no, few or
many escapes, up to more than the 4,096 that the builder gathers in LDS,
against plain BF16 rows, bit for bit (the same operations on the same
values)."""
import numpy as np
import pytest

from conftest import bits_equal, say, to_dev

pytestmark = pytest.mark.gpu


def _rows(rng, n, width, share):
    """n BF16 patterns over `width` neighbouring exponents, `share` of them 20 to 60 binades below."""
    e = rng.integers(118 - width, 118, n)
    e = np.where(rng.random(n) < share, rng.integers(60, 98, n), e)
    return (rng.integers(0, 2, n) << 15 | e << 7 | rng.integers(0, 128, n)).astype(np.uint16)


# (dim, block, exponents, escapes per element): blocks below one octet per thread, partly filled and several
# segments of 16,384 elements; 4- and 2-bit codes; 0.2 of 32,768 and 0.22 of 65,280 elements exceed 4,096
@pytest.mark.parametrize("dim,block,width,share", [(32, 16, 14, 0.05), (64, 128, 14, 0.0), (64, 128, 14, 0.01),
                                                   (64, 128, 3, 0.2), (96, 200, 14, 0.2), (128, 128, 3, 0.3),
                                                   (256, 128, 14, 0.2), (256, 255, 14, 0.22)])
def test_records(ctx, dim, block, width, share):
    import torch

    rng = np.random.default_rng(dim + block)
    seq, n_q, steps = 2 * block - 2, 3, 4  # the appends fill the second block and start a third
    kv = [_rows(rng, (seq + steps) * dim, width, share) for _ in range(2)]
    q = to_dev(_rows(rng, n_q * dim, 14, 0.0), torch.int16)
    dk, dv = (to_dev(x, torch.int16) for x in kv)
    caches = [ctx.cache(dim, seq + steps, block) for _ in range(2)]
    aset = ctx.append_set(caches)
    rows = torch.stack([dk.view(-1, dim), dv.view(-1, dim)])
    aset.append(rows[:, :seq].contiguous(), seq)
    plan = ctx.plan([dict(kx=caches[0].view(), vx=caches[1].view(), seq=seq, splits=2)], n_q, dim, block)
    for n in range(seq, seq + steps + 1):
        if n > seq:
            aset.append(rows[:, n - 1:n].contiguous(), 1)
            plan.update_lengths(n, block)
        say("escape records", dim, block, width, share, n)
        raw = ctx.plan([dict(k=dk[:n * dim], v=dv[:n * dim], seq=n, splits=2)], n_q, dim, block)
        got = plan.run(q, check_errors=True).cpu().numpy()
        assert np.isfinite(got).all()
        assert bits_equal(got, raw.run(q, check_errors=True).cpu().numpy()), n
        raw.close()
    plan.close()
