"""Plan building: indexes and escape counts of every tensor read together, the
host's arrays uploaded as one image. Which error wins, and plans after a refused
one."""
import numpy as np
import pytest

import kvexp_amd
from conftest import bits_equal, say, to_dev
from kvdata import random_kv

pytestmark = pytest.mark.gpu


def _heads(ctx, rng, n, seq, dim, block, splits):
    import torch

    heads = []
    for _ in range(n):
        k, v = (to_dev(random_kv(rng, seq, dim), torch.int16) for _ in range(2))
        heads.append(dict(kx=ctx.encode(k, seq, dim, block), vx=ctx.encode(v, seq, dim, block), seq=seq, splits=splits,
                          k=k, v=v))
    return heads


@pytest.mark.parametrize("dim", [32, 64, 80, 96, 256])
@pytest.mark.parametrize("at", [0, 3])
def test_bad_block_refused(ctx, dim, at):
    """A block header that disagrees with its index fails the plan (checked with
    the indexes), but not before a head without an index; the good container
    builds afterwards and its outputs are the plain rows' bits."""
    import torch

    rng = np.random.default_rng(dim + at)
    seq, block, n_q = 4 * 64 - 5, 64, 3
    heads = _heads(ctx, rng, 3, seq, dim, block, 2)
    xkv = [{k: h[k] for k in ("kx", "vx", "seq", "splits")} for h in heads]
    vx = heads[1]["vx"]
    spot = int(vx.offsets[at].item()) + 4  # the header's head_dim
    good = int(vx.blob[spot].item())
    say("bad block", dim, at)
    vx.blob[spot] = (good + 8) % 256
    with pytest.raises(kvexp_amd.KvexpHipError, match="xkv block dimension or length mismatch"):
        ctx.plan(xkv, n_q, dim, block)
    short = dict(xkv[2], seq=seq + 1)  # more tokens than its index covers
    with pytest.raises(kvexp_amd.KvexpHipError, match="xkv ran out of tokens"):
        ctx.plan([xkv[0], xkv[1], short], n_q, dim, block)
    vx.blob[spot] = good
    q = to_dev(random_kv(rng, 3 * n_q, dim), torch.int16)
    px = ctx.plan(xkv, n_q, dim, block)
    pr = ctx.plan([{k: h[k] for k in ("k", "v", "seq", "splits")} for h in heads], n_q, dim, block)
    assert bits_equal(px.run(q, check_errors=True).cpu().numpy(), pr.run(q, check_errors=True).cpu().numpy())
    px.close()
    pr.close()


def test_plans_of_one_context_in_turn(ctx):
    """Plans of other sizes and kinds built between a plan's runs (they share
    the context's staging): each keeps its own arrays."""
    import torch

    rng = np.random.default_rng(5)
    made = []
    for dim, seq, n_q, splits in ((64, 700, 7, 3), (72, 300, 2, 2), (128, 1300, 12, 5), (32, 129, 1, 1), (96, 64, 8, 4)):
        heads = _heads(ctx, rng, 4, seq, dim, 128, splits)
        q = to_dev(random_kv(rng, 4 * n_q, dim), torch.int16)
        px = ctx.plan([{k: h[k] for k in ("kx", "vx", "seq", "splits")} for h in heads], n_q, dim, 128)
        pr = ctx.plan([{k: h[k] for k in ("k", "v", "seq", "splits")} for h in heads], n_q, dim, 128)
        made.append((px, pr, q, heads))
    for px, pr, q, _ in made + made[::-1]:
        say("plans in turn", px.dim)
        assert bits_equal(px.run(q, check_errors=True).cpu().numpy(), pr.run(q, check_errors=True).cpu().numpy())
    for px, pr, _, _ in made:
        px.close()
        pr.close()


@pytest.mark.parametrize("dim,order", [(32, 0), (64, 0), (96, 0), (96, 1), (128, 0), (256, 1)])
@pytest.mark.parametrize("n_q", [9, 10, 12, 14, 15, 16, 17, 21, 24])
def test_groups_of_query_rows(ctx, oracle, dim, order, n_q):
    """More than eight query rows: groups of equal size in small plans, of eight
    in larger ones (more items than CUs), the oracle's bits in both."""
    import torch

    rng = np.random.default_rng(dim * 100 + n_q)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    seq, splits = 300, 3
    for n_heads in (2, cus // (splits * 2) + 1):
        if n_heads > 2 and n_q not in (12, 17):
            continue
        say("query row groups", dim, order, n_q, n_heads)
        kv = [(random_kv(rng, seq, dim), random_kv(rng, seq, dim)) for _ in range(n_heads)]
        q = random_kv(rng, n_heads * n_q, dim, spread_lo=-4, spread_hi=-2)
        want = oracle.attention_heads("avx512" if order else "scalar", q,
                                      [dict(k=k, v=v, seq=seq, threads=splits) for k, v in kv],
                                      n_q=n_q, dim=dim, split=128)
        dev = [dict(k=to_dev(k, torch.int16), v=to_dev(v, torch.int16), seq=seq, splits=splits) for k, v in kv]
        plan = ctx.plan(dev, n_q, dim, 128, order)
        assert bits_equal(plan.run(to_dev(q, torch.int16), check_errors=True).cpu().numpy(), want)
        plan.update_heads([seq - 1] * n_heads)  # the fast update: the same groups, one token less
        want = oracle.attention_heads("avx512" if order else "scalar", q,
                                      [dict(k=k[:(seq - 1) * dim], v=v[:(seq - 1) * dim], seq=seq - 1, threads=splits)
                                       for k, v in kv], n_q=n_q, dim=dim, split=128)
        assert bits_equal(plan.run(to_dev(q, torch.int16), check_errors=True).cpu().numpy(), want)
        plan.close()
