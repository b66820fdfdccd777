"""kvexp_hip_plan_update's two ways to the GPU: lengths as a kernel argument
(up to 512 heads, byte counts as before) and the uploaded job table (more
heads, or changed byte counts), step by step across a block boundary."""
import numpy as np
import pytest

from conftest import bits_equal, say, to_dev
from kvdata import random_kv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,dim", [(1, 64), (3, 96), (512, 32), (513, 32)])
def test_updates_equal_fresh_plans(ctx, heads, dim):
    import torch

    rng = np.random.default_rng(heads)
    block, n_q, start, steps = 16, 2, 29, 5  # 29 .. 34 tokens: a block ends at 32
    kv = random_kv(rng, 2 * heads * (start + steps), dim).reshape(2 * heads, start + steps, dim)
    caches = [ctx.cache(dim, start + steps, block) for _ in range(2 * heads)]
    aset = ctx.append_set(caches)
    aset.append(to_dev(np.ascontiguousarray(kv[:, :start]).reshape(-1), torch.int16), start)
    q = to_dev(random_kv(rng, heads * n_q, dim), torch.int16)

    def table():
        return [dict(kx=caches[2 * h].view(), vx=caches[2 * h + 1].view(), seq=caches[0].seq, splits=2)
                for h in range(heads)]

    plan = ctx.plan(table(), n_q, dim, block)
    for i in range(steps):
        aset.append(to_dev(np.ascontiguousarray(kv[:, start + i:start + i + 1]).reshape(-1), torch.int16), 1)
        if i == 3:  # byte counts that differ from the last update's
            for c in caches:
                c.size()
            plan.update(table())
        else:
            plan.update_lengths(caches[0].seq, block)
        got = plan.run(q, check_errors=True).cpu().numpy()
        fresh = ctx.plan(table(), n_q, dim, block)
        say("plan lengths", heads, dim, caches[0].seq)
        assert bits_equal(got, fresh.run(q, check_errors=True).cpu().numpy()), i
        fresh.close()
    plan.close()
