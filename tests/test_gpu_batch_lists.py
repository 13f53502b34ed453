"""Batch plans whose lists are cut into tiles of other sizes than the configured one (short lists), for
every operation class, against the per-call entry points."""
import random

import pytest

from grns_amd import largest_primes_below, product

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("tile", [1, 100, 1024, 16384])
@pytest.mark.parametrize("n,lens", [(8, (1, 255, 256, 257)), (20, (1, 2, 300)), (32, (1, 31, 513, 5000)),
                                    (64, (1, 3, 4, 5, 2100))])
def test_short_lists(n, lens, tile):
    import grns_amd as G
    from grns_amd.workload import Synth
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    mod = largest_primes_below(n)
    ctx, syn = G.Context(mod, 0), Synth(mod)
    L = product(mod).bit_length()
    rnd = random.Random(n * tile)
    tasks, checks = [], []
    for k, c in enumerate(lens * 2):
        x, d, D, _ = syn.div(c, seed=100 * n + k, max_bits=L - 2, max_shift=L + 40)
        y = syn.uniform(c, 7, k)
        if rnd.random() < 0.5:
            d[:, ::5] = 0
        q, r, z = torch.zeros_like(x), torch.zeros_like(x), torch.zeros_like(x)
        ev = torch.zeros((c, 4), dtype=torch.float64, device="cuda")
        sg = torch.zeros(c, dtype=torch.int32, device="cuda")
        tasks += [G.make_task("div_fast", c, a=x, b=d, out0=q, out1=r), G.make_task("scale2pow", c, a=x, out0=z, D=D),
                  G.make_task("eval", c, a=x, out0=ev), G.make_task("cmp", c, a=x, b=y, out0=sg)]
        checks.append((x, d, D, y, q, r, z, ev, sg))
    plan = G.Batch(ctx, tasks)
    plan.set_config(tile=tile)
    for _ in range(2):
        plan.launch()
    for x, d, D, y, q, r, z, ev, sg in checks:
        wq, wr = ctx.div(x, d, fast=True)
        assert torch.equal(q, wq) and torch.equal(r, wr)
        assert torch.equal(z, ctx.scale2pow(x, D))
        assert torch.equal(ev.view(torch.int64), ctx.eval(x).view(torch.int64))
        assert torch.equal(sg, ctx.cmp(x, y))
    plan.close()
    ctx.status()
    ctx.close()
