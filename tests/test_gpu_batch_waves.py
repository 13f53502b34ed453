"""Division and scaling lists of a batch plan that are long enough for the forms of long arrays: ragged
vectors, divisors of every length, pairs left to the reference loop, mixed array orders, against short
calls."""
import random

import numpy as np
import pytest

from grns_amd import largest_primes_below, product
from tests.helpers import to_res

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n", [3, 8, 13, 32, 40, 64])
def test_batch_lists_by_waves(n):
    import grns_amd as G
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    mod = largest_primes_below(n)
    ctx = G.Context(mod, 0)
    M, rnd = product(mod), random.Random(n)
    top = M.bit_length() - 2
    base = [rnd.randrange(1 << rnd.randrange(1, top)) for _ in range(400)]
    div = [max(1, x >> rnd.randrange(1, top)) if i % 3 else rnd.randrange(1, 1 << rnd.randrange(1, top))
           for i, x in enumerate(base)]
    xb, db = to_res(base, mod), to_res(div, mod)
    db[:, 11] = 0
    lens = [1, 2, 63, 64, 65, 127, 31, 33, 0, 5000, 9001]
    while sum(lens) < 36000:
        lens.append(rnd.randrange(1, 9000))
    count = sum(lens)
    pick = np.array([rnd.randrange(400) for _ in range(count)])
    x, d = torch.from_numpy(xb[:, pick]).cuda(), torch.from_numpy(db[:, pick]).cuda()
    x[0, ::977] += 3 if mod[0] > 2**31 - 4 else mod[0]  # some past their modulus
    x[0, ::977].clamp_(min=0)
    D = torch.from_numpy(np.array([rnd.randrange(2 * top) for _ in range(count)], np.int32)).cuda()
    q0, r0, s0 = torch.empty_like(x), torch.empty_like(x), torch.empty_like(x)
    for a in range(0, count, 4000):
        b = min(count, a + 4000)
        q, r = ctx.div(x[:, a:b].contiguous(), d[:, a:b].contiguous())
        q0[:, a:b], r0[:, a:b] = q, r
        s0[:, a:b] = ctx.scale2pow(x[:, a:b].contiguous(), D[a:b].contiguous())
    xn, dn = x.t().contiguous().t(), d.t().contiguous().t()
    outs = [torch.full_like(x, -1) for _ in range(3)]
    outn = [torch.full((count, n), -1, dtype=torch.int32, device="cuda").t() for _ in range(3)]
    tasks, at = [], 0
    for i, c in enumerate(lens):
        cut = slice(at, at + c)
        a, b, o = (xn, dn, outn) if i % 4 == 3 else (x, d, outs)
        tasks.append(G.make_task("div_fast", c, a=a[:, cut], b=b[:, cut], out0=o[0][:, cut], out1=o[1][:, cut]))
        tasks.append(G.make_task("scale2pow", c, a=a[:, cut], out0=o[2][:, cut], D=D[cut]))
        at += c
    plan = G.Batch(ctx, tasks)
    for _ in range(2):
        plan.launch()
        at = 0
        for i, c in enumerate(lens):
            cut = slice(at, at + c)
            o = outn if i % 4 == 3 else outs
            for got, want in zip(o, (q0, r0, s0)):
                assert torch.equal(got[:, cut].contiguous(), want[:, cut].contiguous()), (i, c)
                got[:, cut] = -1
            at += c
    plan.close()
    ctx.close()
