"""Evaluation, comparison, arg-max and mixed-radix digits of arrays whose numbers' residues lie side by side
(rows of exactly n or more words, any alignment, ragged counts) against the modulus-major forms."""
import numpy as np
import pytest

from grns_amd import largest_primes_below, product
from tests.helpers import to_res

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _numbers(mod, count, seed):
    rng = np.random.default_rng(seed)
    n, M = len(mod), product(mod)
    x = np.stack([rng.integers(0, m, count) for m in mod]).astype(np.int32)
    edges = to_res([0, 1, M - 1, M // 2, M // 2 + 1, 12345, M - 12345], mod)
    at = rng.integers(0, count, max(1, count // 20))
    x[:, at] = edges[:, at % edges.shape[1]]
    off = rng.integers(0, count, max(1, count // 50))
    x[rng.integers(0, n, off.size), off] += rng.choice([-5, mod[-1]], off.size).astype(np.int32)  # outside [0, m)
    return torch.from_numpy(x).cuda()


def _rows(x, pad, shift):
    """x as a number-major view: rows n + pad words apart, starting `shift` words into the buffer."""
    n, count = x.shape
    buf = torch.full((count * (n + pad) + shift + 8,), -7, dtype=torch.int32, device="cuda")
    view = buf[shift:shift + count * (n + pad)].view(count, n + pad)[:, :n].t()
    view.copy_(x)
    return view


@pytest.mark.parametrize("n", [4, 8, 16, 32, 64])
def test_number_major(n):
    import grns_amd as G
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    mod = largest_primes_below(n)
    ctx = G.Context(mod, 0)
    for count in (1, 2, 63, 64, 65, 255, 257, 1000, 40961):
        x, y = _numbers(mod, count, count + n), _numbers(mod, count, count + n + 1)
        y[:, ::3] = x[:, ::3]
        want = [ctx.eval(x), ctx.eval(x, fast=True), ctx.cmp(x, y), ctx.mrc(x)]
        top, at = ctx.max(x)
        for pad, shift in ((0, 0), (0, 1), (1, 0), (3, 2), (4, 4)):
            xn, yn = _rows(x, pad, shift), _rows(y, pad, shift)
            got = [ctx.eval(xn), ctx.eval(xn, fast=True), ctx.cmp(xn, yn), ctx.mrc(xn, out=torch.empty_like(x))]
            for k, (w, g) in enumerate(zip(want, got)):
                assert torch.equal(w.view(torch.int32), g.contiguous().view(torch.int32)), (count, pad, shift, k)
            assert torch.equal(ctx.cmp(xn, y), want[2])
            dn = _rows(torch.zeros_like(x), pad, shift)
            ctx.mrc(xn, out=dn)
            assert torch.equal(dn.contiguous(), want[3]), (count, pad, shift)
            ctx.mrc(x, out=dn.zero_())
            assert torch.equal(dn.contiguous(), want[3]), (count, pad, shift)
            for mrc in (False, True):
                r, i = ctx.max(xn, mrc=mrc)
                r0, i0 = ctx.max(x, mrc=mrc)
                assert torch.equal(r, r0) and int(i) == int(i0), (count, pad, shift, mrc)
            ctx.mrc(xn, out=xn)  # in place
            assert torch.equal(xn.contiguous(), want[3]), (count, pad, shift)
    ctx.close()
