"""Binary conversions on the matrix cores (long arrays) against the wave-group form (the same numbers
in short calls) and exact integers: partial tiles, both layouts, word strides and alignments,
moduli counts between the padded sizes, residues outside [0, m), values next to 0 and M."""
import random

import numpy as np
import pytest

from grns_amd import largest_primes_below, product
from tests.helpers import to_res

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

SHORT = 4000  # numbers per call of the wave-group form


def _set(name):
    n = int(name.split()[0])
    if "small" in name:
        return [v for v in range(2, 1000) if all(v % p for p in range(2, int(v ** 0.5) + 1))][:n]
    return largest_primes_below(n)


def _long(mod):
    return 16384 if len(mod) > 32 else 8192


def _values(M, count, rnd):
    L = M.bit_length()
    vals = [0, 1, 2, M - 1, M - 2, M // 2, M // 2 + 1]
    for k in range(1, L - 1, max(1, L // 60)):
        e = rnd.randrange(1 << k)
        vals += [e, M - 1 - e, 1 << k, M - (1 << k)]
    vals += [(1 << k) - 1 for k in range(28, L - 1, 28)] + [(1 << k) - 1 for k in range(32, L - 1, 32)]
    vals = [v % M for v in vals]
    return vals + [rnd.randrange(M) for _ in range(count - len(vals))]


def _number_major(x):
    return x.t().contiguous().t()


@pytest.mark.parametrize("name", ["3", "8", "12 small", "16", "20", "32", "50", "64", "64 small"])
def test_to_binary(name):
    import grns_amd as G
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    mod = _set(name)
    M, n = product(mod), len(mod)
    rnd = random.Random(n)
    ctx = G.Context(mod, 0)
    W = ctx.words
    base = _values(M, 1200, rnd)
    for extra in (0, 1, 31, 33):
        count = _long(mod) + extra
        pick = [rnd.randrange(len(base)) for _ in range(count)]
        x = torch.from_numpy(to_res(base, mod)).cuda()[:, torch.tensor(pick, device="cuda")].contiguous()
        want = [base[k].to_bytes(4 * W, "little") for k in pick]
        for layout in (lambda v: v, _number_major):
            got = ctx.to_binary(layout(x)).cpu().numpy().astype("<i4")
            assert [r.tobytes() for r in got] == want
        padded = torch.zeros((count, W + 3), dtype=torch.int32, device="cuda")
        ctx.to_binary(x, out=padded[:, 1:W + 1])
        assert np.array_equal(padded[:, 1:W + 1].cpu().numpy(), got)
        assert not padded[:, 0].any() and not padded[:, W + 1:].any()
        rows = torch.empty((W, count), dtype=torch.int32, device="cuda")
        ctx.to_binary(x, out=rows.t())
        assert np.array_equal(rows.t().cpu().numpy(), got)
    # residues outside [0, m): one number in 50, any int32
    raw = x.clone()
    at = torch.arange(0, count, 50, device="cuda")
    rows = torch.tensor([rnd.randrange(n) for _ in range(at.numel())], device="cuda")
    raw[rows, at] = torch.tensor([rnd.randrange(-1 << 31, 1 << 31) for _ in range(at.numel())], dtype=torch.int32,
                                 device="cuda")
    short = torch.cat([ctx.to_binary(raw[:, k:k + SHORT]) for k in range(0, count, SHORT)])
    assert torch.equal(ctx.to_binary(raw), short)
    ctx.close()


@pytest.mark.parametrize("name", ["3", "8", "12 small", "16", "20", "32", "50", "64", "64 small"])
def test_from_binary(name):
    import grns_amd as G
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    mod = _set(name)
    n = len(mod)
    rng = np.random.default_rng(n)
    ctx = G.Context(mod, 0)
    m = np.array(mod, dtype=object)[:, None]
    for nwords, extra in ((1, 0), (max(1, n - 1), 1), (n, 31), (n + 1, 33), (2 * n + 3, 5)):
        count = _long(mod) + extra
        w = rng.integers(-1 << 31, 1 << 31, size=(count, nwords), dtype=np.int64).astype("<i4")
        w[:200][rng.random((200, nwords)) < 0.5] = 0
        w[200:400][rng.random((200, nwords)) < 0.5] = -1
        sign = rng.integers(0, 2, size=count).astype(np.int32)
        wd, sd = torch.from_numpy(w).cuda(), torch.from_numpy(sign).cuda()
        got = ctx.from_binary(wd, sign=sd)
        short = torch.cat([ctx.from_binary(wd[k:k + SHORT], sign=sd[k:k + SHORT]) for k in range(0, count, SHORT)], 1)
        assert torch.equal(got, short), nwords
        vals = np.array([int.from_bytes(r.tobytes(), "little") * (-1 if s else 1) for r, s in
                         zip(w[:600], sign[:600])], dtype=object)
        assert (got[:, :600].cpu().numpy() == (vals[None, :] % m)).all()
        assert torch.equal(ctx.from_binary(wd), torch.cat([ctx.from_binary(wd[k:k + SHORT]) for k in
                                                           range(0, count, SHORT)], 1))
        nm = _number_major(torch.empty_like(got))
        ctx.from_binary(wd, sign=sd, out=nm)
        assert torch.equal(nm, got)
        odd = torch.empty(count * nwords + 1, dtype=torch.int32, device="cuda")[1:].view(count, nwords)
        odd.copy_(wd)
        assert torch.equal(ctx.from_binary(odd, sign=sd), got)
        assert torch.equal(ctx.from_binary(wd.t().contiguous().t(), sign=sd), got)
    ctx.close()
