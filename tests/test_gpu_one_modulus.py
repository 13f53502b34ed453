"""A set of one modulus has accuracy 0 and no refinement factor: a negative residue, whose sums are
negative, has no row of RNS_POW2 and raises the refinement status."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def test_negative_residue_of_one_modulus():
    import grns_amd as G
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    m = 2147483647
    ctx = G.Context([m], 0)
    x = torch.from_numpy(np.array([[-5, 7, 0, 1 - m, m - 1]], np.int32)).cuda()
    for fast in (False, True):
        ev = ctx.eval(x, fast=fast).view(5, 2, 2)[:, :, 0].cpu().numpy()
        assert np.isnan(ev[[0, 3]]).all() and not np.isnan(ev[[1, 2, 4]]).any(), fast
        assert ctx.status() != 0
        assert ctx.status() == 0
    ctx.close()
