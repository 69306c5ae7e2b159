"""P V on the matrix cores (weights as three bf16 parts): fp32 outputs against the 64-bit oracle at block and split
remainders, for every group size and head dim, and infinite V entries."""
import pytest
import torch

from kvskip_amd import kvskip as K
from oracle import attention as O

pytestmark = pytest.mark.gpu

# A weight's parts sum to it to 2^-24 and the products are exact, so an output is off by the fp32 sums and
# exponentials alone: a few ulps (2^-24 = 6e-8) of the row's 2-norm; measured 2e-7, a tenth of this bound.
F32_REL = 2e-6


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("G", [1, 2, 4, 7, 8])
@pytest.mark.parametrize("T,S", [(1, 1), (64, 1), (65, 2), (255, 1), (1000, 3)])
def test_f32_outputs(gpu, G, D, T, S):
    g = torch.Generator().manual_seed(100 * G + D + T)
    q = torch.randn(2, 2 * G, D, generator=g).to(torch.bfloat16)
    k, v = (torch.randn(2, 2, T, D, generator=g).to(torch.bfloat16) for _ in range(2))
    r = K.decode(q.cuda(), k.cuda(), v.cuda(), D ** -0.5, out_f32=True, num_splits=S)
    ref, lse = O.decode(q, k, v, D ** -0.5)
    assert O.rel_err(r["out_f32"].cpu(), ref) <= F32_REL
    assert (r["lse"].cpu().double() - lse).abs().max().item() <= 2e-5


@pytest.mark.parametrize("G,D", [(4, 128), (4, 64), (7, 128), (8, 64), (1, 128)])
def test_infinite_values(gpu, G, D):
    """An infinite V entry gives that infinity in its dim of every head that weighs its token, and no NaN
    (the parts of a weight may be 0 where the weight is not)."""
    g = torch.Generator().manual_seed(G + D)
    q = (0.2 * torch.randn(1, 2 * G, D, generator=g)).to(torch.bfloat16)   # flat: every weight is far above 0
    k, v = (torch.randn(1, 2, 150, D, generator=g).to(torch.bfloat16) for _ in range(2))
    k[0, 0, 7] = 0.0                                                       # a weight with few significant bits
    v[0, 0, 7, 3], v[0, 1, 140, D - 1] = float("inf"), float("-inf")
    for r in (K.decode(q.cuda(), k.cuda(), v.cuda(), D ** -0.5, out_f32=True, num_splits=1),
              K.decode(q.cuda(), k.cuda(), v.cuda(), D ** -0.5, out_f32=True, num_splits=2)):
        o = r["out_f32"].cpu()
        want = torch.zeros_like(o, dtype=torch.bool)
        want[0, :G, 3] = want[0, G:, D - 1] = True
        assert not o.isnan().any() and torch.equal(o.isinf(), want)
        assert (o[0, :G, 3] > 0).all() and (o[0, G:, D - 1] < 0).all()
