"""P V on the matrix cores (weights as three bf16 parts): fp32 outputs against the 64-bit oracle at block and split
remainders, for every group size and head dim, and infinite V entries."""
import pytest
import torch

from kvskip_amd import ext as E
from kvskip_amd import kvskip as K
from kvskip_amd import planner as P
from kvskip_amd import workloads as W
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


@pytest.mark.parametrize("G,D", [(1, 64), (4, 128), (7, 128), (7, 64), (8, 128)])
@pytest.mark.parametrize("score", [-76.0, -80.0, -85.0])
def test_infinite_values_of_light_tokens(gpu, G, D, score):
    """The same for a token of weight 2^-110, 2^-115 and 2^-123 beside heavy ones, alone in its block (token 140: the
    block's other scores are as low) and not (token 7), in every pass that adds weights times V."""
    g = torch.Generator().manual_seed(G + D)
    T, nb = 150, 3
    q, k = torch.zeros(1, 2 * G, D, dtype=torch.bfloat16), torch.zeros(1, 2, T, D, dtype=torch.bfloat16)
    v = torch.randn(1, 2, T, D, generator=g).to(torch.bfloat16)
    q[..., 0] = 8.0                                                        # scores: 8 k[0], exact in bf16
    k[0, 0, 7, 0] = score / 8
    k[0, 1, 128:, 0] = score / 8
    v[0, 0, 7, 3], v[0, 1, 140, D - 1] = float("inf"), float("-inf")
    q, k, v = q.cuda(), k.cuda(), v.cuda()
    table, kp, vp = W.paged_pools([k], [v], 3)
    every = K.make_plan(torch.ones(1, 2, nb, dtype=torch.bool, device="cuda"))
    lens = torch.tensor([T], dtype=torch.int32, device="cuda")
    outs = [K.decode(q, k, v, 1.0, out_f32=True, num_splits=S, **kw)["out_f32"]
            for S in (1, 2) for kw in ({}, dict(stats=True), dict(stats=True, plan=every))]
    outs += [K.decode(q, k, v, 1.0, out_f32=True, num_splits=2, seq_lens=lens)["out_f32"],
             K.decode(q, kp[0], vp[0], 1.0, out_f32=True, num_splits=2, block_table=table, T=T)["out_f32"],
             K.vskip_one_pass(q, k, v, 1.0, local=nb, out_f32=True, num_splits=1)["out_f32"],
             K.vskip_one_pass(q, kp[0], vp[0], 1.0, local=nb, out_f32=True, num_splits=2, block_table=table, T=T)["out_f32"],
             P.FusedPlanner(P.Policy(), count=False).first(q, k, v, 1.0),
             P.FusedPlanner(P.Policy(), count=False).first(q, kp[0], vp[0], 1.0, block_table=table, T=T)]
    for o in outs:
        o = o.float().cpu()
        want = torch.zeros_like(o, dtype=torch.bool)
        want[0, :G, 3] = want[0, G:, D - 1] = True
        assert not o.isnan().any() and torch.equal(o.isinf(), want)
        assert (o[0, :G, 3] > 0).all() and (o[0, G:, D - 1] < 0).all()


@pytest.mark.parametrize("G,D", [(2, 128), (4, 64), (7, 128), (8, 64), (8, 128)])
@pytest.mark.parametrize("S", [1, 2])
def test_pv_weights_of_any_sign(gpu, G, D, S):
    """Pass 2 of two-pass V-skip takes the caller's P and scales as they are: negative scales beside zeros in P (weights
    of -0), tiny ones, and an infinite V under a tiny weight. Against the 64-bit sum; the bound as above, on the 2-norm of
    the summed magnitudes."""
    g = torch.Generator().manual_seed(10 * G + S)
    Hkv, T = 2, 300
    nb = (T + 63) // 64
    p = torch.rand(1, Hkv * G, nb * 64, generator=g).half()
    p[torch.rand(p.shape, generator=g) < 0.5] = 0.0
    p[:, :, T:] = 0.0
    p[0, :, 5] = 1.0
    v = torch.randn(1, Hkv, T, D, generator=g).to(torch.bfloat16)
    sc = torch.randn(1, Hkv, nb, G, generator=g)
    sc[0, :, 0] = 2.0 ** -112
    sc[0, :, 2] = -sc[0, :, 2].abs()
    every = K.make_plan(torch.ones(1, Hkv, nb, dtype=torch.bool, device="cuda"))
    args = (p.cuda(), sc.cuda(), every.block_idx, every.block_cnt)
    out = E.pv(args[0], v.cuda(), *args[1:], S, True)[1].cpu().double()
    w = (p.double().view(Hkv, G, nb, 64) * sc[0].double().transpose(1, 2)[..., None]).reshape(Hkv, G, -1)[..., :T]
    ref, mag = torch.matmul(w, v[0].double()).view(1, -1, D), torch.matmul(w.abs(), v[0].double().abs()).view(1, -1, D)
    assert not out.isnan().any()
    assert float((out - ref).norm() / mag.norm()) <= F32_REL
    v[0, 0, 5, 3] = float("inf")
    out = E.pv(args[0], v.cuda(), *args[1:], S, True)[1].cpu()
    assert (out[0, :G, 3] == float("inf")).all() and int((~out.isfinite()).sum()) == G
