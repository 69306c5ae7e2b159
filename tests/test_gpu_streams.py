"""How a wavefront takes its blocks: K through LDS in whole rows (short streams) or in the operand's layout (from 24
blocks per wavefront on), steps rotated by the workgroup's place. Sizes on both sides of that line, at one and several
blocks per wavefront and with a ragged last block, against the 64-bit oracle; the paged pass bit for bit as the contiguous one."""
import pytest
import torch

from kvskip_amd import kvskip as K
from kvskip_amd import workloads as W
from oracle import attention as O

pytestmark = pytest.mark.gpu

F32_REL = 2e-6        # fp32 sums of exact products: see test_gpu_mfma_pv.py


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("G", [4, 7])
@pytest.mark.parametrize("T,S", [(64 * 4, 1), (64 * 5 + 1, 1), (64 * 23 * 4 - 3, 1), (64 * 24 * 4, 1), (64 * 25 * 4 + 9, 1),
                                 (64 * 25 * 4 + 9, 2), (64 * 95, 2)])
def test_streams(gpu, D, G, T, S):
    g = torch.Generator().manual_seed(T + G)
    q = torch.randn(2, 2 * G, D, generator=g).to(torch.bfloat16)
    k, v = (torch.randn(2, 2, T, D, generator=g).to(torch.bfloat16) for _ in range(2))
    sc = D ** -0.5
    ref, lse = O.decode(q, k, v, sc)
    M, Z = O.block_stats(q, k, sc)
    gq, gk, gv = q.cuda(), k.cuda(), v.cuda()
    keep = torch.ones(2, 2, (T + 63) // 64, dtype=torch.bool)
    for kw in ({}, dict(stats=True), dict(stats=True, plan=K.make_plan(keep.cuda()))):
        r = K.decode(gq, gk, gv, sc, out_f32=True, num_splits=S, **kw)
        assert O.rel_err(r["out_f32"].cpu(), ref) <= F32_REL
        assert (r["lse"].cpu().double() - lse).abs().max().item() <= 2e-5
        if kw:
            assert (r["blk_max"].cpu().double() - M).abs().max().item() <= 2e-5
            assert ((r["blk_sum"].cpu().double() - Z) / Z).abs().max().item() <= 2e-5
    one = K.decode(gq, gk, gv, sc, stats=True, load_v=False, write_p=True, num_splits=S)
    assert torch.equal(one["blk_max"], r["blk_max"]) and torch.equal(one["blk_sum"], r["blk_sum"])
    table, kp, vp = W.paged_pools([gk], [gv], 3)
    a = K.decode(gq, gk, gv, sc, num_splits=S)
    b = K.decode(gq, kp[0], vp[0], sc, num_splits=S, block_table=table, T=T)
    assert torch.equal(a["out"], b["out"]) and torch.equal(a["lse"], b["lse"])


@pytest.mark.parametrize("D,G", [(128, 4), (64, 7)])
@pytest.mark.parametrize("T,S", [(64 * 4 * 6, 1), (64 * 5 * 4 + 9, 2), (64 * 4 * 26, 1), (64 * 4 * 2 * 25 + 1, 2), (64 * 45, 3)])
def test_batch_slots_alike(gpu, D, G, T, S):
    """A sequence gives the same bits in every slot of a batch and in buffers of any capacity: short and long streams, one
    and several splits, each pass that rotates its steps."""
    B, Hkv = 5, 3
    g = torch.Generator().manual_seed(T + G)
    cap = (T + 2047) // 2048 * 2048
    q = torch.randn(1, Hkv * G, D, generator=g).to(torch.bfloat16).cuda().expand(B, -1, -1).contiguous()
    keep = W.random_block_list(1, Hkv, (T + 63) // 64, 0.6, seed=T).cuda().expand(B, -1, -1).contiguous()
    lens = torch.full((B,), T, dtype=torch.int32, device="cuda")
    plan = K.make_plan(keep)
    rows = [torch.randn(1, Hkv, T, D, generator=g).to(torch.bfloat16).cuda() for _ in range(2)]
    first = None
    for tokens in (cap, cap + 64):
        k, v = (torch.zeros(B, Hkv, tokens, D, dtype=torch.bfloat16, device="cuda")[:, :, :T].copy_(x) for x in rows)
        table, kp, vp = W.paged_pools([k], [v], 3)
        sc = D ** -0.5
        runs = [K.decode(q, k, v, sc, out_f32=True, num_splits=S),
                K.decode(q, k, v, sc, out_f32=True, num_splits=S, stats=True, plan=plan),
                K.decode(q, kp[0], vp[0], sc, out_f32=True, num_splits=S, block_table=table, T=T),
                K.decode(q, k, v, sc, out_f32=True, num_splits=max(S, 2) * B, seq_lens=lens),
                K.decode(q, k, v, sc, stats=True, load_v=False, num_splits=S),
                K.vskip_one_pass(q, k, v, sc, tau=1e-4, out_f32=True, num_splits=S, sync=False)]
        for r in runs:
            for x in ("out_f32", "lse"):
                if x in r:
                    assert all(torch.equal(r[x][b], r[x][0]) for b in range(1, B)), x
        first = first or runs
        assert all(torch.equal(r[x], f[x]) for r, f in zip(runs, first) for x in ("out_f32", "lse") if x in r)
