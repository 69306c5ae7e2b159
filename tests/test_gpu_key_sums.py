"""Key sums from the dense pass of a planner's first step (kvskip_attn_args.key_sums) against block_sums and the 64-bit
sums, and the planner's state after a first step that takes them from there."""
import pytest
import torch

from kvskip_amd import ext as E
from kvskip_amd import planner as P
from kvskip_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("G", [1, 4, 7])
def test_key_sums(gpu, G, D):
    """Blocks of full, one-row and 63-row lengths; what lies past a sequence's end stays as it was. A sum of 64 bf16
    values in fp32 is within 64 ulps (2^-24) of its terms' magnitudes, well under 1e-5 of the block's 2-norm x 8."""
    lens = [1, 64, 65, 64 * 30 + 63, 64 * 100]
    B, Hkv, T, NBC = len(lens), 2, max(lens), max(lens) // 64 + 5
    g = torch.Generator().manual_seed(G * D)
    q = torch.randn(B, Hkv * G, D, generator=g).to(torch.bfloat16).cuda()
    k, v = (torch.randn(B, Hkv, T, D, generator=g).to(torch.bfloat16).cuda() for _ in range(2))
    sl = torch.tensor(lens, dtype=torch.int32, device="cuda")
    nb, S, f32 = (T + 63) // 64, 8, dict(dtype=torch.float32, device="cuda")
    bufs = dict(out=torch.empty(B, Hkv * G, D, dtype=torch.bfloat16, device="cuda"), lse=torch.empty(B, Hkv * G, **f32),
                blk_max=torch.empty(B * Hkv * G * nb, **f32), blk_sum=torch.empty(B * Hkv * G * nb, **f32),
                part_acc=torch.empty(B * Hkv * G * S * D, **f32), part_ml=torch.empty(B * Hkv * G * S * 2, **f32))
    ref = {x: y.clone() for x, y in bufs.items()}
    sums = torch.full((B, Hkv, NBC, D), 7.0, **f32)
    E.decode_into(q, k, v, D ** -0.5, bufs, stats=True, num_splits=S, seq_lens=sl, key_sums=sums)
    E.decode_into(q, k, v, D ** -0.5, ref, stats=True, num_splits=S, seq_lens=sl)
    for x in ("out", "lse", "blk_max", "blk_sum"):
        assert torch.equal(bufs[x], ref[x]), x
    want = E.block_sums(k, NBC, seq_lens=sl)
    for b, n in enumerate(lens):
        m = (n + 63) // 64
        pad = torch.zeros(Hkv, m * 64, D, dtype=torch.float64)
        pad[:, :n] = k[b, :, :n].cpu().double()
        exact = pad.view(Hkv, m, 64, D).sum(2)
        got = sums[b, :, :m].cpu().double()
        assert (got - exact).abs().max().item() <= 1e-5 * 8
        assert (got - want[b, :, :m].cpu().double()).abs().max().item() <= 1e-5 * 8
        assert (sums[b, :, m:] == 7.0).all()


@pytest.mark.parametrize("G,D", [(4, 128), (8, 64), (8, 128)])
def test_key_sums_of_long_streams(gpu, G, D):
    """The same where a wavefront streams 24 blocks and more (its steps then rotate by up to 4 alone, and a pass without
    the sums takes K another way): one and several chunks a sequence, ragged last blocks."""
    lens = [64 * 430 + 17, 64, 64 * 210, 64 * 100 + 1]
    B, Hkv, T, S = len(lens), 2, max(lens), 3
    g = torch.Generator().manual_seed(G * D)
    q = torch.randn(B, Hkv * G, D, generator=g).to(torch.bfloat16).cuda()
    k, v = (torch.randn(B, Hkv, T, D, generator=g).to(torch.bfloat16).cuda() for _ in range(2))
    sl = torch.tensor(lens, dtype=torch.int32, device="cuda")
    nb, f32 = (T + 63) // 64, dict(dtype=torch.float32, device="cuda")
    bufs = dict(out=torch.empty(B, Hkv * G, D, dtype=torch.bfloat16, device="cuda"), lse=torch.empty(B, Hkv * G, **f32),
                blk_max=torch.empty(B * Hkv * G * nb, **f32), blk_sum=torch.empty(B * Hkv * G * nb, **f32),
                part_acc=torch.empty(B * Hkv * G * S * D, **f32), part_ml=torch.empty(B * Hkv * G * S * 2, **f32))
    ref = {x: y.clone() for x, y in bufs.items()}
    sums = torch.full((B, Hkv, nb + 2, D), 7.0, **f32)
    E.decode_into(q, k, v, D ** -0.5, bufs, stats=True, num_splits=S, seq_lens=sl, key_sums=sums)
    E.decode_into(q, k, v, D ** -0.5, ref, stats=True, num_splits=S, seq_lens=sl)
    for x in ("out", "lse"):
        assert torch.equal(bufs[x], ref[x]), x
    for b, n in enumerate(lens):
        m = (n + 63) // 64
        pad = torch.zeros(Hkv, m * 64, D, dtype=torch.float64)
        pad[:, :n] = k[b, :, :n].cpu().double()
        assert (sums[b, :, :m].cpu().double() - pad.view(Hkv, m, 64, D).sum(2)).abs().max().item() <= 1e-5 * 8
        assert (sums[b, :, m:] == 7.0).all()
        for x in ("blk_max", "blk_sum"):
            y, z = (t[x].view(B, Hkv * G, nb)[b, :, :m] for t in (bufs, ref))
            assert torch.equal(y, z), x


@pytest.mark.parametrize("ragged", [False, True])
def test_first_step(gpu, monkeypatch, ragged):
    """A batch's planner from a first step with the sums in its pass, against one with block_sums: the same decisions,
    lists and stored sets at every step, outputs and references to rounding."""
    B, Hkv, G, D, T0, steps = 5, 4, 4, 128, 1900, 6
    lens = [1900, 130, 700, 1024, 65] if ragged else [T0] * B
    run = W.planner_run(layers=1, B=B, Hq=Hkv * G, Hkv=Hkv, D=D, T0=T0, steps=steps, seed=61, ragged=lens)
    k, v, ids = run.k[0].cuda(), run.v[0].cuda(), run.ids.cuda()
    qp = W.QueryProcess(run, 0, p_jump=0.05, revert=True)
    qs = [qp.next().cuda() for _ in range(steps)]
    pol = lambda: P.Policy(calib=0.05, calib_kind="peak", calib_warm=(4, 2), calib_auto_ix=0.1)
    pl = []
    for blocks in (0, 1 << 30):
        monkeypatch.setattr(P, "SUMS_IN_PASS_BLOCKS", blocks)
        p = P.FusedPlanner(pol(), count=False, carrier=P.UpdateCarrier())
        outs = []
        for t in range(steps):
            if ragged:
                sl = torch.tensor([n + t for n in lens], dtype=torch.int32, device="cuda")
                o = p.step(qs[t], k, v, run.scale, ids=ids, seq_lens=sl)
            else:
                o = p.step(qs[t], k[:, :, :T0 + t], v[:, :, :T0 + t], run.scale, ids=ids)
            outs.append(o.float().clone())
            p.carrier.flush()
            outs.append({x: p.state[x].clone() for x in ("keep", "age", "trig", "block_cnt", "lse_att", "csum")})
        pl.append(outs)
    for a, b in zip(*pl):
        if isinstance(a, dict):
            assert all(torch.equal(a[x], b[x]) for x in ("keep", "age", "trig", "block_cnt"))
            assert torch.allclose(a["csum"], b["csum"], rtol=0, atol=1e-4)
            assert torch.allclose(a["lse_att"], b["lse_att"], rtol=0, atol=1e-4)
        else:
            assert float((a - b).norm() / b.norm()) <= 1e-3
