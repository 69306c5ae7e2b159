"""The token index found in the plan's scores pass (ids, idx_out) at the edges of its blocks, wavefronts (8 blocks) and
workgroups (32), against the rule spelled out on the CPU (src/lab.py:149-167): a block is hit if the current token, at
T - 1, also stands earlier at one of the block's tokens, or right before one of them."""
import pytest
import torch

from kvskip_amd import ext as E

pytestmark = pytest.mark.gpu


def _rule(row, T):
    cur, hits = row[T - 1], set()
    for j in range(T):
        if (j < T - 1 and row[j] == cur) or (1 <= j and row[j - 1] == cur):
            hits.add(j // 64)
    return [int(b in hits) for b in range((T + 63) // 64)]


@pytest.mark.parametrize("lens", [[1], [2], [63], [64], [65], [66], [512], [513], [514], [2048], [2049], [2050],
                                  [1, 65, 577, 2113], [128, 129, 2, 1024], [4097, 1, 64, 3000]])
@pytest.mark.parametrize("G,D", [(4, 128), (7, 64)])
def test_index_in_scores(gpu, lens, G, D):
    dev, B, Hkv, T = "cuda", len(lens), 2, max(lens)
    nb = (T + 63) // 64
    NBC = nb + 3
    g = torch.Generator().manual_seed(T + G)
    # rows of few hits each: the current token only at chosen places around block edges
    for spot in (0, 62, 63, 64, 511, 512, 2047, None):
        ids = torch.randint(10, 1000, (B, T), generator=g, dtype=torch.int32)
        for b, n in enumerate(lens):
            ids[b, n - 1] = 5
            if spot is not None and spot < n - 1:
                ids[b, spot] = 5
            if n < T:  # past the sequence's end: never counted
                ids[b, n] = 5
        q = torch.randn(B, Hkv * G, D, generator=g).to(dev, torch.bfloat16)
        k = torch.randn(B, Hkv, T, D, generator=g).to(dev, torch.bfloat16)
        z = lambda *s, dtype=torch.float32: torch.zeros(*s, dtype=dtype, device=dev)  # noqa: E731
        Hq = Hkv * G
        sl = torch.tensor(lens, dtype=torch.int32, device=dev)
        out = torch.full((B, NBC), 9, dtype=torch.uint8, device=dev)
        flags = torch.full((Hkv,), 2, dtype=torch.int32, device=dev)  # heads on the token index
        cnt, lst = z(B, Hkv, dtype=torch.int32), z(B, Hkv, NBC, dtype=torch.int32)
        E.plan(q, k, z(B, Hkv, NBC, D), z(B, Hq, NBC), z(B, Hq, NBC), z(B, Hkv, NBC, dtype=torch.uint8), z(B, Hq),
               z(B, Hkv, dtype=torch.int32), flags, z(B, Hq, NBC), z(B, Hkv, dtype=torch.uint8), lst, cnt, D ** -0.5, 0.05, 32,
               1, False, part=z(E.plan_part_floats(B, Hq, Hkv, NBC)), seq_lens=sl if B > 1 else None, ids=ids.to(dev),
               idx_out=out)
        out, cnt, lst = out.cpu(), cnt.cpu(), lst.cpu()
        for b, n in enumerate(lens):
            want = _rule(ids[b].tolist(), n)
            assert out[b, :len(want)].tolist() == want, (spot, n)
            assert (out[b, len(want):] == 9).all()  # blocks past the sequence are left alone
            attended = [i for i, w in enumerate(want) if w or i == 0 or i == len(want) - 1]
            for h in range(Hkv):
                assert lst[b, h, :int(cnt[b, h])].tolist() == attended, (spot, n, h)
