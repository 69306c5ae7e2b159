"""CPU checks of the native host module (csrc/host.cpp): the split rule count by count, zeroed state
carved from one allocation, and refusals with the messages that the Python checks had."""
import ctypes
import math
import random

import pytest
import torch

from kvskip_amd import _native, ext
from kvskip_amd import kvskip as K
from kvskip_amd import planner as P


def _rule(bh, n_tiles, slots, max_splits, min_tiles):
    def score(s):
        waves = bh * s / slots
        return waves / math.ceil(waves) - 0.002 * s

    most = 1
    while most < max_splits and math.ceil(n_tiles / (most + 1)) >= min_tiles:
        most += 1
    best = 1
    for s in range(2, most + 1):
        if score(s) > score(best) + 1e-9:
            best = s
    return best


@pytest.mark.parametrize("slots", [1, 7, 64, 256, 304])
def test_split_rule(slots):
    rng = random.Random(slots)
    for _ in range(400):
        a = (rng.randint(1, 600), rng.randint(1, 4096))
        kw = dict(max_splits=rng.choice([1, 64, 256]), min_tiles=rng.choice([1, 4, 8]))
        assert K.num_splits_for(*a, sms=slots, **kw) == _rule(*a, slots, *kw.values()), (a, kw)


def test_zeroed_state():
    parts = (("f4", (2, 3, 5)), ("u1", (7,)), ("i4", (1, 4)), ("u1", (2, 0)))
    ts = _native.host().zeroed(parts, torch.empty(0))
    assert [(t.dtype, tuple(t.shape)) for t in ts] == [(torch.float32, (2, 3, 5)), (torch.uint8, (7,)),
                                                       (torch.int32, (1, 4)), (torch.uint8, (2, 0))]
    for i, t in enumerate(ts):                    # apart from each other, and writable
        assert t.is_contiguous() and not t.any()
        t.fill_(i + 1)
    assert all((t == i + 1).all() for i, t in enumerate(ts))


def test_grown_state_keeps_no_old_storage():
    """A planner's state grown to another capacity holds the memory of its tensors (each padded to 256 bytes) and none
    of the replaced ones', with the values carried over."""
    p = P.FusedPlanner(P.Policy(dense_heads=(1,)), count=False)
    B, Hkv, G, D, cap = 3, 4, 4, 64, 900
    p._alloc(torch.zeros(B, Hkv * G, D), torch.zeros(B, Hkv, 64, D), cap)
    for i, x in enumerate(p.state.values()):
        x.fill_(i + 1)
    old = {x: t.clone() for x, t in p.state.items()}
    p._grow(2 * cap)
    held = {t.untyped_storage().data_ptr(): t.untyped_storage().nbytes() for t in p.state.values()}
    need = sum((t.numel() * t.element_size() + 255) // 256 * 256 for t in p.state.values())
    assert sum(held.values()) <= need
    for x, t in p.state.items():
        if x not in ("part", "idx"):                 # a workspace; rewritten by every step
            assert torch.equal(t[:, :, :cap] if t.dim() > 2 else t, old[x]), x


def test_refusals():
    q, k = torch.zeros(1, 32, 128, dtype=torch.bfloat16), torch.zeros(1, 8, 64, 128, dtype=torch.bfloat16)
    f = torch.zeros(1, 32, 1)
    for call, msg in ((lambda: ext.decode(q, k, k, 0.1), "q must be CUDA bf16"),
                      (lambda: ext.decode(None, k, k, 0.1), "q must be a tensor"),
                      (lambda: ext.vskip1(q, k, k, 0.1, 1e-4), "q must be CUDA bf16"),
                      (lambda: ext.pv(q, k, f, f, f), "v must be a CUDA bf16 tensor"),
                      (lambda: ext.select(f, f, 8, "best", 0.9), "rule must be tau or topp"),
                      (lambda: ext.select(f, f, 8, "topp", 0.9), "blk_max must be contiguous CUDA fp32"),
                      (lambda: ext.update(f, f, f, f, f, f, f, f, 64, 0.9, 2), "blk_max must be contiguous CUDA fp32"),
                      (lambda: ext.plan(q, k, *[f] * 11, 0.1, 0.1, 1, 2, True), "q: CUDA bf16"),
                      (lambda: ext.decode_into(q, k, k, 0.1, {}), "q must be CUDA bf16")):
        with pytest.raises(RuntimeError, match=msg):
            call()


def test_launches_refuse_other_devices():
    """A launch goes to the tensor's own CUDA device: host memory is refused before anything is launched."""
    plan, upd, attn = _native.PlanArgs(), _native.UpdateArgs(), _native.AttnArgs()
    host, q = _native.host(), torch.zeros(1, 32, 128)
    for call in (lambda: ext.launch_update(upd, torch.device("cpu")), lambda: ext.plan_scores(plan, "cpu"),
                 lambda: host.plan(ctypes.addressof(plan), q),
                 lambda: host.merge_update(ctypes.addressof(attn), ctypes.addressof(upd), q)):
        with pytest.raises(ValueError, match="Expected a cuda device, but got: cpu"):
            call()
