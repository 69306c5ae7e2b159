"""Operator surface of the reference's torch extension `kvskip_ext`, on the kvskip_amd C ABI.

Same functions, positional/keyword signatures, defaults, output lists and validation messages as
kernels/kvskip_ext.cpp:327-351 (decode, pv, vskip1, plan, update, read_bw). Outputs are allocated
with torch on the inputs' device; launches go to torch's current stream; nothing synchronises.
Absent outputs are returned as None (the reference returns undefined tensors).

Extra operators with no counterpart in kvskip_ext: block_sums and token_index (the device-side
planner initialisation and token index) and decode_into (decode into caller-owned buffers).

Paged caches (block_table and T; not in the reference): k, v are page pools [num_pages, Hkv, 64, D]
whose page block_table[b, j] (int32 [B, >= ceil(T / 64)] on the device) holds tokens 64 j .. 64 j + 63
of sequence b; T is then required (the tokens, or the capacity with seq_lens).

The checks, allocations and launches of most operators are native (csrc/host.cpp)."""

from __future__ import annotations

import ctypes

import torch

from . import _native
from ._native import AttnArgs, PlanArgs, UpdateArgs

TILE = 64


def _fail(msg: str):
    raise RuntimeError(msg)


def _require(cond: bool, msg: str):
    if not cond:
        _fail(msg)


_host = _native.host      # the native argument checks, allocations and launches (csrc/host.cpp)


def _device_index(device) -> int:
    d = torch.device(device)
    if d.type != "cuda":
        raise ValueError(f"Expected a cuda device, but got: {d}")
    return torch.cuda.current_device() if d.index is None else d.index


def _stream(dev: torch.device):
    return ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream)


def check_kv(t: torch.Tensor, name: str):
    """kernels/kvskip_ext.cpp:12-19."""
    _require(t.is_cuda and t.dtype == torch.bfloat16, f"{name} must be a CUDA bf16 tensor")
    _require(t.dim() == 4, f"{name} must be [B, Hkv, T, D]")
    _require(t.stride(3) == 1, f"{name} must have a contiguous last dim")
    _require(t.stride(2) % 8 == 0 and t.stride(1) % 8 == 0 and t.stride(0) % 8 == 0,
             f"{name} strides must be multiples of 8 elements (16-byte rows)")
    _require(t.data_ptr() % 16 == 0, f"{name} must be 16-byte aligned")
    T, D = t.shape[2], t.shape[3]
    _require((T - 1) * t.stride(2) + D < 2**30, f"{name}: one head's rows must span < 2 GiB")


def check_q(q: torch.Tensor):
    _require(q.is_cuda and q.dtype == torch.bfloat16 and q.dim() == 3, "q must be CUDA bf16 [B, Hq, D]")
    _require(q.stride(2) == 1 and q.stride(1) % 8 == 0 and q.stride(0) % 8 == 0 and q.data_ptr() % 16 == 0,
             "q rows must be 16-byte aligned")


def check_f32(t: torch.Tensor, name: str):
    _require(t.is_cuda and t.dtype == torch.float32 and t.is_contiguous(), f"{name} must be contiguous CUDA fp32")


def _attn_args(q, k, v, scale, B, Hq, Hkv, T, D) -> AttnArgs:
    a = AttnArgs()
    if q is not None:
        a.q = q.data_ptr()
        a.q_sb, a.q_sh = q.stride(0), q.stride(1)
    if k is not None:
        a.k = k.data_ptr()
        a.k_sb, a.k_sh, a.k_st = k.stride(0), k.stride(1), k.stride(2)
    if v is not None:
        a.v = v.data_ptr()
        a.v_sb, a.v_sh, a.v_st = v.stride(0), v.stride(1), v.stride(2)
    a.B, a.Hq, a.Hkv, a.T, a.D = B, Hq, Hkv, T, D
    a.scale = float(scale)
    return a


def decode(q, k, v, scale, block_idx=None, block_cnt=None, stats=False, load_v=True, num_splits=1, stages=2,
           want_f32=False, write_p=False, seq_lens=None, block_table=None, T=None, merge=True, list_partition=0):
    """Split-K decode attention (kernels/kvskip_ext.cpp:25-101).

    Returns [out bf16 [B,Hq,D], lse fp32 [B,Hq], blk_max, blk_sum ([B,Hq,nb] or None), out_f32 (or None),
    P fp16 [B,Hq,nb*64] (write_p) or None].

    seq_lens (not in the reference): int32 [B] on the device, a ragged batch; sequence b attends
    tokens [0, clamp(seq_lens[b], 1, T)) of its view; num_splits is then the per-KV-head split
    budget over the whole batch (>= 2). list_partition (not in the reference; block lists with
    seq_lens): 0 cuts each KV head's lists over the batch, 1 all B * Hkv lists by one chunk length
    (kvskip_attn_args.list_partition).
    block_table, T (not in the reference): a paged cache (the pass with V, MFMA engine).
    merge=False (not in the reference; load_v=False): the split pass alone, no merge launch; the block
    statistics and P are whole, lse is not computed (returned as None)."""
    return _host().decode(q, k, v, scale, block_idx, block_cnt, stats, load_v, num_splits, stages, want_f32, write_p,
                          seq_lens, block_table, T, merge, list_partition)


def decode_into(q, k, v, scale, bufs: dict, block_idx=None, block_cnt=None, stats=False, num_splits=1,
                seq_lens=None, phase=3, block_table=None, T=None, list_partition=0, key_sums=None):
    """decode() into caller-owned buffers, allocating nothing (not in the reference): bufs holds
    out bf16, lse fp32 and, as needed, blk_max / blk_sum fp32 (>= B*Hq*nb elements, written as
    [B, Hq, nb], -inf / 0 where a list skips a block) and part_acc / part_ml fp32
    (>= B*Hq*num_splits*D / *2 elements). The fused planner loop runs its passes this way.
    phase: 3 = the whole op, 1 = the split pass only (its merge left to merge_splits / merge_update),
    2 = that merge alone (given the pass's list_partition). block_table, T: a paged cache.
    key_sums: fp32 [B, Hkv, NBC, D]; a dense pass with stats and seq_lens also writes block_sums' sums of the
    sequences' blocks there (kvskip_attn_args.key_sums; blocks past a sequence's end are left alone)."""
    _host().decode_into(q, k, v, scale, bufs, block_idx, block_cnt, stats, num_splits, seq_lens, phase, block_table, T,
                        list_partition, key_sums)


class DecodeOp:
    """One decode-attention op with its arguments and outputs built once (fixed q, k, v views):
    run() = decode(); splits() then merge() = its two launches (kvskip_decode_splits /
    kvskip_merge_splits), for timing each kernel or placing work between them. Not in the
    reference. Outputs: .out bf16 [B, Hq, D], .lse fp32 [B, Hq]."""

    def __init__(self, q, k, v, scale, num_splits, block_idx=None, block_cnt=None):
        check_q(q)
        check_kv(k, "k")
        check_kv(v, "v")
        _require(2 <= num_splits <= 256, "DecodeOp: num_splits in 2..256")
        B, Hq, D = q.shape
        Hkv, T = k.shape[1], k.shape[2]
        dev = q.device
        f32 = dict(dtype=torch.float32, device=dev)
        self.out = torch.empty(B, Hq, D, dtype=torch.bfloat16, device=dev)
        self.lse = torch.empty(B, Hq, **f32)
        self._keep = [q, k, v, block_idx, block_cnt,
                      torch.empty(B, Hq, num_splits, D, **f32), torch.empty(B, Hq, num_splits, 2, **f32)]
        a = _attn_args(q, k, v, scale, B, Hq, Hkv, T, D)
        if block_idx is not None:
            a.block_idx, a.block_cnt, a.max_blocks = block_idx.data_ptr(), block_cnt.data_ptr(), block_idx.shape[2]
        a.num_splits = int(num_splits)
        a.part_acc, a.part_ml = self._keep[5].data_ptr(), self._keep[6].data_ptr()
        a.out, a.lse = self.out.data_ptr(), self.lse.data_ptr()
        self.args, self.dev = a, dev
        self.lib = _native.lib()

    def _call(self, fn):
        _native.check(fn(ctypes.byref(self.args), 0, 1, _stream(self.dev)))

    def run(self):
        self._call(self.lib.kvskip_decode)

    def splits(self):
        self._call(self.lib.kvskip_decode_splits)

    def merge(self):
        self._call(self.lib.kvskip_merge_splits)


def _decode_args(q, k, v, scale, block_idx, block_cnt, num_splits, out, lse, bmax, bsum, out32, pbuf, part_acc,
                 part_ml, seq_lens=None, block_table=None, T=None, list_partition=0) -> AttnArgs:
    a = AttnArgs()
    _host().attn_block(ctypes.addressof(a), q, k, v, scale, block_idx, block_cnt, num_splits, out, lse, bmax, bsum, out32,
                       pbuf, part_acc, part_ml, seq_lens, block_table, T, list_partition)
    return a


def pv(P, v, blk_scale, block_idx, block_cnt, num_splits=1, want_f32=False, block_table=None, T=None):
    """Two-pass V-skip, pass 2 (kernels/kvskip_ext.cpp:106-146). Returns [out bf16, out_f32 or None].
    block_table, T (not in the reference): v is the page pool of a paged cache."""
    return _host().pv(P, v, blk_scale, block_idx, block_cnt, num_splits, want_f32, block_table, T)


def vskip1(q, k, v, scale, tau, local=2, num_splits=1, want_f32=False, count=False, lse_prev=None,
           block_table=None, T=None, v_keep=None):
    """Single-pass V-skip (kernels/kvskip_ext.cpp:149-195). Returns [out, lse, out_f32 or None, vcount or None].
    block_table, T (not in the reference): a paged cache (the MFMA engine).
    v_keep (not in the reference): uint8 [B, Hkv, ceil(T / 64)] on the device, set to 1 where a block's V
    was read, else 0."""
    return _host().vskip1(q, k, v, scale, tau, local, num_splits, want_f32, count, lse_prev, block_table, T, v_keep)


def plan(q, k, csum, lse_ref, cs_ref, keep, lse_att, age, flags, cs_now, trig, block_idx, block_cnt, scale, delta,
         max_age, local, add_token, idx=None, calib=None, est=None, calib_on=False, calib_kind=0, aix=None,
         part=None, seq_lens=None, seq_lens_out=None, ids=None, idx_out=None, block_table=None, T=None,
         ticket=None):
    """Device-side refresh planner before the pass (kernels/kvskip_ext.cpp:205-267); in place.

    part (not in the reference): fp32 workspace of plan_part_floats(...) elements; with it the
    centroid pass is spread over all compute units (two launches instead of one).
    seq_lens (not in the reference): int32 [B] on the device, a ragged batch over views of
    capacity T (sequence b holds seq_lens[b] tokens; add_token adds each one's last row).
    seq_lens_out (not in the reference): int32 [B] on the device; receives each sequence's length
    this step (for the step's update, which may run later).
    ids, idx_out (not in the reference; need part, and idx None): token ids int32 [B, >= T]; the
    plan finds this step's token-index blocks itself and writes them to idx_out (uint8 [B, NBC]).
    block_table, T (not in the reference): k is the page pool of a paged cache.
    ticket (not in the reference; needs part): int32 [B * Hkv] on the device, zero before the first
    call and left zero by each call; the plan is then one launch (each head decided by its last
    scores workgroup, kvskip_plan_args.ticket). Calls sharing one must not overlap in time."""
    p = _plan_args(q, k, csum, lse_ref, cs_ref, keep, lse_att, age, flags, cs_now, trig, block_idx, block_cnt, scale,
                   delta, max_age, local, add_token, idx, calib, est, calib_on, calib_kind, aix, part, seq_lens,
                   seq_lens_out, ids, idx_out, block_table, T, ticket)
    _host().plan(ctypes.addressof(p), q)


def plan_struct(*plan_args, **plan_kwargs) -> PlanArgs:
    """The argument block of plan(*plan_args, **plan_kwargs), checked (it holds raw pointers)."""
    return _plan_args(*plan_args, **plan_kwargs)


def plan_scores(pargs: PlanArgs, device):
    """plan's first launch alone (kvskip_plan_scores; needs part); its decision then runs in
    decode_splits_planned. Not in the reference."""
    _host().plan_scores(ctypes.addressof(pargs), _device_index(device))


DECIDE_PLAN, DECIDE_LISTS, DECIDE_POST = 0, 1, 2      # kvskip_plan_args.decide_mode


def decode_splits_planned(q, k, v, scale, bufs: dict, pargs: PlanArgs, num_splits, update: UpdateArgs | None = None,
                          seq_lens=None, block_table=None, T=None):
    """plan's decision and the masked + statistics split pass in one launch (kvskip_decode_splits_planned;
    after plan_scores(pargs)); the whole op when num_splits == 1. The layer's update must advance the
    age (update_struct(..., age=...)). update: another layer's update to carry, or None. seq_lens: the
    plan's (one sequence, B 1). pargs.decide_mode picks the decision (DECIDE_PLAN, DECIDE_LISTS,
    DECIDE_POST), pargs.slot_base / slot_count the partial slots the pass writes."""
    _host().splits_planned(q, k, v, scale, bufs, None, None, ctypes.addressof(pargs), num_splits,
                           None if update is None else ctypes.addressof(update), seq_lens, block_table, T, 0)


def _plan_args(q, k, csum, lse_ref, cs_ref, keep, lse_att, age, flags, cs_now, trig, block_idx, block_cnt, scale, delta,
         max_age, local, add_token, idx=None, calib=None, est=None, calib_on=False, calib_kind=0, aix=None,
         part=None, seq_lens=None, seq_lens_out=None, ids=None, idx_out=None, block_table=None, T=None,
               ticket=None):
    """kvskip_plan_args of plan(), validated. block_table, T: a paged cache."""
    p = PlanArgs()
    _host().plan_block(ctypes.addressof(p), q, k, csum, lse_ref, cs_ref, keep, lse_att, age, flags, cs_now, trig, block_idx,
                       block_cnt, scale, delta, max_age, local, add_token, idx, calib, est, calib_on, calib_kind, aix, part,
                       seq_lens, seq_lens_out, ids, idx_out, block_table, T, ticket)
    return p


def plan_part_floats(B, Hq, Hkv, NBC) -> int:
    """fp32 elements of plan()'s `part` workspace for a state of capacity NBC blocks."""
    return int(_native.lib().kvskip_plan_part_floats(int(B), int(Hq), int(Hkv), int(NBC)))


def _update_args(blk_max, blk_sum, trig, cs_now, keep, lse_ref, cs_ref, lse_att, T, level, local, flags=None,
                 idx=None, est=None, calib=None, calib_rate=0.0, calib_free=False, calib_kind=0, aix=None,
                 aix_thr=0.0, list_stats=False, seq_lens=None, age=None) -> UpdateArgs:
    """kvskip_update_args of update() (kernels/kvskip_ext.cpp:270-319), validated."""
    p = UpdateArgs()
    _host().update_block(ctypes.addressof(p), blk_max, blk_sum, trig, cs_now, keep, lse_ref, cs_ref, lse_att, T, level, local,
                         flags, idx, est, calib, calib_rate, calib_free, calib_kind, aix, aix_thr, list_stats, seq_lens, age)
    return p


def update(blk_max, blk_sum, trig, cs_now, keep, lse_ref, cs_ref, lse_att, T, level, local, flags=None, idx=None,
           est=None, calib=None, calib_rate=0.0, calib_free=False, calib_kind=0, aix=None, aix_thr=0.0,
           list_stats=False, seq_lens=None, age=None):
    """Device-side refresh planner after the pass (kernels/kvskip_ext.cpp:270-319); in place.

    list_stats (not in the reference): blk_max / blk_sum hold values only for the blocks of this
    step's plan (the masked pass ran on unfilled buffers); the kernel derives the read set from
    trig, keep, flags and idx and ignores the rest. Needs flags (and idx if the plan had one).
    age (not in the reference): advance the plan's age here (after decode_splits_planned)."""
    p = _update_args(blk_max, blk_sum, trig, cs_now, keep, lse_ref, cs_ref, lse_att, T, level, local, flags, idx,
                     est, calib, calib_rate, calib_free, calib_kind, aix, aix_thr, list_stats, seq_lens, age)
    launch_update(p, keep.device)


def merge_update(q, k, v, scale, bufs: dict, num_splits, update_args: tuple, update_kwargs: dict,
                 block_idx=None, block_cnt=None, seq_lens=None, block_table=None, T=None, list_partition=0):
    """The split merge of a decode_into(..., phase=1) pass (same q, k, v, bufs, list, num_splits >= 2)
    and update(*update_args, **update_kwargs), in one launch (kvskip_merge_update; not in the
    reference). block_table, T: the pass's paged cache; list_partition: the pass's."""
    _require(num_splits >= 2, "merge_update needs num_splits >= 2")
    a = _decode_args(q, k, v, scale, block_idx, block_cnt, num_splits, bufs["out"], bufs["lse"], None, None, None,
                     None, bufs["part_acc"], bufs["part_ml"], seq_lens, block_table, T, list_partition)
    u = _update_args(*update_args, **update_kwargs)
    _host().merge_update(ctypes.addressof(a), ctypes.addressof(u), q)


def update_struct(*update_args, **update_kwargs) -> UpdateArgs:
    """The argument block of update(*update_args, **update_kwargs), checked, for a later launch
    (decode_splits_update, launch_update); it holds raw pointers, so the tensors must outlive its use."""
    return _update_args(*update_args, **update_kwargs)


def launch_update(update: UpdateArgs, device):
    """update() from an update_struct, on the current stream of `device`."""
    _host().update(ctypes.addressof(update), _device_index(device))


def decode_splits_update(q, k, v, scale, bufs: dict, block_idx, block_cnt, num_splits, update: UpdateArgs,
                         seq_lens=None, block_table=None, T=None, list_partition=0):
    """decode_into(..., stats=True, phase=1) over a block list (the whole op when num_splits == 1)
    and the update of ANOTHER layer (an update_struct), in one launch (kvskip_decode_splits_update;
    not in the reference). The update reads only its own layer's buffers. block_table, T: a paged cache."""
    _host().splits_update(q, k, v, scale, bufs, block_idx, block_cnt, num_splits, ctypes.addressof(update), seq_lens,
                          block_table, T, list_partition)


def read_bw(x, out, blocks):
    """Streaming read of x (bandwidth ceiling), kernels/kvskip_ext.cpp:321-325."""
    _require(x.is_cuda and x.is_contiguous() and (x.numel() * x.element_size()) % 16 == 0,
             "x: contiguous CUDA, 16-byte multiple")
    dev = x.device
    with torch.cuda.device(dev):
        _native.check(_native.lib().kvskip_read(x.data_ptr(), x.numel() * x.element_size(), out.data_ptr(),
                                                int(blocks), _stream(dev)))


def _seq_lens_ptr(seq_lens, B):
    if seq_lens is None:
        return None
    _require(seq_lens.is_cuda and seq_lens.dtype == torch.int32 and seq_lens.is_contiguous()
             and seq_lens.numel() == B, "seq_lens: contiguous CUDA int32 [B]")
    return seq_lens.data_ptr()


def block_sums(k, NBC, out=None, seq_lens=None, block_table=None, T=None):
    """Per-block key sums [B, Hkv, NBC, D] fp32 of k [B, Hkv, T, D] (blocks >= nb are zero);
    seq_lens: ragged batch (sequence b sums its first seq_lens[b] rows). block_table, T (not in the
    reference): k is a page pool [num_pages, Hkv, 64, D] of a paged cache."""
    check_kv(k, "k")
    if block_table is None:
        B, Hkv, T, D = k.shape
        bt = (None, 0, 0)
    else:
        _require(T is not None and k.dim() == 4 and k.shape[2] == TILE, "paged cache: k [num_pages, Hkv, 64, D] and T")
        _require(block_table.is_cuda and block_table.dtype == torch.int32 and block_table.dim() == 2
                 and block_table.stride(1) == 1, "block_table: int32 [B, >= ceil(T / 64)] on the device, rows contiguous")
        B, (Hkv, D), T = block_table.shape[0], (k.shape[1], k.shape[3]), int(T)
        bt = (block_table.data_ptr(), block_table.stride(0), k.shape[0])
    _require((T + TILE - 1) // TILE <= NBC, "block capacity exceeded")
    if out is None:
        out = torch.empty(B, Hkv, NBC, D, dtype=torch.float32, device=k.device)
    check_f32(out, "csum")
    _require(tuple(out.shape) == (B, Hkv, NBC, D), "csum: [B, Hkv, NBC, D]")
    with torch.cuda.device(k.device):
        _native.check(_native.lib().kvskip_block_sums(k.data_ptr(), k.stride(0), k.stride(1), k.stride(2), B, Hkv, T, D,
                                                      out.data_ptr(), NBC, _seq_lens_ptr(seq_lens, B), *bt,
                                                      _stream(k.device)))
    return out


def token_index(ids, T, NBC, out=None, seq_lens=None):
    """Token-index blocks [B, NBC] uint8 of the step whose current token is ids[:, T-1]
    (ids[b, seq_lens[b] - 1] with seq_lens: ragged batch)."""
    _require(ids.is_cuda and ids.dtype == torch.int32 and ids.dim() == 2 and ids.stride(1) == 1,
             "ids: CUDA int32 [B, >= T]")
    B = ids.shape[0]
    _require(ids.shape[1] >= T >= 1, "ids: CUDA int32 [B, >= T]")
    if out is None:
        out = torch.empty(B, NBC, dtype=torch.uint8, device=ids.device)
    _require(out.dtype == torch.uint8 and out.is_contiguous() and tuple(out.shape) == (B, NBC), "idx: uint8 [B, NBC]")
    with torch.cuda.device(ids.device):
        _native.check(_native.lib().kvskip_token_index(ids.data_ptr(), ids.stride(0), B, int(T), out.data_ptr(), NBC,
                                                       _seq_lens_ptr(seq_lens, B), _stream(ids.device)))
    return out


def select(blk_max, blk_sum, Hkv, rule, value, local=2, keep=None, block_idx=None, block_cnt=None, blk_scale=None):
    """GQA-union block selection on the device (kvskip_select; not in kvskip_ext): from per-block
    statistics [B, Hq, nb] fp32, rule "tau" (weight >= value) or "topp" (fewest blocks reaching value)
    per query head, the union over each KV head's group plus block 0 and the `local` newest blocks.
    Fills whichever outputs are given: keep uint8 [B, Hkv, nb], block_idx / block_cnt int32 ([B, Hkv, nb]
    kept first ascending, [B, Hkv]) and blk_scale fp32 [B, Hkv, nb, G] (exp(blk_max - lse over the kept
    blocks), 0 off the set)."""
    _host().select(blk_max, blk_sum, Hkv, rule, value, local, keep, block_idx, block_cnt, blk_scale)


def pv_select(P, v, blk_max, blk_sum, rule, value, local=2, num_splits=1, want_f32=False, keep=None,
              block_idx=None, block_cnt=None, blk_scale=None):
    """Two-pass V-skip pass 2 with the selection in it (kvskip_pv_select; not in kvskip_ext): select()
    on pass 1's statistics, then pv() over the kept blocks and their scales, in one launch (+ the split
    merge), the same results bit for bit. Contiguous cache. keep / block_idx / block_cnt / blk_scale:
    select()'s outputs, filled if given. Returns [out bf16, out_f32 or None]."""
    return _host().pv_select(P, v, blk_max, blk_sum, rule, value, local, num_splits, want_f32, keep, block_idx, block_cnt,
                             blk_scale)


def block_list(keep, block_idx, block_cnt):
    """The kept-first block list of a keep mask [B, Hkv, nb] (bool or uint8) on the device
    (kvskip_block_list; not in kvskip_ext): block_idx int32 [B, Hkv, nb] (kept blocks ascending, then
    the others ascending), block_cnt int32 [B, Hkv]."""
    _require(keep.is_cuda and keep.dtype in (torch.bool, torch.uint8) and keep.dim() == 3 and keep.is_contiguous(),
             "keep: contiguous bool / uint8 [B, Hkv, nb] on the device")
    B, Hkv, nb = keep.shape
    _require(block_idx.dtype == torch.int32 and block_idx.is_contiguous() and tuple(block_idx.shape) == (B, Hkv, nb),
             "block_idx: int32 [B, Hkv, nb]")
    _require(block_cnt.dtype == torch.int32 and block_cnt.is_contiguous() and tuple(block_cnt.shape) == (B, Hkv),
             "block_cnt: int32 [B, Hkv]")
    dev = keep.device
    with torch.cuda.device(dev):
        _native.check(_native.lib().kvskip_block_list(keep.data_ptr(), B, Hkv, nb, block_idx.data_ptr(),
                                                      block_cnt.data_ptr(), _stream(dev)))
