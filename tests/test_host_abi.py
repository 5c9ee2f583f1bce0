"""CPU-side checks of the shipped library: it loads, exports every symbol the
header declares, and its host-side geometry (tile plan, top-k rule, block-causal
predicate, shard ranges) equals the oracle's restatement of the reference and
the reference's own known answers. No GPU calls.
"""
import ctypes
import os
import re

import numpy as np
import pytest

from util import ROOT

import fv_sdpa
from fv_sdpa import _lib


def test_library_exports_every_declared_symbol():
    header = open(os.path.join(ROOT, "include", "fv_sdpa_hip.h")).read()
    header = re.sub(r"/\*.*?\*/", "", header, flags=re.S)
    declared = set(re.findall(r"\b(fv_[a-z0-9_]+)\s*\(", header))
    assert len(declared) >= 20
    assert declared == set(_lib.SIGNATURES), declared ^ set(_lib.SIGNATURES)
    lib = ctypes.CDLL(_lib.LIB_PATH)
    for name in declared:
        assert hasattr(lib, name), name
    assert fv_sdpa.lib().fv_sdpa_arch() == b"gfx950"
    assert isinstance(fv_sdpa.lib().fv_sdpa_last_error(), bytes)   # "" until a call of this thread fails


def test_supported_table():
    # rt/attn.rs:932-960
    ok = fv_sdpa.sdpa_supported
    assert ok(1, 40, 38001, 38001, 128) and ok(2, 32, 4097, 1024, 128) and ok(1, 1, 1, 1, 128)
    assert ok(1, 32, 125, 1, 64)
    for d in (32, 80, 96, 256, 384):
        assert not ok(1, 8, 1024, 1024, d)
    assert not ok(1, 8, 0, 1024, 128) and not ok(1, 8, 1024, 0, 128)
    assert not ok(0, 8, 1024, 1024, 128) and not ok(2, 40000, 64, 64, 128)


def test_log2_domain_scale_predicate():
    # scale = ln 2 as f32 times the library's f32 log2(e) rounds to exactly one; its neighbours and the
    # usual 1/sqrt(d) do not
    is_log2 = fv_sdpa.lib().fv_sdpa_is_log2_domain_scale
    ln2 = np.float32(np.log(2.0))
    assert is_log2(float(ln2)) == 1
    assert is_log2(float(np.nextafter(ln2, np.float32(0)))) == 0 and is_log2(float(np.nextafter(ln2, np.float32(1)))) == 0
    for d in (64, 128):
        assert is_log2(1.0 / np.sqrt(d)) == 0
    header = open(os.path.join(ROOT, "include", "fv_sdpa_hip.h")).read()
    m = re.search(r"#define FV_SDPA_SCALE_LOG2_DOMAIN ([0-9.]+)f", header)
    assert m and np.float32(float(m.group(1))) == ln2
    rust = open(os.path.join(ROOT, "rust", "fastvideo-hip-sdpa", "src", "ffi.rs")).read()
    m = re.search(r"FV_SDPA_SCALE_LOG2_DOMAIN: f32 = ([0-9._]+);", rust)
    assert m and np.float32(float(m.group(1).replace("_", ""))) == ln2


@pytest.mark.parametrize("grid", [(4, 4, 4), (33, 28, 52), (3, 5, 7), (1, 1, 1), (1, 1, 5), (21, 30, 52), (32, 32, 32)])
def test_tile_plan_equals_oracle(oracle, grid):
    got, want = fv_sdpa.TilePlan(grid), oracle.TilePlan(grid)
    assert got.tiles == want.tiles and got.seq == want.seq and got.padded == want.padded
    assert np.array_equal(got.slot_src, want.slot_src)
    assert np.array_equal(got.token_slot, want.token_slot)
    assert np.array_equal(got.block_sizes.astype(np.uint32), want.block_sizes)


def test_tile_plan_known_answers():
    p = fv_sdpa.TilePlan((1, 1, 5))
    assert list(p.block_sizes) == [4, 1] and list(p.slot_src[:4]) == [0, 1, 2, 3] and p.slot_src[64] == 4
    assert (p.slot_src[4:64] == -1).all()
    assert fv_sdpa.TilePlan((21, 30, 52)).num_tiles == 624
    with pytest.raises(ValueError):
        fv_sdpa.TilePlan((4, 0, 4))


def test_topk_rule(oracle):
    for sp, n, want in [(0.8, 819, 164), (0.0, 819, 819), (1.0, 819, 1), (0.9, 10, 1), (0.8, 624, 125), (0.875, 512, 64)]:
        assert fv_sdpa.topk_for(sp, n) == want == oracle.topk_for(sp, n)


def test_block_causal_host_helpers(oracle):
    for bt, win, sink in [(5, 2, 1), (1, 0, 0), (7, 0, 2), (4, 1, 0), (0, 0, 0), (60, 3, 1)]:
        assert np.array_equal(fv_sdpa.block_causal_dense_mask(bt, win, sink, 50, 61),
                              oracle.block_causal_dense_mask(bt, win, sink, 50, 61))
    for fpb, las, ft in [(3, -1, 1560), (3, 4, 6), (3, 6, 10), (1, 2, 7), (1, -1, 3), (3, 0, 5)]:
        assert fv_sdpa.block_causal_for(fpb, las, ft) == oracle.block_causal_for(fpb, las, ft)
    assert fv_sdpa.block_causal_for(3, 4, 6) is None
    assert fv_sdpa.block_causal_allows(5, 2, 1, 23, 0) and not fv_sdpa.block_causal_allows(5, 2, 1, 23, 5)


def test_shard_ranges(oracle):
    assert fv_sdpa.shard_ranges(10, 2) == [(0, 5), (5, 5)]
    assert fv_sdpa.shard_ranges(11, 2) == [(0, 6), (6, 5)]
    assert fv_sdpa.shard_ranges(32760, 8) == oracle.shard_ranges(32760, 8)


def test_backend_parses_like_the_reference():
    # rt/sdpa_rule.rs:593-604
    for v in ("dense", "cublas", "flash", "host", "sparse"):
        assert fv_sdpa.parse_backend(v) == v
    for v in ("", "fused", " cublas", "dense "):
        assert fv_sdpa.parse_backend(v) == "dense", v
    assert fv_sdpa.backend() == fv_sdpa.parse_backend(os.environ.get("FASTVIDEO_SDPA", "dense").lower())
    with fv_sdpa.with_backend("cublas"):
        assert fv_sdpa.backend() == "cublas"
    assert fv_sdpa.backend() == fv_sdpa.parse_backend(os.environ.get("FASTVIDEO_SDPA", "dense").lower())


def test_shapes_agree_only_when_k_and_v_match_q():
    # rt/sdpa_rule.rs:624-651
    assert fv_sdpa.shape_of((1, 2, 5, 64), (1, 2, 7, 64), (1, 2, 7, 64)) == (5, 7, (1, 2, 5, 7, 64))
    assert fv_sdpa.shape_of((1, 2, 5, 64), (1, 2, 7, 64), (1, 2, 6, 64))[2] is None
    assert fv_sdpa.shape_of((1, 2, 5, 64), (1, 3, 7, 64), (1, 3, 7, 64))[2] is None
    assert fv_sdpa.shape_of((1, 2, 5, 64), (1, 2, 7, 32), (1, 2, 7, 32))[2] is None


def test_dense_route_collapsed():
    # rt/sdpa_rule.rs:409-437 without the cuDNN / cuBLAS / Sage / f32-flash steps
    s = ((1, 12, 320, 128),) * 3
    assert fv_sdpa.dense_route(*s) == ["fused", "composed"]
    assert fv_sdpa.dense_route(*s, masked=True) == ["composed"]
    for b in ("cublas", "flash"):
        assert fv_sdpa.dense_route(*s, backend_name=b) == ["composed"]
    for b in ("host", "sparse"):
        assert fv_sdpa.dense_route(*s, backend_name=b) == ["retired"]
        assert fv_sdpa.dense_route(*s, masked=True, backend_name=b) == ["composed"]   # masked calls never look


@pytest.mark.parametrize("bt,win,sink,sq,sk", [
    (256, 1, 0, 512, 256),      # the second query tile sees no key at all
    (100, 2, 0, 1000, 300), (100, 2, 1, 1000, 300), (64, 0, 0, 700, 130), (1560, 0, 0, 4680, 4680),
    (1560, 2, 1, 6240, 4680), (7, 3, 2, 900, 200), (300, 1, 0, 2000, 500), (128, 1, 3, 1024, 4096),
    (50, 4, 0, 257, 1), (1000, 1, 0, 513, 64)])
def test_block_causal_tile_walk_covers_every_visible_key(bt, win, sink, sq, sk):
    """The key-tile ranges the fused block-causal kernel walks (the function the kernel itself runs):
    ascending, disjoint, inside the key tiles, and covering every key that rt/attn.rs:449-453 lets any
    query of the tile see; a tile whose walk is empty has no visible key at all."""
    lib = fv_sdpa.lib()
    nkt = (sk + 63) // 64
    q = np.arange(sq)[:, None]
    k = np.arange(sk)[None, :]
    tq, tk = q // bt, k // bt
    vis = (tk < sink) | ((tk <= tq) & ((win == 0) | (tq - tk < win)))
    empty_tiles = 0
    for q0 in range(0, sq, 256):
        out = (ctypes.c_int * 4)()
        assert lib.fv_block_causal_tile_walk(bt, win, sink, sq, sk, q0, out) == 0
        n0, a1, n1, total = list(out)
        assert 0 <= n0 <= a1 and n1 >= 0 and a1 + n1 <= nkt and total == n0 + n1
        walked = np.zeros(nkt, bool)
        walked[:n0] = True
        walked[a1:a1 + n1] = True
        need = vis[q0:q0 + 256].any(axis=0)                       # keys some query of the tile sees
        need_tiles = np.zeros(nkt, bool)
        need_tiles[np.nonzero(need)[0] // 64] = True
        assert not (need_tiles & ~walked).any(), (q0, list(out))
        if total == 0:
            assert not need.any()
            empty_tiles += 1
    if (bt, win, sink, sq, sk) == (256, 1, 0, 512, 256):
        assert empty_tiles == 1
    # parameters the kernel declines
    out = (ctypes.c_int * 4)()
    assert lib.fv_block_causal_tile_walk(0, 0, 0, 256, 256, 0, out) == _lib.FV_DECLINED
    assert lib.fv_block_causal_tile_walk(64, 0, 0, 256, 256, 100, out) == _lib.FV_DECLINED


def _fake_tensor(shape, bf16, addr=0x1000):
    """A descriptor whose pointer is never dereferenced on the host: for calls that must fail before a launch."""
    from fv_sdpa.sdpa import _FvTensor

    t = _FvTensor()
    t.data, t.dtype, t.rank, t.plane_rows = addr, int(bf16), len(shape), 0
    for i, s in enumerate(shape):
        t.shape[i] = s
    return t


def _rt_call(q, k, v, kind=0, mask=None):
    from fv_sdpa.sdpa import _FvPlan, _FvTensor

    lib = fv_sdpa.lib()
    p = _FvPlan()
    p.kind, p.kv_flash = kind, -1
    if mask is not None:
        p.mask = ctypes.pointer(mask)
    out = _FvTensor()
    rc = lib.fv_rt_sdpa(ctypes.byref(q), ctypes.byref(k), ctypes.byref(v), ctypes.byref(p), ctypes.byref(out), None)
    return rc, lib.fv_sdpa_last_error().decode()


def test_rt_sdpa_refuses_before_any_device_work():
    """Argument errors of the one entry are host decisions: they come back as -hipErrorInvalidValue with the
    reference's message and touch no device (rt/sdpa.rs:141-164, rt/tensor.rs:1655-1667)."""
    q = _fake_tensor((1, 2, 8, 128), True)
    rc, msg = _rt_call(_fake_tensor((2, 8, 128), True), q, q)
    assert rc == -1 and msg == "sdpa expects BHSD"
    # a masked composed call with no keys: refused, and the mask's batch count is never divided by sq * sk = 0
    k0 = _fake_tensor((1, 2, 0, 128), False)
    rc, msg = _rt_call(_fake_tensor((1, 2, 8, 128), False), k0, k0, kind=1, mask=_fake_tensor((8, 0), False))
    assert rc == -1 and msg == "sdpa: no keys"
    rc, msg = _rt_call(q, q, q, kind=99)
    assert rc == -1 and "unknown plan kind" in msg


def test_rt_sdpa_reports_an_allocation_failure_with_its_own_code():
    """Without a device the first allocation fails: the entry returns that hipError_t (not the code of a
    refused argument) and the message says which step failed. Skipped where a GPU is present (the
    allocation would succeed and the fake operands must never reach a kernel)."""
    import torch

    if torch.cuda.device_count() > 0:
        pytest.skip("needs a host without a GPU")
    q = _fake_tensor((1, 2, 8, 128), True)
    rc, msg = _rt_call(q, q, q)
    assert rc < -1 and msg.startswith("sdpa: device allocation failed: ")
    # no query rows + a mask: an empty result is allocated (no division by sq * sk = 0 on the way)
    q0 = _fake_tensor((1, 2, 0, 128), False)
    kv = _fake_tensor((1, 2, 8, 128), False)
    rc, msg = _rt_call(q0, kv, kv, kind=1, mask=_fake_tensor((0, 8), False))
    assert rc < -1 and msg.startswith("sdpa: device allocation failed: ")


@pytest.mark.parametrize("shape,kind,launch", [
    ((24, 3000, 3000, 128), 0, "flash_fwd_pp2<dense>"),    # the last round of query tiles split
    ((12, 1560, 32760, 128), 0, "flash_fwd_pp2<dense>"),   # every tile split
    ((12, 4096, 4096, 128), 1, "sdpa_composed")])          # a tail cut by key ranges
def test_no_memory_for_partial_results_is_no_error(shape, kind, launch):
    """Without a device every allocation fails. A call into the caller's result buffer whose split partial results get
    no memory goes on unsplit, to the launch (which then reports that there is no device). Skipped where a GPU is
    present: the fake operands must never reach a kernel."""
    import torch
    from fv_sdpa.sdpa import _FvPlan

    if torch.cuda.device_count() > 0:
        pytest.skip("needs a host without a GPU")
    lib = fv_sdpa.lib()
    h, sq, sk, d = shape
    q, k, v = (_fake_tensor((1, h, s, d), kind == 0) for s in (sq, sk, sk))
    p = _FvPlan()
    p.kind, p.kv_flash = kind, -1
    ref = ctypes.byref
    need = (ctypes.c_size_t * 2)()
    assert lib.fv_rt_sdpa_need(ref(q), ref(k), ref(v), ref(p), need) == 0 and need[1] > 0
    rc = lib.fv_rt_sdpa_into(ref(q), ref(k), ref(v), ref(p), 0x1000, h * sq * d * (2 if need[0] else 4), None, 0, None)
    msg = lib.fv_sdpa_last_error().decode()
    assert rc < -1 and launch in msg and "allocation" not in msg, msg


@pytest.mark.parametrize("shape,act16,split", [
    ((24, 3000, 6100, 64), True, True), ((24, 3000, 2300, 64), True, False), ((24, 3000, 2400, 64), True, True),
    ((40, 2000, 3000, 64), True, False), ((40, 2000, 3200, 64), True, True), ((12, 8000, 6100, 64), True, False),
    ((12, 6000, 1500, 128), True, True), ((12, 6000, 1400, 128), True, False), ((12, 8000, 1500, 128), True, False),
    ((38, 1700, 1300, 128), True, True), ((24, 3000, 2200, 64), False, True), ((12, 6000, 1300, 128), False, True)])
def test_a_last_round_of_few_tiles_is_split(shape, act16, split):
    """A few query tiles past whole rounds of the CUs, on walks long enough, are shared out by key ranges (partial results
    in the workspace), whatever kernel takes the walk otherwise; f32 results, which have one kernel, sooner. Past the lines
    the split is faster by up to a seventh (24 x 3000 x 6100 x 64)."""
    from fv_sdpa.sdpa import _FvPlan

    lib, ref, need = fv_sdpa.lib(), ctypes.byref, (ctypes.c_size_t * 2)()
    h, sq, sk, d = shape
    q, k = _fake_tensor((1, h, sq, d), True), _fake_tensor((1, h, sk, d), True)
    p = _FvPlan()
    p.kv_flash = -1
    with fv_sdpa.with_bf16_act(act16):
        assert lib.fv_rt_sdpa_need(ref(q), ref(k), ref(k), ref(p), need) == 0
    assert (need[1] > 0) == split, need[1]


def test_every_fused_kernel_has_a_form_for_the_log2_domain():
    """What fv_sdpa_log2_domain_launches counts is launches of kernels without the multiply of every score: each fused
    kernel is built with and without it (the kernels' symbols, mangled names of their templates)."""
    with open(fv_sdpa._lib.LIB_PATH, "rb") as f:
        text = f.read()
    for d in (64, 128):
        for masked in (0, 1):
            for form in (0, 1):
                assert b"flash_fwd_pp2ILi2ELb%dELi%dELb%dE" % (masked, d, form) in text
                assert b"flash_fwd_duoILb%dELi%dELb%dE" % (masked, d, form) in text
        for waves in (4, 8):
            for form in (0, 1):
                assert b"sdpa_short_kernelILi%dELi1ELi%dELb%dE" % (d // 16, waves, form) in text


@pytest.mark.parametrize("kind", [2, 3])
def test_a_masked_call_keeps_nothing_in_a_workspace_that_is_not_its_own(kind):
    """Two long masked calls on bf16 operands may share a workspace on two streams: only a plan that says that the
    workspace is its own (256) asks for the queue's memory. The flag belongs to these two kinds."""
    from fv_sdpa.sdpa import _FvPlan

    lib, ref, need = fv_sdpa.lib(), ctypes.byref, (ctypes.c_size_t * 2)()
    q, k = _fake_tensor((1, 40, 32760, 128), True), _fake_tensor((1, 40, 32760, 128), True)
    p = _FvPlan()
    p.kv_flash = -1
    p.block_tokens = p.frame_tokens = 1560
    p.frames = 21
    for flag, bytes_ in ((0, 0), (256, 1024)):
        p.kind = kind | flag
        assert lib.fv_rt_sdpa_need(ref(q), ref(k), ref(k), ref(p), need) == 0
        assert need[1] == bytes_, (flag, need[1])
    for other in (0, 1, 4):
        p.kind = other | 256
        assert lib.fv_rt_sdpa_need(ref(q), ref(k), ref(k), ref(p), need) == -1


# (kind, heads, frame, frames, window or chunk, sink or radius, channels, whether its items come from the queue)
QUEUED = [
    (2, 40, 1560, 21, 0, 0, 128, True),      # causal, the mean walk half the longest
    (2, 12, 1560, 21, 0, 0, 128, False),     # six rounds
    (2, 40, 1560, 21, 0, 0, 64, False),
    (2, 40, 1560, 21, 4, 1, 128, True),      # a window: walks of one length, long ...
    (2, 12, 1560, 32, 1, 0, 128, False),     # ... and short
    (2, 12, 1560, 32, 1 << 62, 1 << 62, 128, True),
    (3, 12, 1560, 32, 5, 1, 128, True),
    (3, 40, 880, 18, 5, 2, 128, True),       # the window covers the clip
    (3, 12, 1560, 60, 0, 2, 128, False),     # the first and last frame's walks are much longer than the others
    (3, 40, 390, 40, 0, 0, 128, False),
    (3, 12, 1560, 32, 1 << 62, 1 << 62, 128, True),
]


@pytest.mark.parametrize("kind,h,frame,frames,a,b,d,queued", QUEUED)
def test_which_masked_calls_ask_for_the_queue(kind, h, frame, frames, a, b, d, queued):
    """Eight rounds of query tiles are not enough: walks of very unequal length end late where the queue's lists go head by
    head (12 heads 60 x 1560, radius 2: 8.3 ms instead of 6.6), short ones do not gain."""
    from fv_sdpa.sdpa import _FvPlan

    need = (ctypes.c_size_t * 2)()
    q = _fake_tensor((1, h, frame * frames, d), True)
    p = _FvPlan()
    p.kv_flash, p.kind = -1, kind | 256
    if kind == 2:
        p.block_tokens, p.window, p.sink = frame, a, b
    else:
        p.frame_tokens, p.frames, p.chunk, p.radius = frame, frames, a, b
    assert fv_sdpa.lib().fv_rt_sdpa_need(*[ctypes.byref(q)] * 3, ctypes.byref(p), need) == 0
    assert need[1] == (1024 if queued else 0)


def test_need_is_host_arithmetic_at_any_shape():
    """fv_rt_sdpa_need answers for shapes the call itself refuses (no keys, no queries, no heads, lengths past every
    limit), for every kind of plan and either type: no division by a count of zero, and a workspace of zero or of the
    order of the operands. In a process of its own, which a failure would end."""
    out = _in_subprocess("sys.path.insert(0, %r)" % os.path.join(ROOT, "tests") + """
import ctypes, itertools
from test_host_abi import _fake_tensor
import fv_sdpa
from fv_sdpa.sdpa import _FvPlan
lib, ref, need, n = fv_sdpa.lib(), ctypes.byref, (ctypes.c_size_t * 2)(), 0
sizes = (0, 1, 31, 128, 4096, 75600, 1 << 31, 1 << 40, 1 << 63)
for h, sq, sk, d, bf16, kind in itertools.product((0, 1, 12, 70000), sizes, sizes, (0, 1, 64, 128, 200), (False, True), range(5)):
    q, k = _fake_tensor((1, h, sq, d), bf16), _fake_tensor((1, h, sk, d), bf16)
    p = _FvPlan()
    p.kind, p.kv_flash = kind, -1
    assert lib.fv_rt_sdpa_need(ref(q), ref(k), ref(k), ref(p), need) == 0
    if h * d * (sq + sk) < 1 << 50:
        assert need[1] <= 20 * 4 * h * (sq + 2 * sk + 256) * d + 4096, (h, sq, sk, d, bf16, kind, need[1])
    n += 1
print(n)
""", {})
    assert int(out) == 4 * 9 * 9 * 5 * 2 * 5


@pytest.mark.parametrize("scale", [None, 0.125, 1e40, -1e300, float("inf"), np.float32(0.5), 3])
@pytest.mark.parametrize("numbers", [(1560, 0, 1), (-1, 4, 0), (16, -2, 2**64 + 3), (np.int64(7), 2**63, 0)])
def test_packed_plans_hold_what_the_c_structure_would(scale, numbers):
    """Numbers that do not fit their fields are no Python errors: they reach the library as C has them."""
    from fv_sdpa.sdpa import Plan, _FvPlan, _plan_bytes

    for plan in (Plan.block_causal(scale, fv_sdpa.BlockCausal(*numbers)),
                 Plan.vdn_window(scale, fv_sdpa.VdnWindow(numbers[1], numbers[0], 5, 0, numbers[2])), Plan.kv_window_with(True)):
        want = _FvPlan()
        want.kind = plan.kind
        want.has_scale, want.scale = (0, 0.0) if plan.scale is None else (1, float(plan.scale))
        if plan.causal is not None:
            want.block_tokens, want.window, want.sink = numbers
        if plan.window is not None:
            want.video_start, want.frame_tokens, want.frames, want.chunk, want.radius = plan.window._args()
        want.kv_flash = -1 if plan.kv_flash is None else int(plan.kv_flash)
        got = _FvPlan.from_buffer_copy(_plan_bytes(plan, 0))
        for name, _ in _FvPlan._fields_[:3] + _FvPlan._fields_[4:]:
            assert getattr(got, name) == getattr(want, name), name
    with pytest.raises(TypeError):
        _plan_bytes(Plan.block_causal(None, fv_sdpa.BlockCausal(1.5)), 0)


def test_scans_longer_than_one_launch_are_refused():
    """2^32 work-items and more in a launch are cut off by the runtime without an error: these entries decline instead
    (host arithmetic; the fake operands reach no kernel)."""
    lib, x = fv_sdpa.lib(), 0x1000
    seq = 1 << 26
    assert lib.fv_split_heads_bhsd(x, x, 1, 1, seq, 4, 128, 512, 0, None) == _lib.FV_DECLINED
    assert lib.fv_merge_heads(x, x, 1, 1, 4, seq, 128, None) == _lib.FV_DECLINED
    assert lib.fv_rope_bhsd(x, 1, seq, x, x, 0, x, 1, seq, 4, seq, 128, None) == _lib.FV_DECLINED
    assert lib.fv_qk_norm_rope_bhsd(x, 1, x, 0, None, None, x, 1, 1, seq, 1, 8, 8, 0, 1e-6, 1.0, None) == _lib.FV_DECLINED


def test_log_level_parses_like_the_reference():
    # rt/log.rs:17-37
    parse = fv_sdpa.lib().fv_rt_parse_log_level
    for v, want in [(None, 1), (b"", 1), (b"1", 1), (b"info", 1), (b"anything", 1), (b"0", 0), (b"off", 0), (b" OFF ", 0),
                    (b"false", 0), (b"quiet", 0), (b"error", 0), (b"2", 2), (b"debug", 2), (b"Trace", 2), (b"verbose\n", 2)]:
        assert parse(v) == want, v


def _in_subprocess(code, env):
    import subprocess
    import sys

    e = dict(os.environ)
    e.update(env)
    r = subprocess.run([sys.executable, "-c", "import sys; sys.path[:0] = %r; " % [ROOT, os.path.join(ROOT, "fastvideo-rs_amd")]
                        + code], capture_output=True, text=True, env=e, timeout=120)
    assert r.returncode == 0, r.stderr[-2000:]
    return r.stdout.strip()


def test_environment_defaults_are_read_by_the_library():
    code = "import fv_sdpa; l = fv_sdpa.lib(); print(l.fv_rt_log_level(), l.fv_vsa_default_sparsity())"
    assert _in_subprocess(code, {"FASTVIDEO_LOG": "debug", "FASTVIDEO_VSA_SPARSITY": " 0.875 "}) == "2 0.875"
    assert _in_subprocess(code, {"FASTVIDEO_LOG": "0", "FASTVIDEO_VSA_SPARSITY": "sparse"}) == "0 0.8"
    # the reference trims, then parses with Rust's f64 grammar (settings/parse.rs:43-45): a leading '+' and
    # exponents are numbers, hex floats and "nan(...)" (which strtod alone would take) are not
    for text, want in ((" 0.5", "0.5"), ("+0.25", "0.25"), ("5e-1\n", "0.5"), ("0x1p-1", "0.8"), ("nan(1)", "0.8"),
                       ("0.5 0.6", "0.8"), ("", "0.8")):
        assert _in_subprocess(code, {"FASTVIDEO_LOG": "0", "FASTVIDEO_VSA_SPARSITY": text}) == "0 " + want, text
    env = {k: v for k, v in os.environ.items() if k not in ("FASTVIDEO_LOG", "FASTVIDEO_VSA_SPARSITY")}
    import subprocess
    import sys

    r = subprocess.run([sys.executable, "-c", "import sys; sys.path[:0] = %r; " % [ROOT, os.path.join(ROOT, "fastvideo-rs_amd")]
                        + code], capture_output=True, text=True, env=env, timeout=120)
    assert r.stdout.strip() == "1 0.8", r.stderr[-500:]


def test_static_splitkv_never_refuses_its_own_choice():
    """fv_sdpa_dense_bf16_splitkv_static with splits == 0 runs the library's choice stepped down to what its
    32 MiB buffer holds (host arithmetic: fv_sdpa_splitkv_static_splits); only an explicit count that cannot
    fit is refused; absurd counts are settled, not divided by."""
    lib = fv_sdpa.lib()
    cap = lib.fv_sdpa_splitkv_static_bytes()
    assert cap == 32 << 20
    stepped = 0
    for d in (128, 64):
        for bh in (1, 2, 3, 4, 6, 8, 12, 16, 24, 40):
            for sq in (1, 64, 256, 257, 512, 1024, 1560, 2048, 3000, 4096, 4680, 8192):
                for sk in (64, 512, 1560, 4096, 4680, 16384, 32760, 75600):
                    auto = lib.fv_sdpa_splitkv_static_splits(bh, sq, sk, d, 0)
                    chosen = lib.fv_sdpa_splitkv_choose(bh, sq, sk)
                    assert 1 <= auto <= chosen, (bh, sq, sk, d, auto, chosen)
                    assert lib.fv_sdpa_splitkv_workspace_bytes(bh, sq, d, auto) <= cap
                    if auto < chosen:
                        stepped += 1
                        nxt = auto + 1    # the next count that is a real split count does not fit
                        while nxt <= chosen and lib.fv_sdpa_splitkv_static_splits(bh, sq, sk, d, nxt) == auto:
                            nxt += 1
                        assert nxt > chosen or lib.fv_sdpa_splitkv_static_splits(bh, sq, sk, d, nxt) == 0
    assert stepped > 0
    # the three shapes that used to be refused: 16 splits chosen, partials 262 144 bytes over the buffer
    for bh, sq in ((1, 4096), (2, 2048), (4, 1024)):
        assert lib.fv_sdpa_splitkv_choose(bh, sq, 32760) == 16
        assert lib.fv_sdpa_splitkv_workspace_bytes(bh, sq, 128, 16) == 33816576 > cap
        assert lib.fv_sdpa_splitkv_static_splits(bh, sq, 32760, 128, 0) == 15
        assert lib.fv_sdpa_splitkv_static_splits(bh, sq, 32760, 128, 16) == 0     # explicit and too large: refused
    # explicit counts: settled so that no split is empty, never more than the key tiles
    assert lib.fv_sdpa_splitkv_static_splits(12, 256, 32760, 128, 7) == 7
    assert lib.fv_sdpa_splitkv_static_splits(12, 256, 640, 128, 7) == 5            # 10 tiles / ceil(10 / 7) = 2 per split
    assert lib.fv_sdpa_splitkv_static_splits(1, 256, 640, 128, 2 ** 64 - 1) == 10  # no wrap, no division by zero
    assert lib.fv_sdpa_splitkv_static_splits(1, 256, 64, 128, 5) == 1
