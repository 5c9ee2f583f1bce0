"""Parity of the block-causal flash kernel against the oracle (masked composed
fp32 SDPA and the f64 checker). Cases follow the reference's wan_causal_attn
table (crates/fastvideo-gpucheck/src/kernels_wan.rs:90-169, every case at d = 128
and at d = 64), limit max|delta| <= 1e-2 and cosine >= 0.9999 (the
reference's own limit is 2e-2), plus the schedule invariant of
kernels_wan.rs:230-261: one block spanning the sequence is bit-identical to the
dense kernel.
"""
import numpy as np
import pytest

from util import (REL_L2_F32_OUT, announce, assert_bf16_result_matches_f32_result, assert_parity, qkv, sample_rows,
                  to_dev_bf16)

pytestmark = pytest.mark.gpu

CASES = [  # (bh, s, block_tokens, window, sink)
    (2, 300, 60, 0, 0),
    (6, 257, 37, 2, 0),
    (2, 511, 50, 3, 1),
    (4, 190, 19, 0, 2),
    (1, 129, 1, 0, 0),
    (2, 640, 128, 1, 0),
    (2, 96, 200, 0, 0),
    (2, 1000, 64, 2, 3),
    (1, 777, 100, 1, 0),
    # band walks whose tile counts are odd / even and whose sink tiles are disjoint from the
    # band (the pair-of-tiles phases round an odd count up with a fully masked tile)
    (1, 1280, 64, 2, 1),    # window 2 blocks of one tile, one sink tile: 3-tile walks
    (1, 1280, 128, 1, 1),
    (2, 1500, 192, 2, 2),
    (1, 2049, 256, 3, 0),
    (1, 900, 300, 0, 0),
]


@pytest.fixture(scope="module")
def fv():
    import torch

    assert torch.cuda.is_available()
    import fv_sdpa

    fv_sdpa.lib()
    return fv_sdpa


@pytest.mark.parametrize("d", [128, 64])
@pytest.mark.parametrize("bh,s,bt,win,sink", CASES)
def test_block_causal_matches_masked_oracle(fv, oracle, bh, s, bt, win, sink, d):
    import torch

    seed = 3000 + s + d
    announce(f"causal bh={bh} s={s} d={d} block={bt} window={win} sink={sink} seed={seed}")
    q, k, v = qkv(seed, bh, s, s, d)
    mask = oracle.block_causal_dense_mask(bt, win, sink, s, s)
    want = oracle.sdpa_composed(q, k, v, mask=mask)
    want64 = oracle.sdpa_f64(q, k, v, mask_bc=(bt, win, sink))
    qd, kd, vd = (to_dev_bf16(x) for x in (q, k, v))
    got = fv.sdpa_block_causal_bf16(qd, kd, vd, bt, win, sink)
    torch.cuda.synchronize()
    got = got.cpu().numpy()
    assert_parity(got, want, f"causal_{s}_{bt}_{win}_{sink}_vs_composed")
    assert_parity(got, want64, f"causal_{s}_{bt}_{win}_{sink}_vs_f64")
    got16 = fv.sdpa_block_causal_bf16(qd, kd, vd, bt, win, sink, out_bf16=True)
    torch.cuda.synchronize()
    # launches that write bf16 and whose queries all see key 0 keep the softmax offset of the first 128 keys; the f32
    # launch follows the running max: the same bits unless a row's maximum grows by 2^6 after those keys
    assert_bf16_result_matches_f32_result(got16.float().cpu().numpy(), got, f"causal_{s}_{bt}_{win}_{sink}", exact_share=0.9)


@pytest.mark.parametrize("d", [128, 64])
@pytest.mark.parametrize("out_bf16", [False, True])
def test_one_block_spanning_the_sequence_is_the_dense_kernel(fv, d, out_bf16):
    """gpucheck/src/kernels_wan.rs:230-261 (its shape: 1 x 3 x 333, both head dims, bf16 result), and a longer one."""
    import torch

    for bh, s in ((3, 333), (3, 700)):
        announce(f"causal one-block == dense, {bh}x{s} d={d} out_bf16={out_bf16}")
        q, k, v = (to_dev_bf16(x) for x in qkv(11 + s, bh, s, s, d))
        dense = fv.sdpa_dense_bf16(q, k, v, out_bf16=out_bf16)
        causal = fv.sdpa_block_causal_bf16(q, k, v, max(s, 4096), 0, 0, out_bf16=out_bf16)
        exact = fv.sdpa_block_causal_bf16(q, k, v, s, 0, 0, out_bf16=out_bf16)
        torch.cuda.synchronize()
        assert torch.equal(dense, causal) and torch.equal(dense, exact)


def test_sq_ne_sk_and_first_block_rows(fv, oracle):
    import torch

    # queries of a later chunk against a longer key sequence is not a reference
    # case (its causal calls are square); square only, but check block-0 rows
    # see only block 0 (kernel never loads later tiles for them)
    bh, s, d, bt = 1, 512, 128, 128
    announce("causal first-block rows 1x512")
    q, k, v = qkv(13, bh, s, s, d)
    got = fv.sdpa_block_causal_bf16(*(to_dev_bf16(x) for x in (q, k, v)), bt, 0, 0)
    torch.cuda.synchronize()
    want0 = oracle.sdpa_composed(q[:, :bt], k[:, :bt], v[:, :bt])
    assert_parity(got[:, :bt].cpu().numpy(), want0, "causal_block0_rows")


@pytest.mark.parametrize("d", [128, 64])
@pytest.mark.parametrize("bh,sq,sk,bt,win,sink", [
    (2, 512, 256, 256, 1, 0),     # the second query tile walks no key tile at all
    (1, 1000, 300, 100, 2, 0),    # rows 500.. see nothing; the tile 256..511 is partly visible
    (2, 1000, 300, 100, 2, 1),    # same with a sink block: every row sees block 0
    (1, 700, 130, 64, 0, 0),      # more queries than keys, no window: the late rows see every key
])
def test_more_queries_than_keys_with_a_window(fv, oracle, bh, sq, sk, bt, win, sink, d):
    """sq > sk with a window lets the window slide past the last key: such rows have no visible key and
    come out as zeros (the reference's kernel runs zero iterations and stores acc * 0,
    kernels/attn2.cu:214-221, 330-352), whole tiles of them included; every other row matches the
    masked oracle. The output buffer is poisoned first, so an unwritten row cannot pass."""
    import torch

    seed = 4100 + sq + d
    announce(f"causal sq>sk bh={bh} sq={sq} sk={sk} d={d} block={bt} window={win} sink={sink} seed={seed}")
    q, k, v = qkv(seed, bh, sq, sk, d)
    tq, tk = np.arange(sq)[:, None] // bt, np.arange(sk)[None, :] // bt
    vis = (tk < sink) | ((tk <= tq) & ((win == 0) | (tq - tk < win)))
    live = vis.any(axis=1)
    assert (win == 0 or sink > 0) == bool(live.all())
    want = oracle.sdpa_f64(q, k, v, mask_bc=(bt, win, sink), rows=np.nonzero(live)[0])
    qd, kd, vd = (to_dev_bf16(x) for x in (q, k, v))
    for out_bf16 in (False, True):
        out = torch.full((bh, sq, d), float("nan"), device="cuda", dtype=torch.bfloat16 if out_bf16 else torch.float32)
        fv.sdpa_block_causal_bf16(qd, kd, vd, bt, win, sink, out_bf16=out_bf16, out=out)
        torch.cuda.synchronize()
        got = out.float().cpu().numpy()
        assert np.isfinite(got).all()
        assert np.all(got[:, ~live] == 0.0)
        assert_parity(got[:, live], want, f"causal_sq{sq}_sk{sk}_{bt}_{win}_{sink}_bf16out{int(out_bf16)}",
                      max_abs=2e-2 if out_bf16 else 1e-2)


def test_declines(fv):
    import torch

    y = torch.zeros((1, 4, 128), device="cuda", dtype=torch.bfloat16)
    with pytest.raises(fv.FvDeclined):
        fv.sdpa_block_causal_bf16(y, y, y, 0, 0, 0)


@pytest.mark.parametrize("bt", [1560, 4680])
def test_headline_causal_shape_sampled_rows(fv, oracle, bt):
    """Self-Forcing frame-causal at full size (21 frames x 1560 tokens) and the reference's own 3-frame
    blocks, inputs from numpy's PCG64: parity of every head on more than 512 query rows, the last row of
    every block and the first row of the next among them (both sides of every mask boundary)."""
    import torch

    bh, s, d = 12, 32760, 128
    announce(f"causal headline bh={bh} s={s} block={bt} seed=77")
    qn, kn, vn = qkv(77, bh, s, s, d)
    q, k, v = (to_dev_bf16(x) for x in (qn, kn, vn))
    out = fv.sdpa_block_causal_bf16(q, k, v, bt, 0, 0)
    torch.cuda.synchronize()
    edges = [e for b in range(bt, s, bt) for e in (b - 1, b)]
    rows = sample_rows(3, s, 512, extra=[0, 255, 256, 10 * bt + 5, s - 1] + edges)
    assert rows.size >= 512 and set(edges) <= set(rows.tolist())
    want = oracle.sdpa_composed_rows(qn, kn, vn, rows, mask_bc=(bt, 0, 0))
    assert_parity(out[:, torch.from_numpy(rows).cuda()].cpu().numpy(), want, f"causal_headline_{bt}_{rows.size}_rows",
                  max_rel_l2=REL_L2_F32_OUT)
    # the bf16 output is the RNE rounding of the f32 output, every element
    assert torch.equal(fv.sdpa_block_causal_bf16(q, k, v, bt, 0, 0, out_bf16=True), out.to(torch.bfloat16))


@pytest.mark.parametrize("mode", ["block_causal", "vdn_window"])
def test_full_size_masked_rows_of_ones(fv, mode):
    """With V = 1 every row of a masked call is 1 if its visible weights are normalised right: a check
    of the whole full-size output (tile walks, boundary masks, longest-first order) without an oracle."""
    import torch

    bh, d = 12, 128
    s = 32760 if mode == "block_causal" else 49920
    announce(f"masked rows-of-ones {mode} bh={bh} s={s}")
    g = torch.Generator(device="cuda").manual_seed(12)
    q, k = (torch.randn((bh, s, d), generator=g, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    v = torch.ones((bh, s, d), device="cuda", dtype=torch.bfloat16)
    if mode == "block_causal":
        out = fv.sdpa_block_causal_bf16(q, k, v, 1560, 0, 0)
    else:
        out = fv.sdpa_vdn_window_bf16(q, k, v, 0, 1560, 32, 5, 1)
    torch.cuda.synchronize()
    err = (out - 1.0).abs().max().item()
    print(f"max |out - 1| = {err:.3e}")
    assert err <= 4e-3


@pytest.mark.parametrize("bt,win,sink", [(1560, 0, 0), (4680, 0, 0), (1560, 4, 1)])
def test_full_size_prefix_and_block_properties(fv, bt, win, sink):
    """Whole-output checks at H = 12, S = 21 x 1560 that need no oracle. (1) A block-causal row sees nothing after
    its own block, so the first n blocks of the full call equal the call on the first n blocks alone, every row
    and element, bit for bit: the walks visit the same key tiles in the same order, and the keys past the prefix
    are masked in one call and absent in the other. (2) Without window and sink, the rows of the first block equal
    dense attention over that block (bar: a quarter of the output's standard deviation, and 1e-2)."""
    import torch

    bh, frames, ft, d = 12, 21, 1560, 128
    s = frames * ft
    announce(f"block-causal full size prefix property bt={bt} win={win} sink={sink}")
    g = torch.Generator(device="cuda").manual_seed(4242)
    q, k, v = (torch.randn((bh, s, d), generator=g, device="cuda").to(torch.bfloat16) for _ in range(3))
    full = fv.sdpa_block_causal_bf16(q, k, v, bt, win, sink)
    torch.cuda.synchronize()
    assert torch.isfinite(full).all()
    for blocks in (1, 2, (s // bt) // 2 + 1):
        n = blocks * bt
        part = fv.sdpa_block_causal_bf16(q[:, :n].contiguous(), k[:, :n].contiguous(), v[:, :n].contiguous(), bt, win, sink)
        torch.cuda.synchronize()
        assert torch.equal(part, full[:, :n]), (blocks, (part - full[:, :n]).abs().max().item())
    if win == 0 and sink == 0:
        first = fv.sdpa_dense_bf16(q[:, :bt].contiguous(), k[:, :bt].contiguous(), v[:, :bt].contiguous())
        torch.cuda.synchronize()
        delta = (first - full[:, :bt]).abs().max().item()
        assert delta <= min(1e-2, 0.25 * first.std().item()), delta


@pytest.mark.parametrize("out_bf16", [False, True])
@pytest.mark.parametrize("bh,bt,d", [(2, 513, 128), (40, 600, 64), (40, 880, 128), (12, 1560, 128)])
def test_a_clip_of_one_block_is_the_first_block_of_a_longer_one(fv, bh, bt, d, out_bf16):
    """One block is the dense launch, three are a masked one: the rows of the first block are the same bits, for blocks of
    more than 512 tokens (shorter ones are dense calls that the short kernel takes)."""
    import torch

    announce(f"causal one block and three {bh}x{bt}x{d} out_bf16={out_bf16}")
    g = torch.Generator(device="cuda").manual_seed(bh + bt)
    q, k, v = (torch.randn((bh, 3 * bt, d), generator=g, device="cuda").to(torch.bfloat16) for _ in range(3))
    whole = fv.sdpa_block_causal_bf16(q, k, v, bt, 0, 0, out_bf16=out_bf16)
    one = fv.sdpa_block_causal_bf16(*(x[:, :bt].contiguous() for x in (q, k, v)), bt, 0, 0, out_bf16=out_bf16)
    torch.cuda.synchronize()
    assert torch.equal(one, whole[:, :bt])


@pytest.mark.parametrize("d", [128, 64])
def test_block_causal_pass_with_the_fixed_offset_and_its_rerun(fv, oracle, d):
    """Block-causal launches that write bf16 and in which every query sees key 0 (no window, or sink blocks) make their
    pass with every query's softmax offset fixed at the largest score among the first 128 keys of its tile's walk and
    redo it with the running max where a row outgrew that by more than about 2^90. One head's later keys score hundreds of base-2
    units above its first ones: its workgroups take the second pass (counted), every row matches the f64 host math
    under the mask, the other heads' rows are the bits of a launch without that head; a launch under a window
    with a sink block does the same, and one under a window without a sink (whose queries may see none of the walk's
    first keys) keeps the running max: no rerun, same tolerance."""
    import torch

    bh, s, bt = 3, 700, 100
    announce(f"block-causal fixed-offset pass and its rerun d={d}")
    rng = np.random.Generator(np.random.PCG64(515))
    q = rng.standard_normal((bh, s, d)).astype(np.float32)
    k = rng.standard_normal((bh, s, d)).astype(np.float32)
    v = oracle.quantize_bf16(rng.standard_normal((bh, s, d)).astype(np.float32))
    q[0] = np.abs(q[0]) + 2.0
    k[0, :128] = -0.5
    k[0, 128:] = np.linspace(1.0, 30.0, s - 128, dtype=np.float32)[:, None]
    q, k = oracle.quantize_bf16(q), oracle.quantize_bf16(k)
    tq, tk, tv = (to_dev_bf16(x) for x in (q, k, v))
    lib = fv.lib()
    n0 = lib.fv_sdpa_exact_pass_reruns()
    got = fv.sdpa_block_causal_bf16(tq, tk, tv, bt, 0, 0, out_bf16=True)
    torch.cuda.synchronize()
    n1 = lib.fv_sdpa_exact_pass_reruns()
    # head 0: the query tiles whose rows see keys past the first 128 (all three: the first tile's rows 128.. do)
    assert n1 - n0 == (s + 255) // 256, (n0, n1)
    want = oracle.sdpa_f64(q, k, v, mask_bc=(bt, 0, 0))
    assert_parity(got.float().cpu().numpy(), want, f"causal_rerun_d{d}", max_abs=2e-2)
    rest = fv.sdpa_block_causal_bf16(tq[1:].contiguous(), tk[1:].contiguous(), tv[1:].contiguous(), bt, 0, 0, out_bf16=True)
    torch.cuda.synchronize()
    assert lib.fv_sdpa_exact_pass_reruns() == n1 and torch.equal(rest, got[1:])
    # f32 results and windows without a sink keep the running max
    got32 = fv.sdpa_block_causal_bf16(tq, tk, tv, bt, 0, 0)
    gotw0 = fv.sdpa_block_causal_bf16(tq, tk, tv, bt, 3, 0, out_bf16=True)
    torch.cuda.synchronize()
    assert lib.fv_sdpa_exact_pass_reruns() == n1
    assert_parity(got32.cpu().numpy(), want, f"causal_running_max_d{d}")
    assert_parity(gotw0.float().cpu().numpy(), oracle.sdpa_f64(q, k, v, mask_bc=(bt, 3, 0)), f"causal_window_nosink_d{d}", max_abs=2e-2)
    # a window with a sink block: key 0 is visible to every query, fixed offset, head 0 redone
    gotw = fv.sdpa_block_causal_bf16(tq, tk, tv, bt, 3, 1, out_bf16=True)
    torch.cuda.synchronize()
    assert lib.fv_sdpa_exact_pass_reruns() == n1 + (s + 255) // 256
    assert_parity(gotw.float().cpu().numpy(), oracle.sdpa_f64(q, k, v, mask_bc=(bt, 3, 1)), f"causal_window_d{d}", max_abs=2e-2)
