"""Unsplit dense calls on few keys, two (head dim 64: three) workgroups a CU: the edges of its key and query tiles, one tile
and two, the longest walks it takes, f32 and bf16 results, row windows, rows whose scores outgrow the offset of their
first 128 keys, so that the pass is made again, and the bits of the kernel that takes the same rows in calls of few heads.

Against the f64 softmax on the same operands. P is rounded to bf16, 2^-9 of each weight at most, and so is a bf16 result:
2^-9 in the 2-norm for an f32 one, twice that for a bf16 one."""
import numpy as np
import pytest

from util import announce

pytestmark = pytest.mark.gpu
HEADS = 256   # a query tile for every CU: more than the short kernel takes


@pytest.fixture(scope="module")
def fv():
    import torch

    assert torch.cuda.is_available()
    import fv_sdpa

    fv_sdpa.lib()
    return fv_sdpa


def operands(torch, seed, sq, sk, d):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn((HEADS, s, d), generator=g, device="cuda").to(torch.bfloat16) for s in (sq, sk, sk)]


def want64(torch, q, k, v):
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    for b in range(q.shape[0]):
        s = (q[b].double() @ k[b].double().T) / np.sqrt(q.shape[-1])
        out[b] = torch.softmax(s, -1) @ v[b].double()
    return out


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("sq,sk", [(1, 1), (31, 63), (32, 64), (33, 65), (127, 100), (128, 128), (129, 129), (200, 191),
                                   (257, 192), (40, 513), (20, 1535), (20, 1536), (20, 1537), (20, 6144)])
def test_edges(fv, sq, sk, d):
    import torch

    announce(f"duo {HEADS}x{sq}x{sk}x{d}")
    q, k, v = operands(torch, sq + sk, sq, sk, d)
    want = want64(torch, q, k, v)
    for out_bf16, bound in ((True, 2 * 2.0 ** -9), (False, 2.0 ** -9)):
        got = fv.sdpa_dense_bf16(q, k, v, out_bf16=out_bf16)
        assert torch.isfinite(got).all()
        assert ((got.double() - want).norm() / want.norm()).item() <= bound, out_bf16
        assert torch.equal(got, fv.sdpa(q[None], k[None], v[None], fv.Plan.dense())[0]) or not out_bf16


@pytest.mark.parametrize("d", [64, 128])
def test_windows_and_reruns(fv, d):
    import torch

    announce(f"duo windows and reruns d={d}")
    sq, sk = 70, 300
    q, k, v = operands(torch, d, sq, sk, d)
    plain = fv.sdpa_dense_bf16(q, k, v, out_bf16=True)
    pad = [torch.full((HEADS, x.shape[1] + 9, d), float("nan"), device="cuda", dtype=torch.bfloat16) for x in (q, k, v)]
    for p, x in zip(pad, (q, k, v)):
        p[:, 2:2 + x.shape[1]] = x
    wins = [p[:, 2:2 + x.shape[1]] for p, x in zip(pad, (q, k, v))]
    assert torch.equal(fv.sdpa_dense_bf16_windows(*wins, out_bf16=True), plain)
    # scores of head 0 that climb by hundreds of base-2 units past its first tile: that head's workgroup goes again
    lib = fv.lib()
    n0 = lib.fv_sdpa_exact_pass_reruns()
    kc = k.clone()
    q1 = q.clone()
    q1[0] = 4.0
    kc[0] = (torch.arange(sk, device="cuda", dtype=torch.float32)[:, None] * (8.0 / sk)).to(torch.bfloat16).expand(sk, d)
    got = fv.sdpa_dense_bf16(q1, kc, v, out_bf16=True)
    torch.cuda.synchronize()
    assert lib.fv_sdpa_exact_pass_reruns() == n0 + 1
    want = want64(torch, q1, kc, v)
    assert ((got.double() - want).norm(dim=(1, 2)) / want.norm(dim=(1, 2))).max().item() <= 2.0 ** -7
    assert torch.equal(got[1:], plain[1:])
    # a NaN query is its own row's
    q2 = q.clone()
    q2[3, 5, 7] = float("nan")
    got = fv.sdpa_dense_bf16(q2, k, v, out_bf16=True)
    assert torch.isnan(got[3, 5]).all()
    rest = torch.ones(HEADS, sq, dtype=torch.bool, device="cuda")
    rest[3, 5] = False
    assert torch.isfinite(got[rest]).all()


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("heads,s,mask", [
    (40, 513, ("causal", 100, 0, 0)), (40, 700, ("causal", 64, 2, 1)), (30, 640, ("causal", 128, 2, 0)),
    (40, 640, ("window", 0, 64, 10, 3, 1)), (40, 701, ("window", 13, 40, 16, 0, 2)), (30, 1024, ("window", 0, 128, 8, 2, 1))])
def test_masked(fv, d, heads, s, mask):
    """Masked bf16 launches of more than 128 query tiles of 128: frame boundaries inside, on and off the tiles."""
    import torch

    announce(f"duo masked {heads}x{s}x{d} {mask}")
    g = torch.Generator(device="cuda").manual_seed(s + d)
    q, k, v = (torch.randn((heads, s, d), generator=g, device="cuda").to(torch.bfloat16) for _ in range(3))
    if mask[0] == "causal":
        bias = fv.BlockCausal(*mask[1:]).dense_mask(s, s)
        got = fv.sdpa_block_causal_bf16(q, k, v, *mask[1:], out_bf16=True)
    else:
        bias = fv.VdnWindow(*mask[1:]).dense_mask(s, s)
        got = fv.sdpa_vdn_window_bf16(q, k, v, *mask[1:], out_bf16=True)
    shut = torch.from_numpy(np.asarray(bias).reshape(s, s) < -1e8).cuda()
    assert shut.any() and not shut.all(-1).any()
    want = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    for b in range(heads):
        x = ((q[b].double() @ k[b].double().T) / np.sqrt(d)).masked_fill(shut, float("-inf"))
        want[b] = torch.softmax(x, -1) @ v[b].double()
    rows = ((got.double() - want).norm(dim=-1) / want.norm(dim=-1)).max().item()
    assert ((got.double() - want).norm() / want.norm()).item() <= 2 * 2.0 ** -9 and rows <= 2.0 ** -7, rows


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("sq,sk", [(129, 513), (257, 576), (40, 640), (300, 1535), (256, 1536)])
def test_the_bits_do_not_depend_on_the_number_of_heads(fv, sq, sk, d):
    """A launch of few heads takes flash_fwd_pp2, one of many flash_fwd_duo: the same sums term by term, so each head's
    result is that of a call on a few of them, bit for bit."""
    import torch

    announce(f"duo heads {HEADS}x{sq}x{sk}x{d}")
    q, k, v = operands(torch, 3 * sq + sk, sq, sk, d)
    many = fv.sdpa_dense_bf16(q, k, v, out_bf16=True)
    few = 128 // ((sq + 127) // 128)          # as many as leave no more than 128 tiles of 128 queries
    assert few < HEADS
    for lo in range(0, HEADS, few):
        part = fv.sdpa_dense_bf16(*(x[lo:lo + few].contiguous() for x in (q, k, v)), out_bf16=True)
        assert torch.equal(part, many[lo:lo + few]), lo


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("mask", [("causal", 70, 0, 0), ("causal", 128, 0, 0), ("causal", 66, 3, 1), ("causal", 33, 3, 2), ("causal", 64, 3, 1),
                                  ("causal", 100, 2, 0), ("window", 0, 70, 11, 3, 1), ("window", 20, 50, 14, 0, 1),
                                  ("window", 0, 40, 16, 0, 1)])
def test_masked_bits_do_not_depend_on_heads_or_clip_length(fv, d, mask):
    """Masked bf16 results: a head's rows are those of a call on two heads, and the first blocks of a causal clip are the
    shorter clip's, bit for bit, with and without window and sink, whichever kernel the sizes select."""
    import torch

    heads, s = 60, 770
    announce(f"duo masked bits {heads}x{s}x{d} {mask}")
    g = torch.Generator(device="cuda").manual_seed(s + d + mask[1])
    q, k, v = (torch.randn((heads, s, d), generator=g, device="cuda").to(torch.bfloat16) for _ in range(3))

    def call(h, n):
        x = [t[:h, :n].contiguous() for t in (q, k, v)]
        if mask[0] == "causal":
            return fv.sdpa_block_causal_bf16(*x, *mask[1:], out_bf16=True)
        return fv.sdpa_vdn_window_bf16(*x, *mask[1:], out_bf16=True)

    whole = call(heads, s)
    assert torch.equal(call(2, s), whole[:2])
    if mask[0] == "causal":
        for blocks in (2, 5, s // mask[1]):
            n = blocks * mask[1]
            for h in (2, heads):
                assert torch.equal(call(h, n), whole[:h, :n]), (blocks, h)


def masked_call(fv, mask, q, k, v, **kw):
    entry = fv.sdpa_block_causal_bf16 if mask[0] == "causal" else fv.sdpa_vdn_window_bf16
    return entry(q, k, v, *mask[1:], out_bf16=True, **kw)


def masked64(fv, torch, mask, q, k, v, scale=None):
    """The f64 softmax under the mask; rows that see no key are zeros."""
    spec = fv.BlockCausal(*mask[1:]) if mask[0] == "causal" else fv.VdnWindow(*mask[1:])
    sq, sk = q.shape[1], k.shape[1]
    shut = torch.from_numpy(np.asarray(spec.dense_mask(sq, sk)).reshape(sq, sk) < -1e8).cuda()
    scale = 1.0 / np.sqrt(q.shape[-1]) if scale is None else scale
    want = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    for b in range(q.shape[0]):
        x = ((q[b].double() @ k[b].double().T) * scale).masked_fill(shut, float("-inf"))
        want[b] = torch.softmax(x, -1).nan_to_num(0.0) @ v[b].double()
    return want


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("mask", [None, ("causal", 100, 0, 0), ("causal", 100, 3, 1), ("window", 10, 70, 9, 3, 1)])
def test_the_scale_folded_into_the_queries(fv, d, mask):
    """scale = ln 2 takes the form without the multiply of every score, and is counted."""
    import torch

    announce(f"duo log2 d={d} {mask}")
    ln2 = float(np.float32(np.log(2.0)))
    g = torch.Generator(device="cuda").manual_seed(d)
    heads, s = (60, 650) if mask else (HEADS, 140)
    q, k, v = (torch.randn((heads, s, d), generator=g, device="cuda") for _ in range(3))
    q, k, v = (x.to(torch.bfloat16) for x in (q * (1.4426950408889634 / np.sqrt(d)), k, v))
    n0 = fv.lib().fv_sdpa_log2_domain_launches()
    got = masked_call(fv, mask, q, k, v, scale=ln2) if mask else fv.sdpa_dense_bf16(q, k, v, scale=ln2, out_bf16=True)
    assert fv.lib().fv_sdpa_log2_domain_launches() == n0 + 1
    want = masked64(fv, torch, mask or ("causal", s, 0, 0), q, k, v, ln2)
    assert ((got.double() - want).norm() / want.norm()).item() <= 2 * 2.0 ** -9


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("mask", [("causal", 100, 0, 0), ("causal", 100, 3, 1), ("window", 0, 70, 10, 3, 1)])
def test_masked_reruns(fv, d, mask):
    """One head's keys past the first 128 score hundreds of base-2 units above those: all its workgroups of 128 queries go
    again (each sees some of them), under their masks, and no other head's."""
    import torch

    announce(f"duo masked reruns d={d} {mask}")
    heads, s = 60, 700
    g = torch.Generator(device="cuda").manual_seed(7 * d)
    q, k, v = (torch.randn((heads, s, d), generator=g, device="cuda") for _ in range(3))
    plain = masked_call(fv, mask, *(x.to(torch.bfloat16) for x in (q, k, v)))
    q[0] = q[0].abs() + 2.0
    k[0, :128] = -0.5
    k[0, 128:] = torch.linspace(4.0, 40.0, s - 128, device="cuda")[:, None]
    q, k, v = (x.to(torch.bfloat16) for x in (q, k, v))
    n0 = fv.lib().fv_sdpa_exact_pass_reruns()
    got = masked_call(fv, mask, q, k, v)
    torch.cuda.synchronize()
    assert fv.lib().fv_sdpa_exact_pass_reruns() - n0 == (s + 127) // 128
    assert torch.equal(got[1:], plain[1:])
    want = masked64(fv, torch, mask, q[:1], k[:1], v[:1])
    assert (got[:1].double() - want).abs().max().item() <= 2e-2


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("sq,sk,mask", [(500, 300, (90, 0, 0)), (300, 500, (90, 0, 0)), (500, 200, (70, 2, 1)), (513, 129, (128, 1, 1)),
                                        (500, 200, (70, 2, 0)), (513, 129, (128, 1, 0))])
def test_more_queries_than_keys_and_fewer(fv, sq, sk, mask, d):
    """Causal calls of many heads on rectangles, every row written; a row that sees no key (a window past the last one, no
    sink) is zeros."""
    import torch

    announce(f"duo causal {sq}x{sk}x{d} {mask}")
    heads = 60
    g = torch.Generator(device="cuda").manual_seed(sq + sk + d)
    q, k, v = (torch.randn((heads, s, d), generator=g, device="cuda").to(torch.bfloat16) for s in (sq, sk, sk))
    out = torch.full((heads, sq, d), float("nan"), device="cuda", dtype=torch.bfloat16)
    got = masked_call(fv, ("causal", *mask), q, k, v, out=out)
    want = masked64(fv, torch, ("causal", *mask), q, k, v)
    empty = ~want.abs().amax(-1).gt(0)
    assert empty.any() == (mask[2] == 0 and mask[1] > 0)
    assert not got[empty].any()
    rows = (got.double() - want).norm(dim=-1)[~empty] / want.norm(dim=-1)[~empty]
    assert rows.max().item() <= 2.0 ** -7


@pytest.mark.parametrize("d,sk", [(64, 3100), (128, 1500)])
def test_a_last_round_that_cannot_be_split(fv, d, sk):
    """32 query tiles past a round of the CUs, on a walk long enough for their keys to be shared out: the plain entry, which
    has no workspace for it, takes workgroups of 128 queries (a head of 200 that outgrows its offset is two of them); the bits
    are those of fewer heads."""
    import torch

    heads, sq = 288, 200
    announce(f"duo last round {heads}x{sq}x{sk}x{d}")
    g = torch.Generator(device="cuda").manual_seed(d)
    q, k, v = (torch.randn((heads, s, d), generator=g, device="cuda") for s in (sq, sk, sk))
    q[0] = q[0].abs() + 2.0
    k[0, 128:] = k[0, 128:].abs() + 8.0
    k[0, :128] = -0.5
    q, k, v = (x.to(torch.bfloat16) for x in (q, k, v))
    n0 = fv.lib().fv_sdpa_exact_pass_reruns()
    got = fv.sdpa_dense_bf16(q, k, v, out_bf16=True)
    torch.cuda.synchronize()
    assert fv.lib().fv_sdpa_exact_pass_reruns() == n0 + 2
    few = fv.sdpa_dense_bf16(*(x[200:260].contiguous() for x in (q, k, v)), out_bf16=True)
    assert torch.equal(few, got[200:260])
