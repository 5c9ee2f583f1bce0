"""Split-KV form of the dense kernel (few query tiles, many keys): every split count gives the unsplit
kernel's result to rounding (each split normalises by its own row sum, the merge re-weights by the
base-2 log-sum-exp), parity against the fp32 oracle, row windows read in place, the library's own
choice of the split count, and the `fv_rt_sdpa` entry applying it by itself.
"""
import numpy as np
import pytest

from util import announce, assert_parity, qkv, to_dev_bf16

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fv():
    import torch

    assert torch.cuda.is_available()
    import fv_sdpa

    fv_sdpa.lib()
    return fv_sdpa


@pytest.mark.parametrize("d", [128, 64])
@pytest.mark.parametrize("bh,sq,sk", [(2, 100, 3000), (3, 257, 2049), (1, 1, 4096), (4, 300, 1000)])
def test_every_split_count_matches_the_unsplit_kernel(fv, oracle, bh, sq, sk, d):
    import torch

    announce(f"splitkv bh={bh} sq={sq} sk={sk} d={d}")
    q, k, v = qkv(900 + sk + d, bh, sq, sk, d)
    tq, tk, tv = (to_dev_bf16(x) for x in (q, k, v))
    base = fv.sdpa_dense_bf16(tq, tk, tv)
    want = oracle.sdpa_composed(q, k, v)
    for splits in (1, 2, 3, 5, 16, 1000):
        got = fv.sdpa_dense_bf16_splitkv(tq, tk, tv, splits=splits)
        torch.cuda.synchronize()
        if splits == 1:
            assert torch.equal(got, base)
        assert (got - base).abs().max().item() <= 2e-3, splits
        assert_parity(got.cpu().numpy(), want, f"splitkv_{splits}_{bh}_{sq}_{sk}_{d}")
    got16 = fv.sdpa_dense_bf16_splitkv(tq, tk, tv, splits=4, out_bf16=True)
    torch.cuda.synchronize()
    assert (got16.float() - base).abs().max().item() <= 2e-2


def test_many_split_items(fv, oracle):
    """40 heads x 2 query tiles x 8 splits = 640 workgroups of 4 key tiles (several rounds of short
    items), against the unsplit kernel, the oracle, and the same heads in smaller calls."""
    import torch

    bh, sq, sk, d = 40, 300, 2000, 128
    announce(f"splitkv many items bh={bh} sq={sq} sk={sk}")
    q, k, v = qkv(4242, bh, sq, sk, d)
    tq, tk, tv = (to_dev_bf16(x) for x in (q, k, v))
    got = fv.sdpa_dense_bf16_splitkv(tq, tk, tv, splits=8)
    base = fv.sdpa_dense_bf16(tq, tk, tv)
    torch.cuda.synchronize()
    assert (got - base).abs().max().item() <= 2e-3
    heads = np.array([0, 1, 20, 38, 39])
    assert_parity(got[torch.from_numpy(heads).cuda()].cpu().numpy(), oracle.sdpa_composed(q[heads], k[heads], v[heads]),
                  "splitkv_many_items")
    # the same heads in smaller calls: bit-identical partials and merge
    for lo in range(0, bh, 10):
        part = fv.sdpa_dense_bf16_splitkv(tq[lo:lo + 10].contiguous(), tk[lo:lo + 10].contiguous(),
                                          tv[lo:lo + 10].contiguous(), splits=8)
        assert torch.equal(part, got[lo:lo + 10])


def test_choice_and_windows(fv, oracle):
    import torch

    # a one-frame block of Self-Forcing generation against a 21-frame cache: 7 query tiles x 12 heads
    bh, sq, sk, d = 12, 1560, 32760, 128
    splits = fv.splitkv_choose(bh, sq, sk)
    announce(f"splitkv choice bh={bh} sq={sq} sk={sk}: {splits}")
    assert 2 <= splits <= 16
    assert fv.splitkv_choose(12, 32760, 32760) == 1 and fv.splitkv_choose(12, 4680, 32760) == 1
    assert fv.splitkv_choose(12, 1560, 512) == 1          # too few key tiles to share out
    g = torch.Generator(device="cuda").manual_seed(4)
    cache_k = torch.randn((bh, sk + 500, d), generator=g, device="cuda").to(torch.bfloat16)
    cache_v = torch.randn((bh, sk + 500, d), generator=g, device="cuda").to(torch.bfloat16)
    q = torch.randn((bh, sq, d), generator=g, device="cuda").to(torch.bfloat16)
    kw, vw = cache_k[:, 100:100 + sk], cache_v[:, 100:100 + sk]      # row windows, read in place
    got = fv.sdpa_dense_bf16_splitkv(q, kw, vw)
    base = fv.sdpa_dense_bf16_windows(q, kw, vw)
    torch.cuda.synchronize()
    assert (got - base).abs().max().item() <= 2e-3
    # the plan entry picks the split form by itself for such a shape, and stays within the kernel bar
    t4 = lambda x: x.reshape(1, *x.shape)  # noqa: E731
    with fv.with_bf16_act(False):
        via_plan = fv.sdpa(t4(q), t4(cache_k)[:, :, 100:100 + sk], t4(cache_v)[:, :, 100:100 + sk], fv.Plan.kv_window())
    torch.cuda.synchronize()
    assert torch.equal(via_plan.reshape(bh, sq, d), got)
    with pytest.raises(fv.FvError):
        ws = torch.empty(256, device="cuda", dtype=torch.uint8)
        fv.lib().fv_sdpa_dense_bf16_splitkv.restype  # noqa: B018
        fv._lib.check(fv.lib().fv_sdpa_dense_bf16_splitkv(q.data_ptr(), kw.data_ptr(), vw.data_ptr(), got.data_ptr(), 0, bh, sq,
                                                          sk, d, 0.088, 0, sk + 500, sk + 500, 4, ws.data_ptr(), 256,
                                                          torch.cuda.current_stream().cuda_stream))


@pytest.mark.parametrize("bh,sq,sk,d,act16", [(38, 1700, 2100, 128, True), (37, 1650, 1600, 64, True),
                                              (38, 1537, 4100, 128, False), (261, 33, 1100, 64, True)])
def test_last_round_of_tiles_split(fv, oracle, bh, sq, sk, d, act16):
    """A few query tiles more than one per CU: the first 256 are the unsplit launch's bit for bit, the ones past them took
    the split path (a workspace is asked for, other bits), agree with it to rounding and with the oracle, and every row
    is written. The two forms round P against different offsets and sum in another order, each 2.4e-3 at most from the
    exact sums in the 2-norm: at most 4.8e-3 apart."""
    import ctypes
    import torch

    from fv_sdpa.sdpa import _FvPlan, _desc

    announce(f"splitkv last round bh={bh} sq={sq} sk={sk} d={d}")
    q, k, v = qkv(77 + sq, bh, sq, sk, d)
    tq, tk, tv = (to_dev_bf16(x) for x in (q, k, v))
    base = fv.sdpa_dense_bf16(tq, tk, tv, out_bf16=act16)          # unsplit
    p, need = _FvPlan(), (ctypes.c_size_t * 2)()
    p.kv_flash = -1
    with fv.with_bf16_act(act16):
        assert fv.lib().fv_rt_sdpa_need(*(ctypes.byref(_desc(x[None], "x")) for x in (tq, tk, tv)), ctypes.byref(p), need) == 0
        got = fv.sdpa(tq[None], tk[None], tv[None], fv.Plan.dense())[0]
    torch.cuda.synchronize()
    assert need[1] > 0
    assert got.dtype == (torch.bfloat16 if act16 else torch.float32)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    nqt = (sq + 255) // 256
    full = bh * nqt // cus * cus
    row0 = full // nqt * sq + full % nqt * 256
    assert 0 < row0 < bh * sq
    got_rows, base_rows = got.reshape(-1, d), base.reshape(-1, d)
    assert torch.equal(got_rows[:row0], base_rows[:row0])
    tail, base_tail = got_rows[row0:].double(), base_rows[row0:].double()
    assert not torch.equal(tail, base_tail)
    assert (tail - base_tail).norm() <= 4.8e-3 * base_tail.norm()
    by_row = (tail - base_tail).norm(dim=1) / base_tail.norm(dim=1)   # a misplaced row is off by its whole norm
    assert by_row.max().item() < 0.1
    heads = np.array(sorted({0, row0 // sq, bh - 1}))
    assert_parity(got[torch.from_numpy(heads).cuda()].float().cpu().numpy(),
                  oracle.sdpa_composed(q[heads], k[heads], v[heads]), f"splitkv_last_round_{bh}_{sq}_{sk}_{d}")


@pytest.mark.parametrize("bh,sq,sk,d", [(38, 1700, 2100, 128), (37, 1650, 1600, 64),   # the last round of tiles split
                                        (2, 100, 3000, 128), (3, 257, 2049, 64)])      # every tile split
@pytest.mark.parametrize("act16", [False, True])
def test_nan_rows_stay_nan(fv, bh, sq, sk, d, act16):
    """A NaN in a query makes its row NaN, one in a key the rows of its head, in split and unsplit tiles alike."""
    import torch

    announce(f"splitkv NaN bh={bh} sq={sq} sk={sk} d={d} act16={act16}")
    q, k, v = (to_dev_bf16(x) for x in qkv(5 + sq, bh, sq, sk, d))
    rows = [(0, 3), (bh // 2, sq - 1), (bh - 1, 0), (bh - 1, sq - 2)]
    for h, r in rows:
        q[h, r, d - 1] = float("nan")
    want = torch.zeros((bh, sq, d), dtype=torch.bool, device="cuda")
    for h, r in rows:
        want[h, r] = True
    with fv.with_bf16_act(act16):
        got = fv.sdpa(q[None], k[None], v[None], fv.Plan.dense())[0]
        for h in (0, bh - 1):
            k[h, sk // 2, 1] = float("nan")
            want[h] = True
        keyed = fv.sdpa(q[None], k[None], v[None], fv.Plan.dense())[0]
    torch.cuda.synchronize()
    first = torch.zeros_like(want)
    for h, r in rows:
        first[h, r] = True
    assert torch.equal(got.isnan(), first)
    assert torch.equal(keyed.isnan(), want)


@pytest.mark.parametrize("d", [128, 64])
def test_an_explicit_count_is_the_count_that_runs(fv, oracle, d):
    """Also where it is the library's own, and where fv_rt_sdpa takes another kernel: every split of a bf16 launch checks its
    own offset, so scores that outgrow the first 128 keys' show in the rerun counter. A count of one is the plain entry's
    result bit for bit, for both result types; no count is the choice of fv_rt_sdpa."""
    import torch

    bh, sq, sk = 3, 600, 1100
    announce(f"splitkv explicit counts d={d}")
    assert fv.splitkv_choose(bh, sq, sk) == 2
    q, k, v = (to_dev_bf16(x) for x in qkv(31 + d, bh, sq, sk, d))
    lib = fv.lib()
    for act16 in (True, False):
        plain = fv.sdpa_dense_bf16(q, k, v, out_bf16=act16)
        assert torch.equal(fv.sdpa_dense_bf16_splitkv(q, k, v, splits=1, out_bf16=act16), plain)
        with fv.with_bf16_act(act16):
            assert torch.equal(fv.sdpa_dense_bf16_splitkv(q, k, v, out_bf16=act16)[None], fv.sdpa(q[None], k[None], v[None], fv.Plan.dense()))
        got = fv.sdpa_dense_bf16_splitkv(q, k, v, splits=2, out_bf16=act16)
        assert (got.float() - plain.float()).abs().max().item() <= 2e-2
    q[0] = q[0].abs() + 2.0
    k[0, :128] = -0.5
    k[0, 128:] = torch.linspace(1.0, 40.0, sk - 128, device="cuda")[:, None].to(torch.bfloat16)
    n0 = lib.fv_sdpa_exact_pass_reruns()
    got = fv.sdpa_dense_bf16_splitkv(q, k, v, splits=2, out_bf16=True)
    torch.cuda.synchronize()
    assert lib.fv_sdpa_exact_pass_reruns() >= n0 + (sq + 255) // 256
    want = oracle.sdpa_f64(*(x.float().cpu().numpy() for x in (q, k, v)))
    assert_parity(got.float().cpu().numpy(), want, f"splitkv_explicit_d{d}", max_abs=2e-2)


def test_no_count_and_no_workspace_runs_unsplit(fv):
    """The entry with splits = 0 takes what fv_rt_sdpa would, and is not refused for want of a workspace."""
    import torch

    bh, sq, sk, d = 2, 100, 5000, 128
    announce("splitkv no count, no workspace")
    assert fv.splitkv_choose(bh, sq, sk) > 1
    q, k, v = (to_dev_bf16(x) for x in qkv(32, bh, sq, sk, d))
    out = torch.full((bh, sq, d), float("nan"), device="cuda")
    rc = fv.lib().fv_sdpa_dense_bf16_splitkv(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), 0, bh, sq, sk, d, d ** -0.5, 0,
                                             0, 0, 0, None, 0, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert rc == 0 and torch.equal(out, fv.sdpa_dense_bf16(q, k, v))
