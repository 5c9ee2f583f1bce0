"""The composed kernel (f32 arithmetic on the bf16 matrix cores) at the edges of its tiles: head dims that are no
multiple of 32, of 8 or of 4, one row more and less than a query group and a key tile, every split of the keys over a
workgroup's waves, operands of either type, rows that are not 16-byte units, both kinds of mask, both result types.

Checked against the same sums in 64 bits. Bounds: with f32 arithmetic a weight 2^x carries the rounding of x, |x| at
most about 16 at these inputs, so up to 16 ln 2 2^-24 = 7e-7 relative, and the sums a few 2^-24 more: 2e-6 in the
2-norm. A result rounded to bf16 adds 2^-9 at most: 2e-3."""
import numpy as np
import pytest

from util import announce

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fv():
    import torch

    assert torch.cuda.is_available()
    import fv_sdpa

    fv_sdpa.lib()
    return fv_sdpa


def want64(q, k, v, mask):
    q, k, v = (x.double().cpu().numpy() for x in (q, k, v))
    s = q @ k.swapaxes(-1, -2) / np.sqrt(q.shape[-1])
    if mask is not None:
        s = s + mask.double().cpu().numpy()
    m = s.max(axis=-1, keepdims=True)
    e = np.exp(s - np.where(np.isfinite(m), m, 0.0))
    l = e.sum(axis=-1, keepdims=True)
    return np.where(l > 0, (e / np.where(l > 0, l, 1.0)) @ v, 0.0)


SHAPES = [  # bh, sq, sk, d
    (1, 1, 1, 1), (2, 5, 7, 8), (1, 31, 33, 7), (2, 33, 32, 30), (1, 32, 31, 33), (3, 64, 65, 40), (1, 127, 129, 72),
    (2, 129, 64, 80), (1, 100, 257, 96), (1, 96, 63, 100), (2, 130, 191, 128), (1, 33, 300, 127),
    (40, 500, 90, 64),        # 640 query groups: two shares of the keys
    (70, 500, 70, 128),       # 1120: two (one with three parts)
    (3, 70, 290, 24), (2, 97, 545, 96), (1, 33, 257, 61),   # eight shares, more than one tile each for some
    (66, 1000, 40, 64),       # 2112: one
]


@pytest.mark.parametrize("kinds", ["f32", "bf16", "round", "mixed"])
@pytest.mark.parametrize("bh,sq,sk,d", SHAPES)
def test_edges(fv, bh, sq, sk, d, kinds):
    import torch

    announce(f"composed bh={bh} sq={sq} sk={sk} d={d} {kinds}")
    g = torch.Generator(device="cuda").manual_seed(1000 * sq + sk + d)
    mk = lambda s: torch.randn((1, bh, s, d), generator=g, device="cuda")
    q, k, v = mk(sq), mk(sk), mk(sk)
    act16 = kinds in ("bf16", "round")
    if kinds == "bf16":
        q, k, v = (x.to(torch.bfloat16) for x in (q, k, v))
    elif kinds == "mixed":                        # f32 queries against bf16 keys: nothing may be rounded
        k, v = k.to(torch.bfloat16), v.to(torch.bfloat16)
    shared = torch.randn((1, 1, sq, sk), generator=g, device="cuda")
    shared[..., ::3] = -1e9
    per_head = torch.randn((1, bh, sq, sk), generator=g, device="cuda")
    per_head[:, :, 0, :] = float("-inf")          # a row without a key: zeros
    for mask in (None, shared, per_head):
        with fv.with_bf16_act(act16):
            if kinds == "bf16" or act16:
                plan = fv.Plan.masked(None, mask) if mask is not None else fv.Plan.kv_window_with(False)
            else:
                plan = fv.Plan.composed(None, mask)
            out = fv.sdpa(q, k, v, plan)
        torch.cuda.synchronize()
        assert out.dtype == (torch.bfloat16 if act16 else torch.float32) and tuple(out.shape) == (1, bh, sq, d)
        qq, kk, vv = (x.to(torch.bfloat16) for x in (q, k, v)) if act16 else (q, k, v)
        want = want64(qq, kk, vv, mask)
        got = out.double().cpu().numpy()
        assert np.isfinite(got).all()
        if mask is per_head and bh > 1:
            assert not got[:, :, 0].any()
        norm = np.linalg.norm(want)
        assert np.linalg.norm(got - want) <= (2e-3 if act16 else 2e-6) * norm + 1e-30, np.linalg.norm(got - want) / norm


def test_unaligned_operands(fv):
    """Pointers that are not 16-byte aligned take element loads and stores."""
    import torch

    bh, sq, sk, d = 2, 70, 90, 64
    announce("composed unaligned")
    g = torch.Generator(device="cuda").manual_seed(7)
    lib = fv.lib()
    mk = lambda n: torch.randn(n + 1, generator=g, device="cuda")[1:]
    q, k, v = mk(bh * sq * d), mk(bh * sk * d), mk(bh * sk * d)
    mask, out = mk(sq * sk), torch.full((bh * sq * d + 2,), 7.0, device="cuda")
    rc = lib.fv_sdpa_composed_f32(q.data_ptr(), k.data_ptr(), v.data_ptr(), mask.data_ptr(), 0, out[1:].data_ptr(), bh, sq,
                                  sk, d, 0.125, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    torch.cuda.synchronize()
    want = want64(q.view(bh, sq, d), k.view(bh, sk, d), v.view(bh, sk, d), mask.view(sq, sk))
    got = out[1:-1].view(bh, sq, d).double().cpu().numpy()
    assert np.linalg.norm(got - want) <= 2e-6 * np.linalg.norm(want)
    assert float(out[0]) == 7.0 and float(out[-1]) == 7.0


@pytest.mark.parametrize("scale", [-0.3, 0.0, 0.125, 1.7])
@pytest.mark.parametrize("bh,sq,sk,d,act16", [(9, 65, 97, 64, True), (9, 65, 97, 64, False), (1, 33, 40, 128, False),
                                              (70, 960, 33, 96, True)])
def test_scales(fv, bh, sq, sk, d, act16, scale):
    """Unmasked scores are scaled inside the exponential (sign and zero go into the queries), masked ones before the
    mask is added; item counts that eight does not divide."""
    import torch

    announce(f"composed scale={scale} bh={bh} sq={sq} sk={sk} d={d} {act16}")
    g = torch.Generator(device="cuda").manual_seed(sq + sk + d)
    mk = lambda s: torch.randn((1, bh, s, d), generator=g, device="cuda")
    q, k, v = mk(sq), mk(sk), mk(sk)
    if act16:
        q, k, v = (x.to(torch.bfloat16) for x in (q, k, v))
    for mask in (None, torch.randn((1, 1, sq, sk), generator=g, device="cuda")):
        out = fv.sdpa(q, k, v, fv.Plan.composed(scale, mask))
        torch.cuda.synchronize()
        # 64-bit reference on keys scaled by scale * sqrt(d) (want64 divides by sqrt(d))
        want = want64(q, k.double() * (scale * np.sqrt(d)), v, mask)
        # scores up to |scale| * sqrt(d) * 5 in f32: a rounding of each is that times 2^-24 on its weight
        bound = 2e-6 + abs(scale) * np.sqrt(d) * 5 * 2.0**-24
        err = np.linalg.norm(out.double().cpu().numpy() - want) / np.linalg.norm(want)
        assert err <= bound, (err, bound)


@pytest.mark.parametrize("bh,sq,sk,d", [(35, 1010, 515, 128), (18, 2000, 700, 40), (24, 1400, 900, 63), (257, 128, 1025, 96),
                                        (12, 4096, 1000, 128)])
@pytest.mark.parametrize("masked", ["no", "shared", "per_head"])
def test_split_tail(fv, bh, sq, sk, d, masked):
    """Query tiles past a multiple of the CUs, shared out by key ranges: the rows before them are those of the launch
    that is not cut, bit for bit, the others within f32 rounding of the 64-bit sums; ranges that a row sees no key of."""
    import torch
    from fv_sdpa.sdpa import Plan, _PLAN_BYTES, _desc_bytes

    announce(f"composed split tail bh={bh} sq={sq} sk={sk} d={d} {masked}")
    g = torch.Generator(device="cuda").manual_seed(bh + sq + sk + d)
    q, k, v = (torch.randn((1, bh, s, d), generator=g, device="cuda") for s in (sq, sk, sk))
    mask = None
    if masked != "no":
        mask = torch.randn((1, 1 if masked == "shared" else bh, sq, sk), generator=g, device="cuda")
        mask[..., sq // 2:, : sk // 2] = -float("inf")   # the first ranges hold no key of these rows
        mask[..., sq - 1, : sk - 3] = -1e9
        if masked == "per_head":
            mask[:, -1, sq - 2] = -float("inf")          # no key at all
    lib = fv.lib()
    need = (fv._lib.C.c_size_t * 2)()
    plain = _PLAN_BYTES.pack(Plan.COMPOSED, 0, 0.0, 0, 0, *(0,) * 8, -1)
    assert lib.fv_rt_sdpa_need(*(_desc_bytes(x, "x") for x in (q, k, v)), plain, need) == 0 and need[1] > 0
    scale = float(np.float32(1.0 / np.sqrt(d)))          # the same f32 number for both
    got = fv.sdpa(q, k, v, Plan.composed(scale, mask))
    whole = torch.full_like(got, float("nan"))
    assert lib.fv_sdpa_composed_f32(q.data_ptr(), k.data_ptr(), v.data_ptr(), mask.data_ptr() if mask is not None else None,
                                    int(masked == "per_head"), whole.data_ptr(), bh, sq, sk, d, scale,
                                    torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    nqt = (sq + 127) // 128
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    full = bh * nqt // cus * cus
    row0 = full // nqt * sq + full % nqt * 128
    assert 0 < row0 < bh * sq
    a, b = got.view(bh * sq, d), whole.view(bh * sq, d)
    assert torch.equal(a[:row0], b[:row0])
    h0 = row0 // sq                                      # the heads the tail touches
    want = want64(q[:, h0:], k[:, h0:], v[:, h0:], mask[:, h0:] if masked == "per_head" else mask)
    have = got[:, h0:].double().cpu().numpy()
    assert np.isfinite(have).all()
    assert np.linalg.norm(have - want) <= 2e-6 * np.linalg.norm(want)


@pytest.mark.parametrize("bh,sq,sk,d,dtype", [
    (66, 1000, 40, 64, "bf16"), (40, 500, 90, 64, "bf16"), (3, 70, 200, 64, "bf16"), (3, 70, 290, 64, "bf16"),   # 1, 2, 4, 8 shares
    (3, 70, 200, 64, "f32"), (35, 1010, 515, 128, "f32"),   # three parts: two shares; whole tiles and a tail cut by key ranges
    (2, 5, 300, 200, "f32")])                               # past 128 channels
def test_nan_scores_make_nan_rows(fv, bh, sq, sk, d, dtype):
    """A NaN in a query makes its row NaN and leaves every other row as it was, one in a key makes the rows of its head
    NaN, and a row whose mask closes every key stays zeros."""
    import torch

    announce(f"composed NaN bh={bh} sq={sq} sk={sk} d={d} {dtype}")
    g = torch.Generator(device="cuda").manual_seed(sq + sk)
    q, k, v = (torch.randn((1, bh, s, d), generator=g, device="cuda").to(torch.bfloat16 if dtype == "bf16" else torch.float32)
               for s in (sq, sk, sk))
    mask = torch.zeros((sq, sk), device="cuda")
    mask[3] = float("-inf")
    plan = fv.Plan.masked(None, mask)
    with fv.with_bf16_act(dtype == "bf16"):
        base = fv.sdpa(q, k, v, plan)
        rows = [(0, 0), (bh // 2, 1), (bh - 1, sq - 1)]
        for h, r in rows:
            q[0, h, r, d - 1] = float("nan")
        got = fv.sdpa(q, k, v, plan)
        k[0, bh - 1, sk // 2, 1] = float("nan")
        keyed = fv.sdpa(q, k, v, plan)
    torch.cuda.synchronize()
    assert not bool(base.isnan().any()) and not bool(base[0, :, 3].any())
    for h, r in rows:
        assert bool(got[0, h, r].isnan().all()), (h, r)
        base[0, h, r] = got[0, h, r]
    assert torch.equal(got.nan_to_num(7.0), base.nan_to_num(7.0))
    assert bool(keyed[0, bh - 1].isnan().all())
    assert torch.equal(keyed[0, :bh - 1].nan_to_num(7.0), got[0, :bh - 1].nan_to_num(7.0))


def plain64(q, k, v, mask):
    """The plain sums in 64 bits, with what infinities and NaN make of them; a row without a key is zeros."""
    q, k, v = (x.double().cpu().numpy() for x in (q, k, v))
    with np.errstate(all="ignore"):
        s = q @ k.swapaxes(-1, -2) / np.sqrt(q.shape[-1]) + mask.double().cpu().numpy()
        m = s.max(axis=-1, keepdims=True)
        e = np.exp(s - np.where(m == -np.inf, 0.0, m))
        l = e.sum(axis=-1, keepdims=True)
        return np.where(l == 0, 0.0, (e @ v) / l)


MAX = float(np.finfo(np.float32).max)
OUT_OF_RANGE = {   # name: (what to do to q, k, v of shape [.., s, d]; key 5 is closed)
    "v_max_closed": lambda q, k, v: v[..., 5, 0].fill_(MAX) and v[..., 5, 1].fill_(-MAX),
    "v_inf_closed": lambda q, k, v: v[..., 5, 2].fill_(float("inf")),
    "v_inf_open": lambda q, k, v: v[..., 6, 1].fill_(float("-inf")),
    "k_max_closed": lambda q, k, v: (q[..., 3].mul_(2.0 ** -10), k[..., 5, 3].fill_(MAX)),
    "k_inf_open": lambda q, k, v: (q[..., 1].abs_().add_(0.5), k[..., 7, 1].fill_(float("-inf"))),   # scores of -inf: weight 0
    "q_inf": lambda q, k, v: q[..., 9, 1].fill_(float("inf")),
    "v_tiny": lambda q, k, v: v.mul_(2.0 ** -118),
    "v_tiny_channel": lambda q, k, v: v[..., 3].mul_(2.0 ** -118),
    "v_huge": lambda q, k, v: v.mul_(2.0 ** 115),
    "qk_apart": lambda q, k, v: (q.mul_(2.0 ** -105), k.mul_(2.0 ** 105)),
}


@pytest.mark.parametrize("case", OUT_OF_RANGE)
@pytest.mark.parametrize("bh,sq,sk,d,kinds", [
    (3, 70, 200, 72, "f32"), (2, 40, 70, 33, "f32"), (35, 1010, 515, 128, "f32"),    # three parts; the last: whole tiles and a cut tail
    (3, 70, 290, 64, "round"), (66, 1000, 40, 96, "round"),
    (66, 1000, 40, 64, "bf16"), (40, 500, 90, 128, "bf16"), (3, 70, 200, 80, "bf16"), (3, 70, 290, 30, "bf16")])
def test_operands_outside_the_range_of_the_parts(fv, bh, sq, sk, d, kinds, case):
    """Infinities, f32 numbers past the largest bf16 number and values below bf16's subnormals: what the plain f32 sums give,
    in the rows and channels they concern and nowhere else (a closed key's finite values do not count, whatever they are).
    Twice 2e-6 and 2e-3, the bounds above, as a channel alone has larger relative errors than all together (a tiny bf16
    result, 2^-122, adds its subnormals' 2^-134: 2e-4)."""
    import torch

    announce(f"composed out of range bh={bh} sq={sq} sk={sk} d={d} {kinds} {case}")
    g = torch.Generator(device="cuda").manual_seed(sq + sk + d)
    q, k, v = (torch.randn((1, bh, s, d), generator=g, device="cuda") for s in (sq, sk, sk))
    OUT_OF_RANGE[case](*(x[:, bh - 1:] for x in (q, k, v)))     # in the last head only
    if kinds == "bf16":
        q, k, v = (x.to(torch.bfloat16) for x in (q, k, v))
    mask = torch.zeros((sq, sk), device="cuda")
    mask[:, 5] = float("-inf")
    act16 = kinds != "f32"
    with fv.with_bf16_act(act16):
        got = fv.sdpa(q, k, v, fv.Plan.masked(None, mask))
    torch.cuda.synchronize()
    heads = [0, bh - 1]
    r16 = (lambda x: x.to(torch.bfloat16)) if act16 else (lambda x: x)
    want = plain64(*(r16(x[0, heads]) for x in (q, k, v)), mask)
    got = got[0, heads].double().cpu().numpy()
    for i, name in enumerate(("an untouched head", case)):
        g_, w = got[i], want[i]
        assert np.array_equal(np.isnan(g_), np.isnan(w)), name
        inf = np.isinf(w)
        assert np.array_equal(g_[inf], w[inf]) and np.array_equal(np.isinf(g_), inf), name
        fin = np.isfinite(w)
        for col in range(d):                                  # by channel: a tiny one does not hide behind the others
            f = fin[:, col]
            if f.any():
                err = np.linalg.norm(g_[f, col] - w[f, col]) / np.linalg.norm(w[f, col])
                assert err < (4e-3 if act16 else 4e-6), (name, col, err)


@pytest.mark.parametrize("mask_dtype", ["f32", "bf16"])
def test_a_row_window_as_mask(fv, mask_dtype):
    """A mask of every head's own that is a row window of longer planes (`full[:, :, a:b]`): its own rows, not the memory
    behind its first one."""
    import torch

    g = torch.Generator(device="cuda").manual_seed(8)
    q, k, v = (torch.randn((1, 3, s, 64), generator=g, device="cuda") for s in (40, 72, 72))
    full = torch.randn((1, 3, 100, 72), generator=g, device="cuda").to(torch.bfloat16 if mask_dtype == "bf16" else torch.float32)
    window = full[:, :, 7:47]
    with fv.with_bf16_act(False):
        got = fv.sdpa(q, k, v, fv.Plan.masked(None, window))
        want = fv.sdpa(q, k, v, fv.Plan.masked(None, window.contiguous()))
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    assert np.linalg.norm(got.double().cpu().numpy() - want64(q, k, v, window)) < 2e-6 * np.linalg.norm(want64(q, k, v, window))


def test_more_query_tiles_than_one_launch_holds(fv):
    """65535 heads of 33000 queries are 2^24 query tiles and more, a launch of 2^32 work-items: made in parts, every head
    in its place. One key, whose value is the result; one channel."""
    import torch

    bh, sq = 65535, 33000
    announce(f"composed bh={bh} sq={sq}")
    q = torch.zeros((1, bh, sq, 1), device="cuda", dtype=torch.bfloat16)
    k = torch.ones((1, bh, 1, 1), device="cuda", dtype=torch.bfloat16)
    v = (torch.arange(bh, device="cuda") % 251 + 1).to(torch.bfloat16).reshape(1, bh, 1, 1)
    with fv.with_bf16_act(True):
        got = fv.sdpa(q, k, v, fv.Plan.dense())
    torch.cuda.synchronize()
    for lo in range(0, bh, 8192):
        assert bool((got[:, lo:lo + 8192] == v[:, lo:lo + 8192]).all())


@pytest.mark.parametrize("act16", [True, False])
@pytest.mark.parametrize("per_head", [True, False])
@pytest.mark.parametrize("h,sq,sk,d", [(1, 33, 1, 16), (2, 40, 3, 64), (2, 33, 61, 64), (3, 70, 318, 80), (70, 1000, 95, 40), (40, 1000, 65, 128)])
def test_masks_of_any_row_length_and_start(fv, h, sq, sk, d, per_head, act16):
    """Mask rows that are no whole 16-byte units, in storage that starts one, two and three floats past one: the bits of
    the same mask at an aligned start, and the f64 result."""
    import torch

    announce(f"composed mask rows h={h} sq={sq} sk={sk} d={d} per_head={per_head} act16={act16}")
    g = torch.Generator(device="cuda").manual_seed(sq + sk)
    q, k, v = (torch.randn((1, h, s, d), generator=g, device="cuda") for s in (sq, sk, sk))
    if act16:
        q, k, v = (x.to(torch.bfloat16) for x in (q, k, v))
    n = (h if per_head else 1) * sq * sk
    values = torch.randn(n, generator=g, device="cuda")
    base = None
    for shift in range(4):
        store = torch.full((n + 8,), 1e9, device="cuda")
        store[shift:shift + n] = values
        mask = store[shift:shift + n].view(1, h if per_head else 1, sq, sk)
        with fv.with_bf16_act(act16):
            got = fv.sdpa(q, k, v, fv.Plan.masked(None, mask) if act16 else fv.Plan.composed(None, mask))
        if base is None:
            base = got
            want = want64(q, k, v, mask)
            assert np.linalg.norm(got.double().cpu().numpy() - want) <= (2e-3 if act16 else 2e-6) * np.linalg.norm(want)
        assert torch.equal(got, base), shift
