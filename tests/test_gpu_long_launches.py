"""Operands longer than one launch holds (2^32 work-items in a grid dimension; past it the runtime cuts the size off
without an error): every element, in its place."""
import math

import pytest

from util import announce

pytestmark = pytest.mark.gpu

LN2 = math.log(2.0)


@pytest.fixture(scope="module")
def fv():
    import torch

    assert torch.cuda.is_available()
    import fv_sdpa

    fv_sdpa.lib()
    return fv_sdpa


def test_cast_bf16_f32(fv):
    import torch

    n = (1 << 32) + 4099
    announce(f"cast n={n}")
    x = torch.empty(n, device="cuda", dtype=torch.bfloat16)
    step = 1 << 28
    for lo in range(0, n, step):
        x[lo:lo + step] = (torch.arange(lo, min(n, lo + step), device="cuda") % 251).to(torch.bfloat16)
    y = fv.cast_bf16_f32(x)
    torch.cuda.synchronize()
    assert all(torch.equal(y[lo:lo + step], x[lo:lo + step].float()) for lo in range(0, n, step))


@pytest.mark.parametrize("out_bf16", [False, True])
def test_softmax_of_many_short_rows(fv, out_bf16):
    import torch

    rows, width = (1 << 26) + 7, 3
    announce(f"softmax rows={rows} width={width} out_bf16={out_bf16}")
    x = torch.randn((rows, width), device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    got = fv.softmax_last(x, out_bf16=out_bf16)
    torch.cuda.synchronize()
    step = 1 << 23
    for lo in range(0, rows, step):
        want = torch.softmax(x[lo:lo + step].double(), dim=-1)
        # a few f32 roundings of numbers up to one; a bf16 result: half a unit of its eight bits
        assert float((got[lo:lo + step].double() - want).abs().max()) <= (2.0 ** -8 if out_bf16 else 1e-6)


def test_topk_of_many_short_rows(fv):
    import torch

    rows = (1 << 26) + 5
    announce(f"topk rows={rows}")
    s = torch.randn((rows, 2), device="cuda", generator=torch.Generator(device="cuda").manual_seed(2))
    got = fv.vsa_topk(s, 1)
    torch.cuda.synchronize()
    assert torch.equal(got[:, 0], (s[:, 1] > s[:, 0]).to(torch.int32))


@pytest.mark.parametrize("d", [128, 64])
def test_planes_of_four_gigabytes(fv, d):
    """Keys whose plane passes 4 GB, past which tile loads address by tile: dense, split by key ranges and block-causal, and
    the longest plane below. Two far keys hold the rows, so a wrong address shows; P and the result are rounded to bf16,
    2^-9 each."""
    import torch

    announce(f"planes of 4 GB d={d}")
    rows = (1 << 32) // (2 * d)
    sq, sk = 5, rows + 70
    k = torch.zeros((1, sk, d), device="cuda", dtype=torch.bfloat16)
    v = torch.zeros((1, sk, d), device="cuda", dtype=torch.bfloat16)
    g = torch.Generator(device="cuda").manual_seed(d)
    q = torch.ones((1, sq, d), device="cuda", dtype=torch.bfloat16)
    far = [0, rows // 2 + 3, rows - 70, rows - 1, rows, rows + 5, sk - 1]
    for i, at in enumerate(far):
        k[0, at] = 3.0 + 0.125 * i
        v[0, at] = torch.randn(d, generator=g, device="cuda").to(torch.bfloat16)

    def want(n):
        at = [x for x in far if x < n]
        s = torch.full((1,), 0.0, dtype=torch.float64)
        w = torch.exp(torch.stack([k[0, x].double().sum() / d ** 0.5 for x in at]).cpu())
        others = (n - len(at)) * torch.exp(s)
        return sum(wi * v[0, x].double().cpu() for wi, x in zip(w, at)) / (w.sum() + others)

    def close(got, n):
        ref = want(n)
        assert ((got.double().cpu() - ref).norm(dim=-1) / ref.norm()).max().item() <= 2.0 ** -7

    for out_bf16 in (True, False):
        close(fv.sdpa_dense_bf16(q, k, v, out_bf16=out_bf16)[0], sk)
    close(fv.sdpa(q[None], k[None], v[None], fv.Plan.dense())[0, 0], sk)
    block = rows // 2 + 10
    close(fv.sdpa_block_causal_bf16(q, k, v, block, 0, 2, out_bf16=True)[0], 2 * block)
    close(fv.sdpa_dense_bf16(q, k[:, :rows - 1].contiguous(), v[:, :rows - 1].contiguous(), out_bf16=True)[0], rows - 1)


@pytest.mark.parametrize("d", [128, 64])
def test_planes_of_four_gigabytes_keep_every_form(fv, d):
    """Past 4 GB a call has the forms that it has below: scale * log2(e) = 1 without the multiply (counted), a bf16 result
    with a fixed offset (a late key that outgrows it makes the second pass, counted), query tiles of 128."""
    import torch

    announce(f"forms of planes of 4 GB d={d}")
    lib, rows, sq = fv.lib(), (1 << 32) // (2 * d), 130
    sk = rows + 70
    k = torch.zeros((1, sk, d), device="cuda", dtype=torch.bfloat16)
    v = torch.zeros((1, sk, d), device="cuda", dtype=torch.bfloat16)
    q = torch.ones((1, sq, d), device="cuda", dtype=torch.bfloat16)
    v[0, rows + 5] = torch.randn(d, generator=torch.Generator(device="cuda").manual_seed(d), device="cuda").to(torch.bfloat16)
    k[0, rows + 5] = 0.5   # d / 2 bits above the others, which are 2^24 and 2^25: the row is its value
    want = v[0, rows + 5].double()
    n0, r0 = lib.fv_sdpa_log2_domain_launches(), lib.fv_sdpa_exact_pass_reruns()
    near = [fv.sdpa_dense_bf16(q, k, v, scale=LN2, out_bf16=True)[0],
            fv.sdpa_dense_bf16(q, k, v, scale=LN2)[0],
            fv.sdpa_block_causal_bf16(q, k, v, rows, 0, 2, scale=LN2, out_bf16=True)[0],
            fv.sdpa(q[None], k[None], v[None], fv.Plan.dense(LN2))[0, 0]]
    torch.cuda.synchronize()
    assert lib.fv_sdpa_log2_domain_launches() == n0 + 4 and lib.fv_sdpa_exact_pass_reruns() == r0
    for got in near:   # the others' share of the sum is below 2^(25 - 32); P and the result are rounded to bf16
        assert float((got.double() - want).abs().max()) <= 2.0 ** -6 * float(want.abs().max())
    k[0, rows + 5] = 16.0   # 184 and 261 bits: past the range of the fixed offset
    for fn in (lambda: fv.sdpa_dense_bf16(q, k, v, out_bf16=True), lambda: fv.sdpa_block_causal_bf16(q, k, v, rows, 0, 2, out_bf16=True)):
        r0 = lib.fv_sdpa_exact_pass_reruns()
        far = fn()[0]
        torch.cuda.synchronize()
        assert lib.fv_sdpa_exact_pass_reruns() == r0 + 1
        assert float((far.double() - want).abs().max()) <= 2.0 ** -8 * float(want.abs().max())


@pytest.mark.parametrize("d", [128, 64])
def test_vdn_window_on_planes_of_four_gigabytes(fv, d):
    import torch

    announce(f"VDN window on planes of 4 GB d={d}")
    t, rows = 64, (1 << 32) // (2 * d)
    frames = rows // t + 1
    s, vs = t * frames + 90, 40
    g = torch.Generator(device="cuda").manual_seed(d)
    q, k, v = (torch.randn((1, s, d), generator=g, device="cuda", dtype=torch.bfloat16) for _ in range(3))
    for out_bf16 in (True, False):
        got = fv.sdpa_vdn_window_bf16(q, k, v, vs, t, frames, 0, 1, out_bf16=out_bf16)[0]
        for i in (vs + t, vs + 5 * t - 1, rows // 2, rows - 1, rows, s - 50 - t - 1):
            f = (i - vs) // t
            seen = torch.zeros(s, dtype=torch.bool, device="cuda")
            for a, b in ((0, vs + t), (vs + (f - 1) * t, vs + (f + 2) * t), (vs + (frames - 1) * t, s)):
                seen[a:b] = True
            at = seen.nonzero()[:, 0]
            p = torch.softmax(k[0, at].double() @ q[0, i].double() / d ** 0.5, 0)
            ref = p @ v[0, at].double()
            # P and the result rounded to 8 bits, half a unit of each
            bound = 2.0 ** -8 * (p @ v[0, at].double().abs() + ref.abs()) + 1e-5
            assert bool(((got[i].double() - ref).abs() <= bound).all()), (out_bf16, i)
