"""Operands longer than one launch holds (2^32 work-items in a grid dimension; past it the runtime cuts the size off
without an error): every element, in its place."""
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
