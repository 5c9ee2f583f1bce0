"""Dense calls small enough for the short kernel, at the edges of its rule and of its tiles: one row more and less than a
query group and a key tile, fewer tiles than waves, one more than a whole round of tiles, 256 and 272 (512 and 513, 768 and 792) query
groups, the longest keys it takes, operands that are row windows of longer planes.

Against the f64 softmax on the same operands. P is rounded to bf16, 2^-9 of each weight at most, and so is a bf16 result:
2^-9 in the 2-norm for an f32 one, twice that for a bf16 one."""
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


def operands(torch, seed, b, h, sq, sk, d):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn((b, h, s, d), generator=g, device="cuda").to(torch.bfloat16) for s in (sq, sk, sk)]


def want64(q, k, v):
    q, k, v = (x.double().cpu() for x in (q, k, v))
    return ((q @ k.transpose(-1, -2)) / np.sqrt(q.shape[-1])).softmax(-1) @ v


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("b,h,sq,sk", [
    (1, 1, 1, 1), (1, 2, 31, 31), (2, 1, 32, 32), (1, 3, 33, 33), (1, 2, 64, 127), (1, 1, 40, 128), (1, 2, 97, 129),
    (1, 3, 65, 255), (1, 2, 32, 256), (2, 2, 100, 257), (1, 5, 70, 289), (1, 3, 200, 513),
    (1, 255, 20, 100), (1, 256, 20, 100), (1, 64, 128, 90), (1, 16, 513, 90),    # 255 (and as many query tiles), 256 and 272 groups
    (1, 16, 1024, 90), (1, 19, 864, 90), (1, 24, 1024, 70), (1, 24, 1025, 70),   # 512, 513, 768 and 792
    (1, 2, 100, 3072), (1, 2, 100, 3073), (1, 20, 420, 2048),                    # the longest walks and one key more
])
def test_edges(fv, b, h, sq, sk, d):
    import torch

    announce(f"short {b}x{h}x{sq}x{sk}x{d}")
    q, k, v = operands(torch, sq + sk, b, h, sq, sk, d)
    want = want64(q, k, v)
    for act16, bound in ((True, 2 * 2.0 ** -9), (False, 2.0 ** -9)):
        with fv.with_bf16_act(act16):
            got = fv.sdpa(q, k, v, fv.Plan.dense()).double().cpu()
        assert torch.isfinite(got).all()
        assert (got - want).norm() <= bound * want.norm(), act16


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("sk", [200, 700])
def test_row_windows_and_nan_rows(fv, sk, d):
    """Keys and values read in place from longer planes give the contiguous call's bits; a NaN query is its own row's, a
    NaN key its head's."""
    import torch

    announce(f"short windows sk={sk} d={d}")
    b, h, sq = 2, 3, 75
    q, k, v = operands(torch, sk + d, b, h, sq, sk + 50, d)
    kw, vw = k[:, :, 17:17 + sk], v[:, :, 40:40 + sk]
    base = fv.sdpa(q, kw.contiguous(), vw.contiguous(), fv.Plan.dense())
    assert torch.equal(fv.sdpa(q, kw, vw, fv.Plan.dense()), base)
    q[1, 2, 33, 5] = float("nan")
    k[0, 1, 17 + sk - 1, 3] = float("nan")
    got = fv.sdpa(q, kw, vw, fv.Plan.dense())
    nan = torch.zeros((b, h, sq), dtype=torch.bool, device="cuda")
    nan[1, 2, 33] = True
    nan[0, 1] = True
    assert torch.equal(got.isnan().all(-1), nan) and torch.equal(got.isnan().any(-1), nan)
    assert torch.equal(got[~nan], base[~nan])


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("h,sq,sk", [(12, 320, 320), (3, 100, 700), (16, 640, 513)])   # eight waves, eight, four
def test_the_scale_folded_into_the_queries(fv, h, sq, sk, d):
    """scale = ln 2 takes the form without the multiply of every score, and is counted."""
    import torch

    announce(f"short log2 {h}x{sq}x{sk}x{d}")
    ln2 = float(np.float32(np.log(2.0)))
    q, k, v = operands(torch, sq + sk + d, 1, h, sq, sk, d)
    q = (q.float() * (1.4426950408889634 / np.sqrt(d))).to(torch.bfloat16)
    lib = fv.lib()
    n0 = lib.fv_sdpa_log2_domain_launches()
    got = fv.sdpa(q, k, v, fv.Plan.masked(ln2)).double().cpu()
    assert lib.fv_sdpa_log2_domain_launches() == n0 + 1
    q, k, v = (x.double().cpu() for x in (q, k, v))
    want = ((q @ k.transpose(-1, -2)) * ln2).softmax(-1) @ v
    assert (got - want).norm() <= 2 * 2.0 ** -9 * want.norm()
