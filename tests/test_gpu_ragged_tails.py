"""Rows of a last key tile past the keys: tile loads read zeros there, into LDS as well, and P V multiplies them by a
probability of zero without a mask of its own. What an earlier launch left in LDS, NaN values at worst, must not stay."""
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


# one round of query tiles of 128 and more than one of 256, few queries (half tiles, split keys); keys past one, two and many
# tiles by one, by half a tile and by all but one
@pytest.mark.parametrize("d", [128, 64])
@pytest.mark.parametrize("h,sq", [(12, 4000), (12, 1500), (5, 300)])
def test_nothing_of_an_earlier_launch_stays(fv, h, sq, d):
    import torch

    announce(f"ragged tails h={h} sq={sq} d={d}")
    g = torch.Generator(device="cuda").manual_seed(sq + d)
    rnd = lambda n: torch.randn((h, n, d), generator=g, device="cuda").to(torch.bfloat16)
    lq, lk = rnd(8192), rnd(2048)
    left = [torch.full_like(lk, x) for x in (0.0, float("nan"))]
    q = rnd(sq)

    def forms(n):
        k, v = rnd(n), rnd(n)
        t = max(1, n // 5)
        yield "dense bf16", lambda: fv.sdpa_dense_bf16(q, k, v, out_bf16=True)
        yield "dense f32", lambda: fv.sdpa_dense_bf16(q, k, v)
        yield "split", lambda: fv.sdpa(q[None], k[None], v[None], fv.Plan.kv_window())[0]
        yield "causal bf16", lambda: fv.sdpa_block_causal_bf16(q, k, v, max(t, sq), 0, 2, out_bf16=True)
        yield "causal f32", lambda: fv.sdpa_block_causal_bf16(q, k, v, max(t, sq // 2), 1, 0)
        kq, vq = rnd(sq), rnd(sq)
        yield "window", lambda: fv.sdpa_vdn_window_bf16(q, kq, vq, 3, (sq - 4) // 7, 7, 0, 1, out_bf16=True)

    for n in (65, 96, 127, 129, 2001, 7039):
        for name, run in forms(n):
            got = []
            for v in left:
                for bf16 in (True, False):   # (every CU's buffers, of both kernels)
                    fv.sdpa_dense_bf16(lq, lk, v, out_bf16=bf16)
                fv.sdpa_dense_bf16(lq, lk[:, :512].contiguous(), v[:, :512].contiguous(), out_bf16=True)
                got.append(run())
            torch.cuda.synchronize()
            assert bool(torch.isfinite(got[0]).all()), (name, n)
            assert torch.equal(got[0], got[1]), (name, n)
