"""Masked launches: waves whose queries lie on both sides of a frame boundary, so that whole key tiles are seen by some of
them and hidden from the others, next to tiles that a boundary cuts."""
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


# (block tokens, window, sink) or (video start, frame tokens, frames, chunk, radius): boundaries inside a wave's 32 queries,
# hidden ranges of whole tiles and of one tile with a remainder on either side
CAUSAL = [(300, 1, 0), (333, 2, 1), (200, 0, 0), (129, 1, 1)]
WINDOW = [(0, 300, 6, 0, 0), (10, 210, 8, 2, 0), (65, 190, 9, 0, 1)]


@pytest.mark.parametrize("out_bf16", [False, True])
@pytest.mark.parametrize("d", [128, 64])
@pytest.mark.parametrize("mask", CAUSAL + WINDOW)
def test_tiles_hidden_from_some_queries_of_a_wave(fv, oracle, mask, d, out_bf16):
    """Keys that a query does not see may hold anything: the last frame's are NaN for the queries before it (causal)."""
    import torch

    announce(f"hidden tiles mask={mask} d={d} bf16={out_bf16}")
    s = 1850
    q, k, v = qkv(sum(mask) + d, 2, s, s, d)
    qd, kd, vd = (to_dev_bf16(x) for x in (q, k, v))
    if len(mask) == 3:
        want = oracle.sdpa_composed(q, k, v, mask=oracle.block_causal_dense_mask(*mask, s, s))
        run = lambda kk: fv.sdpa_block_causal_bf16(qd, kk, vd, *mask, out_bf16=out_bf16)
    else:
        want = oracle.sdpa_composed(q, k, v, mask=oracle.vdn_window_dense_mask(*mask, s, s))
        run = lambda kk: fv.sdpa_vdn_window_bf16(qd, kk, vd, *mask, out_bf16=out_bf16)
    got = run(kd).float().cpu().numpy()
    assert_parity(got, want, f"hidden_{mask}_{d}")
    if len(mask) == 3:
        first = (s - 1) // mask[0] * mask[0]   # of the last block
        poisoned = kd.clone()
        poisoned[:, first:] = float("nan")
        again = run(poisoned).float().cpu().numpy()
        # (not the same bits: a wave moves the offsets of all its queries when one of them asks for it)
        assert_parity(again[:, :first], want[:, :first], f"hidden_nan_{mask}_{d}")


# bounds at every place of a tile's word of 64 keys, its ends among them; 33 heads: flash_fwd_duo where the result is bf16
@pytest.mark.parametrize("out_bf16", [False, True])
@pytest.mark.parametrize("d", [128, 64])
@pytest.mark.parametrize("frame", [1, 3, 16, 31, 32, 33, 63, 64, 65, 127, 128])
def test_frames_of_any_length(fv, oracle, frame, d, out_bf16):
    announce(f"frames of {frame} d={d} bf16={out_bf16}")
    h, s = 33, 6 * frame + 130
    q, k, v = qkv(frame + d, h, s, s, d)
    qd, kd, vd = (to_dev_bf16(x) for x in (q, k, v))
    # queries that see few keys have results as large as a value: P and the result are rounded to 8 bits, half a unit each, at
    # most 2^-8 max|v| from either; f32 sums and exponentials are a hundredth of that
    most = 1.01 * 2 * 2.0 ** -8 * float(abs(v).max())
    for args in ((frame, 0, 0), (frame, 2, 1), (frame, 3, 0)):
        want = oracle.sdpa_composed(q, k, v, mask=oracle.block_causal_dense_mask(*args, s, s))
        assert_parity(fv.sdpa_block_causal_bf16(qd, kd, vd, *args, out_bf16=out_bf16).float().cpu().numpy(), want, f"causal_{args}_{d}", max_abs=most)
    for args in ((65, frame, 6, 0, 1), (130, frame, 6, 2, 0), (7, frame, 5, 0, 0)):
        want = oracle.sdpa_composed(q, k, v, mask=oracle.vdn_window_dense_mask(*args, s, s))
        assert_parity(fv.sdpa_vdn_window_bf16(qd, kd, vd, *args, out_bf16=out_bf16).float().cpu().numpy(), want, f"window_{args}_{d}", max_abs=most)
