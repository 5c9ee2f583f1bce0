"""The queue that masked launches of eight rounds and more take their items from through `sdpa`: the bits of the
launch in the order of the workgroups' numbers, which the kernel-level entries make."""
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


# eight rounds of query tiles: lists of shared heads only, of whole and shared ones, of whole ones, with one shared head
QUEUE = [(3, 175200, 64), (12, 44000, 128), (16, 33000, 128), (41, 13000, 64)]


@pytest.mark.parametrize("kind", ["causal", "sink", "window"])
@pytest.mark.parametrize("h,s,d", QUEUE)
def test_the_queue_gives_the_bits_of_the_launch_without_it(fv, h, s, d, kind):
    import torch

    announce(f"queue h={h} s={s} d={d} {kind}")
    g = torch.Generator(device="cuda").manual_seed(h + s)
    q, k, v = (torch.randn((1, h, s, d), generator=g, device="cuda").to(torch.bfloat16) for _ in range(3))
    t = s // 11
    if kind == "window":
        plan = fv.Plan.vdn_window(None, fv.VdnWindow(s - 10 * t - 5, t, 10, 2, 1))
        args = (s - 10 * t - 5, t, 10, 2, 1)
    else:
        args = (t, 0, 0) if kind == "causal" else (t, 5, 1)
        plan = fv.Plan.block_causal(None, fv.BlockCausal(*args))
    fn = fv.sdpa_vdn_window_bf16 if kind == "window" else fv.sdpa_block_causal_bf16
    for bf16 in (True, False):
        want = fn(q[0], k[0], v[0], *args, out_bf16=bf16)
        with fv.with_bf16_act(bf16):
            got = [fv.sdpa(q, k, v, plan) for _ in range(2)]   # (the second one's memory for the queue has been used)
        torch.cuda.synchronize()
        for x in got:
            assert x.dtype == (torch.bfloat16 if bf16 else torch.float32)
            assert torch.equal(x[0], want)


def test_the_queue_in_a_graph(fv):
    """Replays with other work and a synchronisation between them: every one clears its own counters."""
    import torch

    announce("queue in a graph")
    g = torch.Generator(device="cuda").manual_seed(5)
    q, k, v = (torch.randn((1, 12, 44000, 128), generator=g, device="cuda").to(torch.bfloat16) for _ in range(3))
    plan = fv.Plan.block_causal(None, fv.BlockCausal(4400, 0, 0))
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        fv.sdpa(q, k, v, plan)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fv.sdpa(q, k, v, plan)
    for i in range(4):
        q.normal_(generator=g)
        want = fv.sdpa(q, k, v, plan)
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), i
