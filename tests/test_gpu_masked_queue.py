"""The queue that long masked launches at 128 channels take their items from through `sdpa` (fv_masked_workspace_bytes): the
bits of the launch in the order of the workgroups' numbers, which the kernel-level entries make."""
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


def queue_bytes(fv, q, plan):
    import ctypes

    from fv_sdpa.sdpa import _desc_bytes, _plan_bytes

    need = (ctypes.c_size_t * 2)()
    assert fv.lib().fv_rt_sdpa_need(*[_desc_bytes(q, "q")] * 3, _plan_bytes(plan, 0, 256), need) == 0
    return need[1]


# eight rounds of query tiles: lists of shared heads only, of whole and shared ones, of whole ones, with one shared head
# (at 64 channels such launches go without it)
QUEUE = [(3, 175200, 64), (12, 44000, 128), (16, 33000, 128), (41, 13000, 64), (3, 175200, 128), (41, 13000, 128)]


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
    assert queue_bytes(fv, q, plan) == (1024 if d == 128 else 0)
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


def call_into(fv, q, k, v, plan, work, own):
    """fv_rt_sdpa_into with the test's own workspace on the current stream -> the result (bf16)."""
    import ctypes

    import torch
    from fv_sdpa import _lib
    from fv_sdpa.sdpa import _desc_bytes, _plan_bytes

    out = torch.empty_like(q)
    rc = fv.lib().fv_rt_sdpa_into(*(_desc_bytes(x, "x") for x in (q, k, v)), _plan_bytes(plan, 0, 256 if own else 0),
                                  out.data_ptr(), out.numel() * 2, work.data_ptr(), work.numel(), _lib.stream())
    assert rc == 0, ctypes.string_at(fv.lib().fv_sdpa_last_error())
    return out


# lists of shared heads only, of whole and shared ones, with one shared head: 128 channels, where a bf16 result takes the queue
@pytest.mark.parametrize("h,s", [(3, 175200), (12, 44000), (41, 13000)])
def test_the_items_come_from_the_queue(fv, h, s):
    """A call with a workspace of its own draws every item from the eight counters (32 words apart), one that shares its
    workspace leaves it alone; the bits are the same, also where a late key makes items go again with the running max."""
    import torch

    announce(f"queue counters h={h} s={s}")
    g = torch.Generator(device="cuda").manual_seed(h)
    q, k, v = (torch.randn((1, h, s, 128), generator=g, device="cuda").to(torch.bfloat16) for _ in range(3))
    t = s // 11
    plan = fv.Plan.block_causal(None, fv.BlockCausal(t, 0, 0))
    items = h * ((s + 255) // 256)
    for late in (False, True):
        if late:
            k[:, 0, s // 2:] *= 40.0
        n0 = fv.lib().fv_sdpa_exact_pass_reruns()
        want = fv.sdpa_block_causal_bf16(q[0], k[0], v[0], t, 0, 0, out_bf16=True)
        torch.cuda.synchronize()
        n1 = fv.lib().fv_sdpa_exact_pass_reruns()
        assert (n1 > n0) == late
        work = torch.full((1024,), 0x55, device="cuda", dtype=torch.uint8)
        assert torch.equal(call_into(fv, q, k, v, plan, work, own=False)[0], want)
        assert bool((work == 0x55).all())
        n2 = fv.lib().fv_sdpa_exact_pass_reruns()
        assert torch.equal(call_into(fv, q, k, v, plan, work, own=True)[0], want)
        torch.cuda.synchronize()
        assert fv.lib().fv_sdpa_exact_pass_reruns() - n2 == n1 - n0
        drawn = work.view(torch.int32)
        assert int(drawn[::32].sum()) >= items and int(drawn.count_nonzero()) == 8


def test_two_streams_share_a_workspace(fv):
    """Two long masked calls on bf16 operands in flight with one workspace, as they may be: neither has it for its own."""
    import torch

    announce("two streams, one workspace")
    g = torch.Generator(device="cuda").manual_seed(9)
    sets = [[torch.randn((1, 12, 44000, 128), generator=g, device="cuda").to(torch.bfloat16) for _ in range(3)] for _ in range(2)]
    plan = fv.Plan.block_causal(None, fv.BlockCausal(4400, 0, 0))
    want = [fv.sdpa(*x, plan) for x in sets]
    work = torch.zeros(1 << 20, device="cuda", dtype=torch.uint8)
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in sets]
    got = []
    for x, s in zip(sets, streams):
        with torch.cuda.stream(s):
            got.append(call_into(fv, *x, plan, work, own=False))
    torch.cuda.synchronize()
    for a, b in zip(got, want):
        assert torch.equal(a, b)
