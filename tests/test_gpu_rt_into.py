"""`fv_rt_sdpa_into`, the one entry writing into the caller's memory: bit-identical to `fv_rt_sdpa` whatever part of the
workspace is given, and the refusals of a buffer that does not fit. The KV-cache windows `update` returns are views of
one tensor per layer: still valid after the cache object is gone."""
import ctypes

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


def parts(torch, q, k, v, kind=0):
    from fv_sdpa.sdpa import _FvPlan, _desc

    p = _FvPlan()
    p.kind, p.kv_flash = kind, -1
    need = (ctypes.c_size_t * 2)()
    return _desc(q, "q"), _desc(k, "k"), _desc(v, "v"), p, need


@pytest.mark.parametrize("sq,sk,dtype", [(300, 200, "f32"), (100, 4096, "f32"), (100, 4096, "bf16"), (64, 64, "bf16")])
def test_the_workspace_is_optional(fv, sq, sk, dtype):
    """f32 operands (rounded copies) and a split-KV shape (partials): whole workspace, half of it, none."""
    import torch

    announce(f"rt into {sq}x{sk} {dtype}")
    g = torch.Generator(device="cuda").manual_seed(sq + sk)
    q, k, v = (torch.randn((1, 2, s, 128), generator=g, device="cuda") for s in (sq, sk, sk))
    if dtype == "bf16":
        q, k, v = (x.to(torch.bfloat16) for x in (q, k, v))
    dq, dk, dv, p, need = parts(torch, q, k, v)
    lib, st = fv.lib(), torch.cuda.current_stream().cuda_stream
    R = ctypes.byref
    assert lib.fv_rt_sdpa_need(R(dq), R(dk), R(dv), R(p), need) == 0
    assert need[0] == 1 and (need[1] > 0) == (dtype == "f32" or sk == 4096)
    want = fv.sdpa(q, k, v, fv.Plan.dense(None))
    for nbytes in {need[1], need[1] // 2 // 256 * 256, 0}:
        out = torch.full_like(want, float("nan"))
        work = torch.empty(max(nbytes, 256), device="cuda", dtype=torch.uint8)
        assert lib.fv_rt_sdpa_into(R(dq), R(dk), R(dv), R(p), out.data_ptr(), out.numel() * 2, work.data_ptr(), nbytes, st) == 0
        torch.cuda.synchronize()
        assert torch.equal(out, want), nbytes


@pytest.mark.parametrize("h,sq,sk,d,kind", [(24, 3000, 700, 128, 1), (12, 4096, 1024, 64, 1), (38, 1700, 2100, 128, 0)])
def test_a_split_tail_and_its_workspace(fv, h, sq, sk, d, kind):
    """A composed launch on f32 operands whose last query tiles are cut by key ranges: the same bits with the whole
    workspace, half of it and none (then allocated). A dense one whose last round is split: split in the caller's
    workspace only, without it the unsplit launch's bits."""
    import torch

    announce(f"rt into tail {h}x{sq}x{sk}x{d} kind={kind}")
    g = torch.Generator(device="cuda").manual_seed(sq)
    q, k, v = (torch.randn((1, h, s, d), generator=g, device="cuda") for s in (sq, sk, sk))
    if kind == 0:
        q, k, v = (x.to(torch.bfloat16) for x in (q, k, v))
    dq, dk, dv, p, need = parts(torch, q, k, v, kind)
    lib, st = fv.lib(), torch.cuda.current_stream().cuda_stream
    R = ctypes.byref
    assert lib.fv_rt_sdpa_need(R(dq), R(dk), R(dv), R(p), need) == 0 and need[1] > 0
    assert need[0] == (1 if kind == 0 else 0)
    want = fv.sdpa(q, k, v, fv.Plan.dense() if kind == 0 else fv.Plan.composed())
    whole = fv.sdpa_dense_bf16(q[0], k[0], v[0], out_bf16=True)[None] if kind == 0 else want
    assert kind == 1 or not torch.equal(whole, want)
    for nbytes, expect in ((need[1], want), (need[1] // 2 // 256 * 256, whole), (0, whole)):
        out = torch.full_like(want, float("nan"))
        work = torch.empty(max(nbytes, 256), device="cuda", dtype=torch.uint8)
        assert lib.fv_rt_sdpa_into(R(dq), R(dk), R(dv), R(p), out.data_ptr(), out.numel() * out.element_size(),
                                   work.data_ptr(), nbytes, st) == 0
        torch.cuda.synchronize()
        assert torch.equal(out, expect), nbytes


@pytest.mark.parametrize("h,sq,sk", [(38, 1700, 2100), (2, 100, 3000)])
def test_f32_row_windows_and_the_workspace(fv, h, sq, sk):
    """f32 keys and values that are row windows of longer planes are compacted, rounded and split like contiguous ones:
    the workspace holds all three, the bits are the same."""
    import torch

    announce(f"rt into f32 windows {h}x{sq}x{sk}")
    g = torch.Generator(device="cuda").manual_seed(h)
    q = torch.randn((1, h, sq, 128), generator=g, device="cuda")
    k, v = (torch.randn((1, h, sk + 64, 128), generator=g, device="cuda") for _ in range(2))
    want = fv.sdpa(q, k[:, :, 16:16 + sk].contiguous(), v[:, :, :sk].contiguous(), fv.Plan.dense())
    got = fv.sdpa(q, k[:, :, 16:16 + sk], v[:, :, :sk], fv.Plan.dense())
    torch.cuda.synchronize()
    assert torch.equal(got, want)


def test_refusals(fv):
    import torch

    x = torch.zeros((1, 2, 64, 128), device="cuda", dtype=torch.bfloat16)
    out = torch.full_like(x, 3.0)
    dq, dk, dv, p, _ = parts(torch, x, x, x)
    lib, st = fv.lib(), torch.cuda.current_stream().cuda_stream
    R = ctypes.byref
    n = out.numel() * 2
    for args, needle in (((out.data_ptr(), n - 2, None, 0), "result buffer"), ((None, n, None, 0), "null argument"),
                         ((out.data_ptr(), n, out.data_ptr() + 16, 256), "256-byte aligned")):
        assert lib.fv_rt_sdpa_into(R(dq), R(dk), R(dv), R(p), *args, st) == -1
        assert needle in lib.fv_sdpa_last_error().decode()
    p.kind = 9
    assert lib.fv_rt_sdpa_into(R(dq), R(dk), R(dv), R(p), out.data_ptr(), n, None, 0, st) == -1
    torch.cuda.synchronize()
    assert bool((out == 3.0).all())


def test_windows_outlive_their_cache(fv):
    import gc
    import torch

    ft, d = 16, 64
    cache = fv.CausalKvCache(fv.KvSpec.rolling_window(ft, 3, 1), 2)
    k = [torch.randn((1, 2, ft, d), device="cuda").to(torch.bfloat16) for _ in range(6)]
    for i, x in enumerate(k[:5]):
        cache.update(1, x, -x, i * ft)
    kw, vw = cache.update(1, k[5], -k[5], 5 * ft)
    want = torch.cat([k[0], k[4], k[5]], dim=2)       # the sink frame, then the last two
    assert torch.equal(kw, want) and torch.equal(vw, -want)
    del cache
    gc.collect()
    junk = torch.full((1 << 20,), 9.0, device="cuda")
    assert torch.equal(kw, want) and torch.equal(vw, -want) and float(junk[0]) == 9.0


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_windows_of_a_cache_first_written_in_inference_mode(fv, dtype):
    """The windows a later call outside inference mode gets are ordinary tensors: autograd may save them."""
    import torch

    ft, d = 16, 64
    cache = fv.CausalKvCache(fv.KvSpec.global_window(ft, 4), 1)
    mk = lambda: torch.randn((1, 2, ft, d), device="cuda").to(torch.bfloat16 if dtype == "bf16" else torch.float32)
    k = [mk() for _ in range(2)]
    with torch.inference_mode():
        cache.update(0, k[0], k[0], 0)
    kw, vw = cache.update(0, k[1], k[1], ft)
    assert not kw.is_inference() and not vw.is_inference()
    w = torch.ones((), device="cuda", requires_grad=True, dtype=kw.dtype)
    (w * kw).sum().backward()
    assert torch.equal(kw, torch.cat(k, dim=2)) and w.grad is not None
