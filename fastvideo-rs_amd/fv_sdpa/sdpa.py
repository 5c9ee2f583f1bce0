"""Python mirror of `rt::sdpa::sdpa(q, k, v, &Plan)` (crates/fastvideo-cudarc/src/rt/sdpa.rs:29-164)
over the library's C++ host layer (`fv_rt_sdpa`). Same constructors, same error
messages; tensors are torch CUDA tensors (device memory only).
"""
import ctypes as C
import struct
from contextlib import contextmanager

import torch

from . import _lib

__all__ = ["Plan", "BlockCausal", "VdnWindow", "sdpa", "with_bf16_act", "bf16_activations", "with_fold_scale", "fold_scale", "rt_stats", "TensorError",
           "BACKENDS", "STEPS", "parse_backend", "backend", "with_backend", "shape_of", "dense_route"]


class TensorError(RuntimeError):
    """rt/tensor.rs:92-98 `TensorError::Message`. `rc` is the C ABI's return: -hipErrorInvalidValue (-1) for a
    refused argument, the negated hipError_t of a failed allocation (-2 out of memory) or launch otherwise."""

    def __init__(self, message, rc=None):
        super().__init__(message)
        self.rc = rc


class _FvTensor(C.Structure):
    _fields_ = [("data", C.c_void_p), ("dtype", C.c_int), ("rank", C.c_int), ("shape", C.c_size_t * 8),
                ("plane_rows", C.c_size_t)]


class _FvPlan(C.Structure):
    _fields_ = [("kind", C.c_int), ("has_scale", C.c_int), ("scale", C.c_float), ("mask", C.POINTER(_FvTensor)),
                ("fp8_first", C.c_int), ("block_tokens", C.c_size_t), ("window", C.c_size_t), ("sink", C.c_size_t),
                ("video_start", C.c_size_t), ("frame_tokens", C.c_size_t), ("frames", C.c_size_t),
                ("chunk", C.c_size_t), ("radius", C.c_size_t), ("kv_flash", C.c_int)]


class BlockCausal:
    """rt/attn.rs:441-467."""

    def __init__(self, block_tokens, window=0, sink=0):
        self.block_tokens, self.window, self.sink = block_tokens, window, sink

    def allows(self, q, k):
        return bool(_lib.lib().fv_block_causal_allows(self.block_tokens, self.window, self.sink, q, k))

    def dense_mask(self, sq, sk):
        from .vsa import block_causal_dense_mask

        return block_causal_dense_mask(self.block_tokens, self.window, self.sink, sq, sk)


class VdnWindow:
    """rt/attn.rs:469-524."""

    def __init__(self, video_start, frame_tokens, frames, chunk=0, radius=0):
        self.video_start, self.frame_tokens, self.frames, self.chunk, self.radius = (video_start, frame_tokens,
                                                                                     frames, chunk, radius)

    def _args(self):
        return self.video_start, self.frame_tokens, self.frames, self.chunk, self.radius

    def video_end(self):
        return self.video_start + self.frames * self.frame_tokens

    def allows(self, q, k):
        return bool(_lib.lib().fv_vdn_window_allows(*self._args(), q, k))

    def dense_mask(self, sq, sk):
        import numpy as np

        m = np.empty((sq, sk), dtype=np.float32)
        _lib.lib().fv_vdn_window_dense_mask(*self._args(), sq, sk, m.ctypes.data)
        return m


class Plan:
    """rt/sdpa.rs:29-137."""

    DENSE, COMPOSED, BLOCK_CAUSAL, VDN_WINDOW, KV_WINDOW = range(5)

    def __init__(self, kind, scale=None, mask=None, fp8=False, causal=None, kv_flash=None, window=None):
        self.kind, self.scale, self.mask, self.fp8, self.causal, self.kv_flash = kind, scale, mask, fp8, causal, kv_flash
        self.window = window

    @staticmethod
    def dense(scale=None):
        return Plan.masked(scale, None)

    @staticmethod
    def masked(scale=None, mask=None):
        return Plan(Plan.DENSE, scale, mask)

    def fp8_first(self):
        if self.kind == Plan.DENSE and self.mask is None:
            return Plan(Plan.DENSE, self.scale, None, fp8=True)
        return self

    @staticmethod
    def composed(scale=None, mask=None):
        return Plan(Plan.COMPOSED, scale, mask)

    @staticmethod
    def block_causal(scale, mask):
        return Plan(Plan.BLOCK_CAUSAL, scale, causal=mask)

    @staticmethod
    def vdn_window(scale, mask):
        return Plan(Plan.VDN_WINDOW, scale, window=mask)

    @staticmethod
    def kv_window():
        return Plan(Plan.KV_WINDOW)

    @staticmethod
    def kv_window_with(flash):
        return Plan(Plan.KV_WINDOW, kv_flash=bool(flash))


def _window_rows(t):
    """plane_rows of a BHSD tensor that is a row window (`base[:, :, a:b]`) of a contiguous
    [b, h, rows, d] tensor, else None."""
    if t.dim() != 4:
        return None
    b, h, s, d = t.shape
    sb, sh, ss, sd = t.stride()
    if sd != 1 or ss != d or sh % d or sh < s * d or (b > 1 and sb != h * sh):
        return None
    return sh // d


# struct fv_tensor and struct fv_plan as bytes: packing one takes a microsecond where filling a ctypes structure field by
# field takes ten, as much as a small launch.
_TENSOR_BYTES = struct.Struct("@Pii9N")
_PLAN_BYTES = struct.Struct("@iifPi8Ni0P")
assert _TENSOR_BYTES.size == C.sizeof(_FvTensor) and _PLAN_BYTES.size == C.sizeof(_FvPlan)
_NO_SHAPE = (0,) * 8
_OWN_WORKSPACE = 256   # FV_PLAN_OWN_WORKSPACE, of these kinds
_OWN_KINDS = (Plan.BLOCK_CAUSAL, Plan.VDN_WINDOW)
_BF16, _F32 = torch.bfloat16, torch.float32


def _desc_bytes(t, name):
    """`t` as the bytes of a struct fv_tensor."""
    if not (isinstance(t, torch.Tensor) and t.is_cuda):
        raise ValueError(f"{name}: want a contiguous CUDA tensor")
    rows = 0
    if not t.is_contiguous():
        rows = _window_rows(t) or 0
        if not rows:
            raise ValueError(f"{name}: want a contiguous CUDA tensor or a row window of a BHSD one")
    dtype = t.dtype
    if dtype is _BF16:
        bf16 = 1
    elif dtype is _F32:
        bf16 = 0
    else:
        raise ValueError(f"{name}: want f32 or bf16")
    shape = t.shape
    rank = len(shape)
    if rank == 4:
        return _TENSOR_BYTES.pack(t.data_ptr(), bf16, 4, *shape, 0, 0, 0, 0, rows)
    if rank > 8:
        raise ValueError(f"{name}: rank > 8")
    return _TENSOR_BYTES.pack(t.data_ptr(), bf16, rank, *shape, *_NO_SHAPE[rank:], rows)


def _desc(t, name):
    return _FvTensor.from_buffer_copy(_desc_bytes(t, name))


def _plan_bytes(plan, mask, flags=0):
    """`plan` as the bytes of a struct fv_plan; `mask`: the address of its mask's struct fv_tensor, or 0;
    `flags`: or'ed into its kind."""
    scale, causal, window, kind = plan.scale, plan.causal, plan.window, plan.kind
    if flags:
        kind |= flags
    causal = (causal.block_tokens, causal.window, causal.sink) if causal is not None else (0, 0, 0)
    window = window._args() if window is not None else (0, 0, 0, 0, 0)
    kv_flash = -1 if plan.kv_flash is None else int(plan.kv_flash)
    try:
        return _PLAN_BYTES.pack(kind, 0 if scale is None else 1, 0.0 if scale is None else scale, mask,
                                1 if plan.fp8 else 0, *causal, *window, kv_flash)
    except (struct.error, OverflowError):
        # numbers that do not fit their fields (negative, a scale past f32): what C makes of them, for the library to judge
        p = _FvPlan()
        p.kind, p.fp8_first, p.kv_flash = kind, 1 if plan.fp8 else 0, kv_flash
        p.has_scale, p.scale = (0, 0.0) if scale is None else (1, float(scale))
        p.mask = C.cast(C.c_void_p(mask), C.POINTER(_FvTensor))
        p.block_tokens, p.window, p.sink = causal
        p.video_start, p.frame_tokens, p.frames, p.chunk, p.radius = window
        return bytes(p)


def sdpa(q, k, v, plan):
    """rt/sdpa.rs:141-164. Returns a new [b, h, sq, d] tensor (bf16 under bf16 activations, else f32)."""
    lib = _lib.lib()
    dq, dk, dv = _desc_bytes(q, "q"), _desc_bytes(k, "k"), _desc_bytes(v, "v")
    mask = None
    if plan.mask is not None:
        mask = C.create_string_buffer(_desc_bytes(plan.mask, "mask"), _TENSOR_BYTES.size)   # alive until the call is made
    # (the workspace of a block-causal or window call is allocated below, for it alone)
    p = _plan_bytes(plan, 0 if mask is None else C.addressof(mask), _OWN_WORKSPACE if plan.kind in _OWN_KINDS else 0)
    need = (C.c_size_t * 2)()
    rc = lib.fv_rt_sdpa_need(dq, dk, dv, p, need)
    if rc != 0:
        raise TensorError(lib.fv_sdpa_last_error().decode(), rc)
    bf16, nbytes = need
    # (the shape of q is the result's: the library refuses anything else before it writes)
    dtype = _BF16 if bf16 else _F32
    try:
        if type(q) is torch.Tensor and q.dtype is dtype and q.is_contiguous():
            res = torch.empty_like(q, memory_format=torch.contiguous_format)   # half the time of an empty() by shape
        else:
            res = torch.empty(q.shape, device=q.device, dtype=dtype)
    except torch.cuda.OutOfMemoryError as e:
        raise TensorError(f"sdpa: device allocation failed: {e}", -2) from e   # hipErrorOutOfMemory
    try:
        work = torch.empty(nbytes, device=q.device, dtype=torch.uint8) if nbytes else None
    except torch.cuda.OutOfMemoryError:
        nbytes = 0   # the library allocates what it cannot do without, or refuses
    rc = lib.fv_rt_sdpa_into(dq, dk, dv, p, res.data_ptr(), res.numel() * (2 if bf16 else 4),
                             work.data_ptr() if nbytes else None, nbytes, _lib.stream())
    if rc != 0:
        raise TensorError(lib.fv_sdpa_last_error().decode(), rc)
    return res


def bf16_activations():
    return bool(_lib.lib().fv_rt_bf16_activations())


@contextmanager
def with_bf16_act(on):
    """rt/tensor.rs `with_bf16_act(on, f)`."""
    lib = _lib.lib()
    lib.fv_rt_set_bf16_activations(int(bool(on)))
    try:
        yield
    finally:
        lib.fv_rt_set_bf16_activations(-1)


def fold_scale():
    return bool(_lib.lib().fv_rt_fold_scale())


@contextmanager
def with_fold_scale(on):
    """Per-thread override of FASTVIDEO_SDPA_FOLD_SCALE: whether `sdpa` folds scale * log2(e) into the one
    rounding of an f32 q (and runs the kernel at scale = ln 2)."""
    lib = _lib.lib()
    lib.fv_rt_set_fold_scale(int(bool(on)))
    try:
        yield
    finally:
        lib.fv_rt_set_fold_scale(-1)


def rt_stats():
    out = (C.c_uint64 * 5)()
    _lib.lib().fv_rt_stats(out)
    return dict(zip(("fused", "causal", "composed", "casts", "masks"), (int(x) for x in out)))


# rt/sdpa_rule.rs:178-207 `Backend` and the collapsed `Step` (the NVIDIA alternates are gone)
BACKENDS = ("dense", "cublas", "flash", "host", "sparse")
STEPS = ("retired", "fused", "composed")


def parse_backend(v):
    """rt/sdpa_rule.rs:199-207: a FASTVIDEO_SDPA value -> backend name (unknown = "dense")."""
    return BACKENDS[_lib.lib().fv_rt_parse_backend(str(v).encode())]


def backend():
    return BACKENDS[_lib.lib().fv_rt_backend()]


@contextmanager
def with_backend(name):
    """Per-thread override of FASTVIDEO_SDPA for the calls inside the block."""
    lib = _lib.lib()
    lib.fv_rt_set_backend(BACKENDS.index(name))
    try:
        yield
    finally:
        lib.fv_rt_set_backend(-1)


def _shape4(x):
    x = tuple(int(i) for i in x)
    if len(x) != 4:
        raise TensorError("sdpa expects BHSD")
    return (C.c_size_t * 4)(*x)


def dense_route(q_shape, k_shape, v_shape, masked=False, backend_name="dense"):
    """rt/sdpa_rule.rs:409-437: the kernels a dense call tries, in order."""
    steps = (C.c_int * 4)()
    n = _lib.lib().fv_rt_dense_route(_shape4(q_shape), _shape4(k_shape), _shape4(v_shape), int(bool(masked)),
                                     BACKENDS.index(backend_name), steps, None)
    if n < 0:
        raise TensorError("dense_route: bad arguments")
    return [STEPS[steps[i]] for i in range(n)]


def shape_of(q_shape, k_shape, v_shape):
    """rt/sdpa_rule.rs:373-390 `Shape::of`: (sq, sk, dims) with dims = (b, h, sq, sk, d) or None."""
    steps, dims = (C.c_int * 4)(), (C.c_size_t * 5)()
    _lib.lib().fv_rt_dense_route(_shape4(q_shape), _shape4(k_shape), _shape4(v_shape), 0, 0, steps, dims)
    d = tuple(int(x) for x in dims)
    return int(q_shape[2]), int(k_shape[2]), (d if any(d) else None)
