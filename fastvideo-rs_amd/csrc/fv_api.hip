// C ABI of libfv_sdpa_hip.so: argument checks, decline rules and launches.
// Declarations and reference citations live in include/fv_sdpa_hip.h.
#include "../../include/fv_sdpa_hip.h"

#include <limits.h>
#include <stdio.h>

#include <algorithm>
#include <atomic>
#include <string>

#include "fv_common.h"
#include "fv_internal.h"

static thread_local std::string g_last_error;
int fv_fail_hip(hipError_t e, const char* what) {
    char buf[256];
    snprintf(buf, sizeof buf, "%s: %s (hipError %d)", what, hipGetErrorString(e), (int)e);
    g_last_error = buf;
    return -(int)e;
}
int fv_decline(const char* why) {
    g_last_error = why;
    return FV_DECLINED;
}
int fv_invalid(const char* why) {
    g_last_error = why;
    return -(int)hipErrorInvalidValue;
}

namespace {

int fail_hip(hipError_t e, const char* what) { return fv_fail_hip(e, what); }
int decline(const char* why) { return fv_decline(why); }

// y = bf16(x * mul), RNE; mul == 1 is the plain cast (x * 1.0f is x)
__global__ void cast_f32_bf16_kernel(const float* __restrict__ x, uint16_t* __restrict__ y,
                                     size_t n, float mul) {
    const size_t i = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
    if (i + 4 <= n && ((((uintptr_t)x) & 15) == 0) && ((((uintptr_t)y) & 7) == 0)) {
        const fv::f32x4 v = *reinterpret_cast<const fv::f32x4*>(x + i);
        fv::s16x4 o;
#pragma unroll
        for (int j = 0; j < 4; j++) o[j] = (short)fv::bf16_rne_bits(v[j] * mul);
        *reinterpret_cast<fv::s16x4*>(y + i) = o;
    } else {
        for (size_t j = i; j < n && j < i + 4; j++) y[j] = fv::bf16_rne_bits(x[j] * mul);
    }
}

// The operands of one call that arrive as f32, in one launch (blockIdx.y: which). HBM-bound, eight elements a thread:
// 3 x 24 x 7800 x 64 (216 MB) 39 us in three launches, 30 in one; a call of 12 x 500 x 500 x 64 21 us with three, 15 with one.
__global__ __launch_bounds__(256) void cast_operands_kernel(const FvCastOperands ops) {
    const FvCastOperands::One c = ops.at[blockIdx.y];
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 8;
    if (i + 8 <= c.n && ((((uintptr_t)c.x) | ((uintptr_t)c.y)) & 15) == 0) {
        const fv::f32x4 a = *reinterpret_cast<const fv::f32x4*>(c.x + i), b = *reinterpret_cast<const fv::f32x4*>(c.x + i + 4);
        fv::s16x8 o;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            o[j] = (short)fv::bf16_rne_bits(a[j] * c.mul);
            o[4 + j] = (short)fv::bf16_rne_bits(b[j] * c.mul);
        }
        *reinterpret_cast<fv::s16x8*>(c.y + i) = o;
    } else {
        for (size_t j = i; j < c.n && j < i + 8; j++) c.y[j] = fv::bf16_rne_bits(c.x[j] * c.mul);
    }
}

__global__ void cast_bf16_f32_kernel(const uint16_t* __restrict__ x, float* __restrict__ y,
                                     size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = fv::bf16_bits_to_f32(x[i]);
}

// ---- static split-KV buffer ------------------------------------------------------------------
// The partials of fv_sdpa_dense_bf16_splitkv_static: part of the code object, so every GPU the
// library runs on holds its own copy at its own address from module load to process end. In host
// code the array's NAME is only a handle for hipGetSymbolAddress, never a device address: kernels
// and copies get the per-device pointer resolved below.
constexpr size_t kStaticScratchBytes = (size_t)32 << 20;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

constexpr int kMaxDevices = 64;
std::atomic<void*> g_scratch_ptr[kMaxDevices];

// This device's address of `scratch` (resolved once per device, with that device current).
hipError_t static_scratch(void** out) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
    void* p = g_scratch_ptr[dev].load(std::memory_order_acquire);
    if (!p) {
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        if (!p || (((uintptr_t)p) & 255) != 0) return hipErrorInvalidSymbol;
        g_scratch_ptr[dev].store(p, std::memory_order_release);   // racing first calls store the same address
    }
    *out = p;
    return hipSuccess;
}

enum { kMaskNone = 0, kMaskBlockCausal = 1, kMaskVdnWindow = 2 };

// The split count a launch settles on for `nkt` key tiles when `splits` are asked for: never more splits
// than key tiles (also keeps the sums below from wrapping on absurd counts), and no empty split.
size_t settle_splits(size_t nkt, size_t splits) {
    if (splits <= 1 || nkt <= 1) return 1;
    if (splits > nkt) splits = nkt;
    const size_t per = (nkt + splits - 1) / splits;
    return (nkt + per - 1) / per;
}

struct MaskArgs {
    int mode = kMaskNone;
    size_t q_rows = 0, k_rows = 0, v_rows = 0;   // rows per (batch, head) plane; 0 = contiguous (sq / sk)
    size_t splits = 1;                            // split-KV (dense only): key splits per query tile ...
    size_t full = 0;                              // ... past the first `full` ones
    size_t block_m = 0;                           // queries per workgroup (0: the kernel's own)
    int short_waves = 0;                          // > 0: the short kernel, with as many waves a workgroup
    void* workspace = nullptr;                    // ... and their partial results
    size_t workspace_bytes = 0;
    int* queue = nullptr;                         // masked: kFvQueueBytes for the queue of its items, or in the order of their numbers
    size_t block_tokens = 0, window = 0, sink = 0;                           // block-causal
    size_t video_start = 0, frame_tokens = 0, frames = 0, chunk = 0, radius = 0;   // VDN window
};

// flash_fwd_duo for masked launches, where it gives flash_fwd_pp2's bits, so that neither a clip's length nor the number of
// heads shows in a row: the offset is fixed (a bf16 result, and key 0 in every query's sight: fv_internal_launch_duo), and
// the first two tiles of every walk are keys 0 to 127 whatever the query tile's size. Its tiles of 128 queries cross fewer frame boundaries and leave a shorter
// last round, which counts where a query reaches few keys; long walks run at the chip's power limit, where 256 queries to a
// K and V stream cost less. Causal launches without a window, whose walks are half their reach on average, and windows that
// are part of their clip take it up to 8192 keys reached, walks of one length up to 4096; near those lines the two are within
// 7 %. us, flash_fwd_pp2 / flash_fwd_duo, heads x frame x frames (keys reached): causal 12 x 880 x 2 (1760) 46 / 40, 12 x 390 x 6 in
// blocks of 3 (2340) 66 / 51, 24 x 390 x 8 (3120) 78 / 71, 40 x 390 x 12 in blocks of 3 (4680) 257 / 241, 24 x 880 x 8 (7040) 291 / 284,
// 12 x 1560 x 4 (6240) 141 / 140, x 5 (7800) 190 / 200, 24 x 1560 x 6 (9360) 490 / 506; under a window with a sink 12 x 880 x 8 (2640)
// 130 / 113, 24 x 880 x 8 (3520) 245 / 224, 12 x 1560 x 6 (6240) 245 / 261, x 8 343 / 337, 12 x 1560 x 12 (18720) 882 / 893; VDN window
// 40 x 390 x 16 (2730) 415 / 381, 12 x 880 x 10 (4400) 276 / 266, 24 x 390 x 20 (6630) 484 / 448, 12 x 1560 x 24 (7800) 1999 / 2005, 40 x
// 1560 x 12 (7800) 2983 / 3116, 24 x 880 x 12 (9680) 881 / 834, 12 x 1560 x 24 (10920) 2389 / 2464, x 32 (26520) 5962 / 6335, over the whole
// clip 12 x 390 x 8 (3120) 67.8 / 67.2, 12 x 390 x 12 (4680) 109 / 113. At head dim 64 causal 24 x 880 x 4 71 / 68, 12 x 1560 x 21 (32760)
// 1743 / 1617, 40 x 1560 x 21 5543 / 5590, 40 x 1560 x 12 under a window of 3 with a sink 1312 / 1106, VDN window 12 x 1560 x 32 chunk 5
// 4129 / 3800.
bool duo_masked(const fv::FlashParams& p, size_t bh, size_t d) {
    const long ft = p.ft;
    const bool causal = p.mask_mode == kMaskBlockCausal;
    if (!fv_internal_fixed_offset(p.out_is_bf16) || (causal && p.win > 0 && p.sink * ft <= 64) || (!causal && p.vs + ft <= 64)) return false;
    long reach = p.sq, most = 8192;
    if (!causal) {
        const long seen = 2 + (2 * (long)p.radius + 1) * std::max(1, p.chunk);
        if (seen >= p.frames) most = 4096;
        else reach = ft * seen;
    } else if (p.win > 0) {
        reach = ft * ((long)p.win + p.sink), most = 4096;
    }
    return bh * (((size_t)p.sq + 127) / 128) > (size_t)fv_compute_units() / 2 && (d == 64 || reach <= most);
}

int flash_common(const uint16_t* q, const uint16_t* k, const uint16_t* v, void* out,
                 int out_is_bf16, size_t bh, size_t sq, size_t sk, size_t d, float scale,
                 const MaskArgs& m, void* stream) {
    if (!fv_sdpa_supported(1, bh, sq, sk, d)) return decline("sdpa: shape not taken by the fused kernel");
    if (!(scale > 0.0f) || !(scale < 3.0e38f)) return decline("sdpa: the fused kernel needs a finite scale > 0");
    if (!q || !k || !v || !out) return fv_invalid("sdpa: null operand");
    if ((((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out) & 15) != 0)
        return fv_invalid("sdpa: operands must be 16-byte aligned");
    fv::FlashParams p;
    p.q = q;
    p.k = k;
    p.v = v;
    p.out_f32 = out_is_bf16 ? nullptr : (float*)out;
    p.out_bf16 = out_is_bf16 ? (uint16_t*)out : nullptr;
    p.out_is_bf16 = out_is_bf16 ? 1 : 0;
    p.sq = (int)sq;
    p.sk = (int)sk;
    p.sl2 = scale * 1.4426950408889634f;
    const size_t q_rows = m.q_rows ? m.q_rows : sq, k_rows = m.k_rows ? m.k_rows : sk,
                 v_rows = m.v_rows ? m.v_rows : sk;
    if (q_rows < sq || k_rows < sk || v_rows < sk) return fv_invalid("sdpa: plane rows below the sequence length");
    const size_t plane_lim = (size_t)LONG_MAX / (d * (bh ? bh : 1));
    if (q_rows > plane_lim || k_rows > plane_lim || v_rows > plane_lim)
        return decline("sdpa: planes too large");
    p.q_plane = (long)(q_rows * d);
    p.k_plane = (long)(k_rows * d);
    p.v_plane = (long)(v_rows * d);
    const bool far = sk > 0xffffffffull / (2 * d);   // planes of 4 GB and more: flash_fwd_pp2 alone
    const size_t bm = m.block_m ? m.block_m : (size_t)fv_internal_flash_block_m();
    p.nqt = (int)((sq + bm - 1) / bm);
    const size_t total = bh * (size_t)p.nqt;
    if (total > (size_t)INT_MAX / 2) return decline("sdpa: too many query tiles for one launch");
    p.total = (int)total;
    p.per_xcd = (int)((total + 7) / 8);
    p.mask_mode = kMaskNone;
    p.ft = p.win = p.sink = 0;
    p.vs = p.ve = p.frames = p.chunk = p.radius = 0;
    int mode = m.mode;
    const size_t lim = (size_t)INT_MAX;
    if (mode == kMaskBlockCausal) {
        // rt/attn.rs:668-676
        if (m.block_tokens == 0 || m.window > lim || m.sink > lim || (sq > sk ? sq : sk) + m.block_tokens > lim)
            return decline("sdpa: block-causal parameters outside the kernel's int range");
        p.ft = (int)m.block_tokens;
        p.win = (int)m.window;
        p.sink = (int)m.sink;
        // One block spanning both sequences: every key is visible to every query (tq == tk == 0
        // for any window), so this is the dense problem and runs as the launch of the kernel-level dense entry, bit for bit
        // (the reference asserts that identity for its own kernels, gpucheck kernels_wan.rs:230-261).
        if (m.block_tokens >= sq && m.block_tokens >= sk) mode = kMaskNone;
    } else if (mode == kMaskVdnWindow) {
        // rt/attn.rs:544-553: self-attention only, the video rows inside the sequence
        const size_t ve = m.video_start + m.frames * m.frame_tokens;
        if (sq != sk || m.frames == 0 || m.frame_tokens == 0 || m.frames > lim / m.frame_tokens || ve > sk ||
            m.chunk > lim || m.radius > lim / 2 || (m.chunk > 0 && m.radius > lim / (2 * m.chunk)))
            return decline("sdpa: VDN window parameters the kernel cannot run");
        p.ft = (int)m.frame_tokens;
        p.vs = (int)m.video_start;
        p.ve = (int)ve;
        p.frames = (int)m.frames;
        p.chunk = (int)m.chunk;
        // a radius past the clip means every frame: clamp so that (f/c + r + 1) * c stays in int range
        p.radius = (int)(m.radius > m.frames ? m.frames : m.radius);
        if (m.frames <= 2) mode = kMaskNone;   // anchors only: dense
    }
    p.mask_mode = mode;
    p.full = 0;
    p.kv_split = 1;
    p.split_tiles = INT_MAX;
    p.part_row0 = p.part_rows = 0;
    p.part_o = nullptr;
    p.part_lse = nullptr;
    p.queue = nullptr;
    const size_t nkt = (sk + 63) / 64;
    size_t splits = mode == kMaskNone ? settle_splits(nkt, m.splits) : 1;
    if (splits > 1) {
        if (total * splits > (size_t)INT_MAX / 2) return decline("sdpa: too many workgroups for one launch");
        // the split query tiles are the last rows of [bh * sq]
        const size_t full = m.full < total ? m.full : 0;
        const size_t row0 = full / (size_t)p.nqt * sq + full % (size_t)p.nqt * bm, rows = bh * sq - row0;
        const size_t need = fv_sdpa_splitkv_workspace_bytes(1, rows, d, splits);
        if (!m.workspace || m.workspace_bytes < need || (((uintptr_t)m.workspace) & 255) != 0)
            return fv_invalid("sdpa: split-KV needs a 256-byte aligned workspace of fv_sdpa_splitkv_workspace_bytes");
        p.kv_split = (int)splits;
        p.split_tiles = (int)((nkt + splits - 1) / splits);
        p.part_o = (float*)m.workspace;
        p.part_lse = (float*)((char*)m.workspace + ((splits * rows * d * 4 + 255) & ~(size_t)255));
        p.full = (int)full;
        p.part_row0 = (long)row0;
        p.part_rows = (long)rows;
        p.total = (int)((total - full) * splits);
        p.per_xcd = (p.total + 7) / 8;
    }
    // Kernel-level calls take the short kernel up to 512 keys. Past them fv_rt_sdpa alone asks for it (short_waves): there
    // these calls are flash_fwd_pp2's or flash_fwd_duo's, whose bits a block-causal clip of one block then shares with the
    // first block of a longer one, for both result types (one frame has 880 tokens and more); it costs them what the short
    // kernel gains, 22.8 us instead of 16.7 at 12 x 1000 x 1000 x 128, 19.2 instead of 10.8 at 12 x 600 x 1000.
    int short_waves = m.short_waves;
    if (mode == kMaskNone && splits == 1 && !short_waves && sk <= 512) short_waves = fv_short_waves(bh, sq, sk, d);
    if (short_waves) {
        fv::ComposedParams c;
        c.q = q, c.k = k, c.v = v, c.out = out, c.q_is_bf16 = 1, c.out_is_bf16 = out_is_bf16;
        c.sq = p.sq, c.sk = p.sk, c.d = (int)d, c.scale = scale, c.vec = 1;
        c.q_plane = p.q_plane, c.k_plane = p.k_plane, c.v_plane = p.v_plane;
        const hipError_t e = fv_internal_launch_short(&c, short_waves, bh, (hipStream_t)stream);
        return e == hipSuccess ? FV_OK : fail_hip(e, "sdpa_short");
    }
    if (!far && (mode == kMaskNone ? splits == 1 && fv_duo(bh, sq, sk, d, out_is_bf16, false) : duo_masked(p, bh, d))) {
        p.nqt = (int)((sq + 127) / 128);
        p.total = (int)(bh * (size_t)p.nqt);
        p.per_xcd = (p.total + 7) / 8;
        const hipError_t e = fv_internal_launch_duo(&p, mode != kMaskNone ? 1 : 0, (int)d, (hipStream_t)stream);
        return e == hipSuccess ? FV_OK : fail_hip(e, "flash_fwd_duo");
    }
    if (mode != kMaskNone && m.queue) {
        p.queue = m.queue;
        const hipError_t e = fv_internal_clear_queue(p.queue, (hipStream_t)stream);
        if (e != hipSuccess) return fail_hip(e, "clear_queue");
    }
    hipError_t e = fv_internal_launch_flash(&p, mode != kMaskNone ? 1 : 0, (int)d, (int)bm, (hipStream_t)stream);
    if (e != hipSuccess) return fail_hip(e, mode != kMaskNone ? "flash_fwd_pp2<masked>" : "flash_fwd_pp2<dense>");
    if (p.kv_split > 1) {
        void* dst = (char*)out + (size_t)p.part_row0 * d * (out_is_bf16 ? 2 : 4);
        e = fv_internal_launch_splitkv_merge(p.part_o, p.part_lse, dst, out_is_bf16 ? 1 : 0, (size_t)p.part_rows, (int)d,
                                             p.kv_split, (hipStream_t)stream);
        if (e != hipSuccess) return fail_hip(e, "splitkv_merge");
    }
    return FV_OK;
}

}  // namespace

int fv_compute_units() {
    static const int cus = [] {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
            n = 256;
        return n;
    }();
    return cus;
}

// The short kernel (composed_fwd.hip) takes calls whose 32-query groups are one round of resident workgroups: of eight
// waves where each has a CU to itself, of four up to two a CU (three at head dim 64, which has room for four), while the walk of the keys is
// short enough that sharing it out over the chip (split-KV) or reading K and V once for 128 or 256 queries gains less. us in a
// graph, without it / short: at 128 channels 12 x 320 x 320 10.4 / 6.8, 3 x 390 x 200 8.7 / 6.0, 12 x 600 x 1000 19.2 / 10.8,
// x 3000 29.0 / 23.2, 12 x 320 x 4000 25.2 / 24.1, x 5000 32.1 / 30.2, 3 x 390 x 3000 20.2 / 19.2, x 5000 24.1 / 30.1; 264 to 512 groups
// 12 x 680 x 500 12.0 / 10.5, 12 x 1000 x 1000 22.8 / 16.7, x 2000 29.7 / 26.1, x 3000 31.9 / 36.0; 516 groups 12 x 1360 x 500 12.1 / 16.0,
// x 2000 34 / 41. At 64 channels 12 x 320 x 320 7.6 / 5.0, 3 x 390 x 3000 15.0 / 13.0, x 4000 16.7 / 15.9, x 5000 18.2 / 19.0, 12 x 1000 x 3000
// 26.5 / 23.8 (eight waves 22.3), 12 x 1560 x 1500 24.3 / 18.8, x 3000 32.1 / 32.6, 40 x 560 x 500 9.1 / 9.5, x 3000 35.3 / 34.7; 880 groups
// 40 x 700 x 700 11.6 / 14.6.
// (Query tiles of 256 that have a CU each already, of few rows: flash_fwd_pp2 as before.)
int fv_short_waves(size_t bh, size_t sq, size_t sk, size_t d) {
    const size_t cus = (size_t)fv_compute_units(), nq = (sq + 31) / 32, bm = (size_t)fv_internal_flash_block_m();
    if (nq > 3 * cus || bh * nq > (d == 64 ? 3 : 2) * cus || bh * ((sq + bm - 1) / bm) >= cus) return 0;
    if (bh * nq <= cus) return sk <= (d == 64 ? 4000 : 3072) ? 8 : 0;
    return sk <= (d == 64 ? 3072 : 2048) ? 4 : 0;
}

// flash_fwd_duo (two or, at head dim 64, three workgroups a CU) against flash_fwd_pp2, for walks so short that an item's
// ends count. Past them the chip runs at its power limit in either form, and 256 queries to a K and V stream cost less. us,
// flash_fwd_pp2 / flash_fwd_duo: at 128 channels 12 x 32760 x 64 61 / 38, x 200 77 / 64, x 512 109 / 100, x 800 160 / 144, x 1000
// 177 / 171, x 1500 243 / 242; one round 12 x 4000 x 512 17.3 / 17.3, x 700 22.2 / 20.9, x 1024 26.0 / 26.9, x 1500 35.8 / 36.7; 16 x 2560 x 700
// 21.6 / 20.2, 16 x 6144 x 1500 72.9 / 68.5, 24 x 10000 x 1000 115 / 111. At 64: 24 x 4001 x 50 14.2 / 7.6, 12 x 4000 x 4096 58.5 / 55.5,
// 16 x 4096 x 3000 50 / 48, 16 x 6144 x 4000 105 / 99, 16 x 12288 x 6000 270 / 268, x 8000 357 / 355, 16 x 7680 x 6000 178 / 177.
// A last round of a quarter of the CUs or less is shared out by key ranges (fv_split_plan), the sooner the fewer its tiles:
// at 64 channels 16 x 4608 (32 tiles past a round) x 2000 52 / 49, x 2500 61 / 60, x 6000 120 / 136, 16 x 8704 (32 past two) x 2500
// 100 / 96, x 6000 213 / 218, 16 x 5120 (64) x 3000 75 / 71, x 4000 93 / 94; at 128 16 x 4608 x 1300 63 / 58, x 1500 64 / 66,
// 16 x 8960 (48) x 1350 102 / 97, x 1500 106 / 105. (Of a sixteenth or less: at any length, this kernel would pay a round for them.)
// Where it cannot be split (no workspace, or an entry without one), flash_fwd_pp2 pays two whole rounds: 24 x 3000 x 6100 x 64
// 172 / 139, 24 x 3000 x 1500 x 128 72 / 66, 16 x 8960 x 1500 x 128 114 / 105.
// Few query tiles have a CU each, of 128 queries where fv_split_plan says so. f32 results follow the running max, whose
// rescales go by pairs of tiles in flash_fwd_pp2: they stay there, and a block's result does not depend on the clip's length.
bool fv_duo(size_t bh, size_t sq, size_t sk, size_t d, bool out_bf16, bool may_split) {
    const size_t cus = (size_t)fv_compute_units(), bm = (size_t)fv_internal_flash_block_m(), wgs = bh * ((sq + bm - 1) / bm);
    const size_t rest = wgs > cus ? wgs % cus : 0;   // tiles of the last round that flash_fwd_pp2 would split
    size_t most = d == 64 ? 6144 : 1536;
    if (may_split && rest > 0 && rest <= cus / 4) most = d == 128 ? 1408 : rest <= cus / 8 ? 2304 : 3072;
    if (rest > 0 && rest <= cus / 16) most = 0;
    return fv_internal_fixed_offset(out_bf16) && sk <= most && bh * ((sq + 127) / 128) > cus / 2;
}

// Fewer query tiles than CUs: fv_sdpa_splitkv_choose. More: they run in rounds of one per CU, and the last round costs a
// whole walk of the keys however few tiles are left for it. Where they are few, they are shared out over the chip by key
// ranges instead; where they are many it does not pay, because a chip that is half busy runs at a higher clock.
// Measured on MI355X, unsplit and so, us: 24 x 3000 x 3000 x 128 (288 tiles: 256 + 32 x 4) 130 / 102, 40 x 2000 x 2000
// x 64 (320: 256 + 64 x 4) 64 / 55, 40 x 5000 x 5000 x 128 (800: 768 + 32 x 5) 441 / 391, 40 x 75600 x 75600 x 128 (11840: 11776 + 64 x 4)
// 80900 / 80200.
FvSplitPlan fv_split_plan(size_t bh, size_t sq, size_t sk, size_t d, bool out_bf16) {
    const size_t cus = (size_t)fv_compute_units(), bm = (size_t)fv_internal_flash_block_m();
    const size_t nqt = (sq + bm - 1) / bm, wgs = bh * nqt, nkt = (sk + 63) / 64;
    if (wgs < cus || cus % 8 != 0 || wgs > (size_t)INT_MAX / 64) {
        const size_t splits = fv_sdpa_splitkv_choose(bh, sq, sk);
        // Query tiles of 128 where each still has a CU to itself. Measured on MI355X, 256 / 128 queries a workgroup, us:
        // bf16 results past the short kernel's walks and past flash_fwd_duo's 200 x 100 x 2000 x 128 45.9 / 37.1, 200 x 100 x
        // 8000 x 64 123 / 90, 4 x 390 x 8000 x 128 split 32.5 / 27.7; f32 results 12 x 1000 x 1000 x 128 split 26.8 / 23.5, 40 x 700 x
        // 700 x 64 17.5 / 13.4, 12 x 320 x 600 x 128 19.4 / 15.6; past one per CU, 24 x 390 x 4000 x 128 36.7 / 45.5, 24 x 390 x 2000 x
        // 128 f32 26.8 / 33.8, 12 x 4000 x 512 x 128 19.8 / 27.2, 40 x 1000 x 1000 x 64 (320 tiles) 22.1 / 23.1.
        if (splits == 1 && fv_duo(bh, sq, sk, d, out_bf16, false)) return {bm, 0, 1, 0};
        const size_t half = bm / 2, small = bh * ((sq + half - 1) / half) * settle_splits(nkt, splits);
        return {small <= cus ? half : bm, 0, splits, fv_sdpa_splitkv_workspace_bytes(bh, sq, d, splits)};
    }
    const size_t full = wgs / cus * cus, rest = wgs - full;
    if (rest == 0 || fv_duo(bh, sq, sk, d, out_bf16, true)) return {bm, 0, 1, 0};
    const size_t rows = bh * sq - (full / nqt * sq + full % nqt * bm);
    // us: a workgroup's fixed part, and a 64-key tile while `w` workgroups run; partials written and read at 4 TB/s and a launch.
    // Fitted to the kernel on 32x32x16 MFMAs (16 x 4000 x 4000 x 128, 256 tiles: 121 us, half of them 79). Now it
    // takes 104 and 79, at 64 channels 70 and 59: the last tiles of a full chip cost less than this says, so it splits later than it could.
    // 16 x 6144 x 4000 x 128 (128 tiles past a round) 174 as planned, unsplit, 160 in two; elsewhere the plan is within 6 % of the best
    // count: 24 x 3000 x 6000 x 64 125 / 119, 40 x 2000 x 8000 x 64 167 / 159, 24 x 3000 x 3000 x 128 102 / 101, 12 x 8000 x 8000 290 / 290.
    const double fixed = d == 64 ? 5.0 : 8.0;
    auto run = [&](size_t w, size_t tiles) {
        const double x = w <= cus / 2 ? 0.0 : ((double)w / (double)cus - 0.5) * 2.0;
        return fixed + (d == 64 ? 0.8 + 0.25 * x : 1.15 + 0.65 * x) * (double)tiles;
    };
    size_t best = 1;
    double best_cost = 0.95 * run(rest, nkt);
    for (size_t sp = 2; sp <= 16 && sp * 8 <= nkt; sp++) {   // at least 8 key tiles (4 phases) per split
        const size_t per = (nkt + sp - 1) / sp, real = settle_splits(nkt, sp), n = rest * real;
        const double c = (double)(n / cus) * run(cus, per) + (n % cus ? run(n % cus, per) : 0.0) +
                         (double)(real * rows * d) * 4.0 / 4.0e6 + 6.0;
        if (c < best_cost) best_cost = c, best = real;
    }
    if (best == 1) return {bm, 0, 1, 0};
    return {bm, full, best, fv_sdpa_splitkv_workspace_bytes(1, rows, d, best)};
}

int fv_dense_planned(const uint16_t* q, const uint16_t* k, const uint16_t* v, void* out, int out_is_bf16, size_t bh,
                     size_t sq, size_t sk, size_t d, float scale, size_t q_rows, size_t k_rows, size_t v_rows,
                     const FvSplitPlan& plan, void* workspace, size_t workspace_bytes, void* stream) {
    MaskArgs m;
    m.q_rows = q_rows;
    m.k_rows = k_rows;
    m.v_rows = v_rows;
    m.splits = plan.splits;
    m.full = plan.full;
    m.block_m = plan.block_m;
    m.short_waves = plan.short_waves;
    m.workspace = workspace;
    m.workspace_bytes = workspace_bytes;
    return flash_common(q, k, v, out, out_is_bf16, bh, sq, sk, d, scale, m, stream);
}

// The queue (take_item in flash_fwd.hip) saves L2 misses where walks are long, and goes through its lists head by head: the last
// head's longest walk may begin near the end. So it takes launches of eight rounds and more at 128 channels whose walks are
// 4096 keys long on average and whose work is four times a CU's longest walk. us, in the order of the numbers / from the queue, with
// that ratio: causal 40 x 21 x 1560 (10) 8624 / 7979, 12 x 32 x 1560 (4.6) 5795 / 5535, 40 x 21 x 1560 under a window of four with a sink 3863
// / 3747; VDN window 40 x 18 x 880 chunk 5 radius 2 (9.7) 3781 / 3524, 40 x 21 x 1560 radius 2 (7.9) 6917 / 6787, 12 x 32 x 1560 chunk 5
// (5.1) 6033 / 5911, 24 x 24 x 1560 radius 2 (4.8) 4787 / 4782 and f32 results 5310 / 5084. Past the lines: 24 x 40 x 1560 radius 1 (3.9) 6735 /
// 6887, 12 x 60 x 1560 radius 2 (2.5) 6564 / 8292, 40 x 40 x 390 radius 0 (1.2) 766 / 961; causal under a window of one 12 x 32 x 1560
// (1535 keys) 601 / 616, 40 x 34 x 390 267 / 292; f32 results at 64 channels causal 24 x 21 x 1560 3567 / 3634, VDN 12 x 32 x 1560 chunk 5
// 4382 / 4424. (Numbers as they come: the bounds of a mask are judged by the launch.)
size_t fv_masked_workspace_bytes(size_t bh, size_t sq, size_t sk, size_t d, const FvMask& m) {
    const size_t cus = (size_t)fv_compute_units(), bm = (size_t)fv_internal_flash_block_m();
    const double tiles = (double)bh * (double)((sq + bm - 1) / bm), nq = (double)sq, nk = (double)sk;
    if (d != 128 || cus < 8 || tiles < 8.0 * (double)cus) return 0;
    double mean, longest;   // keys of a walk
    if (m.causal) {
        const double seen = ((double)m.window + (double)m.sink) * (double)m.block_tokens;
        longest = std::min(m.window > 0 ? std::min(seen, nk) : nk, nq);
        mean = longest * (1.0 - longest / (2.0 * nq));   // (the first queries see less)
    } else {
        const double frames = (double)m.frames, ft = (double)m.frame_tokens;
        const double seen = std::min(frames, 2.0 + (2.0 * (double)m.radius + 1.0) * std::max(1.0, (double)m.chunk));
        const double inner = std::min(std::max(0.0, frames - 2.0) * ft, nq);
        longest = nk;
        mean = ((nq - inner) * nk + inner * std::max(0.0, nk - (frames - seen) * ft)) / nq;
    }
    return mean >= 4096.0 && tiles * mean >= 4.0 * (double)cus * longest ? kFvQueueBytes : 0;
}

int fv_masked_planned(const uint16_t* q, const uint16_t* k, const uint16_t* v, void* out, int out_is_bf16, size_t bh,
                      size_t sq, size_t sk, size_t d, float scale, const FvMask& mask, void* workspace, void* stream) {
    MaskArgs m;
    m.mode = mask.causal ? kMaskBlockCausal : kMaskVdnWindow;
    m.block_tokens = mask.block_tokens;
    m.window = mask.window;
    m.sink = mask.sink;
    m.video_start = mask.video_start;
    m.frame_tokens = mask.frame_tokens;
    m.frames = mask.frames;
    m.chunk = mask.chunk;
    m.radius = mask.radius;
    if (fv_masked_workspace_bytes(bh, sq, sk, d, mask)) m.queue = (int*)workspace;
    return flash_common(q, k, v, out, out_is_bf16, bh, sq, sk, d, scale, m, stream);
}

int fv_cast_operands(const FvCastOperands& ops, int count, void* stream) {
    size_t most = 0;
    for (int i = 0; i < count; i++) most = ops.at[i].n > most ? ops.at[i].n : most;
    if (most == 0) return FV_OK;
    const size_t blocks = (most + 2047) / 2048;
    if (blocks >= (size_t)1 << 24) return decline("cast: too many elements for one launch");   // 2^32 work-items
    hipLaunchKernelGGL(cast_operands_kernel, dim3((unsigned)blocks, (unsigned)count), dim3(256), 0, (hipStream_t)stream, ops);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? FV_OK : fail_hip(e, "cast_operands");
}

extern "C" {

const char* fv_sdpa_last_error(void) { return g_last_error.c_str(); }
const char* fv_sdpa_arch(void) { return "gfx950"; }

int fv_sdpa_init(void) {
    hipError_t e = fv_internal_init_flash();
    if (e == hipSuccess) e = fv_internal_init_vsa();
    if (e == hipSuccess) e = fv_internal_init_composed();
    void* p = nullptr;
    if (e == hipSuccess) e = static_scratch(&p);
    return e == hipSuccess ? FV_OK : fail_hip(e, "fv_sdpa_init");
}

// the launchers' own test (flash_fwd.hip: FlashParams::sl2, computed as below, equal to one)
int fv_sdpa_is_log2_domain_scale(float scale) { return scale * 1.4426950408889634f == 1.0f ? 1 : 0; }

uint64_t fv_sdpa_exact_pass_reruns(void) {
    unsigned long long n = 0;
    return fv_internal_exact_pass_reruns(&n) == hipSuccess ? (uint64_t)n : 0;
}

int fv_sdpa_supported(size_t b, size_t h, size_t sq, size_t sk, size_t d) {
    if (b != 0 && h > (size_t)65535 / b) return 0;
    const size_t bh = b * h;
    return (d == 128 || d == 64) && sq > 0 && sk > 0 && bh >= 1 && bh <= 65535 && sq <= (size_t)INT_MAX &&
           sk <= (size_t)INT_MAX;
}

int fv_sdpa_dense_bf16(const uint16_t* q, const uint16_t* k, const uint16_t* v, void* out,
                       int out_is_bf16, size_t bh, size_t sq, size_t sk, size_t d, float scale,
                       void* stream) {
    return flash_common(q, k, v, out, out_is_bf16, bh, sq, sk, d, scale, MaskArgs{}, stream);
}

int fv_sdpa_dense_bf16_strided(const uint16_t* q, const uint16_t* k, const uint16_t* v, void* out,
                               int out_is_bf16, size_t bh, size_t sq, size_t sk, size_t d, float scale,
                               size_t q_rows, size_t k_rows, size_t v_rows, void* stream) {
    MaskArgs m;
    m.q_rows = q_rows;
    m.k_rows = k_rows;
    m.v_rows = v_rows;
    return flash_common(q, k, v, out, out_is_bf16, bh, sq, sk, d, scale, m, stream);
}

size_t fv_sdpa_splitkv_workspace_bytes(size_t bh, size_t sq, size_t d, size_t splits) {
    if (splits <= 1) return 0;
    return ((splits * bh * sq * d * 4 + 255) & ~(size_t)255) + ((splits * bh * sq * 4 + 255) & ~(size_t)255);
}

size_t fv_sdpa_splitkv_choose(size_t bh, size_t sq, size_t sk) {
    const int cus = fv_compute_units();
    const size_t bm = (size_t)fv_internal_flash_block_m();
    const size_t wgs = bh * ((sq + bm - 1) / bm), nkt = (sk + 63) / 64;
    if (wgs == 0 || wgs >= (size_t)cus) return 1;               // the query tiles alone fill the CUs
    // Cost model (microseconds): a workgroup costs about 10 fixed + 1.7 per 64-key tile (an early form of the kernel; now 7
    // and 1.1 on a chip that is half full, 1.5 on a full one, so it splits a little early: f32 results 12 x 1000 x 1000 x 128 23.2
    // as it chooses, 21.6 unsplit; 24 x 390 x 4000 36 / 60, 12 x 1560 x 32760 270 / 470), workgroups run in rounds of one per CU, and the merge reads `s` f32 partials at about 4 TB/s. Take the cheapest split count, if it wins by more than 10 %.
    auto cost = [&](size_t sp) {
        const size_t per = (nkt + sp - 1) / sp, real = (nkt + per - 1) / per;
        const double rounds = (double)((wgs * real + cus - 1) / cus);
        const double merge = real > 1 ? (double)(real * bh * sq) * 128.0 * 4.0 / 4.0e6 + 5.0 : 0.0;
        return rounds * (10.0 + 1.7 * (double)per) + merge;
    };
    size_t best = 1;
    double best_cost = cost(1);
    for (size_t sp = 2; sp <= 16 && sp * 8 <= nkt; sp++) {        // at least 8 key tiles (4 phases) per split
        const double c = cost(sp);
        if (c < best_cost) best_cost = c, best = sp;
    }
    return best_cost < 0.9 * cost(1) ? best : 1;
}

int fv_sdpa_dense_bf16_splitkv(const uint16_t* q, const uint16_t* k, const uint16_t* v, void* out,
                               int out_is_bf16, size_t bh, size_t sq, size_t sk, size_t d, float scale,
                               size_t q_rows, size_t k_rows, size_t v_rows, size_t splits, void* workspace,
                               size_t workspace_bytes, void* stream) {
    MaskArgs m;
    m.q_rows = q_rows;
    m.k_rows = k_rows;
    m.v_rows = v_rows;
    m.splits = splits;
    if (splits == 0) {   // the choice of fv_rt_sdpa
        m.short_waves = out_is_bf16 ? fv_short_waves(bh, sq, sk, d) : 0;
        m.splits = m.short_waves ? 1 : fv_sdpa_splitkv_choose(bh, sq, sk);
        if (!workspace || workspace_bytes < fv_sdpa_splitkv_workspace_bytes(bh, sq, d, m.splits)) m.splits = 1;
    }
    m.workspace = workspace;
    m.workspace_bytes = workspace_bytes;
    return flash_common(q, k, v, out, out_is_bf16, bh, sq, sk, d, scale, m, stream);
}

size_t fv_sdpa_splitkv_static_bytes(void) { return kStaticScratchBytes; }

size_t fv_sdpa_splitkv_static_splits(size_t bh, size_t sq, size_t sk, size_t d, size_t splits) {
    const size_t nkt = (sk + 63) / 64;
    if (splits != 0) {   // the caller's count, settled as the launch would; refused when its partials do not fit
        splits = settle_splits(nkt, splits);
        return fv_sdpa_splitkv_workspace_bytes(bh, sq, d, splits) <= kStaticScratchBytes ? splits : 0;
    }
    // the library's own choice never refuses: it steps down to the largest count whose partials fit (1 = unsplit)
    for (size_t s = fv_sdpa_splitkv_choose(bh, sq, sk); s > 1; s--) {
        const size_t real = settle_splits(nkt, s);
        if (fv_sdpa_splitkv_workspace_bytes(bh, sq, d, real) <= kStaticScratchBytes) return real;
    }
    return 1;
}

int fv_sdpa_dense_bf16_splitkv_static(const uint16_t* q, const uint16_t* k, const uint16_t* v, void* out,
                                      int out_is_bf16, size_t bh, size_t sq, size_t sk, size_t d, float scale,
                                      size_t q_rows, size_t k_rows, size_t v_rows, size_t splits, void* stream) {
    if (!fv_sdpa_supported(1, bh, sq, sk, d)) return decline("sdpa: shape not taken by the fused kernel");
    const size_t run = fv_sdpa_splitkv_static_splits(bh, sq, sk, d, splits);
    if (run == 0) {
        char buf[200];
        snprintf(buf, sizeof buf,
                 "sdpa: split-KV partials of this call need %zu bytes, the static buffer holds %zu "
                 "(use fv_sdpa_dense_bf16_splitkv with a workspace)",
                 fv_sdpa_splitkv_workspace_bytes(bh, sq, d, settle_splits((sk + 63) / 64, splits)), kStaticScratchBytes);
        return fv_invalid(buf);
    }
    MaskArgs m;
    m.q_rows = q_rows;
    m.k_rows = k_rows;
    m.v_rows = v_rows;
    m.splits = run;
    if (run > 1) {
        void* p = nullptr;
        const hipError_t e = static_scratch(&p);
        if (e != hipSuccess) return fail_hip(e, "sdpa: resolving the static split-KV buffer");
        m.workspace = p;
        m.workspace_bytes = kStaticScratchBytes;
    }
    return flash_common(q, k, v, out, out_is_bf16, bh, sq, sk, d, scale, m, stream);
}

int fv_sdpa_block_causal_bf16(const uint16_t* q, const uint16_t* k, const uint16_t* v, void* out,
                              int out_is_bf16, size_t bh, size_t sq, size_t sk, size_t d,
                              float scale, size_t block_tokens, size_t window, size_t sink,
                              void* stream) {
    const FvMask mask = {true, block_tokens, window, sink, 0, 0, 0, 0, 0};
    return fv_masked_planned(q, k, v, out, out_is_bf16, bh, sq, sk, d, scale, mask, nullptr, stream);
}

int fv_sdpa_vdn_window_bf16(const uint16_t* q, const uint16_t* k, const uint16_t* v, void* out,
                            int out_is_bf16, size_t bh, size_t sq, size_t sk, size_t d, float scale,
                            size_t video_start, size_t frame_tokens, size_t frames, size_t chunk,
                            size_t radius, void* stream) {
    const FvMask mask = {false, 0, 0, 0, video_start, frame_tokens, frames, chunk, radius};
    return fv_masked_planned(q, k, v, out, out_is_bf16, bh, sq, sk, d, scale, mask, nullptr, stream);
}

// (a launch holds fewer than 2^32 work-items and the runtime does not say so: longer operands in several)
int fv_cast_f32_bf16_scaled(const float* x, uint16_t* y, size_t n, float mul, void* stream) {
    constexpr size_t kMost = (size_t)1 << 33;   // elements: four a thread
    for (size_t at = 0; at < n; at += kMost) {
        const size_t len = n - at < kMost ? n - at : kMost, blocks = (len + 1023) / 1024;
        hipLaunchKernelGGL(cast_f32_bf16_kernel, dim3((unsigned)blocks), dim3(256), 0,
                           (hipStream_t)stream, x + at, y + at, len, mul);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return fail_hip(e, "cast_f32_bf16");
    }
    return FV_OK;
}

int fv_cast_f32_bf16(const float* x, uint16_t* y, size_t n, void* stream) {
    return fv_cast_f32_bf16_scaled(x, y, n, 1.0f, stream);
}

int fv_cast_bf16_f32(const uint16_t* x, float* y, size_t n, void* stream) {
    constexpr size_t kMost = (size_t)1 << 31;   // elements: one a thread
    for (size_t at = 0; at < n; at += kMost) {
        const size_t len = n - at < kMost ? n - at : kMost, blocks = (len + 255) / 256;
        hipLaunchKernelGGL(cast_bf16_f32_kernel, dim3((unsigned)blocks), dim3(256), 0,
                           (hipStream_t)stream, x + at, y + at, len);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return fail_hip(e, "cast_bf16_f32");
    }
    return FV_OK;
}

}  // extern "C"
