// Launch parameter blocks and internal launcher prototypes shared by the kernel
// translation units and the C ABI (fv_api.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

namespace fv {

struct FlashParams {
    const uint16_t* q;
    const uint16_t* k;
    const uint16_t* v;
    float* out_f32;
    uint16_t* out_bf16;
    int out_is_bf16;
    int sq, sk;
    float sl2;          // scale * log2(e)
    int nqt;            // query tiles per (batch, head)
    int total;          // workgroups past the first `full`: (bh * nqt - full) * kv_split
    int per_xcd;        // ceil(total / 8)
    int mask_mode;      // 0 none, 1 block-causal, 2 VDN window
    int ft, win, sink;  // block-causal: block tokens, window blocks, sink blocks; VDN window: ft = frame tokens
    int vs, ve, frames, chunk, radius;   // VDN window: video rows [vs, ve), frame count, chunk, radius
    // elements between consecutive (batch, head) planes of q, k and v: s * d when contiguous, larger
    // when the operand is a row window of a longer plane (a KV cache read in place)
    long q_plane, k_plane, v_plane;
    // Split-KV (dense launches only): the first `full` (a multiple of 8) query tiles of the launch, counted head by
    // head, have a workgroup each. kv_split > 1 gives every later one kv_split workgroups, each walking split_tiles
    // key tiles and writing its own normalised partial output (f32 [split][row][d]) and base-2 log-sum-exp
    // ([split][row]) for the merge kernel, for the part_rows rows of [bh * sq] from part_row0 on.
    int full, kv_split, split_tiles;
    long part_row0, part_rows;
    float* part_o;
    float* part_lse;
    // Masked launches: eight zeroed counters (kFvQueueBytes) from which the workgroups take their items, or null: in the order of
    // their numbers.
    int* queue;
};

struct ComposedParams {
    const void* q = nullptr;      // [bh, sq, d]
    const void* k = nullptr;      // [bh, sk, d]
    const void* v = nullptr;
    const float* mask = nullptr;  // additive, [sq, sk] per mask_bh elements, or null
    long mask_bh = 0;             // elements between the masks of consecutive (batch, head) planes (0: shared)
    void* out = nullptr;          // [bh, sq, d] f32 or bf16 (RNE)
    int q_is_bf16 = 0, out_is_bf16 = 0;
    int sq = 0, sk = 0, d = 0;
    float scale = 1.0f;
    int vec = 0;                  // set by the launcher: 16-byte operand rows
    int nqt = 0, total = 0, per_xcd = 0, by_head = 0;   // set by the launcher: query tiles per head, items past `full`, ceil(total / 8), item order
    // Split tail (fv_composed_plan): the first `full` query tiles have a workgroup each, every later one `splits`, each
    // walking split_tiles key tiles and leaving its sums (f32 [split][row][dpad], unnormalised) and its (max, sum)
    // ([split][row][2]) for the merge kernel, for the part_rows rows of [bh * sq] from part_row0 on. splits <= 1: no tail.
    int full = 0, splits = 1, split_tiles = 0, dpad = 0;
    long part_row0 = 0, part_rows = 0;
    float* part_o = nullptr;
    float* part_ml = nullptr;
    long q_plane = 0, k_plane = 0, v_plane = 0;   // short launches: elements between consecutive (batch, head) planes
};

// How a composed launch is cut (composed_fwd.hip): splits <= 1: one workgroup a query tile throughout.
struct ComposedPlan {
    size_t full, splits, workspace_bytes;
};

struct VsaFineParams {
    const uint16_t* qt;           // tile-ordered bf16 [bh, nb*64, 128]
    const uint16_t* kt;
    const uint16_t* vt;
    const unsigned* selected;     // [bh, nb, topk]
    const int* block_sizes;       // [nb]
    float* out;                   // [bh, q_tiles*64, 128] f32, tile-slot order
    int num_tiles, topk;
    float sl2;
    int q_base, q_tiles;          // query tiles [q_base, q_base + q_tiles)
    int total, per_xcd;           // bh * q_tiles, ceil(total / 8)
    int* pace;                    // zeroed counters (fv_internal_fine_pace) or null
    int gang, pace_stride;        // workgroups that share a set of counters; words a set
    // Fused combine (whole-op entry): when `final_out` is set the kernel writes
    // final_out[token] = coarse[tile] * gate[token] + sparse instead of `out`, in token order.
    float* final_out;             // [bh, seq, 128] f32 or null
    const float* coarse;          // [bh, num_tiles, 128]
    const void* gate;             // [bh, seq, 128] f32 / bf16 or null (gate of one)
    int gate_is_bf16;
    const int* slot_src;          // [num_tiles * 64]
    long seq;
};

// The key-tile walk of one query tile of a masked launch: up to three ascending, non-overlapping
// ranges of 64-key tiles, [0, n0), [a1, a1 + n1) and [a2, a2 + n2), ne = n0 + n1 + n2 tiles in all
// (ne == 0: no query of the tile sees any key). Every key visible to any query of the tile lies in
// a walked tile; which scores inside a walked tile count is decided per lane.
//   block-causal (rt/attn.rs:449-453): the sink tiles, then the band of the tile's blocks;
//   VDN window (rt/attn.rs:483-510): rows before the video + frame 0, the window frames of the
//   tile, the last frame + rows after the video; a tile holding an anchor / global row walks all.
struct TileWalk {
    int a1, a2, n0, n1, ne;
};
// (Params: FlashParams, or the same struct read through another address space)
template <class Params>
__host__ __device__ inline TileWalk mask_tile_walk(const Params& p, int q0, int qlen, int nkt) {
    constexpr int kKeys = 64;
    const int sk = p.sk;
    auto imin = [](int a, int b) { return a < b ? a : b; };
    auto imax = [](int a, int b) { return a > b ? a : b; };
    int a1 = 0, a2 = 0, b0, b1, b2 = 0;
    if (p.mask_mode == 1) {
        const int ft = p.ft, win = p.win;
        const int fq_lo = q0 / ft, fq_hi = (q0 + qlen - 1) / ft;
        const long hi_l = (long)(fq_hi + 1) * ft;
        const int hi_tok = (int)(hi_l < (long)sk ? hi_l : (long)sk);
        const int lo_tok = imin(hi_tok, win > 0 ? imax(0, fq_lo - win + 1) * ft : 0);
        const long sink_l = (long)p.sink * ft;
        const int sink_tok = (int)(sink_l < (long)sk ? sink_l : (long)sk);
        b0 = (sink_tok + kKeys - 1) / kKeys;
        a1 = lo_tok / kKeys;
        b1 = (hi_tok + kKeys - 1) / kKeys;
    } else {
        const int vs = p.vs, ve = p.ve, t = p.ft, last = p.frames - 1, c = p.chunk, r = p.radius;
        auto lo_frame = [&](int f) { return imax(0, c > 0 ? (f / c - r) * c : f - r); };
        auto hi_frame = [&](int f) { return imin(last, c > 0 ? (f / c + r + 1) * c - 1 : f + r); };
        const bool inner_tile = q0 >= vs + t && q0 + qlen <= ve - t;   // frames 1 .. last-1 only
        if (inner_tile) {
            const int fmin = (q0 - vs) / t, fmax = (q0 + qlen - 1 - vs) / t;
            b0 = (vs + t + kKeys - 1) / kKeys;
            a1 = (vs + lo_frame(fmin) * t) / kKeys;
            b1 = (vs + (hi_frame(fmax) + 1) * t + kKeys - 1) / kKeys;
            a2 = (ve - t) / kKeys;
            b2 = nkt;
        } else {
            b0 = nkt;
            b1 = 0;
        }
    }
    // ranges may touch or overlap: each starts no earlier than the previous one ends
    b0 = imin(b0, nkt);
    a1 = imax(a1, b0);
    b1 = imin(imax(b1, a1), nkt);
    a2 = imax(a2, b1);
    b2 = imax(b2, a2);
    TileWalk w;
    w.a1 = a1;
    w.a2 = a2;
    w.n0 = b0;
    w.n1 = b1 - a1;
    w.ne = w.n0 + w.n1 + (imin(b2, nkt) - imin(a2, nkt));
    return w;
}

// The keys query qi of a masked launch sees: x < a_hi || x >= c_lo || (w_lo <= x && x < w_hi).
struct LaneMask {
    int a_hi, c_lo, w_lo, w_hi;
};
template <class Params>
__host__ __device__ inline LaneMask lane_mask(const Params& p, int qi) {
    auto imin = [](int a, int b) { return a < b ? a : b; };
    auto imax = [](int a, int b) { return a > b ? a : b; };
    LaneMask m = {0, 0x7fffffff, 0, 0};
    if (p.mask_mode == 1) {
        // block-causal (rt/attn.rs:449-453): keys of blocks (tq - win, tq], plus the sink blocks
        const int ft = p.ft, win = p.win;
        const int tq = qi / ft;
        const long sink_l = (long)p.sink * ft, hi_l = (long)(tq + 1) * ft;
        m.a_hi = (int)(sink_l < (long)p.sk ? sink_l : (long)p.sk);
        m.w_hi = (int)(hi_l < 0x7fffffffL ? hi_l : 0x7fffffffL);
        m.w_lo = win > 0 ? imax(0, tq - win + 1) * ft : 0;
    } else {
        // VDN window (rt/attn.rs:483-510): rows outside [vs, ve) and the frames 0 and
        // frames-1 are dense both ways; any other frame sees the frames of its window
        const int vs = p.vs, ve = p.ve, t = p.ft, last = p.frames - 1, c = p.chunk, r = p.radius;
        auto lo_frame = [&](int f) { return imax(0, c > 0 ? (f / c - r) * c : f - r); };
        auto hi_frame = [&](int f) { return imin(last, c > 0 ? (f / c + r + 1) * c - 1 : f + r); };
        if (qi >= vs + t && qi < ve - t) {
            const int qf = (qi - vs) / t;
            m.a_hi = vs + t;
            m.c_lo = ve - t;
            m.w_lo = vs + lo_frame(qf) * t;
            m.w_hi = vs + (hi_frame(qf) + 1) * t;
        } else {
            m.a_hi = 0x7fffffff;
        }
    }
    return m;
}

// The walk positions at which each of a wave's 32 queries sees every key, from scalars, once per walk: e < a, w0 <= e < w1 or
// e >= c. At the others the lanes ask key by key; those are the few that a range's ends or a frame boundary among the
// queries cut (and the last, where the keys may end). Every visible range counts in every range of the walk: a query tile
// with a row of an anchor frame walks everything in one. (With ranges matched to ranges its tiles past the first frame were
// taken for cut: VDN windows that cover the clip, 12 heads 12 x 390 174 us instead of 110, 12 x 880 645 instead of 510; 12 heads 32 x
// 1560 chunk 5 5872 instead of 5626.)
struct WalkSight {
    int a, w0, w1, c;
    __host__ __device__ inline bool all(int from, int to) const { return (to < a) | ((from >= w0) & (to < w1)) | (from >= c); }
};
template <class Params>
__host__ __device__ inline WalkSight walk_sight(const Params& p, const TileWalk& w, int first) {
    constexpr int kNone = 0x7fffffff;
    auto imin = [](int a, int b) { return a < b ? a : b; };
    auto imax = [](int a, int b) { return a > b ? a : b; };
    int last = first + 31;
    if (p.mask_mode == 2) {   // the rows of inner frames among them: the others see every key
        first = imax(first, p.vs + p.ft);
        last = imin(last, p.ve - p.ft - 1);
        if (first > last) return {kNone, 0, 0, kNone};
    }
    const LaneMask m0 = lane_mask(p, first), m1 = lane_mask(p, last);   // (both bounds of a window rise with the query)
    const int w_lo = imax(m0.w_lo, m1.w_lo), w_hi = imin(m0.w_hi, m1.w_hi);
    int a = m0.a_hi, c = m0.c_lo;
    if (w_lo < w_hi) {   // a window that touches its neighbours is one range with them
        if (w_lo <= a) a = imax(a, w_hi);
        if (w_hi >= c) c = imin(c, w_lo);
        if (a >= c) a = kNone;
    }
    // positions of the walk whose tile lies before tile t
    auto before = [&](int t) {
        return imin(t, w.n0) + imin(imax(t - w.a1, 0), w.n1) + imin(imax(t - w.a2, 0), w.ne - w.n0 - w.n1);
    };
    auto up = [](int x) { return (x >> 6) + ((x & 63) != 0); };
    return {before(a >> 6), before(up(w_lo)), before(w_hi >> 6), c == kNone ? kNone : before(up(c))};
}

}  // namespace fv

// y = bf16(x * mul), RNE, for up to three operands in one launch
struct FvCastOperands {
    struct One {
        const float* x;
        uint16_t* y;
        size_t n;
        float mul;
    } at[3];
};
int fv_cast_operands(const FvCastOperands& ops, int count, void* stream);

// How a dense launch of this shape is split where the caller has a workspace for it: all of its query tiles into
// `splits` key ranges (full == 0), the ones past the first `full`, or none (splits == 1).
struct FvSplitPlan {
    size_t block_m, full, splits, workspace_bytes;   // block_m: queries per workgroup
    int short_waves = 0;                             // > 0: the short kernel, with as many waves a workgroup
};
FvSplitPlan fv_split_plan(size_t bh, size_t sq, size_t sk, size_t d, bool out_bf16);
// Waves a workgroup of the short kernel where a dense call of this shape that writes bf16 takes it, else 0.
int fv_short_waves(size_t bh, size_t sq, size_t sk, size_t d);
// whether an unsplit dense launch takes the kernel with two workgroups a CU; may_split: where its last round could be split
bool fv_duo(size_t bh, size_t sq, size_t sk, size_t d, bool out_bf16, bool may_split);
// fv_sdpa_dense_bf16_splitkv with such a plan
int fv_dense_planned(const uint16_t* q, const uint16_t* k, const uint16_t* v, void* out, int out_is_bf16, size_t bh,
                     size_t sq, size_t sk, size_t d, float scale, size_t q_rows, size_t k_rows, size_t v_rows,
                     const FvSplitPlan& plan, void* workspace, size_t workspace_bytes, void* stream);

extern "C" int fv_internal_fixed_offset(int out_is_bf16);   // whether results of that type are made with a fixed offset first
// Masked launches of many rounds take their items from a queue where the caller has this much memory for it.
constexpr size_t kFvQueueBytes = 1024;
struct FvMask {
    bool causal;
    size_t block_tokens, window, sink;                            // block-causal
    size_t video_start, frame_tokens, frames, chunk, radius;      // VDN window
};
size_t fv_masked_workspace_bytes(size_t bh, size_t sq, size_t sk, size_t d, const FvMask& mask);
// fv_sdpa_block_causal_bf16 or fv_sdpa_vdn_window_bf16 with such a workspace, or without one (null)
int fv_masked_planned(const uint16_t* q, const uint16_t* k, const uint16_t* v, void* out, int out_is_bf16, size_t bh,
                      size_t sq, size_t sk, size_t d, float scale, const FvMask& mask, void* workspace, void* stream);
extern "C" hipError_t fv_internal_clear_queue(int* queue, hipStream_t stream);
extern "C" int fv_internal_flash_block_m(void);   // queries per workgroup of the flash kernel in use
extern "C" hipError_t fv_internal_launch_duo(const fv::FlashParams* p, int masked, int d, hipStream_t stream);   // total, nqt: of 128 queries
extern "C" hipError_t fv_internal_launch_flash(const fv::FlashParams* p, int masked, int d, int block_m,
                                               hipStream_t stream);
extern "C" hipError_t fv_internal_exact_pass_reruns(unsigned long long* out);
extern "C" hipError_t fv_internal_launch_tile_mean(const void* x, int x_is_bf16, const int* slot_src,
                                                   const int* block_sizes, float* out, size_t bh,
                                                   size_t seq, int dim, int num_tiles, int round16,
                                                   hipStream_t st);
extern "C" hipError_t fv_internal_launch_coarse(const float* qc, const float* kc, const float* vc,
                                                float* scores, float* coarse, size_t bh, int nb,
                                                int dim, float scale, hipStream_t st);
extern "C" hipError_t fv_internal_launch_topk(const float* scores, unsigned* out, int rows, int n, int k,
                                              int* zero, int zeros, hipStream_t st);
extern "C" hipError_t fv_internal_launch_tile_scan3(const void* const x[3], int x_is_bf16, const int* slot_src,
                                                    const int* block_sizes, uint16_t* const tiles[3],
                                                    float* const means[3], const float* copy_mul, size_t bh, size_t seq,
                                                    size_t padded, int num_tiles, hipStream_t st);
extern "C" hipError_t fv_internal_launch_tile_qkv(const void* x, int x_is_bf16, const int* slot_src,
                                                  uint16_t* xt, size_t bh, size_t seq, size_t padded,
                                                  int dim, hipStream_t st);
int fv_compute_units();   // of the first device used
// How a launch on f32 operands that are not rounded (three parts) is cut where the caller has a workspace for it.
fv::ComposedPlan fv_composed_plan(size_t bh, size_t sq, size_t sk, size_t d);
// softmax(scale q k^T + mask) v in f32 arithmetic, head dims 1 .. 128 (composed_fwd.hip). kv_is_bf16: k and v are bf16
// bits (else f32); round16: operands that arrive as f32 are rounded to bf16 first (RNE). A bf16 q with f32 k / v needs
// round16 == 0 to be exact; an f32 q with bf16 k / v is rounded.
extern "C" hipError_t fv_internal_launch_composed(const fv::ComposedParams* p, int kv_is_bf16, int round16, size_t bh,
                                                  hipStream_t st);
extern "C" hipError_t fv_internal_launch_short(const fv::ComposedParams* p, int waves, size_t bh, hipStream_t st);
extern "C" void fv_internal_count_log2_domain(void);
extern "C" hipError_t fv_internal_launch_splitkv_merge(const float* part_o, const float* part_lse, void* out,
                                                       int out_is_bf16, size_t rows, int d, int splits,
                                                       hipStream_t st);
extern "C" hipError_t fv_internal_init_flash(void);
extern "C" hipError_t fv_internal_init_vsa(void);
extern "C" hipError_t fv_internal_init_composed(void);
extern "C" size_t fv_internal_fine_pace(fv::VsaFineParams* p);
extern "C" hipError_t fv_internal_launch_fine(const fv::VsaFineParams* p, hipStream_t st);
extern "C" hipError_t fv_internal_launch_combine(const float* sparse, const float* coarse,
                                                 const void* gate, int gate_is_bf16,
                                                 const int* slot_src, float* out, size_t bh,
                                                 size_t seq, int num_tiles, int q_base, int q_tiles,
                                                 int round16, hipStream_t st);

// Error plumbing of the C ABI (defined in fv_api.hip): the message is kept per thread.
int fv_fail_hip(hipError_t e, const char* what);   // returns -(int)e
int fv_decline(const char* why);                    // returns FV_DECLINED
int fv_invalid(const char* why);                    // returns -(int)hipErrorInvalidValue

// Raise a kernel's dynamic LDS limit once per device (the attribute belongs to the function
// on the current device). `done` holds one bit per device ordinal; concurrent first calls may
// both set the attribute, which is harmless.
inline hipError_t fv_set_max_lds_once(const void* fn, int bytes, std::atomic<unsigned long long>& done) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const unsigned long long bit = 1ull << (dev & 63);
    if (done.load(std::memory_order_acquire) & bit) return hipSuccess;
    e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e == hipSuccess) done.fetch_or(bit, std::memory_order_release);
    return e;
}
