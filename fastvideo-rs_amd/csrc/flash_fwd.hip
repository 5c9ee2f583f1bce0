// Dense and block-causal flash attention forward for gfx950, head dim 128 or 64, bf16.
//
// Replaces the reference's flash_mma_fwd2_d128 / flash_mma_fwd2_causal_d128
// (crates/fastvideo-cudarc/src/rt/kernels/attn2.cu:40-352) behind
// attn::device_mma_sdpa / device_mma_sdpa_causal (rt/attn.rs:225-421, 652-730), and
// flash_mma_fwd2_window_d128 (attn2.cu:356-578) behind device_mma_sdpa_window
// (rt/attn.rs:526-610).
//
// Schedule (not a translation of the CUDA one):
//   * one workgroup = 8 waves = 256 queries of one (batch, head); each wave
//     owns 32 queries and walks the keys in tiles of 64;
//   * the wave computes S^T = K Q^T with v_mfma_f32_16x16x32_bf16: K rows come
//     from LDS as the A operand, each fragment for two MFMAs, Q^T stays in registers as the B operand for
//     the whole kernel. In the 16x16 accumulator layout every lane then holds
//     16 scores of each of TWO queries, so row maxima and row sums are in-lane reductions
//     plus exchanges with lane^32 and lane^16. The shape is a matter of power, at whose limit long launches run: on
//     random operands the chip sustains 2.01 PFLOP/s of it from registers and 1.74 with this kernel's LDS reads,
//     1.73 and 1.52 of v_mfma_f32_32x32x16_bf16 on the same operands (on zeros both 2.45). Its MFMAs are twice as many
//     and take the SIMD's issue port twice as long, so everything else in a phase had to shrink with it. Together, against
//     the 32x32 form: 12 x 32760 x 32760 x 128 4.92 -> 4.40 ms, block-causal 21 x 1560 2.69 -> 2.55, 24 x 7800 x 7800 x 64
//     363 -> 344 us. Launches that the power limit does not hold, of one round, lose by it where the softmax is the longer
//     part: f32 results 12 x 4000 x 4096 x 64 66.2 -> 70.2 us;
//   * P^T (bf16, RNE) is the B operand of O^T = V^T P^T straight from those
//     registers (the contraction index is a fixed permutation of the keys,
//     matched on the V side); V^T fragments are read from the row-major
//     [key][d] LDS tile with ds_read_b64_tr_b16;
//   * online softmax in base 2 with f32 max / sum / accumulators. The
//     accumulator is rescaled only when some row's max grew by more than
//     2^kRescaleLog2 since the last rescale; the final O / l is exact for any
//     such choice because P and l always share the same reference max;
//   * waves 0-3 (group 0) and 4-7 (group 1) share the SIMDs pairwise and run
//     half an iteration apart: while one group is in its MFMA phase (O += P V
//     of the previous tile, S = K Q^T of the current one, operands prefetched
//     from LDS a fixed number of MFMAs ahead) the other is in its VALU phase
//     (softmax of its current tile), separated by workgroup barriers, so each
//     SIMD's matrix pipe and vector ALU are busy at the same time by
//     construction. Interleaving the two instruction kinds inside one wave
//     loses on this hardware: a wave issues in order, so its VALU work stalls
//     behind every MFMA that waits for the matrix pipe;
//   * K/V tiles go global -> LDS directly (buffer_load_dwordx4 ... lds) into
//     XOR-swizzled unpadded tiles, four buffers each; rows past the last key are the descriptor's business;
//   * dense launches remap workgroup ids so that the workgroups resident on one
//     XCD walk consecutive query tiles of the same head (their K/V stream hits
//     that XCD's L2); masked launches run longest tiles first, long ones from a queue head by head (take_item).
//
// Time is counted in slots (one phase each); a phase covers a PAIR of key tiles
// (128 keys): a matrix phase is 128 MFMAs (PV of the previous pair, QK of the
// current pair), a VALU phase the softmax of the pair with one shared max /
// rescale decision. Barriers, the LDS-latency ramp at the head of a matrix phase
// and the per-phase bookkeeping are thus paid once per 128 keys. Group 0 runs
// matrix phase m in slot 2m and VALU phase m in slot 2m+1; group 1 is one slot
// behind. K and V tiles rotate through 4 LDS buffers each (128 KB): matrix phase
// m reads K(2m), K(2m+1), V(2m-2), V(2m-1) and issues K(2m+2), K(2m+3), V(2m),
// V(2m+1) into the buffers phase m-1 read last, all of them during the first tile
// of the pair (a load needs more than a thousand cycles to land), at offsets worked out in the VALU phase before, so the
// matrix phase carries bare DMA instructions and no branches. The VALU phase, in turn, is kept to the softmax itself: the
// other wave's MFMAs leave it about half the issue slots, and every scalar instruction and branch in it counts (the masks
// are asked by position of the walk, WalkSight; with per-lane tests, clamps and 64-bit addresses block-causal launches
// were 5 % slower than in the 32x32 form instead of 9 % faster).
// Every wave waits for its own loads at the end of the same phase, one barrier
// before phase m+1 of either group reads them. Phase 0 has no previous pair and runs its QK half only
// (unrolled apart from the loop). An odd tile count is rounded up: the extra
// tile re-reads the last one and all its scores are masked. Tile indices are walk
// positions: a masked call walks up to three ascending tile ranges (block-causal:
// sink tiles, then the band; VDN window: rows before the video + frame 0, the
// window frames, the last frame + rows after the video).
#include <stdlib.h>
#include <string.h>

#include "attn_core.h"
#include "fv_internal.h"

namespace fv {

constexpr int kBN = 64;          // keys per tile
constexpr int kPpBM = 256;      // queries per workgroup
constexpr int kRing2 = 4;        // K buffers = V buffers: 128 KB of LDS at D = 128, 64 KB at D = 64
constexpr int kVoteBytes = 64;   // behind the rings: one word per wave for the fixed-offset pass's vote

// Workgroups that had to redo their pass with the running max (see flash_item) since the library was loaded on
// this device.
__device__ unsigned long long g_exact_pass_reruns;

// VDN window launches: the r-th query tile in the order of work. Tiles that hold a global row or a row of an anchor
// frame walk every key and come first (the front ones, then the back ones); then the tiles of inner frames upwards
// from the first frame whose window is not cut off by the start of the clip, and last, downwards, the frames before
// it, whose walks are the shortest. Tiles in flight together are neighbours and stream the same keys, and the last
// round is short. The order it replaces took tiles from both ends in turn, so two far windows of every head were in
// flight and the longest inner walks came last: 12 heads, 32 frames x 1560, chunk 5, radius 1: 7.45 -> 6.47 ms;
// 16 frames, chunk 3: 2.43 -> 2.14; 40 heads, 18 frames x 880, chunk 5, radius 2: 4.27 -> 4.10; clips whose windows
// cover everything: equal. (Heads dealt to XCDs besides, so that an L2 serves few of them: equal to 1 %.)
template <int BM, class Params>
FV_DEV int vdn_tile_order(const Params& p, int r) {
    const int n = p.nqt, t = p.ft;
    const int front = min(n, (p.vs + t + BM - 1) / BM);         // tiles [0, front)
    const int back = min(n, max(front, (p.ve - t) / BM));          // tiles [back, n)
    const int first_full = max(1, min(p.frames, (int)min(0x7fffffffL, (long)p.radius * max(1, p.chunk))));
    const int start = min(max((p.vs + first_full * t) / BM, front), back);
    if (r < front) return r;
    r -= front;
    if (r < n - back) return back + r;
    r -= n - back;
    if (r < back - start) return start + r;
    return back - 1 - r;   // r counts on from back - start: start - 1 down to front
}

// The kernel's arguments read again from their segment, of which FlashParams is the whole: for code that runs rarely, so
// that the loop around it keeps none of them in registers.
using ConstParams = const __attribute__((address_space(4))) FlashParams;
FV_DEV ConstParams* params_again() {
    ConstParams* again = (ConstParams*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(again));
    return again;
}
// The first n of 64 bits.
FV_DEV unsigned long long first_bits(int n) {
    const unsigned long long m = ~0ull >> ((64 - n) & 63);
    return n <= 0 ? 0ull : n >= 64 ? ~0ull : m;
}
// Scores of query block g that the lane's query may not see to -inf, and those of keys `left` (counted from the tile's first)
// and on; `at`: the tile's first key. The bounds make one word of 64 keys, and a score costs a test of its bit and a
// select: 3 vector instructions where four comparisons and their scalar joins took 9, and no path apart for tiles that are whole
// for each query. us, 32x32x16 form / comparisons / so: causal 12 heads 21 x 1560 2713 / 2542 / 2480, 40 heads 34 x 390 under
// a window of one 366 / 380 / 290, VDN window 12 heads 32 x 1560 chunk 5 6421 / 5970 / 5872, 24 heads 30 x 100 radius 2 106 / 104 / 77. (The
// bounds worked out anew a tile, two integer divisions a query, took a phase 10 us instead of 2.9: they are kept, see lane_masks and
// duo_item.)
FV_DEV void mask_scores(ScoreTile& s, int g, const LaneMask& m, int at, int q4, int left) {
    const int x = at + 4 * q4;   // bit b: key x + b
    const unsigned long long seen = (first_bits(m.a_hi - x) | ~first_bits(m.c_lo - x) | (first_bits(m.w_hi - x) & ~first_bits(m.w_lo - x))) &
                                    first_bits(left - 4 * q4);
    const unsigned hidden[2] = {~(unsigned)seen, ~(unsigned)(seen >> 32)};
#pragma unroll
    for (int kb = 0; kb < 4; kb++)
#pragma unroll
        for (int i = 0; i < 4; i++) s[kb][g][i] = (hidden[kb >> 1] >> (16 * (kb & 1) + i)) & 1 ? neg_inf() : s[kb][g][i];
}
// The scores as they are, in registers of their own: around code that runs rarely, whose merges would otherwise cost the
// common way copies of them.
FV_DEV void pin_scores(ScoreTile& s) {
#pragma unroll
    for (int kb = 0; kb < 4; kb++) asm volatile("" : "+v"(s[kb][0]), "+v"(s[kb][1]));
}
FV_DEV void mask_keys(ScoreTile& s, int left) {
#pragma unroll
    for (int kb = 0; kb < 4; kb++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const bool vis = 16 * kb + i < left;
            s[kb][0][i] = vis ? s[kb][0][i] : neg_inf();
            s[kb][1][i] = vis ? s[kb][1][i] : neg_inf();
        }
}

// A wave's 32 rows o * inv in bf16, the first of them row `row0` of the result; `rows` (and no more) are stored. `my`:
// 32 x 2D bytes of LDS of the wave's own: scattered 8-byte pieces in, whole rows out, 16 bytes per lane and 1 KB (D = 128)
// of consecutive output per store instruction.
template <int D>
FV_DEV void store_rows16(lds_u8* my, const f32x4 (&o)[D / 16][2], const float (&inv)[2], uint16_t* out, size_t row0, int rows, int lane) {
    const int q4 = lane >> 4, i16 = lane & 15;
    constexpr int kRowB = 2 * D, kCh = kRowB / 16;
#pragma unroll
    for (int db = 0; db < D / 16; db++)
#pragma unroll
        for (int g = 0; g < 2; g++) {
            f32x4 r;
#pragma unroll
            for (int x = 0; x < 4; x++) r[x] = o[db][g][x] * inv[g];
            const bf16x4 rb4 = __builtin_convertvector(r, bf16x4);
            const int ch = (2 * db + (q4 >> 1)) ^ (i16 & (kCh - 1));
            *reinterpret_cast<__attribute__((address_space(3))) bf16x4*>(my + (16 * g + i16) * kRowB + (ch << 4) + 8 * (q4 & 1)) = rb4;
        }
    // (same-wave LDS writes and reads complete in order; the compiler waits on the reads' data)
    constexpr int kRowsPer = 64 / kCh;           // rows one store instruction covers
    const int lr = lane / kCh, lc = lane % kCh;
    uint16_t* ob = out + row0 * D;
#pragma unroll
    for (int i = 0; i < 32 / kRowsPer; i++) {
        const int rr = i * kRowsPer + lr;
        const u32x4 val = *reinterpret_cast<const __attribute__((address_space(3))) u32x4*>(
            my + rr * kRowB + ((lc ^ (rr & (kCh - 1))) << 4));
        if (rr < rows) global_store<u32x4>(ob + (size_t)rr * D + lc * 8, val);
    }
}

// One workgroup's item: the whole pass over its key tiles and the store of its rows. Returns false (FIXED only,
// nothing stored) when the pass has to be made again with the running max.
// FIXED: once the first phase has put every query's offset at the largest score of its first 128 keys, the offset
// stays there: no row max and no rescale decision in the loop (32 three-operand VALU instructions a phase less:
// 2 % of the time of the long launches, 9 % at head dim 64). Exact for any input as long as nothing overflows (P
// and l share the offset), so the pass is checked before anything is stored: if some row's scores grew by more
// than about 2^90 past that first maximum (a row sum of 2^100 or more, whose reciprocal nears the subnormals, or an accumulator not
// finite), the workgroup makes the pass again from the top with the running max. One difference in rounding
// remains: the largest P of a row is exactly 1 under the running max and a rounded bf16 number under the fixed
// offset, so a row that ONE late key dominates can be off by up to 2^-8 relative; the launcher therefore takes
// this form only for results that are rounded to bf16 anyway.
template <int NG, bool MASKED, int D, bool LOG2DOM, bool FIXED, bool FAR, class Params>
FV_DEV bool flash_item(const Params& p, const int wave, const int lane, const int block) {
    // (masked launches: only where every query sees key 0, see launch_flash)
    using G = TileGeo<D>;
    constexpr int kD = D;
    constexpr int kTileBytes = G::kTile;
    constexpr int kBM = 128 * NG;
    static_assert(NG == 2 || (NG == 1 && !MASKED), "one group: dense launches only");
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    lds_u8* smem = (lds_u8*)smem_raw;

    const int tid = wave * 64 + lane;   // (wave is scalar: branches on it stay scalar)
    const int grp = wave >> 2;
    const int q4 = lane >> 4, i16 = lane & 15;   // this lane's queries: rows i16 and 16 + i16 of the wave's 32
    // Work order. Dense (equal tiles): workgroup i runs on XCD i % 8, and XCD x takes the
    // contiguous range [x, x+1) * per_xcd of (head, query tile) items, so its CUs stream one
    // head's K/V through its L2 together. Masked (tiles differ in length by up to the whole
    // sequence): longest first over the whole launch, tile index major and head minor
    // (block-causal: last tile first; VDN window: vdn_tile_order); measured 9 % faster than the
    // dense order, whose per-XCD ranges hold unequal work.
    int bh, qt, sp = 0;   // sp: this workgroup's key split
    bool split = false;   // dense launches: one of the kv_split workgroups of its query tile
    if constexpr (MASKED) {
        const int work = block;
        if (work >= p.total) return true;
        const int nbh = p.total / p.nqt;
        bh = work % nbh;
        const int r = work / nbh;
        qt = p.mask_mode == 2 ? vdn_tile_order<kPpBM>(p, r) : p.nqt - 1 - r;
    } else {
        // (the unsplit query tiles first, dealt like a launch of their own: p.full is a multiple of 8)
        const bool whole = block < p.full;
        const int b = whole ? block : block - p.full;
        int work = (b & 7) * (whole ? p.full >> 3 : p.per_xcd) + (b >> 3);
        if (!whole) {
            if (work >= p.total) return true;
            split = p.kv_split > 1;
            sp = work % p.kv_split;
            work = p.full + work / p.kv_split;
        }
        bh = work / p.nqt;
        qt = work - bh * p.nqt;
    }
    const int q0 = qt * kBM;
    const int sq = p.sq, sk = p.sk;
    const int qlen = min(kBM, sq - q0);
    const float sl2 = p.sl2;
    const float NEG = neg_inf();
    // Fetch the epilogue's arguments now. Left to the compiler, their scalar loads sit
    // right before the main loop, still pending at its head, and a pending scalar load
    // (out-of-order return) turns every LDS wait count in the loop into a full drain.
    float* out_f32 = p.out_f32;
    uint16_t* out_bf16 = p.out_bf16;
    int out_is_bf16 = p.out_is_bf16;
    asm volatile("" : "+s"(out_f32), "+s"(out_bf16), "+s"(out_is_bf16));

    const uint16_t* Qh = p.q + (size_t)bh * p.q_plane + (size_t)q0 * kD;
    const uint16_t* Kh = p.k + (size_t)bh * p.k_plane;
    const uint16_t* Vh = p.v + (size_t)bh * p.v_plane;

    const int nkt_all = (sk + kBN - 1) / kBN;
    // a split walks key tiles [t0, t0 + nkt) of the nkt_all tiles (the whole range without split-KV)
    const int t0 = split ? sp * p.split_tiles : 0;
    const int nkt = split ? min(p.split_tiles, nkt_all - t0) : nkt_all;
    // The key-tile walk of this query tile: up to three ascending tile ranges [a_i, a_i + n_i),
    // n0 + n1 + n2 = ne tiles in all. A lane's query sees key x iff
    //   x < a_hi  ||  x >= c_lo  ||  (w_lo <= x && x < w_hi).
    int a1 = 0, a2 = 0, n0 = nkt, n1 = 0, ne = nkt;
    WalkSight sight = {0, 0, 0, 0};
    // (masked: the bounds of the wave's queries behind the vote, the wave's own business)
    auto* const lane_masks = (__attribute__((address_space(3))) u32x4*)(smem + 2 * kRing2 * kTileBytes + kVoteBytes) + wave * 32;
    if constexpr (MASKED) {
        const TileWalk w = mask_tile_walk(p, q0, qlen, nkt);
        a1 = w.a1;
        a2 = w.a2;
        n0 = w.n0;
        n1 = w.n1;
        ne = w.ne;
        sight = walk_sight(p, w, q0 + wave * 32);
        if (lane < 32) lane_masks[lane] = __builtin_bit_cast(u32x4, lane_mask(p, q0 + wave * 32 + lane));
    }
    if constexpr (MASKED) {
        // No key tile is visible to any query of this tile (block-causal with more queries than keys
        // and a window that has moved past the last key): rows of zeros, what a query without a
        // visible key gets in a partly visible tile too (l == 0). Workgroup-uniform, before any barrier.
        if (ne <= 0) {
            const int units = kD * (out_is_bf16 ? 2 : 4) / 16;   // 16-byte units per output row
            char* ob = out_is_bf16 ? (char*)(out_bf16 + ((size_t)bh * sq + q0) * kD)
                                   : (char*)(out_f32 + ((size_t)bh * sq + q0) * kD);
            const u32x4 zero = {0u, 0u, 0u, 0u};
            for (int u = tid; u < qlen * units; u += 512) global_store<u32x4>(ob + (size_t)u * 16, zero);
            return true;
        }
    }
    const int np = (ne + 1) / 2;             // phases
    // first key of walk position e; positions past the end repeat the last tile (their scores are masked)
    auto kv0_of = [&](int e) -> int {
        e = min(e, ne - 1);
        if constexpr (MASKED) return (e < n0 ? e : e < n0 + n1 ? a1 + (e - n0) : a2 + (e - n0 - n1)) * kBN;
        else return (t0 + e) * kBN;
    };
    // Tile t lives in K buffer t mod 4 and V buffer t mod 4 (behind the K ring).
    using Dma = TileDma<4 * NG, D>;
    Dma dma;
    dma.init(wave, lane);
    constexpr int kUnits = Dma::kUnits;
    const u32x4 kplane = plane_descriptor(Kh, FAR ? 0u : (unsigned)sk * G::kRow), vplane = plane_descriptor(Vh, FAR ? 0u : (unsigned)sk * G::kRow);
    // (planes of 4 GB and more: a descriptor per tile)
    auto load_k = [&](int kv0, unsigned lds, int u) {
        if constexpr (FAR) dma.template issue<false>(plane_descriptor(Kh + (size_t)kv0 * kD, (unsigned)min(sk - kv0, kBN) * G::kRow), 0, lds, u);
        else dma.template issue<false>(kplane, (unsigned)kv0 * G::kRow, lds, u);
    };
    auto load_v = [&](int kv0, unsigned lds, int u) {
        if constexpr (FAR) dma.template issue<true>(plane_descriptor(Vh + (size_t)kv0 * kD, (unsigned)min(sk - kv0, kBN) * G::kRow), 0, lds, u);
        else dma.template issue<true>(vplane, (unsigned)kv0 * G::kRow, lds, u);
    };
    const unsigned ring = (unsigned)__builtin_amdgcn_readfirstlane((int)(size_t)smem);
    {
        const int k0 = kv0_of(0), k1 = kv0_of(1);
#pragma unroll
        for (int u = 0; u < kUnits; u++) {
            load_k(k0, ring, u);
            load_k(k1, ring + kTileBytes, u);
        }
    }
    bf16x8 qf[D / 32][2];
    const TileReadBases rb = tile_read_bases<D>(lane);
    // The wave's 32 query rows come through LDS: whole rows by LDS-DMA (1 KB of consecutive global memory per
    // instruction) into the wave's own slice of the V ring (group 0: buffers 0, 1, idle until the first matrix
    // phase requests V(0); group 1: buffers 2, 3, idle a phase longer), in the K tiles' swizzle, then the fragments
    // with the K operand's conflict-free read pattern. (Loading the fragments straight from global memory takes
    // 16-byte pieces of 32 rows per instruction: 2 - 3 % slower on 512-key launches, whose prologue shows.)
    // Group 1, which idles through the first slot anyway, waits for its rows only then: group 0 starts as soon as
    // K(0), K(1) and its own rows are there.
    lds_u8* qs = smem + kRing2 * kTileBytes + wave * (32 * G::kRow);
    auto q_request = [&]() {
        const unsigned qlds = __builtin_amdgcn_readfirstlane((unsigned)(size_t)qs);
        constexpr int kQIt = 32 * G::kRow / 1024;
#pragma unroll
        for (int it = 0; it < kQIt; it++) {
            const int r = it * G::kRowsPerDma + lane / G::kChunks, pch = lane % G::kChunks;
            const int rg = min(wave * 32 + r, qlen - 1);   // rows past the end re-read the last one (zeroed below)
            lds_dma16_s(qlds + it * 1024, Qh, (unsigned)(rg * G::kRow + ((pch ^ G::kswz(r)) << 4)));
        }
    };
    auto q_read = [&]() {
        wait_vmcnt<0>();   // this wave's rows (and its parts of K(0), K(1)) have landed
#pragma unroll
        for (int g = 0; g < 2; g++) {
            const bool ok = wave * 32 + 16 * g + i16 < qlen;
#pragma unroll
            for (int dk = 0; dk < D / 32; dk++) {
                bf16x8 t = lds_read_b128(qs + (rb.k ^ (dk << 6)) + 16 * g * G::kRow);
                if (!ok) t = __builtin_bit_cast(bf16x8, u32x4{0u, 0u, 0u, 0u});
                qf[dk][g] = t;
            }
        }
        __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): the slice is read before the wave passes its next barrier
    };
    if (grp == 0) {
        q_request();
        q_read();
    } else {
        q_request();
        wait_vmcnt<32 * G::kRow / 1024>();   // this wave's parts of K(0), K(1); its query rows are still in flight
    }

    constexpr int kNO = D / 16;   // 16-wide d blocks of the accumulator
    f32x4 o[kNO][2];
#pragma unroll
    for (int db = 0; db < kNO; db++)
#pragma unroll
        for (int g = 0; g < 2; g++) o[db][g] = f32x4{0.f, 0.f, 0.f, 0.f};
    SoftmaxOffState st;
    st.init();
    // the C operand every S block starts from: minus the lane's softmax offset (zero until the first rescale)
    f32x4 s_init[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    ScoreTile s0, s1;
    ProbTile pb0, pb1;     // P of the previous pair of tiles (first read in phase 1; defined from the start)
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int g = 0; g < 2; g++) pb0[t][g] = pb1[t][g] = __builtin_bit_cast(bf16x8, u32x4{0u, 0u, 0u, 0u});

    // What the next matrix phase loads: V of the tiles at positions 2 m and 2 m + 1 (first keys kv[0], kv[1]), K of the two behind
    // them (kk), and the LDS addresses of their pairs of buffers.
    int kv[2] = {kv0_of(0), kv0_of(1)}, kk[2] = {kv0_of(2), kv0_of(3)};
    unsigned vlds = ring + kRing2 * kTileBytes, klds = ring + 2 * kTileBytes;
    // Per-lane LDS addresses of the operand fragments of the first tile of the pair a matrix phase reads: K tiles
    // 2m, 2m+1 sit in buffers 2 (m & 1) + {0, 1}, V tiles 2m-2, 2m-1 in buffers 2 (1 - m & 1) + {0, 1}, so every
    // phase flips one bit (two tiles' worth) in each register instead of adding a buffer base to every read.
    const lds_u8* ka[D / 32];
    const lds_u8* va[D / 16];
#pragma unroll
    for (int dk = 0; dk < D / 32; dk++) ka[dk] = smem + (rb.k ^ (dk << 6));
#pragma unroll
    for (int db = 0; db < D / 16; db++) va[db] = smem + ((rb.v ^ (db << 5)) + (kRing2 + 2) * kTileBytes);
    // (the ring starts at LDS address 0 and spans a power of two, so flipping an address bit moves between buffers)
    auto flip = [](const lds_u8* q, unsigned bit) -> const lds_u8* {
        return (const lds_u8*)(__attribute__((address_space(3))) void*)(size_t)((unsigned)(size_t)q ^ bit);
    };

    block_barrier();                 // K(0), K(1) resident
    if (grp == 1) {                  // group 1 takes its query rows in slot 0, in which it has nothing else to do
        q_read();
        block_barrier();
    }

    // scores of walk position e, whose first key is kv0: keys past the end (or a position past the walk) to -inf; masked
    // launches: keys this lane's queries may not see to -inf
    auto mask_tile = [&](ScoreTile& s, int e, int kv0) {
        const int left = (e >= ne ? 0 : sk) - kv0;
        if constexpr (MASKED) {
#pragma unroll
            for (int g = 0; g < 2; g++) mask_scores(s, g, __builtin_bit_cast(LaneMask, (u32x4)lane_masks[16 * g + i16]), kv0, q4, left);
        } else {
            mask_keys(s, left - 4 * q4);
        }
    };
    const bool ragged = (ne & 1) != 0 || kv0_of(ne - 1) + kBN > sk;   // keys past the end in the last phase

    // The first phase of a walk has no previous pair to multiply: it is unrolled apart (part 0) and runs
    // the K groups only.
#pragma unroll
    for (int part = 0; part < 2; part++) {
    const bool first = part == 0;
    const int m_begin = part == 0 ? 0 : 1;
    const int m_end = part == 0 ? 1 : np;
#pragma unroll 1
    for (int m = m_begin; m < m_end; m++) {
        // ---- matrix phase: group 0 in slot 2m, group 1 in slot 2m+1 ----
        __builtin_amdgcn_s_setprio(1);
        constexpr int kAhead = 3;
        // All of the phase's loads go out during the FIRST tile of the pair, a unit after each of its first groups, in the
        // order the next phase reads the tiles (V of its first tile, K of its first tile, then the second tile's). A load takes well over
        // a thousand cycles to land when every CU streams K/V; issued from the second tile's groups
        // they were still in flight at the end of the phase (330 cycles of every matrix phase
        // spent in the wait below, measured with shader-clock stamps).
        auto hook_dma = [&](int i) {
            const int x = i / kUnits, u = i % kUnits;
            if (x >= 4) return;
            if (x & 1) load_k(kk[x >> 1], klds + (x >> 1) * kTileBytes, u);
            else load_v(kv[x >> 1], vlds + (x >> 1) * kTileBytes, u);
        };
        const ProbTile* const pbs[2] = {&pb0, &pb1};
        ScoreTile* const ss[2] = {&s0, &s1};
        if (first) mfma_phase<false, kAhead, 2, D>(va, ka, pbs, o, qf, ss, s_init, hook_dma);
        else mfma_phase<true, kAhead, 2, D>(va, ka, pbs, o, qf, ss, s_init, hook_dma);
        __builtin_amdgcn_s_setprio(0);
        if constexpr (NG == 2) {
            wait_vmcnt<0>();             // this wave's loads of this phase have landed
            __builtin_amdgcn_sched_barrier(0);
            block_barrier();
        }
        __builtin_amdgcn_sched_barrier(0);
        // ---- VALU phase: group 0 in slot 2m+1, group 1 in slot 2m+2 ----
        if ((m == np - 1 && ragged) || (MASKED && !sight.all(2 * m, 2 * m + 1))) {
            if constexpr (MASKED) pin_scores(s0), pin_scores(s1);
            mask_tile(s0, 2 * m, kv[0]);
            mask_tile(s1, 2 * m + 1, kv[1]);
            if constexpr (MASKED) pin_scores(s0), pin_scores(s1);
        }
        if (FIXED && !first) softmax_tile_pair_fixed<!LOG2DOM>(s0, s1, st, sl2, pb0, pb1);
        else softmax_tile_pair_off<!LOG2DOM, kNO>(s0, s1, st, o, s_init, sl2, pb0, pb1);
        // P and the row sum must be complete before the barrier: without this the
        // compiler sinks the exponentials past it, into the matrix phase
        asm volatile("" ::"v"(pb0[0][0]), "v"(pb0[0][1]), "v"(pb0[1][0]), "v"(pb0[1][1]), "v"(pb1[0][0]), "v"(pb1[0][1]),
                     "v"(pb1[1][0]), "v"(pb1[1][1]), "v"(st.l_acc[0]), "v"(st.l_acc[1]));
#pragma unroll
        for (int dk = 0; dk < D / 32; dk++) ka[dk] = flip(ka[dk], 2 * kTileBytes);   // the other pair of K buffers
#pragma unroll
        for (int db = 0; db < D / 16; db++) va[db] = flip(va[db], 2 * kTileBytes);   // ... and of V buffers
        vlds ^= 2 * kTileBytes;
        klds ^= 2 * kTileBytes;
        kv[0] = kk[0];               // for matrix phase m + 1
        kv[1] = kk[1];
        kk[0] = kv0_of(2 * m + 4);
        kk[1] = kv0_of(2 * m + 5);
        // (here and not behind the barrier, at the head of the matrix phase, where the compiler would put them)
#pragma unroll
        for (int dk = 0; dk < D / 32; dk++) asm volatile("" : "+v"(ka[dk]));
#pragma unroll
        for (int db = 0; db < D / 16; db++) asm volatile("" : "+v"(va[db]));
        asm volatile("" : "+s"(kk[0]), "+s"(kk[1]), "+s"(vlds), "+s"(klds));
        if (NG == 1 || grp == 0 || m + 1 < np) {
            __builtin_amdgcn_sched_barrier(0);
            // (one group: the only barrier of a phase, behind which its loads are resident and its tiles read)
            if constexpr (NG == 1) wait_vmcnt<0>();
            block_barrier();
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    }
    // O += P V of the last pair (their V landed before the last barrier both groups passed)
    lds_u8* const vlast = smem + (kRing2 + ((2 * np - 2) & (kRing2 - 1))) * kTileBytes;
    pv_tile<D>(vlast, rb.v, pb0, o);
    pv_tile<D>(vlast + kTileBytes, rb.v, pb1, o);

    if constexpr (FIXED) {
        // Did the fixed offset hold? Every row sum below 2^100 (its reciprocal a normal number with room to spare) and every accumulator finite
        // (x * 0 is NaN for an infinite or NaN x). One vote per wave through 8 words of LDS behind the rings.
        float chk = 0.f;
#pragma unroll
        for (int db = 0; db < kNO; db++)
#pragma unroll
            for (int g = 0; g < 2; g++)
#pragma unroll
                for (int i = 0; i < 4; i++) chk = __builtin_fmaf(o[db][g][i], 0.f, chk);
        const bool lane_ok = quad_sum(st.l_acc[0]) < 0x1p+100f && quad_sum(st.l_acc[1]) < 0x1p+100f && chk == 0.f;
        auto* votes = (__attribute__((address_space(3))) unsigned*)(smem + 2 * kRing2 * kTileBytes);
        const bool wave_ok = __builtin_amdgcn_ballot_w64(!lane_ok) == 0;   // (of all lanes: outside the branch below)
        if (lane == 0) votes[wave] = wave_ok ? 0u : 1u;
        __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): the vote is written before the barrier
        block_barrier();   // ... behind which every wave is past its last read of both rings
        const u32x4 v0 = *reinterpret_cast<const __attribute__((address_space(3))) u32x4*>(votes);
        unsigned any = v0[0] | v0[1] | v0[2] | v0[3];
        if constexpr (NG == 2) {
            const u32x4 v1 = *reinterpret_cast<const __attribute__((address_space(3))) u32x4*>(votes + 4);
            any |= v1[0] | v1[1] | v1[2] | v1[3];
        }
        if (__builtin_amdgcn_readfirstlane(any) != 0) {
            if (tid == 0) atomicAdd(&g_exact_pass_reruns, 1ull);
            return false;
        }
    }

    float l_tot[2], inv[2];
#pragma unroll
    for (int g = 0; g < 2; g++) {
        l_tot[g] = quad_sum(st.l_acc[g]);
        inv[g] = l_tot[g] > 0.f ? 1.f / l_tot[g] : 0.f;
    }
    const int row = wave * 32 + i16;   // and row + 16
    if constexpr (!MASKED) {
        if (split) {
            // partial result of this split: O / l in f32 and log2 of the sum of 2^(s * sl2) it covers
#pragma unroll
            for (int g = 0; g < 2; g++) {
                if (row + 16 * g >= qlen) continue;
                const size_t prow = (size_t)sp * p.part_rows + ((size_t)bh * sq + q0 + row + 16 * g - p.part_row0);
                float* po = p.part_o + prow * kD;
#pragma unroll
                for (int db = 0; db < kNO; db++) {
                    f32x4 r;
#pragma unroll
                    for (int x = 0; x < 4; x++) r[x] = o[db][g][x] * inv[g];
                    global_store<f32x4>(po + 16 * db + 4 * q4, r);
                }
                if (q4 == 0)
                    p.part_lse[prow] = l_tot[g] == 0.f ? NEG : st.template log2_offset<!LOG2DOM>(g, sl2) + __builtin_log2f(l_tot[g]);   // (NaN stays)
            }
            return true;
        }
    }
    // (store_rows16() written out: its call costs the long masked launches 1 %)
    if (out_is_bf16) {
        // bf16 rows through this wave's own 32 x 2D-byte slice of the K ring (every K read is behind the last
        // barrier and no load is in flight): scattered 8-byte pieces in, whole rows out, 16 bytes per
        // lane and 1 KB (D = 128) of consecutive output per store instruction
        constexpr int kRowB = 2 * kD, kCh = kRowB / 16;
        lds_u8* my = smem + wave * (32 * kRowB);
#pragma unroll
        for (int db = 0; db < kNO; db++)
#pragma unroll
            for (int g = 0; g < 2; g++) {
                f32x4 r;
#pragma unroll
                for (int x = 0; x < 4; x++) r[x] = o[db][g][x] * inv[g];
                const bf16x4 rb4 = __builtin_convertvector(r, bf16x4);
                const int ch = (2 * db + (q4 >> 1)) ^ (i16 & (kCh - 1));
                *reinterpret_cast<__attribute__((address_space(3))) bf16x4*>(my + (16 * g + i16) * kRowB + (ch << 4) + 8 * (q4 & 1)) = rb4;
            }
        // (same-wave LDS writes and reads complete in order; the compiler waits on the reads' data)
        constexpr int kRowsPer = 64 / kCh;           // rows one store instruction covers
        const int lr = lane / kCh, lc = lane % kCh;
        uint16_t* ob = out_bf16 + ((size_t)bh * sq + q0 + wave * 32) * kD;
#pragma unroll
        for (int i = 0; i < 32 / kRowsPer; i++) {
            const int rr = i * kRowsPer + lr;
            const u32x4 val = *reinterpret_cast<const __attribute__((address_space(3))) u32x4*>(
                my + rr * kRowB + ((lc ^ (rr & (kCh - 1))) << 4));
            if (wave * 32 + rr < qlen) global_store<u32x4>(ob + (size_t)rr * kD + lc * 8, val);
        }
    } else {
#pragma unroll
        for (int g = 0; g < 2; g++) {
            if (row + 16 * g >= qlen) continue;
            float* po = out_f32 + ((size_t)bh * sq + q0 + row + 16 * g) * kD;
#pragma unroll
            for (int db = 0; db < kNO; db++) {
                f32x4 r;
#pragma unroll
                for (int x = 0; x < 4; x++) r[x] = o[db][g][x] * inv[g];
                global_store<f32x4>(po + 16 * db + 4 * q4, r);
            }
        }
    }
    return true;
}

// The queue of a long masked launch. A workgroup takes the next item of its XCD's list when it starts, and where that is used up
// one of another's: XCDs differ in speed by 5 %, and an eighth more workgroups than items are launched, so that the fast ones may
// take more (the rest find nothing and end). A list is the whole heads x * a .. one after the other and, tile by tile, a share of the
// heads past the last multiple of eight: one head at a time goes through an L2. An item is a (head, query tile), counted as
// `work` in flash_item.
// Which launches gain by it: fv_masked_workspace_bytes (causal 40 heads 21 x 1560 8624 us in the order of the numbers, where 36 % of the
// L2 lines missed, 7979 so). One workgroup a CU that walks item after item needs registers that the main loop then misses: 8649 and 3863
// where this form had 8345 and 3712 (those two: before a tile's bounds were one word of bits).
template <class Params>
FV_DEV int queue_item(const Params& p, int x, int j) {
    const int nqt = p.nqt, nbh = p.total / nqt, a = nbh >> 3, c = nbh & 7;
    if (j < a * nqt) return j % nqt * nbh + x * a + j / nqt;
    const int i = (j - a * nqt) * 8 + x;
    return i < c * nqt ? i / c * nbh + 8 * a + i % c : -1;
}
constexpr int kQueueStep = 32;   // words between the XCDs' counters: a line each
// The workgroup's item into `block`; false: there is none left.
template <int D, class Params>
FV_DEV bool take_item(const Params& p, const int wave, const int lane, int& block) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    auto* word = (__attribute__((address_space(3))) int*)((lds_u8*)smem_raw + 2 * kRing2 * TileGeo<D>::kTile + kVoteBytes / 2);
    if (wave == 0) {
        int got = -1;
        for (int i = 0; i < 8 && got < 0; i++) {
            const int x = (blockIdx.x + i) & 7;
            int j = 0;
            if (lane == 0) j = __hip_atomic_fetch_add((__attribute__((address_space(1))) int*)p.queue + x * kQueueStep, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            got = queue_item(p, x, __builtin_amdgcn_readfirstlane(j));
        }
        if (lane == 0) *word = got;
        __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): the word is written before the barrier
    }
    block_barrier();
    block = __builtin_amdgcn_readfirstlane(*word);
    return block >= 0;
}

// The softmax offset rides in the C operand of the K Q^T MFMAs (softmax_tile_pair_off): a score costs one multiply,
// one exponential and one add. LOG2DOM: the call's scale * log2(e) is exactly 1 (scores are base-2 logarithms as
// they leave the MFMAs) and the multiply is gone too. FIXED (launches that write bf16 and whose queries all see key 0): the first pass keeps
// the offset of the first 128 keys (flash_item); the others keep the running max throughout.
// NG: groups of four waves. Two (256 queries) alternate; one (128) runs its matrix and VALU phases in turn, with one
// barrier a phase and no slot in which a group waits for the other's first or last phase: for launches whose query tiles
// of 128 still have a CU each (fv_split_plan). Bit for bit the same rows. A phase takes 2.1 us instead of 2.4, a launch of
// one phase 7.1 instead of 8.2.
template <int NG, bool MASKED, int D, bool LOG2DOM, bool FIXED, bool FAR>
__global__ __launch_bounds__(256 * NG, 2) void flash_fwd_pp2(const FlashParams p) {
    const int tid = threadIdx.x;
    int wave = __builtin_amdgcn_readfirstlane(tid >> 6), block = blockIdx.x;
    if constexpr (MASKED)
        if (p.queue && !take_item<D>(p, wave, tid & 63, block)) return;
    if constexpr (!FIXED) {
        flash_item<NG, MASKED, D, LOG2DOM, false, FAR>(p, wave, tid & 63, block);
    } else {
        if (flash_item<NG, MASKED, D, LOG2DOM, true, FAR>(p, wave, tid & 63, block)) return;
        // The second pass shares nothing with the first but two scalars: its inputs are made opaque (the lane
        // index counted anew from the execution mask, the kernel arguments read again from their segment, of which
        // FlashParams is the whole), so that the compiler keeps no value of the first pass alive for it. It runs
        // once in a blue moon; the first pass is the kernel.
        ConstParams* again = params_again();
        int lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
        asm volatile("" : "+v"(lane), "+s"(wave), "+s"(block));
        flash_item<NG, MASKED, D, LOG2DOM, false, FAR>(*again, wave, lane, block);
    }
}

// Walks of few keys under a fixed offset (fv_duo, duo_masked): two workgroups a CU, three at head dim 64. flash_fwd_pp2
// gives an item the CU and pays its first loads, its first and last slot and its store in the open, half of the time at
// eight key tiles. Here an item is four waves x 32 queries with five buffers of a tile (80 KB at D = 128), so that two share
// a CU unsynchronised and one's ends pass under the other's arithmetic. A phase is one key tile: the matrix part (O += P V of
// the tile before, S = K Q^T, with the loads of the next K and of this V going out behind the first MFMAs), the softmax, one
// barrier; the first phase has two. Every sum is flash_fwd_pp2's, term by term: the offset of a row is the largest score of the walk's first two
// tiles, so the two kernels give the same bits and the line between them is drawn by time alone (a workgroup that goes
// again with the running max is one of 128 queries here and of 256 there: its rows differ by the rounding of P).
constexpr int kDuoBM = 128;
template <int D>
constexpr int kDuoLds = 5 * TileGeo<D>::kTile;
template <bool MASKED, int D, bool LOG2DOM, bool FIXED, class Params>
FV_DEV bool duo_item(const Params& p, const int wave, const int lane, const int block) {
    using G = TileGeo<D>;
    using Dma = TileDma<4, D>;
    constexpr int kTileBytes = G::kTile, kNO = D / 16, kIt = Dma::ITER, kUnits = Dma::kUnits;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    lds_u8* smem = (lds_u8*)smem_raw;
    const int q4 = lane >> 4, i16 = lane & 15;
    // work order as in flash_item: XCD x takes a contiguous eighth of the (head, query tile) items; masked, longest first
    const int work = MASKED ? block : (block & 7) * p.per_xcd + (block >> 3);
    if (work >= p.total) return true;
    int bh, qt;
    if constexpr (MASKED) {
        const int nbh = p.total / p.nqt, r = work / nbh;
        bh = work - r * nbh;
        qt = p.mask_mode == 2 ? vdn_tile_order<kDuoBM>(p, r) : p.nqt - 1 - r;
    } else {
        bh = work / p.nqt;
        qt = work - bh * p.nqt;
    }
    const int q0 = qt * kDuoBM, sq = p.sq, sk = p.sk, qlen = min(kDuoBM, sq - q0), nkt = (sk + kBN - 1) / kBN;
    int a1 = 0, a2 = 0, n0 = nkt, n1 = 0, ne = nkt;   // the walk, as in flash_item (key 0 is in it)
    WalkSight sight = {0, 0, 0, 0};
    // Masked: bounds of one of the wave's queries a lane, row lane % 32, which is query block q4 & 1; a tile that asks for them
    // gets both blocks' by an exchange (mask_tile). There is no LDS left for them at D = 128, bounds of both queries a lane
    // spilled accumulators, and worked out anew a tile they cost up to a fifth (VDN window 12 heads 8 x 390 107 / 78 us).
    LaneMask mine = {0, 0x7fffffff, 0, 0};
    if constexpr (MASKED) {
        const TileWalk w = mask_tile_walk(p, q0, qlen, nkt);
        a1 = w.a1, a2 = w.a2, n0 = w.n0, n1 = w.n1, ne = w.ne;
        sight = walk_sight(p, w, q0 + wave * 32);
        mine = lane_mask(p, q0 + wave * 32 + (lane & 31));
    }
    const float sl2 = p.sl2;
    uint16_t* out = p.out_bf16;
    asm volatile("" : "+s"(out));   // (fetched now, see flash_item)
    // first key of walk position e; positions past the end repeat the last tile
    auto kv0_of = [&](int e) -> int {
        e = min(e, ne - 1);
        if constexpr (MASKED) return (e < n0 ? e : e < n0 + n1 ? a1 + (e - n0) : a2 + (e - n0 - n1)) * kBN;
        else return e * kBN;
    };
    const uint16_t* Qh = p.q + (size_t)bh * p.q_plane + (size_t)q0 * D;
    const uint16_t* Kh = p.k + (size_t)bh * p.k_plane;
    const uint16_t* Vh = p.v + (size_t)bh * p.v_plane;

    // Buffers: K(0), K(1), V(0), V(1), K(2) each in its own; from then on odd phases read V(m - 1) and K(m) from 0 and 1 and
    // load V(m) and K(m + 1) into 3 and 4, even ones the other way round.
    auto kbuf = [&](int t) -> lds_u8* { return smem + (t == 0 ? 0 : t & 1 ? 1 : 4) * kTileBytes; };
    auto vbuf = [&](int t) -> lds_u8* { return smem + (t == 0 ? 2 : t & 1 ? 3 : 0) * kTileBytes; };
    Dma dma;
    dma.init(wave, lane);
    const u32x4 kplane = plane_descriptor(Kh, (unsigned)sk * G::kRow), vplane = plane_descriptor(Vh, (unsigned)sk * G::kRow);
    auto lds_of = [](lds_u8* b) { return (unsigned)__builtin_amdgcn_readfirstlane((int)(size_t)b); };
    auto load_k = [&](int t, int kv0, int u) { dma.template issue<false>(kplane, (unsigned)kv0 * G::kRow, lds_of(kbuf(t)), u); };
    auto load_v = [&](int t, int kv0, int u) { dma.template issue<true>(vplane, (unsigned)kv0 * G::kRow, lds_of(vbuf(t)), u); };
    bf16x8 qf[D / 32][2];
    const TileReadBases rb = tile_read_bases<D>(lane);
    {
        // the wave's query rows through its slice of buffers 2 and 3, as in flash_item; K(0) and K(1) besides
        lds_u8* qs = smem + 2 * kTileBytes + wave * (32 * G::kRow);
        const unsigned qlds = __builtin_amdgcn_readfirstlane((unsigned)(size_t)qs);
#pragma unroll
        for (int it = 0; it < 32 * G::kRow / 1024; it++) {
            const int r = it * G::kRowsPerDma + lane / G::kChunks, pch = lane % G::kChunks;
            const int rg = min(wave * 32 + r, qlen - 1);   // rows past the end re-read the last one (zeroed below)
            lds_dma16_s(qlds + it * 1024, Qh, (unsigned)(rg * G::kRow + ((pch ^ G::kswz(r)) << 4)));
        }
        const int k0 = kv0_of(0), k1 = kv0_of(1);
#pragma unroll
        for (int u = 0; u < kUnits; u++) load_k(0, k0, u);
        if (ne > 1) {
#pragma unroll
            for (int u = 0; u < kUnits; u++) load_k(1, k1, u);
            wait_vmcnt<2 * kIt>();
        } else {
            wait_vmcnt<kIt>();
        }
#pragma unroll
        for (int g = 0; g < 2; g++) {
            const bool ok = wave * 32 + 16 * g + i16 < qlen;
#pragma unroll
            for (int dk = 0; dk < D / 32; dk++) {
                bf16x8 t = lds_read_b128(qs + (rb.k ^ (dk << 6)) + 16 * g * G::kRow);
                if (!ok) t = __builtin_bit_cast(bf16x8, u32x4{0u, 0u, 0u, 0u});
                qf[dk][g] = t;
            }
        }
        __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): the slice is read before the wave passes its next barrier
    }
    auto mask_tile = [&](ScoreTile& s, int e) {
        if (e < ne - 1 && (!MASKED || sight.all(e, e))) return;
        const int kv0 = kv0_of(e), left = sk - kv0;
        if constexpr (MASKED) {
            const u32x4 m = __builtin_bit_cast(u32x4, mine);
            u32x4 both[2];   // the even rows of 16 lanes hold block 0's, the odd ones block 1's
#pragma unroll
            for (int x = 0; x < 4; x++) {
                const auto r = __builtin_amdgcn_permlane16_swap(m[x], m[x], false, false);
                both[0][x] = (unsigned)r[0];
                both[1][x] = (unsigned)r[1];
            }
#pragma unroll
            for (int g = 0; g < 2; g++) mask_scores(s, g, __builtin_bit_cast(LaneMask, both[g]), kv0, q4, left);
        } else {
            if (kv0 + kBN > sk) mask_keys(s, left - 4 * q4);
        }
    };
    f32x4 o[kNO][2], s_init[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    SoftmaxOffState st;
    ProbTile pb;
    // Two waves of a SIMD that are in step halve its rate: both multiply, then both are at their softmax. Where walks are of one
    // length and the launch is one round they start so, and the softmax, the longer part, goes first: whoever reaches it
    // gets its issue slots while the other multiplies. With the matrix part first, which served the 32x32x16 form well, waves stayed
    // in step. At 64 channels four groups of operands are read ahead, whose MFMAs leave the port to the other wave's softmax.
    // us, 32x32x16 form / matrix part first, three ahead / now, at 64 channels: 9 x 4000 x 512 12.3 / 13.0 / 12.5, x 1024 18.2 / 20.4 / 18.6,
    // x 4096 54.4 / 63.0 / 54.6, 16 x 2560 x 2048 30.9 / 34.9 / 30.8, 16 x 4000 x 4096 70.9 / 72.6 / 66.6, 16 x 7680 x 3000 103.5 / 101.0 / 98.1; at
    // 128: 9 x 4000 x 512 16.5 / 17.6 / 17.1, 16 x 4000 x 700 26.8 / 25.8 / 25.2, 12 x 32760 x 512 108.6 / 103.4 / 103.3. (Masked walks,
    // which differ in length, lose by it: causal 24 x 8 x 880 at 64 channels 183.5 / 187.5.)
    constexpr int kAhead = D == 64 && !MASKED ? 4 : 3, kMatrixPrio = MASKED ? 1 : 0, kSoftmaxPrio = 1 - kMatrixPrio;
    int kv = kv0_of(0), kk = kv0_of(1);   // first keys of the tiles that the next matrix part loads: V, K
    wait_vmcnt<0>();
    block_barrier();   // K(0), K(1) resident, every wave has its queries
    // The first two tiles have one offset, the largest score of their 128 keys: the one flash_fwd_pp2 gives them, and with
    // it the result's bits.
    {
        if (ne > 2) {
            const int k2 = kv0_of(2);
#pragma unroll
            for (int u = 0; u < kUnits; u++) load_k(2, k2, u);
        }
        ScoreTile s0, s1;
        auto hook_v0 = [&](int i) {
            if (i < kUnits) load_v(0, kv, i);
        };
        auto hook_v1 = [&](int i) {
            if (i < kUnits) load_v(1, kk, i);
        };
        __builtin_amdgcn_s_setprio(kMatrixPrio);
        mfma_phase<false, kAhead, D>(vbuf(0), kbuf(0), rb, pb, o, qf, s0, s_init, hook_v0);
        ProbTile pa;
        if (ne > 1) {
            mfma_phase<false, kAhead, D>(vbuf(0), kbuf(1), rb, pb, o, qf, s1, s_init, hook_v1);
            __builtin_amdgcn_s_setprio(kSoftmaxPrio);
            __builtin_amdgcn_sched_barrier(0);
            mask_tile(s0, 0);
            mask_tile(s1, 1);
            softmax_first_off<!LOG2DOM>(s0, s1, st, s_init, sl2, pa, pb);
        } else {
            __builtin_amdgcn_s_setprio(kSoftmaxPrio);
            __builtin_amdgcn_sched_barrier(0);
            mask_tile(s0, 0);
            softmax_first_off<!LOG2DOM>(s0, st, s_init, sl2, pa);
#pragma unroll
            for (int t = 0; t < 2; t++) pb[t][0] = pa[t][0], pb[t][1] = pa[t][1];
        }
        asm volatile("" ::"v"(pa[0][0]), "v"(pa[0][1]), "v"(pa[1][0]), "v"(pa[1][1]), "v"(pb[0][0]), "v"(pb[0][1]), "v"(pb[1][0]),
                     "v"(pb[1][1]), "v"(st.l_acc[0]), "v"(st.l_acc[1]));
        __builtin_amdgcn_sched_barrier(0);
        wait_vmcnt<0>();
        block_barrier();   // V(0), V(1), K(2) resident, K(0) and K(1) read by every wave
#pragma unroll
        for (int db = 0; db < kNO; db++)
#pragma unroll
            for (int g = 0; g < 2; g++) o[db][g] = f32x4{0.f, 0.f, 0.f, 0.f};
        __builtin_amdgcn_s_setprio(kMatrixPrio);
        pv_tile<D>(vbuf(0), rb.v, pa, o);
        kk = kv0_of(3);
        kv = kv0_of(2);
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll 1
    for (int m = 2; m < ne; m++) {
        ScoreTile s;
        auto hook_dma = [&](int i) {
            if (i < kUnits) load_v(m, kv, i);
            else if (i < 2 * kUnits) load_k(m + 1, kk, i - kUnits);
        };
        __builtin_amdgcn_s_setprio(kMatrixPrio);
        mfma_phase<true, kAhead, D>(vbuf(m - 1), kbuf(m), rb, pb, o, qf, s, s_init, hook_dma);
        __builtin_amdgcn_s_setprio(kSoftmaxPrio);
        __builtin_amdgcn_sched_barrier(0);
        mask_tile(s, m);
        if constexpr (FIXED) {
            softmax_off_tile<!LOG2DOM>(s, st, sl2, pb);
        } else {
            softmax_tile_off<!LOG2DOM>(s, st, o, s_init, sl2, pb);
        }
        asm volatile("" ::"v"(pb[0][0]), "v"(pb[0][1]), "v"(pb[1][0]), "v"(pb[1][1]), "v"(st.l_acc[0]), "v"(st.l_acc[1]));
        kv = kk;
        kk = kv0_of(m + 2);
        __builtin_amdgcn_sched_barrier(0);
        wait_vmcnt<0>();
        block_barrier();   // K(m+1), V(m) resident; this phase's tiles read by every wave
        __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_s_setprio(kMatrixPrio);
    if (ne > 1) pv_tile<D>(vbuf(ne - 1), rb.v, pb, o);
    __builtin_amdgcn_s_setprio(kSoftmaxPrio);

    if constexpr (FIXED) {   // did the fixed offset hold (flash_item)?
        float chk = 0.f;
#pragma unroll
        for (int db = 0; db < kNO; db++)
#pragma unroll
            for (int g = 0; g < 2; g++)
#pragma unroll
                for (int i = 0; i < 4; i++) chk = __builtin_fmaf(o[db][g][i], 0.f, chk);
        const bool lane_ok = quad_sum(st.l_acc[0]) < 0x1p+100f && quad_sum(st.l_acc[1]) < 0x1p+100f && chk == 0.f;
        // (in buffer 4: its last K is behind the last barrier, and a second pass loads it behind its first)
        auto* votes = (__attribute__((address_space(3))) unsigned*)(smem + 4 * kTileBytes);
        const bool wave_ok = __builtin_amdgcn_ballot_w64(!lane_ok) == 0;
        if (lane == 0) votes[wave] = wave_ok ? 0u : 1u;
        __builtin_amdgcn_s_waitcnt(0xC07F);
        block_barrier();
        const u32x4 v = *reinterpret_cast<const __attribute__((address_space(3))) u32x4*>(votes);
        if (__builtin_amdgcn_readfirstlane(v[0] | v[1] | v[2] | v[3]) != 0) {
            if (wave == 0 && lane == 0) atomicAdd(&g_exact_pass_reruns, 1ull);
            return false;
        }
    }
    float inv[2];
#pragma unroll
    for (int g = 0; g < 2; g++) {
        const float l_tot = quad_sum(st.l_acc[g]);
        inv[g] = l_tot > 0.f ? 1.f / l_tot : 0.f;
    }
    // (through buffers 0 and 1 behind the vote, else 1 and 4, which the last P V does not read: half of one a wave)
    store_rows16<D>((FIXED ? smem + (wave >> 1) * kTileBytes : kbuf(1 + (wave >> 1))) + (wave & 1) * (kTileBytes / 2), o,
                    inv, out, (size_t)bh * sq + q0 + wave * 32, qlen - wave * 32, lane);
    return true;
}
template <bool MASKED, int D, bool LOG2DOM>
__global__ __launch_bounds__(256, D == 64 ? 3 : 2) void flash_fwd_duo(const FlashParams p) {
    int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), block = blockIdx.x;
    if (duo_item<MASKED, D, LOG2DOM, true>(p, wave, threadIdx.x & 63, block)) return;
    ConstParams* again = params_again();   // (as in flash_fwd_pp2)
    int lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    asm volatile("" : "+v"(lane), "+s"(wave), "+s"(block));
    duo_item<MASKED, D, LOG2DOM, false>(*again, wave, lane, block);
}

// Merge of the split-KV partials: out[row] = sum_s w_s O_s / sum_s w_s with w_s = 2^(lse_s - max lse).
// One thread per (row, 4 d).
template <bool OUT16>
__global__ __launch_bounds__(256) void splitkv_merge_kernel(const float* __restrict__ part_o,
                                                            const float* __restrict__ part_lse, void* __restrict__ out,
                                                            size_t rows, int d, int splits) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    const int d4 = d >> 2;
    if (i >= rows * d4) return;
    const size_t row = i / d4;
    const int c = (int)(i - row * d4) * 4;
    float m = neg_inf();
    bool nan = false;   // (a split whose sum is NaN: max drops it)
    for (int s = 0; s < splits; s++) {
        const float lse = part_lse[(size_t)s * rows + row];
        m = __builtin_fmaxf(m, lse);
        nan |= lse != lse;
    }
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    float wsum = 0.f;
    if (m != neg_inf() || nan) {
        for (int s = 0; s < splits; s++) {
            const float w = fast_exp2(part_lse[(size_t)s * rows + row] - m);
            const f32x4 o = *reinterpret_cast<const f32x4*>(part_o + ((size_t)s * rows + row) * d + c);
            wsum += w;
#pragma unroll
            for (int x = 0; x < 4; x++) acc[x] += w * o[x];
        }
    }
    const float inv = wsum == 0.f ? 0.f : 1.f / wsum;
#pragma unroll
    for (int x = 0; x < 4; x++) acc[x] *= inv;
    if constexpr (OUT16) {
        *reinterpret_cast<bf16x4*>((uint16_t*)out + row * d + c) = __builtin_convertvector(acc, bf16x4);
    } else {
        *reinterpret_cast<f32x4*>((float*)out + row * d + c) = acc;
    }
}

}  // namespace fv

extern "C" hipError_t fv_internal_launch_splitkv_merge(const float* part_o, const float* part_lse, void* out,
                                                       int out_is_bf16, size_t rows, int d, int splits,
                                                       hipStream_t st) {
    const size_t n = rows * (size_t)(d / 4), blocks = (n + 255) / 256;
    if (blocks == 0) return hipSuccess;
    if (out_is_bf16)
        hipLaunchKernelGGL(fv::splitkv_merge_kernel<true>, dim3((unsigned)blocks), dim3(256), 0, st, part_o, part_lse,
                           out, rows, d, splits);
    else
        hipLaunchKernelGGL(fv::splitkv_merge_kernel<false>, dim3((unsigned)blocks), dim3(256), 0, st, part_o, part_lse,
                           out, rows, d, splits);
    return hipGetLastError();
}

// ---- host launchers -------------------------------------------------------------

// (a kernel, not a memset: a caller may capture it into a graph)
static __global__ void clear_queue_kernel(int* queue) { queue[threadIdx.x] = 0; }
extern "C" hipError_t fv_internal_clear_queue(int* queue, hipStream_t stream) {
    static_assert(8 * fv::kQueueStep * sizeof(int) == kFvQueueBytes, "a counter an XCD");
    hipLaunchKernelGGL(clear_queue_kernel, dim3(1), dim3(8 * fv::kQueueStep), 0, stream, queue);
    return hipGetLastError();
}

extern "C" int fv_internal_flash_block_m(void) { return fv::kPpBM; }

// FASTVIDEO_SDPA_RUNNING_MAX=1: every launch keeps the running max (no fixed-offset first pass).
extern "C" int fv_internal_fixed_offset(int out_is_bf16) {
    static const bool forced = [] {
        const char* e = getenv("FASTVIDEO_SDPA_RUNNING_MAX");
        return e && *e && strcmp(e, "0") != 0;
    }();
    return out_is_bf16 && !forced;
}

namespace {
template <bool MASKED, int D>
constexpr int flash_lds = 2 * fv::kRing2 * fv::TileGeo<D>::kTile + fv::kVoteBytes + (MASKED ? fv::kPpBM * (int)sizeof(fv::LaneMask) : 0);
// The kernel's dynamic LDS limit (128 KB at D = 128), once per device.
template <int NG, bool MASKED, int D, bool LOG2DOM, bool FIXED, bool FAR>
hipError_t flash_attr() {
    static std::atomic<unsigned long long> attr_done;
    constexpr int lds = flash_lds<MASKED, D>;
    return fv_set_max_lds_once((const void*)fv::flash_fwd_pp2<NG, MASKED, D, LOG2DOM, FIXED, FAR>, lds, attr_done);
}
template <int NG, bool MASKED, int D, bool LOG2DOM, bool FIXED, bool FAR>
hipError_t launch_flash_as(const fv::FlashParams* p, hipStream_t stream) {
    constexpr int lds = flash_lds<MASKED, D>;
    hipError_t e = flash_attr<NG, MASKED, D, LOG2DOM, FIXED, FAR>();
    if (e != hipSuccess) return e;
    const int grid = p->full + (p->queue ? p->per_xcd + p->per_xcd / 8 : p->per_xcd) * 8;
    hipLaunchKernelGGL((fv::flash_fwd_pp2<NG, MASKED, D, LOG2DOM, FIXED, FAR>), dim3(grid), dim3(256 * NG), lds, stream, *p);
    return hipGetLastError();
}
template <bool MASKED, int D, bool LOG2DOM>
hipError_t duo_attr() {
    static std::atomic<unsigned long long> attr_done;
    return fv_set_max_lds_once((const void*)fv::flash_fwd_duo<MASKED, D, LOG2DOM>, fv::kDuoLds<D>, attr_done);
}
template <bool MASKED, int D, bool LOG2DOM>
hipError_t launch_duo_as(const fv::FlashParams* p, hipStream_t stream) {
    hipError_t e = duo_attr<MASKED, D, LOG2DOM>();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((fv::flash_fwd_duo<MASKED, D, LOG2DOM>), dim3(p->per_xcd * 8), dim3(256), fv::kDuoLds<D>, stream, *p);
    return hipGetLastError();
}
// A call whose scale * log2(e) is exactly 1 (scale = ln 2: the caller folded the softmax scale into Q) runs
// the form without the per-score multiply.
std::atomic<unsigned long long> g_log2_domain_launches{0};
template <int NG, bool MASKED, int D, bool FIXED, bool FAR>
hipError_t launch_flash_fixed(const fv::FlashParams* p, hipStream_t stream) {
    if (p->sl2 != 1.0f) return launch_flash_as<NG, MASKED, D, false, FIXED, FAR>(p, stream);
    g_log2_domain_launches.fetch_add(1, std::memory_order_relaxed);
    return launch_flash_as<NG, MASKED, D, true, FIXED, FAR>(p, stream);
}
// Launches whose result is rounded to bf16 make their first pass with the fixed offset: on a row that one late
// key dominates, that key's P is then a rounded bf16 number instead of exactly 1 (up to 2^-8 relative on the row),
// which a bf16 result absorbs; f32 results keep the running max. Masked launches take it where every query sees
// key 0, the first key of every tile's walk, so that its offset is a score of its own: block-causal without a
// window or with sink blocks, and the VDN mask (rows before the video and frame 0 are visible to every query).
// Under a window without a sink a query's first visible key may lie anywhere in the walk: running max.
template <bool MASKED>
bool takes_fixed_offset(const fv::FlashParams* p) {
    const bool offset_is_a_score = !MASKED || p->mask_mode == 2 || (p->mask_mode == 1 && (p->win == 0 || p->sink > 0));
    return fv_internal_fixed_offset(p->out_is_bf16) && offset_is_a_score;
}
template <int NG, bool MASKED, int D, bool FAR>
hipError_t launch_flash_planes(const fv::FlashParams* p, hipStream_t stream) {
    return takes_fixed_offset<MASKED>(p) ? launch_flash_fixed<NG, MASKED, D, true, FAR>(p, stream)
                                         : launch_flash_fixed<NG, MASKED, D, false, FAR>(p, stream);
}
template <int NG, bool MASKED, int D>
hipError_t launch_flash(const fv::FlashParams* p, hipStream_t stream) {
    return fv::plane_fits<D>(p->sk) ? launch_flash_planes<NG, MASKED, D, false>(p, stream)
                                    : launch_flash_planes<NG, MASKED, D, true>(p, stream);
}
template <bool MASKED, int D>
hipError_t launch_duo(const fv::FlashParams* p, hipStream_t stream) {
    if (!takes_fixed_offset<MASKED>(p)) return hipErrorInvalidValue;
    if (p->sl2 != 1.0f) return launch_duo_as<MASKED, D, false>(p, stream);
    g_log2_domain_launches.fetch_add(1, std::memory_order_relaxed);
    return launch_duo_as<MASKED, D, true>(p, stream);
}
template <bool MASKED, int D>
hipError_t init_duo() {
    const hipError_t e = duo_attr<MASKED, D, false>();
    return e == hipSuccess ? duo_attr<MASKED, D, true>() : e;
}
template <int NG, bool MASKED, int D, bool FAR>
hipError_t init_flash_planes() {
    hipError_t e = flash_attr<NG, MASKED, D, false, false, FAR>();
    if (e == hipSuccess) e = flash_attr<NG, MASKED, D, true, false, FAR>();
    if (e == hipSuccess) e = flash_attr<NG, MASKED, D, false, true, FAR>();
    if (e == hipSuccess) e = flash_attr<NG, MASKED, D, true, true, FAR>();
    return e;
}
template <int NG, bool MASKED, int D>
hipError_t init_flash() {
    const hipError_t e = init_flash_planes<NG, MASKED, D, false>();
    return e == hipSuccess ? init_flash_planes<NG, MASKED, D, true>() : e;
}
}  // namespace

extern "C" void fv_internal_count_log2_domain(void) { g_log2_domain_launches.fetch_add(1, std::memory_order_relaxed); }
extern "C" uint64_t fv_sdpa_log2_domain_launches(void) { return g_log2_domain_launches.load(std::memory_order_relaxed); }

extern "C" hipError_t fv_internal_exact_pass_reruns(unsigned long long* out) {
    return hipMemcpyFromSymbol(out, HIP_SYMBOL(fv::g_exact_pass_reruns), sizeof *out, 0, hipMemcpyDeviceToHost);
}

extern "C" hipError_t fv_internal_init_flash(void) {
    hipError_t e = init_flash<2, false, 128>();
    if (e == hipSuccess) e = init_flash<2, true, 128>();
    if (e == hipSuccess) e = init_flash<2, false, 64>();
    if (e == hipSuccess) e = init_flash<2, true, 64>();
    if (e == hipSuccess) e = init_flash<1, false, 128>();
    if (e == hipSuccess) e = init_flash<1, false, 64>();
    if (e == hipSuccess) e = init_duo<false, 128>();
    if (e == hipSuccess) e = init_duo<false, 64>();
    if (e == hipSuccess) e = init_duo<true, 128>();
    if (e == hipSuccess) e = init_duo<true, 64>();
    return e;
}

extern "C" hipError_t fv_internal_launch_duo(const fv::FlashParams* p, int masked, int d, hipStream_t stream) {
    if (d == 128) return masked ? launch_duo<true, 128>(p, stream) : launch_duo<false, 128>(p, stream);
    if (d == 64) return masked ? launch_duo<true, 64>(p, stream) : launch_duo<false, 64>(p, stream);
    return hipErrorInvalidValue;
}

extern "C" hipError_t fv_internal_launch_flash(const fv::FlashParams* p, int masked, int d, int block_m,
                                               hipStream_t stream) {
    const bool half = block_m == fv::kPpBM / 2;
    if ((block_m != fv::kPpBM && !half) || (half && masked)) return hipErrorInvalidValue;
    if (d == 128)
        return masked ? launch_flash<2, true, 128>(p, stream)
                      : half ? launch_flash<1, false, 128>(p, stream) : launch_flash<2, false, 128>(p, stream);
    if (d == 64)
        return masked ? launch_flash<2, true, 64>(p, stream)
                      : half ? launch_flash<1, false, 64>(p, stream) : launch_flash<2, false, 64>(p, stream);
    return hipErrorInvalidValue;
}
