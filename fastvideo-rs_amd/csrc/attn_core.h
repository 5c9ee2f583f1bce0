// Building blocks shared by the gfx950 attention kernels that stage K/V tiles
// with direct global->LDS loads into XOR-swizzled,
// unpadded [64 keys][128 d] bf16 tiles.
//
// LDS tile layout (16 KB): row r is 256 B = 16 chunks of 16 B; logical chunk c
// of row r lives at chunk position c ^ swz(r), with
//   K tiles: swz(r) = r & 15        (32 consecutive keys reading one chunk
//                                    column hit 16 distinct positions)
//   V tiles: swz(r) = (r & 7) << 1  (8 rows of a transposed 4x16 read, two blocks of
//                                    16 lanes, land in 8 disjoint 32 B bank groups)
// The LDS-DMA write puts lane i's 16 B at base + 16 i, so the swizzle is applied
// on the global side: lane i fetches the chunk that belongs at its position.
#pragma once
#include "fv_common.h"
#include <type_traits>

namespace fv {

constexpr int kTileRows = 64;
constexpr int kRowBytes = 256;
constexpr int kTileBytes = kTileRows * kRowBytes;   // 16 KB (head dim 128)

// Tile geometry by head dim D (128 or 64): rows of 2 D bytes, 16-byte chunks, and the XOR
// swizzles that make the operand reads bank-conflict free.
//   D = 128 (256 B rows, 16 chunks): K chunk ^ (row & 15); V chunk ^ ((row & 7) << 1).
//   D = 64  (128 B rows,  8 chunks): two rows share a 256 B bank line, so both swizzles
//     advance every second row: K chunk ^ ((row >> 1) & 7), V chunk ^ (((row >> 1) & 3) << 1).
// (vswz32: of the kernels whose V^T operands are 32 channels wide.)
template <int D>
struct TileGeo {
    static_assert(D == 128 || D == 64, "head dim 128 or 64");
    static constexpr int kRow = 2 * D;                   // bytes per row
    static constexpr int kTile = kTileRows * kRow;       // bytes per tile
    static constexpr int kChunks = kRow / 16;            // 16-byte chunks per row
    static constexpr int kRowsPerDma = 1024 / kRow;      // rows one wave-wide DMA instruction covers
    static constexpr int kDmaPerTile = kTile / 1024;
    static constexpr int kVGroups = D / 16;              // PV groups per tile (two operand fragments, 4 MFMAs each)
    static constexpr int kKGroups = D / 16;              // QK groups per tile (the same)
    static constexpr int kGroups = kVGroups + kKGroups;
    static FV_DEV int kswz(int r) { return D == 128 ? (r & 15) : ((r >> 1) & 7); }
    static FV_DEV int vswz(int r) { return D == 128 ? ((r & 7) << 1) : (((r >> 1) & 3) << 1); }
    static FV_DEV int vswz32(int r) { return D == 128 ? ((r & 3) << 2) : (((r >> 1) & 1) << 2); }
};

typedef __attribute__((address_space(1))) void glb_void;
typedef __attribute__((address_space(3))) void lds_void;

// LDS-DMA: one wave-wide `global_load_lds_dwordx4` copies, per lane i, 16 B from the lane's global
// address to LDS byte address lds_base + 16 i (lds_base wave-uniform, in m0). It is issued as inline
// asm so that the compiler's wait-count insertion does not serialise later LDS reads of OTHER buffers
// behind it; the kernels order these loads with wait_vmcnt<N>() + block_barrier() themselves.

// Workgroup barrier without the memory fences of __syncthreads() (a fence
// would wait for every outstanding LDS-DMA load, defeating the prefetch). LDS
// reads issued before it have been consumed by then (their MFMA waited on them).
FV_DEV void block_barrier() { asm volatile("s_barrier" ::: "memory"); }

// s_waitcnt vmcnt(N) alone (expcnt / lgkmcnt untouched), gfx9 encoding.
template <int N>
FV_DEV void wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// LDS-DMA with a wave-uniform 64-bit base (SGPR pair) + per-lane byte offset.
FV_DEV void lds_dma16_s(unsigned lds_base, const void* sbase_in, unsigned voff) {
    // pin the base to an SGPR pair even where the compiler's divergence analysis
    // (branches on the wave index) would otherwise place it in VGPRs
    const unsigned long long a = (unsigned long long)sbase_in;
    // (readfirstlane returns int: widen through unsigned, or a low half with bit 31 set
    // would sign-extend over the high half)
    const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)a);
    const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(a >> 32));
    const unsigned long long sbase = ((unsigned long long)hi << 32) | (unsigned long long)lo;
    asm volatile(
        "s_mov_b32 m0, %0\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %1, %2"
        :
        : "s"(lds_base), "v"(voff), "s"(sbase)
        : "memory");   // m0 is a reserved scratch register: the compiler sets it right before each of
                       // its own uses and keeps nothing live in it across statements
}

// The first `rows` rows of one plane of K or V as a buffer descriptor: lanes that read past them (the rows of a last
// tile past the keys) get zeros from the hardware's range check, in LDS as well, so a tile load needs no clamp. Bytes and
// offsets are 32 bits: plane_fits() says which planes that holds. (Before, a phase clamped its lanes' offsets to the last
// row: 8 registers, four branches and 60 scalar instructions.)
FV_DEV u32x4 plane_descriptor(const void* base, unsigned bytes) {
    const unsigned long long a = (unsigned long long)base;
    u32x4 r;
    r[0] = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)a);
    r[1] = (unsigned)__builtin_amdgcn_readfirstlane((int)((unsigned)(a >> 32) & 0xffffu));   // (stride 0: raw)
    r[2] = (unsigned)__builtin_amdgcn_readfirstlane((int)bytes);
    r[3] = 0x00020000u;   // 32-bit data
    return r;
}
template <int D>
__host__ __device__ constexpr bool plane_fits(long rows) { return rows <= 0xffffffffl / (2 * D); }

// Per-lane source offsets of the tile loads, computed once per kernel: a wave-wide
// DMA instruction moves 1 KB = 4 rows of 256 B (D = 128) or 8 rows of 128 B (D = 64);
// with NW waves sharing a 64-row tile a wave issues ITER = (tile KB) / NW of them, two (one where ITER is 1) to a unit;
// lane i fetches the 16 B chunk that belongs at its position of its row.
template <int NW, int D = 128>
struct TileDma {
    using G = TileGeo<D>;
    static constexpr int ITER = G::kDmaPerTile / NW;
    static constexpr int kUnits = ITER > 1 ? ITER / 2 : 1;   // units a tile
    static_assert(ITER >= 1 && (ITER == 1 || ITER % 2 == 0), "one load or pairs of them");
    // byte offset from the tile's first row, K or V swizzle; of a unit's second load less the 1 KB that its immediate
    // offset adds (to the LDS address as well: m0 is written once a unit)
    unsigned koff[ITER], voff[ITER];
    unsigned slot;           // wave-uniform: the wave's part of a tile's LDS bytes
    FV_DEV void init(int wave, int lane) {
        const int p = lane % G::kChunks;
#pragma unroll
        for (int it = 0; it < ITER; it++) {
            const int r = (wave * ITER + it) * G::kRowsPerDma + lane / G::kChunks;
            koff[it] = r * G::kRow + ((p ^ G::kswz(r)) << 4) - (it & 1) * 1024;
            voff[it] = r * G::kRow + ((p ^ G::vswz(r)) << 4) - (it & 1) * 1024;
        }
        slot = (unsigned)__builtin_amdgcn_readfirstlane(wave * ITER * 1024);
    }
    // Unit u of the tile whose first row lies `at` bytes into the plane (wave-uniform, within it), into the tile buffer at
    // LDS byte address `lds` + the wave's slot.
    template <bool IS_V>
    FV_DEV void issue(const u32x4& plane, unsigned at, unsigned lds, int u) const {
        at = (unsigned)__builtin_amdgcn_readfirstlane((int)at);   // (free where the compiler knows it to be uniform)
        const unsigned m0 = (unsigned)__builtin_amdgcn_readfirstlane((int)(lds + slot + u * 2048));
        const unsigned o0 = IS_V ? voff[2 * u] : koff[2 * u];
        if constexpr (ITER == 1) {
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                         :: "s"(m0), "v"(o0), "s"(plane), "s"(at) : "memory");
        } else {
            const unsigned o1 = IS_V ? voff[2 * u + 1] : koff[2 * u + 1];
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %3, %4 offen lds\n\t"
                         "buffer_load_dwordx4 %2, %3, %4 offen offset:1024 lds"
                         :: "s"(m0), "v"(o0), "v"(o1), "s"(plane), "s"(at) : "memory");
        }
    }
};

// Per-lane read bases into a swizzled tile.
struct TileReadBases {
    int k;   // K A-operand (16 keys x 32 d): ^ (dk << 6), + kb * 16 rows
    int v;   // V^T A-operand (16 d x 32 keys, two transposed reads): ^ (db << 5), + 32 t rows, + 16 for the second
};
template <int D = 128>
FV_DEV TileReadBases tile_read_bases(int lane) {
    using G = TileGeo<D>;
    const int q4 = lane >> 4, i16 = lane & 15;
    TileReadBases b;
    // K: lane reads logical chunk 4 dk + q4 of row i16 (+ 16 kb)
    b.k = i16 * G::kRow + ((G::kswz(i16) ^ q4) << 4);
    // V^T: lane reads 8 bytes at d = 16 db + 4 (i16 & 3) of row 4 q4 + i16 / 4 (+ 32 t, + 16)
    const int r = 4 * q4 + (i16 >> 2);
    b.v = r * G::kRow + ((G::vswz(r) ^ ((i16 & 3) >> 1)) << 4) + 8 * (i16 & 1);
    return b;
}
// The same for operands of 32 rows: K ^ (dk << 5), + kb * 32 rows; V^T ^ (db << 6), + (16 t + 8 g) rows (vswz32).
template <int D = 128>
FV_DEV TileReadBases tile_read_bases32(int lane) {
    using G = TileGeo<D>;
    const int h = lane >> 5, c32 = lane & 31;
    const int b16 = lane >> 4, i16 = lane & 15;
    TileReadBases b;
    // K: lane reads logical chunk 2 dk + h of row c32 (+32): physical (2 dk + h) ^ kswz(row)
    b.k = c32 * G::kRow + ((G::kswz(c32) ^ h) << 4);
    // V^T: lane reads 8 bytes at d = 32 db + 16 (b16 & 1) + 4 (i16 & 3) of row 4 h + i16/4 (+16 t, +8)
    const int r = 4 * h + (i16 >> 2);
    const int c_lane = 2 * (b16 & 1) + ((i16 & 3) >> 1);
    b.v = r * G::kRow + ((G::vswz32(r) ^ c_lane) << 4) + 8 * (i16 & 1);
    return b;
}

constexpr float kRescaleLog2 = 6.0f;

// Scores of a 64-key tile against the wave's 32 queries, S^T in blocks of 16 keys x 16 queries: [kb][g], a lane holds
// keys 16 kb + 4 (lane / 16) + i of query 16 g + lane % 16. P of the tile is [t][g], the B operand of 32 keys x 16 queries:
// a lane's eight keys are its four of blocks 2 t and 2 t + 1 (the V^T operand is read in that order).
typedef f32x4 ScoreTile[4][2];
typedef bf16x8 ProbTile[2][2];

// Online softmax in base 2 with the offset riding in the matrix pipe. The K Q^T MFMAs of every S block start from
// `negoff` (4 copies of minus the lane's offset, in raw score units) as their C operand, so the scores arrive as
// x = s - off and P = 2^(sl2 * x): one two-operand multiply and one v_exp_f32 per score, no three-operand
// multiply-add (measured on MI355X against P = exp2(fma(s, sl2, -m * sl2)): same cycles, 1.7 % less time on the
// long dense launches and 2.3 % on block-causal ones, which run at the chip's power limit). SCALED == false is
// the form for calls whose sl2 = scale * log2(e) is exactly 1 (the caller folded the softmax scale into Q, e.g.
// into the q RMSNorm output): the multiply is gone as well.
// State per lane, for each of its two queries (lanes l, l ^ 16, l ^ 32 and l ^ 48 hold the same ones): `off` the offset,
// `r` the running max relative to it (-inf until the query has seen a finite score), `l_acc` the lane's share of the row
// sum. When sl2 * r exceeds kRescaleLog2 in some lane (or a query sees its first finite score) every lane moves its
// offsets to its running maxima: l and O are scaled by 2^(-sl2 r), this phase's scores lose r, negoff is rewritten
// (wave-uniform branch, rare). The final O / l is exact for any such policy: P and l always share an offset.
struct SoftmaxOffState {
    float r[2], off[2], l_acc[2];
    FV_DEV void init() {
#pragma unroll
        for (int g = 0; g < 2; g++) r[g] = neg_inf(), off[g] = 0.f, l_acc[g] = 0.f;
    }
    // base-2 logarithm of the row sum's scale: sum_k 2^(sl2 s_k) = l * 2^(sl2 off)
    template <bool SCALED>
    FV_DEV float log2_offset(int g, float sl2) const { return SCALED ? off[g] * sl2 : off[g]; }
};

// The largest of query g's scores over NS tiles, in every lane that holds the query.
template <int NS>
FV_DEV float score_max(const ScoreTile* const (&sc)[NS], int g) {
    float mx = (*sc[0])[0][g][0];
#pragma unroll
    for (int b = 0; b < NS; b++)
#pragma unroll
        for (int kb = 0; kb < 4; kb++)
#pragma unroll
            for (int i = 0; i < 4; i++) mx = __builtin_fmaxf(mx, (*sc[b])[kb][g][i]);
    return quad_max(mx);
}

// The rescale decision and its (rare) execution for NS tiles: updates st, o, the scores and negoff.
template <bool SCALED, int NO, int NS>
FV_DEV void softmax_off_rescale(SoftmaxOffState& st, f32x4 (&o)[NO][2], f32x4 (&negoff)[2], float sl2,
                                ScoreTile* const (&sc)[NS]) {
    const float NEG = neg_inf();
    const ScoreTile* csc[NS];
#pragma unroll
    for (int b = 0; b < NS; b++) csc[b] = sc[b];
    float r_new[2];
    bool need = false;
#pragma unroll
    for (int g = 0; g < 2; g++) {
        r_new[g] = __builtin_fmaxf(st.r[g], score_max<NS>(csc, g));
        need |= ((SCALED ? r_new[g] * sl2 : r_new[g]) > kRescaleLog2) || (st.r[g] == NEG && r_new[g] != NEG);
    }
    if (__builtin_amdgcn_ballot_w64(need) != 0) {
#pragma unroll
        for (int g = 0; g < 2; g++) {
            const float delta = (r_new[g] == NEG) ? 0.f : r_new[g];
            const float alpha = (st.r[g] == NEG) ? 0.f : fast_exp2(SCALED ? -delta * sl2 : -delta);
            st.l_acc[g] *= alpha;
#pragma unroll
            for (int db = 0; db < NO; db++)
#pragma unroll
                for (int i = 0; i < 4; i++) o[db][g][i] *= alpha;
#pragma unroll
            for (int b = 0; b < NS; b++)
#pragma unroll
                for (int kb = 0; kb < 4; kb++)
#pragma unroll
                    for (int i = 0; i < 4; i++) (*sc[b])[kb][g][i] -= delta;   // -inf stays -inf
            st.off[g] += delta;
#pragma unroll
            for (int i = 0; i < 4; i++) negoff[g][i] = -st.off[g];
            st.r[g] = (r_new[g] == NEG) ? NEG : 0.f;
        }
    } else {
        st.r[0] = r_new[0];
        st.r[1] = r_new[1];
    }
}

// A tile of scores (relative to the offset) to P: exponentials, row-sum shares, bf16 pack (RNE).
template <bool SCALED>
FV_DEV void softmax_off_tile(const ScoreTile& s, SoftmaxOffState& st, float sl2, ProbTile& pb) {
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int g = 0; g < 2; g++) {
            f32x8 e;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float x = s[2 * t + (i >> 2)][g][i & 3];
                e[i] = fast_exp2(SCALED ? x * sl2 : x);
                st.l_acc[g] += e[i];
            }
            pb[t][g] = __builtin_convertvector(e, bf16x8);
        }
}

// A pair of tiles (128 keys) with one shared max / rescale decision.
template <bool SCALED, int NO>
FV_DEV void softmax_tile_pair_off(ScoreTile& s0, ScoreTile& s1, SoftmaxOffState& st, f32x4 (&o)[NO][2],
                                  f32x4 (&negoff)[2], float sl2, ProbTile& pb0, ProbTile& pb1) {
    ScoreTile* const sc[2] = {&s0, &s1};
    softmax_off_rescale<SCALED, NO, 2>(st, o, negoff, sl2, sc);
    softmax_off_tile<SCALED>(s0, st, sl2, pb0);
    softmax_off_tile<SCALED>(s1, st, sl2, pb1);
}

// A pair of tiles with the offset left where it is: no row max, no rescale decision. For walks whose caller
// checks afterwards that no row sum outgrew the f32 range comfortably (and redoes the walk with
// softmax_tile_pair_off if one did).
template <bool SCALED>
FV_DEV void softmax_tile_pair_fixed(const ScoreTile& s0, const ScoreTile& s1, SoftmaxOffState& st, float sl2,
                                    ProbTile& pb0, ProbTile& pb1) {
    softmax_off_tile<SCALED>(s0, st, sl2, pb0);
    softmax_off_tile<SCALED>(s1, st, sl2, pb1);
}

// The first pair of a walk (or its only tile), before anything has been added up: the same offset and the same P.
template <int NS>
FV_DEV void softmax_first_offset(ScoreTile* const (&sc)[NS], SoftmaxOffState& st, f32x4 (&negoff)[2]) {
    const float NEG = neg_inf();
    const ScoreTile* csc[NS];
#pragma unroll
    for (int b = 0; b < NS; b++) csc[b] = sc[b];
#pragma unroll
    for (int g = 0; g < 2; g++) {
        const float r = __builtin_fmaxf(NEG, score_max<NS>(csc, g));   // (a NaN: as no score)
        st.off[g] = r == NEG ? 0.f : r;
        st.r[g] = r == NEG ? NEG : 0.f;
        st.l_acc[g] = 0.f;
#pragma unroll
        for (int b = 0; b < NS; b++)
#pragma unroll
            for (int kb = 0; kb < 4; kb++)
#pragma unroll
                for (int i = 0; i < 4; i++) (*sc[b])[kb][g][i] -= st.off[g];
#pragma unroll
        for (int i = 0; i < 4; i++) negoff[g][i] = -st.off[g];
    }
}
template <bool SCALED>
FV_DEV void softmax_first_off(ScoreTile& s0, ScoreTile& s1, SoftmaxOffState& st, f32x4 (&negoff)[2], float sl2,
                              ProbTile& pb0, ProbTile& pb1) {
    ScoreTile* const sc[2] = {&s0, &s1};
    softmax_first_offset<2>(sc, st, negoff);
    softmax_tile_pair_fixed<SCALED>(s0, s1, st, sl2, pb0, pb1);
}
template <bool SCALED>
FV_DEV void softmax_first_off(ScoreTile& s, SoftmaxOffState& st, f32x4 (&negoff)[2], float sl2, ProbTile& pb) {
    ScoreTile* const sc[1] = {&s};
    softmax_first_offset<1>(sc, st, negoff);
    softmax_off_tile<SCALED>(s, st, sl2, pb);
}

// One tile.
template <bool SCALED, int NO>
FV_DEV void softmax_tile_off(ScoreTile& s, SoftmaxOffState& st, f32x4 (&o)[NO][2], f32x4 (&negoff)[2], float sl2,
                             ProbTile& pb) {
    ScoreTile* const sc[1] = {&s};
    softmax_off_rescale<SCALED, NO, 1>(st, o, negoff, sl2, sc);
    softmax_off_tile<SCALED>(s, st, sl2, pb);
}

// The V^T operand of 16 channels x 32 keys at `a0` of a tile.
template <int D>
FV_DEV bf16x8 read_v_frag(const lds_u8* a0) {
    s16x8 a;
    a.lo = lds_read_tr16_b64(a0);
    a.hi = lds_read_tr16_b64(a0 + 16 * TileGeo<D>::kRow);
    return __builtin_bit_cast(bf16x8, a);
}

// O^T (D d x 32 queries) += V^T P^T.
template <int D = 128>
FV_DEV void pv_tile(const lds_u8* vb, int v_base, const ProbTile& pb, f32x4 (&o)[D / 16][2]) {
    constexpr int kRow = TileGeo<D>::kRow;
#pragma unroll
    for (int t = 0; t < 2; t++) {
#pragma unroll
        for (int db = 0; db < D / 16; db++) {
            const bf16x8 a = read_v_frag<D>(vb + (v_base ^ (db << 5)) + 32 * t * kRow);
#pragma unroll
            for (int g = 0; g < 2; g++) o[db][g] = mfma16(a, pb[t][g], o[db][g]);
        }
    }
}

// One MFMA phase over NT key tiles with a deep, explicit LDS prefetch: for each of them O^T += V^T P^T of the
// tile NT before it (if DO_PV), then S^T = K Q^T. A group is 2 operand fragments (8 VGPRs), each feeding the MFMAs of both
// query blocks; the first K MFMAs of a key block take `s_init` as their C operand (zeros, or minus the
// softmax offset of the lane's queries). kAhead (3, or 4 where the registers allow it) groups are always in flight ahead of the group
// being multiplied, so an MFMA waits on a read issued kAhead x 64 cycles of
// matrix-pipe time earlier instead of on LDS latency plus the 64 B/clk per-SIMD
// LDS return path. sched_barrier keeps the compiler from re-serialising reads
// behind MFMAs.
// The operand fragments are addressed through per-lane LDS pointers that already hold the buffer's place
// (`va[db]`: V^T fragments of d block db, `ka[dk]`: K fragments of d chunk dk, both for the FIRST tile; the others follow it
// and are immediates of the reads), so a read costs no address arithmetic.
template <bool DO_PV, int kAhead, int NT, int D, class Hook>
FV_DEV void mfma_phase(const lds_u8* const (&va)[D / 16], const lds_u8* const (&ka)[D / 32],
                       const ProbTile* const (&pb)[NT], f32x4 (&o)[D / 16][2], const bf16x8 (&qf)[D / 32][2],
                       ScoreTile* const (&s)[NT], const f32x4 (&s_init)[2], Hook&& hook) {
    using G = TileGeo<D>;
    constexpr int NV = G::kVGroups, kPer = DO_PV ? G::kGroups : G::kKGroups, kAll = NT * kPer;
    constexpr int kPerT = D / 32;   // V groups per 32-key group t (each covers two 16-wide d blocks)
    bf16x8 f[kAll][2];
    auto issue = [&](int i, int x) {
        const int t = i / kPer, n = i % kPer + (DO_PV ? 0 : NV);
        if (n < NV)           // V^T fragments: key group n / kPerT, d blocks 2*(n % kPerT) + {0, 1}
            f[i][x] = read_v_frag<D>(va[2 * (n % kPerT) + x] + (32 * (n / kPerT) * G::kRow + t * G::kTile));
        else                  // K fragments: d chunk dk = (n - NV) / 2, key blocks 2 * ((n - NV) % 2) + {0, 1}
            f[i][x] = lds_read_b128(ka[(n - NV) / 2] + ((2 * ((n - NV) & 1) + x) * 16 * G::kRow + t * G::kTile));
    };
    auto run = [&](int i, int x, int g) {
        const int t = i / kPer, n = i % kPer + (DO_PV ? 0 : NV);
        if (n < NV) {
            f32x4& acc = o[2 * (n % kPerT) + x][g];
            acc = mfma16(f[i][x], (*pb[t])[n / kPerT][g], acc);
        } else {   // S is born at dk == 0, not before the PV part, from the C operand s_init
            const int dk = (n - NV) / 2;
            f32x4& acc = (*s[t])[2 * ((n - NV) & 1) + x][g];
            acc = mfma16(f[i][x], qf[dk][g], dk == 0 ? s_init[g] : acc);
        }
    };
#pragma unroll
    for (int i = 0; i < kAhead && i < kAll; i++) issue(i, 0), issue(i, 1);
#pragma unroll
    for (int i = 0; i < kAll; i++) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            __builtin_amdgcn_sched_barrier(0);
            run(i, j >> 1, j & 1);
            __builtin_amdgcn_sched_barrier(0);
            // A wave issues in order and an instruction takes it four cycles: after an MFMA of 16 cycles there is room
            // for three others before the next one is due, so the reads and the side work are dealt out over the gaps.
            if (j < 2 && i + kAhead < kAll) issue(i + kAhead, j);
            if (j == 2) hook(i);   // side work (tile DMA issue) that rides under the matrix pipe
        }
    }
}

// mfma_phase for one tile given by its V and K buffers (wave-uniform) and the lane's read bases: the fragment
// addresses are formed here, an add per fragment.
template <bool DO_PV, int kAhead, int D, class Hook>
FV_DEV void mfma_phase(const lds_u8* vb, const lds_u8* kb, const TileReadBases& rb,
                       const ProbTile& pb, f32x4 (&o)[D / 16][2], const bf16x8 (&qf)[D / 32][2],
                       ScoreTile& s, const f32x4 (&s_init)[2], Hook&& hook) {
    const lds_u8* va[D / 16];
    const lds_u8* ka[D / 32];
#pragma unroll
    for (int db = 0; db < D / 16; db++) va[db] = vb + (rb.v ^ (db << 5));
#pragma unroll
    for (int dk = 0; dk < D / 32; dk++) ka[dk] = kb + (rb.k ^ (dk << 6));
    const ProbTile* const pbs[1] = {&pb};
    ScoreTile* const ss[1] = {&s};
    mfma_phase<DO_PV, kAhead, 1, D>(va, ka, pbs, o, qf, ss, s_init, static_cast<Hook&&>(hook));
}

// Q^T fragments for the wave's 32 queries: rows row0 + lane%32 of a row-major
// [rows][128] bf16 tensor; rows >= nrows read as zero.
template <int D = 128>
FV_DEV void load_q_frags(const uint16_t* q, int row, bool ok, int lane, bf16x8 (&qf)[D / 16]) {
    const uint16_t* src = q + (size_t)row * D + 8 * (lane >> 5);
#pragma unroll
    for (int dk = 0; dk < D / 16; dk++) {
        u32x4 t = {0u, 0u, 0u, 0u};
        if (ok) t = *reinterpret_cast<const u32x4*>(src + 16 * dk);
        qf[dk] = __builtin_bit_cast(bf16x8, t);
    }
    // Drain these (compiler-tracked) loads here: a wait the compiler would
    // otherwise place inside the main loop also counts the untracked LDS-DMA
    // loads in flight there and would stall on them.
    __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
}

}  // namespace fv
