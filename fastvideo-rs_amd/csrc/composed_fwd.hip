// Composed SDPA, softmax(scale * q k^T + mask) v with f32 arithmetic, on the bf16 matrix cores: the path of the
// plans the reference runs through its composed tensor ops (rt/sdpa.rs:328-342: masked calls, Plan::composed, the
// block-causal / KV-window fallbacks, FASTVIDEO_SDPA=cublas) — there materialised scores through cuBLAS f32
// (rt/attn.rs:748-865), here an online softmax over key tiles, so no [bh, sq, sk] buffer exists. Head dims up to 128;
// longer heads keep the scalar kernel of rt_sdpa.hip.
//
// f32 on bf16 matrix cores: an f32 value is the sum of three bf16 values exactly (24 significant bits = 3 x 8, each
// part the nearest bf16 of what the ones before it leave; magnitudes from 2^-110 to the largest bf16 number, for the others
// see composed_redo), and a product of two of them, x y = sum over the parts, is
// exact in f32. Of the nine part products the six that matter are multiplied (hi.hi, hi.mid, mid.hi, mid.mid, hi.lo,
// lo.hi): the three left out are below 2^-24 of the product, the size of one f32 rounding, and the accumulators are
// f32. v_mfma_f32_32x32x16_bf16 has sixteen times the rate of v_mfma_f32_32x32x2_f32, so six of them cost 0.375 of the
// one f32 product they replace. Operands that are bf16 numbers already (bf16 tensors, or f32 ones that the caller
// wants rounded: PARTS = 1) have one part, so K Q^T is one product and P V, whose P is f32, three.
// Measured against the same sums in 64 bits, rel_l2: 5.4e-7 at 4096 x 4096 x 128, 3.9e-7 at 1024 x 1024 x 64; the
// v_mfma_f32_32x32x2_f32 form: 8.1e-7 and 6.1e-7. Time against that form with its casts, in us: 12 x 4096 x 4096 x 128 with a shared mask (f32 operands)
// 1376 -> 615 in 384 workgroups of two a CU, 531 with their last 128 cut in two (fv_composed_plan); 64 x 512 x 512 x 64 with a mask per
// head (bf16; 67 MB of mask) 306 -> 22, bound by the softmax's and the splitting of P's vector instructions; 16 x 257 x
// 257 x 80, which used to take the scalar kernel, 136 -> 10, a chain of two tiles with little to hide their latency.
//
// One workgroup = 4 waves (8 with eight shares). KS waves share 32 queries, each walking every KS-th key tile with its own
// running max and sum; their results are merged through LDS at the end, every wave a part of the channels (one wave
// merging and dividing them all took 2.9 of 11 us at 16 x 257 x 257 x 80, shader-clock stamps). KS = 1 (128 queries a workgroup) where the query tiles fill
// the chip, more where they do not. Tiles go global -> registers -> (split into parts) -> LDS; the next tile's loads
// are in flight under the arithmetic of the current one, and two workgroups share a CU, so that one wave's softmax and
// splitting run under the other's MFMAs.
//
//   S^T (32 keys x 32 queries) = K Q^T     A = K[key = l%32][16 j + 8 (l/32) ..], B = Q of the lane's query, same d
//   C layout                               lane l, register i: query l%32, key 8*(i/4) + 4*(l/32) + i%4
//   O^T (d x 32 queries) += V^T P^T        B = eight score registers as they are; A = V of the same keys, read
//                                          transposed from the row-major tile (ds_read_b64_tr_b16)
//
// LDS rows are padded so that both read patterns spread over all banks: K rows to 2 D + 16 bytes (a multiple of 16
// bytes that is odd in 16-byte units: 16 consecutive rows hit 16 different 16-byte columns), V rows to an odd multiple
// of 64 bytes (the 4 rows of a transposed read land in 4 different 64-byte bank groups).
#include <limits.h>

#include <initializer_list>

#include "../../include/fv_sdpa_hip.h"
#include "attn_core.h"
#include "fv_internal.h"

namespace fv {
namespace {

struct Parts3 {
    bf16x8 p[3];
};

// x = p[0] + p[1] + p[2] exactly (nearest bf16 each time)
FV_DEV Parts3 split3(const f32x8 x) {
    Parts3 r;
    f32x8 e = x;
#pragma unroll
    for (int t = 0; t < 3; t++) {
        r.p[t] = __builtin_convertvector(e, bf16x8);
        if (t < 2) {
            const u32x4 w = __builtin_bit_cast(u32x4, r.p[t]);   // the parts as f32 again, straight from the packed pairs
#pragma unroll
            for (int i = 0; i < 4; i++) {
                e[2 * i] -= __builtin_bit_cast(float, w[i] << 16);
                e[2 * i + 1] -= __builtin_bit_cast(float, w[i] & 0xffff0000u);
            }
        }
    }
    return r;
}

// Eight consecutive elements [c, c + 8) of a row of d, zeros past d; `vec`: rows are whole 16-byte units at 16-byte
// aligned addresses.
template <bool IS16>
FV_DEV f32x8 load8_f32(const void* row, int c, int d, bool vec) {
    f32x8 v = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if constexpr (IS16) {
        const uint16_t* p = (const uint16_t*)row + c;
        if (vec) {
            if (c < d) v = __builtin_convertvector(*reinterpret_cast<const bf16x8*>(p), f32x8);
        } else {
#pragma unroll
            for (int x = 0; x < 8; x++)
                if (c + x < d) v[x] = bf16_bits_to_f32(p[x]);
        }
    } else {
        const float* p = (const float*)row + c;
        if (vec) {
            if (c < d) {
                const f32x4 a = *reinterpret_cast<const f32x4*>(p), b = *reinterpret_cast<const f32x4*>(p + 4);
#pragma unroll
                for (int x = 0; x < 4; x++) v[x] = a[x], v[4 + x] = b[x];
            }
        } else {
#pragma unroll
            for (int x = 0; x < 8; x++)
                if (c + x < d) v[x] = p[x];
        }
    }
    return v;
}

template <int D>
struct ComposedGeo {
    static constexpr int kKRow = 2 * D + 16;
    static constexpr int kVRow = (D / 32) % 2 == 1 ? 2 * D : 2 * D + 64;
};
constexpr int composed_waves(int ks) { return ks < 4 ? 4 : ks; }
// O of one wave in the merge: D / 8 groups of four registers, then max and sum
template <int D>
constexpr int kMergeShare = D / 8 * 1024 + 512;
template <int D, int PARTS, int KS>
constexpr int composed_lds() {
    constexpr int tiles = KS * PARTS * 32 * (ComposedGeo<D>::kKRow + ComposedGeo<D>::kVRow);
    constexpr int merge = KS > 1 ? composed_waves(KS) * kMergeShare<D> : 0;
    return tiles > merge ? tiles : merge;
}

// One workgroup's item: its (batch, head) plane, query tile and key tiles; split < 0: all of them, else that key range of
// a cut tail. Workgroup i runs on XCD i % 8. A mask of every head's own (or none): XCD x takes a contiguous eighth of the
// (head, query tile) items, so that a head's keys and values pass through one L2. A shared mask: the query tiles go round
// the XCDs, so that a mask row is read through one L2 for all heads.
struct ComposedItem {
    bool none;
    long bh;
    int qt, tile0, tiles, split;
};
template <int KS, class Params>
FV_DEV ComposedItem composed_item(const Params& p, int item) {
    ComposedItem r = {false, 0, 0, 0, (p.sk + 31) / 32, -1};
    if (KS == 1 && item < p.full) {          // (full is a multiple of 8)
        if (p.by_head) item = (item & 7) * (p.full >> 3) + (item >> 3);
    } else {
        if constexpr (KS == 1) item -= p.full;
        if (p.by_head) item = (item & 7) * p.per_xcd + (item >> 3);
        if (item >= p.total) {
            r.none = true;
            return r;
        }
        if constexpr (KS == 1) {
            if (p.splits > 1) {
                const int tile = item / p.splits;
                r.split = item - tile * p.splits;
                item = tile;
                r.tile0 = r.split * p.split_tiles;
                r.tiles = min(p.split_tiles, r.tiles - r.tile0);
            }
            item += p.full;
        }
    }
    r.bh = item / p.nqt;
    r.qt = item - (int)r.bh * p.nqt;
    return r;
}

// Unmasked scores are compared unscaled, so the scale's sign goes into Q and its magnitude into the exponent; a scale of
// zero makes Q zero. With a mask the scores are s * scale + mask before they are compared.
template <class Params>
FV_DEV float composed_q_mul(const Params& p) {
    return p.mask || p.scale > 0.f ? 1.f : p.scale < 0.f ? -1.f : p.scale;
}
template <class Params>
FV_DEV float composed_to_log2(const Params& p) {
    return p.mask || p.scale == 0.f ? 1.4426950408889634f : __builtin_fabsf(p.scale) * 1.4426950408889634f;
}

// The additive mask of the lane's 16 keys, four consecutive ones per load: vector loads need no more than the alignment
// of a float. Element by element only in a tile that a row ends in between two such groups, where a whole group would
// reach past the mask's last row. (Rows of any other length than whole 16-byte units used to be read element by element
// throughout: 32 rows touched by each of 16 instructions, 787 -> 476 us at 64 x 2611 x 2611 x 80 with a shared mask,
// 58.7 -> 41.6 at 64 x 523 x 523 x 80 with a mask per head.)
FV_DEV void load_mask(const float* mr, int kv0, int h, int sk, f32x16& mk) {
    typedef f32x4 __attribute__((aligned(4))) f32x4_any;
    if (!mr) return;
    if ((sk & 3) == 0 || kv0 + 32 <= sk) {
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const f32x4 t = *reinterpret_cast<const f32x4_any*>(mr + min(kv0 + 8 * g + 4 * h, sk - 4));
#pragma unroll
            for (int x = 0; x < 4; x++) mk[4 * g + x] = t[x];
        }
    } else {
#pragma unroll
        for (int i = 0; i < 16; i++) mk[i] = mr[min(kv0 + 8 * (i >> 2) + 4 * h + (i & 3), sk - 1)];
    }
}

// out = o / l for four consecutive channels from d0 on of query qi; l == 0 (no key): zeros. A NaN score is not the largest
// of its row (max drops it) but makes l NaN, and the row with it. PLAIN: o may be infinite (otherwise composed_redo stores
// over it).
template <bool PLAIN, class Params>
FV_DEV void composed_store4(const Params& p, long bh, int qi, f32x4 r, float l, float inv, int d0) {
#pragma clang fp contract(off)
    const int d = p.d;
    const bool vec = p.vec != 0;
#pragma unroll
    for (int x = 0; x < 4; x++) {
        // one Newton step on the quotient: the rounding of o / l without the division's scaling (1 <= l < 2^32); it makes
        // an infinity NaN
        const float v = r[x] * inv;
        const float n = __builtin_fmaf(__builtin_fmaf(-v, l, r[x]), inv, v);
        r[x] = l == 0.f ? 0.f : !PLAIN || __builtin_fabsf(v) < __builtin_inff() ? n : v;
    }
    const long at = (bh * p.sq + qi) * (long)d + d0;
    if (p.out_is_bf16) {
        uint16_t* dst = (uint16_t*)p.out + at;
        const bf16x4 r16 = __builtin_convertvector(r, bf16x4);
        if (vec) {
            if (d0 < d) *reinterpret_cast<bf16x4*>(dst) = r16;
        } else {
#pragma unroll
            for (int x = 0; x < 4; x++)
                if (d0 + x < d) reinterpret_cast<__bf16*>(dst)[x] = r16[x];
        }
    } else {
        float* dst = (float*)p.out + at;
        if (vec) {
            if (d0 < d) *reinterpret_cast<f32x4*>(dst) = r;
        } else {
#pragma unroll
            for (int x = 0; x < 4; x++)
                if (d0 + x < d) dst[x] = r[x];
        }
    }
}

// A wave's rows where it has walked all keys of its item: the result, or (split >= 0: a part of the keys) the sums for the
// merge kernel. STEP > 1: every STEP-th group of four channels from `first` on.
template <int NO, int STEP, bool PLAIN, class Params>
FV_DEV void composed_store_rows(const Params& p, long bh, int qi, int split, int h, float m, float l, const f32x16 (&o)[NO],
                                int first) {
    const long row = split * p.part_rows + (bh * p.sq + qi - p.part_row0);
    if (split >= 0 && h == 0) *reinterpret_cast<f32x2*>(p.part_ml + 2 * row) = f32x2{m, l};
    const float inv = __builtin_amdgcn_rcpf(l);
#pragma unroll
    for (int db = 0; db < NO; db++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            if (STEP > 1 && (4 * db + g) % STEP != first) continue;
            const int d0 = 32 * db + 8 * g + 4 * h;
            f32x4 r;
#pragma unroll
            for (int x = 0; x < 4; x++) r[x] = o[db][4 * g + x];
            if (split < 0) composed_store4<PLAIN>(p, bh, qi, r, l, inv, d0);
            else if (d0 < p.d) *reinterpret_cast<f32x4*>(p.part_o + row * p.dpad + d0) = r;
        }
}

// Do sums of weighted values, or l, the sum of their weights, ask for the plain products below? Gathered four at a time.
template <int PARTS>
struct ComposedSuspect {
    f32x4 chk = {0.f, 0.f, 0.f, 0.f};   // NaN once an infinity or a NaN has been seen
    unsigned least = ~0u;               // the least magnitude but zero
    FV_DEV void add(const f32x4 r) {
#pragma unroll
        for (int x = 0; x < 4; x++) {
            const float v = r[x];       // (a bit cast of the vector's element itself reads element 0)
            chk[x] = __builtin_fmaf(v, 0.f, chk[x]);
            if constexpr (PARTS == 3) least = min(least, (__builtin_bit_cast(unsigned, v) << 1) - 1u);
        }
    }
    FV_DEV bool operator()(float l) const {
        bool bad = !((chk[0] + chk[1]) + (chk[2] + chk[3]) + l * 0.f == 0.f);
        if constexpr (PARTS == 3) bad |= least < (__builtin_bit_cast(unsigned, l * 0x1p-104f) << 1) - 1u;
        return bad;
    }
};

// Operands outside the range of the parts. One past the largest bf16 number (infinities, and f32 numbers above 3.396e38)
// has parts that do not add up to it, and so has an infinity under the signed parts of P: the sums they enter are NaN. An
// f32 value below 2^-110 has fewer than three whole parts, which costs a result its last bits when it is that small itself
// (a score's error, 2^-134 times the other operand, stays below f32's own up to operands of 2^96). Where a query's sums
// end with a NaN, an infinity or so small a result, its wave makes the walk over its item's keys again in plain f32
// products (v_mfma_f32_32x32x2_f32: the two k slots of a product are the lane halves), operands straight from memory, no
// LDS, no barrier, and stores that for the queries with `redo`: 0 times a finite number, the weights of -inf scores and
// NaN rows come out as in the plain sums, and the other queries keep their bits. The last thing a wave does, with a softmax
// of its own: sharing the first walk's, or keeping its values alive, cost that walk registers (12 x 1024 x 1024 x 128 in
// f32 107 -> 117 us; so 107, and the check 0 - 2 % of a launch, 0.6 of 21 us at 12 x 300 x 300 x 80). A launch whose every
// head holds an infinity takes 5 to 14 times as long: 12 x 4096 x 4096 x 128 3.7 ms (f32), 5.0 (bf16).
template <int D, int PARTS, int KS, bool KV16>
FV_DEV void composed_redo(const __attribute__((address_space(4))) ComposedParams& p, int block, int wave, int lane, bool redo) {
    constexpr int QG = composed_waves(KS) / KS, kElem = KV16 ? 2 : 4, NO = D / 32;
    const int h = lane >> 5, c32 = lane & 31;
    const ComposedItem it = composed_item<KS>(p, block);
    const int sq = p.sq, sk = p.sk, d = p.d, qi = it.qt * (32 * QG) + (wave % QG) * 32 + c32;
    const bool q_ok = qi < sq, vec = p.vec != 0, q16 = p.q_is_bf16 != 0;
    const long qrow = (it.bh * sq + (q_ok ? qi : 0)) * d;
    const char* kb = (const char*)p.k + it.bh * sk * (long)d * kElem;
    const char* vb = (const char*)p.v + it.bh * sk * (long)d * kElem;
    const char* qr = (const char*)p.q + qrow * (q16 ? 2 : 4);
    const float* mr = p.mask ? p.mask + it.bh * p.mask_bh + (long)(q_ok ? qi : 0) * sk : nullptr;
    const float q_mul = composed_q_mul(p), to_log2 = composed_to_log2(p), scale = p.scale;
    f32x16 o[NO];
#pragma unroll
    for (int db = 0; db < NO; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) o[db][i] = 0.f;
    float m_run = neg_inf(), l_run = 0.f;
    auto operand = [&](f32x8 x) {
        if constexpr (PARTS == 1) return __builtin_convertvector(__builtin_convertvector(x, bf16x8), f32x8);
        else return x;
    };
#pragma unroll 1
    for (int t = 0; t < it.tiles; t++) {
        const int kv0 = (it.tile0 + t) * 32;
        f32x16 mk, s;
        load_mask(mr, kv0, h, sk, mk);
#pragma unroll
        for (int i = 0; i < 16; i++) s[i] = 0.f;
        const char* krow = kb + (long)min(kv0 + c32, sk - 1) * d * kElem;
#pragma unroll 1
        for (int c = 0; c < D; c += 16) {
            const f32x8 a = operand(load8_f32<KV16>(krow, c + 8 * h, d, vec));
            f32x8 b = q16 ? load8_f32<true>(qr, c + 8 * h, d, vec) : load8_f32<false>(qr, c + 8 * h, d, vec);
            if (!q_ok) b = f32x8{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            b = operand(b * q_mul);
#pragma unroll
            for (int x = 0; x < 8; x++) s = __builtin_amdgcn_mfma_f32_32x32x2f32(a[x], b[x], s, 0, 0, 0);
        }
        float mx = neg_inf(), ls = 0.f;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            if (mr) s[i] = __builtin_fmaf(s[i], scale, mk[i]);
            if (kv0 + 8 * (i >> 2) + 4 * h + (i & 3) >= sk) s[i] = neg_inf();
            mx = __builtin_fmaxf(mx, s[i]);
        }
        const float m_new = __builtin_fmaxf(m_run, pair_max(mx));
        const float alpha = m_run == neg_inf() ? 0.f : fast_exp2((m_run - m_new) * to_log2);
        const float off = m_new == neg_inf() ? 0.f : m_new;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            s[i] = fast_exp2((s[i] - off) * to_log2);
            ls += s[i];
        }
        m_run = m_new;
        l_run = l_run * alpha + ls;
#pragma unroll
        for (int db = 0; db < NO; db++)
#pragma unroll
            for (int i = 0; i < 16; i++) o[db][i] *= alpha;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int key = kv0 + 8 * (i >> 2) + 4 * h + (i & 3);
            const char* vrow = vb + (long)min(key, sk - 1) * d * kElem;
#pragma unroll
            for (int db = 0; db < NO; db++) {
                const int c = 32 * db + c32;
                float a = 0.f;
                if (key < sk && c < d) {
                    if constexpr (KV16) a = bf16_bits_to_f32(((const uint16_t*)vrow)[c]);
                    else a = ((const float*)vrow)[c];
                }
                if constexpr (PARTS == 1 && !KV16) a = (float)(__bf16)a;
                o[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, s[i], o[db], 0, 0, 0);
            }
            asm volatile("" ::: "memory");   // (few loads in flight, few registers)
        }
    }
    l_run = pair_sum(l_run);
    if (redo) composed_store_rows<NO, KS, true>(p, it.bh, qi, it.split, h, m_run, l_run, o, wave / QG);
}

template <int D, int PARTS, int KS, bool KV16>
__global__ __launch_bounds__(64 * composed_waves(KS), 2) void sdpa_composed_kernel(const ComposedParams p) {
    static_assert(D % 32 == 0 && (PARTS == 1 || PARTS == 3) && (KS == 1 || KS == 2 || KS == 4 || KS == 8) &&
                  !(KV16 && PARTS == 3), "instantiations");
    using G = ComposedGeo<D>;
    constexpr int QG = composed_waves(KS) / KS;   // 32-query groups per workgroup
    constexpr int kGroup = 64 * QG;          // threads that share a key tile
    constexpr int kKP = 32 * G::kKRow, kVP = 32 * G::kVRow;   // bytes of one part of a K / V tile
    constexpr int kUnits = 32 * (D / 8);     // 8-element units per tile
    constexpr int kPer = (kUnits + kGroup - 1) / kGroup;
    constexpr int NO = D / 32, NC = D / 16;
    constexpr int kMine = KV16 ? 4 : 8;      // 32-bit registers per unit in flight
    extern __shared__ __attribute__((aligned(16))) unsigned char csm[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, c32 = lane & 31;
    const int qg = wave % QG, ks = wave / QG;
    const int gt = tid - ks * kGroup;        // thread within the group
    lds_u8* kt = (lds_u8*)csm + ks * (PARTS * (kKP + kVP));
    lds_u8* vt = kt + PARTS * kKP;
    const int sq = p.sq, sk = p.sk, d = p.d;
    const ComposedItem it = composed_item<KS>(p, blockIdx.x);
    if (it.none) return;
    const long bh = it.bh;
    const int qt = it.qt, tile0 = it.tile0, tiles = it.tiles, split = it.split;
    const bool vec = p.vec != 0;
    const int qi = qt * (32 * QG) + qg * 32 + c32;   // this lane's query
    const bool q_ok = qi < sq;
    const float NEG = neg_inf();
    const float q_mul = composed_q_mul(p), to_log2 = composed_to_log2(p);
    const char* kb = (const char*)p.k + bh * sk * (long)d * (KV16 ? 2 : 4);
    const char* vb = (const char*)p.v + bh * sk * (long)d * (KV16 ? 2 : 4);
    const float* mr = p.mask ? p.mask + bh * p.mask_bh + (long)(q_ok ? qi : 0) * sk : nullptr;

    // One 8-element unit of the group's tile in registers: raw bf16, or f32.
    struct Unit {
        u32x4 r[kMine / 4];
    };
    // Byte offsets of this thread's units from the tile's first row; units past d are never loaded and stay zero.
    constexpr int kElem = KV16 ? 2 : 4;
    int uoff[kPer];
    bool uok[kPer];
#pragma unroll
    for (int r = 0; r < kPer; r++) {
        const int un = gt + kGroup * r, row = un / (D / 8), c = 8 * (un % (D / 8));
        uoff[r] = (row * d + c) * kElem;
        uok[r] = un < kUnits && c < d;
    }
    // Rows past the end re-read the last one: their scores are masked, and the last row's values times zero.
    auto load_units = [&](const char* base, int kv0, Unit (&u)[kPer]) {
        const char* tile = base + (long)kv0 * d * kElem;
        const int last = sk - 1 - kv0;
#pragma unroll
        for (int r = 0; r < kPer; r++) {
            const int un = gt + kGroup * r, row = un / (D / 8), c = 8 * (un % (D / 8));
            if (!uok[r]) continue;
            const char* src = tile + (uoff[r] - max(0, row - last) * d * kElem);
            if (vec) {
#pragma unroll
                for (int x = 0; x < kMine / 4; x++) u[r].r[x] = *reinterpret_cast<const u32x4*>(src + 16 * x);
            } else {
                // rows that are not whole 16-byte units: element by element
#pragma unroll
                for (int x = 0; x < kMine / 4; x++) u[r].r[x] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
                for (int x = 0; x < 8; x++) {
                    if (c + x < d) {
                        if constexpr (KV16)
                            u[r].r[0][x >> 1] |= (unsigned)reinterpret_cast<const uint16_t*>(src)[x] << (16 * (x & 1));
                        else
                            u[r].r[(x >> 2) % (kMine / 4)][x & 3] = reinterpret_cast<const unsigned*>(src)[x];
                    }
                }
            }
        }
    };
    auto store_units = [&](lds_u8* dst, int row_bytes, int part_bytes, const Unit (&u)[kPer]) {
#pragma unroll
        for (int r = 0; r < kPer; r++) {
            const int un = gt + kGroup * r, row = un / (D / 8), c = 8 * (un % (D / 8));
            if (un >= kUnits) continue;
            lds_u8* at = dst + row * row_bytes + 2 * c;
            if constexpr (KV16) {
                lds_write_b128(at, u[r].r[0]);
            } else {
                const f32x4 a = __builtin_bit_cast(f32x4, u[r].r[0]), b = __builtin_bit_cast(f32x4, u[r].r[kMine / 4 - 1]);
                const f32x8 x = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
                if constexpr (PARTS == 1) {
                    lds_write_b128(at, __builtin_bit_cast(u32x4, __builtin_convertvector(x, bf16x8)));
                } else {
                    const Parts3 s = split3(x);
#pragma unroll
                    for (int t = 0; t < 3; t++) lds_write_b128(at + t * part_bytes, __builtin_bit_cast(u32x4, s.p[t]));
                }
            }
        }
    };

    // A tile belongs to one wave where every wave walks keys of its own: its LDS writes and reads complete in order.
    auto tile_barrier = [&]() {
        if constexpr (KS >= 4) __builtin_amdgcn_wave_barrier();
        else __syncthreads();
    };

    f32x16 o[NO];
#pragma unroll
    for (int db = 0; db < NO; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) o[db][i] = 0.f;
    float m_run = NEG, l_run = 0.f;

    const lds_u8* ka = kt + c32 * G::kKRow + 16 * h;
    const int b16 = lane >> 4, i16 = lane & 15;
    const lds_u8* va = vt + (4 * h + (i16 >> 2)) * G::kVRow + 32 * (b16 & 1) + 8 * (i16 & 3);

    const int steps = (tiles + KS - 1) / KS;
    Unit ku[kPer], vu[kPer];
#pragma unroll
    for (int r = 0; r < kPer; r++)
#pragma unroll
        for (int x = 0; x < kMine / 4; x++) ku[r].r[x] = vu[r].r[x] = u32x4{0u, 0u, 0u, 0u};
    f32x16 mk;
    load_units(kb, (tile0 + ks) * 32, ku);
    load_units(vb, (tile0 + ks) * 32, vu);
    load_mask(mr, (tile0 + ks) * 32, h, sk, mk);

    // Q operand, in parts: this lane's query, d = 16 j + 8 h ..
    bf16x8 qf[PARTS][NC];
    {
        const long row = (bh * sq + (q_ok ? qi : 0)) * d;
#pragma unroll
        for (int j = 0; j < NC; j++) {
            const int c = 16 * j + 8 * h;
            f32x8 x = p.q_is_bf16 ? load8_f32<true>((const uint16_t*)p.q + row, c, d, vec)
                                  : load8_f32<false>((const float*)p.q + row, c, d, vec);
            if (!q_ok) x = f32x8{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            if (q_mul != 1.f) x = x * q_mul;
            if constexpr (PARTS == 1) {
                qf[0][j] = __builtin_convertvector(x, bf16x8);
            } else {
                const Parts3 s = split3(x);
#pragma unroll
                for (int t = 0; t < 3; t++) qf[t][j] = s.p[t];
            }
        }
    }

#pragma unroll 1
    for (int step = 0; step < steps; step++) {
        const int kv0 = (tile0 + step * KS + ks) * 32;
        store_units(kt, G::kKRow, kKP, ku);
        store_units(vt, G::kVRow, kVP, vu);
        tile_barrier();
        if (step + 1 < steps) {   // in flight under this tile's arithmetic (rows past the end: zeros)
            load_units(kb, kv0 + 32 * KS, ku);
            load_units(vb, kv0 + 32 * KS, vu);
        }
        if (kv0 < sk) {           // (a wave whose share has ended keeps the barriers only)
            // ---- S^T = K Q^T ----
            f32x16 s;
#pragma unroll
            for (int i = 0; i < 16; i++) s[i] = 0.f;
#pragma unroll
            for (int j = 0; j < NC; j++) {
                bf16x8 a[PARTS];
#pragma unroll
                for (int t = 0; t < PARTS; t++) a[t] = lds_read_b128(ka + t * kKP + 32 * j);
                if constexpr (PARTS == 3) {   // small products first
                    s = mfma32(a[2], qf[0][j], s);
                    s = mfma32(a[0], qf[2][j], s);
                    s = mfma32(a[1], qf[1][j], s);
                    s = mfma32(a[1], qf[0][j], s);
                    s = mfma32(a[0], qf[1][j], s);
                }
                s = mfma32(a[0], qf[0][j], s);
            }
            // ---- mask, online softmax (per lane = per query; the halves share the max, each sums its own keys) ----
            // Without a mask the scores stay unscaled up to the exponential; with one they are s * scale + mask.
            {
                if (mr) {
#pragma unroll
                    for (int i = 0; i < 16; i++) s[i] = __builtin_fmaf(s[i], p.scale, mk[i]);
                }
                if (kv0 + 32 > sk) {
                    asm volatile("");   // a branch, not sixteen selects on every tile
#pragma unroll
                    for (int i = 0; i < 16; i++)
                        if (kv0 + 8 * (i >> 2) + 4 * h + (i & 3) >= sk) s[i] = NEG;
                }
                float mx = NEG;
#pragma unroll
                for (int i = 0; i < 16; i++) mx = __builtin_fmaxf(mx, s[i]);
                mx = pair_max(mx);
                const float m_new = __builtin_fmaxf(m_run, mx);
                const float alpha = (m_run == NEG) ? 0.f : fast_exp2((m_run - m_new) * to_log2);
                const float off = (m_new == NEG) ? 0.f : m_new;   // a row that has seen no key: every P is 2^-inf = 0
                float ls = 0.f;
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const float e = fast_exp2((s[i] - off) * to_log2);
                    s[i] = e;
                    ls += e;
                }
                l_run = l_run * alpha + ls;
                m_run = m_new;
                if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
#pragma unroll
                    for (int db = 0; db < NO; db++)
#pragma unroll
                        for (int i = 0; i < 16; i++) o[db][i] *= alpha;
                }
            }
            // the next tile's mask, in flight under the rest of this tile (rows past the end: nothing)
            if (step + 1 < steps) load_mask(mr, kv0 + 32 * KS, h, sk, mk);
            // ---- O^T += V^T P^T, 16 keys at a time ----
#pragma unroll
            for (int t = 0; t < 2; t++) {
                f32x8 e;
#pragma unroll
                for (int x = 0; x < 8; x++) e[x] = s[8 * t + x];
                const Parts3 pp = split3(e);
#pragma unroll
                for (int db = 0; db < NO; db++) {
                    bf16x8 a[PARTS];
#pragma unroll
                    for (int x = 0; x < PARTS; x++) {
                        const lds_u8* at = va + x * kVP + 64 * db + 16 * t * G::kVRow;
                        s16x8 w;
                        w.lo = lds_read_tr16_b64(at);
                        w.hi = lds_read_tr16_b64(at + 8 * G::kVRow);
                        a[x] = __builtin_bit_cast(bf16x8, w);
                    }
                    if constexpr (PARTS == 3) {
                        o[db] = mfma32(a[2], pp.p[0], o[db]);
                        o[db] = mfma32(a[1], pp.p[1], o[db]);
                        o[db] = mfma32(a[0], pp.p[2], o[db]);
                        o[db] = mfma32(a[1], pp.p[0], o[db]);
                    } else {
                        o[db] = mfma32(a[0], pp.p[2], o[db]);
                    }
                    o[db] = mfma32(a[0], pp.p[1], o[db]);
                    o[db] = mfma32(a[0], pp.p[0], o[db]);
                }
            }
        }
        tile_barrier();
    }
    l_run = pair_sum(l_run);

    ComposedSuspect<PARTS> suspect;
    bool redo;
    if constexpr (KS == 1) {
#pragma unroll
        for (int db = 0; db < NO; db++)
#pragma unroll
            for (int g = 0; g < 4; g++) suspect.add(f32x4{o[db][4 * g], o[db][4 * g + 1], o[db][4 * g + 2], o[db][4 * g + 3]});
        redo = pair_max(suspect(l_run) ? 1.f : 0.f) > 0.f;   // (a query is a pair of lanes)
        if (q_ok) composed_store_rows<NO, 1, false>(p, bh, qi, split, h, m_run, l_run, o, 0);
    } else {
        // Merge of a query's KS shares, every wave its part of the channels: all leave O, max and sum in LDS (over the
        // tiles, which every wave is done with), each adds up every KS-th group of four registers over the shares.
        typedef __attribute__((address_space(3))) f32x4 lds_f4;
        typedef __attribute__((address_space(3))) f32x2 lds_f2;
        if constexpr (KS >= 4) __syncthreads();   // (KS = 2: the loop ends with one)
        auto share = [&](int t) { return (lds_u8*)csm + (t * QG + qg) * kMergeShare<D>; };
#pragma unroll
        for (int db = 0; db < NO; db++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
                f32x4 r;
#pragma unroll
                for (int x = 0; x < 4; x++) r[x] = o[db][4 * g + x];
                *(lds_f4*)(share(ks) + ((4 * db + g) * 64 + lane) * 16) = r;
            }
        *(lds_f2*)(share(ks) + D / 8 * 1024 + lane * 8) = f32x2{m_run, l_run};
        __syncthreads();
        float w[KS], l = 0.f, m_all = NEG;
        f32x2 ml[KS];
#pragma unroll
        for (int t = 0; t < KS; t++) ml[t] = *(const lds_f2*)(share(t) + D / 8 * 1024 + lane * 8);
#pragma unroll
        for (int t = 0; t < KS; t++) m_all = __builtin_fmaxf(m_all, ml[t][0]);
#pragma unroll
        for (int t = 0; t < KS; t++) {
            w[t] = ml[t][0] == NEG ? 0.f : fast_exp2((ml[t][0] - m_all) * to_log2);
            l = __builtin_fmaf(ml[t][1], w[t], l);
        }
        const float inv = __builtin_amdgcn_rcpf(l);
#pragma unroll 1
        for (int gi = ks; gi < D / 8; gi += KS) {
            f32x4 r = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int t = 0; t < KS; t++) {
                const f32x4 x4 = *(const lds_f4*)(share(t) + (gi * 64 + lane) * 16);
#pragma unroll
                for (int x = 0; x < 4; x++) r[x] = __builtin_fmaf(x4[x], w[t], r[x]);
            }
            suspect.add(r);
            if (q_ok) composed_store4<false>(p, bh, qi, r, l, inv, 8 * gi + 4 * h);
        }
        redo = suspect(l);
    }
    redo &= q_ok;
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(redo) != 0, 0)) {
        __builtin_amdgcn_s_waitcnt(0);   // (behind the stores above; each wave for the channels it has stored)
        // (nothing of the first walk is kept alive for this: indices counted anew, arguments read again from their segment)
        using ConstParams = const __attribute__((address_space(4))) ComposedParams;
        ConstParams* again = (ConstParams*)__builtin_amdgcn_kernarg_segment_ptr();
        int lane2 = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)), wave2 = wave, block = blockIdx.x;
        asm volatile("" : "+v"(lane2), "+s"(wave2), "+s"(block), "+s"(again));
        composed_redo<D, PARTS, KS, KV16>(*again, block, wave2, lane2, redo);
    }
}

// ---- short launches on bf16 operands --------------------------------------------------------
// For launches whose time is one chain of latencies and not the matrix pipe. One workgroup = 32 queries of one (batch,
// head); wave w of its KS = 8 or 4 walks the 32-key tiles w, w + KS, ... with K and V buffers, running max and sums of its
// own, and the shares are merged through LDS: one barrier when the query rows are there, none until the merge. Tiles and
// query rows come by LDS-DMA (whole rows: fragments straight from memory touch every row with every instruction), the
// next K tile while the softmax runs, the next V tile behind the products. PP: parts of P, 3 for the composed plans
// (masks, head dims in steps of 8, exact P), 1 for the fused kernels' plans (P rounded to bf16, no mask, head dims 64
// and 128). Shader-clock stamps at 12 x 320 x 320 x 128, 13 k cycles: arguments 0.6, issue of 17 loads a wave
// 1.6, query rows and K 2.2, two tiles 4.3, merge 3.8 (128 KB written, 128 KB read), drain
// 0.5. us, in a graph, the kernels it replaces / this: 12 x 320 x 320 x 128 11.0 / 6.8 (flash_fwd_pp2, 24 k cycles in five phases),
// 16 x 257 x 257 x 80 10.2 / 7.8, 12 x 668 x 668 x 128 17.8 / 9.7, 12 x 1200 x 1200 x 64 19.5 / 12.9.
template <int NC>
struct ShortGeo {
    static constexpr int D = NC <= 4 ? 64 : 128;      // channels an LDS row has room for
    using G = TileGeo<D>;
    static constexpr int kTile = 32 * G::kRow;        // 32 rows
    static constexpr int kIt = kTile / 1024;          // LDS-DMA instructions a tile
    static constexpr int NO = (NC + 1) / 2;           // 32-channel blocks of the result
};
template <int NC, int KS>
constexpr int short_lds() {
    constexpr int tiles = (2 * KS + 1) * ShortGeo<NC>::kTile, merge = KS * kMergeShare<32 * ShortGeo<NC>::NO>;
    return tiles > merge ? tiles : merge;
}

// LOG2DOM: scale * log2(e) is one, no multiply of a score.
template <int NC, int PP, int KS, bool LOG2DOM>
__global__ __launch_bounds__(64 * KS, NC <= 4 ? 4 : 2) void sdpa_short_kernel(const ComposedParams p) {
    using SG = ShortGeo<NC>;
    using G = typename SG::G;
    constexpr int kTile = SG::kTile, kIt = SG::kIt, NO = SG::NO;
    extern __shared__ __attribute__((aligned(16))) unsigned char csm[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, c32 = lane & 31;
    const ComposedItem it = composed_item<KS>(p, blockIdx.x);
    if (it.none) return;
    const int sq = p.sq, sk = p.sk, d = PP == 1 ? SG::D : p.d, tiles = it.tiles;
    const int rowb = 2 * d, nch = d >> 3;             // bytes and 16-byte chunks of a row in memory
    const long bh = it.bh;
    const int qi = it.qt * 32 + c32;
    const bool q_ok = qi < sq;
    const float NEG = neg_inf();
    const char* qb = (const char*)p.q + (bh * p.q_plane + (long)it.qt * 32 * d) * 2;
    const char* kb = (const char*)p.k + bh * p.k_plane * 2;
    const char* vb = (const char*)p.v + bh * p.v_plane * 2;
    lds_u8* kt = (lds_u8*)csm + wave * (2 * kTile);
    lds_u8* vt = kt + kTile;
    lds_u8* qs = (lds_u8*)csm + 2 * KS * kTile;
    const int lr = lane / G::kChunks, lc = lane % G::kChunks;
    // One instruction's rows of a tile of `rows` valid ones (the ones past them re-read the last): whole 16-byte chunks of
    // the row, each to its swizzled place; lanes whose chunk lies past d fetch nothing. Every instruction has lanes that do.
    auto request_one = [&](lds_u8* dst, const char* base, int rows, int it_, bool is_v) {
        const int r = it_ * G::kRowsPerDma + lr, c = lc ^ (is_v ? G::vswz32(r) : G::kswz(r));
        const unsigned at = __builtin_amdgcn_readfirstlane((unsigned)(size_t)dst) + it_ * 1024;
        const unsigned off = (unsigned)(min(r, rows - 1) * rowb + (c << 4));
        if (PP == 1 || c < nch) lds_dma16_s(at, base, off);
    };
    auto request = [&](lds_u8* dst, const char* base, int t, bool is_v) {
        const char* tile = base + (long)t * 32 * rowb;
#pragma unroll
        for (int i = 0; i < kIt; i++) request_one(dst, tile, sk - 32 * t, i, is_v);
    };
#pragma unroll
    for (int i = 0; i < (kIt + KS - 1) / KS; i++)
        if (i * KS + wave < kIt) request_one(qs, qb, sq - it.qt * 32, i * KS + wave, false);
    if (wave < tiles) {
        request(kt, kb, wave, false);
        request(vt, vb, wave, true);
    }
    const float* mr = PP == 3 && p.mask ? p.mask + bh * p.mask_bh + (long)(q_ok ? qi : 0) * sk : nullptr;
    f32x16 mk;
    if (PP == 3 && wave < tiles) load_mask(mr, wave * 32, h, sk, mk);
    if (PP == 3 && nch < 2 * NC) {   // the channels between d and the products' last: zeros, in K for each wave and in Q
#pragma unroll
        for (int i = 0; i < kIt; i++) {
            const int r = i * G::kRowsPerDma + lr, c = lc ^ G::kswz(r);
            if (c >= nch && c < 2 * NC) {
                lds_write_b128(kt + i * 1024 + lane * 16, u32x4{0u, 0u, 0u, 0u});
                if (wave == 0) lds_write_b128(qs + i * 1024 + lane * 16, u32x4{0u, 0u, 0u, 0u});
            }
        }
    }
    // (2 kIt loads after the query rows'; a wave without keys has no other)
    if (wave < tiles) wait_vmcnt<2 * kIt>();
    else wait_vmcnt<0>();
    __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): the zeros are written
    block_barrier();
    const TileReadBases rb = tile_read_bases32<SG::D>(lane);
    const float q_mul = PP == 3 ? composed_q_mul(p) : 1.f, to_log2 = LOG2DOM ? 1.f : composed_to_log2(p);
    bf16x8 qf[NC];
#pragma unroll
    for (int j = 0; j < NC; j++) {
        qf[j] = lds_read_b128(qs + (rb.k ^ (j << 5)));
        if (q_mul != 1.f) qf[j] = __builtin_convertvector(__builtin_convertvector(qf[j], f32x8) * q_mul, bf16x8);
    }
    f32x16 o[NO];
#pragma unroll
    for (int db = 0; db < NO; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) o[db][i] = 0.f;
    float m_run = NEG, l_run = 0.f;
#pragma unroll 1
    for (int t = wave; t < tiles; t += KS) {
        const int kv0 = 32 * t;
        const bool more = t + KS < tiles;
        wait_vmcnt<kIt>();                // K(t) has landed; V(t) may be in flight
        f32x16 s;
#pragma unroll
        for (int i = 0; i < 16; i++) s[i] = 0.f;
#pragma unroll
        for (int j = 0; j < NC; j++) s = mfma32(lds_read_b128(kt + (rb.k ^ (j << 5))), qf[j], s);
        __builtin_amdgcn_s_waitcnt(0xC07F);   // (every K read has returned)
        __builtin_amdgcn_sched_barrier(0);
        if (more) request(kt, kb, t + KS, false);
        if (PP == 3 && mr) {
#pragma unroll
            for (int i = 0; i < 16; i++) s[i] = __builtin_fmaf(s[i], p.scale, mk[i]);
        }
        if (kv0 + 32 > sk) {
            asm volatile("");
#pragma unroll
            for (int i = 0; i < 16; i++)
                if (kv0 + 8 * (i >> 2) + 4 * h + (i & 3) >= sk) s[i] = NEG;
        }
        float mx = NEG;
#pragma unroll
        for (int i = 0; i < 16; i++) mx = __builtin_fmaxf(mx, s[i]);
        const float m_new = __builtin_fmaxf(m_run, pair_max(mx));
        const float alpha = (m_run == NEG) ? 0.f : fast_exp2((m_run - m_new) * to_log2);
        const float off = (m_new == NEG) ? 0.f : m_new;
        float ls = 0.f;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            s[i] = fast_exp2((s[i] - off) * to_log2);
            ls += s[i];
        }
        l_run = l_run * alpha + ls;
        m_run = m_new;
        if (t >= KS && __builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
#pragma unroll
            for (int db = 0; db < NO; db++)
#pragma unroll
                for (int i = 0; i < 16; i++) o[db][i] *= alpha;
        }
        if (PP == 3 && more) load_mask(mr, kv0 + 32 * KS, h, sk, mk);
        if (more) wait_vmcnt<kIt>();      // V(t) has landed; K of the next tile may be in flight
        else wait_vmcnt<0>();
#pragma unroll
        for (int g = 0; g < 2; g++) {
            f32x8 e;
#pragma unroll
            for (int x = 0; x < 8; x++) e[x] = s[8 * g + x];
            Parts3 pp;
            if constexpr (PP == 1) pp.p[0] = __builtin_convertvector(e, bf16x8);
            else pp = split3(e);
#pragma unroll
            for (int db = 0; db < NO; db++) {
                const lds_u8* at = vt + ((rb.v ^ (db << 6)) + 16 * g * G::kRow);
                s16x8 w;
                w.lo = lds_read_tr16_b64(at);
                w.hi = lds_read_tr16_b64(at + 8 * G::kRow);
                const bf16x8 a = __builtin_bit_cast(bf16x8, w);
#pragma unroll
                for (int x = PP - 1; x >= 0; x--) o[db] = mfma32(a, pp.p[x], o[db]);   // small products first
            }
        }
        if (more) {
            __builtin_amdgcn_s_waitcnt(0xC07F);   // (every V read has returned)
            __builtin_amdgcn_sched_barrier(0);
            request(vt, vb, t + KS, true);
        }
    }
    l_run = pair_sum(l_run);

    typedef __attribute__((address_space(3))) f32x4 lds_f4;
    typedef __attribute__((address_space(3))) f32x2 lds_f2;
    __syncthreads();   // every wave is done with its tiles
    constexpr int kShare = kMergeShare<32 * NO>;
    lds_u8* shares = (lds_u8*)csm;
#pragma unroll
    for (int db = 0; db < NO; db++)
#pragma unroll
        for (int g = 0; g < 4; g++)
            *(lds_f4*)(shares + wave * kShare + ((4 * db + g) * 64 + lane) * 16) =
                f32x4{o[db][4 * g], o[db][4 * g + 1], o[db][4 * g + 2], o[db][4 * g + 3]};
    *(lds_f2*)(shares + wave * kShare + NO * 4096 + lane * 8) = f32x2{m_run, l_run};
    __syncthreads();
    float w[KS], l = 0.f, m_all = NEG;
    f32x2 ml[KS];
#pragma unroll
    for (int t = 0; t < KS; t++) ml[t] = *(const lds_f2*)(shares + t * kShare + NO * 4096 + lane * 8);
    constexpr int kOwn = (4 * NO + KS - 1) / KS;   // groups of four channels a wave adds up
    f32x4 part[kOwn][KS];
#pragma unroll
    for (int i = 0; i < kOwn; i++)
#pragma unroll
        for (int t = 0; t < KS; t++)
            part[i][t] = *(const lds_f4*)(shares + t * kShare + (min(wave + i * KS, 4 * NO - 1) * 64 + lane) * 16);
#pragma unroll
    for (int t = 0; t < KS; t++) m_all = __builtin_fmaxf(m_all, ml[t][0]);
#pragma unroll
    for (int t = 0; t < KS; t++) {
        w[t] = ml[t][0] == NEG ? 0.f : fast_exp2((ml[t][0] - m_all) * to_log2);
        l = __builtin_fmaf(ml[t][1], w[t], l);
    }
    const float inv = __builtin_amdgcn_rcpf(l);
    ComposedSuspect<1> suspect;
#pragma unroll
    for (int i = 0; i < kOwn; i++) {
        const int gi = wave + i * KS;
        if (gi >= nch) break;
        f32x4 r = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < KS; t++)
#pragma unroll
            for (int x = 0; x < 4; x++) r[x] = __builtin_fmaf(part[i][t][x], w[t], r[x]);
        if constexpr (PP == 3) suspect.add(r);
        if (q_ok) composed_store4<PP == 1>(p, bh, qi, r, l, inv, 8 * gi + 4 * h);
    }
    if constexpr (PP == 3) {
        const bool redo = suspect(l) && q_ok;
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(redo) != 0, 0)) {
            __builtin_amdgcn_s_waitcnt(0);
            using ConstParams = const __attribute__((address_space(4))) ComposedParams;
            ConstParams* again = (ConstParams*)__builtin_amdgcn_kernarg_segment_ptr();
            int lane2 = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)), wave2 = wave, block = blockIdx.x;
            asm volatile("" : "+v"(lane2), "+s"(wave2), "+s"(block), "+s"(again));
            composed_redo<32 * NO, 1, KS, true>(*again, block, wave2, lane2, redo);
        }
    }
}

// out = sum over the splits of O 2^(m - max) / sum of l 2^(m - max), four channels a thread. HBM-bound: the
// partial sums are read once and the result is written once.
__global__ __launch_bounds__(256) void composed_merge_kernel(const ComposedParams p) {
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    const int d4 = p.dpad >> 2;
    const long row = i / d4;
    const int c = (int)(i - row * d4) * 4;
    if (row >= p.part_rows) return;
    const float to_log2 = composed_to_log2(p);
    float m = neg_inf(), l = 0.f;
    for (int t = 0; t < p.splits; t++) m = __builtin_fmaxf(m, p.part_ml[2 * (t * p.part_rows + row)]);
    f32x4 r = {0.f, 0.f, 0.f, 0.f};
    for (int t = 0; t < p.splits; t++) {
        const long at = t * p.part_rows + row;
        const f32x2 ml = *reinterpret_cast<const f32x2*>(p.part_ml + 2 * at);
        const float w = ml[0] == neg_inf() ? 0.f : fast_exp2((ml[0] - m) * to_log2);
        l = __builtin_fmaf(ml[1], w, l);
        const f32x4 o = *reinterpret_cast<const f32x4*>(p.part_o + at * p.dpad + c);
#pragma unroll
        for (int x = 0; x < 4; x++) r[x] = __builtin_fmaf(o[x], w, r[x]);
    }
    const long dst = (p.part_row0 + row) * p.d + c;
#pragma unroll
    for (int x = 0; x < 4; x++) {
        if (c + x >= p.d) continue;
        const float v = l == 0.f ? 0.f : r[x] / l;   // (no key: zeros; NaN stays)
        if (p.out_is_bf16) ((__bf16*)p.out)[dst + x] = (__bf16)v;
        else ((float*)p.out)[dst + x] = v;
    }
}

// The kernels' dynamic LDS limits, once per device.
template <int D, int PARTS, int KS, bool KV16>
hipError_t composed_attr() {
    constexpr int lds = composed_lds<D, PARTS, KS>();
    if (lds <= 64 * 1024) return hipSuccess;
    static std::atomic<unsigned long long> attr_done;
    return fv_set_max_lds_once((const void*)sdpa_composed_kernel<D, PARTS, KS, KV16>, lds, attr_done);
}
template <int NC, int PP, int KS, bool LOG2DOM>
hipError_t short_attr() {
    static std::atomic<unsigned long long> attr_done;
    return fv_set_max_lds_once((const void*)sdpa_short_kernel<NC, PP, KS, LOG2DOM>, short_lds<NC, KS>(), attr_done);
}

template <int D, int PARTS, int KS, bool KV16>
hipError_t launch_as(const ComposedParams& p, size_t bh, hipStream_t st) {
    constexpr int lds = composed_lds<D, PARTS, KS>();
    const hipError_t ae = composed_attr<D, PARTS, KS, KV16>();
    if (ae != hipSuccess) return ae;
    constexpr int rows = 32 * (composed_waves(KS) / KS);
    ComposedParams a = p;
    a.nqt = (p.sq + rows - 1) / rows;
    const size_t total = bh * (size_t)a.nqt;
    if (total > (size_t)INT_MAX - 8) return hipErrorInvalidValue;
    size_t items = total;
    if (KS == 1 && p.splits > 1) {
        items = (total - (size_t)p.full) * (size_t)p.splits;
        const int tiles = (p.sk + 31) / 32;
        a.split_tiles = (tiles + p.splits - 1) / p.splits;
        a.dpad = (p.d + 3) & ~3;
        a.part_row0 = (long)(p.full / a.nqt) * p.sq + (long)(p.full % a.nqt) * rows;
        a.part_rows = (long)bh * p.sq - a.part_row0;
    } else {
        a.full = 0, a.splits = 1;
    }
    a.total = (int)items;
    a.per_xcd = (int)((items + 7) / 8);
    a.by_head = !p.mask || p.mask_bh != 0;
    hipLaunchKernelGGL((sdpa_composed_kernel<D, PARTS, KS, KV16>), dim3((unsigned)(a.full + a.per_xcd * 8)), dim3(64 * composed_waves(KS)), lds, st, a);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess && a.splits > 1) {
        const size_t n = (size_t)a.part_rows * (size_t)(a.dpad / 4);
        hipLaunchKernelGGL(composed_merge_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, a);
        e = hipGetLastError();
    }
    return e;
}

template <int D>
hipError_t launch_d(const ComposedParams& p, int parts, bool kv16, int ks, size_t bh, hipStream_t st) {
    if (parts == 3) return ks == 1 ? launch_as<D, 3, 1, false>(p, bh, st) : launch_as<D, 3, 2, false>(p, bh, st);
    if (!kv16) return ks == 1 ? launch_as<D, 1, 1, false>(p, bh, st) : launch_as<D, 1, 2, false>(p, bh, st);
    if (ks == 1) return launch_as<D, 1, 1, true>(p, bh, st);
    if constexpr (D <= 96) {
        if (ks == 4) return launch_as<D, 1, 4, true>(p, bh, st);
        if (ks == 8) return launch_as<D, 1, 8, true>(p, bh, st);
    }
    return launch_as<D, 1, 2, true>(p, bh, st);
}
template <int NC, int PP, int KS, bool LOG2DOM>
hipError_t launch_short_as(const ComposedParams& p, size_t bh, hipStream_t st) {
    constexpr int lds = short_lds<NC, KS>();
    const hipError_t e = short_attr<NC, PP, KS, LOG2DOM>();
    if (e != hipSuccess) return e;
    if (LOG2DOM) fv_internal_count_log2_domain();
    ComposedParams a = p;
    a.nqt = (p.sq + 31) / 32;
    a.full = 0, a.splits = 1;
    const size_t total = bh * (size_t)a.nqt;
    if (total > ((size_t)1 << 22)) return hipErrorInvalidValue;   // (2^32 work-items a launch)
    a.total = (int)total;
    a.per_xcd = (int)((total + 7) / 8);
    a.by_head = !p.mask || p.mask_bh != 0;
    hipLaunchKernelGGL((sdpa_short_kernel<NC, PP, KS, LOG2DOM>), dim3((unsigned)(a.per_xcd * 8)), dim3(64 * KS), lds, st, a);
    return hipGetLastError();
}
template <int NC, int PP>
hipError_t launch_short_nc(const ComposedParams& p, int waves, size_t bh, hipStream_t st) {
    if constexpr (PP == 1) {
        if (fv_sdpa_is_log2_domain_scale(p.scale))
            return waves == 8 ? launch_short_as<NC, PP, 8, true>(p, bh, st) : launch_short_as<NC, PP, 4, true>(p, bh, st);
    }
    return waves == 8 ? launch_short_as<NC, PP, 8, false>(p, bh, st) : launch_short_as<NC, PP, 4, false>(p, bh, st);
}
template <int PP>
hipError_t launch_short(const ComposedParams& p, int waves, size_t bh, hipStream_t st) {
    if (p.d <= 64) return launch_short_nc<4, PP>(p, waves, bh, st);
    if constexpr (PP == 3) {
        if (p.d <= 80) return launch_short_nc<5, PP>(p, waves, bh, st);
        if (p.d <= 96) return launch_short_nc<6, PP>(p, waves, bh, st);
        if (p.d <= 112) return launch_short_nc<7, PP>(p, waves, bh, st);
    }
    return launch_short_nc<8, PP>(p, waves, bh, st);
}

hipError_t first_error(std::initializer_list<hipError_t> all) {
    for (const hipError_t e : all)
        if (e != hipSuccess) return e;
    return hipSuccess;
}
template <int D>
hipError_t init_composed_d() {   // (launch_d)
    hipError_t e = first_error({composed_attr<D, 3, 1, false>(), composed_attr<D, 3, 2, false>(), composed_attr<D, 1, 1, false>(),
                                composed_attr<D, 1, 2, false>(), composed_attr<D, 1, 1, true>(), composed_attr<D, 1, 2, true>()});
    if constexpr (D <= 96)
        if (e == hipSuccess) e = first_error({composed_attr<D, 1, 4, true>(), composed_attr<D, 1, 8, true>()});
    return e;
}
template <int NC, int PP>
hipError_t init_short_nc() {
    hipError_t e = first_error({short_attr<NC, PP, 4, false>(), short_attr<NC, PP, 8, false>()});
    if constexpr (PP == 1)
        if (e == hipSuccess) e = first_error({short_attr<NC, PP, 4, true>(), short_attr<NC, PP, 8, true>()});
    return e;
}
}  // namespace
}  // namespace fv

extern "C" hipError_t fv_internal_init_composed(void) {
    using namespace fv;
    return first_error({init_composed_d<32>(), init_composed_d<64>(), init_composed_d<96>(), init_composed_d<128>(),
                        init_short_nc<4, 1>(), init_short_nc<8, 1>(), init_short_nc<4, 3>(), init_short_nc<5, 3>(),
                        init_short_nc<6, 3>(), init_short_nc<7, 3>(), init_short_nc<8, 3>()});
}

// Query tiles (128 queries) past a multiple of the CUs hold up the launch for a whole walk of the keys while other CUs
// have none left: they are shared out by key ranges, in as many as fill the CUs best, where that saves more than writing
// and merging the partial sums costs (a quarter above the estimate). A 32-key tile of a workgroup that has its CU to
// itself takes 3.4 us at 128 channels. Measured on MI355X, a shared mask, uncut / cut, us: 12 x 4096 x 4096 x 128 (384 tiles:
// 256 + 128 x 2) 618 / 531, 24 x 3000 x 700 x 128 (576: 512 + 64 x 4) 187 / 151, 12 x 3000 x 1024 x 128 (288) 159 / 131,
// 24 x 3000 x 800 x 80 (576) 158 / 124, 12 x 4096 x 1024 x 64 (384) 94 / 84; a mask per head, 64 x 700 x 700 x 128 (384)
// 122 / 110, 64 x 600 x 900 x 80 (320) 112 / 97. Where the rule leaves a launch whole the key walk is too short for the
// merge (12 x 4096 x 300 x 128, 60) or the rest fills the CUs (24 x 2600 x 1000 x 128: 248 of 256 tiles). Launches of one
// part are not cut: a tile costs them a third of that, and the same merge.
fv::ComposedPlan fv_composed_plan(size_t bh, size_t sq, size_t sk, size_t d) {
    const size_t cus = (size_t)fv_compute_units(), groups = bh * ((sq + 31) / 32), total = bh * ((sq + 127) / 128);
    const size_t full = total / cus * cus, rest = total - full, tiles = (sk + 31) / 32;
    if (d < 1 || d > 128 || bh > 65535 || sk == 0 || sq > (size_t)INT_MAX - 256 || sk > (size_t)INT_MAX - 256 ||
        groups < 1024 || full == 0 || rest == 0 || cus % 8 != 0 || total > (size_t)INT_MAX / 16)
        return {0, 1, 0};
    const size_t nqt = (sq + 127) / 128, rows = bh * sq - (full / nqt * sq + full % nqt * 128), dpad = (d + 3) & ~(size_t)3;
    const double tile_us = 3.4 * (double)((d + 31) / 32) / 4.0;
    size_t best = 1, best_bytes = 0;
    double best_gain = 0.0;
    for (size_t want = 2; want <= 8; want++) {
        const size_t per = (tiles + want - 1) / want, s = (tiles + per - 1) / per;
        if (per < 4 || s != want) continue;
        const size_t bytes = s * rows * (dpad + 2) * 4;
        const double walk = (double)((rest * s + cus - 1) / cus) * (double)per;
        const double gain = ((double)tiles - walk) * tile_us - 1.25 * (6.0 + 2.0 * (double)bytes / 4.0e6);
        if (gain > best_gain) best_gain = gain, best = s, best_bytes = bytes;
    }
    return {best > 1 ? full : 0, best, best_bytes};
}

extern "C" hipError_t fv_internal_launch_composed(const fv::ComposedParams* params, int kv_is_bf16, int round16, size_t bh,
                                                  hipStream_t st) {
    fv::ComposedParams p = *params;
    const int d = p.d;
    if (d < 1 || d > 128 || p.sk > INT_MAX - 256 || p.sq > INT_MAX - 256) return hipErrorInvalidValue;
    // A launch holds fewer than 2^32 work-items: heads in several where their query tiles are more (a tail is not cut there).
    const size_t tiles = ((size_t)p.sq + 127) / 128, most = ((size_t)1 << 24) - 8;
    if (bh > 1 && bh > most / (tiles ? tiles : 1)) {
        const size_t heads = most / tiles ? most / tiles : 1;
        for (size_t h0 = 0; h0 < bh; h0 += heads) {
            fv::ComposedParams part = *params;
            const size_t qe = h0 * (size_t)p.sq * d, ke = h0 * (size_t)p.sk * d * (kv_is_bf16 ? 2 : 4);
            part.q = (const char*)p.q + qe * (p.q_is_bf16 ? 2 : 4);
            part.k = (const char*)p.k + ke, part.v = (const char*)p.v + ke;
            part.out = (char*)p.out + qe * (p.out_is_bf16 ? 2 : 4);
            if (p.mask) part.mask = p.mask + (long)h0 * p.mask_bh;
            part.full = 0, part.splits = 1, part.part_o = nullptr;
            const hipError_t e = fv_internal_launch_composed(&part, kv_is_bf16, round16, heads < bh - h0 ? heads : bh - h0, st);
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    }
    const uintptr_t any = (uintptr_t)p.q | (uintptr_t)p.k | (uintptr_t)p.v | (uintptr_t)p.out;
    p.vec = (any & 15) == 0 && d % 8 == 0;
    const int parts = kv_is_bf16 || round16 ? 1 : 3;
    // 1024 groups are one wave on every SIMD of the chip: below two waves (one with three parts, whose second share of
    // the tiles leaves room for one workgroup per CU) the keys are shared out over a workgroup's waves. bf16 keys, us with 1 /
    // 2 / 4 / 8 shares: 64 x 1024 x 300 x 80 (2048 groups) 33 / 39 / 56 / 83, 64 x 512 x 512 x 64 (1024) 28 / 24 / 27 / 38. Four and
    // eight are left for what the short kernel (below) does not take: f32 queries on bf16 keys 16 x 257 x 257 x 80 (144) 15.9 /
    // 12.4 / 10.4 / 9.6, 24 x 300 x 300 x 80 (240) 17.2 / 12.6 / 10.8 / 10.0, 24 x 500 x 500 x 80 (384) 24.3 / 17.3 / 16.5 / 20.5;
    // rows that are no whole 16-byte units 16 x 257 x 257 x 76 40.0 / 32.0 / 34.5 / 28.7, 12 x 500 x 500 x 76 (192) 63.5 / 46.1 / 44.3 / 30.9,
    // 12 x 200 x 200 x 60 (84) 21.4 / 20.0 / 18.2 / 14.5, 24 x 500 x 500 x 76 64 / 47 / 51 / 59; unaligned ones 24 x 300 x 300 x 80 46.7
    // / 34.5 / 37.1 / 34.4, 24 x 500 x 500 x 80 67 / 49 / 57 / 69 (the line does not follow the alignment). Three parts, 1 / 2
    // shares: 64 x 3000 x 700 x 80 (6016) 284 / 331, 12 x 4096 x 4096 x 128 (1536) 606 / 1459, 24 x 1024 x 1024 x 64 (768) 71 / 62. Four
    // and eight shares take the registers of whole tiles in flight: bf16 keys up to 96 channels only (f32 keys, 12 x 700 x 700 x
    // 112: 39 / 29 / 61, with spills).
    // Between 1024 and 2047 groups, bf16, one / two shares: 12 x 4096 x 4096 x 64 (1536) 189 / 158, 64 x 700 x 700 x 64
    // (1408) 41.5 / 34.5, 40 x 1000 x 300 x 80 (1280) 26.4 / 23.9, 12 x 3000 x 1024 x 64 (1128) 53.2 / 43.6; but at 128
    // channels (two shares stage every tile for half as many queries) 12 x 4096 x 4096 (1536) 264 / 283, 24 x
    // 2000 x 2000 (1512) 142 / 151, 12 x 4000 x 300 (1500) 33.4 / 37.2: the line does not follow the head dim.
    int ks = 1;
    const size_t groups = bh * (size_t)((p.sq + 31) / 32);   // 32-query groups
    // bf16 operands in whole 16-byte units: the short kernel, eight waves a query group while each has a CU to itself, four
    // while they are about one resident round. us, that / the kernels below: 16 x 257 x 257 x 80 (144 groups) 7.8 / 10.2,
    // 12 x 111 x 111 x 128 under a mask (48) 7.5 / 12.5, 16 x 1000 x 1000 x 80 (512) 22.9 / 29.5, 24 x 512 x 512 x 128 under
    // a mask (384) 17.4 / 24.4; past two a CU, up to 64 channels (half the registers and LDS) 24 x 1024 x 1024 x 64 (768)
    // 27.7 / 37.4, 64 x 512 x 512 x 64 with a mask per head (1024) 22.3 / 24.4, past 96 (whole LDS rows) 12 x 1500 x 1500 x
    // 112 (564) 52.6 / 64.8, 32 x 1000 x 1000 x 112 (1024) 46.4 / 49.4; between them 24 x 900 x 900 x 80 (696) 34.8 / 34.8,
    // 64 x 300 x 300 x 80 under a mask (640) 18.6 / 18.1.
    const size_t cus = (size_t)fv_compute_units(), most_short = (d <= 64 || d > 96 ? 4 : 2) * cus;
    if (p.vec && kv_is_bf16 && p.q_is_bf16 && groups <= most_short) {
        p.q_plane = (long)p.sq * d, p.k_plane = p.v_plane = (long)p.sk * d;
        return fv::launch_short<3>(p, groups <= cus ? 8 : 4, bh, st);
    }
    if (groups < (parts == 3 ? 1024 : 2048)) ks = 2;
    if (groups < 512) ks = 4;
    if (groups <= 256 && p.sk > 256) ks = 8;
    if (parts != 3 || !p.part_o) p.full = 0, p.splits = 1;   // (a plan has at least 1024 groups: ks is 1)
    if (d <= 32) return fv::launch_d<32>(p, parts, kv_is_bf16 != 0, ks, bh, st);
    if (d <= 64) return fv::launch_d<64>(p, parts, kv_is_bf16 != 0, ks, bh, st);
    if (d <= 96) return fv::launch_d<96>(p, parts, kv_is_bf16 != 0, ks, bh, st);
    return fv::launch_d<128>(p, parts, kv_is_bf16 != 0, ks, bh, st);
}

// The same for the plans of the fused kernels: P rounded to bf16, no mask (fv_short_waves).
extern "C" hipError_t fv_internal_launch_short(const fv::ComposedParams* p, int waves, size_t bh, hipStream_t st) {
    if (p->d != 64 && p->d != 128) return hipErrorInvalidValue;
    return fv::launch_short<1>(*p, waves, bh, st);
}
