// Video Sparse Attention stages for gfx950: tile mean, coarse scores, coarse
// softmax x V, bitwise-descent top-k, tile permute, block-sparse fine attention,
// gated combine. Reference stages: crates/fastvideo-cudarc/src/rt/vsa.rs:358-470
// and the kernels cited per function below (kernels/core.cu, kernels/attn3.cu).
#include <algorithm>

#include "attn_core.h"
#include "fv_internal.h"

namespace fv {

constexpr int kTileElems = 64;   // VSA cube = 4x4x4 tokens (rt/vsa.rs:29-31)

// ---- tile mean (kernels/core.cu:550-570, kernels/attn3.cu:208-226) --------------
// One 32-lane group per tile, 4 consecutive d per lane; the sum runs over the
// tile's real tokens in slot order with one f32 add per token, then / n — the
// same order and operations as the reference, so the result is bit-identical
// to its host restatement.
template <bool IN_BF16>
FV_DEV void tile_mean_body(const void* __restrict__ x, const int* __restrict__ slot_src,
                           const int* __restrict__ block_sizes, float* __restrict__ out, long seq, int dim,
                           int num_tiles, int round16) {
    const int grp = threadIdx.x >> 5, ln = threadIdx.x & 31;
    const int tile = blockIdx.x * 8 + grp;
    const long bh = blockIdx.y;
    if (tile >= num_tiles) return;
    const int n = block_sizes[tile];
    // slot_src == null: x is already tile-ordered, slot j of the tile is row tile*64 + j
    const int* src = slot_src ? slot_src + (long)tile * kTileElems : nullptr;
    const long row0 = (long)tile * kTileElems;
    float* ob = out + (bh * num_tiles + tile) * (long)dim;
    auto load_tok = [&](long tok, int d0) -> f32x4 {
        f32x4 v;
        if constexpr (IN_BF16) {
            const u32x2 raw = *reinterpret_cast<const u32x2*>(
                (const uint16_t*)x + (bh * seq + tok) * dim + d0);
            v[0] = __builtin_bit_cast(float, raw[0] << 16);
            v[1] = __builtin_bit_cast(float, raw[0] & 0xffff0000u);
            v[2] = __builtin_bit_cast(float, raw[1] << 16);
            v[3] = __builtin_bit_cast(float, raw[1] & 0xffff0000u);
        } else {
            v = *reinterpret_cast<const f32x4*>((const float*)x + (bh * seq + tok) * dim + d0);
            if (round16) {
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] = bf16_bits_to_f32(bf16_rne_bits(v[e]));
            }
        }
        return v;
    };
    for (int d0 = ln * 4; d0 < dim; d0 += 128) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        int j = 0;
        // eight loads in flight, then their adds in slot order (the order is the contract)
        for (; j + 8 <= n; j += 8) {
            f32x4 v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = load_tok(src ? src[j + u] : row0 + j + u, d0);
#pragma unroll
            for (int u = 0; u < 8; u++)
#pragma unroll
                for (int e = 0; e < 4; e++) acc[e] = __fadd_rn(acc[e], v[u][e]);
        }
        for (; j < n; j++) {
            const f32x4 v = load_tok(src ? src[j] : row0 + j, d0);
#pragma unroll
            for (int e = 0; e < 4; e++) acc[e] = __fadd_rn(acc[e], v[e]);
        }
        f32x4 r;
#pragma unroll
        for (int e = 0; e < 4; e++) r[e] = n > 0 ? __fdiv_rn(acc[e], (float)n) : 0.0f;
        *reinterpret_cast<f32x4*>(ob + d0) = r;
    }
}

template <bool IN_BF16>
__global__ __launch_bounds__(256) void vsa_tile_mean_kernel(
    const void* __restrict__ x, const int* __restrict__ slot_src,
    const int* __restrict__ block_sizes, float* __restrict__ out, long seq, int dim,
    int num_tiles, int round16) {
    tile_mean_body<IN_BF16>(x, slot_src, block_sizes, out, seq, dim, num_tiles, round16);
}
// ---- tile pass and tile means in one scan (the whole op; rt/vsa.rs:378-384 and 406-414) ----------------
// dim == 128. 16 lanes per tile, a lane owns 8 consecutive d of every slot: it reads the slot's 16 (bf16) or 32
// (f32) bytes, writes them as bf16 (RNE) to the tile-ordered copy if there is one (zeros for padding slots), and adds
// them in f32, in slot order over the tile's real tokens, to its share of the mean: the same values in the same
// order as vsa_tile_mean_kernel, so the means (and the selection that follows from them) are bit-identical.
// slot_src == null: x is already tile-ordered. Eight slots in flight per lane. (Measured and not kept: the tile's 64
// slot indices fetched once and handed round the 16-lane row, the next batch's rows requested before a batch is
// stored and added: 124 registers and 10 % slower.)
struct ThreeScan {
    const void* in[3];
    uint16_t* tiles[3];   // null: no copy wanted
    float* means[3];
    float mul[3];         // f32 operands: factor on the values of the copy before their one rounding (1 = none);
                          // the means pool the operand as it is
};
template <bool IN_BF16>
__global__ __launch_bounds__(256) void vsa_tile_scan3_kernel(ThreeScan t, const int* __restrict__ slot_src,
                                                             const int* __restrict__ block_sizes, long seq, long padded,
                                                             int num_tiles) {
    constexpr int kDim = 128;
    const int grp = threadIdx.x >> 4, c = threadIdx.x & 15;
    const int tile = blockIdx.x * 16 + grp;
    if (tile >= num_tiles) return;
    const long bh = blockIdx.y;
    const void* __restrict__ x = t.in[blockIdx.z];
    uint16_t* __restrict__ xt = t.tiles[blockIdx.z];
    const int n = block_sizes[tile];
    const long row0 = (long)tile * kTileElems;
    const int* src = slot_src ? slot_src + row0 : nullptr;
    float acc[8];
#pragma unroll
    for (int e = 0; e < 8; e++) acc[e] = 0.f;
    for (int j = 0; j < kTileElems; j += 8) {
        float v[8][8];
        u32x4 packed[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const long tok = src ? (long)src[j + u] : row0 + j + u;
            const bool real = tok >= 0;
            if constexpr (IN_BF16) {
                u32x4 raw = {0u, 0u, 0u, 0u};
                if (real) raw = *reinterpret_cast<const u32x4*>((const uint16_t*)x + (bh * seq + tok) * kDim + c * 8);
                packed[u] = raw;
#pragma unroll
                for (int w = 0; w < 4; w++) {
                    v[u][2 * w] = __builtin_bit_cast(float, raw[w] << 16);
                    v[u][2 * w + 1] = __builtin_bit_cast(float, raw[w] & 0xffff0000u);
                }
            } else {
                f32x4 a = {0.f, 0.f, 0.f, 0.f}, b = a;
                if (real) {
                    const float* px = (const float*)x + (bh * seq + tok) * kDim + c * 8;
                    a = *reinterpret_cast<const f32x4*>(px);
                    b = *reinterpret_cast<const f32x4*>(px + 4);
                }
#pragma unroll
                for (int w = 0; w < 4; w++) v[u][w] = a[w], v[u][4 + w] = b[w];
                if (xt) {
                    const float m = t.mul[blockIdx.z];
#pragma unroll
                    for (int w = 0; w < 4; w++)
                        packed[u][w] = bf16_rne_bits(v[u][2 * w] * m) | ((unsigned)bf16_rne_bits(v[u][2 * w + 1] * m) << 16);
                }
            }
        }
        if (xt) {
#pragma unroll
            for (int u = 0; u < 8; u++)
                *reinterpret_cast<u32x4*>(xt + (bh * padded + row0 + j + u) * kDim + c * 8) = packed[u];
        }
#pragma unroll
        for (int u = 0; u < 8; u++) {
            if (j + u < n) {   // uniform over the tile's 16 lanes
#pragma unroll
                for (int e = 0; e < 8; e++) acc[e] = __fadd_rn(acc[e], v[u][e]);
            }
        }
    }
    float* ob = t.means[blockIdx.z] + (bh * num_tiles + tile) * (long)kDim + c * 8;
    f32x4 r0, r1;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        r0[e] = n > 0 ? __fdiv_rn(acc[e], (float)n) : 0.0f;
        r1[e] = n > 0 ? __fdiv_rn(acc[4 + e], (float)n) : 0.0f;
    }
    *reinterpret_cast<f32x4*>(ob) = r0;
    *reinterpret_cast<f32x4*>(ob + 4) = r1;
}

// The same scan for bf16 operands that want their tile-ordered copy, one wave per tile: the wave reads the tile's 64
// rows as whole 256-byte rows, four consecutive slots (1 KB, contiguous where the slots' tokens are) per load
// instruction, all 16 in flight; writes them to the copy the same way and to 16 KB of LDS; then lane c adds word c
// (two d) of every real slot in slot order. Same values, same order: means bit-identical to the kernel above.
// 99 - 108 us at 12 x 32768 / 32760 tokens x 3 operands where the 16-lanes-per-tile form takes 126 - 136 (its loads
// touch four tiles, 256 bytes each, per instruction); for pooling alone (no copy) that form is the faster one.
__global__ __launch_bounds__(64) void vsa_tile_scan3_staged_kernel(ThreeScan t, const int* __restrict__ slot_src,
                                                                   const int* __restrict__ block_sizes, long seq,
                                                                   long padded, int num_tiles) {
    __shared__ __attribute__((aligned(16))) unsigned stage[kTileElems * 64];   // 64 rows x 64 words
    const int lane = threadIdx.x;
    const int tile = blockIdx.x;
    const long bh = blockIdx.y;
    const uint16_t* __restrict__ x = (const uint16_t*)t.in[blockIdx.z];
    uint16_t* __restrict__ xt = t.tiles[blockIdx.z];
    const long row0 = (long)tile * kTileElems;
    const int n = block_sizes[tile];
    const int my_tok = slot_src ? slot_src[row0 + lane] : (int)(row0 + lane);   // lane = slot
    const int c = lane & 15;
    u32x4 v[16];
#pragma unroll
    for (int it = 0; it < 16; it++) {
        const int slot = it * 4 + (lane >> 4);
        const int tok = __shfl(my_tok, slot);
        v[it] = u32x4{0u, 0u, 0u, 0u};
        if (tok >= 0) v[it] = *reinterpret_cast<const u32x4*>(x + (bh * seq + tok) * 128 + c * 8);
    }
#pragma unroll
    for (int it = 0; it < 16; it++) {
        const int slot = it * 4 + (lane >> 4);
        *reinterpret_cast<u32x4*>(xt + (bh * padded + row0 + slot) * 128 + c * 8) = v[it];
        *reinterpret_cast<u32x4*>(&stage[slot * 64 + c * 4]) = v[it];
    }
    __syncthreads();   // one wave: orders its LDS writes before the reads below
    float a0 = 0.f, a1 = 0.f;
#pragma unroll 8
    for (int j = 0; j < kTileElems; j++) {
        const unsigned w = stage[j * 64 + lane];
        if (j < n) {
            a0 = __fadd_rn(a0, __builtin_bit_cast(float, w << 16));
            a1 = __fadd_rn(a1, __builtin_bit_cast(float, w & 0xffff0000u));
        }
    }
    float* ob = t.means[blockIdx.z] + (bh * num_tiles + tile) * 128L + lane * 2;
    float2 r;
    r.x = n > 0 ? __fdiv_rn(a0, (float)n) : 0.0f;
    r.y = n > 0 ? __fdiv_rn(a1, (float)n) : 0.0f;
    *reinterpret_cast<float2*>(ob) = r;
}

// ... and for f32 operands: the tile in two halves of 32 slots (16 KB of f32 each), two consecutive slots per load
// instruction; the copy is rounded to bf16 (RNE), the sums take the unrounded values, lane c owning d = c and c + 64.
__global__ __launch_bounds__(64) void vsa_tile_scan3_staged_f32_kernel(ThreeScan t, const int* __restrict__ slot_src,
                                                                       const int* __restrict__ block_sizes, long seq,
                                                                       long padded, int num_tiles) {
    __shared__ __attribute__((aligned(16))) unsigned stage[32 * 128];   // 32 rows x 128 words
    const int lane = threadIdx.x;
    const int tile = blockIdx.x;
    const long bh = blockIdx.y;
    const float* __restrict__ x = (const float*)t.in[blockIdx.z];
    uint16_t* __restrict__ xt = t.tiles[blockIdx.z];
    const long row0 = (long)tile * kTileElems;
    const int n = block_sizes[tile];
    const int my_tok = slot_src ? slot_src[row0 + lane] : (int)(row0 + lane);   // lane = slot
    const int c = lane & 31;
    const float mul = t.mul[blockIdx.z];   // x * 1.0f is x
    float a0 = 0.f, a1 = 0.f;
    u32x4 v[2][16];
    auto load_half = [&](int half, u32x4 (&r)[16]) {
#pragma unroll
        for (int it = 0; it < 16; it++) {
            const int slot = 32 * half + it * 2 + (lane >> 5);
            const int tok = __shfl(my_tok, slot);
            r[it] = u32x4{0u, 0u, 0u, 0u};
            if (tok >= 0) r[it] = *reinterpret_cast<const u32x4*>(x + (bh * seq + tok) * 128 + c * 4);
        }
    };
    load_half(0, v[0]);
#pragma unroll
    for (int half = 0; half < 2; half++) {
        if (half == 0) load_half(1, v[1]);   // in flight while the first half is stored and added
#pragma unroll
        for (int it = 0; it < 16; it++) {
            const int sl = it * 2 + (lane >> 5);
            const u32x4 w = v[half][it];
            // (the vector cast as a whole: __builtin_bit_cast(float, w[i]) read element 0 for every i with hipcc 7.2)
            const f32x4 f = __builtin_bit_cast(f32x4, w);
            u32x2 packed;
            packed[0] = bf16_rne_bits(f[0] * mul) | ((unsigned)bf16_rne_bits(f[1] * mul) << 16);
            packed[1] = bf16_rne_bits(f[2] * mul) | ((unsigned)bf16_rne_bits(f[3] * mul) << 16);
            *reinterpret_cast<u32x2*>(xt + (bh * padded + row0 + 32 * half + sl) * 128 + c * 4) = packed;
            *reinterpret_cast<u32x4*>(&stage[sl * 128 + c * 4]) = w;
        }
        __syncthreads();   // one wave: orders its LDS writes before the reads below
#pragma unroll 8
        for (int j = 0; j < 32; j++) {
            const float w0 = __builtin_bit_cast(float, stage[j * 128 + lane]);
            const float w1 = __builtin_bit_cast(float, stage[j * 128 + 64 + lane]);
            if (32 * half + j < n) {
                a0 = __fadd_rn(a0, w0);
                a1 = __fadd_rn(a1, w1);
            }
        }
        __syncthreads();   // ... and the reads before the next half's writes
    }
    float* ob = t.means[blockIdx.z] + (bh * num_tiles + tile) * 128L;
    ob[lane] = n > 0 ? __fdiv_rn(a0, (float)n) : 0.0f;
    ob[64 + lane] = n > 0 ? __fdiv_rn(a1, (float)n) : 0.0f;
}

// ---- coarse scores (rt/vsa.rs:385-388; arithmetic of the host oracle, rt/vsa.rs:185-189) ----
// scores[bh, qt, kt] = f32( (f64 dot of the tile means, d ascending from -0.0) * f64(scale) ).
// The product of two f32 values is exact in f64, so one v_fma_f64 per term is the oracle's
// multiply-then-add, and the scores (and with them the selected tiles) equal the host oracle's
// bit for bit. (The reference's device path runs cuBLAS f32 here, whose order is unspecified.)
// A 64 x 64 block of scores per workgroup, 4 x 4 per thread, the means staged in LDS as f32.
__global__ __launch_bounds__(256) void vsa_coarse_scores_kernel(
    const float* __restrict__ qc, const float* __restrict__ kc, float* __restrict__ scores,
    int nb, int dim, float scale) {
    __shared__ float qs[32][65];   // [d][tile]: the 4 tiles of a thread are consecutive words
    __shared__ float ks[32][65];
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    const int q0 = blockIdx.y * 64, k0 = blockIdx.x * 64;
    const long bh = blockIdx.z;
    const float* qb = qc + bh * nb * (long)dim;
    const float* kb = kc + bh * nb * (long)dim;
    double acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = -0.0;   // the identity of Rust's f64 Sum
    for (int d0 = 0; d0 < dim; d0 += 32) {
        for (int e = threadIdx.x; e < 64 * 32; e += 256) {
            const int r = e >> 5, c = e & 31;
            qs[c][r] = (q0 + r < nb && d0 + c < dim) ? qb[(long)(q0 + r) * dim + d0 + c] : 0.f;
            ks[c][r] = (k0 + r < nb && d0 + c < dim) ? kb[(long)(k0 + r) * dim + d0 + c] : 0.f;
        }
        __syncthreads();
        const int dn = min(32, dim - d0);
        for (int c = 0; c < dn; c++) {
            double a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; i++) a[i] = (double)qs[c][ty * 4 + i];
#pragma unroll
            for (int j = 0; j < 4; j++) b[j] = (double)ks[c][tx * 4 + j];
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) acc[i][j] = __builtin_fma(a[i], b[j], acc[i][j]);
        }
        __syncthreads();
    }
    const double sc = (double)scale;
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int qi = q0 + ty * 4 + i, kj = k0 + tx * 4 + j;
            if (qi < nb && kj < nb) scores[(bh * nb + qi) * (long)nb + kj] = (float)(acc[i][j] * sc);
        }
}

// ---- coarse softmax x V (rt/vsa.rs:389-393, kernels/core.cu:177-252) ---------------
// coarse[bh, qt, :] = softmax(scores[bh, qt, :]) vc[bh]; eight query tiles per block
// share every vc row they read. dim = 128.
constexpr int kCoarseRows = 8;
__global__ __launch_bounds__(256) void vsa_coarse_pv_kernel(
    const float* __restrict__ scores, const float* __restrict__ vc, float* __restrict__ coarse,
    int nb) {
    extern __shared__ __attribute__((aligned(16))) float p_lds[];   // [kCoarseRows][nbp], rows 16-byte aligned
    __shared__ float red[kCoarseRows][4];
    __shared__ float stat[kCoarseRows];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int q0 = blockIdx.x * kCoarseRows;
    const long bh = blockIdx.y;
    const int rows = min(kCoarseRows, nb - q0);
    const int nbp = (nb + 3) & ~3;
    const float* sb = scores + (bh * nb + q0) * (long)nb;
    for (int r = 0; r < rows; r++)
        for (int j = tid; j < nb; j += 256) p_lds[r * nbp + j] = sb[(long)r * nb + j];
    __syncthreads();
    // row max
    for (int r = 0; r < rows; r++) {
        float m = neg_inf();
        for (int j = tid; j < nb; j += 256) m = fmaxf(m, p_lds[r * nbp + j]);
        for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
        if (lane == 0) red[r][wave] = m;
    }
    __syncthreads();
    if (tid < rows) stat[tid] = fmaxf(fmaxf(red[tid][0], red[tid][1]), fmaxf(red[tid][2], red[tid][3]));
    __syncthreads();
    for (int r = 0; r < rows; r++) {
        const float m = stat[r];
        float s = 0.f;
        for (int j = tid; j < nb; j += 256) {
            const float e = expf(p_lds[r * nbp + j] - m);
            p_lds[r * nbp + j] = e;
            s += e;
        }
        for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
        if (lane == 0) red[r][wave] = s;
    }
    __syncthreads();
    if (tid < rows) stat[tid] = 1.0f / (red[tid][0] + red[tid][1] + red[tid][2] + red[tid][3]);
    __syncthreads();
    // each half-block owns four rows; lane d accumulates over all key tiles in ascending order, four
    // vc rows in flight per step and the four weights of a row in one 16-byte LDS read
    constexpr int kOwn = kCoarseRows / 2;
    const int d = tid & 127, rh = tid >> 7;
    const float* vb = vc + bh * nb * 128L + d;
    const float* pr = p_lds + (kOwn * rh) * nbp;
    float a[kOwn];
#pragma unroll
    for (int r = 0; r < kOwn; r++) a[r] = 0.f;
    int kt = 0;
    for (; kt + 4 <= nb; kt += 4) {
        float vv[4];
#pragma unroll
        for (int u = 0; u < 4; u++) vv[u] = vb[(long)(kt + u) * 128];
#pragma unroll
        for (int r = 0; r < kOwn; r++) {
            const f32x4 p4 = *reinterpret_cast<const f32x4*>(pr + r * nbp + kt);
#pragma unroll
            for (int u = 0; u < 4; u++) a[r] += p4[u] * vv[u];
        }
    }
    for (; kt < nb; kt++) {
        const float vv = vb[(long)kt * 128];
#pragma unroll
        for (int r = 0; r < kOwn; r++) a[r] += pr[r * nbp + kt] * vv;
    }
#pragma unroll
    for (int r = 0; r < kOwn; r++)
        if (kOwn * rh + r < rows) coarse[(bh * nb + q0 + kOwn * rh + r) * 128L + d] = a[r] * stat[kOwn * rh + r];
}

// ---- top-k (kernels/core.cu:576-619, kernels/attn3.cu:279-363) ----------------------
// Output contract: T = the k-th largest sortable key of the row; the indices whose key is
// above T in ascending order, then those equal to T in ascending order, k in all, zero padded
// (k > n: every index, then zeros). Integer work, bit-exact.
//
// One wave owns one row and keeps it in registers: lane l holds the keys of indices
// l, 64 + l, 128 + l, ... (KPL of them; slots past n hold key 0 and are never emitted).
// T is built bit by bit from the top: a bit stays set if at least k keys are >= the candidate.
// A count is the sum of the popcounts of KPL wave-wide compare masks, so it lands in a scalar
// register and the decision is a scalar branch: no LDS, no atomics, no barrier. The emit pass
// walks the registers in index order; a lane's output slot is the running total plus the number
// of set mask bits below it.
FV_DEV unsigned sortable_key(float x) {
    const unsigned u = __builtin_bit_cast(unsigned, x);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

constexpr int kTopkMaxN = 4096;
constexpr int kTopkRowsPerBlock = 4;

FV_DEV int lanes_below(unsigned long long m) {
    return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}

template <int KPL>
__global__ __launch_bounds__(64 * kTopkRowsPerBlock) void vsa_topk_kernel(const float* __restrict__ scores,
                                                                          unsigned* __restrict__ out, int rows,
                                                                          int n, int k, int* zero, int zeros) {
    for (int i = blockIdx.x * (64 * kTopkRowsPerBlock) + threadIdx.x; i < zeros; i += gridDim.x * (64 * kTopkRowsPerBlock)) zero[i] = 0;
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * kTopkRowsPerBlock + (threadIdx.x >> 6);
    if (row >= rows) return;   // the whole wave leaves; waves never meet at a barrier
    const float* s = scores + (long)row * n;
    unsigned key[KPL];
#pragma unroll
    for (int j = 0; j < KPL; j++) {
        const int i = 64 * j + lane;
        key[j] = i < n ? sortable_key(s[i]) : 0u;
    }
    unsigned t = 0u;           // k > n: threshold 0 lets every index through
    if (k <= n) {
#pragma unroll 1
        for (unsigned bit = 0x80000000u; bit != 0u; bit >>= 1) {
            const unsigned cand = t | bit;
            int at_least = 0;
#pragma unroll
            for (int j = 0; j < KPL; j++)
                at_least += __builtin_popcountll(__builtin_amdgcn_ballot_w64(key[j] >= cand));
            if (at_least >= k) t = cand;
        }
    }
    unsigned* dst = out + (long)row * k;
    int filled = 0;            // wave-uniform count of slots written so far
#pragma unroll
    for (int pass = 0; pass < 2; pass++) {
#pragma unroll
        for (int j = 0; j < KPL; j++) {
            const int i = 64 * j + lane;
            const bool take = i < n && (pass == 0 ? key[j] > t : key[j] == t);
            const unsigned long long m = __builtin_amdgcn_ballot_w64(take);
            const int pos = filled + lanes_below(m);
            if (take && pos < k) dst[pos] = (unsigned)i;
            filled += __builtin_popcountll(m);
        }
    }
    for (int pos = filled + lane; pos < k; pos += 64) dst[pos] = 0u;
}

// ---- tile permute (kernels/core.cu:1659-1672, kernels/attn3.cu:230-244) --------------
// [bh, seq, 128] -> tile-contiguous bf16 [bh, padded, 128]; padding slots are zero.
template <bool IN_BF16>
FV_DEV void tile_qkv_body(const void* __restrict__ x, const int* __restrict__ slot_src, uint16_t* __restrict__ xt,
                          long seq, long padded, int dim) {
    const long chunks = dim / 8;
    const long rem = blockIdx.x * 256L + threadIdx.x;
    if (rem >= padded * chunks) return;
    const long bh = blockIdx.y;
    const long slot = rem / chunks;
    const long c = rem - slot * chunks;
    const int src = slot_src[slot];
    u32x4 v = {0u, 0u, 0u, 0u};
    if (src >= 0) {
        if constexpr (IN_BF16) {
            v = *reinterpret_cast<const u32x4*>((const uint16_t*)x + (bh * seq + src) * dim + c * 8);
        } else {
            const float* px = (const float*)x + (bh * seq + src) * dim + c * 8;
            const f32x4 a = *reinterpret_cast<const f32x4*>(px);
            const f32x4 b = *reinterpret_cast<const f32x4*>(px + 4);
            v[0] = bf16_rne_bits(a[0]) | ((unsigned)bf16_rne_bits(a[1]) << 16);
            v[1] = bf16_rne_bits(a[2]) | ((unsigned)bf16_rne_bits(a[3]) << 16);
            v[2] = bf16_rne_bits(b[0]) | ((unsigned)bf16_rne_bits(b[1]) << 16);
            v[3] = bf16_rne_bits(b[2]) | ((unsigned)bf16_rne_bits(b[3]) << 16);
        }
    }
    *reinterpret_cast<u32x4*>(xt + (bh * padded + slot) * dim + c * 8) = v;
}
template <bool IN_BF16>
__global__ __launch_bounds__(256) void vsa_tile_qkv_kernel(const void* __restrict__ x,
                                                           const int* __restrict__ slot_src,
                                                           uint16_t* __restrict__ xt, long seq,
                                                           long padded, int dim) {
    tile_qkv_body<IN_BF16>(x, slot_src, xt, seq, padded, dim);
}

// ---- fine stage (kernels/core.cu:1029-1179) ---------------------------------------------
// One workgroup of two waves per (query tile, batch*head): online softmax over the selected key tiles in list order;
// key columns >= block_sizes[tile] are -inf. Both waves hold all 64 queries and share the keys out, 32 at a time, so
// each wave has a ring of its own, fed by its own LDS-DMA, and waits for nobody but its own loads until the end, where
// the two results are merged through LDS, every wave finishing 32 queries. The ring has five slots of 4 KB; 32 keys
// pass through it as four chunks (K: channels 0 - 63, then 64 - 127; V: keys 0 - 15, then 16 - 31), each requested into
// the slot its predecessor but four has just left: a whole step ahead of its use.
// Padding is left out. A selected tile of more than 32 keys is a step of each wave; one of up to 32 a step of one wave,
// the waves taking turns; two of up to 16 share a step. A query tile of up to 32 queries (whole op only: the stage entry
// writes the padding rows too) is walked for those 32 alone (NB = 1), and one wave finishes them.
// Workgroups in step (FinePace). A selection that is spread over the sequence reads K and V as many times as it
// has tiles a row (31 GB at 12 heads, 125 of 624 tiles), and what misses the 4 MB of an XCD's L2 comes at 6.8 TB/s
// however the kernel is scheduled. The workgroups resident on an XCD belong to one or two heads and walk their ascending lists
// from the front together, but drift apart; so a wave enters the next window of kPaceTiles key tiles (2 MB of K and V)
// only when half the waves of its gang, the workgroups that one XCD holds at a time, have entered the one before: lines that
// miss the L2s 107 -> 70 M of 191 on ragged tiles, 130 -> 92 M of 257 on full ones with a uniformly random selection.
// Measured on MI355X, 12 heads, 624 tiles, 125 selected, us: the form this replaces (a wave 32 queries, both waves on
// every key tile behind three barriers) / steps as above / in step: ragged tiles of 21 x 30 x 52 2400 / 2010 / 1650, full
// tiles with a uniformly random selection 2350 / 2430 / 2150, a banded one 2075 / 1900 / 1965. All waves instead of half
// of them: 2860, 3100 and 2820; windows of 48, 96 tiles with 7/8: 1900, 1720 (ragged).
constexpr int kFineSlot = 4096;
constexpr int kFineWave = 5 * kFineSlot;
constexpr int kFineLds = 2 * kFineWave;
struct FineState {
    float thr, off, l;   // rescale above thr (-inf: no finite score yet); P = 2^(sl2 s - off); the lane's share of the sum
};
// Two blocks of 16 keys: their first rows in the tile-ordered copies and how many of their keys count.
struct FineStep {
    int row_a, row_b, valid_a, valid_b;
    bool none;
};

// How far the waves of a gang have got: counters[w] of them have entered window w or a later one. Only a hint: no result
// depends on it, a wave that has polled kPaceTries times (about 30 us) stops asking, and the atomics are those of one
// workgroup's scope, which are carried out in the L2 that the gang shares (agent scope, past the L2s: 4.7 ms a launch).
constexpr int kPaceTiles = 64, kPaceTries = 30;
struct FinePace {
    int* counters;   // null: no pace is kept
    int half;        // of the gang's waves
    int window;      // the one this wave has entered
    bool asks;
    FV_DEV void enter(int w, int lane) {
        if (lane == 0)
            for (int x = window + 1; x <= w; x++) __hip_atomic_fetch_add(counters + x, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        window = w;
    }
    FV_DEV void wait(int lane) {
        for (int tries = 0; asks; tries++) {
            int n = 0;
            asm volatile("" : "+v"(n));   // (an addition of nothing, not a load: that may come from the L1)
            if (lane == 0) n = __hip_atomic_fetch_add(counters + window - 1, n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            if (__builtin_amdgcn_readfirstlane(n) >= half) break;
            if (tries == kPaceTries) asks = false;
            __builtin_amdgcn_s_sleep(16);
        }
    }
};

template <int NB>
FV_DEV void fine_item(const VsaFineParams& p, lds_u8* smem, const int wave, const int lane, const int bh, const int qtile,
                      FinePace pace) {
    lds_u8* ring = smem + wave * kFineWave;
    const int h = lane >> 5, c32 = lane & 31;
    const int nb = p.num_tiles, topk = p.topk;
    const size_t padded = (size_t)nb * kTileElems;
    const char* kb = (const char*)(p.kt + (size_t)bh * padded * 128);
    const char* vb = (const char*)(p.vt + (size_t)bh * padded * 128);
    const unsigned* sel = p.selected + ((size_t)bh * nb + qtile) * topk;
    const float sl2 = p.sl2;
    const float NEG = neg_inf();

    // query block 0 is the one this wave finishes: queries 32 wave ..; block 1 the other wave's
    bf16x8 qf[NB][8];
#pragma unroll
    for (int b = 0; b < NB; b++)
        load_q_frags(p.qt + ((size_t)bh * padded + (size_t)qtile * kTileElems) * 128, (NB == 2 ? wave ^ b : 0) * 32 + c32,
                     true, lane, qf[b]);
    int krd = tile_read_bases32<64>(lane).k, vrd = tile_read_bases32<128>(lane).v;

    f32x16 o[NB][4];
    FineState st[NB];
#pragma unroll
    for (int b = 0; b < NB; b++) {
#pragma unroll
        for (int db = 0; db < 4; db++)
#pragma unroll
            for (int i = 0; i < 16; i++) o[b][db][i] = 0.f;
        st[b] = {NEG, 0.f, 0.f};
    }

    // The list, 64 entries at a time: lane l holds entry l (tile, keys); `mine` the entries this wave takes, `small` those
    // of up to 16 keys.
    int entry = 0, base = 0, turn_s = 0, turn_t = 0;
    unsigned long long mine = 0, small = 0;
    auto refill = [&]() {
        const int at = base + lane;
        base += 64;
        const bool in = at < topk;
        const int tile = min(max((int)sel[min(at, topk - 1)], 0), nb - 1);
        const int keys = in ? min(max(p.block_sizes[tile], 0), kTileElems) : kTileElems;
        entry = (tile << 7) | keys;
        const bool one = keys <= 32 && keys > 16, two = keys <= 16;
        const unsigned long long s = __builtin_amdgcn_ballot_w64(one);
        small = __builtin_amdgcn_ballot_w64(two);
        const int turn1 = lanes_below(s) + turn_s, turn2 = (lanes_below(small) >> 1) + turn_t, turn = two ? turn2 : turn1;
        mine = __builtin_amdgcn_ballot_w64(in & ((keys > 32) | ((turn & 1) == wave)));
        turn_s += __builtin_popcountll(s);
        turn_t += (__builtin_popcountll(small) + 1) >> 1;
    };
    auto next = [&]() -> FineStep {
        while (mine == 0 && base < topk) refill();
        FineStep r = {0, 16, 16, 16, mine == 0};   // (past the end: rows that exist, loaded and not used)
        if (mine == 0) return r;
        const int i = __builtin_ctzll(mine);
        mine &= mine - 1;
        const int e = __builtin_amdgcn_readlane(entry, i), keys = e & 127, half = keys > 32 ? 32 * wave : 0;
        r.row_a = (e >> 7) * kTileElems + half;
        r.valid_a = keys - half;
        r.row_b = r.row_a + 16;
        r.valid_b = r.valid_a - 16;
        const unsigned long long pair = mine & small;
        if (keys <= 16 && pair != 0) {
            const int j = __builtin_ctzll(pair);
            mine &= ~(1ull << j);
            const int f = __builtin_amdgcn_readlane(entry, j);
            r.row_b = (f >> 7) * kTileElems;
            r.valid_b = f & 127;
        }
        return r;
    };

    // A DMA instruction moves 1 KB: eight rows of a K chunk (128 bytes each, K swizzle of 64 channels) or four of a V chunk
    const int dr = lane >> 4;
    unsigned koff = (lane >> 3) * kRowBytes + (((lane & 7) ^ dr) << 4);   // (row >> 1) & 7 = 4 (it & 1) + l / 16
    const unsigned voff = dr * kRowBytes + (((lane & 15) ^ (dr << 2)) << 4);
    const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(size_t)ring);
    auto load_k = [&](unsigned slot, const FineStep s, int half, int it) {
        const int row = it < 2 ? s.row_a : s.row_b;
        const char* src = kb + (size_t)(unsigned)row * kRowBytes;
        lds_dma16_s(lds0 + slot + it * 1024, src + (it & 1) * 8 * kRowBytes + half * 128, koff ^ ((it & 1) << 6));
    };
    auto load_v = [&](unsigned slot, const FineStep s, int half, int it) {
        const int row = half ? s.row_b : s.row_a;
        const char* src = vb + (size_t)(unsigned)row * kRowBytes;
        lds_dma16_s(lds0 + slot + it * 1024, src + it * 1024, voff);
    };

    unsigned sk0 = 0, sk1 = kFineSlot, sv0 = 2 * kFineSlot, sv1 = 3 * kFineSlot, spare = 4 * kFineSlot;
    FineStep cur = next();
#pragma unroll
    for (int x = 0; x < 8; x++) load_k(x < 4 ? sk0 : sk1, cur, x >> 2, x & 3);
#pragma unroll
    for (int x = 0; x < 8; x++) load_v(x < 4 ? sv0 : sv1, cur, x >> 2, x & 3);
    if (pace.counters) pace.enter(0, lane);
    constexpr int kAhead = 2;   // a fragment feeds NB MFMAs and is read kAhead fragments before them
    while (!cur.none) {
        const FineStep nx = next();
        if (pace.counters) {
            const int w = nx.row_a / (kPaceTiles * kTileElems);
            if (w > pace.window) {
                pace.enter(w, lane);
                pace.wait(lane);
            }
        }
        // (addresses are formed where they are used: kept across the loop they would take 16 registers that it has not got)
        asm volatile("" : "+v"(krd), "+v"(vrd), "+v"(koff));
        f32x16 s[NB];
        {
            bf16x8 f[8];
            auto read = [&](int dk) { f[dk] = lds_read_b128(ring + (dk < 4 ? sk0 : sk1) + (krd ^ ((dk & 3) << 5))); };
            wait_vmcnt<12>();   // the first K chunk has landed; the other three may be in flight
            // The two waves of a SIMD come from workgroups that know nothing of each other: the one in a matrix part goes before
            // one that waits, forms addresses or is at its softmax. us, without / so, 12 heads 21 x 30 x 52 at 0.8 1878 / 1824, 16 x 32
            // x 64 at 0.9 1000 / 982, 24 heads 9 x 21 x 50 462 / 459. (Priority over the softmax too: 1853, 990, 461.)
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int dk = 0; dk < kAhead; dk++) read(dk);
#pragma unroll
            for (int dk = 0; dk < 8; dk++) {
                if (dk + kAhead == 4) wait_vmcnt<12>();   // the second one (in flight: both V chunks, the next K chunk)
                if (dk + kAhead < 8) read(dk + kAhead);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int b = 0; b < NB; b++) {
                    if (dk == 0)
#pragma unroll
                        for (int e = 0; e < 16; e++) s[b][e] = 0.f;
                    s[b] = mfma32(f[dk], qf[b][dk], s[b]);
                }
                __builtin_amdgcn_sched_barrier(0);
                if (dk < 2) load_k(spare, nx, 0, 2 * dk), load_k(spare, nx, 0, 2 * dk + 1);
                if (dk >= 4) load_k(sk0, nx, 1, dk - 4);   // (every read of the slot has been multiplied)
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __builtin_amdgcn_s_setprio(0);
        if (cur.valid_a < 16 || cur.valid_b < 16) {
            const int va = cur.valid_a - 4 * h, vb16 = cur.valid_b - 4 * h;
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const bool out = 8 * ((e >> 2) & 1) + (e & 3) >= (e < 8 ? va : vb16);
#pragma unroll
                for (int b = 0; b < NB; b++) s[b][e] = out ? NEG : s[b][e];
            }
        }
        float mx[NB];
        bool grown = false;
#pragma unroll
        for (int b = 0; b < NB; b++) {
            mx[b] = s[b][0];
#pragma unroll
            for (int e = 1; e < 16; e++) mx[b] = __builtin_fmaxf(mx[b], s[b][e]);
            mx[b] = pair_max(mx[b]) * sl2;
            grown |= mx[b] > st[b].thr;
        }
        if (__builtin_amdgcn_ballot_w64(grown) != 0) {
#pragma unroll
            for (int b = 0; b < NB; b++) {
                const bool need = mx[b] > st[b].thr;
                const float off = need ? mx[b] : st[b].off;
                const float alpha = st[b].thr == NEG ? 1.f : fast_exp2(st[b].off - off);   // (no finite score yet: zeros)
                st[b].off = off;
                if (need) st[b].thr = off + kRescaleLog2;
                st[b].l *= alpha;
#pragma unroll
                for (int db = 0; db < 4; db++)
#pragma unroll
                    for (int e = 0; e < 16; e++) o[b][db][e] *= alpha;
            }
        }
        bf16x8 pb[NB][2];
#pragma unroll
        for (int b = 0; b < NB; b++) {
#pragma unroll
            for (int t = 0; t < 2; t++) {
                f32x8 e;
#pragma unroll
                for (int x = 0; x < 8; x++) {
                    e[x] = fast_exp2(__builtin_fmaf(s[b][8 * t + x], sl2, -st[b].off));
                    st[b].l += e[x];
                }
                pb[b][t] = __builtin_convertvector(e, bf16x8);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int it = 0; it < 2 / NB; it++) load_v(sk1, nx, 0, NB == 2 ? 2 * b + t : 2 * t + it);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        wait_vmcnt<16>();   // the first V chunk
        __builtin_amdgcn_s_setprio(1);
        {
            bf16x8 f[8];
            auto read = [&](int g) {
                const lds_u8* a0 = ring + (g < 4 ? sv0 : sv1) + (vrd ^ ((g & 3) << 6));
                s16x8 a;
                a.lo = lds_read_tr16_b64(a0);
                a.hi = lds_read_tr16_b64(a0 + 8 * kRowBytes);
                f[g] = __builtin_bit_cast(bf16x8, a);
            };
#pragma unroll
            for (int g = 0; g < kAhead; g++) read(g);
#pragma unroll
            for (int g = 0; g < 8; g++) {
                if (g + kAhead == 4) wait_vmcnt<12>();   // the second one
                if (g + kAhead < 8) read(g + kAhead);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int b = 0; b < NB; b++) o[b][g & 3] = mfma32(f[g], pb[b][g >> 2], o[b][g & 3]);
                __builtin_amdgcn_sched_barrier(0);
                if (g >= 4) load_v(sv0, nx, 1, g - 4);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __builtin_amdgcn_s_setprio(0);
        const unsigned left_slot = sv1;   // the ring moves on by four of its five slots
        sv1 = sv0, sv0 = sk1, sk1 = sk0, sk0 = spare, spare = left_slot;
        cur = nx;
    }

    if (pace.counters) pace.enter((nb - 1) / kPaceTiles, lane);
    wait_vmcnt<0>();   // (the loads past the end)
    // The merge: each wave hands the other one's queries over in its own ring.
    typedef __attribute__((address_space(3))) f32x4 lds_f32x4;
    typedef __attribute__((address_space(3))) f32x2 lds_f32x2;
    constexpr int kMl = 4 * kFineSlot;   // behind the sums: offset and row sum, a pair a lane
    if (NB == 2 || wave == 1) {
        constexpr int B = NB - 1;
#pragma unroll
        for (int j = 0; j < 16; j++) {
            f32x4 r;
#pragma unroll
            for (int x = 0; x < 4; x++) r[x] = o[B][j >> 2][4 * (j & 3) + x];
            *reinterpret_cast<lds_f32x4*>(ring + (j * 64 + lane) * 16) = r;
        }
        *reinterpret_cast<lds_f32x2*>(ring + kMl + lane * 8) = f32x2{st[B].thr == NEG ? NEG : st[B].off, pair_sum(st[B].l)};
    }
    __syncthreads();
    if (NB == 1 && wave == 1) return;
    const lds_u8* other = smem + (wave ^ 1) * kFineWave;
    const f32x2 om = *reinterpret_cast<const lds_f32x2*>(other + kMl + lane * 8);
    const float off0 = st[0].thr == NEG ? NEG : st[0].off;
    const float m = __builtin_fmaxf(off0, om[0]);
    const float w0 = off0 == NEG ? 0.f : fast_exp2(off0 - m), w1 = om[0] == NEG ? 0.f : fast_exp2(om[0] - m);
    const float l_tot = pair_sum(st[0].l) * w0 + om[1] * w1;
    const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
    auto merged = [&](int db, int g) {
        const f32x4 t = *reinterpret_cast<const lds_f32x4*>(other + ((4 * db + g) * 64 + lane) * 16);
        f32x4 r;
#pragma unroll
        for (int x = 0; x < 4; x++) r[x] = (o[0][db][4 * g + x] * w0 + t[x] * w1) * inv;
        return r;
    };
    if (p.final_out) {
        // fused combine (kernels/core.cu:803-835): out[token] = coarse[tile] * gate[token] + sparse,
        // the product rounded to f32 before the add as on the host; padding slots write nothing
#pragma clang fp contract(off)
        const int token = p.slot_src[(size_t)qtile * kTileElems + wave * 32 + c32];
        if (token < 0) return;
        const float* co = p.coarse + ((size_t)bh * nb + qtile) * 128;
        const size_t row = ((size_t)bh * p.seq + token) * 128;
#pragma unroll
        for (int db = 0; db < 4; db++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const int d0 = 32 * db + 8 * g + 4 * h;
                const f32x4 c4 = *reinterpret_cast<const f32x4*>(co + d0);
                f32x4 ga = {1.f, 1.f, 1.f, 1.f};
                if (p.gate) {
                    if (p.gate_is_bf16) {
                        const u32x2 raw = *reinterpret_cast<const u32x2*>((const uint16_t*)p.gate + row + d0);
                        ga[0] = __builtin_bit_cast(float, raw[0] << 16);
                        ga[1] = __builtin_bit_cast(float, raw[0] & 0xffff0000u);
                        ga[2] = __builtin_bit_cast(float, raw[1] << 16);
                        ga[3] = __builtin_bit_cast(float, raw[1] & 0xffff0000u);
                    } else {
                        ga = *reinterpret_cast<const f32x4*>((const float*)p.gate + row + d0);
                    }
                }
                const f32x4 sp = merged(db, g);
                f32x4 r;
#pragma unroll
                for (int x = 0; x < 4; x++) r[x] = c4[x] * ga[x] + sp[x];
                *reinterpret_cast<f32x4*>(p.final_out + row + d0) = r;
            }
        return;
    }
    float* ob = p.out + (((size_t)bh * p.q_tiles + (qtile - p.q_base)) * kTileElems + wave * 32 + c32) * 128;
#pragma unroll
    for (int db = 0; db < 4; db++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            *reinterpret_cast<f32x4*>(ob + 32 * db + 8 * g + 4 * h) = merged(db, g);
        }
}

__global__ __launch_bounds__(128, 2) void vsa_fine_kernel(const VsaFineParams p) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int work = (blockIdx.x & 7) * p.per_xcd + (blockIdx.x >> 3);
    if (work >= p.total) return;
    const int bh = work / p.q_tiles;
    const int qtile = p.q_base + work % p.q_tiles;
    if (qtile >= p.num_tiles) return;
    FinePace pace = {nullptr, 0, -1, true};
    if (p.pace) {
        const int xcd = blockIdx.x & 7, at = blockIdx.x >> 3, gang = at / p.gang;
        pace.counters = p.pace + ((size_t)xcd * ((p.per_xcd + p.gang - 1) / p.gang) + gang) * p.pace_stride;
        pace.half = min(p.gang, min(p.per_xcd, p.total - xcd * p.per_xcd) - gang * p.gang);   // workgroups, of two waves
    }
    if (p.final_out && p.block_sizes[qtile] <= 32) fine_item<1>(p, (lds_u8*)smem_raw, wave, lane, bh, qtile, pace);
    else fine_item<2>(p, (lds_u8*)smem_raw, wave, lane, bh, qtile, pace);
}

// ---- combine (kernels/core.cu:803-835) -----------------------------------------------------
// out[token] = coarse[tile] * gate[token] + sparse[slot]; gate == null is a gate of one.
// ROUND16 is the bf16 combine of the H3 family (kernels/core.cu:825-830, kernels/attn3.cu:247-270):
// bf16(bf16(sparse) + bf16(bf16(coarse) * bf16(gate))), every step rounded to nearest even and the
// result stored as the f32 of that bf16 value; without a gate the product is bf16(coarse) itself.
template <bool GATE_BF16, bool ROUND16>
__global__ __launch_bounds__(256) void vsa_combine_kernel(
    const float* __restrict__ sparse, const float* __restrict__ coarse,
    const void* __restrict__ gate, const int* __restrict__ slot_src, float* __restrict__ out,
    long seq, int num_tiles, int q_base, int q_tiles, int has_gate) {
#pragma clang fp contract(off)   // coarse * gate rounds to f32 before the add, as on the host
    // one thread per (slot, 4 d): 32 threads per slot, 8 slots per block
    const long slot_lin = blockIdx.x * 8L + (threadIdx.x >> 5);   // over q_tiles * 64
    const int d0 = (threadIdx.x & 31) * 4;
    const long bh = blockIdx.y;
    if (slot_lin >= (long)q_tiles * kTileElems) return;
    const int g = (int)(slot_lin / kTileElems);
    const int tile = q_base + g;
    if (tile >= num_tiles) return;
    const int src = slot_src[(long)tile * kTileElems + (slot_lin - (long)g * kTileElems)];
    if (src < 0) return;
    const f32x4 sp = *reinterpret_cast<const f32x4*>(sparse + (bh * q_tiles * kTileElems + slot_lin) * 128 + d0);
    const f32x4 co = *reinterpret_cast<const f32x4*>(coarse + (bh * num_tiles + tile) * 128L + d0);
    f32x4 ga = {1.f, 1.f, 1.f, 1.f};
    if (has_gate) {
        if constexpr (GATE_BF16) {
            const u32x2 raw = *reinterpret_cast<const u32x2*>((const uint16_t*)gate + (bh * seq + src) * 128 + d0);
            ga[0] = __builtin_bit_cast(float, raw[0] << 16);
            ga[1] = __builtin_bit_cast(float, raw[0] & 0xffff0000u);
            ga[2] = __builtin_bit_cast(float, raw[1] << 16);
            ga[3] = __builtin_bit_cast(float, raw[1] & 0xffff0000u);
        } else {
            ga = *reinterpret_cast<const f32x4*>((const float*)gate + (bh * seq + src) * 128 + d0);
        }
    }
    f32x4 r;
    if constexpr (ROUND16) {
        auto r16 = [](float x) { return bf16_bits_to_f32(bf16_rne_bits(x)); };
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float c = r16(co[e]);
            const float p = has_gate ? r16(c * r16(ga[e])) : c;
            r[e] = r16(r16(sp[e]) + p);
        }
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++) r[e] = co[e] * ga[e] + sp[e];
    }
    *reinterpret_cast<f32x4*>(out + (bh * seq + src) * 128 + d0) = r;
}

}  // namespace fv

// ---- host launchers -----------------------------------------------------------------------

using namespace fv;

extern "C" hipError_t fv_internal_launch_tile_mean(const void* x, int x_is_bf16, const int* slot_src,
                                                   const int* block_sizes, float* out, size_t bh,
                                                   size_t seq, int dim, int num_tiles, int round16,
                                                   hipStream_t st) {
    const dim3 grid((num_tiles + 7) / 8, (unsigned)bh), block(256);
    if (x_is_bf16)
        hipLaunchKernelGGL(vsa_tile_mean_kernel<true>, grid, block, 0, st, x, slot_src, block_sizes, out,
                           (long)seq, dim, num_tiles, round16);
    else
        hipLaunchKernelGGL(vsa_tile_mean_kernel<false>, grid, block, 0, st, x, slot_src, block_sizes, out,
                           (long)seq, dim, num_tiles, round16);
    return hipGetLastError();
}

// Tile pass (tiles != null) and tile means of q, k and v in one launch; dim == 128. copy_mul (f32 operands only,
// null = none): factors on the values of the three copies before their rounding to bf16.
extern "C" hipError_t fv_internal_launch_tile_scan3(const void* const x[3], int x_is_bf16, const int* slot_src,
                                                    const int* block_sizes, uint16_t* const tiles[3],
                                                    float* const means[3], const float* copy_mul, size_t bh, size_t seq,
                                                    size_t padded, int num_tiles, hipStream_t st) {
    if (copy_mul && x_is_bf16) return hipErrorInvalidValue;   // a second rounding of values already rounded
    ThreeScan t;
    for (int i = 0; i < 3; i++)
        t.in[i] = x[i], t.tiles[i] = tiles ? tiles[i] : nullptr, t.means[i] = means[i], t.mul[i] = copy_mul ? copy_mul[i] : 1.0f;
    const dim3 grid((num_tiles + 15) / 16, (unsigned)bh, 3), block(256);
    if (tiles) {
        if (x_is_bf16)
            hipLaunchKernelGGL(vsa_tile_scan3_staged_kernel, dim3(num_tiles, (unsigned)bh, 3), dim3(64), 0, st, t, slot_src,
                               block_sizes, (long)seq, (long)padded, num_tiles);
        else
            hipLaunchKernelGGL(vsa_tile_scan3_staged_f32_kernel, dim3(num_tiles, (unsigned)bh, 3), dim3(64), 0, st, t,
                               slot_src, block_sizes, (long)seq, (long)padded, num_tiles);
        return hipGetLastError();
    }
    if (x_is_bf16)
        hipLaunchKernelGGL(vsa_tile_scan3_kernel<true>, grid, block, 0, st, t, slot_src, block_sizes, (long)seq, (long)padded, num_tiles);
    else
        hipLaunchKernelGGL(vsa_tile_scan3_kernel<false>, grid, block, 0, st, t, slot_src, block_sizes, (long)seq, (long)padded, num_tiles);
    return hipGetLastError();
}

// The coarse PV kernel's dynamic LDS limit (8 rows of up to 4096 scores), once per device.
extern "C" hipError_t fv_internal_init_vsa(void) {
    static std::atomic<unsigned long long> attr_done;
    return fv_set_max_lds_once((const void*)vsa_coarse_pv_kernel, (int)(sizeof(float) * kCoarseRows * kTopkMaxN),
                               attr_done);
}

extern "C" hipError_t fv_internal_launch_coarse(const float* qc, const float* kc, const float* vc,
                                                float* scores, float* coarse, size_t bh, int nb,
                                                int dim, float scale, hipStream_t st) {
    const dim3 g1((nb + 63) / 64, (nb + 63) / 64, (unsigned)bh);
    hipLaunchKernelGGL(vsa_coarse_scores_kernel, g1, dim3(256), 0, st, qc, kc, scores, nb, dim, scale);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || !coarse) return e;
    const size_t lds = sizeof(float) * kCoarseRows * (size_t)((nb + 3) & ~3);
    e = fv_internal_init_vsa();
    if (e != hipSuccess) return e;
    const dim3 g2((nb + kCoarseRows - 1) / kCoarseRows, (unsigned)bh);
    hipLaunchKernelGGL(vsa_coarse_pv_kernel, g2, dim3(256), lds, st, scores, vc, coarse, nb);
    return hipGetLastError();
}

// Counters of FinePace that a launch of `total` query tiles asks for (none where the key tiles of a head, 32 KB each, fit
// an XCD's L2), and its layout: gangs of as many workgroups as an XCD holds at a time, each with whole cache lines.
extern "C" size_t fv_internal_fine_pace(fv::VsaFineParams* p) {
    p->pace_stride = ((p->num_tiles + kPaceTiles - 1) / kPaceTiles + 31) & ~31;
    p->gang = std::max(1, fv_compute_units() / 8 * 4);
    if (p->num_tiles <= 128) return 0;
    return (size_t)8 * ((p->per_xcd + p->gang - 1) / p->gang) * p->pace_stride;
}

// zero: so many words set to zero besides (fv_internal_fine_pace)
extern "C" hipError_t fv_internal_launch_topk(const float* scores, unsigned* out, int rows, int n, int k,
                                              int* zero, int zeros, hipStream_t st) {
    if (n < 1 || n > kTopkMaxN) return hipErrorInvalidValue;
    // keys per lane: the smallest instantiated count that holds the row (624 tiles: 10)
    const int need = (n + 63) / 64;
    constexpr int kMost = 1 << 25;   // rows a launch, 64 threads each: it holds fewer than 2^32 work-items
    for (int at = 0; at < rows;) {
        const int some = rows - at < kMost ? rows - at : kMost;
        const dim3 grid((some + kTopkRowsPerBlock - 1) / kTopkRowsPerBlock), block(64 * kTopkRowsPerBlock);
        const float* src = scores + (size_t)at * n;
        unsigned* dst = out + (size_t)at * k;
#define FV_TOPK(K) hipLaunchKernelGGL(vsa_topk_kernel<K>, grid, block, 0, st, src, dst, some, n, k, zero, zeros)
        if (need <= 4) FV_TOPK(4);
        else if (need <= 8) FV_TOPK(8);
        else if (need <= 10) FV_TOPK(10);
        else if (need <= 12) FV_TOPK(12);
        else if (need <= 16) FV_TOPK(16);
        else if (need <= 24) FV_TOPK(24);
        else if (need <= 32) FV_TOPK(32);
        else if (need <= 48) FV_TOPK(48);
        else FV_TOPK(64);
#undef FV_TOPK
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        at += some;
    }
    return hipSuccess;
}

extern "C" hipError_t fv_internal_launch_tile_qkv(const void* x, int x_is_bf16, const int* slot_src,
                                                  uint16_t* xt, size_t bh, size_t seq, size_t padded,
                                                  int dim, hipStream_t st) {
    const size_t per = padded * (size_t)(dim / 8);
    const dim3 grid((unsigned)((per + 255) / 256), (unsigned)bh), block(256);
    if (x_is_bf16)
        hipLaunchKernelGGL(vsa_tile_qkv_kernel<true>, grid, block, 0, st, x, slot_src, xt, (long)seq,
                           (long)padded, dim);
    else
        hipLaunchKernelGGL(vsa_tile_qkv_kernel<false>, grid, block, 0, st, x, slot_src, xt, (long)seq,
                           (long)padded, dim);
    return hipGetLastError();
}

// (40 KB of LDS a workgroup: four fill a CU)
extern "C" hipError_t fv_internal_launch_fine(const fv::VsaFineParams* p, hipStream_t st) {
    hipLaunchKernelGGL(vsa_fine_kernel, dim3(p->per_xcd * 8), dim3(128), kFineLds, st, *p);
    return hipGetLastError();
}

extern "C" hipError_t fv_internal_launch_combine(const float* sparse, const float* coarse,
                                                 const void* gate, int gate_is_bf16,
                                                 const int* slot_src, float* out, size_t bh,
                                                 size_t seq, int num_tiles, int q_base, int q_tiles,
                                                 int round16, hipStream_t st) {
    const dim3 grid((unsigned)(((size_t)q_tiles * kTileElems + 7) / 8), (unsigned)bh), block(256);
    const int has_gate = gate != nullptr;
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, block, 0, st, sparse, coarse, gate, slot_src, out, (long)seq, num_tiles,
                           q_base, q_tiles, has_gate);
    };
    if (gate_is_bf16) {
        if (round16) launch(vsa_combine_kernel<true, true>);
        else launch(vsa_combine_kernel<true, false>);
    } else {
        if (round16) launch(vsa_combine_kernel<false, true>);
        else launch(vsa_combine_kernel<false, false>);
    }
    return hipGetLastError();
}
