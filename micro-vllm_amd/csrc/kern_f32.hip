// kern_f32.hip -- f32-weight GEMMs on the gfx950 matrix cores (v_mfma_f32_16x16x4_f32):
// moe_block with fmt 0 experts (the shared experts, src/model/kimi_k3.cpp:192-209,
// src/model/glm53.cpp:2000-2027), the router scores (src/gpu/metal_ops.cpp:213-231) and
// fmt 0 dense linears (QuantMat::gemm, src/quant/weight.cpp:47-64).
//
// C[r, o] = sum_k X[r, k] * W[o, k] with f32 products and f32 sums (the reference's
// matmul_f32 in another summation order).  Work item = (expert, block of up to 16 * MT
// rows) x (block of columns).  Lane (t, q) loads 16 bytes of row t of each operand at K
// offset 4 q, and MFMA step s takes element s of them, so the four steps of a 16-wide K
// block cover its K indices once.
// I8: a linear on QuantMat's int8 rows (fmt 8; quant::matmul_int8_row,
// src/quant/quant.cpp:255-268): each code converts exactly to f32, and the row's f32 scale
// multiplies the finished sum once, as the reference does.
#include "mfma_common.h"

#include <algorithm>

namespace mvllm_hip {

struct F32Item {
    int a, r0, nrow, pad;
};

struct F32Args {
    const ExpertWork *ew;   // per expert: w[0..2] = gate, up, down f32 [O][K]
                            // (I8: w[mi] int8 [O][K], s[mi] f32 [O])
    const F32Item *items;   // null: one expert (ew1), items of 16 * MT rows over nrows_all
    ExpertWork ew1;
    int nrows_all;
    const float *in;        // input rows [*][K]
    const int *in_rows;     // compact row -> input row (null: identity)
    float *out;             // output rows [rcap][O]
    float *out2;            // the second half of K's sums when K is split (ksl = 1)
    int mi;                 // single: which matrix of the expert (2 = down; 0 = a linear)
    int n_items, ksl;       // items; log2 of the K splits across workgroups (0 or 1)
    int nbn;                // k_f32mm_wave: workgroups per item
    int n_tasks, K, O;
    int act;
    float act_a, act_b;
};

// How the int8 codes of one row reach a lane: none (f32 rows), 4 codes of each 16-wide K
// block, or 16 codes of each 64-wide one (K % 64 == 0 and 16-byte aligned rows).
enum : int { kRowsF32 = 0, kRowsI8x4 = 1, kRowsI8x16 = 2 };

// With few rows the weights' stream is the bound, and a wave per column tile walking all of
// K left most of the chip idle (7168 x 384 at one row: 3 workgroups, 221 us for 11 MB).  So
// the W waves of a workgroup split K of the same NT tiles of 16 weight rows and meet once
// in LDS, where one thread per output adds the W partial sums in wave order (a fixed order:
// equal inputs give equal bits; chains W times shorter, so no less exact).  Dual: the gate
// and the up rows of 16 columns (NT = 2) or of 8 columns, side by side in one tile (NT = 1).
// Two groups of U K blocks per operand are in flight per wave; loads past the wave's range
// repeat its last block and are not multiplied.  Against the wave-per-tile kernel: the f32
// expert of 7168 x 2048 at one row 300 -> 54 us per call (176 MB, 3.2 TB/s with the
// combine), int8 7168 x 7168 167 -> 22 us, f32 7168 x 7168 at 61 rows 526 -> 103 us.
template <bool DUAL, int MT, int NT, int WK, int W>
__global__ __launch_bounds__(64 * W) void k_f32mm_rows(F32Args A) {
    static_assert(!(WK && DUAL), "int8 rows: single projections only");
    constexpr int KBW = WK == kRowsI8x16 ? 64 : 16;  // K indices of a block
    constexpr int XV = KBW / 16;                     // float4 of an input row per lane and block
    constexpr int U = WK == kRowsI8x16 ? (MT == 1 ? 2 : 1) : (MT == 1 ? 4 : 2);
    __shared__ float red[W][MT * NT * 256];
    const int task = xcd_task(blockIdx.x, A.n_tasks);
    const int cs = task / A.n_items, item = task - cs * A.n_items;
    const int ks = cs & ((1 << A.ksl) - 1), cb = cs >> A.ksl;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, t = lane & 15, q = lane >> 4;
    const int K = A.K, O = A.O;
    constexpr int CW = DUAL ? 8 * NT : 16 * NT;  // output columns of a workgroup
    const int col0 = cb * CW;
    F32Item it;
    if (A.items) {
        it = A.items[item];
    } else {
        it.a = 0;
        it.r0 = item * 16 * MT;
        it.nrow = min(16 * MT, A.nrows_all - it.r0);
    }
    const ExpertWork &ew = A.items ? A.ew[it.a] : A.ew1;
    const int jbase = ew.row0 + it.r0;
    const float4 *xr[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int r = min(mt * 16 + t, it.nrow - 1);  // rows past the item repeat the last
        const int src = A.in_rows ? A.in_rows[jbase + r] : jbase + r;
        xr[mt] = reinterpret_cast<const float4 *>(A.in + (size_t)src * K) + XV * q;
    }
    const char *wr[NT];
#pragma unroll
    for (int m = 0; m < NT; ++m) {
        const int row = DUAL ? col0 + (NT == 1 ? t & 7 : t) : col0 + 16 * m + t;
        const char *w = static_cast<const char *>(ew.w[DUAL ? (NT == 1 ? t >> 3 : m) : A.mi]);
        wr[m] = w + (size_t)row * (size_t)K * (WK ? 1 : 4) + (WK == kRowsI8x4 ? 4 : 16) * q;
    }
    f4v acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int m = 0; m < NT; ++m)
            acc[mt][m] = f4v{0.f, 0.f, 0.f, 0.f};
    // this wave's K blocks [kb0, kb1)
    const unsigned nkb = (unsigned)(K / KBW), part = (unsigned)(ks * W + wave);
    constexpr int LW = W == 16 ? 4 : W == 8 ? 3 : 2;
    const int kb0 = (int)(nkb * part >> (LW + A.ksl));
    const int kb1 = (int)(nkb * (part + 1) >> (LW + A.ksl));
    const int klast = max(kb1 - 1, 0);
    struct Buf {
        float4 x[U][MT][XV];
        u32x4 w[U][NT];  // kRowsI8x4: word 0 only
    };
    auto load = [&] __attribute__((always_inline)) (Buf &b, int kb) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = min(kb + u, klast);
#pragma unroll
            for (int m = 0; m < NT; ++m) {
                const char *p = wr[m] + (size_t)k * (WK ? KBW : 64);
                if constexpr (WK == kRowsI8x4)
                    b.w[u][m].x = *reinterpret_cast<const uint32_t *>(p);
                else
                    b.w[u][m] = *reinterpret_cast<const u32x4 *>(p);
            }
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int v = 0; v < XV; ++v)
                    b.x[u][mt][v] = xr[mt][(size_t)k * (KBW / 4) + v];
        }
    };
    auto mma = [&] __attribute__((always_inline)) (const Buf &b, int u) {
#pragma unroll
        for (int v = 0; v < XV; ++v)
#pragma unroll
            for (int m = 0; m < NT; ++m) {
                float w[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if constexpr (WK == kRowsF32)
                        w[e] = __uint_as_float(b.w[u][m][e]);
                    else
                        w[e] = (float)(int8_t)(b.w[u][m][v] >> (8 * e));
                }
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    const float4 x = b.x[u][mt][v];
                    acc[mt][m] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.x, w[0], acc[mt][m], 0, 0, 0);
                    acc[mt][m] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.y, w[1], acc[mt][m], 0, 0, 0);
                    acc[mt][m] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.z, w[2], acc[mt][m], 0, 0, 0);
                    acc[mt][m] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.w, w[3], acc[mt][m], 0, 0, 0);
                }
            }
    };
    // groups of U blocks, two buffers; the pair loop has no exit between its two halves, and
    // the last group(s) run after it with a uniform test per block
    Buf b0, b1;
    int kb = kb0;
    load(b0, kb);
    for (; kb + 2 * U <= kb1; kb += 2 * U) {
        load(b1, kb + U);
#pragma unroll
        for (int u = 0; u < U; ++u)
            mma(b0, u);
        load(b0, kb + 2 * U);
#pragma unroll
        for (int u = 0; u < U; ++u)
            mma(b1, u);
    }
    load(b1, kb + U);
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (kb + u < kb1)
            mma(b0, u);
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (kb + U + u < kb1)
            mma(b1, u);
    // C[4 q + i][t] of row tile mt and tile m -> LDS, then the W partial sums in wave order
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int m = 0; m < NT; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                red[wave][(mt * NT + m) * 256 + i * 64 + lane] = acc[mt][m][i];
    __syncthreads();
    auto sum = [&] __attribute__((always_inline)) (int at) {
        float v = red[0][at];
#pragma unroll
        for (int w = 1; w < W; ++w)
            v += red[w][at];
        return v;
    };
    for (int e = tid; e < MT * (DUAL ? 1 : NT) * 256; e += 64 * W) {
        const int tile = e >> 8, pos = e & 255;
        const int mt = DUAL ? tile : tile / NT, m = DUAL ? 0 : tile - mt * NT;
        const int r = mt * 16 + 4 * ((pos >> 4) & 3) + (pos >> 6);
        const int col = col0 + 16 * m + (pos & 15);
        if (r >= it.nrow || (DUAL && NT == 1 && (pos & 8)))
            continue;
        float *dst = (ks ? A.out2 : A.out) + (size_t)(jbase + r) * O + col;
        if constexpr (DUAL)
            *dst = mf_act(A.act, sum(NT * tile * 256 + pos),
                          sum(NT == 1 ? e + 8 : (2 * tile + 1) * 256 + pos), A.act_a, A.act_b);
        else if constexpr (WK != kRowsF32)
            *dst = sum(e) * static_cast<const float *>(ew.s[A.mi])[col];
        else
            *dst = sum(e);
    }
}

// Many rows: 64 input rows x 16 NB weight rows a workgroup, through LDS.  In the kernel above
// each wave reads 64 bytes, half a line, of 96 rows for 32 matrix instructions, and the waves
// of a workgroup read different parts of K, so nothing is shared.  Here
// a K step of 32 is a whole line of every row, read once for the four waves that share it, two
// steps ahead (registers, then one of two LDS buffers; 16-byte chunks XOR-swizzled by the
// row, so that eight rows' reads of one chunk lie in different banks); wave w multiplies row
// tile w with all NB weight tiles.  int8 codes convert to f32 as they are staged.  Two such
// groups of four waves split K and add at the end: with one, a CU that has a single workgroup
// waits on its loads (1024 x 7168 at 512 rows 112 us, 91 with two).  Each 512 of K sum in
// their own chain, which then adds to the total: no less exact than eight waves' split.
// The f32 expert of 6144 x 2048 over 300 rows 386 -> 291 us per call (59 -> 78 TFLOP/s), f32
// 7168 x 7168 over 1024 rows 1178 -> 964 us (109 of the f32 matrix cores' 157 TFLOP/s), int8
// 1116 -> 963 us.  Counted, the matrix cores are busy 48 and 53 % (gate/up, down of the
// expert) and 69 % (1024 rows) of the time; the waves wait 61-68 % of theirs, 7 % on LDS reads
// (no bank conflicts), and the address units do not stall: the rest goes to the waits of each
// step of 16 matrix instructions a wave (its barrier, its loads).
template <bool DUAL, int NB, int WK>
__global__ __launch_bounds__(512) void k_f32mm_tile(F32Args A) {
    constexpr int BK = 32, XC = 64 * BK / 4 / 256;      // chunks of x a thread stages
    constexpr int WC = 16 * NB * BK / 4 / 256;          // and of the weights
    constexpr int CT = DUAL ? NB / 2 : NB;              // output column tiles
    static_assert(NB % 2 == 0 && WC >= 1, "weight tiles in pairs");
    __shared__ float4 lx[2][2][64 * BK / 4];
    __shared__ float4 lw[2][2][16 * NB * BK / 4];
    const int task = xcd_task(blockIdx.x, A.n_tasks);
    const int cb = task / A.n_items, item = task - cb * A.n_items;
    const int tid = threadIdx.x & 255;
    const int grp = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    auto &sx = lx[grp];
    auto &sw = lw[grp];
    const int lane = tid & 63, t = lane & 15, q = lane >> 4;
    const int K = A.K, O = A.O, col0 = cb * 16 * CT;
    F32Item it;
    if (A.items) {
        it = A.items[item];
    } else {
        it.a = 0;
        it.r0 = item * 64;
        it.nrow = min(64, A.nrows_all - it.r0);
    }
    const ExpertWork &ew = A.items ? A.ew[it.a] : A.ew1;
    const int jbase = ew.row0 + it.r0;
    // this thread's chunks: chunk tid % 8 of rows tid / 8 + 32 j (rows past the item or the
    // matrix repeat the last; their results are not stored)
    const int c = tid & 7, r0 = tid >> 3;
    const float *xr[XC];
#pragma unroll
    for (int j = 0; j < XC; ++j) {
        const int r = min(r0 + 32 * j, it.nrow - 1);
        const int src = A.in_rows ? A.in_rows[jbase + r] : jbase + r;
        xr[j] = A.in + (size_t)src * K;
    }
    const char *wr[WC];
#pragma unroll
    for (int j = 0; j < WC; ++j) {
        const int r = r0 + 32 * j, m = r >> 4;
        const int row = min(col0 + 16 * (m % CT) + (r & 15), O - 1);
        const char *w = static_cast<const char *>(ew.w[DUAL ? m / CT : A.mi]);
        wr[j] = w + (size_t)row * (size_t)K * (WK ? 1 : 4);
    }
    struct Stage {
        float4 x[XC];
        u32x4 w[WC];  // int8: word 0 only
    };
    // this group's K steps: [s0, s0 + ns); the second group's may end past K
    const int ns = ((K + BK - 1) / BK + 1) / 2, s0 = grp * ns;
    auto load = [&] __attribute__((always_inline)) (Stage &b, int s) {
        const int k = (s0 + min(s, ns - 1)) * BK + 4 * c;
        const int kc = min(k, K - 4);  // past K: zeros (set at the store)
#pragma unroll
        for (int j = 0; j < WC; ++j) {
            if constexpr (WK)
                b.w[j].x = *reinterpret_cast<const uint32_t *>(wr[j] + kc);
            else
                b.w[j] = *reinterpret_cast<const u32x4 *>(wr[j] + 4 * (size_t)kc);
        }
#pragma unroll
        for (int j = 0; j < XC; ++j)
            b.x[j] = *reinterpret_cast<const float4 *>(xr[j] + kc);
    };
    auto store = [&] __attribute__((always_inline)) (const Stage &b, int s, int buf) {
        const bool in = s < ns && (s0 + s) * BK + 4 * c < K;
        const int at = 8 * r0 + (c ^ (r0 & 7));  // rows 32 apart swizzle alike
#pragma unroll
        for (int j = 0; j < XC; ++j)
            sx[buf][at + 256 * j] = in ? b.x[j] : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int j = 0; j < WC; ++j) {
            float4 w;
            if constexpr (WK)
                w = make_float4((float)(int8_t)b.w[j].x, (float)(int8_t)(b.w[j].x >> 8),
                                (float)(int8_t)(b.w[j].x >> 16), (float)(int8_t)(b.w[j].x >> 24));
            else
                w = __builtin_bit_cast(float4, b.w[j]);
            sw[buf][at + 256 * j] = in ? w : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    };
    f4v acc[NB], tot[NB];
#pragma unroll
    for (int m = 0; m < NB; ++m)
        acc[m] = tot[m] = f4v{0.f, 0.f, 0.f, 0.f};
    const bool live = 16 * wave < it.nrow;
    auto mma = [&] __attribute__((always_inline)) (int buf) {
        if (!live)  // wave-uniform: a row tile past the item
            return;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int at = 8 * t + ((4 * h + q) ^ (t & 7));
            const float4 x = sx[buf][128 * wave + at];
            float4 w[NB];
#pragma unroll
            for (int m = 0; m < NB; ++m)
                w[m] = sw[buf][128 * m + at];
#pragma unroll
            for (int m = 0; m < NB; ++m)
                acc[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.x, w[m].x, acc[m], 0, 0, 0);
#pragma unroll
            for (int m = 0; m < NB; ++m)
                acc[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.y, w[m].y, acc[m], 0, 0, 0);
#pragma unroll
            for (int m = 0; m < NB; ++m)
                acc[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.z, w[m].z, acc[m], 0, 0, 0);
#pragma unroll
            for (int m = 0; m < NB; ++m)
                acc[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.w, w[m].w, acc[m], 0, 0, 0);
        }
    };
    auto fold = [&] __attribute__((always_inline)) () {
#pragma unroll
        for (int m = 0; m < NB; ++m) {
            tot[m] += acc[m];
            acc[m] = f4v{0.f, 0.f, 0.f, 0.f};
        }
    };
    // step s: LDS buffer s & 1; its successor waits in one register set while the one after it
    // is loaded into the other.  One barrier a step: the buffer that a step writes was last
    // read before the barrier that ended the step before.
    Stage g0, g1;
    load(g0, 0);
    load(g1, 1);
    store(g0, 0, 0);
    __syncthreads();
    for (int s = 0; s < ns; s += 2) {
        load(g0, s + 2);
        mma(0);
        store(g1, s + 1, 1);  // past the last step: zeros
        __syncthreads();
        load(g1, s + 3);
        mma(1);
        store(g0, s + 2, 0);
        if ((s & 14) == 14)
            fold();
        __syncthreads();
    }
    fold();
    // the second group's sums are added to the first's
    f4v *part = reinterpret_cast<f4v *>(&lx[0][0][0]);  // 256 NB of its 2048 chunks
    if (grp)
#pragma unroll
        for (int m = 0; m < NB; ++m)
            part[256 * m + tid] = tot[m];
    __syncthreads();
    if (grp)
        return;
#pragma unroll
    for (int m = 0; m < NB; ++m)
        tot[m] += part[256 * m + tid];
    // C[4 q + i][t] of row tile `wave` and weight tile m
#pragma unroll
    for (int m = 0; m < CT; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = 16 * wave + 4 * q + i, col = col0 + 16 * m + t;
            if (r >= it.nrow || col >= O)
                continue;
            float *dst = A.out + (size_t)(jbase + r) * O + col;
            if constexpr (DUAL)
                *dst = mf_act(A.act, tot[m][i], tot[m + CT][i], A.act_a, A.act_b);
            else if constexpr (WK != kRowsF32)
                *dst = tot[m][i] * static_cast<const float *>(ew.s[A.mi])[col];
            else
                *dst = tot[m][i];
        }
}

constexpr int kF32Waves = 4;

// Short K, or more column tiles than the chip holds workgroups: a wave of its own for each tile
// of 16 MT rows x 32 columns (dual: 16) over all of K.  The splits above then start eight waves
// and meet in LDS for a few blocks each.  int8 codes come as 4 of each 16-wide block.  K sums in
// P chains, by the block's parity (P = 2, as the two groups above) and by the matrix
// instruction's step in it (P = 8, as eight waves), added in order at the end: as exact as the
// split (f32 24576 x 512 1.5e-7 from 64 bits, one chain 4.0e-7).
template <bool DUAL, int MT, bool I8, int P>
__global__ __launch_bounds__(64 * kF32Waves)
__attribute__((amdgpu_waves_per_eu(MT == 2 ? 2 : 1, 8))) void k_f32mm_wave(F32Args A) {
    static_assert(!(I8 && DUAL), "int8 rows: single projections only");
    const int item = blockIdx.x / A.nbn;
    const int nb = blockIdx.x - item * A.nbn;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63, t = lane & 15, q = lane >> 4;
    const int K = A.K, O = A.O;
    const int col0 = DUAL ? (nb * kF32Waves + wave) * 16 : (nb * kF32Waves + wave) * 32;
    if (col0 >= O)
        return;  // past the last column tile (waves share nothing: no barrier below)
    F32Item it;
    if (A.items) {
        it = A.items[item];
    } else {
        it.a = 0;
        it.r0 = item * 16 * MT;
        it.nrow = min(16 * MT, A.nrows_all - it.r0);
    }
    const ExpertWork &ew = A.items ? A.ew[it.a] : A.ew1;
    const int jbase = ew.row0 + it.r0;
    // operand row pointers of this lane: MT input rows, two weight rows
    const float4 *xr[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int r = min(mt * 16 + t, it.nrow - 1);  // rows past the item repeat the last
        const int src = A.in_rows ? A.in_rows[jbase + r] : jbase + r;
        xr[mt] = reinterpret_cast<const float4 *>(A.in + (size_t)src * K) + q;
    }
    const float4 *wr[2];
    const int *wr8[2];  // I8: 4 codes of row t at K offset 4 q of each 16-wide block
#pragma unroll
    for (int m = 0; m < 2; ++m) {
        const int row = DUAL ? col0 + t : col0 + 16 * m + t;
        if constexpr (I8) {
            const int8_t *w = static_cast<const int8_t *>(ew.w[A.mi]);
            wr8[m] = reinterpret_cast<const int *>(w + (size_t)row * K) + q;
        } else {
            const float *w = static_cast<const float *>(ew.w[DUAL ? m : A.mi]);
            wr[m] = reinterpret_cast<const float4 *>(w + (size_t)row * K) + q;
        }
    }
    f4v acc[P][MT][2];
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
            acc[p][mt][0] = acc[p][mt][1] = f4v{0.f, 0.f, 0.f, 0.f};
    const int nkb = K >> 4;  // 16-wide K blocks; a block is 4 float4 per row
    float4 xa[2][MT], wb[2][2];
    int wq[2][2];  // I8: raw codes
    auto load = [&](int kb, int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
            xa[buf][mt] = xr[mt][4 * kb];
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            if constexpr (I8)
                wq[buf][m] = wr8[m][4 * kb];
            else
                wb[buf][m] = wr[m][4 * kb];
        }
    };
    auto mma = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                float4 b;
                if constexpr (I8) {
                    const int v = wq[buf][m];
                    b = float4{(float)(int8_t)(v & 0xff), (float)(int8_t)((v >> 8) & 0xff),
                               (float)(int8_t)((v >> 16) & 0xff), (float)(int8_t)(v >> 24)};
                } else {
                    b = wb[buf][m];
                }
                const float4 a = xa[buf][mt];
                auto step = [&](float x, float w, int s) __attribute__((always_inline)) {
                    f4v &c = acc[P == 8 ? 4 * buf + s : P == 2 ? buf : 0][mt][m];
                    c = __builtin_amdgcn_mfma_f32_16x16x4f32(x, w, c, 0, 0, 0);
                };
                step(a.x, b.x, 0);
                step(a.y, b.y, 1);
                step(a.z, b.z, 2);
                step(a.w, b.w, 3);
            }
    };
    // two blocks in flight: block kb + 1 loads while block kb multiplies (past the end:
    // the last block again, never consumed)
    load(0, 0);
    for (int kb = 0; kb < nkb; kb += 2) {
        load(min(kb + 1, nkb - 1), 1);
        mma(0);
        if (kb + 1 >= nkb)
            break;
        load(min(kb + 2, nkb - 1), 0);
        mma(1);
    }
#pragma unroll
    for (int p = 1; p < P; ++p)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int m = 0; m < 2; ++m)
                acc[0][mt][m] += acc[p][mt][m];
    // C[4 q + i][t] of row tile mt and column tile m
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = mt * 16 + 4 * q + i;
            if (r >= it.nrow)
                continue;
            float *dst = A.out + (size_t)(jbase + r) * O;
            if constexpr (DUAL) {
                dst[col0 + t] = mf_act(A.act, acc[0][mt][0][i], acc[0][mt][1][i], A.act_a, A.act_b);
            } else if constexpr (I8) {
                const float *sc = static_cast<const float *>(ew.s[A.mi]);
                dst[col0 + t] = acc[0][mt][0][i] * sc[col0 + t];
                dst[col0 + 16 + t] = acc[0][mt][1][i] * sc[col0 + 16 + t];
            } else {
                dst[col0 + t] = acc[0][mt][0][i];
                dst[col0 + 16 + t] = acc[0][mt][1][i];
            }
        }
}

bool f32mm_fits(bool dual, int K, int O) {
    return K >= 16 && K % 16 == 0 && O % (dual ? 16 : 32) == 0;
}

// Whether a wave of its own for each tile is the faster form: by K and the number of column
// tiles of all items (32 columns; dual 16), from calls of 1 to 4096 rows and 32 to 163840
// columns in both forms.  At few tiles it wins while K has no blocks for eight waves (f32 2048
// x 64 at 16 rows 5.8 us with the split, 4.4 with a wave a tile); where the tiles are more
// workgroups of eight waves than the chip holds, also beyond (f32 32768 x 512 at 16 rows 25 ->
// 20, 65536 x 1024 92 -> 62, int8 163840 x 16 60 -> 9; against the blocks of 64 rows through
// LDS, f32 16384 x 16 at 4096 rows 240 -> 51).  One chain of K is some 20 % faster still, but
// 2.6 times as far from 64 bits.  The lines weigh single
// matrices: small experts of 17 to 32 rows take up to 0.7 us more than with the split (eight of
// 20 rows, 32 x 96 16.5 -> 17.2 us, 64 x 64 17.7 -> 18.0).  Up to four rows the split stays
// ahead for longer: there the tiles of a longer K count half.
static bool f32_wave_fits(bool i8, int mt, int K, long long tiles, int rows) {
    constexpr int kNever = 1 << 30;
    struct Line {
        int K, tiles;  // up to this K, from this many tiles
    };
    static const Line lines[2][3][7] = {
        {{{96, 0}, {128, 224}, {320, 384}, {384, 768}, {512, 1024}, {768, kNever}, {1024, 1024}},
         {{64, 0}, {192, 384}, {256, 768}, {512, 1024}, {1024, 2048}, {kNever, kNever}},
         {{32, 0}, {64, 640}, {96, 1536}, {128, 24576}, {192, 5120}, {kNever, kNever}}},
        {{{64, 0}, {128, 224}, {256, 384}, {384, 768}, {512, 1024}, {kNever, kNever}},
         {{96, 384}, {256, 1024}, {kNever, kNever}},
         {{16, 640}, {32, 896}, {96, 1536}, {192, 5120}, {256, kNever}, {320, 6144},
          {kNever, kNever}}},
    };
    if (mt == 1 && rows <= 4 && K > (i8 ? 128 : 320))
        tiles /= 2;
    for (const Line &l : lines[i8 ? 1 : 0][mt == 4 ? 2 : mt - 1])
        if (K <= l.K)
            return tiles >= l.tiles;
    return false;
}

hipError_t launch_f32mm(bool dual, int mt, const ExpertWork *ew, const void *items, int n_items,
                        const ExpertWork *ew1, int nrows_all, const float *in,
                        const int *in_rows, float *out, int mi, int K, int O, int act,
                        float act_a, float act_b, hipStream_t st, bool i8, float *out2) {
    if (!f32mm_fits(dual, K, O) || (mt != 1 && mt != 2 && mt != 4) || (!items && !ew1) ||
        (i8 && (dual || out2)) || (dual && out2))
        return hipErrorInvalidValue;
    F32Args a{};
    a.ew = ew;
    a.items = static_cast<const F32Item *>(items);
    if (ew1)
        a.ew1 = *ew1;
    a.nrows_all = nrows_all;
    a.in = in;
    a.in_rows = in_rows;
    a.out = out;
    a.out2 = out2;
    a.ksl = out2 ? 1 : 0;
    a.mi = mi;
    a.K = K;
    a.O = O;
    a.act = act;
    a.act_a = act_a;
    a.act_b = act_b;
    if (!items)
        n_items = (nrows_all + 16 * mt - 1) / (16 * mt);
    if (n_items <= 0)
        return hipSuccess;
    a.n_items = n_items;
    const long long tiles = (long long)n_items * (O / (dual ? 16 : 32));
    if (!out2 && f32_wave_fits(i8, mt, K, tiles, nrows_all)) {
        a.nbn = (O / (dual ? 16 : 32) + kF32Waves - 1) / kF32Waves;
        const dim3 grid((unsigned)(n_items * a.nbn)), block(64 * kF32Waves);
#define MVLLM_F32W(D, M, I, P) \
    hipLaunchKernelGGL((k_f32mm_wave<D, M, I, P>), grid, block, 0, st, a)
#define MVLLM_F32W_MT(D, I)                               \
    do {                                                  \
        if (mt == 1) MVLLM_F32W(D, 1, I, 8);              \
        else if (mt == 2) MVLLM_F32W(D, 2, I, 8);         \
        else MVLLM_F32W(D, 4, I, 2);                      \
    } while (0)
        if (dual)
            MVLLM_F32W_MT(true, false);
        else if (K == 16 && mt == 4 && i8)  // one block: no second chain
            MVLLM_F32W(false, 4, true, 1);
        else if (K == 16 && mt == 4)
            MVLLM_F32W(false, 4, false, 1);
        else if (i8)
            MVLLM_F32W_MT(false, true);
        else
            MVLLM_F32W_MT(false, false);
#undef MVLLM_F32W_MT
#undef MVLLM_F32W
        return hipGetLastError();
    }
    // Blocks of 64 rows through LDS where they are more than a workgroup a CU (at 256 of them:
    // int8 1024 x 7168 at 512 rows 91 us against 82 of the rows' kernel, f32 91 against 88; at
    // 320, 2048 x 6144 at 300 rows, 128 against 144, int8 128 against 137).  Four weight tiles
    // a workgroup where their rounds of 256 cost no more than those of two.
    if (mt == 4 && !out2) {
        const auto tasks = [&](int nb) {
            const int cw = dual ? 8 * nb : 16 * nb;
            return (long long)n_items * ((O + cw - 1) / cw);
        };
        const long long t2 = tasks(2), t4 = tasks(4);
        if (t2 > 256) {
            const bool four = (t4 + 255) / 256 * 2 <= (t2 + 255) / 256;
            a.n_tasks = (int)(four ? t4 : t2);
            const dim3 grid((unsigned)a.n_tasks), block(512);
#define MVLLM_F32T(D, I)                                                                  \
    do {                                                                                  \
        if (four) hipLaunchKernelGGL((k_f32mm_tile<D, 4, I>), grid, block, 0, st, a);     \
        else hipLaunchKernelGGL((k_f32mm_tile<D, 2, I>), grid, block, 0, st, a);          \
    } while (0)
            if (dual)
                MVLLM_F32T(true, kRowsF32);
            else if (i8)
                MVLLM_F32T(false, kRowsI8x4);
            else
                MVLLM_F32T(false, kRowsF32);
#undef MVLLM_F32T
            return hipGetLastError();
        }
    }
    const bool wide8 = i8 && K % 64 == 0 && ew1 && (reinterpret_cast<uintptr_t>(ew1->w[mi]) & 15) == 0;
    // Two tiles a wave read the input rows once for twice the weights; one tile a wave gives
    // twice the workgroups.  Two from 448 one-tile tasks on (the 256 CUs then have about a
    // workgroup each): int8 7168 x 7168 at 16 rows 28 us against 42 us with one tile, f32
    // 7168 x 7168 at 61 rows 103 against 154 us; below, one: the f32 expert of 7168 x 2048 at
    // one row 54 against 77 us, 2048 x 2048 at 8 rows 11 against 22 us.  Sixteen waves split a
    // long K of a launch that leaves CUs to spare (the same expert 54 against 57 us with
    // eight, int8 7168 x 7168 22 against 25 us); shorter rows pay more for the larger
    // workgroup's start than they gain (2048 x 2048 14 against 11 us).
    const long long t1 = (long long)n_items * (O / (dual ? 8 : 16)) << a.ksl;
    const int nt = t1 >= 448 ? 2 : 1;
    const int w = mt == 1 && K >= 4096 && t1 / nt <= 256 ? 16 : 8;
    a.n_tasks = (int)(t1 / nt);
    const dim3 grid((unsigned)a.n_tasks), block((unsigned)(64 * w));
#define MVLLM_F32(D, M, N, I, W_) \
    hipLaunchKernelGGL((k_f32mm_rows<D, M, N, I, W_>), grid, block, 0, st, a)
#define MVLLM_F32_MT(D, N, I)                                     \
    do {                                                          \
        if (mt == 1 && w == 16) MVLLM_F32(D, 1, N, I, 16);        \
        else if (mt == 1) MVLLM_F32(D, 1, N, I, 8);               \
        else if (mt == 2) MVLLM_F32(D, 2, N, I, 8);               \
        else MVLLM_F32(D, 4, N, I, 8);                            \
    } while (0)
    if (dual && nt == 2)
        MVLLM_F32_MT(true, 2, kRowsF32);
    else if (dual)
        MVLLM_F32_MT(true, 1, kRowsF32);
    else if (!i8 && nt == 2)
        MVLLM_F32_MT(false, 2, kRowsF32);
    else if (!i8)
        MVLLM_F32_MT(false, 1, kRowsF32);
    else if (wide8 && nt == 2)
        MVLLM_F32_MT(false, 2, kRowsI8x16);
    else if (wide8)
        MVLLM_F32_MT(false, 1, kRowsI8x16);
    else if (nt == 2)
        MVLLM_F32_MT(false, 2, kRowsI8x4);
    else
        MVLLM_F32_MT(false, 1, kRowsI8x4);
#undef MVLLM_F32_MT
#undef MVLLM_F32
    return hipGetLastError();
}

// ---- the router's elementwise tail (src/gpu/metal_ops.cpp:218-231) ------------------

// scores [n][E] (the router GEMM) -> mix = sigmoid(score) and choice = mix + bias[e],
// written in place of scores (mix) and into choice.  Sigmoid split by sign as the
// reference's (src/quant/quant.hpp:22-29).
__global__ void k_route_tail(float *scores, const float *bias, float *choice, int n, int E) {
    const size_t total = (size_t)n * E;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < total;
         i += (size_t)gridDim.x * blockDim.x) {
        const float s = mf_sigmoid(scores[i]);
        scores[i] = s;
        choice[i] = s + (bias ? bias[i % E] : 0.f);
    }
}

// w[n][k] *= rscale (after moe_topk normalized them)
__global__ void k_scale(float *w, size_t count, float rscale) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < count;
         i += (size_t)gridDim.x * blockDim.x)
        w[i] *= rscale;
}

hipError_t launch_route_tail(float *scores, const float *bias, float *choice, int n, int E,
                             hipStream_t st) {
    const size_t total = (size_t)n * E;
    const unsigned grid = (unsigned)std::min<size_t>((total + 255) / 256, 4096);
    hipLaunchKernelGGL(k_route_tail, dim3(grid), dim3(256), 0, st, scores, bias, choice, n, E);
    return hipGetLastError();
}

hipError_t launch_scale(float *w, size_t count, float rscale, hipStream_t st) {
    const unsigned grid = (unsigned)std::min<size_t>((count + 255) / 256, 1024);
    hipLaunchKernelGGL(k_scale, dim3(grid), dim3(256), 0, st, w, count, rscale);
    return hipGetLastError();
}

// ---- RMSNorm (src/quant/quant.cpp:384-398), one workgroup per row -------------------

__global__ __launch_bounds__(256) void k_rmsnorm(const float *x, const float *w, float *y,
                                                 int n, float eps) {
    const float *xr = x + (size_t)blockIdx.x * n;
    float *yr = y + (size_t)blockIdx.x * n;
    float ss = 0.f;
    for (int i = threadIdx.x; i < n; i += 256)
        ss = fmaf(xr[i], xr[i], ss);
    // wave sums, then across the four waves in fixed order
    for (int o = 32; o > 0; o >>= 1)
        ss += __shfl_xor(ss, o);
    __shared__ float part[4];
    if ((threadIdx.x & 63) == 0)
        part[threadIdx.x >> 6] = ss;
    __syncthreads();
    const float tot = ((part[0] + part[1]) + part[2]) + part[3];
    const float inv = 1.f / sqrtf(tot / (float)n + eps);
    for (int i = threadIdx.x; i < n; i += 256)
        yr[i] = w ? xr[i] * inv * w[i] : xr[i] * inv;
}

// The same with the row in registers (n % 4 == 0, n <= 4 * NV * NT, 16-byte aligned rows): x
// and w are read once, every load issued before the first is needed.  The loop above waits
// for memory 2 n / 256 times over (27 us at one row of 7168; this one: 5).
template <int NT, int NV>
__global__ __launch_bounds__(NT) void k_rmsnorm_reg(const float4 *x, const float4 *w, float4 *y,
                                                    int n4, float eps) {
    const int tid = threadIdx.x;
    const float4 *xr = x + (size_t)blockIdx.x * n4;
    float4 xv[NV], wv[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int i = tid + NT * j;
        xv[j] = i < n4 ? xr[i] : make_float4(0.f, 0.f, 0.f, 0.f);
        wv[j] = w && i < n4 ? w[i] : make_float4(1.f, 1.f, 1.f, 1.f);
    }
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        ss = fmaf(xv[j].x, xv[j].x, ss);
        ss = fmaf(xv[j].y, xv[j].y, ss);
        ss = fmaf(xv[j].z, xv[j].z, ss);
        ss = fmaf(xv[j].w, xv[j].w, ss);
    }
    for (int o = 32; o > 0; o >>= 1)
        ss += __shfl_xor(ss, o);
    __shared__ float part[NT / 64];
    if ((tid & 63) == 0)
        part[tid >> 6] = ss;
    __syncthreads();
    float tot = part[0];
#pragma unroll
    for (int v = 1; v < NT / 64; ++v)
        tot += part[v];
    const float inv = 1.f / sqrtf(tot / (float)(4 * n4) + eps);
    float4 *yr = y + (size_t)blockIdx.x * n4;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int i = tid + NT * j;
        if (i < n4)
            yr[i] = make_float4(xv[j].x * inv * wv[j].x, xv[j].y * inv * wv[j].y,
                                xv[j].z * inv * wv[j].z, xv[j].w * inv * wv[j].w);
    }
}

hipError_t launch_rmsnorm(const float *x, const float *w, float *y, int rows, int n, float eps,
                          hipStream_t st) {
    const uintptr_t al = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w) |
                         reinterpret_cast<uintptr_t>(y);
    const float4 *x4 = reinterpret_cast<const float4 *>(x), *w4 = reinterpret_cast<const float4 *>(w);
    float4 *y4 = reinterpret_cast<float4 *>(y);
    const dim3 grid((unsigned)rows);
    if (n % 4 || al % 16 || n > 16384)  // other rows: the loop
        hipLaunchKernelGGL(k_rmsnorm, grid, dim3(256), 0, st, x, w, y, n, eps);
    else if (n <= 2048)
        hipLaunchKernelGGL((k_rmsnorm_reg<256, 2>), grid, dim3(256), 0, st, x4, w4, y4, n / 4, eps);
    else if (n <= 8192)
        hipLaunchKernelGGL((k_rmsnorm_reg<512, 4>), grid, dim3(512), 0, st, x4, w4, y4, n / 4, eps);
    else
        hipLaunchKernelGGL((k_rmsnorm_reg<1024, 4>), grid, dim3(1024), 0, st, x4, w4, y4, n / 4, eps);
    return hipGetLastError();
}

}  // namespace mvllm_hip
