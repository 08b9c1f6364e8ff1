// kern_qrows.hip -- int4-g64 / MXFP4 matrices of any width on the gfx950 matrix cores with
// exact f32 activations: experts whose widths are not multiples of 256 (the decode and the
// grouped-GEMM kernels need that), and dense linears over few rows.
//
// C[r, o] = sum_k X[r, k] * W[o, k], W formed exactly (src/quant/quant.cpp:203-228, 298-321).
// An f32 x is the sum of three bf16 terms (its 24 significant bits cut in three: hi =
// the upper 16 bits of x, mid = those of x - hi, lo = the rest), so every product
// with a decoded weight is exact in f32 and only the sums round, as in the element-wise
// kernel this replaces for these shapes.
//
// Work item = (expert, block of up to 16 * MT rows) x (block of columns).  K goes in blocks
// of 64: lane (t, q) holds 8 bytes of weight row t (K elements 16 q .. + 15 of the block) and
// the same 16 elements of input row t, and MFMA step s takes its 8 elements 8 s .. + 7.  The
// W waves of a workgroup split the blocks of the same NT tiles of 16 weight rows and add
// their partial sums in LDS in wave order.
//   int4: nibbles decode to bf16(n - 8), one chain per 64-wide group and tile, then one f32
//   FMA applies the group's scale.  (A chain over n from -8 sum x decodes with fewer
//   instructions, but its cancellation cost accuracy: 2.5e-7 against 1.5e-7 of 64 bits.)
//   MXFP4: the block's scale is folded into the decode (exact for bytes 2..252), one chain
//   per 64-wide block that then adds to the sum (experts of 1568 x 928 are 1.21e-7 from 64
//   bits; one chain over all of a wave's K 1.80e-7, the element-wise kernel 1.35e-7).
// A wave that meets an activation of 2^118 or more (a group's unscaled sum could overflow
// where the reference's does not), a non-finite int4 scale or another MXFP4 scale byte forms
// its sums again element by element, as the reference does.
//
// Bound by the latency of the loads of the few waves that its registers allow, then by the
// vector ALU (the split of x, the decode): NT tiles share one split.  24 tokens, 32 int4
// experts of 2112 x 704 (81 MB): gate/up 186 -> 33 us, down 99 -> 17 us against the
// element-wise kernel (one nibble a lane and step).
#include "mfma_common.h"

#include <algorithm>

namespace mvllm_hip {

struct QItem {
    int a, r0, nrow, pad;
};

struct QArgs {
    const ExpertWork *ew;
    const QItem *items;     // null: one expert (ew1), items of 16 * MT rows over nrows_all
    ExpertWork ew1;
    int nrows_all;
    const float *in;        // input rows [*][K]
    const int *in_rows;     // compact row -> input row (null: identity)
    float *out;             // output rows [rcap][O]
    int mi;                 // single: which matrix of the expert
    int nbn, n_tasks;       // column blocks; items * nbn
    int K, O;
    int act;
    float act_a, act_b;
};

// x's upper 16 bits (a bf16 by truncation) as f32
__device__ __forceinline__ float bf_top(float x) {
    return __uint_as_float(__float_as_uint(x) & 0xffff0000u);
}
// the upper halves of two f32 as a bf16 pair (a first)
__device__ __forceinline__ uint32_t bf_pair(float a, float b) {
    return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}

template <int FMT, bool DUAL, int MT, int NT, int W>
__global__ __launch_bounds__(64 * W) void k_q_rows(QArgs A) {
    constexpr int U = MT == 1 ? 2 : 1;  // K blocks a group: two groups in flight
    constexpr int CT = DUAL ? NT / 2 : NT;  // column tiles of 16
    static_assert(!DUAL || NT % 2 == 0, "dual: gate and up tiles in pairs");
    __shared__ float red[W][MT * NT * 256];
    const int task = xcd_task(blockIdx.x, A.n_tasks);
    const int item = task / A.nbn, cb = task - item * A.nbn;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, t = lane & 15, q = lane >> 4;
    const int K = A.K, O = A.O, col0 = cb * 16 * CT;
    const int rowb = K >> 1, ngs = FMT == 4 ? (K + 63) / 64 : (K + 31) / 32;
    QItem it;
    if (A.items) {
        it = A.items[item];
    } else {
        it.a = 0;
        it.r0 = item * 16 * MT;
        it.nrow = min(16 * MT, A.nrows_all - it.r0);
    }
    const ExpertWork &ew = A.items ? A.ew[it.a] : A.ew1;
    const int jbase = ew.row0 + it.r0;
    auto src_row = [&] __attribute__((always_inline)) (int r) {
        const int j = jbase + min(r, it.nrow - 1);  // rows past the item repeat the last
        return A.in_rows ? A.in_rows[j] : j;
    };
    auto mat = [&] __attribute__((always_inline)) (int m) { return DUAL ? m & 1 : A.mi; };
    // weight row of tile m at this lane; past the matrix: its last row, not stored
    auto wrow = [&] __attribute__((always_inline)) (int m) {
        return min(col0 + 16 * (DUAL ? m >> 1 : m) + t, O - 1);
    };
    const float4 *xr[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
        xr[mt] = reinterpret_cast<const float4 *>(A.in + (size_t)src_row(mt * 16 + t) * K) + 4 * q;
    const uint8_t *wr[NT];
    const uint8_t *sr[NT];
#pragma unroll
    for (int m = 0; m < NT; ++m) {
        const size_t row = (size_t)wrow(m);
        wr[m] = static_cast<const uint8_t *>(ew.w[mat(m)]) + row * rowb + 8 * q;
        sr[m] = static_cast<const uint8_t *>(ew.s[mat(m)]) + row * ngs * (FMT == 4 ? 4 : 1) +
                (FMT == 4 ? 0 : q >> 1);
    }
    f4v acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int m = 0; m < NT; ++m)
            acc[mt][m] = f4v{0.f, 0.f, 0.f, 0.f};
    struct Buf {
        float4 x[U][MT][4];
        u32x2 w[U][NT];
        float s[U][NT];  // the f32 scale, or the ue8m0 byte's value
    };
    const int nb = K / 64, kb0 = nb * wave / W, kb1 = nb * (wave + 1) / W;
    const int klast = max(kb1 - 1, 0);
    auto load = [&] __attribute__((always_inline)) (Buf &b, int kb) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = min(kb + u, klast);
#pragma unroll
            for (int m = 0; m < NT; ++m) {
                b.w[u][m] = *reinterpret_cast<const u32x2 *>(wr[m] + 32 * (size_t)k);
                if constexpr (FMT == 4)
                    b.s[u][m] = reinterpret_cast<const float *>(sr[m])[k];
                else
                    b.s[u][m] = __uint_as_float((uint32_t)sr[m][2 * (size_t)k] << 23);
            }
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    b.x[u][mt][v] = xr[mt][16 * (size_t)k + v];
        }
    };
    float xmax = 0.f;   // largest |x| met (2^118 up: the wave's sums are formed again)
    uint32_t exc = 0;   // a scale that the decode does not reproduce
    auto compute = [&] __attribute__((always_inline)) (const Buf &b, int u) {
        __builtin_amdgcn_sched_barrier(0);
        bf16x8 w[NT][2];
#pragma unroll
        for (int m = 0; m < NT; ++m) {
            if constexpr (FMT == 4) {
                w[m][0] = decode_b4_signed(b.w[u][m].x);
                w[m][1] = decode_b4_signed(b.w[u][m].y);
            } else {
                w[m][0] = decode_b<FMT>(b.w[u][m].x, b.s[u][m]);
                w[m][1] = decode_b<FMT>(b.w[u][m].y, b.s[u][m]);
            }
            exc |= (uint32_t)(FMT == 4 ? nonfinite(b.s[u][m]) : b7_exceptional(b.s[u][m]));
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            __builtin_amdgcn_sched_barrier(0);  // one row tile's terms live at a time
            bf16x8 a[3][2];
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const float4 f0 = b.x[u][mt][2 * s], f1 = b.x[u][mt][2 * s + 1];
                const float x[8] = {f0.x, f0.y, f0.z, f0.w, f1.x, f1.y, f1.z, f1.w};
                float mid[8], lo[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    xmax = fmaxf(xmax, fabsf(x[e]));
                    mid[e] = x[e] - bf_top(x[e]);
                    lo[e] = mid[e] - bf_top(mid[e]);
                }
                // pairs of elements in the operand's slot order (int4: 0 2 4 6 1 3 5 7)
                auto pack = [&] __attribute__((always_inline)) (const float (&v)[8]) {
                    if constexpr (FMT == 4)
                        return __builtin_bit_cast(bf16x8, u32x4{bf_pair(v[0], v[2]), bf_pair(v[4], v[6]),
                                                                bf_pair(v[1], v[3]), bf_pair(v[5], v[7])});
                    else
                        return __builtin_bit_cast(bf16x8, u32x4{bf_pair(v[0], v[1]), bf_pair(v[2], v[3]),
                                                                bf_pair(v[4], v[5]), bf_pair(v[6], v[7])});
                };
                a[0][s] = pack(x);
                a[1][s] = pack(mid);
                a[2][s] = pack(lo);
            }
#pragma unroll
            for (int m = 0; m < NT; ++m) {
                f4v c = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int tm = 2; tm >= 0; --tm)
#pragma unroll
                    for (int s = 0; s < 2; ++s)
                        c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[tm][s], w[m][s], c, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    acc[mt][m][i] = FMT == 4 ? fmaf(b.s[u][m], c[i], acc[mt][m][i])
                                             : acc[mt][m][i] + c[i];
            }
        }
    };
    // groups of U blocks, two buffers; the pair loop has no exit between its two halves
    Buf b0, b1;
    int kb = kb0;
    load(b0, kb);
    for (; kb + 2 * U <= kb1; kb += 2 * U) {
        load(b1, kb + U);
#pragma unroll
        for (int u = 0; u < U; ++u)
            compute(b0, u);
        load(b0, kb + 2 * U);
#pragma unroll
        for (int u = 0; u < U; ++u)
            compute(b1, u);
    }
    load(b1, kb + U);
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (kb + u < kb1)
            compute(b0, u);
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (kb + U + u < kb1)
            compute(b1, u);
    // the last, partial block of K (16, 32 or 48 elements): lanes past it hold zeros
    const int krem = K - 64 * nb;
    if (krem && wave == W - 1) {
        const bool in = 16 * q < krem;
#pragma unroll
        for (int m = 0; m < NT; ++m) {
            b0.w[0][m] = *reinterpret_cast<const u32x2 *>(wr[m] + (in ? 32 * (size_t)nb : 0));
            if constexpr (FMT == 4)
                b0.s[0][m] = reinterpret_cast<const float *>(sr[m])[nb];
            else
                b0.s[0][m] = in ? __uint_as_float((uint32_t)sr[m][2 * (size_t)nb] << 23) : 1.f;
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                b0.x[0][mt][v] = in ? xr[mt][16 * (size_t)nb + v] : make_float4(0.f, 0.f, 0.f, 0.f);
        compute(b0, 0);
    }
    // C[4 q + i][t] of row tile mt and tile m -> LDS
    float *mine = red[wave];
    if (__any(exc != 0 || xmax >= 0x1p118f)) {
        const int k0 = 64 * kb0, k1 = wave == W - 1 ? K : 64 * kb1;
        for (int e = 0; e < MT * NT * 4; ++e) {
            const int mt = e / (4 * NT), m = e / 4 % NT, i = e & 3;
            const float *x = A.in + (size_t)src_row(mt * 16 + 4 * q + i) * K;
            const size_t row = (size_t)wrow(m);
            const uint8_t *wp = static_cast<const uint8_t *>(ew.w[mat(m)]) + row * rowb;
            float v = 0.f;
            for (int k = k0; k < k1; ++k) {
                const uint32_t n = (wp[k >> 1] >> (4 * (k & 1))) & 15u;
                float w;
                if constexpr (FMT == 4)
                    w = (float)((int)n - 8) *
                        static_cast<const float *>(ew.s[mat(m)])[row * ngs + k / 64];
                else
                    w = e2m1_val(n) *
                        ue8m0_ref(static_cast<const uint8_t *>(ew.s[mat(m)])[row * ngs + k / 32]);
                v += x[k] * w;
            }
            mine[(mt * NT + m) * 256 + i * 64 + lane] = v;
        }
    } else {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int m = 0; m < NT; ++m)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    mine[(mt * NT + m) * 256 + i * 64 + lane] = acc[mt][m][i];
    }
    __syncthreads();
    auto sum = [&] __attribute__((always_inline)) (int at) {
        float v = red[0][at];
#pragma unroll
        for (int w = 1; w < W; ++w)
            v += red[w][at];
        return v;
    };
    for (int e = tid; e < MT * CT * 256; e += 64 * W) {
        const int tile = e >> 8, pos = e & 255;
        const int mt = tile / CT, ct = tile - mt * CT;
        const int r = mt * 16 + 4 * ((pos >> 4) & 3) + (pos >> 6);
        const int col = col0 + 16 * ct + (pos & 15);
        if (r >= it.nrow || col >= O)
            continue;
        float *dst = A.out + (size_t)(jbase + r) * O + col;
        if constexpr (DUAL) {
            const int g = (mt * NT + 2 * ct) * 256 + pos;
            *dst = mf_act(A.act, sum(g), sum(g + 256), A.act_a, A.act_b);
        } else {
            *dst = sum((mt * NT + ct) * 256 + pos);
        }
    }
}

// K >= 64: the loads before the partial block read a whole 64-wide one (rows of fewer elements
// end before lane q's 16 of it).
bool q_rows_fits(int fmt, int K) { return (fmt == 4 || fmt == 7) && K >= 64 && K % 16 == 0; }

// Weight tiles of 16 a wave holds and, with them, the workgroups of a launch.  Four tiles share
// one split of x, two give more workgroups: 4 from 512 two-tile tasks on (2 per CU).
static int q_rows_tiles(bool dual, int mt, long long n_items, int O) {
    const long long t2 = n_items * ((O + (dual ? 15 : 31)) / (dual ? 16 : 32));
    return mt == 1 && t2 >= 512 ? 4 : 2;
}
static long long q_rows_tasks(bool dual, long long n_items, int O, int nt) {
    const int cols = (dual ? 8 : 16) * nt;
    return n_items * ((O + cols - 1) / cols);
}

// A linear's few rows of a short K as one launch, where the planes, the GEMM and the sum of its
// splits are three (7168 x 512 at 1 row 9.2 -> 6.0 us, at 32 rows 11.5 -> 6.8; 7168 x 1024 at
// 16 rows 13.0 -> 9.9, 7168 x 2048 at 1 row 12.8 -> 11.0; equal at 2048 and 16 rows, behind past
// it: 6144 at 1 row 14.6 -> 19.6).  A workgroup's time grows with K and a second one on a CU
// runs after the first, so only launches of at most a workgroup a CU, two of a shorter K, are
// ahead of the planes, which take three terms for such calls and whose GEMM reads wide
// matrices at the HBM's rate (32768 x 512 at 33 rows 37 us against 14, 65536 x 2048 at 1 row 49
// against 23, 28672 x 512 at 1 row 11.9 against 9.9; MXFP4 12288 x 1024 at 32 rows 19.6 against
// 17.2, at 4 rows 10.8 against 12.2, 7168 x 256 at 100 rows 17.8 against 9.9).
bool q_rows_linear(int K, int O, int n) {
    const int mt = n <= 16 ? 1 : 2, nb = (n + 15) / 16, items = (n + 16 * mt - 1) / (16 * mt);
    const bool wide = O > 8192;
    const long long tasks = q_rows_tasks(false, items, O, q_rows_tiles(false, mt, items, O));
    if (wide && (O > 16384 || K > 1024 || (K == 1024 && n > 8)))
        return false;
    return (long long)K * nb <= (wide ? 1536 : 2048) && tasks <= (wide || K <= 768 ? 512 : 256);
}

hipError_t launch_q_rows(int fmt, bool dual, int mt, const ExpertWork *ew, const void *items,
                         int n_items, const ExpertWork *ew1, int nrows_all, const float *in,
                         const int *in_rows, float *out, int mi, int K, int O, int act,
                         float act_a, float act_b, hipStream_t st) {
    if (!q_rows_fits(fmt, K) || O < 1 || (mt != 1 && mt != 2) || (!items && !ew1))
        return hipErrorInvalidValue;
    QArgs a{};
    a.ew = ew;
    a.items = static_cast<const QItem *>(items);
    if (ew1)
        a.ew1 = *ew1;
    a.nrows_all = nrows_all;
    a.in = in;
    a.in_rows = in_rows;
    a.out = out;
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
    // Four waves a workgroup: its start and end weigh less than a finer split of these short
    // rows gains.  24 tokens, 32 int4 experts of 2112 x 704, per call: 55 us (4 tiles), 61 (2
    // tiles), 74 and 91 us with eight waves; 100 tokens, 64 MXFP4 experts of 2080 x 1056: 144 /
    // 168 / 181 / 222 us; one token, 4 of 2592 x 1248: 34 / 32 / 34 / 38.
    const int nt = q_rows_tiles(dual, mt, n_items, O), w = mt == 1 ? 4 : 8;
    const int cols = (dual ? 8 : 16) * nt;
    a.nbn = (O + cols - 1) / cols;
    a.n_tasks = (int)q_rows_tasks(dual, n_items, O, nt);
    const dim3 grid((unsigned)a.n_tasks), block((unsigned)(64 * w));
#define MVLLM_Q(F, D, M, N, W_) hipLaunchKernelGGL((k_q_rows<F, D, M, N, W_>), grid, block, 0, st, a)
#define MVLLM_Q_MT(F, D)                          \
    do {                                          \
        if (mt == 2) MVLLM_Q(F, D, 2, 2, 8);      \
        else if (nt == 4) MVLLM_Q(F, D, 1, 4, 4); \
        else MVLLM_Q(F, D, 1, 2, 4);              \
    } while (0)
    if (fmt == 4) {
        if (dual) MVLLM_Q_MT(4, true); else MVLLM_Q_MT(4, false);
    } else {
        if (dual) MVLLM_Q_MT(7, true); else MVLLM_Q_MT(7, false);
    }
#undef MVLLM_Q_MT
#undef MVLLM_Q
    return hipGetLastError();
}

}  // namespace mvllm_hip
