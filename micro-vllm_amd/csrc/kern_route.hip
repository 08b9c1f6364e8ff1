// kern_route.hip -- the routing in front of the expert block, on the device: moe_topk of
// every token (src/model/ops.cpp:860-889), then the moe_block segments of one batched
// call (the union of src/model/ops.cpp:1082-1099 and the per-expert gather of
// src/model/glm53.cpp:1938-1971 / src/model/kimi_k3.cpp:2009-2050).  Integer work and a
// few f32 additions and divisions in the reference's order: bit-exact.
//
//   k_moe_topk      one wave per token: k rounds of a wave-wide argmax under the
//                   reference's order (larger score first, lower index on ties), then the
//                   weights summed in pick order by every lane alike; for the router also
//                   the sigmoid, the bias and the weights' scale;
//   k_seg_count     per (token, slot): the expert's count of tokens whose summed weight
//                   is non-zero, and its presence (union membership: any slot);
//   k_seg_scan      one workgroup: experts in ascending id -> positions, row offsets,
//                   the capacity checks;
//   k_seg_rows      one workgroup per kept expert: its tokens in ascending order by a
//                   ballot per 256 tokens (two chunks a pass), written at the expert's
//                   row offset.
#include "mfma_common.h"

#include <algorithm>

namespace mvllm_hip {

constexpr int kTopkWaves = 4;

// A score as an unsigned key of the same order (-0 and +0 alike); 0 is kept for "taken".  The
// reference's sort has no order for NaN; by key it has one, so that every round picks some
// expert (a NaN that compared with nothing left lanes without one, and their -1 was read as an
// index).
__device__ __forceinline__ uint32_t rank_key(float v) {
    const uint32_t b = __float_as_uint(v + 0.f);  // -0 + 0 = +0
    return max(b ^ ((uint32_t)((int)b >> 31) | 0x80000000u), 1u);
}

// Wave-wide maximum of non-negative keys, by row shifts and broadcasts (lane 63 ends with
// it); a masked or missing source counts as 0.
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t dpp_max(uint32_t v) {
    return max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false));
}
__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
    v = dpp_max<0x111, 0xf>(v);  // row_shr 1, 2, 4, 8: lane 15 of each row
    v = dpp_max<0x112, 0xf>(v);
    v = dpp_max<0x114, 0xf>(v);
    v = dpp_max<0x118, 0xf>(v);
    v = dpp_max<0x142, 0xa>(v);  // row_bcast 15, 31
    v = dpp_max<0x143, 0xc>(v);
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// NV > 0: the lane's scores (elements lane + 64 s, s < NV) stay in registers as keys for
// all k rounds (n_exp <= 64 NV), each round one DPP maximum and a ballot: the chain of k
// rounds is the whole time, and an argmax by twelve cross-lane LDS permutes a round took
// 10 us at 384 experts, k = 8 (this one: 4.6, about a launch's own time).  NV = 0
// reads the scores again each round (up to 4096 experts).
// ROUTE: the router's tail in the same launch: choice (and part2, when K was split over two
// workgroups) hold the router GEMM's sums, mix = sigmoid(sum) is written to mix_out, mix +
// bias to choice_out, and the weights are scaled by rscale at the end
// (src/gpu/metal_ops.cpp:218-231).  The sums may lie in mix_out and choice_out: a wave
// reads its token's row before it writes it, and no other wave touches that row.
template <int NV, bool ROUTE>
__global__ __launch_bounds__(64 * kTopkWaves) void k_moe_topk(const float *choice,
                                                                const float *mix, int n_tok,
                                                                int n_exp, int k, int *idx,
                                                                float *wt, const float *part2,
                                                                const float *bias, float rscale,
                                                                float *mix_out,
                                                                float *choice_out) {
    static_assert(!ROUTE || NV > 0, "the router's tail keeps its row in registers");
    const int tok = blockIdx.x * kTopkWaves + (int)(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (tok >= n_tok)  // wave-uniform
        return;
    const float *row = choice + (size_t)tok * n_exp;
    int mine = -1;  // lane i < k: the i-th pick
    float w = 0.f;  // and its weight
    if constexpr (NV > 0) {
        uint32_t key[NV];
        float mx[ROUTE ? NV : 1];
        if constexpr (ROUTE) {
            float sc[NV], s2[NV], bv[NV];
#pragma unroll
            for (int s = 0; s < NV; ++s) {
                const int j = min(lane + 64 * s, n_exp - 1);
                sc[s] = row[j];
                s2[s] = part2 ? part2[(size_t)tok * n_exp + j] : 0.f;
                bv[s] = bias ? bias[j] : 0.f;
            }
#pragma unroll
            for (int s = 0; s < NV; ++s) {
                const int j = lane + 64 * s;
                mx[s] = mf_sigmoid(part2 ? sc[s] + s2[s] : sc[s]);
                const float c = mx[s] + bv[s];
                key[s] = j < n_exp ? rank_key(c) : 0u;
                if (j < n_exp) {
                    mix_out[(size_t)tok * n_exp + j] = mx[s];
                    choice_out[(size_t)tok * n_exp + j] = c;
                }
            }
        } else {
#pragma unroll
            for (int s = 0; s < NV; ++s)
                key[s] = lane + 64 * s < n_exp ? rank_key(row[lane + 64 * s]) : 0u;
        }
        for (int i = 0; i < k; ++i) {
            uint32_t bk = 0;
            int bs = 0;
            float bm = 0.f;
#pragma unroll
            for (int s = 0; s < NV; ++s)
                if (key[s] > bk) {  // the lane's lowest index on ties
                    bk = key[s];
                    bs = s;
                    if constexpr (ROUTE)
                        bm = mx[s];
                }
            const uint32_t m = wave_max(bk);
            const uint64_t cand = __ballot(bk == m);
            int win = __builtin_ctzll(cand);
            if (cand & (cand - 1))  // equal scores in several lanes: the lowest index
                win = (int)(~wave_max(bk == m ? ~(uint32_t)(bs * 64 + lane) : 0u) & 63u);
            const int ws = __builtin_amdgcn_readlane(bs, win);
            if (lane == win) {
#pragma unroll
                for (int s = 0; s < NV; ++s)
                    key[s] = s == bs ? 0u : key[s];
            }
            const int wm = __builtin_amdgcn_readlane((int)__float_as_uint(bm), win);
            if (lane == i) {
                mine = ws * 64 + win;
                w = __uint_as_float((uint32_t)wm);
            }
        }
    } else {
        uint64_t taken = 0;  // bit s: element lane + 64 s is picked (n_exp <= 4096)
        for (int i = 0; i < k; ++i) {
            uint32_t bk = 0;  // larger key first, lower index on ties (the reference comparator)
            int bi = -1;
            for (int s = 0; lane + 64 * s < n_exp; ++s) {
                const int j = lane + 64 * s;
                if ((taken >> s) & 1u)
                    continue;
                const uint32_t key = rank_key(row[j]);
                if (key > bk) {
                    bk = key;
                    bi = j;
                }
            }
            // the order is total on the candidates, so any reduction tree finds the same one
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) {
                const uint32_t ok = __shfl_xor(bk, off);
                const int oi = __shfl_xor(bi, off);
                if (ok > bk || (ok == bk && ok && oi < bi)) {
                    bk = ok;
                    bi = oi;
                }
            }
            if ((bi & 63) == lane)
                taken |= 1ull << (bi >> 6);
            if (lane == i)
                mine = bi;
        }
    }
    // weights: clipped at 0, summed in pick order (every lane adds the same sequence)
    if (lane < k) {
        if constexpr (!ROUTE)
            w = mix ? mix[(size_t)tok * n_exp + mine] : row[mine];
        if (w < 0.f)
            w = 0.f;
    }
    float sum = 0.f;
    for (int i = 0; i < k; ++i)
        sum += __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(w), i));
    if (lane < k) {
        idx[(size_t)tok * k + lane] = mine;
        float v = sum > 0.f ? w / sum : 1.f / (float)k;
        if constexpr (ROUTE)
            v = rscale != 1.f ? v * rscale : v;
        wt[(size_t)tok * k + lane] = v;
    }
}

// work layout (ints): cnt[n_exp] | pos[n_exp] (0 = absent, 1 = present; the scan turns
// it into the expert's position or -1) | flag (1: an id >= n_exp was seen)
__global__ __launch_bounds__(256) void k_seg_zero(int *work, int n) {
    for (int i = blockIdx.x * 256 + (int)threadIdx.x; i < n; i += (int)gridDim.x * 256)
        work[i] = 0;
}

// Summed weight of token c for expert e over its slots, in slot order from +0 (the
// reference's wsum).  Slots naming another expert add +0, which leaves the sum as it is:
// a sum started at +0 never becomes -0, and x + 0 = x otherwise (inf and NaN included).
// So every slot is loaded unconditionally and the loads issue together.
__device__ __forceinline__ float slot_wsum(const int *idx, const float *wt, int c, int topk,
                                           int e) {
    float ws = 0.f;
    for (int t = 0; t < topk; ++t) {
        const int id = idx[(size_t)c * topk + t];
        const float w = wt[(size_t)c * topk + t];
        ws += id == e ? w : 0.f;
    }
    return ws;
}

// One thread per (token, slot): the token's first slot naming an expert counts the token
// for it when the summed weight is non-zero; every named expert is present.
__global__ __launch_bounds__(256) void k_seg_count(const int *idx, const float *wt, int n_tok,
                                                   int topk, int n_exp, int *work) {
    const int i = blockIdx.x * 256 + (int)threadIdx.x;
    if (i >= n_tok * topk)
        return;
    const int c = i / topk, t = i - c * topk;
    const int e = idx[i];
    if (e < 0)
        return;
    if (e >= n_exp) {
        work[2 * n_exp] = 1;
        return;
    }
    bool first = true;
    for (int u = 0; u < t; ++u)
        first = first && idx[(size_t)c * topk + u] != e;
    if (!first)
        return;
    const float ws = slot_wsum(idx, wt, c, topk, e);
    work[n_exp + e] = 1;
    if (ws != 0.f)
        atomicAdd(work + e, 1);
}

// One workgroup of 1024: experts in ascending id.  counts = {nb, rows}, or {-1, -1} when
// cap_rows is short or an id is out of range.  The union keeps its cap_experts smallest
// ids, as the reference's union does.
__global__ __launch_bounds__(1024) void k_seg_scan(int n_exp, int *work, int cap_experts,
                                                   int cap_rows, int *eids, int *xoff, int *nr,
                                                   int *counts) {
    __shared__ int wsum_p[16], wsum_r[16];
    __shared__ int base_p, base_r;
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (tid == 0) {
        base_p = 0;
        base_r = 0;
    }
    __syncthreads();
    for (int e0 = 0; e0 < n_exp; e0 += 1024) {
        const int e = e0 + tid;
        const int p = e < n_exp ? work[n_exp + e] : 0;
        const int r = e < n_exp && p ? work[e] : 0;
        // inclusive scans within the wave
        int sp = p, sr = r;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int up = __shfl_up(sp, off), ur = __shfl_up(sr, off);
            if (lane >= off) {
                sp += up;
                sr += ur;
            }
        }
        if (lane == 63) {
            wsum_p[wave] = sp;
            wsum_r[wave] = sr;
        }
        __syncthreads();
        int bp = base_p, br = base_r;
        for (int w = 0; w < wave; ++w) {
            bp += wsum_p[w];
            br += wsum_r[w];
        }
        const int ui = bp + sp - p;  // exclusive: position among present experts
        const int ro = br + sr - r;  // rows before this expert
        if (e < n_exp) {
            const bool kept = p && ui < cap_experts;
            work[n_exp + e] = kept ? ui : -1;
            if (kept) {
                eids[ui] = e;
                xoff[ui] = ro;
                nr[ui] = r;
            }
        }
        __syncthreads();
        if (tid == 1023) {
            base_p = bp + sp;
            base_r = br + sr;
        }
        __syncthreads();
    }
    if (tid == 0) {
        // rows of the kept experts only: the dropped ones have the larger ids
        int nb = base_p < cap_experts ? base_p : cap_experts;
        int rows = 0;
        if (base_p <= cap_experts) {
            rows = base_r;
        } else {
            for (int e = 0; e < n_exp; ++e)  // truncated union (rare): count again
                if (work[n_exp + e] >= 0)
                    rows += work[e];
        }
        const bool bad = work[2 * n_exp] != 0 || rows > cap_rows;
        counts[0] = bad ? -1 : nb;
        counts[1] = bad ? -1 : rows;
    }
}

// One workgroup per expert id: the kept ones write their tokens (ascending) and sums.
// A pass covers kRowsChunks chunks of 256 tokens (token base + 256 r + thread), their
// id loads issued together, placed by one ballot per chunk and one barrier pair per
// pass.  Weights are loaded only for the slots that name the expert (loading every
// slot's weight measured 50 % slower here).
constexpr int kRowsChunks = 2;

__global__ __launch_bounds__(256) void k_seg_rows(const int *idx, const float *wt, int n_tok,
                                                  int topk, int n_exp, const int *work,
                                                  const int *xoff, const int *counts,
                                                  int *rows, float *rw) {
    __shared__ int wcnt[kRowsChunks][4];
    const int e = blockIdx.x;
    const int ui = work[n_exp + e];
    if (ui < 0 || counts[0] < 0)  // workgroup-uniform
        return;
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint64_t below = (1ull << lane) - 1ull;
    int j = xoff[ui];
    for (int base = 0; base < n_tok; base += 256 * kRowsChunks) {
        float ws[kRowsChunks];
        uint64_t m[kRowsChunks];
#pragma unroll
        for (int r = 0; r < kRowsChunks; ++r) {
            const int c = base + 256 * r + tid;
            ws[r] = 0.f;  // the reference's wsum: matching slots in slot order from +0
            if (c < n_tok)
                for (int t = 0; t < topk; ++t)
                    if (idx[(size_t)c * topk + t] == e)
                        ws[r] += wt[(size_t)c * topk + t];
            m[r] = __ballot(c < n_tok && ws[r] != 0.f);
            if (lane == 0)
                wcnt[r][wave] = __popcll(m[r]);
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kRowsChunks; ++r) {
            int before = 0, total = 0;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const int v = wcnt[r][w];
                total += v;
                before += w < wave ? v : 0;
            }
            if ((m[r] >> lane) & 1u) {
                const int pos = j + before + __popcll(m[r] & below);
                rows[pos] = base + 256 * r + tid;
                rw[pos] = ws[r];
            }
            j += total;
        }
        __syncthreads();  // wcnt is rewritten by the next pass
    }
}

// Small calls (at most kSegPairs (token, slot) pairs and kSegExperts experts): the whole
// construction in one workgroup and one launch instead of four, each of which costs a
// launch's ~4.6 us whatever it does.  One thread per pair: the token's first slot naming an
// expert stands for the token; its rank among the same expert's pairs of its wave's 64
// comes from 64 lane reads, the counts of the waves before from a table [wave][expert] in
// LDS, the row offsets from a scan over the experts.  Same results.
constexpr int kSegPairs = 1024, kSegExperts = 1024, kSegWaves = kSegPairs / 64;

__global__ __launch_bounds__(1024) void k_seg_small(const int *idx, const float *wt, int n_tok,
                                                    int topk, int n_exp, int cap_experts,
                                                    int cap_rows, int *eids, int *xoff, int *nr,
                                                    int *rows, float *rw, int *counts) {
    __shared__ int sid[kSegPairs];
    __shared__ float swt[kSegPairs];
    __shared__ uint8_t wcnt[kSegWaves][kSegExperts];  // rows of expert e among wave v's pairs
    __shared__ int ebase[kSegExperts];                // row offset of expert e, -1: not kept
    __shared__ uint8_t present[kSegExperts];
    __shared__ int wsum_p[16], wsum_r[16], flag, kept_rows, kept_n;
    const int tid = (int)threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int pairs = n_tok * topk, nv = (pairs + 63) / 64;
    if (tid == 0)
        flag = kept_rows = kept_n = 0;
    if (tid < pairs) {
        sid[tid] = idx[tid];
        swt[tid] = wt[tid];
    }
    for (int v = 0; v < nv; ++v)
        if (tid < n_exp)
            wcnt[v][tid] = 0;
    if (tid < n_exp)
        present[tid] = 0;
    __syncthreads();
    const int p = tid;     // this thread's pair
    int key = -1, rank = 0;  // the pair's expert when it makes a row; its rank in the wave
    float ws = 0.f;
    if (wave < nv) {  // wave-uniform
        if (p < pairs) {
            const int e = sid[p], c = p / topk, t0 = c * topk;
            bool first = e >= 0;
            if (e >= n_exp) {
                flag = 1;
                first = false;
            }
            for (int u = t0; u < p; ++u)
                first = first && sid[u] != e;
            if (first) {
                // the summed weight over the token's slots, in slot order from +0
                for (int u = 0; u < topk; ++u)
                    ws += sid[t0 + u] == e ? swt[t0 + u] : 0.f;
                present[e] = 1;
                if (ws != 0.f)
                    key = e;
            }
        }
        bool last = true;
        const int n = min(64, pairs - 64 * wave);
        for (int i = 0; i < n; ++i) {
            const int o = __builtin_amdgcn_readlane(key, i);
            rank += o == key && i < lane;
            last = last && !(o == key && i > lane);
        }
        if (key >= 0 && last)
            wcnt[wave][key] = (uint8_t)(rank + 1);
    }
    __syncthreads();
    // experts in ascending id: rows and presence, scanned over the workgroup
    const int e = tid;
    int r = 0;
    const int pr = e < n_exp ? present[e] : 0;
    if (e < n_exp)
        for (int v = 0; v < nv; ++v)
            r += wcnt[v][e];
    int sp = pr, sr = r;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int up = __shfl_up(sp, off), ur = __shfl_up(sr, off);
        if (lane >= off) {
            sp += up;
            sr += ur;
        }
    }
    if (lane == 63) {
        wsum_p[wave] = sp;
        wsum_r[wave] = sr;
    }
    __syncthreads();
    int bp = 0, br = 0;
    for (int w = 0; w < wave; ++w) {
        bp += wsum_p[w];
        br += wsum_r[w];
    }
    const int ui = bp + sp - pr, ro = br + sr - r;
    const bool kept = pr && ui < cap_experts;  // the union keeps its smallest ids
    if (e < n_exp)
        ebase[e] = kept ? ro : -1;
    if (kept) {
        eids[ui] = e;
        xoff[ui] = ro;
        nr[ui] = r;
        // the kept experts are a prefix of the present ones: the last one ends the rows
        atomicMax(&kept_n, ui + 1);
        atomicMax(&kept_rows, ro + r);
    }
    __syncthreads();
    const bool bad = flag != 0 || kept_rows > cap_rows;
    if (tid == 0) {
        counts[0] = bad ? -1 : kept_n;
        counts[1] = bad ? -1 : kept_rows;
    }
    if (bad)
        return;
    if (key >= 0 && ebase[key] >= 0) {
        int pos = ebase[key] + rank;
        for (int v = 0; v < wave; ++v)
            pos += wcnt[v][key];
        rows[pos] = p / topk;
        rw[pos] = ws;
    }
}

// NV of a row of n_exp scores: the smallest instance that holds it (0: none).
#define MVLLM_TOPK(ROUTE, ...)                                                              \
    do {                                                                                    \
        const dim3 grid((unsigned)((n_tok + kTopkWaves - 1) / kTopkWaves));                 \
        const dim3 block(64 * kTopkWaves);                                                  \
        const int nv = (n_exp + 63) / 64;                                                   \
        if (nv <= 1)                                                                        \
            hipLaunchKernelGGL((k_moe_topk<1, ROUTE>), grid, block, 0, st, __VA_ARGS__);    \
        else if (nv <= 2)                                                                   \
            hipLaunchKernelGGL((k_moe_topk<2, ROUTE>), grid, block, 0, st, __VA_ARGS__);    \
        else if (nv <= 4)                                                                   \
            hipLaunchKernelGGL((k_moe_topk<4, ROUTE>), grid, block, 0, st, __VA_ARGS__);    \
        else if (nv <= 6)                                                                   \
            hipLaunchKernelGGL((k_moe_topk<6, ROUTE>), grid, block, 0, st, __VA_ARGS__);    \
        else if (nv <= 8)                                                                   \
            hipLaunchKernelGGL((k_moe_topk<8, ROUTE>), grid, block, 0, st, __VA_ARGS__);    \
        else                                                                                \
            hipLaunchKernelGGL((k_moe_topk<0, false>), grid, block, 0, st, __VA_ARGS__);    \
    } while (0)

hipError_t launch_moe_topk(const float *choice, const float *mix, int n_tok, int n_exp, int k,
                           int *idx, float *wt, hipStream_t st) {
    if (n_tok < 1 || n_exp < 1 || n_exp > kRouteMaxExperts || k < 1 || k > 64 || k > n_exp)
        return hipErrorInvalidValue;
    MVLLM_TOPK(false, choice, mix, n_tok, n_exp, k, idx, wt, nullptr, nullptr, 1.f, nullptr,
               nullptr);
    return hipGetLastError();
}

hipError_t launch_route_topk(const float *sums, const float *sums2, const float *bias,
                             float rscale, int n_tok, int n_exp, int k, float *mix,
                             float *choice, int *idx, float *wt, hipStream_t st) {
    if (n_tok < 1 || n_exp < 1 || n_exp > kRouteTopkMax || k < 1 || k > 64 || k > n_exp)
        return hipErrorInvalidValue;
    MVLLM_TOPK(true, sums, nullptr, n_tok, n_exp, k, idx, wt, sums2, bias, rscale, mix, choice);
    return hipGetLastError();
}
#undef MVLLM_TOPK

hipError_t launch_moe_segments(const int *idx, const float *wt, int n_tok, int topk, int n_exp,
                               int *work, int *eids, int *xoff, int *nr, int *rows, float *rw,
                               int cap_experts, int cap_rows, int *counts, hipStream_t st) {
    if (n_tok < 1 || topk < 1 || n_exp < 1 || cap_experts < 1 || cap_rows < 1 ||
        (long long)n_tok * topk > (1ll << 30))
        return hipErrorInvalidValue;
    // one workgroup where a thread a pair covers the call (back to back, 384 experts, top 8: 1
    // token 14.1 -> 6.5 us, 61 tokens 14.1 -> 10.6, 128 tokens 14.1 -> 13.8; with two pairs a
    // thread it was slower than the four launches, 256 tokens 16.5 -> 19.3 us)
    if ((long long)n_tok * topk <= kSegPairs && n_exp <= kSegExperts) {
        hipLaunchKernelGGL(k_seg_small, dim3(1), dim3(1024), 0, st, idx, wt, n_tok, topk, n_exp,
                           cap_experts, cap_rows, eids, xoff, nr, rows, rw, counts);
        return hipGetLastError();
    }
    const int nw = 2 * n_exp + 1;
    hipLaunchKernelGGL(k_seg_zero, dim3((unsigned)std::min((nw + 255) / 256, 1024)), dim3(256), 0,
                       st, work, nw);
    const int pairs = n_tok * topk;
    hipLaunchKernelGGL(k_seg_count, dim3((unsigned)((pairs + 255) / 256)), dim3(256), 0, st, idx,
                       wt, n_tok, topk, n_exp, work);
    hipLaunchKernelGGL(k_seg_scan, dim3(1), dim3(1024), 0, st, n_exp, work, cap_experts, cap_rows,
                       eids, xoff, nr, counts);
    hipLaunchKernelGGL(k_seg_rows, dim3((unsigned)n_exp), dim3(256), 0, st, idx, wt, n_tok, topk,
                       n_exp, work, xoff, counts, rows, rw);
    return hipGetLastError();
}

hipError_t launch_moe_route(const float *choice, const float *mix, int n_tok, int n_exp, int k,
                            int *idx, float *wt, int *work, int *eids, int *xoff, int *nr,
                            int *rows, float *rw, int cap_experts, int cap_rows, int *counts,
                            hipStream_t st) {
    hipError_t e = launch_moe_topk(choice, mix, n_tok, n_exp, k, idx, wt, st);
    if (e != hipSuccess)
        return e;
    return launch_moe_segments(idx, wt, n_tok, k, n_exp, work, eids, xoff, nr, rows, rw,
                               cap_experts, cap_rows, counts, st);
}

}  // namespace mvllm_hip
