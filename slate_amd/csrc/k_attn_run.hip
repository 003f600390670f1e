// k_attn_run.hip -- ragged attention of many query tokens over f32 caches:
// runs of consecutive tokens share their K/V rows on the f32 MFMA.
//
// attention_ragged takes its tokens one by one (sequence and position per
// token, in device memory), so a prompt chunk arrives as tokens that follow
// each other in one sequence.  attn_token_kernel (k_attn.hip) finds these
// runs on the device and cuts them into units of up to 16 / G tokens (16 query
// rows with the G heads of a group) times a chunk of 256 keys; attn_run_kernel
// streams each unit's K and V rows once for all its rows.  A token that
// follows no other is a unit of its own.
//
// A unit's four waves own up to 64 keys each.  Scores are S^T = K Q^T (16 keys x 16
// rows per MFMA tile, 4 dims a step): a lane holds scores of one row, keys
// 4g .. 4g+3 of each tile, which is the layout that O^T += V^T P^T takes as
// its second operand, so probabilities never leave their registers.  A wave
// passes its K tiles, then its V tiles, through one LDS tile of its own:
// whole lines in (global -> LDS copies; operand loads straight from the rows
// touch 16 lines each), a tile into registers, and the next copy in flight
// while the tile is used.  All values, products and sums are f32, added in
// short chains and trees, so that the result is no further from 64 bits than
// the token-by-token kernel's (1.11e-7 against 1.16e-7 at 8 kv heads of 128,
// 35 decode tokens and two chunks of up to 127).
//
// Bound: the f32 MFMA (64 flops a clock and SIMD; busy 40 % of the time) and
// the vector ALUs beside it (softmax, tree sums).  13 decode tokens at ~900
// keys and three chunks of 121-172 tokens (32 q / 8 kv heads of 128), the
// whole call: 139 us token by token, 89 here; 32 q and kv heads of 128, four
// chunks of up to 98 tokens: 55 and 28 us; 16 q / 4 kv heads of 64, four of up
// to 68 beside nine decode tokens: 32 and 23.  Lone tokens gain nothing, and
// lose at short contexts: such calls go to the token kernel (attn_runs.h).  32
// rows a unit halve the K/V traffic but leave two waves a SIMD: 102 us.  Chains of four MFMAs fit 128
// registers (four waves; 86 us where these took 93), but round 3 to 10 % worse.
#include <algorithm>
#include <cfloat>

#include "launch.h"
#include "attn_runs.h"
#include "mfma.h"

namespace slate_hip {

constexpr int ARN_KW = 64;           // keys per wave, at most

template <int HD>
struct RunGeom {
    static constexpr int NT = HD / 16;                      // 16-byte K pieces of a lane, 16-dim output tiles
    static constexpr int VW = NT < 4 ? NT : 4;              // floats of a V load
    static constexpr int NB = NT / VW;                      // V loads of a row
    static constexpr int CPR = HD / 4;                      // 16-byte pieces of a row
    static constexpr int TILE = 16 * HD;                    // floats of 16 rows
    // LDS floats per wave: a K or V tile, then the outputs of 16 rows (or the
    // probabilities of 16 rows and 64 keys)
    static constexpr int WAVE = ARN_ROWS * (HD > ARN_KW ? HD : ARN_KW);
    // float offset of element d of row r in an LDS tile: the row's 16-byte
    // pieces are stored in an order of its own, so that one piece of 16
    // consecutive rows covers every bank once
    static __device__ __forceinline__ int at(int r, int d) {
        const int c = d >> 2;
        return 4 * (c & ~15) + (r * HD + 4 * ((c & 15) ^ swz(r))) + (d & 3);
    }
    static __device__ __forceinline__ int swz(int r) { return CPR >= 16 ? r & 15 : (r >> 1) & (CPR - 1); }
};

// The wave's own loads and LDS operations, ordered against LDS accesses
// before and after (the copies below are not known to the compiler).
__device__ __forceinline__ void wait_copies() { asm volatile("s_waitcnt vmcnt(0)" : : : "memory"); }
__device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory"); }

template <int HD, int G>
__device__ __forceinline__ void attn_run_unit(const float* q, const float* Kp, const float* Vp, const RunUnit& un,
                                              int h, int Hq, int64_t head_stride, int nch_max,
                                              float* __restrict__ po, float* __restrict__ pml, float* s_o,
                                              float* s_q) {
    using Geo = RunGeom<HD>;
    constexpr int NT = Geo::NT, VW = Geo::VW, NB = Geo::NB, CPR = Geo::CPR, KT = ARN_KW / 16, R = ARN_ROWS;
    typedef float vf_t __attribute__((ext_vector_type(VW)));
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));   // the unit's LDS offsets are computed here, not held across the units' loop
    const int lane = tid & 63, j = lane & 15, g = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int k0 = un.c * ARN_CHUNK;
    const int nk = min(un.p0 + un.n - k0, ARN_CHUNK);       // keys some row of the unit sees
    // the chunk's keys in whole tiles over the four waves (a chunk of 130 keys
    // as 48 + 48 + 34, not 64 + 64 + 2)
    const int kw = (nk + 63) / 64 * 16, kw0 = wv * kw;
    const int kn = min(nk - kw0, kw);                       // the wave's keys
    const bool active = kn > 0;
    const float scale = 1.0f / sqrtf((float)HD);
    const int64_t key0 = un.kvb + (int64_t)h * head_stride + (int64_t)k0 * HD;   // the chunk's first key
    const float* Kh = Kp + key0;
    const float* Vh = Vp + key0;
    float* so = s_o + wv * Geo::WAVE;
    // ---- the unit's query rows (row r: token r / G, head r % G; rows past
    // its tokens repeat the last one), and the wave's first K tile
    constexpr int QJ = (R * CPR + 255) / 256;
    floatx4 qv[QJ];
#pragma unroll
    for (int x = 0; x < QJ; ++x) {
        const int idx = min(tid + 256 * x, R * CPR - 1), r = idx / CPR, c = idx % CPR;
        qv[x] = *(const floatx4*)(q + ((size_t)(un.t0 + min(r / G, un.n - 1)) * Hq + h * G + r % G) * HD + 4 * c);
    }
    __builtin_amdgcn_sched_barrier(0);
    // 16 rows from key kw0 + 16 kt of a pool into the wave's LDS tile, RP rows
    // a copy.  Piece c of row x * RP + hi lies at piece c ^ swz(row): the
    // lane's source offset within a copy's rows differs from copy to copy in
    // the bits of x alone.  Rows past the last key repeat it.
    constexpr int RP = 64 / CPR;
    auto copy = [&](const float* src, int kt) {
        int ln = lane;
        asm volatile("" : "+v"(ln));                        // offsets computed per tile, not kept from K for V
        const int hi = ln / CPR;
        const int row0 = kw0 + 16 * kt;
        if (row0 + 16 <= nk) {
            const uint32_t off = (uint32_t)(hi * HD * 4 | ((ln % CPR) ^ Geo::swz(hi)) << 4);
#pragma unroll
            for (int x = 0; x < NT; ++x)
                lds_copy16(src + (size_t)(row0 + x * RP) * HD, off ^ (uint32_t)(Geo::swz(x * RP) << 4),
                           lds_addr(so + x * 256));
        } else {
#pragma unroll
            for (int x = 0; x < NT; ++x) {
                const int r = x * RP + hi, c = (ln % CPR) ^ Geo::swz(r);
                lds_copy16(src, (uint32_t)((min(row0 + r, nk - 1) * HD + 4 * c) * 4), lds_addr(so + x * 256));
            }
        }
    };
    if (active) copy(Kh, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int x = 0; x < QJ; ++x) {
        const int idx = tid + 256 * x, r = idx / CPR, c = idx % CPR;
        if (idx < R * CPR) *(floatx4*)(s_q + Geo::at(r, 4 * c)) = qv[x];
    }
    __syncthreads();
    floatx4 qf[NT];
#pragma unroll
    for (int m = 0; m < NT; ++m) qf[m] = *(const floatx4*)(s_q + Geo::at(j, 16 * m + 4 * g));
    __syncthreads();                                        // s_q is free: the waves' maxima and sums go there
    float* s_m = s_q;                                       // [row][wave]
    float* s_l = s_q + 4 * R;                               // [wave][row]
    floatx4 s[KT];
    if (active) {
        const int vis = un.p0 + min(j / G, un.n - 1) - k0;  // last key of the chunk that the lane's row sees
        // ---- scores: chains of two MFMAs (8 dims) from zero, added pairwise
        // (one chain over all dims rounds on growing sums: 1.9e-7 against 64
        // bits where these show 1.2e-7)
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) {
            s[kt] = floatx4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
            if (16 * kt >= kn) continue;
            wait_copies();
            floatx4 kf[NT];
#pragma unroll
            for (int m = 0; m < NT; ++m) kf[m] = *(const floatx4*)(so + Geo::at(j, 16 * m + 4 * g));
            wait_lds();                                     // the tile is in registers: the next one may land
            if (16 * (kt + 1) < kn) copy(Kh, kt + 1);
            else copy(Vh, 0);
            __builtin_amdgcn_sched_barrier(0);
            floatx4 tr[4];                                  // pending partial sums of the pairwise tree
#pragma unroll
            for (int m = 0; m < NT; ++m) {
                floatx4 t[2] = {floatx4{0.f, 0.f, 0.f, 0.f}, floatx4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
                for (int e = 0; e < 2; ++e)
#pragma unroll
                    for (int x = 0; x < 2; ++x)
                        t[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[m][2 * x + e], qf[m][2 * x + e], t[x],
                                                                    0, 0, 0);
                t[0] += t[1];
                int lv = 0;
#pragma unroll
                for (; (m >> lv) & 1; ++lv) t[0] = tr[lv] + t[0];
                tr[lv] = t[0];
                // two chains at a time: left to itself the scheduler starts
                // more than the registers hold
                __builtin_amdgcn_sched_barrier(0);
            }
            s[kt] = tr[NT == 8 ? 3 : (NT == 4 ? 2 : 1)];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int k = kw0 + 16 * kt + 4 * g + i;
                s[kt][i] = k <= vis ? s[kt][i] * scale : -INFINITY;   // (vis < nk)
            }
        }
        // ---- the rows' maxima over the unit's keys (lanes j, j+16, j+32, j+48
        // share a row), so that the waves' sums simply add
        float mw = -INFINITY;
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
            for (int i = 0; i < 4; ++i) mw = fmaxf(mw, s[kt][i]);
        mw = fmaxf(mw, __shfl_xor(mw, 16));
        mw = fmaxf(mw, __shfl_xor(mw, 32));
        if (g == 0) s_m[4 * j + wv] = mw;
    } else if (g == 0) {
        s_m[4 * j + wv] = -INFINITY;
    }
    __syncthreads();
    if (active) {
        const floatx4 m4 = *(const floatx4*)(s_m + 4 * j);
        const float mx = fmaxf(fmaxf(m4[0], m4[1]), fmaxf(m4[2], m4[3]));
        float st[KT];
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float x = s[kt][i];
                s[kt][i] = x == -INFINITY ? 0.f : expf(x - mx);
            }
            st[kt] = (s[kt][0] + s[kt][1]) + (s[kt][2] + s[kt][3]);
        }
        float sum = (st[0] + st[1]) + (st[2] + st[3]);
        sum += __shfl_xor(sum, 16);
        sum += __shfl_xor(sum, 32);
        // ---- output: tile b*VW + c, register i of lane (j, g): row j, dim
        // 16*VW*b + VW*(4g + i) + c; a tile's 16 keys as two chains
        floatx4 acc[NT];
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[n] = floatx4{0.f, 0.f, 0.f, 0.f};
        // keys that some row of the wave's range does not see: 0 * V there
        // would carry an infinity or NaN of a later token's V row into it
        const int diag = un.p0 - k0;
        bool bad = false;
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) {
            if (16 * kt >= kn) continue;
            wait_copies();
            // lane (j, g): key 4g + i, dims VW*j .. of each VW*16-dim block
            vf_t vf[4][NB];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int b = 0; b < NB; ++b) vf[i][b] = *(const vf_t*)(so + Geo::at(4 * g + i, 16 * VW * b + VW * j));
            wait_lds();
            if (16 * (kt + 1) < kn) copy(Vh, kt + 1);
            __builtin_amdgcn_sched_barrier(0);
            if (kw0 + 16 * kt + 15 > diag)
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int b = 0; b < NB; ++b)
#pragma unroll
                        for (int c = 0; c < VW; ++c) bad |= !(fabsf(vf[i][b][c]) <= FLT_MAX);
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int c = 0; c < VW; ++c) {
                    floatx4 t[2] = {floatx4{0.f, 0.f, 0.f, 0.f}, floatx4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int x = 0; x < 2; ++x)
                            t[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[2 * x + i][b][c], s[kt][2 * x + i],
                                                                        t[x], 0, 0, 0);
                    acc[b * VW + c] += t[0] + t[1];
                    __builtin_amdgcn_sched_barrier(0);
                }
        }
        if (__any(bad)) {
            // some V value there is not finite: each row over its own keys alone
#pragma unroll
            for (int kt = 0; kt < KT; ++kt)
#pragma unroll
                for (int i = 0; i < 4; ++i) so[j * ARN_KW + 16 * kt + 4 * g + i] = s[kt][i];
#pragma unroll
            for (int n = 0; n < NT; ++n) acc[n] = floatx4{0.f, 0.f, 0.f, 0.f};
            wait_lds();
            for (int k = 0; k < kn; ++k)
                if (k0 + kw0 + k <= un.p0 + min(j / G, un.n - 1)) {
                    const float pk = so[j * ARN_KW + k];
                    const float* vr = Vh + (int64_t)(kw0 + k) * HD;
#pragma unroll
                    for (int b = 0; b < NB; ++b)
#pragma unroll
                        for (int i = 0; i < 4; ++i)
#pragma unroll
                            for (int c = 0; c < VW; ++c)
                                acc[b * VW + c][i] = __builtin_fmaf(pk, vr[16 * VW * b + VW * (4 * g + i) + c],
                                                                    acc[b * VW + c][i]);
                }
            wait_lds();
        }
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                vf_t o;
#pragma unroll
                for (int c = 0; c < VW; ++c) o[c] = acc[b * VW + c][i];
                *(vf_t*)(so + Geo::at(j, 16 * VW * b + VW * (4 * g + i))) = o;
            }
        if (g == 0) s_l[wv * R + j] = sum;
    }
    __syncthreads();
    const int nw = (nk + kw - 1) / kw;                      // waves that had keys
    for (int idx = tid; idx < R * CPR; idx += 256) {
        const int r = idx / CPR, d = 4 * (idx % CPR), i = r / G;
        if (i >= un.n || un.p0 + i < k0) continue;          // the merge reads no chunk past a token's end
        floatx4 o = *(const floatx4*)(s_o + Geo::at(r, d));
        for (int w = 1; w < nw; ++w) o += *(const floatx4*)(s_o + w * Geo::WAVE + Geo::at(r, d));
        const size_t pidx = ((size_t)(un.t0 + i) * Hq + h * G + r % G) * nch_max + un.c;
        *(floatx4*)(po + pidx * HD + d) = o;
        if (d == 0) {
            const floatx4 m4 = *(const floatx4*)(s_m + 4 * r);
            float L = s_l[r];
            for (int w = 1; w < nw; ++w) L += s_l[w * R + r];
            pml[pidx * 2 + 0] = fmaxf(fmaxf(m4[0], m4[1]), fmaxf(m4[2], m4[3]));
            pml[pidx * 2 + 1] = L;
        }
    }
}

// Workgroup (h, y) takes units y, y + gridDim.y, ... of kv head h.  Consecutive
// workgroups run on consecutive XCDs, so with 8 kv heads an XCD stays on one
// head, whose K/V rows its L2 holds for the units that share them.
template <int HD, int G>
__global__ __launch_bounds__(256, HD == 128 ? 3 : 4) void attn_run_kernel(const float* q, const float* Kp, const float* Vp, int Hq,
                                                       int64_t head_stride, int nch_max, float* __restrict__ po,
                                                       float* __restrict__ pml, const int32_t* __restrict__ list) {
    __shared__ __attribute__((aligned(1024))) float s_o[4 * RunGeom<HD>::WAVE];
    __shared__ __attribute__((aligned(16))) float s_q[ARN_ROWS * HD];
    const int h = blockIdx.x, total = list[0];
    for (int u = blockIdx.y; u < total; u += gridDim.y) {
        const RunUnit un = arn_unpack(((const int4*)(list + 4))[u]);
        attn_run_unit<HD, G>(q, Kp, Vp, un, h, Hq, head_stride, nch_max, po, pml, s_o, s_q);
        __syncthreads();
    }
}

constexpr int ARN_GRID = 4096;

template <int HD>
static int launch_run_hd(int G, dim3 grid, hipStream_t s, const float* q, const float* Kp, const float* Vp, int Hq,
                         int64_t head_stride, int nch_max, float* po, float* pml, const int32_t* list) {
    switch (G) {
        case 1: hipLaunchKernelGGL((attn_run_kernel<HD, 1>), grid, dim3(256), 0, s, q, Kp, Vp, Hq, head_stride,
                                   nch_max, po, pml, list); return 0;
        case 2: hipLaunchKernelGGL((attn_run_kernel<HD, 2>), grid, dim3(256), 0, s, q, Kp, Vp, Hq, head_stride,
                                   nch_max, po, pml, list); return 0;
        case 4: hipLaunchKernelGGL((attn_run_kernel<HD, 4>), grid, dim3(256), 0, s, q, Kp, Vp, Hq, head_stride,
                                   nch_max, po, pml, list); return 0;
        case 8: hipLaunchKernelGGL((attn_run_kernel<HD, 8>), grid, dim3(256), 0, s, q, Kp, Vp, Hq, head_stride,
                                   nch_max, po, pml, list); return 0;
        default: return -5;
    }
}

// Partials of the units in `list` (at most one per token and chunk of n tokens).
int launch_attention_runs(const float* q, const float* Kp, const float* Vp, int n, int Hq, int Hkv, int HD,
                          int64_t head_stride, int nch_max, float* po, float* pml, const int32_t* list,
                          hipStream_t s) {
    const int G = Hq / Hkv;
    if (attn_chunk_size() != ARN_CHUNK) return -5;
    const dim3 grid(Hkv, (unsigned)std::min<int64_t>(std::max(1, ARN_GRID / Hkv), (int64_t)n * nch_max));
    const int rc = HD == 128 ? launch_run_hd<128>(G, grid, s, q, Kp, Vp, Hq, head_stride, nch_max, po, pml, list)
                   : HD == 64 ? launch_run_hd<64>(G, grid, s, q, Kp, Vp, Hq, head_stride, nch_max, po, pml, list)
                   : HD == 32 ? launch_run_hd<32>(G, grid, s, q, Kp, Vp, Hq, head_stride, nch_max, po, pml, list)
                              : -5;
    if (rc) return rc;
    SH_CHECK_LAUNCH();
    return 0;
}

}  // namespace slate_hip
