// attn_runs.h -- which kernel a token of a large ragged attention call goes
// to, and the unit list of the run kernel (k_attn.hip builds it, k_attn_run.hip
// reads it).
#pragma once
#include "common.h"

namespace slate_hip {

constexpr int ARN_CHUNK = 256;       // keys per unit: the merge kernel's chunk
constexpr int ARN_ROWS = 16;         // query rows per unit
constexpr int ARN_LIST = 1024;       // entries per pass of the list builder

__host__ __device__ constexpr int arn_tokens(int G) { return ARN_ROWS / G; }

// The tokens of the call: sequence and position of each, and the sequences'
// K/V bases.
struct RunTokens {
    const int32_t* seq;
    const int32_t* pos;
    const int64_t* kv_base;
    int n;
};

// Token i continues token i - 1: the next position of the same sequence.
__device__ __forceinline__ bool arn_follows(const RunTokens& tk, int i) {
    return i > 0 && i < tk.n && tk.seq[i] == tk.seq[i - 1] && tk.pos[i] == tk.pos[i - 1] + 1;
}

// Whether token i is left to the token kernel: the run kernel's 16-byte
// copies need rows that start on 16 bytes, and kv_base may be any offset.
__device__ __forceinline__ bool arn_single(const RunTokens& tk, int i) {
    return (tk.kv_base[tk.seq[i]] & 3) != 0;
}

// A unit: up to arn_tokens(G) tokens of a run, one chunk of keys.
struct RunUnit {
    int t0, n, p0, c;        // first token, tokens, first position, key chunk
    int64_t kvb;             // the sequence's K/V base
};
__device__ __forceinline__ int4 arn_pack(const RunUnit& u) {
    return make_int4(u.t0 * 65536 + u.c, u.p0, (int)(uint32_t)((uint64_t)u.kvb & 0xffffffffu),
                     (int)(((uint32_t)((uint64_t)u.kvb >> 32) & 0xffffffu) | ((uint32_t)u.n << 24)));
}
__device__ __forceinline__ RunUnit arn_unpack(const int4& d) {
    return RunUnit{d.x >> 16, (int)((uint32_t)d.w >> 24), d.y, d.x & 0xffff,
                   ((int64_t)(((uint64_t)(uint32_t)d.w << 32) | (uint32_t)d.z) << 8) >> 8};
}

// Exclusive scan over a workgroup of 256 threads (sum, or maximum).
template <bool MAX>
__device__ __forceinline__ int arn_scan(int v, int* s_w) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    int r = MAX ? INT32_MIN : 0;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int u = __shfl_up(v, o, 64);
        if (lane >= o) v = MAX ? max(v, u) : v + u;
    }
    const int u = __shfl_up(v, 1, 64);
    if (lane > 0) r = u;
    if (lane == 63) s_w[wv] = v;
    __syncthreads();
    for (int w = 0; w < wv; ++w) r = MAX ? max(r, s_w[w]) : r + s_w[w];
    __syncthreads();
    return r;
}

// The unit list, built by one workgroup of 256 threads: list[0] = count, then
// one int4 per unit from list + 4.  A run is a series of tokens that continue
// each other; entries ARN_LIST apart are never joined.  At most one unit per
// token and chunk.
__device__ __forceinline__ void arn_build(const RunTokens& tk, int nch_max, int tb, int32_t* __restrict__ list) {
    constexpr int E = ARN_LIST / 256;              // consecutive entries of a thread
    __shared__ int s_w[4], s_tot;
    __shared__ unsigned char s_start[ARN_LIST];
    int4* units = (int4*)(list + 4);
    const int e0 = threadIdx.x * E;
    int base = 0;
    for (int i0 = 0; i0 < tk.n; i0 += ARN_LIST) {
        int first = INT32_MIN;                     // the thread's last start
        bool start[E];
#pragma unroll
        for (int k = 0; k < E; ++k) {
            start[k] = e0 + k == 0 || !arn_follows(tk, i0 + e0 + k);
            s_start[e0 + k] = start[k];
            if (start[k]) first = e0 + k;
        }
        first = arn_scan<true>(first, s_w);        // (its barriers publish s_start too)
        RunUnit un[E];
        int nc[E], sum = 0;
#pragma unroll
        for (int k = 0; k < E; ++k) {
            const int e = e0 + k, i = i0 + e;
            if (start[k]) first = e;
            nc[k] = 0;
            if (i < tk.n && (e - first) % tb == 0 && !arn_single(tk, i)) {
                int n = 1;
                while (n < tb && e + n < ARN_LIST && !s_start[e + n]) ++n;
                un[k] = RunUnit{i, n, tk.pos[i], 0, tk.kv_base[tk.seq[i]]};
                nc[k] = max(0, min((un[k].p0 + n - 1 + ARN_CHUNK) / ARN_CHUNK, nch_max));
            }
            sum += nc[k];
        }
        int at = base + arn_scan<false>(sum, s_w);
        if (threadIdx.x == 255) s_tot = at + sum;
#pragma unroll
        for (int k = 0; k < E; ++k)
            for (int c = 0; c < nc[k]; ++c) {
                un[k].c = c;
                units[at++] = arn_pack(un[k]);
            }
        __syncthreads();
        base = s_tot;
        __syncthreads();
    }
    if (threadIdx.x == 0) list[0] = base;
}

}  // namespace slate_hip
