// attn_runs.h -- which kernel a token of a large ragged attention call goes
// to, and the unit list of the run kernel (k_attn.hip builds it, k_attn_run.hip
// reads it).
#pragma once
#include "lanes.h"

namespace slate_hip {

constexpr int ARN_CHUNK = 256;       // keys per unit: the merge kernel's chunk
constexpr int ARN_ROWS = 16;         // query rows per unit
constexpr int ARN_PASS = 1024;       // tokens that go to one kernel or the other together

__host__ __device__ constexpr int arn_tokens(int G) { return ARN_ROWS / G; }

// The tokens of the call: sequence and position of each, and the sequences'
// K/V bases.
struct RunTokens {
    const int32_t* seq;
    const int32_t* pos;
    const int64_t* kv_base;
    int n;
};

// Keys that a pass's tokens read token by token (each, times the tokens of a
// unit) and in units (runs, a run's first token counted as a unit of its
// own).  Whole numbers: every workgroup that adds them up agrees.
struct RunCost {
    int each = 0, runs = 0;
    bool off = false;        // rows that start off 16 bytes: kv_base may be any offset
    __device__ __forceinline__ void add(int pos, bool follows, int64_t kvb, int tb) {
        const int keys = min(max(pos, -1) + 1, 65536);
        each += keys * tb;
        runs += follows ? keys : keys * tb;
        off |= (kvb & 3) != 0;
    }
    // This thread's wave's part into s_c.
    __device__ __forceinline__ void put(int (*s_c)[3]) const {
        const int e = wave_sum_int(each), r = wave_sum_int(runs);
        const bool any = __any(off);
        if ((threadIdx.x & 63) == 0) {
            s_c[threadIdx.x >> 6][0] = e;
            s_c[threadIdx.x >> 6][1] = r;
            s_c[threadIdx.x >> 6][2] = any;
        }
    }
};

// Whether the run kernel takes a pass of n tokens (after a barrier).  Its
// copies need rows that start on 16 bytes.  A unit of one token costs more
// than the token kernel's, so sharing has to save a third of the keys: at 1.2
// times the keys (40 decode tokens at ~500 keys, a chunk of 60, heads of 64)
// 19.0 us in units and 18.0 without, at 2 (pairs of tokens at ~300 keys) 16.3
// and 18.1.  Only with heads of 128 and more than a chunk of keys a token the
// two are level (128 lone tokens at ~300 keys 67.4 and 68.8 us, at ~60 28.0
// and 21.2).
__device__ __forceinline__ bool arn_shared(const int (*s_c)[3], int n, int tb, int HD) {
    int64_t each = 0, runs = 0;
    int off = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        each += s_c[w][0];
        runs += s_c[w][1];
        off |= s_c[w][2];
    }
    return !off && (2 * each >= 3 * runs || (HD == 128 && each >= (int64_t)ARN_CHUNK * tb * n));
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

// Exclusive scan over a workgroup of 256 threads (sum, or maximum), one
// barrier; s_w keeps the waves' totals.
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
    return r;
}

// The unit list, built by one workgroup of 256 threads: list[0] = count, then
// one int4 per unit from list + 4.  A run is a series of tokens at positions
// one apart in one sequence; it ends at the end of its pass.  At most one
// unit per token and chunk.
__device__ __forceinline__ void arn_build(const RunTokens& tk, int nch_max, int tb, int HD,
                                          int32_t* __restrict__ list) {
    constexpr int E = ARN_PASS / 256;              // consecutive tokens of a thread
    __shared__ int s_m[4], s_w[4], s_c[4][3];
    __shared__ unsigned char s_start[ARN_PASS];
    int4* units = (int4*)(list + 4);
    const int e0 = threadIdx.x * E;
    int base = 0;
    for (int i0 = 0; i0 < tk.n; i0 += ARN_PASS) {
        // the tokens and the one before them, in one round of loads
        int p[E + 1], q[E + 1];
        int64_t kvb[E];
#pragma unroll
        for (int k = 0; k <= E; ++k) {
            const int i = min(max(i0 + e0 + k - 1, 0), tk.n - 1);
            p[k] = tk.pos[i];
            q[k] = tk.seq[i];
        }
#pragma unroll
        for (int k = 0; k < E; ++k) kvb[k] = tk.kv_base[q[k + 1]];
        int first = INT32_MIN;                     // the thread's last start
        bool start[E];
        RunCost cost;
#pragma unroll
        for (int k = 0; k < E; ++k) {
            const int i = i0 + e0 + k;
            const bool follows = i > 0 && i < tk.n && q[k + 1] == q[k] && p[k + 1] == p[k] + 1;
            if (i < tk.n) cost.add(p[k + 1], follows, kvb[k], tb);
            start[k] = !follows || e0 + k == 0;
            s_start[e0 + k] = start[k];
            if (start[k]) first = e0 + k;
        }
        cost.put(s_c);
        first = arn_scan<true>(first, s_m);        // (its barrier publishes s_start and s_c too)
        const bool shared = arn_shared(s_c, min(tk.n - i0, ARN_PASS), tb, HD);
        int n[E], nc[E], sum = 0;
#pragma unroll
        for (int k = 0; k < E; ++k) {
            const int e = e0 + k;
            if (start[k]) first = e;
            n[k] = 1;
            nc[k] = 0;
            if (shared && i0 + e < tk.n && (e - first) % tb == 0) {
                while (n[k] < tb && e + n[k] < ARN_PASS && !s_start[e + n[k]]) ++n[k];
                nc[k] = max(0, min((p[k + 1] + n[k] - 1 + ARN_CHUNK) / ARN_CHUNK, nch_max));
            }
            sum += nc[k];
        }
        int at = base + arn_scan<false>(sum, s_w);
#pragma unroll
        for (int k = 0; k < E; ++k)
            for (int c = 0; c < nc[k]; ++c)
                units[at++] = arn_pack(RunUnit{i0 + e0 + k, n[k], p[k + 1], c, kvb[k]});
        base += (s_w[0] + s_w[1]) + (s_w[2] + s_w[3]);
        __syncthreads();
    }
    if (threadIdx.x == 0) list[0] = base;
}

// The (token, chunk) pairs of a pass that the run kernel does not take, as
// each workgroup of 256 threads numbers them for itself: thread t's tokens
// are t, t + 256, ... of the pass.
struct TokenPass {
    int s_w[4], s_c[4][3];
    int at[256];             // pairs before thread t's
    int nc[ARN_PASS];        // chunks of a token

    // Their count; 0 where the run kernel takes the pass.
    __device__ __forceinline__ int number(const RunTokens& tk, int i0, int nch_max, int tb, int HD) {
        constexpr int E = ARN_PASS / 256;
        const int tid = threadIdx.x;
        int p[E], q[E], p1[E], q1[E];
#pragma unroll
        for (int k = 0; k < E; ++k) {
            const int i = min(i0 + tid + 256 * k, tk.n - 1), j = max(i - 1, 0);
            p[k] = tk.pos[i];
            q[k] = tk.seq[i];
            p1[k] = tk.pos[j];
            q1[k] = tk.seq[j];
        }
        RunCost cost;
        int sum = 0;
#pragma unroll
        for (int k = 0; k < E; ++k) {
            const int i = i0 + tid + 256 * k;
            int n = 0;
            if (i < tk.n) {
                cost.add(p[k], i > 0 && q[k] == q1[k] && p[k] == p1[k] + 1, tk.kv_base[q[k]], tb);
                n = max(0, min((p[k] + ARN_CHUNK) / ARN_CHUNK, nch_max));
            }
            nc[tid + 256 * k] = n;
            sum += n;
        }
        cost.put(s_c);
        __syncthreads();
        if (arn_shared(s_c, min(tk.n - i0, ARN_PASS), tb, HD)) return 0;
        at[tid] = arn_scan<false>(sum, s_w);
        __syncthreads();
        return (s_w[0] + s_w[1]) + (s_w[2] + s_w[3]);
    }
    // Pair r: token (of the pass) and chunk.
    __device__ __forceinline__ void pair(int r, int& token, int& chunk) const {
        int t = 0;
#pragma unroll
        for (int o = 128; o > 0; o >>= 1)
            if (at[t + o] <= r) t += o;
        r -= at[t];
        while (r >= nc[t]) {
            r -= nc[t];
            t += 256;
        }
        token = __builtin_amdgcn_readfirstlane(t);
        chunk = __builtin_amdgcn_readfirstlane(r);
    }
};

}  // namespace slate_hip
