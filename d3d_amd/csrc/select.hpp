// Selection over one logits row by one workgroup of 1024 threads, shared by
// the row filter and the top-k / nucleus kernels: order-preserving keys,
// fixed-point masses, the general (any row) filter and the draw from a sorted
// support.
#pragma once

#include "d3d_common.hpp"
#include "rowstats.hpp"
#include "../../include/d3d_hip.h"

#include <limits.h>

namespace d3d {
namespace filt {

using rows::Scale;

constexpr int NTF = 1024;              // threads per row workgroup
constexpr int kWaves = NTF / kWave;    // 16
constexpr int kIdBits = 18;            // ids < 2^18 in a support key
constexpr int64_t kMaxV = 1 << kIdBits;
constexpr int kMassBits = 40;  // the cuts' masses are in units of 2^-40

// Largest k of the kernels that select from candidates in LDS (select.hip),
// and the candidates they hold.
constexpr int kSelectMaxK = 4096;
constexpr int kMaxSel = 8192;
// Rows per launch of those kernels (their per-row scratch is reused by the
// next batch, in stream order).
constexpr int kRowBatch = 256;

// Order-preserving key of a float: a < b (as floats) iff key(a) < key(b);
// -0 is read as +0 and NaN as the lowest key.
__device__ __forceinline__ uint32_t key_of(float z) {
    if (z != z) return 0u;
    if (z == 0.f) z = 0.f;
    const uint32_t u = __float_as_uint(z);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ __forceinline__ float float_of(uint32_t k) {
    const uint32_t u = (k & 0x80000000u) ? (k & 0x7fffffffu) : ~k;
    return __uint_as_float(u);
}

// The largest float below z > -inf (-0 is read as +0).
__device__ __forceinline__ float float_below(float z) {
    const uint32_t k = key_of(z) - 1;
    return float_of(k == 0x7fffffffu ? k - 1 : k);  // 0x7fffffff: the key -0 would have
}

template <int DT>
__device__ __forceinline__ float scaled(const void* row, int e, float T, bool unit) {
    const float x = rows::load_one<DT>(row, e);
    return unit ? x : x / T;
}

// Calls f(e, z) for every entry of the row; thread t visits e = t, t + NTF, ...
template <int DT, typename F>
__device__ __forceinline__ void for_row(const void* row, int V, float T, bool unit, F&& f) {
    for (int e = threadIdx.x; e < V; e += NTF) f(e, scaled<DT>(row, e, T, unit));
}

__device__ __forceinline__ uint64_t block_sum_u64(uint64_t v, uint64_t* s) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
    __syncthreads();
    if ((threadIdx.x & (kWave - 1)) == 0) s[threadIdx.x / kWave] = v;
    __syncthreads();
    uint64_t t = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) t += s[w];
    return t;
}

__device__ __forceinline__ float block_max_f(float v, float* s) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, kWave));
    __syncthreads();
    if ((threadIdx.x & (kWave - 1)) == 0) s[threadIdx.x / kWave] = v;
    __syncthreads();
    float t = s[0];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) t = fmaxf(t, s[w]);
    return t;
}

// exp(z - M) in units of 2^-BITS, rounded down.
template <int BITS = kMassBits>
__device__ __forceinline__ uint64_t weight_fx(float z, float M) {
    // NaN (and +inf against itself) carries no mass; -inf gives exp = 0.  No
    // branch, so that the chains of a thread's entries overlap.  The same
    // errors as with expf (4M points of each of seven ranges of [-87, 0]: at
    // most 0.85 units in the last place, 0.30 rms), without its range checks.
    const float d = z - M;
    const float e = exp_reduced(
        __builtin_amdgcn_fmed3f(d, -104.f, 0.f), [](float f) { return __builtin_amdgcn_exp2f(f); },
        [](float p, int n) { return __builtin_amdgcn_ldexpf(p, n); });
    const float f = d <= 0.f ? e * (float)(1ull << BITS) : 0.f;
    // Both halves of the 24-bit product are exact.
    const uint32_t hi = (uint32_t)(f * 0x1p-32f);
    const uint32_t lo = (uint32_t)__builtin_fmaf((float)hi, -0x1p32f, f);
    return ((uint64_t)hi << 32) | lo;
}

// weight_fx for a draw, at least one unit where expf(z - M) is not 0: every kept
// entry can be drawn.
template <int BITS>
__device__ __forceinline__ uint64_t draw_fx(float z, float M) {
    const float d = z - M;
    const uint64_t w = weight_fx<BITS>(z, M);
    return d <= 0.f && d > -103.f && w == 0 ? 1 : w;
}

// Id of the q-th entry (1-based, ascending id) with key == v, by a pass in
// id order (rounds of NTF consecutive entries, block-wide exclusive scans of
// the per-round counts).
template <int DT>
__device__ int nth_tie(const void* row, int V, float T, bool unit, uint32_t v, uint32_t q, uint32_t* s_u, int* s_i) {
    uint32_t before = 0;
    for (int base = 0; base < V; base += NTF) {
        const int e = base + threadIdx.x;
        const bool hit = e < V && key_of(scaled<DT>(row, e, T, unit)) == v;
        const uint64_t bal = __ballot(hit);
        const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
        __syncthreads();
        if (lane == 0) s_u[w] = (uint32_t)__popcll(bal);
        __syncthreads();
        uint32_t off = before;
        for (int k = 0; k < w; ++k) off += s_u[k];
        uint32_t total = before;
        for (int k = 0; k < kWaves; ++k) total += s_u[k];
        const uint32_t rank = off + (uint32_t)__popcll(bal & ((1ull << lane) - 1)) + 1;
        if (threadIdx.x == 0) *s_i = -1;
        __syncthreads();
        if (hit && rank == q) *s_i = e;
        __syncthreads();
        if (*s_i >= 0) return *s_i;
        before = total;
    }
    return V - 1;
}

// Scratch of the general filter.
struct FilterScratch {
    unsigned long long mass[256];
    uint64_t u64[kWaves];
    uint32_t cnt[256];
    uint32_t u[kWaves];
    float f[kWaves];
    uint32_t pick[2];
    int i;
};

// The filter (zf, lim) of one row by one workgroup, for rows of any length
// and any values; several passes over the row.  `exact`: the top-k filter
// keeps exactly top_k entries (ties by id).
template <int DT>
__device__ void filter_general(const void* row, int V, float T, bool unit, int top_k, float top_p, bool exact,
                               FilterScratch& sc, float& zf, int& lim) {
    // Top-k: the key K of the k-th largest entry, by digit-wise descent on
    // counts of the entries that share the digits chosen so far.
    uint32_t K = 0;      // keep key >= K (all ties) unless exact
    int lim_k = INT_MAX;
    const bool use_k = top_k > 0 && top_k < V;
    if (use_k) {
        uint32_t prefix = 0, mask = 0, need = (uint32_t)top_k;
        for (int shift = 24; shift >= 0; shift -= 8) {
            for (int b = threadIdx.x; b < 256; b += NTF) sc.cnt[b] = 0;
            __syncthreads();
            for_row<DT>(row, V, T, unit, [&](int, float z) {
                const uint32_t k = key_of(z);
                if ((k & mask) == prefix) atomicAdd(&sc.cnt[(k >> shift) & 255u], 1u);
            });
            __syncthreads();
            if (threadIdx.x == 0) {
                uint32_t acc = 0;
                int b = 255;
                for (; b > 0; --b) {
                    if (acc + sc.cnt[b] >= need) break;
                    acc += sc.cnt[b];
                }
                sc.pick[0] = (uint32_t)b;
                sc.pick[1] = need - acc;  // rank of the k-th entry within bin b
            }
            __syncthreads();
            prefix |= sc.pick[0] << shift;
            mask |= 255u << shift;
            need = sc.pick[1];
            __syncthreads();
        }
        K = prefix;
        // Exactly top_k entries: the `need` lowest ids among the ties at K.
        if (exact) lim_k = nth_tie<DT>(row, V, T, unit, K, need, sc.u, &sc.i);
    }
    zf = use_k ? float_of(K) : -INFINITY;
    lim = use_k ? lim_k : INT_MAX;

    if (top_p < 1.0f) {
        auto kept = [&](int e, float z) {
            const uint32_t k = key_of(z);
            return !use_k || k > K || (k == K && e <= lim_k);
        };
        // Row maximum and total mass over the entries the top-k filter keeps.
        float mx = -INFINITY;
        for_row<DT>(row, V, T, unit, [&](int e, float z) {
            if (kept(e, z) && z > mx) mx = z;
        });
        const float M = block_max_f(mx, sc.f);
        uint64_t tot = 0;
        for_row<DT>(row, V, T, unit, [&](int e, float z) {
            if (kept(e, z)) tot += weight_fx(z, M);
        });
        const uint64_t S = block_sum_u64(tot, sc.u64);
        const uint64_t target = (uint64_t)((double)top_p * (double)S);
        // The largest key v with mass(key >= v) > target: digit descent on
        // the mass of the entries that share the digits chosen so far; A is
        // the mass strictly above the current range.
        uint32_t prefix = 0, mask = 0;
        uint64_t A = 0;
        bool cut = true;
        for (int shift = 24; shift >= 0 && cut; shift -= 8) {
            for (int b = threadIdx.x; b < 256; b += NTF) sc.mass[b] = 0;
            __syncthreads();
            for_row<DT>(row, V, T, unit, [&](int e, float z) {
                const uint32_t k = key_of(z);
                if ((k & mask) == prefix && kept(e, z)) {
                    const uint64_t w = weight_fx(z, M);
                    if (w) atomicAdd(&sc.mass[(k >> shift) & 255u], (unsigned long long)w);
                }
            });
            __syncthreads();
            if (threadIdx.x == 0) {
                uint64_t acc = 0;
                int b = 255;
                for (; b >= 0; --b) {
                    if (A + acc + sc.mass[b] > target) break;
                    acc += sc.mass[b];
                }
                sc.pick[0] = b < 0 ? 0xffffffffu : (uint32_t)b;
                sc.u64[0] = A + acc;
            }
            __syncthreads();
            if (sc.pick[0] == 0xffffffffu) {
                cut = false;  // rounding left the whole mass at or below target
            } else {
                prefix |= sc.pick[0] << shift;
                mask |= 255u << shift;
                A = sc.u64[0];
            }
            __syncthreads();
        }
        if (cut) {
            // Entries with key == prefix all weigh w; the cut keeps the first
            // q of them (ascending id): A + q w > target >= A + (q - 1) w.
            const float zc = float_of(prefix);
            const uint64_t w = weight_fx(zc, M);
            const uint64_t q = w ? (target - A) / w + 1 : 1;
            zf = zc;
            // Every entry with key == prefix >= K passes the top-k filter
            // (ties with the k-th value are kept), so the count runs over all.
            lim = nth_tie<DT>(row, V, T, unit, prefix, (uint32_t)q, sc.u, &sc.i);
        }
    }
}

__device__ __forceinline__ float key_value(uint64_t k) {
    return float_of(~(uint32_t)(k >> kIdBits));
}

// Inclusive scan over the workgroup in thread order.
__device__ __forceinline__ float block_incl(float v, float* s, float* tot) {
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const float t = __shfl_up(v, o, kWave);
        if (lane >= o) v += t;
    }
    __syncthreads();
    if (lane == kWave - 1) s[w] = v;
    __syncthreads();
    float off = 0.f, t = 0.f;
#pragma unroll
    for (int k = 0; k < kWaves; ++k) {
        if (k < w) off += s[k];
        t += s[k];
    }
    *tot = t;
    return v + off;
}

// Sum over the workgroup in double: the normalisers of a support, so that their
// rounding adds nothing to the probabilities' own.
__device__ __forceinline__ double block_sum_f64(double v, double* s) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
    __syncthreads();
    if ((threadIdx.x & (kWave - 1)) == 0) s[threadIdx.x / kWave] = v;
    __syncthreads();
    double t = 0.;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) t += s[w];
    return t;
}

// One workgroup per row over its sorted support keys [S]: ids, softmax over
// the support (max = the first value), the nucleus filter in support order,
// the draw.  A slot the gather left unwritten (only a NaN logit can leave
// the filter short of S entries) holds ~0: weight 0, id -1.
__device__ void support_draw(const uint64_t* k, int S, float top_p, float u, int64_t* tok, int64_t* ids,
                             float* probs, float* tok_prob, float* s_w, int* s_i) {
    const float M = key_value(k[0]);
    auto weight = [&](int s) {
        const uint64_t kk = k[s];
        const float z = key_value(kk);
        return (kk != ~0ull && z > -INFINITY) ? expf(z - M) : 0.f;
    };
    // Z = sum of the weights, in a fixed order.
    __shared__ double s_d[kWaves];
    double sum = 0.;
    for (int s = threadIdx.x; s < S; s += NTF) sum += (double)weight(s);
    const float Z = (float)block_sum_f64(sum, s_d);
    // Nucleus filter: entry s > 0 goes when the inclusive probability of
    // entries 0..s-1 exceeds top_p; `keep` is the kept prefix length.
    int keep = S;
    if (top_p < 1.0f && Z > 0.f) {
        float carry = 0.f;
        if (threadIdx.x == 0) s_i[0] = S;
        __syncthreads();
        for (int base = 0; base < S; base += NTF) {
            const int s = base + threadIdx.x;
            const float p = s < S ? weight(s) / Z : 0.f;
            float t;
            const float incl = carry + block_incl(p, s_w, &t);
            if (s < S && s > 0 && incl - p > top_p) atomicMin(&s_i[0], s);
            __syncthreads();
            carry += t;
            if (s_i[0] < S) break;
        }
        keep = s_i[0];
        __syncthreads();
    }
    float Zk = Z;
    if (keep < S) {
        sum = 0.;
        for (int s = threadIdx.x; s < keep; s += NTF) sum += (double)weight(s);
        Zk = (float)block_sum_f64(sum, s_d);
    }
    auto prob = [&](int s) { return (s < keep && Zk > 0.f) ? weight(s) / Zk : 0.f; };
    float tot_p = 0.f, part = 0.f;
    for (int s = threadIdx.x; s < S; s += NTF) {
        const float p = prob(s);
        ids[s] = k[s] == ~0ull ? -1 : (int64_t)(k[s] & ((1ull << kIdBits) - 1));
        probs[s] = p;
        part += p;
    }
    block_incl(part, s_w, &tot_p);
    // Draw in support order over the same probabilities.
    const float target = u * tot_p;
    float carry = 0.f;
    if (threadIdx.x == 0) {
        s_i[0] = INT_MAX;
        s_i[1] = -1;
    }
    __syncthreads();
    for (int base = 0; base < S; base += NTF) {
        const int s = base + threadIdx.x;
        const float p = s < S ? prob(s) : 0.f;
        float t;
        const float incl = carry + block_incl(p, s_w, &t);
        if (s < S && p > 0.f) {
            atomicMax(&s_i[1], s);
            if (incl > target) atomicMin(&s_i[0], s);
        }
        __syncthreads();
        carry += t;
        if (s_i[0] != INT_MAX) break;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const int pick = s_i[0] != INT_MAX ? s_i[0] : s_i[1];
        *tok = pick >= 0 ? (int64_t)(k[pick] & ((1ull << kIdBits) - 1)) : (int64_t)D3D_TOKEN_EMPTY_DISTRIBUTION;
        if (tok_prob) *tok_prob = pick >= 0 ? prob(pick) : 0.f;
    }
}


// ---- host side (select.hip) ----

// Bytes of per-row scratch for N rows of at most `chunks` 4096-entry chunks.
size_t select_scratch_bytes(int N, int chunks, bool lse);

// The S largest z = x / T of each row (S <= kSelectMaxK, V <= kMaxV), sorted,
// then softmax, nucleus filter and draw over them, as d3d_sample_support_wide.
hipError_t select_support(const void* logits, int dtype, int N, int V, float T, int S, float top_p, const float* u,
                          int64_t* tok, int64_t* ids, float* probs, float* tok_prob, void* scratch, hipStream_t s);

// The k largest entries of each row, as d3d_topk_rows.
hipError_t select_topk(const void* logits, int dtype, int N, int V, int k, bool lse, int64_t* ids, float* vals,
                       void* scratch, hipStream_t s);

}  // namespace filt
}  // namespace d3d
