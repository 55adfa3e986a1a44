// Top-k and nucleus selection over rows of V <= 2^18 logits.
//
// Reference behaviour (D3D repository):
//   single/eval_sync.py:292-303  the top-k and top-p filters of _sampling_probs
//   single/eval_sync.py:308-338  a draw from the filtered softmax
//   single/eval_sync.py:341-367  _sample_with_sparse_probs (sorted top-S support)
//   serving/backend.py:84-93     logits.topk(k).indices
//
// Top-k (any caller with k <= kSelectMaxK): one pass over the logits leaves
// the maximum of every 16-entry group (a thread's share of a 4096-entry
// chunk).  The k-th largest group maximum is a lower bound t of the row's
// k-th largest entry, because k different groups hold an entry >= t.  One
// workgroup per row finds such a t among the 9,728 maxima of a
// 151,936-entry row by a bit-wise search on counts (it stops early once few
// more than k groups pass), re-reads only the passing groups, and sorts their
// entries >= t in LDS.  No assumption on the values is needed: where a long run
// of equal values at the k-th largest entry does not fit, the entries above it
// and the run's first ids do (masked rows); only a run that carries mass under
// a filter, or k of several thousand spread over few groups, is left to the
// general multi-pass selection.
//
// Nucleus over the whole vocabulary (top_p < 1, no top-k): (1) row maxima M;
// (2) a histogram per part of the row of the masses w = exp(z - M) over bins
// of M - z, 1/32 wide; entries beyond 28 weigh less than one fixed-point
// unit (2^-40); (3) the entries of the bin where the running mass crosses
// top_p * S are gathered;
// (4) one workgroup per row narrows them down the same way and places the cut.
// All masses are 64-bit integers, so the cut does not depend on the order of
// the sums and equals the general filter's.  A draw uses integers too (the same
// ones, or of a finer unit where few entries are kept): the parts' masses, then
// one part's entries in id order.
//
// Measured, 64 bf16 rows of 151,936 (19.4 MB, 3 us at the rate of a plain read): sorted
// top-64 with its draw 236 -> 21.6 us (k rounds of argmaxes over every chunk
// and over the chunk winners before), nucleus draw 541 -> 55 us (one
// workgroup per row and about ten passes before).  Launches: maxima 5.7 us,
// selection 12-16 us (one workgroup's chain of dependent steps: search,
// gather, sort, draw); nucleus 5.7 + 16 + 16 + 21 us.
#include "select.hpp"
#include "../../include/d3d_hip.h"

#include <algorithm>

namespace d3d {
namespace filt {
namespace {

using rows::kChunk;
using rows::NT;
constexpr int kGroup = kChunk / NT;      // entries per group
constexpr int kMaxChunks = (int)(kMaxV / kChunk);
constexpr int kRegKeys = kMaxChunks * NT / NTF;  // group maxima per thread: 16
constexpr int kMaxGroups = 6144;         // passing groups listed in LDS
constexpr int kFine = 16, kCoarse = 56, kBins = kFine * kCoarse;  // 1/32-wide bins of M - z < 28
constexpr float kBinScale = 32.f;

enum SelMode : int { kSupport = 0, kTopk = 1, kFilter = 2 };

// What the nucleus passes hand on, per row.
struct NucRec {
    uint64_t above;   // mass of the bins before the crossing one
    uint64_t target;  // top_p * S
    float M;
    int bin;          // crossing bin, -1: none (every entry is kept)
};

struct SelParams {
    const void* logits;  // [N, V]
    int V, C;
    float T;
    int k;         // top-k / support size; 0: none (nucleus)
    float top_p;   // >= 1: off
    const float* u;
    // outputs (by mode)
    int64_t* tok;
    int64_t* ids;
    float* probs;      // support probabilities, or top-k values
    float* tok_prob;
    float* zf;
    int32_t* lim;
    // scratch
    float* gmax;           // [N][C][NT]
    float2* lse;           // [N][C], top-k with log-probabilities
    float* cmax;           // [N][C]
    uint64_t* hist;        // [N][parts][kBins]
    uint64_t* coarse;      // [N][parts][64]
    uint64_t* list;        // [N][kMaxSel]
    uint32_t* counter;     // [N]
    NucRec* rec;           // [N]
    int parts, span;       // parts per row, chunks per part
};

// ---------------------------------------------------------------- pass 1

// Workgroup (chunk, row): group maxima (GROUPS) or the chunk maximum alone,
// and for log-probabilities the chunk's (max, sum exp(x - max)).  NaN is
// ignored.  HBM-bound: the logits are read once.
template <int DT, bool VEC, bool GROUPS, bool LSE>
__global__ __launch_bounds__(NT) void max_kernel(SelParams P) {
    constexpr int E = rows::Vec<DT>::E;
    __shared__ float sv[NT / kWave];
    const int c = blockIdx.x, n = blockIdx.y;
    const int first = c * kChunk + (int)threadIdx.x * E;
    float x[kGroup];
    rows::load_tile<DT, VEC, false, kGroup>(rows::row_ptr<DT>(P.logits, n, P.V), P.V, first, NT * E, -INFINITY, x);
    float m = -INFINITY;
#pragma unroll
    for (int l = 0; l < kGroup; ++l) m = fmaxf(m, x[l]);
    if constexpr (GROUPS) P.gmax[((size_t)n * P.C + c) * NT + threadIdx.x] = m;
    if constexpr (LSE || !GROUPS) {
        const float wv = block_max<NT>(m, sv);
        if constexpr (LSE) {
            float se = 0.f;
            if (wv != -INFINITY) {
#pragma unroll
                for (int l = 0; l < kGroup; ++l)
                    if (rows::tile_index<DT>(first, NT * E, l) < P.V) se += expf(x[l] - wv);
            }
            se = block_sum<NT>(se, sv);
            if (threadIdx.x == 0) P.lse[(size_t)n * P.C + c] = make_float2(wv, se);
        } else if (threadIdx.x == 0) {
            P.cmax[(size_t)n * P.C + c] = P.T == 1.0f ? wv : wv / P.T;
            if (c == 0) P.counter[n] = 0;
        }
    }
}

// ---------------------------------------------------------------- row workgroup

union SelScratch {
    FilterScratch general;
    struct {
        uint32_t cnt[2][kWaves];
        uint32_t n_groups, n_cand;
        float f[kWaves];
        int i[2];
        uint64_t w64[kWaves];
        uint64_t mass[kMaxChunks];
        uint64_t base;
        float fx;
        uint32_t rank[512];  // kRankSort
    } s;
};

// Ascending sort of a[0, m), m <= kRankSort, into its first m slots: every
// key's rank is counted by kWaves threads (the keys are distinct).  At 100
// keys 28 bitonic steps took 7.7 us, this 1 us; past about 500 the m^2
// compares outgrow the steps.
constexpr int kRankSort = 512;
__device__ void rank_sort(uint64_t* a, int m, uint32_t* rank) {
    for (int i = threadIdx.x; i < m; i += NTF) rank[i] = 0;
    __syncthreads();
    // Wave w counts against its share of the keys, a lane per key.
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    const int per = (m + kWaves - 1) / kWaves, b0 = w * per, b1 = min(b0 + per, m);
    for (int i = lane; i < m; i += kWave) {
        const uint64_t mine = a[i];
        uint32_t c = 0;
#pragma unroll 4
        for (int b = b0; b < b1; ++b) c += a[b] < mine ? 1u : 0u;
        if (c) atomicAdd(&rank[i], c);
    }
    __syncthreads();
    uint64_t v = 0;
    const bool have = (int)threadIdx.x < m;  // m <= NTF
    if (have) v = a[threadIdx.x];
    __syncthreads();
    if (have) a[rank[threadIdx.x]] = v;
    __syncthreads();
}

// Ascending bitonic sort of a[0, P2), P2 a power of two.  Steps of distance
// <= 64 stay within the 128 entries one wave owns, so only the longer ones
// need the workgroup's barrier.
__device__ void sort_lds(uint64_t* a, int P2) {
    const int half = P2 / 2;
    for (int k = 2; k <= P2; k <<= 1) {
        for (int j = k >> 1, lj = __builtin_ctz(k) - 1; j > 0; j >>= 1, --lj) {
            if (j >= kWave * 2 || (j == kWave && k > 2 * kWave)) __syncthreads();
            else __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            for (int i = threadIdx.x; i < half; i += NTF) {
                const int lo = ((i >> lj) << (lj + 1)) + (i & (j - 1)), hi = lo + j;
                const uint64_t x = a[lo], y = a[hi];
                const bool up = (lo & k) == 0;
                if ((x > y) == up) {
                    a[lo] = y;
                    a[hi] = x;
                }
            }
        }
    }
    __syncthreads();
}

// Pads list[m, p2) with ~0, p2 the power of two that holds m entries and at
// least `want`, and sorts it; the caller has synchronised.
__device__ __forceinline__ void pad_and_sort(uint64_t* list, int m, int want, uint32_t* rank) {
    if (max(m, want) <= kRankSort) {
        for (int i = m + threadIdx.x; i < want; i += NTF) list[i] = ~0ull;
        rank_sort(list, m, rank);
        return;
    }
    int p2 = 2;
    while (p2 < max(m, want)) p2 <<= 1;
    for (int i = m + threadIdx.x; i < p2; i += NTF) list[i] = ~0ull;
    __syncthreads();
    sort_lds(list, p2);
}

__device__ __forceinline__ uint64_t support_key(float z, int e) {
    return ((uint64_t)(~key_of(z)) << kIdBits) | (uint64_t)e;
}

// Notes group i as passing (any order).
__device__ __forceinline__ void list_group(int i, bool hit, uint16_t* groups, SelScratch& sc) {
    const int lane = threadIdx.x & (kWave - 1);
    const uint64_t bal = __ballot(hit);
    if (bal) {
        uint32_t base = 0;
        if (lane == 0) base = atomicAdd(&sc.s.n_groups, (uint32_t)__popcll(bal));
        base = (uint32_t)__shfl((int)base, 0, kWave) + (uint32_t)__popcll(bal & ((1ull << lane) - 1));
        if (hit && base < (uint32_t)kMaxGroups) groups[base] = (uint16_t)i;
    }
}

// The passing groups' entries with z > lo (none has x < x_lo) into list;
// returns their number, or -1 when they or the groups do not fit.
template <int DT, bool VEC>
__device__ __forceinline__ int gather_groups(const SelParams& P, const void* row, float x_lo, float lo, bool unit,
                                             uint64_t* list, const uint16_t* groups, SelScratch& sc) {
    constexpr int E = rows::Vec<DT>::E;
    __syncthreads();
    const int ng = (int)sc.s.n_groups;
    if (ng > kMaxGroups) return -1;
    constexpr int PP = kGroup / E;  // 16-byte pieces of a group
    for (int p = threadIdx.x; p < ng * PP; p += NTF) {
        const int gi = groups[p / PP];
        const int e0 = (gi / NT) * kChunk + (gi % NT) * E + (p % PP) * NT * E;
        float x[E];
        rows::load_tile<DT, VEC, false, E>(row, P.V, e0, 0, -INFINITY, x);
#pragma unroll
        for (int q = 0; q < E; ++q) {
            if (e0 + q < P.V && !(x[q] < x_lo)) {
                const float z = unit ? x[q] : x[q] / P.T;
                if (z > lo) {
                    const uint32_t slot = atomicAdd(&sc.s.n_cand, 1u);
                    if (slot < (uint32_t)kMaxSel) list[slot] = support_key(z, e0 + q);
                }
            }
        }
    }
    __syncthreads();
    const int m = (int)sc.s.n_cand;
    return m <= kMaxSel ? m : -1;
}

// The row's entries z >= z_t into list (any order), z_t at most its k-th
// largest z; returns their number, or -1 when they do not fit.  When they do
// not, or z_t = -inf, only the entries above z_t: fewer than k of those leave
// the others of the k largest to append_ties(z_t).  That is a row with a long
// run of equal values at its k-th largest, above all a masked one (-inf or a
// dtype's lowest value): in the general selection's passes every count of such
// a run hits one bin.  64 bf16 rows of 151,936, 20 entries not masked, us,
// general / this: top-64 592 / 17, support of 64 600 / 24, top-50 draw 697 / 22.
template <int DT, bool VEC>
__device__ int collect(const SelParams& P, const void* row, const float* gmax, int k, bool unit, uint64_t* list,
                       uint16_t* groups, SelScratch& sc, float& z_t) {
    const int G = P.C * NT, lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    float g[kRegKeys];
    uint32_t key[kRegKeys];
#pragma unroll
    for (int j = 0; j < kRegKeys; ++j) {
        const int i = j * NTF + (int)threadIdx.x;
        g[j] = gmax[min(i, G - 1)];
        if (i >= G) g[j] = -INFINITY;
    }
#pragma unroll
    for (int j = 0; j < kRegKeys; ++j) key[j] = j * NTF + (int)threadIdx.x < G ? key_of(g[j]) : 0u;
    const int J = (G + NTF - 1) / NTF;
    if (threadIdx.x == 0) {
        sc.s.n_groups = 0;
        sc.s.n_cand = 0;
    }
    // The search runs on maxima over several groups while those still number
    // at least four times k (any k disjoint sets with an entry >= t each will
    // do): one key per thread at k <= 256, four at k <= 1024.
    uint32_t sk[4] = {0u, 0u, 0u, 0u};
    uint32_t* s_key = reinterpret_cast<uint32_t*>(list);  // free until the entries are collected
    const int fold = k * 4 <= NTF && J > 1 ? 1 : (k <= NTF && J > 4 ? 4 : 0);
    if (fold) {
#pragma unroll
        for (int j = 0; j < kRegKeys; ++j) sk[j % 4] = max(sk[j % 4], key[j]);
        if (fold == 1) {
            sk[0] = max(max(sk[0], sk[1]), max(sk[2], sk[3]));
            sk[1] = sk[2] = sk[3] = 0u;
        }
    }
    // The largest prefix t with at least k maxima >= t, bit by bit from the
    // top, until few more than k pass.  bf16 maxima differ in their upper 16
    // bits only.
    uint32_t t = 0;
    const uint32_t enough = (uint32_t)(k + k / 8 + 32);
    if (fold == 1) {
        // One wave does the search, 16 maxima per lane, without barriers.
        s_key[threadIdx.x] = sk[0];
        __syncthreads();
        if (w == 0) {
            uint32_t q[kWaves];
            uint32_t mx = 0;
#pragma unroll
            for (int j = 0; j < kWaves; ++j) {
                q[j] = s_key[j * kWave + lane];
                mx = max(mx, q[j]);
            }
            mx = max(mx, xor_partner_desc<32>(mx));
            mx = max(mx, xor_partner_desc<16>(mx));
            mx = max(mx, xor_partner_desc<8>(mx));
            mx = max(mx, xor_partner_desc<4>(mx));
            mx = max(mx, xor_partner_desc<2>(mx));
            mx = max(mx, xor_partner_desc<1>(mx));
            mx = (uint32_t)__builtin_amdgcn_readfirstlane((int)mx);
            auto count = [&](uint32_t cand) {
                uint32_t c = 0;
#pragma unroll
                for (int j = 0; j < kWaves; ++j) c += (uint32_t)__popcll(__ballot(q[j] >= cand));
                return c;
            };
            // The sign and the exponent's upper bits are mostly the maximum's.
            int bit = 31;
            if (count(mx & 0xfe000000u) >= (uint32_t)k) {
                t = mx & 0xfe000000u;
                bit = 24;
            }
            for (; bit >= (DT == kBF16 ? 16 : 0); --bit) {
                const uint32_t cand = t | (1u << bit);
                const uint32_t c = count(cand);
                if (c >= (uint32_t)k) {
                    t = cand;
                    if (c <= enough) break;
                }
            }
            if (lane == 0) sc.s.cnt[0][0] = t;
        }
        __syncthreads();
        t = sc.s.cnt[0][0];
    } else if (G >= k) {
        for (int bit = 31; bit >= (DT == kBF16 ? 16 : 0); --bit) {
            const uint32_t cand = t | (1u << bit);
            uint32_t cw = 0;
            if (fold == 4) {
#pragma unroll
                for (int j = 0; j < 4; ++j) cw += (uint32_t)__popcll(__ballot(sk[j] >= cand));
            } else {
#pragma unroll
                for (int j = 0; j < kRegKeys; ++j)
                    if (j < J) cw += (uint32_t)__popcll(__ballot(key[j] >= cand));
            }
            uint32_t* slot = sc.s.cnt[bit & 1];
            if (lane == 0) slot[w] = cw;
            __syncthreads();
            uint32_t c = 0;
#pragma unroll
            for (int q = 0; q < kWaves; ++q) c += slot[q];
            if (c >= (uint32_t)k) {
                t = cand;
                if (c <= enough) break;
            }
        }
    }
    __syncthreads();
    // A negative bf16 maximum's key ends in ones.
    if (DT == kBF16 && t < 0x80000000u) t |= 0xffffu;
    const float x_t = t > 0x007fffffu ? float_of(t) : -INFINITY;  // 0x007fffff: the key of -inf
    z_t = unit ? x_t : x_t / P.T;
    // Nothing below x_lo scales to z_t: numerators of equal quotients lie within
    // T times the quotient's ulp, a few ulp of x_t, or T 2^-149 where the
    // quotient is denormal.
    const float x_lo = x_t - fmaxf(fabsf(x_t) * 0x1p-20f, P.T * 0x1p-147f);
    // Entries above lo are taken.
    const float lo = z_t == -INFINITY ? z_t : float_below(z_t);
#pragma unroll
    for (int j = 0; j < kRegKeys; ++j) {
        if (j >= J) break;
        const int i = j * NTF + (int)threadIdx.x;
        list_group(i, i < G && !(g[j] < x_lo) && (unit ? g[j] : g[j] / P.T) > lo, groups, sc);
    }
    int m = gather_groups<DT, VEC>(P, row, x_lo, lo, unit, list, groups, sc);
    if (m >= 0 || lo == z_t) return m;
    __syncthreads();
    if (threadIdx.x == 0) {
        sc.s.n_groups = 0;
        sc.s.n_cand = 0;
    }
    __syncthreads();
    for (int j = 0; j < J; ++j) {
        const int i = j * NTF + (int)threadIdx.x;
        const float x = gmax[min(i, G - 1)];
        list_group(i, i < G && !(x < x_lo) && (unit ? x : x / P.T) > z_t, groups, sc);
    }
    return gather_groups<DT, VEC>(P, row, x_lo, z_t, unit, list, groups, sc);
}

// Appends the row's first entries (by id) with z == v to the m entries of list
// until it holds k, and returns the count; a masked row has enough of them in
// its first thousand.
template <int DT>
__device__ int append_ties(const SelParams& P, const void* row, float v, int m, int k, bool unit, uint64_t* list,
                           SelScratch& sc) {
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    for (int base = 0, par = 0; base < P.V && m < k; base += NTF, par ^= 1) {
        const int e = base + (int)threadIdx.x;
        const bool hit = e < P.V && scaled<DT>(row, e, P.T, unit) == v;
        const uint64_t bal = __ballot(hit);
        uint32_t* slot = sc.s.cnt[par];
        if (lane == 0) slot[w] = (uint32_t)__popcll(bal);
        __syncthreads();
        int at = m + __popcll(bal & ((1ull << lane) - 1)), total = 0;
#pragma unroll
        for (int q = 0; q < kWaves; ++q) {
            at += q < w ? (int)slot[q] : 0;
            total += (int)slot[q];
        }
        if (hit && at < k) list[at] = support_key(v, e);
        m = min(m + total, k);
    }
    __syncthreads();
    return m;
}

// Exactly the k largest entries (ties by id) of a row collect() could not
// hold, by the general selection; k <= kSelectMaxK.
template <int DT>
__device__ int collect_general(const SelParams& P, const void* row, int k, bool unit, uint64_t* list,
                               SelScratch& sc) {
    float zf;
    int lim;
    filter_general<DT>(row, P.V, P.T, unit, k < P.V ? k : 0, 1.0f, true, sc.general, zf, lim);
    const uint32_t kf = key_of(zf);
    __syncthreads();
    if (threadIdx.x == 0) sc.s.n_cand = 0;
    __syncthreads();
    for_row<DT>(row, P.V, P.T, unit, [&](int e, float z) {
        const uint32_t key = key_of(z);
        if (key > kf || (key == kf && e <= lim)) {
            const uint32_t slot = atomicAdd(&sc.s.n_cand, 1u);
            if (slot < (uint32_t)kMaxSel) list[slot] = support_key(z, e);
        }
    });
    __syncthreads();
    return min((int)sc.s.n_cand, kMaxSel);
}

template <int O>
__device__ __forceinline__ void wave_scan_step_u64(uint64_t& v, int lane) {
    const uint64_t t = ((uint64_t)up_partner<O>((uint32_t)(v >> 32)) << 32) | up_partner<O>((uint32_t)v);
    if (lane >= O) v += t;
}

__device__ __forceinline__ uint64_t wave_incl_u64(uint64_t v, int lane) {
    wave_scan_step_u64<1>(v, lane);
    wave_scan_step_u64<2>(v, lane);
    wave_scan_step_u64<4>(v, lane);
    wave_scan_step_u64<8>(v, lane);
    wave_scan_step_u64<16>(v, lane);
    wave_scan_step_u64<32>(v, lane);
    return v;
}

__device__ __forceinline__ uint64_t read_lane_u64(uint64_t v, int l) {
    l = __builtin_amdgcn_readfirstlane(l);
    return ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(v >> 32), l) << 32) |
           (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, l);
}

// Inclusive scan in thread order; *total is the workgroup's sum.
__device__ __forceinline__ uint64_t block_incl_u64(uint64_t v, uint64_t* s, uint64_t* total) {
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    if (__ballot(v != 0)) v = wave_incl_u64(v, lane);
    __syncthreads();
    if (lane == kWave - 1) s[w] = v;
    __syncthreads();
    // Each 16-lane row scans the 16 wave totals.
    static_assert(kWaves == 16, "one lane per wave total");
    uint64_t t = s[lane & 15];
    wave_scan_step_u64<1>(t, lane & 15);
    wave_scan_step_u64<2>(t, lane & 15);
    wave_scan_step_u64<4>(t, lane & 15);
    wave_scan_step_u64<8>(t, lane & 15);
    *total = read_lane_u64(t, 15);
    return v + (w ? read_lane_u64(t, w - 1) : 0);
}

// First position of the sorted list[0, m) where A + the running mass exceeds
// target, or m.
__device__ int first_crossing(const uint64_t* list, int m, float M, uint64_t A, uint64_t target, SelScratch& sc) {
    if (threadIdx.x == 0) sc.s.i[0] = m;
    for (int base = 0; base < m; base += NTF) {
        const int i = base + (int)threadIdx.x;
        uint64_t tot;
        const uint64_t incl = block_incl_u64(i < m ? weight_fx(key_value(list[i]), M) : 0, sc.s.w64, &tot);
        if (i < m && A + incl > target) atomicMin(&sc.s.i[0], i);
        __syncthreads();
        A += tot;
        if (sc.s.i[0] < m) break;
    }
    const int r = sc.s.i[0];
    __syncthreads();
    return r;
}

// Units of a draw's weights, as fine as their sum allows (at most 2^64): a
// top-k's kept entries in LDS, a whole row.
constexpr int kListBits = 50, kRowBits = 45;
static_assert(kMaxSel <= 1 << (63 - kListBits) && kMaxV <= 1 << (63 - kRowBits), "sum of the weights");

// Inverse-CDF draw over the kept entries (zf, lim) in id order, from the
// masses of the row's `segs` segments of SPAN chunks in sc.s.mass, sums of
// draw_fx<BITS>: first t with C_t > u * W, else the last with mass.
template <int DT, int SPAN, int BITS>
__device__ void draw_from_segments(const SelParams& P, const void* row, int n, int segs, float M, float zf, int lim,
                                   const Scale& scale, SelScratch& sc) {
    const int lane = threadIdx.x & (kWave - 1);
    __syncthreads();
    if (threadIdx.x < kWave) {
        const uint64_t m = lane < segs ? sc.s.mass[lane] : 0;
        const uint64_t incl = wave_incl_u64(m, lane);
        const uint64_t W = __shfl((unsigned long long)incl, kWave - 1, kWave);
        const uint64_t target = (uint64_t)((double)P.u[n] * (double)W);
        const uint64_t over = __ballot(incl > target), has = __ballot(m > 0);
        const int c = over ? __builtin_ctzll(over) : (has ? 63 - __builtin_clzll(has) : -1);
        if (lane == max(c, 0)) {
            sc.s.i[0] = c;
            // Mass still to pass inside the segment; all of it when nothing crosses.
            sc.s.base = over ? target - (incl - m) : ~0ull;
            sc.s.fx = (float)((double)W / (double)(1ull << BITS));
        }
    }
    __syncthreads();
    const int c = sc.s.i[0];
    const uint64_t need = sc.s.base;
    const float W = sc.s.fx;
    if (c < 0) {
        if (threadIdx.x == 0) {
            P.tok[n] = (int64_t)D3D_TOKEN_EMPTY_DISTRIBUTION;
            if (P.tok_prob) P.tok_prob[n] = 0.f;
        }
        return;
    }
    constexpr int PER = SPAN * kChunk / NTF;  // consecutive entries per thread
    const int e0 = c * SPAN * kChunk + (int)threadIdx.x * PER;
    float z[PER];
    uint64_t wt[PER], sum = 0;
#pragma unroll
    for (int q = 0; q < PER; ++q) z[q] = rows::load_one<DT>(row, min(e0 + q, P.V - 1));
    scale.tile(z);
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const bool kept = e0 + q < P.V && (z[q] > zf || (z[q] == zf && e0 + q <= lim));
        wt[q] = kept ? draw_fx<BITS>(z[q], M) : 0;
        sum += wt[q];
    }
    uint64_t tot;
    uint64_t run = block_incl_u64(sum, sc.s.w64, &tot) - sum;
    int first = INT_MAX, last = -1;
    float z_first = 0.f, z_last = 0.f;
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        run += wt[q];
        if (wt[q]) {
            last = q;
            z_last = z[q];
            if (first == INT_MAX && run > need) {
                first = q;
                z_first = z[q];
            }
        }
    }
    if (threadIdx.x == 0) {
        sc.s.i[0] = INT_MAX;
        sc.s.i[1] = -1;
    }
    __syncthreads();
    if (first != INT_MAX) atomicMin(&sc.s.i[0], e0 + first);
    if (last >= 0) atomicMax(&sc.s.i[1], e0 + last);
    __syncthreads();
    // The segment has mass, so one of the two names an entry; its thread writes.
    const bool crossed = sc.s.i[0] != INT_MAX;
    const int e = crossed ? sc.s.i[0] : sc.s.i[1];
    if (crossed ? (first != INT_MAX && e == e0 + first) : (last >= 0 && e == e0 + last)) {
        P.tok[n] = e;
        if (P.tok_prob) P.tok_prob[n] = expf((crossed ? z_first : z_last) - M) / W;
    }
}

// The filter and draw of a row whose candidates did not fit: several passes
// over the row.
template <int DT>
__device__ void filter_row_general(const SelParams& P, const void* row, int n, float M, bool unit, SelScratch& sc) {
    float zf;
    int lim;
    filter_general<DT>(row, P.V, P.T, unit, P.k, P.top_p, false, sc.general, zf, lim);
    if (threadIdx.x == 0 && P.zf) {
        P.zf[n] = zf;
        P.lim[n] = lim;
    }
    if (!P.tok) return;
    __syncthreads();
    for (int c = threadIdx.x; c < kMaxChunks; c += NTF) sc.s.mass[c] = 0;
    __syncthreads();
    // A wave's 64 consecutive entries lie in one chunk.
    for (int base = 0; base < P.V; base += NTF) {
        const int e = base + (int)threadIdx.x;
        uint64_t w = 0;
        if (e < P.V) {
            const float z = scaled<DT>(row, e, P.T, unit);
            if (z > zf || (z == zf && e <= lim)) w = draw_fx<kRowBits>(z, M);
        }
        const uint64_t s = wave_incl_u64(w, threadIdx.x & (kWave - 1));
        if ((threadIdx.x & (kWave - 1)) == kWave - 1 && s)
            atomicAdd((unsigned long long*)&sc.s.mass[e / kChunk], (unsigned long long)s);
    }
    draw_from_segments<DT, 1, kRowBits>(P, row, n, P.C, M, zf, lim, Scale(P.T), sc);
}

// Row maximum of the scaled logits (the caller's value is per thread).
__device__ __forceinline__ float row_max(float m, SelScratch& sc) {
    const float r = block_max_f(m, sc.s.f);
    __syncthreads();
    return r;
}

// One workgroup per row: the sorted support and its draw (kSupport), the
// sorted top-k (kTopk), or the top-k (and top-p) filter and its draw (kFilter).
template <int DT, bool VEC, SelMode M>
__global__ __launch_bounds__(NTF) void select_kernel(SelParams P) {
    __shared__ uint64_t list[kMaxSel];
    __shared__ uint16_t groups[kMaxGroups];
    __shared__ SelScratch sc;
    const int n = blockIdx.x, k = P.k;
    const bool unit = P.T == 1.0f;
    const void* row = rows::row_ptr<DT>(P.logits, n, P.V);
    float tie;
    int m = collect<DT, VEC>(P, row, P.gmax + (size_t)n * P.C * NT, k, unit, list, groups, sc, tie);
    const bool fits = m >= 0, tied = fits && m < k;
    if (tied) m = append_ties<DT>(P, row, tie, m, k, unit, list, sc);
    if constexpr (M == kFilter) {
        // NaN entries may be among the k largest only if fewer others exist.
        bool general = !fits || m < k;
        if (tied && !general) {
            // Every entry at the tie is kept; the list holds the first few of
            // them, which is enough if they weigh nothing.
            float mx = -INFINITY;
            for (int i = threadIdx.x; i < m; i += NTF) mx = fmaxf(mx, key_value(list[i]));
            general = draw_fx<kMassBits>(tie, row_max(mx, sc)) != 0;
        }
        if (general) {
            const float* gm = P.gmax + (size_t)n * P.C * NT;
            float mx = -INFINITY;
            for (int i = threadIdx.x; i < P.C * NT; i += NTF) mx = fmaxf(mx, gm[i]);
            __syncthreads();
            mx = row_max(mx, sc);
            filter_row_general<DT>(P, row, n, unit ? mx : mx / P.T, unit, sc);
            return;
        }
        pad_and_sort(list, m, 0, sc.s.rank);
        const float mx = key_value(list[0]);
        const uint32_t K = ~(uint32_t)(list[k - 1] >> kIdBits);
        // The kept prefix: everything at or above the k-th largest value.
        if (threadIdx.x == 0) sc.s.i[1] = m;
        __syncthreads();
        for (int i = k + (int)threadIdx.x; i < m; i += NTF)
            if (~(uint32_t)(list[i] >> kIdBits) < K) atomicMin(&sc.s.i[1], i);
        __syncthreads();
        int keep = sc.s.i[1];
        float zf = float_of(K);
        int lim = INT_MAX;
        if (P.top_p < 1.0f) {
            uint64_t part = 0, S;
            for (int i = threadIdx.x; i < keep; i += NTF) part += weight_fx(key_value(list[i]), mx);
            block_incl_u64(part, sc.s.w64, &S);
            const int at = first_crossing(list, keep, mx, 0, (uint64_t)((double)P.top_p * (double)S), sc);
            if (at < keep) {
                keep = at + 1;
                zf = key_value(list[at]);
                lim = (int)(list[at] & ((1ull << kIdBits) - 1));
            }
        }
        if (threadIdx.x == 0 && P.zf) {
            P.zf[n] = zf;
            P.lim[n] = lim;
        }
        if (!P.tok) return;
        for (int c = threadIdx.x; c < kMaxChunks; c += NTF) sc.s.mass[c] = 0;
        __syncthreads();
        for (int i = threadIdx.x; i < keep; i += NTF) {
            const uint64_t w = draw_fx<kListBits>(key_value(list[i]), mx);
            const int c = (int)(list[i] & ((1ull << kIdBits) - 1)) / kChunk;
            if (w) atomicAdd((unsigned long long*)&sc.s.mass[c], (unsigned long long)w);
        }
        draw_from_segments<DT, 1, kListBits>(P, row, n, P.C, mx, zf, lim, Scale(P.T), sc);
    } else if constexpr (M == kSupport) {
        // A support short of k entries (NaN elsewhere): up to 64 the slots stay
        // empty, as with the top-k kernels, wider ones list NaN entries by id.
        if (!fits || (m < k && k > 64 && k < P.V)) m = collect_general<DT>(P, row, k, unit, list, sc);
        pad_and_sort(list, m, k, sc.s.rank);
        support_draw(list, k, P.top_p, P.u[n], P.tok + n, P.ids + (size_t)n * k, P.probs + (size_t)n * k,
                     P.tok_prob ? P.tok_prob + n : nullptr, sc.s.f, sc.s.i);
    } else {
        if (!fits) m = collect_general<DT>(P, row, k, unit, list, sc);
        pad_and_sort(list, m, k, sc.s.rank);
        float logz = 0.f;
        if (P.lse) {
            // logsumexp over the chunk records, in a fixed order.
            const float2 r = (int)threadIdx.x < P.C ? P.lse[(size_t)n * P.C + threadIdx.x] : make_float2(-INFINITY, 0.f);
            const float mx = row_max(r.x, sc);
            // Only the first wave holds records.
            if (threadIdx.x < kWave) {
                const float se = wave_sum(r.x != -INFINITY ? r.y * expf(r.x - mx) : 0.f);
                if (threadIdx.x == 0) sc.s.fx = mx + logf(se);
            }
            __syncthreads();
            logz = sc.s.fx;
        }
        for (int r = threadIdx.x; r < k; r += NTF) {
            const bool has = list[r] != ~0ull;
            const int e = has ? (int)(list[r] & ((1ull << kIdBits) - 1)) : -1;
            P.ids[(size_t)n * k + r] = e;
            // The value as the row holds it (the key has lost the sign of zero).
            if (P.probs) {
                const float x = has ? rows::load_one<DT>(row, e) : -INFINITY;
                P.probs[(size_t)n * k + r] = P.lse ? x - logz : x;
            }
        }
    }
}

template <int DT, bool VEC, SelMode M>
void launch_select(const SelParams& P, int N, hipStream_t s) {
    if (M == kTopk && P.lse)
        hipLaunchKernelGGL((max_kernel<DT, VEC, true, true>), dim3(P.C, N), dim3(NT), 0, s, P);
    else
        hipLaunchKernelGGL((max_kernel<DT, VEC, true, false>), dim3(P.C, N), dim3(NT), 0, s, P);
    hipLaunchKernelGGL((select_kernel<DT, VEC, M>), dim3(N), dim3(NTF), 0, s, P);
}

// Calls f(P, rows) for batches of rows: P's row pointers moved to the batch,
// its scratch the same for every batch.
template <typename F>
hipError_t for_batches(SelParams P, int dtype, int N, F&& f) {
    const size_t esize = dtype == kF32 ? 4 : 2;
    const size_t k = P.k;
    const bool vec = ((uintptr_t)P.logits % 16 == 0) && ((size_t)P.V * esize) % 16 == 0;
    for (int n0 = 0; n0 < N; n0 += kRowBatch) {
        const int nb = std::min(kRowBatch, N - n0);
        f(P, nb, vec);
        const hipError_t err = hipGetLastError();
        if (err != hipSuccess) return err;
        P.logits = static_cast<const char*>(P.logits) + (size_t)nb * P.V * esize;
        if (P.u) P.u += nb;
        if (P.tok) P.tok += nb;
        if (P.ids) P.ids += nb * k;
        if (P.probs) P.probs += nb * k;
        if (P.tok_prob) P.tok_prob += nb;
        if (P.zf) P.zf += nb;
        if (P.lim) P.lim += nb;
    }
    return hipSuccess;
}

template <SelMode M>
hipError_t run_select(const SelParams& P, int dtype, int N, hipStream_t s) {
    return for_batches(P, dtype, N, [&](const SelParams& B, int nb, bool vec) {
        if (dtype == kF32) {
            if (vec) launch_select<kF32, true, M>(B, nb, s);
            else launch_select<kF32, false, M>(B, nb, s);
        } else {
            if (vec) launch_select<kBF16, true, M>(B, nb, s);
            else launch_select<kBF16, false, M>(B, nb, s);
        }
    });
}

// ---------------------------------------------------------------- nucleus

__device__ __forceinline__ float max_of_chunks(const SelParams& P, int n, float* s) {
    if (threadIdx.x < kWave) {
        const float m = (int)threadIdx.x < P.C ? P.cmax[(size_t)n * P.C + threadIdx.x] : -INFINITY;
        const float r = wave_max(m);
        if (threadIdx.x == 0) *s = r;
    }
    __syncthreads();
    return *s;
}

// Bin of M - z for entries with mass (M - z < 28), kBins past them.
__device__ __forceinline__ int mass_bin(float d) {
    return d < (float)kBins / kBinScale ? (int)(d * kBinScale) : kBins;
}

// Workgroup (part, row): the part's mass histogram, and its sums over runs
// of kFine bins.
template <int DT, bool VEC>
__global__ __launch_bounds__(NT) void mass_hist_kernel(SelParams P) {
    constexpr int E = rows::Vec<DT>::E;
    __shared__ unsigned long long h[kBins];
    __shared__ float s_m;
    const int p = blockIdx.x, n = blockIdx.y;
    for (int b = threadIdx.x; b < kBins; b += NT) h[b] = 0;
    const float M = max_of_chunks(P, n, &s_m);
    const void* row = rows::row_ptr<DT>(P.logits, n, P.V);
    const Scale scale(P.T);
    const int c1 = min((p + 1) * P.span, P.C);
    for (int c = p * P.span; c < c1; ++c) {
        float x[kGroup];
        rows::load_tile<DT, VEC, false, kGroup>(row, P.V, c * kChunk + (int)threadIdx.x * E, NT * E, -INFINITY, x);
        scale.tile(x);
        uint64_t w[kGroup];
#pragma unroll
        for (int l = 0; l < kGroup; ++l) w[l] = weight_fx(x[l], M);
#pragma unroll
        for (int l = 0; l < kGroup; ++l)
            if (w[l]) atomicAdd(&h[min(mass_bin(M - x[l]), kBins - 1)], (unsigned long long)w[l]);
    }
    __syncthreads();
    uint64_t* out = P.hist + ((size_t)n * P.parts + p) * kBins;
    for (int b = threadIdx.x; b < kBins; b += NT) out[b] = h[b];
    if (threadIdx.x < 64) {
        uint64_t s = 0;
        if (threadIdx.x < kCoarse)
            for (int f = 0; f < kFine; ++f) s += h[threadIdx.x * kFine + f];
        P.coarse[((size_t)n * P.parts + p) * 64 + threadIdx.x] = s;
    }
}

// The row's crossing bin from the parts' histograms; every workgroup of the
// row gets the same record.
__device__ __forceinline__ NucRec find_bin(const SelParams& P, int n, float M, uint64_t (*s_part)[64], NucRec* s_rec,
                                           unsigned long long* s_fine) {
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    const uint64_t* co = P.coarse + (size_t)n * P.parts * 64;
    uint64_t acc = 0;
    for (int p = w; p < P.parts; p += NT / kWave) acc += co[p * 64 + lane];
    s_part[w][lane] = acc;
    if (threadIdx.x < kFine) s_fine[threadIdx.x] = 0;
    __syncthreads();
    if (w == 0) {
        uint64_t t = 0;
#pragma unroll
        for (int q = 0; q < NT / kWave; ++q) t += s_part[q][lane];
        const uint64_t incl = wave_incl_u64(t, lane);
        const uint64_t S = __shfl((unsigned long long)incl, kWave - 1, kWave);
        const uint64_t target = (uint64_t)((double)P.top_p * (double)S);
        const uint64_t over = __ballot(incl > target);
        const int b = over ? __builtin_ctzll(over) : -1;
        if (lane == max(b, 0)) *s_rec = NucRec{incl - t, target, M, b};
    }
    __syncthreads();
    NucRec r = *s_rec;
    if (r.bin < 0) return r;
    const uint64_t* hi = P.hist + (size_t)n * P.parts * kBins + r.bin * kFine;
    for (int i = threadIdx.x; i < P.parts * kFine; i += NT) {
        const uint64_t v = hi[(size_t)(i / kFine) * kBins + (i % kFine)];
        if (v) atomicAdd(&s_fine[i % kFine], (unsigned long long)v);
    }
    __syncthreads();
    if (w == 0) {
        const uint64_t t = lane < kFine ? s_fine[lane] : 0;
        const uint64_t incl = r.above + wave_incl_u64(t, lane);
        const uint64_t over = __ballot(incl > r.target);
        const int b = __builtin_ctzll(over);  // the coarse sum crosses, so one of its bins does
        if (lane == b) *s_rec = NucRec{incl - t, r.target, M, r.bin * kFine + b};
    }
    __syncthreads();
    return *s_rec;
}

// Workgroup (part, row): the part's entries of the crossing bin as support
// keys into the row's list.
template <int DT, bool VEC>
__global__ __launch_bounds__(NT) void nucleus_gather_kernel(SelParams P) {
    constexpr int E = rows::Vec<DT>::E;
    __shared__ uint64_t s_part[NT / kWave][64];
    __shared__ unsigned long long s_fine[kFine];
    __shared__ NucRec s_rec;
    __shared__ float s_m;
    const int p = blockIdx.x, n = blockIdx.y, lane = threadIdx.x & (kWave - 1);
    const float M = max_of_chunks(P, n, &s_m);
    const NucRec rec = find_bin(P, n, M, s_part, &s_rec, s_fine);
    if (p == 0 && threadIdx.x == 0) P.rec[n] = rec;
    const void* row = rows::row_ptr<DT>(P.logits, n, P.V);
    if (rec.bin < 0) return;
    const Scale scale(P.T);
    // The bin's entries lie in (M - (bin + 1) / 32, M - bin / 32] T; a range of
    // x widened by more than the roundings of M - z, z = x / T and this
    // product is tested first, and only a wave with an entry in it scales that
    // entry (a few of 64 in a bin's worth of a row).
    const float z_hi = M - (float)rec.bin / kBinScale, z_lo = z_hi - 1.f / kBinScale;
    const float pad = (fabsf(M) + 32.f) * P.T * 0x1p-18f;
    const float x_mid = (0.5f * z_hi + 0.5f * z_lo) * P.T;
    // Out of range: every entry is taken for near.
    const float x_half = fabsf(x_mid) < INFINITY ? (0.5f / kBinScale) * P.T + pad : INFINITY;
    uint64_t* list = P.list + (size_t)n * kMaxSel;
    const int c1 = min((p + 1) * P.span, P.C);
    for (int c = p * P.span; c < c1; ++c) {
        const int first = c * kChunk + (int)threadIdx.x * E;
        float x[kGroup];
        rows::load_tile<DT, VEC, false, kGroup>(row, P.V, first, NT * E, -INFINITY, x);
        uint32_t hits = 0;  // bit l: entry l lies in the crossing bin
#pragma unroll
        for (int l = 0; l < kGroup; ++l) {
            const bool near = !(fabsf(x[l] - x_mid) > x_half);
            if (!__ballot(near)) continue;
            float z[1] = {x[l]};
            scale.tile(z);
            x[l] = z[0];
            hits |= (near && mass_bin(M - z[0]) == rec.bin ? 1u : 0u) << l;
        }
        // One slot reservation per wave that holds such entries.
        const uint32_t cnt = __popc(hits);
        if (__ballot(cnt != 0)) {
            uint32_t incl = cnt;
#pragma unroll
            for (int o = 1; o < kWave; o <<= 1) {
                const uint32_t t = __shfl_up(incl, o, kWave);
                if (lane >= o) incl += t;
            }
            uint32_t base = 0;
            if (lane == kWave - 1) base = atomicAdd(&P.counter[n], incl);
            uint32_t slot = (uint32_t)__shfl((int)base, kWave - 1, kWave) + incl - cnt;
#pragma unroll
            for (int l = 0; l < kGroup; ++l)
                if ((hits >> l) & 1u) {
                    if (slot < (uint32_t)kMaxSel) list[slot] = support_key(x[l], rows::tile_index<DT>(first, NT * E, l));
                    ++slot;
                }
        }
    }
}

// One workgroup per row: places the cut among the gathered entries and draws.
template <int DT>
__global__ __launch_bounds__(NTF) void nucleus_finish_kernel(SelParams P) {
    __shared__ uint64_t list[kMaxSel];
    __shared__ unsigned long long s_sub[NTF];
    __shared__ SelScratch sc;
    const int n = blockIdx.x;
    const bool unit = P.T == 1.0f;
    const void* row = rows::row_ptr<DT>(P.logits, n, P.V);
    // The record, the count and this thread's first gathered entry load
    // together (the list has kMaxSel slots, whatever they hold).
    const NucRec rec = P.rec[n];
    const uint32_t counted = P.counter[n];
    const uint64_t key0 = P.list[(size_t)n * kMaxSel + threadIdx.x];
    const uint32_t m = rec.bin < 0 ? 0u : counted;
    if (m > (uint32_t)kMaxSel) {
        filter_row_general<DT>(P, row, n, rec.M, unit, sc);
        return;
    }
    const uint64_t* src = P.list + (size_t)n * kMaxSel;
    float zf = -INFINITY;
    int lim = INT_MAX;
    if (P.tok) {
        // Mass of each part's entries in the bins before the crossing one.
        const int lane = threadIdx.x & (kWave - 1), b = rec.bin < 0 ? kBins : rec.bin;
        for (int p = threadIdx.x / kWave; p < P.parts; p += kWaves) {
            uint64_t v = 0;
            if (lane < b / kFine) v = P.coarse[((size_t)n * P.parts + p) * 64 + lane];
            if (lane < b % kFine) v += P.hist[((size_t)n * P.parts + p) * kBins + b / kFine * kFine + lane];
            v = wave_incl_u64(v, lane);
            if (lane == kWave - 1) sc.s.mass[p] = v;
        }
    }
    uint64_t cut = 0;  // key of the last kept entry
    if (rec.bin >= 0) {
        // A second histogram, of the gathered entries over 1,024 parts of the
        // bin; only the part where the running mass crosses is sorted (entries
        // of one or a few equal values, mostly).
        auto sub_of = [&](uint64_t key) {
            const float d = (rec.M - key_value(key)) * kBinScale - (float)rec.bin;
            return min(max((int)(d * (float)NTF), 0), NTF - 1);
        };
        s_sub[threadIdx.x] = 0;
        if (threadIdx.x == 0) {
            sc.s.n_cand = 0;
            sc.s.i[0] = NTF - 1;
        }
        __syncthreads();
        for (int i = threadIdx.x; i < (int)m; i += NTF) {
            const uint64_t key = i < NTF ? key0 : src[i], w = weight_fx(key_value(key), rec.M);
            if (w) atomicAdd(&s_sub[sub_of(key)], (unsigned long long)w);
        }
        __syncthreads();
        uint64_t tot;
        const uint64_t mine = s_sub[threadIdx.x];
        const uint64_t incl = rec.above + block_incl_u64(mine, sc.s.w64, &tot);
        if (incl > rec.target) atomicMin(&sc.s.i[0], (int)threadIdx.x);
        __syncthreads();
        const int b = sc.s.i[0];
        if ((int)threadIdx.x == b) sc.s.base = incl - mine;
        for (int i = threadIdx.x; i < (int)m; i += NTF) {
            const uint64_t key = i < NTF ? key0 : src[i];
            if (sub_of(key) == b) list[atomicAdd(&sc.s.n_cand, 1u)] = key;
        }
        __syncthreads();
        const int m2 = (int)sc.s.n_cand;
        const uint64_t above = sc.s.base;
        pad_and_sort(list, m2, 0, sc.s.rank);
        // The part's mass crosses the target, so one of its entries does.
        const int at = max(min(first_crossing(list, m2, rec.M, above, rec.target, sc), m2 - 1), 0);
        cut = list[at];
        zf = key_value(cut);
        lim = (int)(cut & ((1ull << kIdBits) - 1));
    }
    if (threadIdx.x == 0 && P.zf) {
        P.zf[n] = zf;
        P.lim[n] = lim;
    }
    if (!P.tok) return;
    __syncthreads();
    for (int i = threadIdx.x; i < (int)m; i += NTF) {
        const uint64_t key = i < NTF ? key0 : src[i], w = key <= cut ? weight_fx(key_value(key), rec.M) : 0;
        const int c = (int)(key & ((1ull << kIdBits) - 1)) / (kChunk * P.span);
        if (w) atomicAdd((unsigned long long*)&sc.s.mass[c], (unsigned long long)w);
    }
    // The cut's entry weighs at least one unit, so every kept one does, and the
    // masses are draw_fx's.
    if (P.span == 2)
        draw_from_segments<DT, 2, kMassBits>(P, row, n, P.parts, rec.M, zf, lim, Scale(P.T), sc);
    else
        draw_from_segments<DT, 1, kMassBits>(P, row, n, P.parts, rec.M, zf, lim, Scale(P.T), sc);
}

template <int DT, bool VEC>
void launch_nucleus(const SelParams& P, int N, hipStream_t s) {
    hipLaunchKernelGGL((max_kernel<DT, VEC, false, false>), dim3(P.C, N), dim3(NT), 0, s, P);
    hipLaunchKernelGGL((mass_hist_kernel<DT, VEC>), dim3(P.parts, N), dim3(NT), 0, s, P);
    hipLaunchKernelGGL((nucleus_gather_kernel<DT, VEC>), dim3(P.parts, N), dim3(NT), 0, s, P);
    hipLaunchKernelGGL((nucleus_finish_kernel<DT>), dim3(N), dim3(NTF), 0, s, P);
}

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

int chunks_of(int64_t V) { return (int)((V + kChunk - 1) / kChunk); }

// Chunks per part of a nucleus row: two (half the histograms to merge), one
// while that would leave most of the 256 CUs without two workgroups.
int part_span(int N, int C) { return N * ((C + 1) / 2) >= 512 ? 2 : 1; }

struct FilterLayout {
    size_t hist, coarse, cmax, list, counter, rec, total;
};

// Scratch of one batch of rows (whichever of the two ways needs more).
FilterLayout filter_layout(int N, int64_t V) {
    const size_t n = std::min(N, kRowBatch), C = chunks_of(V);
    const size_t parts = (C + part_span((int)n, (int)C) - 1) / part_span((int)n, (int)C);
    FilterLayout l;
    l.hist = 0;
    l.coarse = l.hist + align256(n * parts * kBins * sizeof(uint64_t));
    l.cmax = l.coarse + align256(n * parts * 64 * sizeof(uint64_t));
    l.list = l.cmax + align256(n * C * sizeof(float));
    l.counter = l.list + align256(n * kMaxSel * sizeof(uint64_t));
    l.rec = l.counter + align256(n * sizeof(uint32_t));
    l.total = std::max(l.rec + align256(n * sizeof(NucRec)), select_scratch_bytes((int)n, (int)C, false));
    return l;
}

}  // namespace

size_t select_scratch_bytes(int N, int chunks, bool lse) {
    const size_t n = std::min(N, kRowBatch);
    return align256(n * chunks * NT * sizeof(float)) + (lse ? align256(n * chunks * sizeof(float2)) : 0);
}

hipError_t select_support(const void* logits, int dtype, int N, int V, float T, int S, float top_p, const float* u,
                          int64_t* tok, int64_t* ids, float* probs, float* tok_prob, void* scratch, hipStream_t s) {
    SelParams P{};
    P.logits = logits;
    P.V = V;
    P.C = chunks_of(V);
    P.T = T;
    P.k = S;
    P.top_p = top_p;
    P.u = u;
    P.tok = tok;
    P.ids = ids;
    P.probs = probs;
    P.tok_prob = tok_prob;
    P.gmax = static_cast<float*>(scratch);
    return run_select<kSupport>(P, dtype, N, s);
}

hipError_t select_topk(const void* logits, int dtype, int N, int V, int k, bool lse, int64_t* ids, float* vals,
                       void* scratch, hipStream_t s) {
    SelParams P{};
    P.logits = logits;
    P.V = V;
    P.C = chunks_of(V);
    P.T = 1.0f;
    P.k = k;
    P.top_p = 1.0f;
    P.ids = ids;
    P.probs = vals;
    P.gmax = static_cast<float*>(scratch);
    if (lse)
        P.lse = reinterpret_cast<float2*>(static_cast<char*>(scratch) +
                                          align256((size_t)std::min(N, kRowBatch) * P.C * NT * sizeof(float)));
    return run_select<kTopk>(P, dtype, N, s);
}

}  // namespace filt
}  // namespace d3d

using namespace d3d;

extern "C" size_t d3d_filter_rows_workspace_bytes(int N, int64_t V) {
    using namespace filt;
    if (N < 1 || V < 1 || V > kMaxV) return 0;
    return filter_layout(N, V).total;
}

extern "C" int d3d_filter_rows(const void* logits, int dtype, int N, int64_t V, float temperature, int top_k,
                               float top_p, const float* uniforms, float* zfloor_out, int32_t* zlimit_out,
                               int64_t* tokens_out, float* probs_out, void* workspace, size_t workspace_bytes,
                               void* stream) {
    using namespace filt;
    if (N < 0 || N > 65535 || V < 1 || V > kMaxV || top_k < 0) return D3D_E_SHAPE;
    if (dtype != D3D_DTYPE_F32 && dtype != D3D_DTYPE_BF16) return D3D_E_DTYPE;
    if (!(temperature > 1e-5f)) return D3D_E_UNSUPPORTED;
    if (!(top_p > 0.f && top_p <= 1.f)) return D3D_E_VALUE;
    const int k = top_k < V ? top_k : 0;
    if (k > kSelectMaxK || (k == 0 && !(top_p < 1.f))) return D3D_E_UNSUPPORTED;
    if (N == 0) return D3D_OK;
    const bool filter = zfloor_out != nullptr, draw = tokens_out != nullptr;
    if (!logits || !workspace || (!filter && !draw) || filter != (zlimit_out != nullptr) || (draw && !uniforms))
        return D3D_E_NULL;
    const FilterLayout l = filter_layout(N, V);
    if (workspace_bytes < l.total) return D3D_E_WORKSPACE;
    char* ws = static_cast<char*>(workspace);
    hipStream_t s = static_cast<hipStream_t>(stream);
    SelParams P{};
    P.logits = logits;
    P.V = (int)V;
    P.C = chunks_of(V);
    P.T = temperature;
    P.k = k;
    P.top_p = top_p;
    P.u = uniforms;
    P.tok = tokens_out;
    P.tok_prob = probs_out;
    P.zf = zfloor_out;
    P.lim = zlimit_out;
    if (k > 0) {
        P.gmax = reinterpret_cast<float*>(ws);
        return (int)run_select<kFilter>(P, dtype, N, s);
    }
    P.hist = reinterpret_cast<uint64_t*>(ws + l.hist);
    P.coarse = reinterpret_cast<uint64_t*>(ws + l.coarse);
    P.cmax = reinterpret_cast<float*>(ws + l.cmax);
    P.list = reinterpret_cast<uint64_t*>(ws + l.list);
    P.counter = reinterpret_cast<uint32_t*>(ws + l.counter);
    P.rec = reinterpret_cast<NucRec*>(ws + l.rec);
    P.span = part_span(std::min(N, kRowBatch), P.C);
    P.parts = (P.C + P.span - 1) / P.span;
    return (int)for_batches(P, dtype, N, [&](const SelParams& B, int nb, bool vec) {
        if (dtype == D3D_DTYPE_F32) {
            if (vec) launch_nucleus<kF32, true>(B, nb, s);
            else launch_nucleus<kF32, false>(B, nb, s);
        } else {
            if (vec) launch_nucleus<kBF16, true>(B, nb, s);
            else launch_nucleus<kBF16, false>(B, nb, s);
        }
    });
}
