// Row filters of the draft's proposal distributions, and wide sparse
// supports, over rows of V logits.
//
// Reference behaviour (D3D repository):
//   single/eval_sync.py:292-295  top-k: z = logits.float() / T, entries with
//       z below the k-th largest z are masked out (ties with it are kept)
//   single/eval_sync.py:296-303  top-p: sort z descending, softmax, cumsum;
//       entry j > 0 of the sorted order goes when the cumulative probability
//       of entries 0..j-1 exceeds top_p (the crossing entry is kept)
//   single/eval_sync.py:341-367  _sample_with_sparse_probs: the support is
//       torch.topk(z, S) in descending order (S = V when top_k = 0), the
//       nucleus filter over that order, softmax, a draw from the support
//
// A filter is one record per row, (zf, lim): entry e with scaled logit z is
// kept iff z > zf, or z == zf and e <= lim.  Sorted orders break ties by the
// lower id (the order of a stable descending sort), so a cut through a run
// of equal values keeps its lowest ids.
//
// d3d_row_filter is the general selection, for rows and top-k of any size
// (select.hip holds the faster one for V <= 2^18 and top_k <= 4096): one
// workgroup per row makes several passes over the row (it stays in L2 after
// the first): the row maximum, an exact radix
// select of the k-th largest value (four 8-bit digit passes of counts over
// order-preserving 32-bit keys), and for top-p a radix descent over the same
// digits with mass histograms: each entry adds w = exp(z - max) as a 64-bit
// fixed-point integer (2^-40 units), so the sums are exact integers and the
// cut does not depend on the order of the atomic adds.  The entry where the
// cumulative mass first exceeds top_p * sum(w) fixes (zf, lim); one more
// pass in id order finds the tie limit when the cut falls inside a run of
// equal values.
//
// Supports wider than kSelectMaxK: support_gather_kernel writes each kept entry of the
// exact top-S filter as one 50-bit key ((~key(z)) << 18 | id: ascending
// keys are descending values, ties by ascending id, every key distinct),
// rocPRIM's segmented radix sort orders them, and one workgroup per row
// forms softmax over the support, the nucleus filter in support order and
// the inverse-CDF draw (first s with C_s > u * W, else the last s with
// positive weight).
#include "d3d_common.hpp"
#include "rowstats.hpp"
#include "select.hpp"
#include "../../include/d3d_hip.h"

#include <limits.h>

#include <algorithm>
#include <rocprim/device/device_segmented_radix_sort.hpp>

namespace d3d {
namespace filt {

struct FilterParams {
    const void* logits;  // [N, V]
    int V;
    float T;
    int top_k;    // 0: off
    float top_p;  // >= 1: off
    int exact;    // the top-k filter keeps exactly top_k entries (ties by id)
    float* zf;    // [N]
    int32_t* lim; // [N]
};

template <int DT>
__global__ __launch_bounds__(NTF) void row_filter_kernel(FilterParams P) {
    __shared__ FilterScratch sc;
    const int n = blockIdx.x;
    float zf;
    int lim;
    filter_general<DT>(rows::row_ptr<DT>(P.logits, n, P.V), P.V, P.T, P.T == 1.0f, P.top_k, P.top_p, P.exact != 0, sc,
                       zf, lim);
    if (threadIdx.x == 0) {
        P.zf[n] = zf;
        P.lim[n] = lim;
    }
}

// Wide supports ---------------------------------------------------------------

// Workgroup (chunk, row): the kept entries of its 4096-entry chunk, as
// support keys, at consecutive slots reserved with one atomic per chunk.
template <int DT>
__global__ __launch_bounds__(rows::NT) void support_gather_kernel(const void* logits, int V, float T,
                                                                  const float* zf, const int32_t* lim, int S,
                                                                  uint64_t* keys, uint32_t* counters) {
    constexpr int NT = rows::NT;
    const int c = blockIdx.x, n = blockIdx.y;
    const void* row = rows::row_ptr<DT>(logits, n, V);
    const bool unit = T == 1.0f;
    const float f = zf[n];
    const int l = lim[n];
    const uint32_t kf = key_of(f);
    __shared__ uint32_t s_w[NT / kWave];
    __shared__ uint32_t s_base;
    constexpr int PER = rows::kChunk / NT;  // 16 entries per thread
    uint64_t mine[PER];
    uint32_t cnt = 0;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int e = c * rows::kChunk + j * NT + threadIdx.x;
        mine[j] = ~0ull;
        if (e < V) {
            const uint32_t k = key_of(scaled<DT>(row, e, T, unit));
            if (k > kf || (k == kf && e <= l)) {
                mine[j] = ((uint64_t)(~k) << kIdBits) | (uint64_t)e;
                ++cnt;
            }
        }
    }
    // Exclusive offset of this thread among the chunk's kept entries.
    uint32_t incl = cnt;
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const uint32_t t = __shfl_up(incl, o, kWave);
        if (lane >= o) incl += t;
    }
    if (lane == kWave - 1) s_w[w] = incl;
    __syncthreads();
    uint32_t off = incl - cnt, total = 0;
#pragma unroll
    for (int k = 0; k < NT / kWave; ++k) {
        if (k < w) off += s_w[k];
        total += s_w[k];
    }
    if (threadIdx.x == 0) s_base = total ? atomicAdd(&counters[n], total) : 0u;
    __syncthreads();
    uint64_t* out = keys + (size_t)n * S;
    uint32_t slot = s_base + off;
#pragma unroll
    for (int j = 0; j < PER; ++j)
        if (mine[j] != ~0ull) {
            if (slot < (uint32_t)S) out[slot] = mine[j];  // the filter keeps exactly S
            ++slot;
        }
}

// One workgroup per row over its sorted support keys [S].
__global__ __launch_bounds__(NTF) void support_draw_kernel(const uint64_t* keys, int S, float top_p, const float* u,
                                                           int64_t* tok, int64_t* ids, float* probs,
                                                           float* tok_prob) {
    __shared__ float s_w[kWaves];
    __shared__ int s_i[2];
    const size_t n = blockIdx.x;
    support_draw(keys + n * S, S, top_p, u[n], tok + n, ids + n * S, probs + n * S, tok_prob ? tok_prob + n : nullptr,
                 s_w, s_i);
}

// Supports of at most kSelectMaxK entries: select.hip's group maxima (the
// vocabulary is not known when the workspace is sized, so for the longest).
static size_t select_bytes(int N) { return select_scratch_bytes(N, (int)(kMaxV / rows::kChunk), false); }

struct SupportLayout {
    size_t keys_in, keys_out, counters, offsets, temp, temp_bytes, total;
};

static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

static hipError_t sort_temp_bytes(int N, int S, size_t* bytes) {
    *bytes = 0;
    return rocprim::segmented_radix_sort_keys(nullptr, *bytes, (const uint64_t*)nullptr, (uint64_t*)nullptr,
                                              (unsigned int)((size_t)N * S), (unsigned int)N, (const int*)nullptr,
                                              (const int*)nullptr, 0, 32 + kIdBits, (hipStream_t)0, false);
}

static SupportLayout support_layout(int N, int S, size_t temp) {
    SupportLayout l;
    const size_t keys = align256((size_t)N * S * sizeof(uint64_t));
    l.keys_in = 0;
    l.keys_out = keys;
    l.counters = 2 * keys;
    l.offsets = l.counters + align256((size_t)N * sizeof(uint32_t));
    l.temp = l.offsets + align256((size_t)(N + 1) * sizeof(int));
    l.temp_bytes = temp;
    l.total = l.temp + align256(temp);
    return l;
}

// Per-row slot counters at 0, segment offsets n * S, every key slot ~0.
__global__ void support_setup_kernel(uint32_t* counters, int* offsets, uint64_t* keys, int N, int S) {
    const size_t total = (size_t)N * S;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x)
        keys[i] = ~0ull;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < N) counters[i] = 0;
    if (i <= N) offsets[i] = i * S;
}

}  // namespace filt
}  // namespace d3d

using namespace d3d;

extern "C" int d3d_row_filter(const void* logits, int dtype, int N, int64_t V, float temperature, int top_k,
                              float top_p, float* zfloor_out, int32_t* zlimit_out, void* stream) {
    using namespace filt;
    if (N < 0 || N > 65535 || V < 1 || V > (int64_t)INT_MAX / 2 || top_k < 0) return D3D_E_SHAPE;
    if (dtype != D3D_DTYPE_F32 && dtype != D3D_DTYPE_BF16) return D3D_E_DTYPE;
    if (!(temperature > 1e-5f)) return D3D_E_UNSUPPORTED;
    if (!(top_p > 0.f && top_p <= 1.f)) return D3D_E_VALUE;
    if (N == 0) return D3D_OK;
    if (!logits || !zfloor_out || !zlimit_out) return D3D_E_NULL;
    FilterParams P{logits, (int)V, temperature, top_k, top_p, 0, zfloor_out, zlimit_out};
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dtype == D3D_DTYPE_F32)
        hipLaunchKernelGGL(row_filter_kernel<kF32>, dim3(N), dim3(NTF), 0, s, P);
    else
        hipLaunchKernelGGL(row_filter_kernel<kBF16>, dim3(N), dim3(NTF), 0, s, P);
    const hipError_t err = hipGetLastError();
    return err == hipSuccess ? D3D_OK : (int)err;
}

extern "C" size_t d3d_support_workspace_bytes(int N, int S) {
    using namespace filt;
    if (N < 1 || S < 1) return 0;
    if (S <= kSelectMaxK) return select_bytes(N);
    size_t temp = 0;
    if (sort_temp_bytes(N, S, &temp) != hipSuccess) return 0;
    return support_layout(N, S, temp).total;
}

extern "C" int d3d_sample_support_wide(const void* logits, int dtype, int N, int64_t V, float temperature, int S,
                                       float top_p, const float* uniforms, int64_t* tokens_out,
                                       int64_t* support_ids_out, float* support_probs_out, float* token_probs_out,
                                       void* workspace, size_t workspace_bytes, void* stream) {
    using namespace filt;
    if (N < 0 || N > 65535 || V < 1 || V > kMaxV || S < 1 || S > V) return D3D_E_SHAPE;
    if ((size_t)N * S > (size_t)UINT_MAX) return D3D_E_SHAPE;
    if (dtype != D3D_DTYPE_F32 && dtype != D3D_DTYPE_BF16) return D3D_E_DTYPE;
    if (!(temperature > 1e-5f)) return D3D_E_UNSUPPORTED;
    if (!(top_p > 0.f && top_p <= 1.f)) return D3D_E_VALUE;
    if (N == 0) return D3D_OK;
    if (!logits || !uniforms || !tokens_out || !support_ids_out || !support_probs_out || !workspace)
        return D3D_E_NULL;
    if (S <= kSelectMaxK) {
        if (workspace_bytes < select_bytes(N)) return D3D_E_WORKSPACE;
        return (int)select_support(logits, dtype, N, (int)V, temperature, S, top_p, uniforms, tokens_out,
                                   support_ids_out, support_probs_out, token_probs_out, workspace,
                                   static_cast<hipStream_t>(stream));
    }
    size_t temp = 0;
    hipError_t err = sort_temp_bytes(N, S, &temp);
    if (err != hipSuccess) return (int)err;
    const SupportLayout lay = support_layout(N, S, temp);
    if (workspace_bytes < lay.total) return D3D_E_WORKSPACE;
    char* ws = static_cast<char*>(workspace);
    uint64_t* kin = reinterpret_cast<uint64_t*>(ws + lay.keys_in);
    uint64_t* kout = reinterpret_cast<uint64_t*>(ws + lay.keys_out);
    uint32_t* counters = reinterpret_cast<uint32_t*>(ws + lay.counters);
    int* offsets = reinterpret_cast<int*>(ws + lay.offsets);
    // The exact top-S filter's (zf, lim) live in the keys_out region until
    // the gather has read them (the sort writes keys_out afterwards).
    float* zf = reinterpret_cast<float*>(kout);
    int32_t* lim = reinterpret_cast<int32_t*>(kout) + N;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const size_t slots = (size_t)N * S;
    const int setup_blocks = (int)std::min<size_t>(1024, std::max<size_t>((N + 1 + 255) / 256, (slots + 255) / 256));
    hipLaunchKernelGGL(support_setup_kernel, dim3(setup_blocks), dim3(256), 0, s, counters, offsets, kin, N, S);
    FilterParams P{logits, (int)V, temperature, S < V ? S : 0, 1.0f, 1, zf, lim};
    const int C = (int)((V + rows::kChunk - 1) / rows::kChunk);
    if (S == V) {
        // The whole vocabulary: every entry is kept (zf = -inf keeps all but
        // NaN, which the key maps below -inf; those are dropped).
        FilterParams Q = P;
        Q.top_k = 0;
        if (dtype == D3D_DTYPE_F32)
            hipLaunchKernelGGL(row_filter_kernel<kF32>, dim3(N), dim3(NTF), 0, s, Q);
        else
            hipLaunchKernelGGL(row_filter_kernel<kBF16>, dim3(N), dim3(NTF), 0, s, Q);
    } else if (dtype == D3D_DTYPE_F32) {
        hipLaunchKernelGGL(row_filter_kernel<kF32>, dim3(N), dim3(NTF), 0, s, P);
    } else {
        hipLaunchKernelGGL(row_filter_kernel<kBF16>, dim3(N), dim3(NTF), 0, s, P);
    }
    if (dtype == D3D_DTYPE_F32)
        hipLaunchKernelGGL(support_gather_kernel<kF32>, dim3(C, N), dim3(rows::NT), 0, s, logits, (int)V,
                           temperature, zf, lim, S, kin, counters);
    else
        hipLaunchKernelGGL(support_gather_kernel<kBF16>, dim3(C, N), dim3(rows::NT), 0, s, logits, (int)V,
                           temperature, zf, lim, S, kin, counters);
    err = hipGetLastError();
    if (err != hipSuccess) return (int)err;
    size_t tb = lay.temp_bytes;
    err = rocprim::segmented_radix_sort_keys(ws + lay.temp, tb, kin, kout, (unsigned int)((size_t)N * S),
                                             (unsigned int)N, offsets, offsets + 1, 0, 32 + kIdBits, s, false);
    if (err != hipSuccess) return (int)err;
    hipLaunchKernelGGL(support_draw_kernel, dim3(N), dim3(NTF), 0, s, kout, S, top_p, uniforms, tokens_out,
                       support_ids_out, support_probs_out, token_probs_out);
    err = hipGetLastError();
    return err == hipSuccess ? D3D_OK : (int)err;
}
