// Weight-streaming GEMM for blocks of at most 192 rows:  Y[M, N] = X[M, K] W[N, K]^T
// (bf16 in, fp32 accumulation), the projections of a verify or draft block of
// up to twelve requests (serving/vendor/ssd/layers/linear.py: F.linear on bf16
// weights).
//
// Each weight is read once, each activation once per column tile, so the
// kernel is built to stream W:
//
// * Workgroup (column tile of TN, K split s); each k step moves a TN x TK tile
//   of W and the MR x TK tile of X (MR: M rounded up to 16, 32, 64, 128 or
//   192).  Every wave instruction reads whole 128- or 256-byte row segments
//   (16 bytes per lane), the order that streams the weights fastest of those
//   measured.  Within a row the 16-byte chunk q is stored at slot q ^ (row & 7)
//   of LDS, so the MFMA operand reads of 16 consecutive rows spread over the
//   banks.
// * Register-staged pipeline (rows_kernel): the loads of the next P k steps
//   are in flight in registers while a step is stored to one of two LDS
//   buffers and multiplied from it, one barrier per step.  The k loop is
//   unrolled for the step counts the models use (STEPS), so the compiler's
//   wait before each store counts exactly the loads issued after it; as a
//   loop, with a wait for every load at its head, it ran 5-12 % longer.
//   Other step counts of up to 64 rows run on gemm_rows64_dma_kernel (direct
//   global -> LDS loads, two stages, two barriers per step).
// * The tile per row count (us, graph-replayed on HBM-resident weights; the
//   weights alone take 7.5 / 5.0 / 15.0 us for the target's qkv / o / down, 2.5
//   / 1.3 / 3.8 for the draft's, at the 6.7 TB/s that a plain read of 4 GiB
//   reaches -- a copy moves 4.9 and bounds no read):
//     M <= 16, 32: four waves, TK 128.  In the 64-row kernel three quarters
//       of the X loads, LDS traffic and MFMAs were repeats of the last row.
//       16 rows: target 12.9 / 8.3 / 19.7 -> 11.5 / 7.5 / 18.7, draft
//       5.9 / 4.3 / 7.3 -> 5.0 / 3.8 / 6.3.
//     M <= 64: four waves; TK 64 and three stages in flight below 2^24
//       weights, TK 128 and two from there: draft 7.3 / 5.6 / 8.9 with the
//       latter, 6.8 / 5.6 / 8.4 with the former; target 15.4 / 10.0 / 22.4
//       and 15.6 / 9.6 / 22.6 alone, but beside the packed prediction on the
//       other stream the verify forward takes 8.40 ms with TK 128 and 8.84
//       with TK 64 (engine loop 90.7 against 88.7 steps/s).
//     M <= 128, 192: eight waves, TK 64, two stages (hipBLASLt before).
//       128 rows: target 25.7 / 24.4 / 67.4 -> 19.7 / 12.3 / 29.8, draft
//       14.7 / 11.2 / 17.8 -> 8.6 / 6.9 / 10.9; 192 rows: target
//       34.4 / 33.2 / 90.8 -> 24.3 / 15.4 / 37.0, draft 21.4 / 11.9 / 22.6 ->
//       10.7 / 8.4 / 13.4.  Every workgroup reads the whole X of its k range
//       through L2, which is what grows with M: four waves with TK 128 took
//       22.8 / 15.3 / 34.9 at 128 rows (one wave per SIMD, nothing beside its
//       LDS reads), column tiles of 128 halve that traffic but leave half the
//       CUs idle at these splits (25.4 / 16.0 / 38.9).
// * The waves split the tile (WR rows of waves x WC columns) and multiply
//   with v_mfma_f32_16x16x32_bf16, both operands read from LDS.  The sum over
//   k of an entry runs in the same order in every variant.
// * Small N leaves too few column tiles to fill 256 CUs, so K is split over
//   `splits` workgroups per tile (d3d_gemm_rows64_splits picks the count).
//   With one split the result is rounded to bf16 into Y; with several,
//   each split writes its fp32 partial [splits][M][N] and the consumer of
//   the product sums the splits in order (d3d_add_rmsnorm_parts,
//   d3d_qk_rope_append_parts) -- no extra launch, no atomics, and the sum
//   has the same bits on every call.
#include "d3d_common.hpp"
#include "gemm_rows.hpp"
#include "../../include/d3d_hip.h"

namespace d3d {
namespace gemm {

// gemm_rows64_dma_kernel's tiles.
constexpr int NT = 256;                  // four waves
constexpr int TN = 64;                   // output columns per workgroup
constexpr int TK = 128;                  // k per stage
constexpr int ST = 2;                    // stages
constexpr int ROWB = TK * 2;             // bytes of one tile row
constexpr int CPR = ROWB / 16;           // 16-byte chunks per tile row
constexpr int TILEB = 64 * ROWB;         // one 64-row tile (W or X), 16 KB
constexpr int STAGEB = 2 * TILEB;        // W tile, then X tile
constexpr int RPI = kWave / CPR;         // tile rows per wave instruction
constexpr int LPW = TILEB / 1024 / 4;    // load instructions per wave per tile
constexpr int kMaxSplits = 16;
static_assert(ST * STAGEB <= 64 * 1024, "LDS per workgroup");

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// One k step from an LDS stage (W tile, then X tile): wave wv multiplies the
// 64 rows of X by columns 16 wv .. 16 wv + 15 of the tile.
__device__ __forceinline__ void mma_step(const char* cur, f32x4 (&acc)[4], int wv, int c16, int g4) {
    const int rB = 16 * wv + c16;
#pragma unroll
    for (int ks = 0; ks < TK / 32; ++ks) {
        const int q = 4 * ks + g4;
        const u32x4 bw = *reinterpret_cast<const u32x4*>(cur + rB * ROWB + 16 * (q ^ (rB & 7)));
        u32x4 ax[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int m = 16 * t + c16;
            ax[t] = *reinterpret_cast<const u32x4*>(cur + TILEB + m * ROWB + 16 * (q ^ (m & 7)));
        }
#pragma unroll
        for (int t = 0; t < 4; ++t)
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, ax[t]),
                                                             __builtin_bit_cast(bf16x8, bw), acc[t], 0, 0, 0);
    }
}

// Lane (c16, g4) holds rows 16t + 4 g4 + r of column n: bf16 into Y (one
// split) or the fp32 partial of split blockIdx.y.
__device__ __forceinline__ void store_tile(const f32x4 (&acc)[4], uint16_t* y, float* parts, int M, int N, int n,
                                           int g4) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = 16 * t + 4 * g4 + r;
            if (m < M) {
                if (gridDim.y == 1)
                    y[(size_t)m * N + n] = f32_to_bf16_bits(acc[t][r]);
                else
                    parts[((size_t)blockIdx.y * M + m) * N + n] = acc[t][r];
            }
        }
}

// Direct global -> LDS form (global_load_lds, two stages): the kernel for
// step counts rows_kernel is not unrolled for.
__global__ __launch_bounds__(NT) void gemm_rows64_dma_kernel(const uint16_t* __restrict__ x,
                                                         const uint16_t* __restrict__ w,
                                                         uint16_t* __restrict__ y, float* __restrict__ parts,
                                                         int M, int N, int K, int KR) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    const int c16 = lane & 15, g4 = lane >> 4;
    const int n0 = blockIdx.x * TN;
    const int kb = blockIdx.y * KR;
    const int steps = KR / TK;
    // This lane's source rows and LDS rows: wave wv fills rows
    // (wv * LPW + j) * RPI + lane / CPR of both tiles, chunk lane % CPR
    // read from global chunk (lane % CPR) ^ (row & 7).
    const int lr = lane / CPR, lc = lane % CPR;
    const uint16_t* wsrc[LPW];
    const uint16_t* xsrc[LPW];
    int lofs[LPW];
#pragma unroll
    for (int j = 0; j < LPW; ++j) {
        const int rb = (wv * LPW + j) * RPI, r = rb + lr;
        const int q = lc ^ (r & 7);
        wsrc[j] = w + (size_t)(n0 + r) * K + kb + 8 * q;
        xsrc[j] = x + (size_t)min(r, M - 1) * K + kb + 8 * q;
        lofs[j] = rb * ROWB;
    }
    f32x4 acc[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t] = {0.f, 0.f, 0.f, 0.f};
    // Stage 0 in flight before the loop; each iteration issues the next
    // stage, waits for the current one (its own loads, then the barrier for
    // everyone's), multiplies it, and frees it with a second barrier.
#pragma unroll
    for (int j = 0; j < LPW; ++j) {
        __builtin_amdgcn_global_load_lds(wsrc[j], smem + lofs[j], 16, 0, 0);
        __builtin_amdgcn_global_load_lds(xsrc[j], smem + TILEB + lofs[j], 16, 0, 0);
    }
    for (int step = 0; step < steps; ++step) {
        if (step + 1 < steps) {
            char* nxt = smem + ((step + 1) % ST) * STAGEB;
            const int ko = (step + 1) * TK;
#pragma unroll
            for (int j = 0; j < LPW; ++j) {
                __builtin_amdgcn_global_load_lds(wsrc[j] + ko, nxt + lofs[j], 16, 0, 0);
                __builtin_amdgcn_global_load_lds(xsrc[j] + ko, nxt + TILEB + lofs[j], 16, 0, 0);
            }
            wait_vmcnt<2 * LPW>();
        } else {
            wait_vmcnt<0>();
        }
        __syncthreads();
        mma_step(smem + (step % ST) * STAGEB, acc, wv, c16, g4);
        __syncthreads();
    }
    store_tile(acc, y, parts, M, N, n0 + 16 * wv + c16, g4);
}

}  // namespace gemm
}  // namespace d3d

using namespace d3d;

extern "C" int d3d_gemm_rows64_splits(int N, int K) {
    if (N < gemm::TN || N % gemm::TN || K < gemm::TK || K % gemm::TK) return 1;
    // The most splits whose grid is at most one workgroup per CU (256),
    // leaving every split at least two k steps, and -- below K = 8192, where
    // more splits buy less -- at most 16,384 partial floats per output row:
    // the consumer of the product reads every partial back, about 1 us per
    // 4 MB at 64 rows.  Measured with that consumer (d3d_add_rmsnorm_parts)
    // on rotating HBM-resident weights: 4096 x 12288 at 4 splits 27.6 us
    // against 31.2 at 8 (a full round of two per CU), 4096 x 4096 at 4
    // splits 14.9 against 17.9 at 8, 2048 x 6144 at 8 splits 13.8 against
    // 15.4 at 4 and 16.6 at 16.
    const int tiles = N / gemm::TN;
    int s = 1;
    while (s < gemm::kMaxSplits && tiles * 2 * s <= 256 && K % (gemm::TK * 2 * s) == 0 &&
           K / (2 * s) >= 2 * gemm::TK && (K >= 8192 || (int64_t)2 * s * N <= 16384))
        s *= 2;
    return s;
}

namespace {

struct Call {
    const uint16_t *x, *w;
    uint16_t* y;
    float* parts;
    int M, N, K, splits;
    hipStream_t s;
};

template <int MR, int TN, int NW, int WC, int TK, int P, int STEPS>
void launch(const Call& c) {
    hipLaunchKernelGGL((gemm::rows_kernel<MR, TN, NW, WC, TK, P, STEPS, false>), dim3(c.N / TN, c.splits),
                       dim3(NW * kWave), 0, c.s, c.x, c.w, c.y, c.parts, c.M, c.N, c.K, c.K / c.splits);
}

// Launches the variant built for this step count (steps of 128); false if
// there is none.
template <int MR, int TN, int NW, int WC, int TK, int P>
bool launch_steps(const Call& c) {
    constexpr int F = gemm::TK / TK;
    switch (c.K / c.splits / gemm::TK) {
        case 2: launch<MR, TN, NW, WC, TK, P, 2 * F>(c); return true;
        case 4: launch<MR, TN, NW, WC, TK, P, 4 * F>(c); return true;
        case 6: launch<MR, TN, NW, WC, TK, P, 6 * F>(c); return true;
        case 8: launch<MR, TN, NW, WC, TK, P, 8 * F>(c); return true;
        case 12: launch<MR, TN, NW, WC, TK, P, 12 * F>(c); return true;
        case 16: launch<MR, TN, NW, WC, TK, P, 16 * F>(c); return true;
        case 24: launch<MR, TN, NW, WC, TK, P, 24 * F>(c); return true;
        case 32: launch<MR, TN, NW, WC, TK, P, 32 * F>(c); return true;
    }
    if constexpr (MR <= 64) {
        switch (c.K / c.splits / gemm::TK) {
            case 1: launch<MR, TN, NW, WC, TK, P, F>(c); return true;
            case 3: launch<MR, TN, NW, WC, TK, P, 3 * F>(c); return true;
        }
    }
    return false;
}

int check(const void* x, const void* w, const void* y, const float* parts, int M, int max_rows, int N, int K,
          int splits) {
    if (M < 1 || M > max_rows || N < gemm::TN || N % gemm::TN || K < gemm::TK) return D3D_E_SHAPE;
    if (splits < 1 || splits > gemm::kMaxSplits || K % (gemm::TK * splits)) return D3D_E_SHAPE;
    if (!x || !w || (splits == 1 ? !y : !parts)) return D3D_E_NULL;
    if (reinterpret_cast<uintptr_t>(x) % 16 || reinterpret_cast<uintptr_t>(w) % 16) return D3D_E_UNSUPPORTED;
    return D3D_OK;
}

}  // namespace

extern "C" int d3d_gemm_rows64(const void* x, const void* w, void* y, float* parts, int M, int N, int K,
                               int splits, void* stream) {
    const int st = check(x, w, y, parts, M, 64, N, K, splits);
    if (st != D3D_OK) return st;
    const Call c{static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(w), static_cast<uint16_t*>(y), parts,
                 M, N, K, splits, static_cast<hipStream_t>(stream)};
    // An LM head's many rounds of workgroups take column tiles of 128 from 33
    // rows (half the reads of X; 64 rows of 151,936 x 2048: 140.6 -> 133 us).
    const bool wide = splits == 1 && N % 128 == 0 && N / 128 >= 1024;
    const bool done = M <= 16   ? launch_steps<16, 64, 4, 4, 128, 2>(c)
                      : M <= 32 ? launch_steps<32, 64, 4, 4, 128, 2>(c)
                      : wide    ? launch_steps<64, 128, 4, 4, 64, 2>(c)
                      : (int64_t)N * K < (1 << 24) ? launch_steps<64, 64, 4, 4, 64, 3>(c)
                                                   : launch_steps<64, 64, 4, 4, 128, 2>(c);
    if (!done)
        hipLaunchKernelGGL(gemm::gemm_rows64_dma_kernel, dim3(N / gemm::TN, splits), dim3(gemm::NT),
                           gemm::ST * gemm::STAGEB, c.s, c.x, c.w, c.y, parts, M, N, K, K / splits);
    const hipError_t err = hipGetLastError();
    return err == hipSuccess ? D3D_OK : (int)err;
}

extern "C" int d3d_gemm_rows192(const void* x, const void* w, void* y, float* parts, int M, int N, int K, int splits,
                                void* stream) {
    if (M <= 64) return d3d_gemm_rows64(x, w, y, parts, M, N, K, splits, stream);
    const int st = check(x, w, y, parts, M, gemm::kMaxRows, N, K, splits);
    if (st != D3D_OK) return st;
    const Call c{static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(w), static_cast<uint16_t*>(y), parts,
                 M, N, K, splits, static_cast<hipStream_t>(stream)};
    if (!(M <= 128 ? launch_steps<128, 64, 8, 2, 64, 2>(c) : launch_steps<192, 64, 8, 2, 64, 2>(c)))
        return D3D_E_UNSUPPORTED;
    const hipError_t err = hipGetLastError();
    return err == hipSuccess ? D3D_OK : (int)err;
}
