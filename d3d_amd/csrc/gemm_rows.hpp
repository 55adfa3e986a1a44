// The register-staged weight-streaming GEMM kernel of gemm.hip (which says
// why it looks like this), shared with gemm_silu.hip.
#pragma once

#include "d3d_common.hpp"

namespace d3d {
namespace gemm {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Rows the kernels take in all.
constexpr int kMaxRows = 192;

// Bytes of LDS the main loop needs.
template <int MR, int TN, int TK>
constexpr int rows_lds() { return 2 * (TN + MR) * TK * 2; }

// The main loop of a workgroup of NW waves (WC of them across the tile's TN
// columns): acc[a][b] += X[rows, kb ..] W[wrow(0 .. TN - 1), kb ..]^T over STEPS
// k steps of TK, P of them in flight in registers.  Wave wv holds rows ar0 +
// 16a, columns bc0 + 16b, with ar0 = (wv / WC) (MR / WR), bc0 = (wv % WC) (TN / WC).
// The lane's source rows and LDS slots: global 16-byte chunk (lane % chunks) ^
// (row & 7) of a tile row goes to LDS chunk lane % chunks.  Rows of X past M
// repeat the last one.
template <int MR, int TN, int NW, int WC, int TK, int P, int STEPS, typename WRow>
__device__ __forceinline__ void rows_main_loop(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, int M,
                                               int K, int kb, char* smem, WRow&& wrow,
                                               f32x4 (&acc)[MR * WC / NW / 16][TN / WC / 16]) {
    constexpr int RB = TK * 2, CPRW = RB / 16, RPIW = kWave / CPRW;  // bytes, 16-byte chunks of a tile row
    constexpr int WT = TN * RB, XT = MR * RB, STAGE = WT + XT;
    constexpr int NWL = WT / 1024 / NW, NXL = XT / 1024 / NW;  // load instructions per wave
    constexpr int WR = NW / WC, AR = MR / WR / 16, BC = TN / WC / 16;
    static_assert(AR * WR * 16 == MR && BC * WC * 16 == TN && NWL * NW * 1024 == WT && NXL * NW * 1024 == XT, "tile");
    const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    const int c16 = lane & 15, g4 = lane >> 4;
    const int lr = lane / CPRW, lc = lane % CPRW;
    const uint16_t* wsrc[NWL];
    const uint16_t* xsrc[NXL];
    int wofs[NWL], xofs[NXL];
#pragma unroll
    for (int j = 0; j < NWL; ++j) {
        const int r = (wv * NWL + j) * RPIW + lr, q = lc ^ (r & 7);
        wsrc[j] = w + (size_t)wrow(r) * K + kb + 8 * q;
        wofs[j] = r * RB + lc * 16;
    }
#pragma unroll
    for (int j = 0; j < NXL; ++j) {
        const int r = (wv * NXL + j) * RPIW + lr, q = lc ^ (r & 7);
        xsrc[j] = x + (size_t)min(r, M - 1) * K + kb + 8 * q;
        xofs[j] = WT + r * RB + lc * 16;
    }
    u32x4 rw[P][NWL], rx[P][NXL];
    auto load = [&](int st, int sl) {
#pragma unroll
        for (int j = 0; j < NWL; ++j)
            rw[sl][j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wsrc[j] + st * TK));
#pragma unroll
        for (int j = 0; j < NXL; ++j) rx[sl][j] = *reinterpret_cast<const u32x4*>(xsrc[j] + st * TK);
    };
#pragma unroll
    for (int a = 0; a < AR; ++a)
#pragma unroll
        for (int b = 0; b < BC; ++b) acc[a][b] = {0.f, 0.f, 0.f, 0.f};
    const int ar0 = (wv / WC) * (MR / WR), bc0 = (wv % WC) * (TN / WC);
#pragma unroll
    for (int p = 0; p < P; ++p)
        if (p < STEPS) load(p, p);
#pragma unroll
    for (int st = 0; st < STEPS; ++st) {
        // Buffer st % 2 was last read in step st - 2, which every wave
        // finished before the barrier of step st - 1.
        char* buf = smem + (st & 1) * STAGE;
#pragma unroll
        for (int j = 0; j < NWL; ++j) *reinterpret_cast<u32x4*>(buf + wofs[j]) = rw[st % P][j];
#pragma unroll
        for (int j = 0; j < NXL; ++j) *reinterpret_cast<u32x4*>(buf + xofs[j]) = rx[st % P][j];
        if (st + P < STEPS) load(st + P, st % P);
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < TK / 32; ++ks) {
            const int q = 4 * ks + g4;
            u32x4 bw[BC], ax[AR];
#pragma unroll
            for (int b = 0; b < BC; ++b) {
                const int r = bc0 + 16 * b + c16;
                bw[b] = *reinterpret_cast<const u32x4*>(buf + r * RB + 16 * (q ^ (r & 7)));
            }
#pragma unroll
            for (int a = 0; a < AR; ++a) {
                const int r = ar0 + 16 * a + c16;
                ax[a] = *reinterpret_cast<const u32x4*>(buf + WT + r * RB + 16 * (q ^ (r & 7)));
            }
#pragma unroll
            for (int a = 0; a < AR; ++a)
#pragma unroll
                for (int b = 0; b < BC; ++b)
                    acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        __builtin_bit_cast(bf16x8, ax[a]), __builtin_bit_cast(bf16x8, bw[b]), acc[a][b], 0, 0, 0);
        }
    }
}

// SILU: W is a gate-up weight [2 H, K] (gate rows, then up rows) and Y
// [M, H] = silu(bf16(X Wg^T)) * bf16(X Wu^T), each product rounded as the
// bf16 GEMM output would be, then evaluated as d3d_silu_mul does.  Tile t
// stands for output columns TN/2 t .. TN/2 t + TN/2 - 1: tile row 16 w + c is
// the gate row of column TN/2 t + 8 w + c (c < 8) or the up row of column
// TN/2 t + 8 w + c - 8, so a lane's gate and up products of one column sit in
// lanes c and c + 8 of its 16-lane row.
template <int MR, int TN, int NW, int WC, int TK, int P, int STEPS, bool SILU>
__global__ __launch_bounds__(NW * kWave) void rows_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
                                                          uint16_t* __restrict__ y, float* __restrict__ parts, int M,
                                                          int N, int K, int KR) {
    constexpr int WR = NW / WC, AR = MR / WR / 16, BC = TN / WC / 16;
    __shared__ __attribute__((aligned(16))) char smem[rows_lds<MR, TN, TK>()];
    const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    const int c16 = lane & 15, g4 = lane >> 4;
    const int n0 = blockIdx.x * TN, ar0 = (wv / WC) * (MR / WR), bc0 = (wv % WC) * (TN / WC);
    f32x4 acc[AR][BC];
    rows_main_loop<MR, TN, NW, WC, TK, P, STEPS>(
        x, w, M, K, (int)blockIdx.y * KR, smem,
        [&](int r) {
            if constexpr (!SILU) return n0 + r;
            const int col = TN / 2 * (int)blockIdx.x + 8 * (r >> 4) + (r & 7);
            return (r & 8) ? N / 2 + col : col;
        },
        acc);
    // Lane (c16, g4) holds rows 16a + 4 g4 + r of column 16b + c16: bf16 into
    // Y (one split) or the fp32 partial of split blockIdx.y.
#pragma unroll
    for (int a = 0; a < AR; ++a)
#pragma unroll
        for (int b = 0; b < BC; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = ar0 + 16 * a + 4 * g4 + r;
                if constexpr (SILU) {
                    const float mine = acc[a][b][r], other = __shfl_xor(mine, 8, kWave);
                    const int H = N / 2, col = TN / 2 * blockIdx.x + 8 * (bc0 / 16 + b) + (c16 & 7);
                    if (c16 < 8 && m < M) {
                        const float gv = bf16_bits_to_f32(f32_to_bf16_bits(mine));
                        const float uv = bf16_bits_to_f32(f32_to_bf16_bits(other));
                        y[(size_t)m * H + col] = __builtin_bit_cast(uint16_t, (__bf16)(gv / (1.0f + expf(-gv)) * uv));
                    }
                } else {
                    const int n = n0 + bc0 + 16 * b + c16;
                    if (m < M) {
                        if (gridDim.y == 1) y[(size_t)m * N + n] = f32_to_bf16_bits(acc[a][b][r]);
                        else parts[((size_t)blockIdx.y * M + m) * N + n] = acc[a][b][r];
                    }
                }
            }
}

}  // namespace gemm
}  // namespace d3d
