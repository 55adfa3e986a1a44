// The gate-up projection of a block of at most 192 rows and its SiLU-mul in
// one launch, on the weight-streaming kernel of gemm.hip (SILU form).
#include "gemm_rows.hpp"
#include "../../include/d3d_hip.h"

namespace d3d {
namespace gemm {
namespace {

struct SiluCall {
    const uint16_t *x, *w;
    uint16_t* y;
    int M, H, K;
    hipStream_t s;
};

template <int MR, int TN, int NW, int WC, int TK, int P, int STEPS>
void launch(const SiluCall& c) {
    hipLaunchKernelGGL((rows_kernel<MR, TN, NW, WC, TK, P, STEPS, true>), dim3(2 * c.H / TN), dim3(NW * kWave), 0, c.s,
                       c.x, c.w, c.y, nullptr, c.M, 2 * c.H, c.K, c.K);
}

// K / 128 in {8, 16, 24, 32, 48, 64}; false otherwise.
template <int MR, int TN, int NW, int WC, int TK>
bool launch_steps(const SiluCall& c) {
    constexpr int F = 128 / TK;
    switch (c.K / 128) {
        case 8: launch<MR, TN, NW, WC, TK, 2, 8 * F>(c); return true;
        case 16: launch<MR, TN, NW, WC, TK, 2, 16 * F>(c); return true;
        case 24: launch<MR, TN, NW, WC, TK, 2, 24 * F>(c); return true;
        case 32: launch<MR, TN, NW, WC, TK, 2, 32 * F>(c); return true;
        case 48: launch<MR, TN, NW, WC, TK, 2, 48 * F>(c); return true;
        case 64: launch<MR, TN, NW, WC, TK, 2, 64 * F>(c); return true;
    }
    return false;
}

// Column tiles of 64 while they make at most one round of 256 workgroups, or
// up to 32 rows, where a workgroup takes little of a CU; else of 96 where
// those make a round, or of 128: fewer workgroups read X.  Target gate-up,
// 24576 x 4096 (30 us at the rate of a plain read), tiles of 64 / 96 / 128, us: 64 rows
// 51.5 / 43.7 / 46.5 (hipBLASLt 49.5 and a SiLU-mul of 5), 128 rows 67.2 /
// 50.6 / 57.0 (52.9), 192 rows 80.3 / 63.6 / 60.9 (60.4); 16 rows 43.1 with 64.
int column_tile(int M, int H) {
    if (M <= 32 || H / 32 <= 256) return 64;
    if (M <= 128 && H % 48 == 0 && H / 48 <= 256) return 96;
    return H % 64 == 0 ? 128 : 64;
}

int run(const SiluCall& c) {
    bool done = false;
    const int tn = column_tile(c.M, c.H);
    if (c.M <= 16) done = launch_steps<16, 64, 4, 4, 128>(c);
    else if (c.M <= 32) done = launch_steps<32, 64, 4, 4, 128>(c);
    else if (c.M <= 64)
        done = tn == 96    ? launch_steps<64, 96, 8, 2, 128>(c)
               : tn == 128 ? launch_steps<64, 128, 8, 4, 128>(c)
                           : launch_steps<64, 64, 4, 4, 128>(c);
    else if (c.M <= 128)
        done = tn == 96    ? launch_steps<128, 96, 4, 2, 64>(c)
               : tn == 128 ? launch_steps<128, 128, 8, 4, 64>(c)
                           : launch_steps<128, 64, 8, 2, 64>(c);
    else
        done = tn == 128 ? launch_steps<192, 128, 8, 4, 64>(c) : launch_steps<192, 64, 8, 2, 64>(c);
    if (!done) return D3D_E_UNSUPPORTED;
    const hipError_t err = hipGetLastError();
    return err == hipSuccess ? D3D_OK : (int)err;
}

int check_and_run(const void* x, const void* w, void* y, int M, int max_rows, int H, int K, void* stream) {
    if (M < 1 || M > max_rows || H < 32 || H % 32 || K < 128 || K % 128) return D3D_E_SHAPE;
    if (!x || !w || !y) return D3D_E_NULL;
    if (reinterpret_cast<uintptr_t>(x) % 16 || reinterpret_cast<uintptr_t>(w) % 16) return D3D_E_UNSUPPORTED;
    return run(SiluCall{static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(w), static_cast<uint16_t*>(y), M, H,
                        K, static_cast<hipStream_t>(stream)});
}

}  // namespace
}  // namespace gemm
}  // namespace d3d

using namespace d3d;

extern "C" int d3d_gemm_rows64_silu_mul(const void* x, const void* w_gate_up, void* y, int M, int H, int K,
                                        void* stream) {
    return gemm::check_and_run(x, w_gate_up, y, M, 64, H, K, stream);
}

extern "C" int d3d_gemm_rows192_silu_mul(const void* x, const void* w_gate_up, void* y, int M, int H, int K,
                                         void* stream) {
    return gemm::check_and_run(x, w_gate_up, y, M, gemm::kMaxRows, H, K, stream);
}
