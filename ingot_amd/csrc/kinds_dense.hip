// Per-format kernels (see kind_launch.h): GGML types 0 1 8 30.
#include "kind_launch.cuh"

#include "dense_q8.cuh"

INGOT_INSTANTIATE_KIND(0)
INGOT_INSTANTIATE_KIND(1)
INGOT_INSTANTIATE_KIND(8)
INGOT_INSTANTIATE_KIND(30)
INGOT_INSTANTIATE_FUSED(8, 8)
INGOT_INSTANTIATE_F16(8)

namespace ingot {

void launch_dense_q8(hipStream_t s, bool gateup, int xord, const uint8_t* w0, const uint8_t* w1, uint64_t stride0,
                     uint64_t stride1, uint32_t rows, uint32_t kdim, const _Float16* ah, const _Float16* al, uint32_t T,
                     float limit, float* out, const float* xstat, uint32_t* rowmax) {
    // One tile per block (more blocks) up to 256 tokens, four above (weights read and
    // decoded a quarter as often): 512 x 2048 gate/up us, one against four, 17 / 30 at
    // 100 and 130 tokens, 52 / 39 at 509.
    const uint32_t mt = T <= 256u ? 1u : 4u;
    const dim3 grid(rows / (gateup ? 16u : 32u), (T + 16u * mt - 1u) / (16u * mt));
#define DQ_(GU, XO, MT)                                                                                       \
    hipLaunchKernelGGL((k_dense_q8<GU, XO, MT>), grid, dim3(256), 0, s, w0, w1, stride0, stride1, rows, kdim, \
                       ah, al, T, limit, out, xstat, rowmax)
#define DQ(GU, XO)                    \
    do {                              \
        if (mt == 1u) DQ_(GU, XO, 1); \
        else DQ_(GU, XO, 4);          \
    } while (0)
    if (!gateup) DQ(false, A_NATURAL);
    else if (xord == A_IQ3XXS) DQ(true, A_IQ3XXS);
    else if (xord == A_Q6K) DQ(true, A_Q6K);
    else DQ(true, A_NATURAL);
#undef DQ
#undef DQ_
}

}  // namespace ingot
