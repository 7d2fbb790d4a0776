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
    // Four tiles per block (weights read and decoded a quarter as often, but one block
    // per CU) where those blocks fill the rounds they take of the 256 CUs to 85 %, else one (three per
    // CU). Gate/up stage us, one against four: 512 x 2048 at 400 / 509 / 640 tokens (224,
    // 256, 320 blocks of four) 57 / 63 / 72 against 52 / 58 / 83; 1408 x 4096 at 256 / 509
    // (352, 704) 123 / 203 against 129 / 191; down at H = 2048, K = 1024, 256 / 320 (256,
    // 320) 30 / 32 against 27 / 37.
    const uint32_t br = gateup ? 16u : 32u, b4 = rows / br * ((T + 63u) / 64u);
    const uint32_t mt = 100u * b4 >= 85u * 256u * ((b4 + 255u) / 256u) ? 4u : 1u;
    const dim3 grid(rows / br, (T + 16u * mt - 1u) / (16u * mt));
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
