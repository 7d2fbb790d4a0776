// Q8_0 shared expert beside routed experts of another format: dense products on
// f16 MFMA (numerics as k_gemm_f16: A split hi + lo, B the int8 value, fp32 sums).
//
// The matrices are small (1 MB of gate and up at 512 x 2048), so what bounds a
// batch is one wave's chain through K. A block is therefore one 16-row block (down:
// two) of one tile of 16 tokens (or of four: launch_dense_q8) with K split over its 4
// waves, superblock by superblock; a superblock's weights (and with one tile its A
// operands) are all loaded before the first is used, and the waves' sums meet in LDS.
// 512 x 2048 at 65 / 130 / 509 tokens, gate/up 12 / 16 / 27 us and down 8 / 10 / 17 (with
// the split of act), against 86 / 86 / 88 and 25 / 26 / 26 on the fp32 GEMM.
#pragma once
#include "moe_kernels.cuh"

namespace ingot {

// GATEUP: act[t][r] = SwiGLU over x as split by the dispatch in column order XORD,
// written in fp32 with each row's maximum raised in rowmax; else out = W act with
// act split by k_split_act (natural order, scaled by rowmax). grid: row blocks x
// tiles of 16 tokens.
template <bool GATEUP, int XORD, int MT>
__global__ __launch_bounds__(256) void k_dense_q8(const uint8_t* __restrict__ w0, const uint8_t* __restrict__ w1,
                                                  uint64_t stride0, uint64_t stride1, uint32_t rows, uint32_t kdim,
                                                  const _Float16* __restrict__ ah, const _Float16* __restrict__ al,
                                                  uint32_t T, float limit, float* __restrict__ out,
                                                  const float* __restrict__ xstat, uint32_t* __restrict__ rowmax) {
    static_assert(XORD != A_IQ4NL, "an order that keeps runs of 8 columns");
    constexpr int NB = 2;
    constexpr uint32_t NW = 4, BR = GATEUP ? 16u : 32u;
    __shared__ float red[NW][MT * NB * 4][64];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, kq = lane >> 4, ln = lane & 15u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t r0 = BR * blockIdx.x, t0 = 16u * MT * blockIdx.y, n = min(16u * MT, T - t0);
    BStream<8, NB, GATEUP, false> B;
    B.init(w0, w1, stride0, stride1, rows, kdim, r0, lane);
    const __amdgpu_buffer_rsrc_t ra_h = make_rsrc(ah, kdim * 2u * T), ra_l = make_rsrc(al, kdim * 2u * T);
    // rows past the tile: an offset past the buffer, which reads zero
    uint32_t arow[MT];
#pragma unroll
    for (uint32_t k = 0; k < MT; ++k) arow[k] = 16u * k + ln < n ? 2u * (t0 + 16u * k + ln) * kdim : 0xffffff00u;
    floatx4 tot[MT][NB];
#pragma unroll
    for (int k = 0; k < MT; ++k)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) tot[k][nb] = floatx4{0.f, 0.f, 0.f, 0.f};
    // A of K steps 2 s, 2 s + 1 (32-column blocks, of which the lane takes columns
    // 8 kq .. + 7) of superblock sb
    struct Frag {
        uint4 h[MT][2], l[MT][2];
    };
    auto load_a = [&](Frag& f, uint32_t sb, uint32_t s) {
#pragma unroll
        for (uint32_t gi = 0; gi < 2; ++gi) {
            const uint32_t o = 2u * a_pos<XORD>(32u * (2u * s + gi) + 8u * kq);
#pragma unroll
            for (uint32_t k = 0; k < MT; ++k) {
                const uint32_t v = 16u * k + ln < n ? arow[k] + o : arow[k];
                f.h[k][gi] = buf_load16(ra_h, v, 512u * sb);
                f.l[k][gi] = buf_load16(ra_l, v, 512u * sb);
            }
        }
    };
    const uint32_t slabs = B.slabs, nsb = (slabs + 3u) >> 2;
    constexpr uint32_t AHEAD = MT == 1 ? 4u : 2u;  // slabs of A in flight
    for (uint32_t sb = wave; sb < nsb; sb += NW) {
        Frag f[AHEAD];
#pragma unroll
        for (uint32_t s = 0; s < 4u; ++s) B.load_slab(s, 4u * sb + s, (s & 1u) == 0u);
#pragma unroll
        for (uint32_t s = 0; s < AHEAD; ++s) load_a(f[s], sb, s);
#pragma unroll
        for (uint32_t s = 0; s < 4u; ++s) {
            half8 fb[NB][2], fe[NB][2];
            float dg[NB][2];
            typename BStream<8, NB, GATEUP, false>::SbState st;
            if ((s & 1u) == 0u) B.take_pair(s);
            B.decode(st, s, B.nq[s], B.nd[s], fb, dg, fe);
            // (slabs past K: clamped weights over columns past it, not added)
            const bool live = 4u * sb + s < slabs;
#pragma unroll
            for (uint32_t gi = 0; gi < 2; ++gi)
#pragma unroll
                for (uint32_t k = 0; k < MT; ++k) {
                    const half8 a0 = __builtin_bit_cast(half8, f[s % AHEAD].h[k][gi]);
                    const half8 a1 = __builtin_bit_cast(half8, f[s % AHEAD].l[k][gi]);
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb) {
                        floatx4 p =
                            __builtin_amdgcn_mfma_f32_16x16x32_f16(a0, fb[nb][gi], floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                        p = __builtin_amdgcn_mfma_f32_16x16x32_f16(a1, fb[nb][gi], p, 0, 0, 0);
                        if (live) {
#pragma unroll
                            for (int j = 0; j < 4; ++j) tot[k][nb][j] += dg[nb][gi] * p[j];
                        }
                    }
                }
            if (s + AHEAD < 4u) load_a(f[s % AHEAD], sb, s + AHEAD);
        }
    }
#pragma unroll
    for (int k = 0; k < MT; ++k)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int j = 0; j < 4; ++j) red[wave][4 * (NB * k + nb) + j][lane] = tot[k][nb][j];
    __syncthreads();
    // thread -> token m of each tile, column c of the block: lane 16 (m / 4) + c held it
    // in value m % 4
    const uint32_t m = tid >> 4, c = tid & 15u, l = 16u * (m >> 2) + c, j = m & 3u;
#pragma unroll
    for (uint32_t k = 0; k < MT; ++k) {
        const bool live = 16u * k + m < n;
        const uint32_t t = t0 + (live ? 16u * k + m : 0u);
        float v[NB];
#pragma unroll
        for (uint32_t nb = 0; nb < NB; ++nb) {
            const uint32_t i = 4u * (NB * k + nb) + j;
            v[nb] = (red[0][i][l] + red[1][i][l]) + (red[2][i][l] + red[3][i][l]);
        }
        if constexpr (GATEUP) {
            const int e = x_exp(ld_xstat(xstat, t).x);
            const float s = swiglu(ldexpf(v[0], -e), ldexpf(v[1], -e), limit);
            if (live) out[(uint64_t)t * rows + r0 + c] = s;
            const uint32_t rm = row_max16(__float_as_uint(fabsf(s)));
            if (live && c == 0u) atomicMax(rowmax + t, rm);
        } else if (live) {
            const int e = x_exp(__uint_as_float(rowmax[t]));
#pragma unroll
            for (uint32_t nb = 0; nb < NB; ++nb) out[(uint64_t)t * rows + r0 + 16u * nb + c] = ldexpf(v[nb], -e);
        }
    }
}

}  // namespace ingot
