// Grouped GEMM on f16 MFMA for batches with a few pairs per expert (decode
// batches, small prompt blocks), over tiles of at most TMS = 16 pairs. Included by the kinds_*.hip units.
//
// Same numerics as k_gemm_f16 (x and act split into f16 hi + lo, weights as
// exact f16 integers, fp32 sums), for the case in which a tile's cost is its
// weights: reading them from HBM and decoding them. What bounds k_gemm_f16
// there is stalls: 2 waves per SIMD, a barrier and an A DMA per 64 columns.
// Here
//   * a block is 4 waves over 64 act columns (gate/up: 16 gate and the same 16
//     up rows per wave) or 128 down rows (32 per wave). From the tiled copies
//     four blocks fit a CU (at most 128 VGPRs, 33 to 40 KB of LDS), three for
//     Q8_0 and Q6_K (up to 142 VGPRs) and IQ2_S (45 KB); in GGUF order three of
//     those that need more than 128 VGPRs, two of Q6_K. Each wave keeps four
//     slabs of its weights in flight;
//   * A is staged in LDS in chunks of 16 KB (two buffers, one barrier per
//     chunk): tiles of at most 8 pairs hold their hi rows in MFMA rows 0..7 and
//     the lo rows in rows 8..15 of ONE operand (512 columns per chunk), so each
//     decoded B fragment feeds one MFMA instead of two and the halves meet in
//     the epilogue; tiles of 9..16 pairs hold hi and lo operands of 16 rows
//     (256 columns per chunk; a superblock each measured 3 % slower packed);
//   * each superblock is summed from zero and then added to the total times its
//     unit (one fma per value), which needs no reciprocal of the next unit.
// Gate/up + down, k_gemm_f16 against this kernel: a Qwen3-30B-A3B-shaped layer
// (Q4_K / Q6_K) at 32 tokens 109 -> 88 us (4.0 TB/s of weights in gate/up), the
// GLM-shaped IQ3_XXS / IQ4_NL layer at 64 tokens 266 -> 227 us. By counters, gate/up
// of the first then issues VALU instructions in 40 % of its SIMD cycles and its waves
// spend 47 % of theirs waiting for loads and the barrier; in the second's LDS bank
// conflicts, nearly all of the codebook reads, take 43 % of a CU's cycles.
#pragma once
#include "moe_kernels.cuh"

namespace ingot {

template <int KIND, bool GATEUP, int AORD, bool TL>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(!TL ? 2 : KIND == 8 || KIND == 14 ? 3 : 4))) void k_gemm_small(
    const uint8_t* __restrict__ w0, const uint8_t* __restrict__ w1, const uint8_t* __restrict__ ws0,
    const uint8_t* __restrict__ ws1, uint32_t e_shared, uint64_t stride0, uint64_t stride1, uint32_t rows_per_expert,
    uint32_t kdim, const _Float16* __restrict__ ah, const _Float16* __restrict__ al, const float* __restrict__ gs,
    const uint32_t* __restrict__ pairs, uint32_t K, const uint32_t* __restrict__ tiles, uint32_t ldo, float limit,
    float* __restrict__ out, _Float16* __restrict__ out_h, _Float16* __restrict__ out_l, float* __restrict__ out_gs,
    uint32_t nblk, uint32_t a_rows, const float* __restrict__ xstat, uint32_t* __restrict__ rowmax,
    uint32_t* __restrict__ flags, const uint32_t* __restrict__ slot_of, uint32_t flat) {
    static_assert(AORD == A_NATURAL || GATEUP, "the permuted act layout is written by the gate/up kernel");
    constexpr int NB = 2;
    constexpr uint32_t NW = 4;
    using BS = BStream<KIND, NB, GATEUP, TL>;
    constexpr bool Q4K = BS::Q4K, IQG = BS::IQG, IQN = BS::IQN, Q6K = BS::Q6K, Q8 = BS::Q8;
    static_assert(!Q8 || !GATEUP || AORD == A_F32, "Q8_0 gate/up writes fp32 act (k_split_act)");
    __shared__ __align__(16) _Float16 As[2][8192];
    // Q4_K group sums / 32 of the chunk, f16: per superblock 16 rows x 8 groups
    // (packed: rows 0..7 the hi, 8..15 the lo parts) or 16 rows x {8 hi, 8 lo}
    __shared__ __align__(16) _Float16 Ss[Q4K ? 2 : 1][Q4K ? 256 : 8];
    __shared__ int2 s_rowe[TMS];
    __shared__ float gpart[GATEUP ? NW : 1][TMS];
    __shared__ uint32_t rpart[GATEUP ? NW : 1][TMS];
    // flat: tiles in order, a tile's row blocks side by side on all XCDs; whole tiles
    // per XCD leave up to a tile's blocks of imbalance, and a tile's few rows of A cost
    // little to fetch into each L2 (gate/up us, 128 experts Q4_K / GLM shape at 16
    // tokens: 39.8 -> 33.8, 101.6 -> 92.0). With more rows, and experts of several
    // tiles, tile rounds of 8, one tile per XCD, alternating direction, as k_gemm_f16
    // (512 experts at 9.9 pairs each: 163 against 167 us flat).
    const uint32_t nt = tiles[3], slot = blockIdx.x >> 3, ti = slot / nblk, xcd = blockIdx.x & 7u;
    const uint32_t t = flat ? blockIdx.x / nblk : ti * 8u + ((ti & 1u) ? 7u - xcd : xcd);
    const uint32_t blk = flat ? blockIdx.x - t * nblk : slot - ti * nblk;
    if (t >= nt) return;
    const uint32_t* tile = tiles + 4u * t;
    const uint32_t n = tile[2];
    if (n == 0) return;
    const uint32_t e = tile[0], q0 = tile[1];
    const uint32_t ew = slot_of ? slot_of[e] : e;  // cached experts, as in k_gemm_f16
    if (ew == NO_SLOT) return;
    const uint32_t row0 = blk * (GATEUP ? 64u : 128u);
    const uint32_t ngroups = kdim / 32u;

    const bool sh_tile = e == e_shared;
    const uint8_t* const wb0 = sh_tile ? ws0 : w0 + (uint64_t)ew * rows_per_expert * stride0;
    const uint8_t* const wb1 = GATEUP ? (sh_tile ? ws1 : w1 + (uint64_t)ew * rows_per_expert * stride1) : wb0;
    const __amdgpu_buffer_rsrc_t ra_h = make_rsrc(ah, (uint32_t)(kdim * 2u) * a_rows);
    const __amdgpu_buffer_rsrc_t ra_l = make_rsrc(al, (uint32_t)(kdim * 2u) * a_rows);
    const __amdgpu_buffer_rsrc_t rgs = make_rsrc(gs, ngroups * 4u * a_rows);
    if constexpr (!Q4K && !Q6K && !Q8) stage_f16_tables<KIND>();

    auto run = [&](auto packed_tag) {
        const uint32_t tid = threadIdx.x, lane = tid & 63u, kq = lane >> 4, ln = lane & 15u;
        const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        BS B;
        B.init(wb0, wb1, stride0, stride1, rows_per_expert, kdim, row0 + 16u * (GATEUP ? 1u : 2u) * wave, lane);
        const uint32_t slabs = B.slabs;
        if constexpr (GATEUP) {
            if (tid < TMS) {
                const uint32_t q = q0 + (tid < n ? tid : 0u);
                const float2 st = ld_xstat(xstat, pairs ? pairs[q] / K : q);
                s_rowe[tid] = make_int2(x_exp(st.x), act_exp(st));
            }
        } else if constexpr (Q8) {
            if (tid < TMS) s_rowe[tid].x = x_exp(__uint_as_float(rowmax[q0 + (tid < n ? tid : 0u)]));
        } else {
            if (rowmax != nullptr && row0 == 0u) {
                bool bad = false;
                if (tid < n) {
                    const float m = __uint_as_float(rowmax[q0 + tid]);
                    bad = !(m == 0.f || (m >= ACT_RANGE_LO && m < ACT_RANGE_HI));  // NaN: bad
                }
                if (__any(bad) && lane == 0u) atomicOr(flags, FLAG_RANGE);
            }
        }
        constexpr bool PK = decltype(packed_tag)::value;
        constexpr uint32_t CH = PK ? 512u : 256u;  // columns per A chunk
        constexpr uint32_t CSB = CH / 256u, ROWT = PK ? 8u : 16u, DEPTH = 4u;
        // A staging: thread tid copies the 16-byte piece tid % (CH / 8) of tile rows
        // tid / (CH / 8) and ROWT / 2 further, hi and lo (rows past n: an offset past
        // the buffer, which reads zero without a fetch; no branch, so that the waits
        // count loads exactly and never drain the B ring).
        // Operand rows: hi 0 .. ROWT - 1, lo from ROWT; piece c of row r sits at slot
        // c ^ (r & 15), so a fragment read (16 rows at one piece) touches every bank
        // once.
        const uint32_t ac = tid % (CH / 8u), ar = tid / (CH / 8u);
        uint32_t avo[2];
#pragma unroll
        for (uint32_t j = 0; j < 2u; ++j) {
            const uint32_t r = ar + (ROWT / 2u) * j, q = q0 + (r < n ? r : 0u);
            avo[j] = r < n ? 2u * ((GATEUP && pairs ? pairs[q] / K : q) * kdim + 8u * ac) : 0xffffff00u;
        }
        uint4 areg[4];
        auto load_a = [&](uint32_t c) {
#pragma unroll
            for (uint32_t j = 0; j < 4u; ++j) areg[j] = buf_load16(j < 2u ? ra_h : ra_l, avo[j & 1u], 2u * CH * c);
        };
        auto store_a = [&](_Float16* A) {
#pragma unroll
            for (uint32_t j = 0; j < 4u; ++j) {
                const uint32_t r = ar + (ROWT / 2u) * (j & 1u) + (j < 2u ? 0u : ROWT);
                *reinterpret_cast<uint4*>(&A[r * CH + 8u * (ac ^ (r & 15u))]) = areg[j];
            }
        };
        // Q4_K group sums: thread tid < 128 owns one (row, group) of the chunk.
        const uint32_t sg = tid % (CH / 32u), sr = tid / (CH / 32u);
        float sreg = 0.f;
        uint32_t svo = 0;
        if constexpr (Q4K) {
            const uint32_t q = q0 + (sr < n ? sr : 0u);
            svo = 4u * ((GATEUP && pairs ? pairs[q] / K : q) * ngroups + sg);
        }
        auto load_s = [&](uint32_t c) { sreg = __uint_as_float(buf_load4(rgs, svo, (CH / 8u) * c)); };
        auto store_s = [&](_Float16* S) {
            _Float16 h, l;
            split_f16(sreg * 0.03125f, h, l);  // exact; they reach 2^16 for x and 2^19 for act within range
            if (tid < 128u) {
                if constexpr (PK) {
                    S[(sg >> 3) * 128u + sr * 8u + (sg & 7u)] = h;
                    S[(sg >> 3) * 128u + (sr + 8u) * 8u + (sg & 7u)] = l;
                } else {
                    S[sr * 16u + sg] = h;
                    S[sr * 16u + 8u + sg] = l;
                }
            }
        };
        floatx4 tot[NB];
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) tot[nb] = floatx4{0.f, 0.f, 0.f, 0.f};
        load_a(0u);
        if constexpr (Q4K) load_s(0u);
        if constexpr (!IQN) B.load_hdr(0u);
#pragma unroll
        for (uint32_t d = 0; d < DEPTH; ++d) B.load_slab(d, d, (d & 1u) == 0u);
        store_a(As[0]);
        if constexpr (Q4K) store_s(Ss[0]);
        __syncthreads();  // A chunk 0, the tables and s_rowe
        typename BS::SbState cur;
        if constexpr (!IQN) B.take_hdr(cur, 0u);
        const uint32_t nsb = (slabs + 3u) >> 2;
        // superblock sb, the part-th of its A chunk
        auto superblock = [&](uint32_t sb, auto part_tag) {
            constexpr uint32_t PART = decltype(part_tag)::value;
            const uint32_t c = sb / CSB;
            const _Float16* const A = As[c & 1u];
            const bool more = (c + 1u) * CSB < nsb;
            if constexpr (PART == 0u) {
                load_a(more ? c + 1u : c);
                if constexpr (Q4K) load_s(more ? c + 1u : c);
            }
            floatx4 acc[NB];
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) acc[nb] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (uint32_t sq = 0; sq < 4u; ++sq) {
                const uint32_t s = 4u * sb + sq;
                // B of slab s out of the ring, B(s + DEPTH) into its slot
                uint4 qv[NB];
                uint2 dv[NB];
                if ((sq & 1u) == 0u) B.take_pair(sq);
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    qv[nb] = B.nq[sq][nb];
                    if constexpr (IQN && !Q8) qv[nb].z = B.n1[sq][nb];
                    if constexpr (IQN || Q6K) dv[nb] = B.nd[sq][nb];
                }
                half8 fb[NB][2], fe[NB][2];
                float dg[NB][2];
                B.decode(cur, sq, qv, dv, fb, dg, fe);
                B.load_slab(sq, s + DEPTH, (sq & 1u) == 0u);
                if constexpr (!IQN) {
                    if (sq == 0) B.load_hdr(sb + 1u);
                }
#pragma unroll
                for (uint32_t gi = 0; gi < 2; ++gi) {
                    const uint32_t ch = 32u * PART + 8u * sq + (IQG ? 2u * kq + gi : 4u * gi + kq);
                    const half8 a0 = *reinterpret_cast<const half8*>(&A[ln * CH + 8u * (ch ^ ln)]);
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb) {
                        const floatx4 z = IQN ? floatx4{0.f, 0.f, 0.f, 0.f} : acc[nb];
                        acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a0, fb[nb][gi], z, 0, 0, 0);
                        if constexpr (Q6K)
                            acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a0, fe[nb][gi], acc[nb], 0, 0, 0);
                    }
                    if constexpr (!PK) {
                        const half8 a1 = *reinterpret_cast<const half8*>(&A[(16u + ln) * CH + 8u * (ch ^ ln)]);
#pragma unroll
                        for (int nb = 0; nb < NB; ++nb)
                            acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a1, fb[nb][gi], acc[nb], 0, 0, 0);
                    }
                    if constexpr (IQN) {
                        // (a last superblock cut short: clamped weights over columns past K,
                        // not added)
                        if (s < slabs) {
#pragma unroll
                            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                                for (int j = 0; j < 4; ++j) tot[nb][j] += dg[nb][gi] * acc[nb][j];
                        }
                    }
                }
            }
            if constexpr (!IQN) {
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                    for (int j = 0; j < 4; ++j) tot[nb][j] += cur.dsc[nb] * acc[nb][j];
                if constexpr (Q4K) {
                    const half8 sa = *reinterpret_cast<const half8*>(
                        &Ss[c & 1u][PK ? PART * 128u + ln * 8u : ln * 16u + 8u * (kq & 1u)]);
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb) {
                        const uint4 v = kq < (PK ? 1u : 2u) ? make_uint4(bytes01(cur.mn[nb][0]), bytes23(cur.mn[nb][0]),
                                                                         bytes01(cur.mn[nb][1]), bytes23(cur.mn[nb][1]))
                                                            : make_uint4(0, 0, 0, 0);
                        const floatx4 mc = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                            sa, __builtin_bit_cast(half8, v), floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                        for (int j = 0; j < 4; ++j) tot[nb][j] -= cur.dmn[nb] * mc[j];
                    }
                }
                B.take_hdr(cur, sb + 1u);  // past the last superblock: the clamped header, never used
            }
            if (PART + 1u == CSB && more) {
                // the other buffer was last read before the last barrier
                store_a(As[(c + 1u) & 1u]);
                if constexpr (Q4K) store_s(Ss[(c + 1u) & 1u]);
                __syncthreads();
            }
        };
        for (uint32_t sb = 0; sb < nsb; sb += CSB) {
            superblock(sb, std::integral_constant<uint32_t, 0>{});
            if constexpr (CSB == 2u) {
                if (sb + 1u >= nsb) break;
                superblock(sb + 1u, std::integral_constant<uint32_t, 1>{});
            }
        }
        // packed: rows 8..15 hold the lo products of rows 0..7 (lane + 32)
        if constexpr (PK) {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int j = 0; j < 4; ++j) tot[nb][j] += __shfl_xor(tot[nb][j], 32);
        }
        const uint32_t mr = PK ? (kq & 1u) : kq;
        const bool own = !PK || kq < 2u;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t m = 4u * mr + j;
            const uint64_t q = q0 + m;
            const bool live = own && m < n;
            if constexpr (GATEUP) {
                // g, u in true units, then act 2^a_t; act column row0 + 16 w + ln
                const int ex = s_rowe[m].x, ea = s_rowe[m].y;
                const float sw = swiglu(ldexpf(tot[0][j], -ex), ldexpf(tot[1][j], -ex), limit);
                const float v = Q8 ? sw : ldexpf(sw, ea);
                const uint32_t rm = row_max16(__float_as_uint(fabsf(v)));
                if (own && ln == 0u) rpart[wave][m] = rm;
                if constexpr (Q8) {
                    if (live) out[q * ldo + row0 + 16u * wave + ln] = v;
                    continue;
                }
                _Float16 hh, ll;
                split_f16(v, hh, ll);
                if (live) {
                    const uint64_t o = q * ldo + a_pos<AORD>(row0 + 16u * wave + ln);
                    out_h[o] = hh;
                    out_l[o] = ll;
                }
                if (out_gs != nullptr) {
                    float gsum = v;
                    gsum += dpp_mov<0xb1>(gsum);
                    gsum += dpp_mov<0x4e>(gsum);
                    gsum += dpp_mov<0x141>(gsum);
                    gsum += dpp_mov<0x140>(gsum);
                    if (own && ln == 0u) gpart[wave][m] = gsum;  // half of a 32-column group
                }
            } else if (live) {
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)
                    out[q * ldo + row0 + 32u * wave + 16u * nb + ln] = Q8 ? ldexpf(tot[nb][j], -s_rowe[m].x) : tot[nb][j];
            }
        }
        if constexpr (GATEUP) {
            __syncthreads();
            // 32-column group g of the block's 64 act columns = waves 2 g, 2 g + 1
            if (out_gs != nullptr && tid < 2u * TMS) {
                const uint32_t g = tid / TMS, m = tid % TMS;
                if (m < n)
                    out_gs[(q0 + m) * (ldo / 32u) + row0 / 32u + g] = gpart[2u * g][m] + gpart[2u * g + 1u][m];
            }
            if (tid < n)
                atomicMax(rowmax + q0 + tid,
                          max(max(rpart[0][tid], rpart[1][tid]), max(rpart[2][tid], rpart[3][tid])));
        }
    };
    if (n <= 8u) run(std::true_type{});
    else run(std::false_type{});
}

}  // namespace ingot
