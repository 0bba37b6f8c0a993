// bf16/f16 dots of few rows (m <= 64, decode): D[m, n] = A[m, k] B[n, k]^T, both contiguous along k.
//
// Reading B once is all the work, so what bounds it is HBM bandwidth, given enough workgroups and bytes in flight;
// 128 x 128 tiles of 16 rows are a quarter of the chip's workgroups, with a split-k pass and its reduction after
// them. Here a workgroup takes 16 columns and its NW waves divide k (64 at a time, in turn), so [16, 2048] x
// [8192, 2048] is 512 workgroups with no partial products in memory. Fragments come straight from memory: a
// v_mfma_f32_16x16x32 operand is 16 rows of 64 contiguous bytes, A's rows stay in the L2, and U chunks of 64 k are in
// flight a wave. The waves' sums are added through LDS in wave order.
// [16, 2048] x [8192, 2048]: 17.4 (two splits and their sum) -> 9.7 us, 3.5 TB/s; [16, 8192] x [2048, 8192]: 19.0 -> 16.4.
#pragma once

#include "gemm.h"

namespace nhipk {

template <bool F16>
__device__ __forceinline__ f32x4_t mfma16(uint4 a, uint4 b, f32x4_t c) {
    if constexpr (F16)
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0,
                                                       0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                        0, 0, 0);
}

// MT: 16-row groups of A (m <= 16 MT). Needs k % 8 == 0 and 16-byte aligned rows. `epi.visit(f)` calls f with the
// store: st(s, batch offset, row, column, sum).
template <bool F16, int MT, int NW, class Epi>
__device__ __forceinline__ void gemm_skinny_tile(const GemmShape &s, const uint16_t *__restrict__ a,
                                                 const uint16_t *__restrict__ b, const Epi &epi) {
    constexpr int U = MT >= 4 ? 2 : 4;  // chunks of 64 k in flight
    __shared__ f32x4_t sums[NW][MT][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15, g = lane >> 4;
    int64_t oa, ob, od;
    batch_offsets(s, blockIdx.y, oa, ob, od);
    const int64_t n0 = int64_t(blockIdx.x) * 16;
    // rows past the last one: the last one again, never stored
    const uint16_t *pb = b + ob + min(n0 + l16, s.n - 1) * s.b_n + 8 * g;
    const uint16_t *pa[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) pa[i] = a + oa + min(int64_t(16 * i + l16), s.m - 1) * s.a_m + 8 * g;

    f32x4_t acc[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    const int k = int(s.k), step = 64 * NW;
    int k0 = 64 * wave;
    for (; k0 + (U - 1) * step + 64 <= k; k0 += U * step) {
        uint4 fb[U][2], fa[U][2][MT];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int c = 0; c < 2; ++c) fb[u][c] = *reinterpret_cast<const uint4 *>(pb + k0 + u * step + 32 * c);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int i = 0; i < MT; ++i)
                    fa[u][c][i] = *reinterpret_cast<const uint4 *>(pa[i] + k0 + u * step + 32 * c);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int i = 0; i < MT; ++i) acc[i] = mfma16<F16>(fa[u][c][i], fb[u][c], acc[i]);
    }
    for (; k0 < k; k0 += step)  // the last chunks, a lane's 8 k past the end as zeros
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const bool in = k0 + 32 * c + 8 * g < k;
            const uint4 fb = in ? *reinterpret_cast<const uint4 *>(pb + k0 + 32 * c) : make_uint4(0, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < MT; ++i)
                acc[i] = mfma16<F16>(in ? *reinterpret_cast<const uint4 *>(pa[i] + k0 + 32 * c) : make_uint4(0, 0, 0, 0),
                                     fb, acc[i]);
        }
#pragma unroll
    for (int i = 0; i < MT; ++i) sums[wave][i][lane] = acc[i];
    __syncthreads();
    // C layout of a 16 x 16 block: lane holds column lane % 16, rows 4 (lane / 16) + e
    if (wave >= MT) return;
    f32x4_t v = sums[0][wave][lane];
#pragma unroll
    for (int w = 1; w < NW; ++w) v += sums[w][wave][lane];
    const int64_t col = n0 + l16, row = 16 * wave + 4 * g;
    if (col >= s.n) return;
    epi.visit([&](auto st) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (row + e < s.m) st(s, od, row + e, col, v[e]);
    });
}

template <bool F16, int MT, int NW>
__global__ __launch_bounds__(64 * NW) void gemm_skinny(GemmShape s, const uint16_t *__restrict__ a,
                                                        const uint16_t *__restrict__ b, AnyStore out) {
    gemm_skinny_tile<F16, MT, NW>(s, a, b, out);
}

}  // namespace nhipk
