// The float32 dot_general: each output is the reference's sequential k-order fold, the product and every partial
// sum rounded to float32 (lumen/reference/mod.rs:981-993), so two VALU instructions a multiply-add and one
// dependent chain an output (the matrix cores' float32 instructions round the product and sum together).
//
// What bounds it is VALU issue where results fill the chip, and the latency of A and B where they leave a wave or
// two a SIMD: all workgroups walk k together, so each line is first asked for by everyone at once, from beyond
// the L2. Hence:
//  * A wave computes RM rows x 64 columns, a column a lane (the launcher picks RM): few rows a wave leave enough
//    waves for small results.
//  * A's values are uniform over the wave, so they come through the scalar cache into SGPRs and enter the
//    multiply as its scalar operand: no LDS reads, no vector registers. Broadcast from LDS the same values would
//    take its whole 128 bytes a clock; made scalar with v_readlane they cost a VALU instruction each (2048^3:
//    750 us, 384 us with scalar loads).
//  * Scalar loads return out of order, so only one chunk of KC k can be ahead. A vector load a stage, three
//    stages ahead, brings A's lines into the L2 first.
//  * B's tile (32 k x 64 columns, shared by the workgroup's four waves) goes through registers, three stages
//    ahead, into a double-buffered LDS tile, so that either memory order is read along its contiguous axis, 16
//    bytes at a time (with 4 bytes at a time [256, 512] x [512, 1024] took 16.6 us).
// Measured: [256, 512] x [512, 1024] 14.1 us, of which the VALU's 4 cycles an instruction are 7; 64 x 64 tiles
// of 16 outputs a thread read through LDS (64 workgroups, one SIMD in four at work) took 81. 2048^3 with B
// contiguous along k 352 us, 49 TFLOP/s.
#pragma once

#include "gemm.h"

namespace nhipk {

// 4-byte aligned vectors in the constant address space: read by scalar loads where the address is uniform.
template <int N>
struct ScalarVec {
    typedef float type __attribute__((ext_vector_type(N), aligned(4)));
    typedef const type __attribute__((address_space(4))) * ptr;
};
template <>
struct ScalarVec<1> {
    typedef const float __attribute__((address_space(4))) * ptr;
};

// AK: A contiguous along k, else along m. BN: B contiguous along n, else along k.
// Needs m >= RM and k < 2^30. `epi.visit(f)` calls f with the store: st(s, batch offset, row, column, sum).
template <int RM, bool AK, bool BN, class Epi>
__device__ __forceinline__ void gemm_fold_tile(const GemmShape &s, const float *__restrict__ a, const float *__restrict__ b,
                                               const Epi &epi) {
    constexpr int KB = 32;                           // k of a staged B tile
    constexpr int KC = RM <= 2 ? 16 : 32 / RM;       // k of a register chunk: 2 RM KC <= 64 SGPRs
    constexpr int CH = KB / KC;
    constexpr int AHEAD = 3;                         // stages in flight
    constexpr int PITCH = BN ? 64 : 65;              // a transposing store meets 64 different banks at 65
    __shared__ float Bs[2][KB * PITCH];
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    int tm, tn;
    tile_of(blockIdx.x, s.tiles_m, s.tiles_n, tm, tn);
    int64_t oa, ob, od;
    batch_offsets(s, blockIdx.y, oa, ob, od);
    // the wave's rows: the last RM ones where fewer are left, of which those before `own` are another wave's to store
    const int64_t own = int64_t(tm) * (4 * RM) + wave * RM;
    const int64_t m0 = min(own, s.m - RM), n0 = int64_t(tn) * 64;
    const int ktot = int(s.k);

    // B's tile at k0, 16 bytes at a time along its contiguous axis: thread t takes 4 columns of rows t / 16 and 16
    // more (BN), or 4 k of columns t / 8 and 32 more. Past the last row or column: the last one again, never used.
    typedef float vec __attribute__((ext_vector_type(4), aligned(4)));
    const int bcol = BN ? (t & 15) * 4 : t >> 3, brow = BN ? t >> 4 : (t & 7) * 4;
    const float *bp = b + ob;
    const int64_t c0 = min(n0 + bcol, s.n - 1) * s.b_n, c1 = min(n0 + bcol + 32, s.n - 1) * s.b_n;
    const bool cols = n0 + bcol + 3 < s.n;
    auto load_b = [&](float (&x)[8], int k0) {
        if constexpr (BN) {
            const float *p = bp + int64_t(min(k0 + brow, ktot - 1)) * s.b_k;
            const float *q = bp + int64_t(min(k0 + brow + 16, ktot - 1)) * s.b_k;
            if (cols) {
                const vec u = *reinterpret_cast<const vec *>(p + n0 + bcol), v = *reinterpret_cast<const vec *>(q + n0 + bcol);
#pragma unroll
                for (int i = 0; i < 4; ++i) x[i] = u[i], x[4 + i] = v[i];
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) x[i] = (i < 4 ? p : q)[min(n0 + bcol + (i & 3), s.n - 1)];
            }
        } else if (k0 + KB <= ktot) {
            const vec u = *reinterpret_cast<const vec *>(bp + c0 + k0 + brow), v = *reinterpret_cast<const vec *>(bp + c1 + k0 + brow);
#pragma unroll
            for (int i = 0; i < 4; ++i) x[i] = u[i], x[4 + i] = v[i];
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) x[i] = bp[(i < 4 ? c0 : c1) + min(k0 + brow + (i & 3), ktot - 1)];
        }
    };
    auto store_b = [&](const float (&x)[8], int buf) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            Bs[buf][BN ? (brow + (i & 4) * 4) * PITCH + bcol + (i & 3) : (brow + (i & 3)) * PITCH + bcol + (i & 4) * 8] = x[i];
    };
    const float *ap = a + oa + m0 * s.a_m;
    // one word of each 32 bytes of the wave's part of A at [k0, k0 + KB)
    auto touch_a = [&](int k0) {
        const int r = AK ? min(lane >> 2, RM - 1) : 0, kk = AK ? (lane & 3) * 8 : lane & (KB - 1);
        return ap[r * s.a_m + int64_t(min(k0 + kk, ktot - 1)) * (AK ? 1 : s.a_k)];
    };
    auto load_a = [&](float (&x)[RM][KC], int k0) {
        if constexpr (AK) {
#pragma unroll
            for (int r = 0; r < RM; ++r) {
                const char *p = reinterpret_cast<const char *>(ap + r * s.a_m);
                const auto v = *(typename ScalarVec<KC>::ptr)(p + uint32_t(k0) * 4u);
#pragma unroll
                for (int i = 0; i < KC; ++i) x[r][i] = v[i];
            }
        } else {
#pragma unroll
            for (int i = 0; i < KC; ++i) {
                const auto v = *(typename ScalarVec<RM>::ptr)(ap + int64_t(k0 + i) * s.a_k);
                if constexpr (RM == 1) {
                    x[0][i] = v;
                } else {
#pragma unroll
                    for (int r = 0; r < RM; ++r) x[r][i] = v[r];
                }
            }
        }
    };
    auto read_b = [&](float (&y)[KC], int buf, int c) {
#pragma unroll
        for (int i = 0; i < KC; ++i) y[i] = Bs[buf][(c * KC + i) * PITCH + lane];
    };

    float acc[RM];
#pragma unroll
    for (int r = 0; r < RM; ++r) acc[r] = 0.0f;

    const int stages = ktot / KB;  // whole ones
    float st[AHEAD][8], touched[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
        load_b(st[i], i * KB);
        touched[i] = touch_a(i * KB);
    }
    store_b(st[0], 0);
    __syncthreads();
    if (stages > 0) {
        float xa[2][RM][KC], yb[2][KC];
        load_a(xa[0], 0);
        read_b(yb[0], 0, 0);
        __builtin_amdgcn_s_waitcnt(0xc07f);
        for_tiles<AHEAD>(stages, [&](int kt, auto phase) {
            constexpr int P = decltype(phase)::value;
            const int k0 = kt * KB, buf = kt & 1;
            asm volatile("" ::"v"(touched[P]));
            load_b(st[P], k0 + AHEAD * KB);
            touched[P] = touch_a(k0 + AHEAD * KB);
#pragma unroll
            for (int c = 0; c < CH; ++c) {
                const int cur = c & 1, nxt = cur ^ 1;
                // the empty asm keeps each chunk's reads and sums in their place: merged or moved together,
                // several chunks of A would not fit the scalar registers. The last chunk's next one is read
                // whether or not it exists (from the last whole chunk then), so that no branch parts a chunk's
                // reads from their use.
                int next = min(k0 + (c + 1) * KC, stages * KB - KC);
                asm volatile("" : "+s"(next));
                load_a(xa[nxt], next);
                read_b(yb[nxt], c + 1 < CH ? buf : buf ^ 1, (c + 1) % CH);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < KC; ++i)
#pragma unroll
                    for (int r = 0; r < RM; ++r) acc[r] = __fadd_rn(acc[r], __fmul_rn(xa[cur][r][i], yb[cur][i]));
#pragma unroll
                for (int r = 0; r < RM; ++r) asm volatile("" : "+v"(acc[r]));
                __builtin_amdgcn_sched_barrier(0);
                __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the next chunk is there
                // this stage's last LDS reads have returned: after the barrier its buffer may be refilled
                if (c == CH - 2) {
                    store_b(st[(P + 1) % AHEAD], buf ^ 1);
                    __syncthreads();
                }
            }
        });
    }
    // the remaining k, which stop at the last one: a product with a padded zero could change a sum's sign or
    // make a NaN of an infinity
    const float *tail = Bs[stages & 1];
    for (int i = 0; i < ktot - stages * KB; ++i) {
        const float y = tail[i * PITCH + lane];
#pragma unroll
        for (int r = 0; r < RM; ++r)
            acc[r] = __fadd_rn(acc[r], __fmul_rn(ap[r * s.a_m + int64_t(stages * KB + i) * s.a_k], y));
    }
    const int64_t col = n0 + lane;
    if (col >= s.n) return;
    epi.visit([&](auto out) {
#pragma unroll
        for (int r = 0; r < RM; ++r)
            if (m0 + r >= own) out(s, od, m0 + r, col, acc[r]);
    });
}

template <int RM, bool AK, bool BN, class Epi>
__global__ __launch_bounds__(256) void gemm_fold(GemmShape s, const float *__restrict__ a, const float *__restrict__ b,
                                                 Epi epi) {
    gemm_fold_tile<RM, AK, BN>(s, a, b, epi);
}

}  // namespace nhipk
