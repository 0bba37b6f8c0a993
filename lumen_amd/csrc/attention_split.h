// Flash attention forward for few query rows: the keys of a (batch, key/value head) are divided over waves and
// workgroups instead of the queries.
//
// With one query a sequence (decode) the work is reading K and V once, so what bounds it is HBM bandwidth, given
// enough bytes in flight. flash_fwd_kernel gives a head one workgroup whose four waves share one 64-key tile in
// flight behind a barrier, three of them without a query. Here:
//  * 32 query rows are one MFMA tile: the rows of a key/value head's whole group, query heads times queries, so
//    grouped heads read K and V once.
//  * Each of a workgroup's four waves streams 32-key tiles of its own through a private double-buffered LDS ring:
//    no barrier in the loop, two tiles (32 KiB at head dim 128) in flight a wave.
//  * Where there are too few heads to fill the chip the keys are split over workgroups too; their float32 partial
//    sums, maxima and sums of exponentials go through a workspace that flash_combine_kernel reduces in order.
// Measured: batch 16, 16 heads of 128, one query, 4096 keys: 151 -> 97 us, 3.5 -> 5.5 TB/s (a copy reaches 4.6); batch
// 1: 109 -> 20 us; batch 3, 27958 keys: 923 -> 126 us.
// The arithmetic is flash_fwd_kernel's: base 2, the running maximum raised lazily, P rounded to 16 bits.
#pragma once

#include "attention.h"

namespace nhipk {

struct SplitParams {
    int64_t rows;      // query rows of a key/value head: heads / kv_heads * sq
    int64_t tiles;     // 32-row tiles of them
    int64_t splits;    // workgroups a row tile
    int64_t keytiles;  // 32-key tiles a workgroup
    float *sums;       // [unit][split][rows of a tile][value head dim], null with one split
    float2 *stats;     // [unit][split][rows of a tile] maximum (base 2), sum of exponentials
};

// Rows [k0, k0 + 32) of a [*, D] operand into one wave's swizzled tile (the one-wave form of load_tile_async).
template <int D>
__device__ __forceinline__ void load_tile32(const uint16_t *src, int64_t rs, int64_t k0, int64_t rows, uint16_t *dst,
                                            int lane, int64_t cols) {
    constexpr int RPS = 1024 / (D * 2), SEGS = 32 / RPS;
    const int64_t bytes = ((rows - 1) * rs + D) * 2;
    if (bytes < (int64_t(1) << 31) && (k0 + 32) * rs * 2 < (int64_t(1) << 31)) {
        const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)src, (short)0, int(bytes), 0x00020000);
        const uint32_t so = uint32_t(k0 * rs * 2);
        auto seg_load = [&](int seg, bool masked) {
            const int r = seg * RPS + lane / (D / 8);
            const int sc = (lane % (D / 8)) ^ kv_swz<D>(r);
            const uint32_t vo = uint32_t((r * rs + (sc << 3)) * 2);
            if (!masked || (8 * sc < cols && k0 + r < rows))
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void_t *)(dst + seg * 512), 16, vo, so, 0, 0);
        };
        if (k0 + 32 <= rows && cols >= D) {
#pragma unroll
            for (int seg = 0; seg < SEGS; ++seg) seg_load(seg, false);
        } else {
#pragma unroll
            for (int seg = 0; seg < SEGS; ++seg) seg_load(seg, true);
        }
        return;
    }
#pragma unroll
    for (int seg = 0; seg < SEGS; ++seg) {
        const int r = seg * RPS + lane / (D / 8);
        const int64_t row = min(k0 + r, rows - 1);
        __builtin_amdgcn_global_load_lds(src + row * rs + (((lane % (D / 8)) ^ kv_swz<D>(r)) << 3),
                                         (lds_void_t *)(dst + seg * 512), 16, 0, 0);
    }
}

// The K and V tiles of keys [k0, k0 + 32).
template <int D>
__device__ __forceinline__ void load_pair32(const AttnParams &p, const uint16_t *kp, const uint16_t *vp, int64_t k0,
                                            uint16_t *dst, int lane) {
    load_tile32<D>(kp, p.k_s, k0, p.sk, dst, lane, p.hd);
    load_tile32<D>(vp, p.v_s, k0, p.sk, dst + 32 * D, lane, p.hdv);
}

// As in flash_fwd_body the two stages are arrays of their own; the first holds the waves' sums at the end.
template <int D, bool F16, bool CAUSAL>
__device__ __forceinline__ void flash_split_body(const AttnParams &p, const SplitParams &sp) {
    constexpr int BN = 32, DS = D / 16, DT = D / 32, TILE = BN * D;
    __shared__ __align__(1024) uint16_t rings0[4][2 * TILE], rings1[4][2 * TILE];
    __shared__ float2 ml[4][32];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int h = lane >> 5, l32 = lane & 31, g = lane >> 4, s16 = lane & 15;
    // The workgroups of a (batch, key/value head) run on one XCD, whose L2 then holds the keys its row tiles share: 32 x 8
    // heads of 64, 256 rows, 4096 keys 291 us spread over the XCDs, 153 (7 TB/s of K and V read again); 8 x 16 heads, 200
    // rows 133, 61. As xcd_order, in 32-bit scalars: from vector values the addresses would put each load into a loop
    // over the lanes.
    const uint32_t heads = uint32_t(p.batch * p.kv_heads), per = uint32_t(sp.tiles * sp.splits), wg = blockIdx.x;
    const uint32_t at = heads % 8 ? wg : (wg / 8 / per * 8 + wg % 8) * per + wg / 8 % per;
    const int64_t head = __builtin_amdgcn_readfirstlane(at / per);
    const int64_t rt = __builtin_amdgcn_readfirstlane(at % per / uint32_t(sp.splits));
    const int64_t split = __builtin_amdgcn_readfirstlane(at % uint32_t(sp.splits)), unit = head * sp.tiles + rt;
    const int64_t b = head / p.kv_heads, nkv = head % p.kv_heads;
    const int64_t row = rt * 32 + l32, group = p.heads / p.kv_heads;
    const int live = int(min(int64_t(32), sp.rows - rt * 32));  // rows of this tile
    const bool qvalid = l32 < live;
    const int64_t n = nkv * group + (qvalid ? row / p.sq : 0), qi = qvalid ? row % p.sq : 0;
    const int64_t shift = p.sk - p.sq;

    const uint16_t *qp = p.q + b * p.q_b + n * p.q_n + qi * p.q_s;
    const uint16_t *kp = p.k + b * p.k_b + nkv * p.k_n;
    const uint16_t *vp = p.v + b * p.v_b + nkv * p.v_n;

    // the last key any row sees, and the first key some row does not (a tile that spans heads holds every query)
    int64_t kend = p.sk, full_end = p.sk;
    if (CAUSAL) {
        const int64_t first = rt * 32 % p.sq, last = first + live - 1;
        kend = min(p.sk, min(last, p.sq - 1) + shift + 1);
        full_end = min(p.sk, (last < p.sq ? first : 0) + shift + 1);
    }
    const int64_t t0 = split * sp.keytiles;
    const int64_t t1 = min(t0 + sp.keytiles, (kend + BN - 1) / BN);

    uint16_t *const ring0 = rings0[wave], *const ring1 = rings1[wave];
    if (p.sk % BN || p.hd < D || p.hdv < D)  // chunks the loads leave out hold zeros
        for (int i = lane * 8; i < 2 * TILE; i += 512) {
            *reinterpret_cast<uint4 *>(ring0 + i) = make_uint4(0, 0, 0, 0);
            *reinterpret_cast<uint4 *>(ring1 + i) = make_uint4(0, 0, 0, 0);
        }

    uint4 qf[DS];
#pragma unroll
    for (int t = 0; t < DS; ++t)
        qf[t] = qvalid && 16 * t + 8 * h < p.hd ? *reinterpret_cast<const uint4 *>(qp + 16 * t + 8 * h)
                                                : make_uint4(0, 0, 0, 0);
    f32x16_t acc[DT];
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][e] = 0.0f;
    const float c2 = p.scale * 1.4426950408889634f;
    float m = -1e30f, l = 0.0f;

    __builtin_amdgcn_s_waitcnt(0xc07f);  // the zeros are written before a load can land on them
    auto tile = [&](int64_t t, const uint16_t *cur, uint16_t *next) __attribute__((always_inline)) {
        // tile t has landed; the other stage's reads were waited for by the MFMAs that used them
        __builtin_amdgcn_s_waitcnt(0x0f70);
        if (t + 4 < t1) load_pair32<D>(p, kp, vp, (t + 4) * BN, next, lane);
        const char *Kb = reinterpret_cast<const char *>(cur);
        const char *Vb = Kb + TILE * 2;
        const int64_t k0 = t * BN;
        f32x16_t s;
#pragma unroll
        for (int e = 0; e < 16; ++e) s[e] = 0.0f;
#pragma unroll
        for (int u = 0; u < DS; ++u)
            s = mfma32<F16>(*reinterpret_cast<const uint4 *>(Kb + kv_off<D>(l32, 16 * u + 8 * h)), qf[u], s);
        if (k0 + BN > full_end) {
            const int lim = int(max(min(min(CAUSAL ? qi + shift : p.sk - 1, p.sk - 1) - k0 - 4 * h, int64_t(BN)), int64_t(-1)));
#pragma unroll
            for (int e = 0; e < 16; ++e) s[e] = 8 * (e / 4) + (e % 4) <= lim ? s[e] : -INFINITY;
        }
        float mx = s[0];
#pragma unroll
        for (int e = 1; e < 16; ++e) mx = fmaxf(mx, s[e]);
        mx = max_halves(mx) * c2;
        if (__any(mx > m + 8.0f)) {
            const float mnew = fmaxf(m, mx);
            const float alpha = fast_exp2(m - mnew);
            l *= alpha;
#pragma unroll
            for (int i = 0; i < DT; ++i)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[i][e] *= alpha;
            m = mnew;
        }
        uint4 pb[2];
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            uint32_t w[4];
#pragma unroll
            for (int j = 0; j < 8; j += 2) {
                const float e0 = fast_exp2(fmaf(s[8 * half + j], c2, -m));
                const float e1 = fast_exp2(fmaf(s[8 * half + j + 1], c2, -m));
                l += e0 + e1;  // this half-wave's keys; the halves are added at the end
                w[j / 2] = pack2<F16>(e0, e1);
            }
            pb[half] = make_uint4(w[0], w[1], w[2], w[3]);
        }
#pragma unroll
        for (int t2 = 0; t2 < 2; ++t2) {
            const int key = 16 * t2 + 4 * h + s16 / 4;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                const int col = 32 * dt + 16 * (g & 1) + 4 * (s16 & 3);
                v4i16_t x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_t *)(Vb + kv_off<D>(key, col)));
                v4i16_t y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_t *)(Vb + kv_off<D>(key + 8, col)));
                uint2 xa = __builtin_bit_cast(uint2, x), ya = __builtin_bit_cast(uint2, y);
                acc[dt] = mfma32<F16>(make_uint4(xa.x, xa.y, ya.x, ya.y), pb[t2], acc[dt]);
            }
        }
    };
    const int64_t first_tile = t0 + wave;
    if (first_tile < t1) load_pair32<D>(p, kp, vp, first_tile * BN, ring0, lane);
    for (int64_t t = first_tile; t < t1; t += 8) {
        tile(t, ring0, ring1);
        if (t + 4 < t1) tile(t + 4, ring1, ring0);
    }
    l += __shfl_xor(l, 32, 64);

    // the four waves' sums, scaled to the common maximum, added in wave order
    if (h == 0) ml[wave][l32] = make_float2(m, l);
    __syncthreads();
    float top = ml[0][l32].x;
#pragma unroll
    for (int w = 1; w < 4; ++w) top = fmaxf(top, ml[w][l32].x);
    const float own = fast_exp2(m - top);
    static_assert(sizeof(rings0) >= 4 * 32 * D * sizeof(float), "the waves' sums fit the first stage");
    float *red = reinterpret_cast<float *>(&rings0[0][0]);  // [wave][row][D], chunks of 4 swizzled by row
    if (qvalid) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int e4 = 0; e4 < 4; ++e4) {
                const int c = 8 * dt + 2 * e4 + h;
                *reinterpret_cast<float4 *>(red + (wave * 32 + l32) * D + ((c ^ (l32 & 7)) << 2)) =
                    make_float4(acc[dt][4 * e4] * own, acc[dt][4 * e4 + 1] * own, acc[dt][4 * e4 + 2] * own,
                                acc[dt][4 * e4 + 3] * own);
            }
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < live * (D / 4); idx += 256) {
        const int r = idx / (D / 4), c = idx % (D / 4);
        if (4 * c >= p.hdv) continue;
        float tm = ml[0][r].x, tl = 0.0f;
        for (int w = 1; w < 4; ++w) tm = fmaxf(tm, ml[w][r].x);
        for (int w = 0; w < 4; ++w) tl += ml[w][r].y * fast_exp2(ml[w][r].x - tm);
        float4 o = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        for (int w = 0; w < 4; ++w) {
            const float4 x = *reinterpret_cast<const float4 *>(red + (w * 32 + r) * D + ((c ^ (r & 7)) << 2));
            o.x += x.x, o.y += x.y, o.z += x.z, o.w += x.w;
        }
        if (sp.sums) {
            const int64_t at = (unit * sp.splits + split) * min(int64_t(32), sp.rows) + r;
            *reinterpret_cast<float4 *>(sp.sums + at * p.hdv + 4 * c) = o;
            if (c == 0) sp.stats[at] = make_float2(tm, tl);
            continue;
        }
        const int64_t rr = rt * 32 + r, rn = nkv * group + rr / p.sq, ri = rr % p.sq;
        const float inv = tl > 0.0f ? 1.0f / tl : 0.0f;
        *reinterpret_cast<uint2 *>(p.o + b * p.o_b + rn * p.o_n + ri * p.o_s + 4 * c) =
            make_uint2(pack2<F16>(o.x * inv, o.y * inv), pack2<F16>(o.z * inv, o.w * inv));
        if (c == 0 && p.lse)
            p.lse[(b * p.heads + rn) * p.sq + ri] = tl > 0.0f ? (tm + __log2f(tl)) * 0.6931471805599453f : -INFINITY;
    }
}

template <int D, bool F16, bool CAUSAL>
__global__ __launch_bounds__(256) void flash_split_kernel(AttnParams p, SplitParams sp) {
    flash_split_body<D, F16, CAUSAL>(p, sp);
}

// A wave a query row: the splits' sums scaled to their common maximum and added in split order.
template <bool F16>
__global__ __launch_bounds__(256) void flash_combine_kernel(AttnParams p, SplitParams sp) {
    const int lane = threadIdx.x & 63;
    const int64_t id = int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
    if (id >= p.batch * p.kv_heads * sp.rows) return;
    const int64_t head = id / sp.rows, row = id % sp.rows;
    const int64_t per = min(int64_t(32), sp.rows);
    const int64_t at = (head * sp.tiles + row / 32) * sp.splits * per + row % 32;  // + split * per
    float top = -INFINITY, l = 0.0f;
    for (int64_t s = 0; s < sp.splits; ++s) top = fmaxf(top, sp.stats[at + s * per].x);
    for (int64_t s = 0; s < sp.splits; ++s) {
        const float2 x = sp.stats[at + s * per];
        l += x.y * fast_exp2(x.x - top);
    }
    const int64_t b = head / p.kv_heads, n = head % p.kv_heads * (p.heads / p.kv_heads) + row / p.sq, qi = row % p.sq;
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    uint16_t *op = p.o + b * p.o_b + n * p.o_n + qi * p.o_s;
    for (int c = 2 * lane; c < p.hdv; c += 128) {
        float x = 0.0f, y = 0.0f;
        for (int64_t s = 0; s < sp.splits; ++s) {
            const float w = fast_exp2(sp.stats[at + s * per].x - top);
            const float2 v = *reinterpret_cast<const float2 *>(sp.sums + (at + s * per) * p.hdv + c);
            x += v.x * w;
            y += v.y * w;
        }
        *reinterpret_cast<uint32_t *>(op + c) = pack2<F16>(x * inv, y * inv);
    }
    if (lane == 0 && p.lse)
        p.lse[(b * p.heads + n) * p.sq + qi] = l > 0.0f ? (top + __log2f(l)) * 0.6931471805599453f : -INFINITY;
}

}  // namespace nhipk
