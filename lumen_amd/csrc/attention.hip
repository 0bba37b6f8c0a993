// C entry points of the flash attention kernels (attention.h): nhip_flash_fwd, nhip_flash_bwd and the
// allocation-free nhip_flash_bwd_noalloc.
#include <algorithm>
#include <map>
#include <mutex>
#include <string>

#include "attention.h"
#include "attention_split.h"
#include "nhip_internal.h"

using namespace nhip;

namespace {

// Scratch of nhip_flash_bwd_noalloc: the backward's workspace (delta and base-2 LSE, 2 floats a query row, then
// the mode's dS tiles or dQ accumulator), for callers that cannot allocate. One copy per GPU, held until the
// process ends; 16 MiB covers 2^21 query rows (batch x heads x sq) in mode 2, e.g. [4, 4096, 16, 128] uses
// 2 MiB there.
constexpr size_t kFlashScratchBytes = size_t(16) << 20;
__device__ __align__(256) unsigned char scratch[kFlashScratchBytes];

std::mutex scratch_mutex;
std::map<int, void *> scratch_address;  // device -> its copy of `scratch` (device address)

// The device address of the current device's `scratch`, looked up once per device. The array's name is a
// host-side stand-in, never passed to a kernel or a copy itself.
int scratch_of_current(void **out) {
    int dev = -1;
    if (check(hipGetDevice(&dev), "hipGetDevice")) return 1;
    std::lock_guard<std::mutex> lock(scratch_mutex);
    auto it = scratch_address.find(dev);
    if (it == scratch_address.end()) {
        void *ptr = nullptr;
        if (check(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)")) return 1;
        it = scratch_address.emplace(dev, ptr).first;
    }
    *out = it->second;
    return 0;
}

}  // namespace

namespace nhip {

// How flash_split_kernel would divide a forward's keys, and the time of that in quarters of a 64-key tile's time in
// flash_fwd_kernel (1.5 us). A wave's 32-key tile takes three of them, a workgroup's start and end ten, the
// second kernel eight; the chip holds 256 workgroups at head dim 128, 512 at 64.
struct Split {
    int64_t splits, cost;
};

static Split best_split(const nhip_attn_desc *d, int64_t units, int64_t keytiles) {
    const int64_t slots = kernel_dim(d) == 64 ? 512 : 256;
    Split best{1, INT64_MAX};
    for (int64_t s = 1; s <= 64 && (s == 1 || keytiles >= 8 * s); ++s) {
        const int64_t rounds = (units * s + slots - 1) / slots;
        const int64_t cost = rounds * (3 * ((keytiles + 4 * s - 1) / (4 * s)) + 10) + (s > 1 ? 8 : 0);
        if (cost < best.cost) best = {s, cost};
    }
    return best;
}

static nhipk::SplitParams split_params(const nhip_attn_desc *d, int64_t *cost) {
    nhipk::SplitParams sp{};
    sp.rows = d->heads / d->kv_heads * d->sq;
    sp.tiles = (sp.rows + 31) / 32;
    const int64_t keytiles = (d->sk + 31) / 32;
    const Split s = best_split(d, d->batch * d->kv_heads * sp.tiles, keytiles);
    sp.keytiles = (keytiles + s.splits - 1) / s.splits;
    sp.splits = (keytiles + sp.keytiles - 1) / sp.keytiles;
    if (cost) *cost = s.cost;
    return sp;
}

// Where flash_fwd_kernel would clearly take longer: its longest workgroup, every key, or where they are more than the
// chip holds (two a CU, three at head dim 64) their total. Dividing the keys shares a tile of them between fewer
// queries, so it has to be the faster by a third, less a small constant that few keys gain. Of 900 measured shapes
// where a division's cost is below that time, this keeps 832, one of which the division slows by more than 5% (10%); of
// the others, 36 (to 1.8 times). us of flash_fwd_kernel and this (batch, queries, keys, heads / key heads, head dim): 16, 1,
// 4096, 16 / 16, 128: 151, 97 (5.5 TB/s); 1, 1, 4096, 16 / 16, 128: 109, 20; 3, 1, 27958, 16 / 16, 128: 923, 126; 21, 1,
// 963, 32 / 8, 64: 38, 15; 1, 1000, 1000, 4 / 1, 64: 22, 15. Not: 2, 8310, 8310, 4 / 1, 40: 165, 301; 26, 599, 1661,
// 4 / 1, 40: 51, 77; 2, 317, 21981, 32 / 32, 96: 532, 730; 4, 512, 512, 8 / 8, 128: 18, 23.
bool split_keys(const nhip_attn_desc *d) {
    if (d->config >= 0 || kernel_dim(d) > 128 || d->sk == 0) return false;
    int64_t cost;
    split_params(d, &cost);
    const int64_t slots = kernel_dim(d) == 64 ? 768 : 512;
    const int64_t whole = 4 * ((d->sk + 63) / 64) * std::max(slots, (d->sq + 127) / 128 * d->heads * d->batch) / slots;
    return cost < whole && 3 * cost < 2 * whole + 40;
}

static size_t fwd_workspace_bytes(const nhip_attn_desc *d) {
    if (!split_keys(d)) return 0;
    const nhipk::SplitParams sp = split_params(d, nullptr);
    if (sp.splits < 2) return 0;
    const size_t rows = size_t(d->batch) * d->kv_heads * sp.tiles * sp.splits * std::min<int64_t>(32, sp.rows);
    return rows * (value_head_dim(d) * sizeof(float) + sizeof(float2));
}

template <int D, bool F16, bool CAUSAL>
static int launch_split_kernel(hipStream_t s, const nhipk::AttnParams &p, const nhip_attn_desc *d, nhipk::SplitParams sp,
                               void *ws) {
    const int64_t units = d->batch * d->kv_heads * sp.tiles;
    if (sp.splits > 1 && ws) {
        const int64_t rows = units * sp.splits * std::min<int64_t>(32, sp.rows);
        sp.sums = static_cast<float *>(ws);
        sp.stats = reinterpret_cast<float2 *>(sp.sums + rows * p.hdv);
    } else {
        sp.splits = 1;
        sp.keytiles = (d->sk + 31) / 32;
    }
    hipLaunchKernelGGL((nhipk::flash_split_kernel<D, F16, CAUSAL>), dim3(unsigned(units * sp.splits)), dim3(256), 0, s, p, sp);
    if (check(hipGetLastError(), "flash split launch")) return 1;
    if (sp.splits == 1) return 0;
    hipLaunchKernelGGL((nhipk::flash_combine_kernel<F16>), dim3(unsigned((d->batch * d->kv_heads * sp.rows + 3) / 4)),
                       dim3(256), 0, s, p, sp);
    return check(hipGetLastError(), "flash combine launch");
}

int launch_split(hipStream_t s, const nhipk::AttnParams &p, const nhip_attn_desc *d, void *ws) {
    const nhipk::SplitParams sp = split_params(d, nullptr);
    const bool f16 = d->dtype == NHIP_F16;
#define NHIP_SPLIT(DD)                                                                                        \
    return f16 ? (d->causal ? launch_split_kernel<DD, true, true>(s, p, d, sp, ws)                             \
                            : launch_split_kernel<DD, true, false>(s, p, d, sp, ws))                           \
               : (d->causal ? launch_split_kernel<DD, false, true>(s, p, d, sp, ws)                            \
                            : launch_split_kernel<DD, false, false>(s, p, d, sp, ws))
    if (kernel_dim(d) == 64) NHIP_SPLIT(64);
    NHIP_SPLIT(128);
#undef NHIP_SPLIT
}

}  // namespace nhip

extern "C" {

int nhip_flash_fwd(const nhip_attn_desc *desc, const void *q, const void *k, const void *v, void *o, float *lse) {
    hipStream_t s = stream_of_current();
    if (!s) return fail("no HIP stream: call nhip_set_device first");
    return flash_fwd_on(s, desc, q, k, v, o, lse, nullptr);
}

int nhip_flash_fwd_ws(const nhip_attn_desc *desc, const void *q, const void *k, const void *v, void *o, float *lse,
                      void *workspace) {
    hipStream_t s = stream_of_current();
    if (!s) return fail("no HIP stream: call nhip_set_device first");
    return flash_fwd_on(s, desc, q, k, v, o, lse, workspace);
}

int nhip_flash_fwd_workspace(const nhip_attn_desc *desc, size_t *bytes) {
    *bytes = 0;
    if (check_attn(desc, "flash attention", 256)) return 1;
    *bytes = fwd_workspace_bytes(desc);
    return 0;
}

int nhip_flash_fwd_divides_keys(const nhip_attn_desc *desc, int *divides) {
    *divides = 0;
    if (check_attn(desc, "flash attention", 256)) return 1;
    *divides = split_keys(desc);
    return 0;
}

int nhip_flash_bwd(const nhip_attn_desc *desc, const void *q, const void *k, const void *v, const void *o,
                   const void *d_o, const float *lse, void *dq, void *dk, void *dv, void *workspace) {
    hipStream_t s = stream_of_current();
    if (!s) return fail("no HIP stream: call nhip_set_device first");
    return flash_bwd_on(s, desc, q, k, v, o, d_o, lse, dq, dk, dv, workspace);
}

int nhip_attn_config_count(int *count) {
    *count = kNumAttnConfigs;
    return 0;
}

int nhip_flash_bwd_workspace(const nhip_attn_desc *desc, size_t *bytes) {
    *bytes = flash_bwd_workspace_bytes(desc);
    return 0;
}

int nhip_flash_bwd_noalloc(const nhip_attn_desc *desc, const void *q, const void *k, const void *v, const void *o,
                           const void *d_o, const float *lse, void *dq, void *dk, void *dv) {
    hipStream_t s = stream_of_current();
    if (!s) return fail("no HIP stream: call nhip_set_device first");
    const size_t need = flash_bwd_workspace_bytes(desc);
    if (need > kFlashScratchBytes)
        return fail("nhip_flash_bwd_noalloc: " + std::to_string(desc->batch * desc->heads * desc->sq) +
                    " query rows need " + std::to_string(need) + " bytes of scratch, above its " +
                    std::to_string(kFlashScratchBytes) + " (mode 2 takes " + std::to_string(kFlashScratchBytes / 8) +
                    " rows); use nhip_flash_bwd with a workspace, or deterministic = 2");
    void *ws = nullptr;
    if (scratch_of_current(&ws)) return 1;
    // every scratch word the kernels read is written first in the same call (delta and LSE by the prep
    // kernel), so nothing needs clearing between calls
    return flash_bwd_on(s, desc, q, k, v, o, d_o, lse, dq, dk, dv, ws);
}

}  // extern "C"
