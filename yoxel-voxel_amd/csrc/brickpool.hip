// Brick pool manager for brick volumes (the compositing volume's brick table +
// per-slot parameters): CuBrickPoolManager::allocMap
// (reaction/voxtree/brickpool/BrickPool.cpp:21-62) and UpdateBrickPool
// (reaction/voxtree/density.cu:240-284), on the GPU.
//
// The pool manages arrays its caller owns (yx_volume_dev: the int32 brick
// table and the float4 parameters of `num_slots` slots). The reference
// allocates from the least-filled slices of a 3D texture and enumerates the
// mapped bricks in request order; here the pool is one linear HBM array and
// the policy is: the bricks of a request that have no slot, in order of their
// first appearance in the list, get the lowest free slots in increasing order.
// Allocation runs as claim (atomicMin of the list position per brick) and free
// slots as bit masks -> new bricks as bit masks -> a scan over either's bit
// counts -> assign, so the result does not depend on thread timing.
//
// A call is a few launches of a few microseconds each, so what bounds it is
// their number and the waits of the host. Claims carry the call's number
// (later calls' claims are smaller), so nothing is cleared between calls; what
// the host must know is written to pinned memory by the kernels, and it waits
// once, for the last kernel that writes there; a kernel that must not run after
// a failed check reads the check itself. An update's copy is enqueued before
// the wait for its check and runs on behind the host. Two releases, allocations
// and updates of 2,621 of 26,214 bricks: 410 us with cleared arrays and a wait
// for every count, 162 with one wait for each call's whole work, 143 so; with
// an allocation's assignment behind the host too, 173 (another event to record
// for a kernel of a few microseconds).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <new>

#include "internal.h"
#include "prims.h"

#define BP_HIP(call)                                                                           \
    do {                                                                                       \
        hipError_t e_ = (call);                                                                \
        if (e_ != hipSuccess) return fail(YX_ERR_HIP, "%s: %s", #call, hipGetErrorString(e_)); \
    } while (0)

namespace yx {
namespace {

// Device-side state between the kernels of a call.
struct BpState {
    uint32_t bad;       // creation: a slot referenced twice / out of range; else the last call with a bad index
    uint32_t released;  // slots freed so far by a release
    uint32_t blocks;    // blocks of a release that are done
    uint32_t want, have;  // new bricks and free slots of an allocation
};

// What a call tells the host (pinned memory).
struct BpResult {
    uint32_t bad;  // the last call with a bad index
    uint32_t released;
    uint32_t want, have;
};

// A claim of list position `pos` in call `call`: smaller than any earlier call's.
__device__ __forceinline__ uint64_t bp_claim(uint32_t call, uint32_t pos) { return (uint64_t)~call << 32 | pos; }

__global__ void bp_init_used_kernel(const int32_t* __restrict__ table, uint32_t nb, uint32_t cap,
                                    uint32_t* __restrict__ used, BpState* state) {
    const uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nb) return;
    const int32_t s = table[b];
    if (s < 0) return;
    if ((uint32_t)s >= cap || atomicExch(&used[s], 1u) != 0u) atomicOr(&state->bad, 1u);
}

__global__ void bp_fill_kernel(uint32_t* __restrict__ p, uint32_t n, uint32_t v) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// The first blocks claim the listed bricks - FIRST: for the first position that
// lists a brick, else for the last one, which an update writes - and, in an
// allocation, the others write the free slots as masks of 64.
template <bool FIRST>
__global__ __launch_bounds__(256) void bp_claim_kernel(const int32_t* __restrict__ bricks, uint32_t n, uint32_t nb,
                                                       uint32_t call, uint64_t* __restrict__ claim, BpState* state,
                                                       BpResult* result, const uint32_t* __restrict__ used,
                                                       uint32_t cap, uint64_t* __restrict__ free_mask) {
    const uint32_t list_blocks = (n + 255u) / 256u;
    if (blockIdx.x >= list_blocks) {
        const uint32_t j = (blockIdx.x - list_blocks) * 256u + threadIdx.x;
        const uint64_t mask = __ballot(j < cap && used[j] == 0u);
        if ((j & 63u) == 0u && j < cap) free_mask[j >> 6] = mask;
        return;
    }
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= n) return;
    const int32_t b = bricks[i];
    if (b < 0 || (uint32_t)b >= nb) {
        state->bad = call;
        result->bad = call;
        return;
    }
    atomicMin((unsigned long long*)&claim[b], (unsigned long long)bp_claim(call, FIRST ? i : n - 1u - i));
}

// The list's new bricks as masks of 64: first in the list, without a slot.
__global__ __launch_bounds__(256) void bp_new_kernel(const int32_t* __restrict__ bricks, uint32_t n, uint32_t nb,
                                                     uint32_t call, const uint64_t* __restrict__ claim,
                                                     const int32_t* __restrict__ table,
                                                     uint64_t* __restrict__ new_mask) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    bool fresh = false;
    if (i < n) {
        const int32_t b = bricks[i];
        fresh = b >= 0 && (uint32_t)b < nb && claim[b] == bp_claim(call, i) && table[b] < 0;
    }
    const uint64_t mask = __ballot(fresh);
    if ((i & 63u) == 0u && i < n) new_mask[i >> 6] = mask;
}

// Position of set bit number k (from 0) of a mask with more than k set bits.
__device__ __forceinline__ uint32_t bp_select(uint64_t mask, uint32_t k) {
    uint32_t at = 0;
#pragma unroll
    for (uint32_t half = 32u; half != 0u; half >>= 1) {
        const uint32_t low = (uint32_t)__popcll(mask >> at & ((1ull << half) - 1ull));
        if (k >= low) {
            k -= low;
            at += half;
        }
    }
    return at;
}

// The new brick of rank r gets free slot number r: the mask of 64 slots that
// holds it is found in the scan of their bit counts. A brick listed again takes
// its claimant's rank, whether its table entry is written yet or not.
__global__ __launch_bounds__(256) void bp_assign_kernel(const int32_t* __restrict__ bricks, uint32_t n, uint32_t call,
                                                        const uint64_t* __restrict__ claim,
                                                        const uint64_t* __restrict__ new_mask,
                                                        const uint32_t* __restrict__ new_before,
                                                        const uint64_t* __restrict__ free_mask,
                                                        const uint32_t* __restrict__ free_before, uint32_t free_masks,
                                                        int32_t* table, uint32_t* __restrict__ used,
                                                        int32_t* __restrict__ slots_out, const BpState* state,
                                                        BpResult* result) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    const uint32_t want = state->want, have = state->have;
    if (i == 0u) {
        result->want = want;
        result->have = have;
    }
    if (i >= n || state->bad == call || want > have) return;
    const int32_t b = bricks[i];
    int32_t s = __hip_atomic_load(&table[b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t owner = (uint32_t)claim[b];
    const uint64_t mask = new_mask[owner >> 6];
    if (mask >> (owner & 63u) & 1ull) {
        const uint32_t rank =
            new_before[owner >> 6] + (uint32_t)__popcll(mask & ((1ull << (owner & 63u)) - 1ull));
        uint32_t lo = 0, hi = free_masks;  // free_before[lo] <= rank < free_before[hi]
        while (hi - lo > 1u) {
            const uint32_t mid = (lo + hi) >> 1;
            if (free_before[mid] <= rank)
                lo = mid;
            else
                hi = mid;
        }
        s = (int32_t)(lo * 64u + bp_select(free_mask[lo], rank - free_before[lo]));
        if (owner == i) {
            __hip_atomic_store(&table[b], s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            used[s] = 1u;
        }
    }
    if (slots_out) slots_out[i] = s;
}

__global__ __launch_bounds__(256) void bp_release_kernel(const int32_t* __restrict__ bricks, uint32_t n, uint32_t nb,
                                                         uint32_t call, int32_t* __restrict__ table,
                                                         uint32_t* __restrict__ used, BpState* state,
                                                         BpResult* result) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    bool freed = false;
    if (i < n) {
        const int32_t b = bricks[i];
        if (b < 0 || (uint32_t)b >= nb) {
            result->bad = call;
        } else {
            const int32_t s = atomicExch(&table[b], -1);
            freed = s >= 0;
            if (freed) used[s] = 0u;
        }
    }
    const int count = __syncthreads_count(freed);
    if (threadIdx.x == 0) {
        if (count) atomicAdd(&state->released, (uint32_t)count);
        __threadfence();
        if (atomicAdd(&state->blocks, 1u) == gridDim.x - 1u) {  // the last block
            result->released = atomicExch(&state->released, 0u);
            atomicExch(&state->blocks, 0u);
        }
    }
}

// one workgroup per listed brick: its packed voxels into its slot
__global__ __launch_bounds__(256) void bp_update_kernel(const int32_t* __restrict__ bricks, uint32_t n, uint32_t call,
                                                        const int32_t* __restrict__ table,
                                                        const uint64_t* __restrict__ claim, uint32_t vox,
                                                        const float4* __restrict__ packed,
                                                        float4* __restrict__ params, const BpState* state) {
    const uint32_t i = blockIdx.x;
    if (i >= n || state->bad == call) return;
    const int32_t b = bricks[i];
    if (claim[b] != bp_claim(call, n - 1u - i)) return;
    const int32_t s = table[b];
    if (s < 0) return;
    const float4* src = packed + (size_t)i * vox;
    float4* dst = params + (size_t)s * vox;
    for (uint32_t t = threadIdx.x; t < vox; t += blockDim.x) dst[t] = src[t];
}

inline dim3 bp_grid(uint64_t n) { return dim3((unsigned)std::max<uint64_t>(1, (n + 255u) / 256u)); }

}  // namespace
}  // namespace yx

using namespace yx;

struct yx_brick_pool {
    yx_volume_dev vol;  // caller-owned table and params
    uint32_t nb = 0;    // bricks in the table: (grid / brick)^3
    uint32_t vox = 0;   // voxels per brick
    uint32_t used_count = 0;
    uint32_t call = 0;  // number of the current call, from 1
    uint32_t* d_used = nullptr;   // [num_slots]
    uint64_t* d_claim = nullptr;  // [nb]
    BpState* d_state = nullptr;
    BpResult* h_result = nullptr;  // pinned
    hipEvent_t checked = nullptr;  // an update's check is done
    uint64_t *d_new_mask = nullptr, *d_free_mask = nullptr;      // a bit per list entry, per slot
    uint32_t *d_new_before = nullptr, *d_free_before = nullptr;  // bits before each mask
    uint32_t cap_masks = 0;  // masks of list entries
    void* scan_tmp = nullptr;
    size_t scan_bytes = 0;
    ~yx_brick_pool() {
        for (void* p : {(void*)d_used, (void*)d_claim, (void*)d_state, (void*)d_new_mask, (void*)d_free_mask,
                        (void*)d_new_before, (void*)d_free_before, scan_tmp})
            if (p) (void)hipFree(p);
        if (h_result) (void)hipHostFree(h_result);
        if (checked) (void)hipEventDestroy(checked);
    }
};

template <class T>
static int bp_alloc(T** p, size_t n) {
    if (hipMalloc((void**)p, std::max<size_t>(n, 1) * sizeof(T)) != hipSuccess) {
        *p = nullptr;
        return fail(YX_ERR_OOM, "hipMalloc(%zu) for the brick pool", n * sizeof(T));
    }
    return YX_OK;
}

static uint32_t bp_masks(uint32_t n) { return n / 64u + (n % 64u ? 1u : 0u); }

// Space for a scan or a sum of `items` items: a pool's creation sums the used
// slots themselves, the calls scan masks of 64 slots or list entries.
static int bp_scan_space(yx_brick_pool* p, uint32_t items) {
    const size_t bytes = scan_workspace_bytes(std::max(items, 1u));
    if (bytes <= p->scan_bytes) return YX_OK;
    if (p->scan_tmp) BP_HIP(hipFree(p->scan_tmp));
    p->scan_tmp = nullptr;
    p->scan_bytes = 0;
    int rc = bp_alloc((uint8_t**)&p->scan_tmp, bytes);
    if (rc != YX_OK) return rc;
    p->scan_bytes = bytes;
    return YX_OK;
}

static void bp_reset_claims(yx_brick_pool* p, hipStream_t st) {
    // two words a claim; a table has fewer than 2^31 entries
    hipLaunchKernelGGL(bp_fill_kernel, bp_grid((uint64_t)p->nb * 2u), dim3(256), 0, st, (uint32_t*)p->d_claim,
                       p->nb * 2u, 0xFFFFFFFFu);
}

// The next call's number: 1 and up, never that of a claim, a bad index or a
// result that is still around.
static uint32_t bp_next_call(yx_brick_pool* p, hipStream_t st) {
    if (++p->call == 0xFFFFFFFFu) {
        bp_reset_claims(p, st);
        hipLaunchKernelGGL(bp_fill_kernel, dim3(1), dim3(256), 0, st, &p->d_state->bad, 1u, 0u);
        p->h_result->bad = 0u;
        p->call = 1u;
    }
    return p->call;
}

extern "C" int yx_brick_pool_create(const yx_volume_dev* vol, void* stream, yx_brick_pool** out) {
    clear_error();
    if (!vol || !out || !vol->table || (!vol->params && vol->num_slots))
        return fail(YX_ERR_INVALID_ARG, "null argument");
    *out = nullptr;
    if (vol->brick < 1 || vol->grid < vol->brick || vol->grid % vol->brick)
        return fail(YX_ERR_INVALID_ARG, "grid %d must be a positive multiple of brick %d", vol->grid, vol->brick);
    const uint64_t g = (uint64_t)(vol->grid / vol->brick);
    if (g * g * g >= 0x80000000ull || (uint64_t)vol->brick * vol->brick * vol->brick > (1u << 20))
        return fail(YX_ERR_RANGE, "volume too large for the brick pool");
    if (vol->num_slots >= 0x80000000u) return fail(YX_ERR_RANGE, "at most 2^31 slots");
    const hipStream_t st = (hipStream_t)stream;
    yx_brick_pool* p = new (std::nothrow) yx_brick_pool();
    if (!p) return fail(YX_ERR_OOM, "out of host memory");
    p->vol = *vol;
    p->nb = (uint32_t)(g * g * g);
    p->vox = (uint32_t)(vol->brick * vol->brick * vol->brick);
    int rc;
    const uint32_t slot_masks = bp_masks(vol->num_slots);
    if ((rc = bp_alloc(&p->d_used, vol->num_slots)) != YX_OK || (rc = bp_alloc(&p->d_claim, p->nb)) != YX_OK ||
        (rc = bp_alloc(&p->d_state, 1)) != YX_OK || (rc = bp_alloc(&p->d_free_mask, slot_masks)) != YX_OK ||
        (rc = bp_alloc(&p->d_free_before, slot_masks)) != YX_OK ||
        (rc = bp_scan_space(p, vol->num_slots)) != YX_OK) {
        delete p;
        return rc;
    }
    if (hipHostMalloc((void**)&p->h_result, sizeof(BpResult), hipHostMallocDefault) != hipSuccess) {
        p->h_result = nullptr;
        delete p;
        return fail(YX_ERR_OOM, "hipHostMalloc(%zu) for the brick pool", sizeof(BpResult));
    }
    *p->h_result = BpResult{};
    if (hipEventCreateWithFlags(&p->checked, hipEventDisableTiming) != hipSuccess) {
        p->checked = nullptr;
        delete p;
        return fail(YX_ERR_HIP, "hipEventCreate for the brick pool");
    }
    auto give_up = [&](int code) {
        delete p;
        return code;
    };
    hipLaunchKernelGGL(bp_fill_kernel, bp_grid(vol->num_slots), dim3(256), 0, st, p->d_used, vol->num_slots, 0u);
    bp_reset_claims(p, st);
    hipLaunchKernelGGL(bp_fill_kernel, dim3(1), dim3(256), 0, st, (uint32_t*)p->d_state,
                       (uint32_t)(sizeof(BpState) / 4), 0u);
    hipLaunchKernelGGL(bp_init_used_kernel, bp_grid(p->nb), dim3(256), 0, st, vol->table, p->nb, vol->num_slots,
                       p->d_used, p->d_state);
    if (hipGetLastError() != hipSuccess) return give_up(fail(YX_ERR_HIP, "brick pool set-up launch"));
    BpState f;
    if (hipMemcpyAsync(&f, p->d_state, sizeof(f), hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess)
        return give_up(fail(YX_ERR_HIP, "brick pool set-up"));
    if (f.bad) return give_up(fail(YX_ERR_FORMAT, "brick table references a slot twice or beyond %u slots",
                                   vol->num_slots));
    // used slots: count them with a reduction over the used map
    uint32_t* d_cnt = nullptr;
    if ((rc = bp_alloc(&d_cnt, 1)) != YX_OK) return give_up(rc);
    uint32_t cnt = 0;
    const bool ok = vol->num_slots == 0 ||
                    (reduce_sum_u32(p->d_used, vol->num_slots, d_cnt, p->scan_tmp, p->scan_bytes, st) == YX_OK &&
                     hipMemcpyAsync(&cnt, d_cnt, 4, hipMemcpyDeviceToHost, st) == hipSuccess &&
                     hipStreamSynchronize(st) == hipSuccess);
    (void)hipFree(d_cnt);
    if (!ok) return give_up(fail(YX_ERR_HIP, "counting used slots"));
    p->used_count = cnt;
    *out = p;
    return YX_OK;
}

extern "C" void yx_brick_pool_destroy(yx_brick_pool* p) { delete p; }

static int ensure_list(yx_brick_pool* p, uint32_t n) {
    const uint32_t masks = bp_masks(n);
    if (masks <= p->cap_masks && p->d_new_mask && p->d_new_before) return YX_OK;
    if (p->d_new_mask) BP_HIP(hipFree(p->d_new_mask));
    p->d_new_mask = nullptr;
    if (p->d_new_before) BP_HIP(hipFree(p->d_new_before));
    p->d_new_before = nullptr;
    p->cap_masks = 0;
    int rc;
    if ((rc = bp_alloc(&p->d_new_mask, masks)) != YX_OK || (rc = bp_alloc(&p->d_new_before, masks)) != YX_OK ||
        (rc = bp_scan_space(p, masks)) != YX_OK)
        return rc;
    p->cap_masks = masks;
    return YX_OK;
}

extern "C" int yx_brick_pool_alloc(yx_brick_pool* p, const int32_t* bricks, uint32_t n, int32_t* slots_out,
                                   uint32_t* new_count, void* stream) {
    clear_error();
    if (!p || (!bricks && n)) return fail(YX_ERR_INVALID_ARG, "null argument");
    if (new_count) *new_count = 0;
    if (n == 0) return YX_OK;
    if (n >= 0x80000000u) return fail(YX_ERR_RANGE, "at most 2^31 bricks per call");
    const hipStream_t st = (hipStream_t)stream;
    int rc = ensure_list(p, n);
    if (rc != YX_OK) return rc;
    const uint32_t cap = p->vol.num_slots, call = bp_next_call(p, st);
    int32_t* table = const_cast<int32_t*>(p->vol.table);
    const uint32_t blocks = (n + 255u) / 256u, slot_blocks = cap / 256u + (cap % 256u ? 1u : 0u);
    hipLaunchKernelGGL(bp_claim_kernel<true>, dim3(blocks + slot_blocks), dim3(256), 0, st, bricks, n, p->nb, call,
                       p->d_claim, p->d_state, p->h_result, p->d_used, cap, p->d_free_mask);
    hipLaunchKernelGGL(bp_new_kernel, dim3(blocks), dim3(256), 0, st, bricks, n, p->nb, call, p->d_claim, table,
                       p->d_new_mask);
    BP_HIP(hipGetLastError());
    if ((rc = scan_excl_popc64(p->d_new_mask, p->d_new_before, bp_masks(n), &p->d_state->want, p->scan_tmp,
                               p->scan_bytes, st)) != YX_OK)
        return rc;
    if (cap && (rc = scan_excl_popc64(p->d_free_mask, p->d_free_before, bp_masks(cap), &p->d_state->have, p->scan_tmp,
                                      p->scan_bytes, st)) != YX_OK)
        return rc;
    hipLaunchKernelGGL(bp_assign_kernel, dim3(blocks), dim3(256), 0, st, bricks, n, call, p->d_claim, p->d_new_mask,
                       p->d_new_before, p->d_free_mask, p->d_free_before, bp_masks(cap), table, p->d_used, slots_out,
                       p->d_state, p->h_result);
    BP_HIP(hipGetLastError());
    BP_HIP(hipStreamSynchronize(st));
    const BpResult res = *p->h_result;
    if (res.bad == call)
        return fail(YX_ERR_RANGE, "brick index outside the %u bricks of the table", p->nb);
    if (res.want > res.have)
        return fail(YX_ERR_RANGE, "%u new bricks but %u free slots (nothing allocated)", res.want, res.have);
    p->used_count += res.want;
    if (new_count) *new_count = res.want;
    return YX_OK;
}

extern "C" int yx_brick_pool_release(yx_brick_pool* p, const int32_t* bricks, uint32_t n, uint32_t* released,
                                     void* stream) {
    clear_error();
    if (!p || (!bricks && n)) return fail(YX_ERR_INVALID_ARG, "null argument");
    if (released) *released = 0;
    if (n == 0) return YX_OK;
    const hipStream_t st = (hipStream_t)stream;
    const uint32_t call = bp_next_call(p, st);
    hipLaunchKernelGGL(bp_release_kernel, bp_grid(n), dim3(256), 0, st, bricks, n, p->nb, call,
                       const_cast<int32_t*>(p->vol.table), p->d_used, p->d_state, p->h_result);
    BP_HIP(hipGetLastError());
    BP_HIP(hipStreamSynchronize(st));
    const BpResult res = *p->h_result;
    p->used_count -= res.released;
    if (released) *released = res.released;
    if (res.bad == call)
        return fail(YX_ERR_RANGE, "brick index outside the %u bricks of the table (valid ones released)", p->nb);
    return YX_OK;
}

extern "C" int yx_brick_pool_update(yx_brick_pool* p, const int32_t* bricks, uint32_t n, const float* packed,
                                    void* stream) {
    clear_error();
    if (!p || (n && (!bricks || !packed))) return fail(YX_ERR_INVALID_ARG, "null argument");
    if (n == 0) return YX_OK;
    if (!p->vol.params) return fail(YX_ERR_INVALID_ARG, "the volume has no parameter slots");
    if (n >= 0x80000000u) return fail(YX_ERR_RANGE, "at most 2^31 bricks per call");
    const hipStream_t st = (hipStream_t)stream;
    const uint32_t call = bp_next_call(p, st);
    hipLaunchKernelGGL(bp_claim_kernel<false>, bp_grid(n), dim3(256), 0, st, bricks, n, p->nb, call, p->d_claim,
                       p->d_state, p->h_result, (const uint32_t*)nullptr, 0u, (uint64_t*)nullptr);
    BP_HIP(hipEventRecord(p->checked, st));
    hipLaunchKernelGGL(bp_update_kernel, dim3(n), dim3(256), 0, st, bricks, n, call, p->vol.table, p->d_claim, p->vox,
                       reinterpret_cast<const float4*>(packed),
                       reinterpret_cast<float4*>(const_cast<float*>(p->vol.params)), p->d_state);
    BP_HIP(hipGetLastError());
    BP_HIP(hipEventSynchronize(p->checked));
    if (p->h_result->bad == call)
        return fail(YX_ERR_RANGE, "brick index outside the %u bricks of the table (nothing copied)", p->nb);
    return YX_OK;
}

extern "C" int yx_brick_pool_stats(const yx_brick_pool* p, uint32_t* used, uint32_t* capacity) {
    clear_error();
    if (!p || !used || !capacity) return fail(YX_ERR_INVALID_ARG, "null argument");
    *used = p->used_count;
    *capacity = p->vol.num_slots;
    return YX_OK;
}
