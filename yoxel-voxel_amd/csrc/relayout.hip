// Breadth-first re-layout of a VoxNode tree on the GPU: the traversal records
// and LOD colours of build_gpu_tree (scene.cpp), computed from the device copy
// of the node array that yx_renderer_update_scene keeps in sync page by page
// (CudaSVO::Update, reaction/report/main.tex:69-71).
//
// Level by level, one thread per node of the level:
//   visit:  its present children (leaves + non-null node ids), with the id
//           checks of the host re-layout (id in range, no node reached twice);
//   totals: the blocks' sums scanned by one block, which also lays down the
//           next level's place and size in a device table;
//   gather: every node's first child record and the place of its node children
//           in the next level's list, and that list's ids and record indices.
// The level sizes stay on the device: the host enqueues levels ahead (a level
// beyond the last has no nodes) and waits once for all of them where it guesses
// their number right, instead of once per level. The top levels, which fill no
// compute unit, run in one workgroup.
// Then, from the bottom up, every level writes its node records, its leaves'
// records and the mean colours, from the sums of the level below. Integer work
// throughout: the result equals the host re-layout bit for bit.
// Bound by the bytes of the node array, 40 a node read three times.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <new>
#include <vector>

#include "internal.h"
#include "prims.h"

#define RL_HIP(call)                                                                           \
    do {                                                                                       \
        hipError_t e_ = (call);                                                                \
        if (e_ != hipSuccess) return fail(YX_ERR_HIP, "%s: %s", #call, hipGetErrorString(e_)); \
    } while (0)

namespace yx {

namespace {

constexpr uint32_t kNull = 0x80000000u;

constexpr int kTopLevels = 4;          // levels 0..3 (at most 8^3 nodes) in one workgroup
constexpr int kLevels = kMaxDepth + 2;  // table entries: levels 0..kMaxDepth, and one after the last
constexpr uint32_t kParts = 2048;       // blocks of a level's visit and gather, two per thread of the totals

// One level in the device table. Errors are kept by level, so that the first
// one is reported as a walk level by level would find it.
struct RlLevel {
    uint32_t n;           // nodes
    uint32_t off;         // their place in the node lists
    uint32_t first_rec;   // first record of their children
    uint32_t child_nodes; // node children
    uint64_t child_recs;  // children
    uint32_t bad_id;      // 1 + the largest child id >= number of nodes
    uint32_t shared;      // 1 + the largest id of a node reached twice
    uint32_t too_deep;    // children below the last level that may have some
    uint32_t too_many;    // records beyond 2^32
    uint32_t pad[2];
};

struct RlTable {
    RlLevel lv[kLevels];
};

// The node lists of all levels, laid end to end.
struct RlLists {
    const uint32_t* vox;
    uint32_t nn, root;
    uint32_t* ids;     // canonical ids
    uint32_t* rec;     // their record indices
    uint32_t* first;   // first child record
    uint32_t* noff;    // place of the first node child in the next level
    uint16_t* mask;    // leaf mask | node child mask << 8
    uint32_t* claim;   // per node id: the list position and slot (position << 3 | slot) that names it
    uint2* parts;      // per block of a level: children, node children; then their exclusive sums
    RlTable* table;
};

// A node's 10 words, as the 8-byte words that its 40 bytes are aligned to.
__device__ __forceinline__ void rl_load(const uint32_t* vox, uint32_t id, uint32_t v[10]) {
    const uint2* w = reinterpret_cast<const uint2*>(vox) + (size_t)id * 5;
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        const uint2 x = w[k];
        v[2 * k] = x.x;
        v[2 * k + 1] = x.y;
    }
}

// Children of list position p (in the level that starts at `off`). Every node
// child is claimed by the slot that names it: a claim by a slot of an earlier
// level that does name it (whatever the array held before this call, so it is
// never cleared) means that the node is reached again; two claims of one level
// are found by the gather, where one of them no longer holds. Plain loads and
// stores: an atomic exchange per node ran at 20 G/s and took most of the walk.
__device__ __forceinline__ uint2 rl_visit(const RlLists& r, RlLevel* lv, uint32_t off, uint32_t p) {
    uint32_t v[10];
    rl_load(r.vox, r.ids[p], v);
    const uint32_t lm = v[0] & 0xffu;
    uint32_t cm = 0;
#pragma unroll
    for (uint32_t c = 0; c < 8; ++c) {
        const uint32_t ch = v[2 + c];
        if (((lm >> c) & 1u) || (ch & kNull)) continue;
        if (ch >= r.nn) {
            atomicMax(&lv->bad_id, ch + 1u);
            continue;
        }
        const uint32_t old = r.claim[ch], q = old >> 3;
        r.claim[ch] = (p << 3) | c;
        bool again = ch == r.root;
        if (q < off) {
            const uint32_t* w = r.vox + (size_t)r.ids[q] * 10;
            again = again || (w[2 + (old & 7u)] == ch && !((w[0] >> (old & 7u)) & 1u));
        }
        if (again) atomicMax(&lv->shared, ch + 1u);
        cm |= 1u << c;
    }
    r.mask[p] = (uint16_t)(lm | (cm << 8));
    return make_uint2((uint32_t)__popc(lm | cm), (uint32_t)__popc(cm));
}

// Places of the children of list position p, from the exclusive sums before it.
__device__ __forceinline__ void rl_place(const RlLists& r, RlLevel* lv, uint32_t p, uint32_t recs, uint32_t nodes) {
    const uint32_t m = r.mask[p], lm = m & 0xffu, cm = m >> 8;
    const uint32_t first = lv->first_rec + recs;
    r.first[p] = first;
    r.noff[p] = nodes;
    if (cm == 0) return;
    uint32_t v[10];
    rl_load(r.vox, r.ids[p], v);
    uint32_t at = lv->off + lv->n + nodes, k = 0;
#pragma unroll
    for (uint32_t c = 0; c < 8; ++c) {
        if ((cm >> c) & 1u) {
            const uint32_t ch = v[2 + c];
            if (r.claim[ch] != ((p << 3) | c)) atomicMax(&lv->shared, ch + 1u);
            if (at < r.nn) {  // more only when some node is reached twice
                r.ids[at] = ch;
                r.rec[at] = first + k;
            }
            ++at;
        }
        k += ((lm | cm) >> c) & 1u;
    }
}

// The level's sums are known: the next level's entry, or none after an error
// (one found by the gather before counts too).
__device__ __forceinline__ void rl_next(RlLevel* lv, int l, uint32_t nn, uint64_t recs, uint32_t nodes) {
    lv[l].child_recs = recs;
    lv[l].child_nodes = nodes;
    lv[l].too_deep = recs > 0 && l + 1 > kMaxDepth ? 1u : 0u;
    const uint64_t total = (uint64_t)lv[l].first_rec + recs;
    lv[l].too_many = total + 8 > 0xFFFFFFF0ull ? 1u : 0u;
    const bool stop = lv[l].bad_id || lv[l].shared || (l > 0 && lv[l - 1].shared) || lv[l].too_deep || lv[l].too_many;
    RlLevel nx = {};
    nx.off = lv[l].off + lv[l].n;
    nx.n = stop ? 0u : min(nodes, nn - nx.off);
    nx.first_rec = (uint32_t)total;
    lv[l + 1] = nx;
}

__device__ __forceinline__ uint64_t rl_pack(uint2 v) { return ((uint64_t)v.y << 32) | v.x; }

// Levels 0 .. kTopLevels - 1 by one workgroup: a level's visits, a barrier,
// then its places in rounds of 1024 nodes with a running sum.
__global__ __launch_bounds__(1024) void rl_top_kernel(RlLists r) {
    __shared__ uint64_t shw[1024 / 64];
    RlLevel* lv = r.table->lv;
    if (threadIdx.x == 0) {
        RlLevel top = {};
        top.n = 1;
        top.first_rec = 1;
        lv[0] = top;
        r.ids[0] = r.root;
        r.rec[0] = 0;
    }
    __syncthreads();
    for (int l = 0; l < kTopLevels; ++l) {
        const uint32_t n = lv[l].n, off = lv[l].off;
        uint64_t sum = 0, total = 0;
        for (uint32_t i = threadIdx.x; i < n; i += 1024u) sum += rl_pack(rl_visit(r, lv + l, off, off + i));
        (void)block_excl_scan<uint64_t, 1024>(sum, shw, total);
        if (threadIdx.x == 0) rl_next(lv, l, r.nn, total & 0xFFFFFFFFull, (uint32_t)(total >> 32));
        __syncthreads();
        uint64_t carry = 0;
        for (uint32_t base = 0; base < n; base += 1024u) {
            const uint32_t i = base + threadIdx.x;
            uint64_t mine = 0, all = 0;
            if (i < n) {
                const uint32_t m = r.mask[off + i];
                mine = rl_pack(make_uint2((uint32_t)__popc((m | (m >> 8)) & 0xffu), (uint32_t)__popc(m >> 8)));
            }
            const uint64_t ex = carry + block_excl_scan<uint64_t, 1024>(mine, shw, all);
            if (i < n) rl_place(r, lv + l, off + i, (uint32_t)ex, (uint32_t)(ex >> 32));
            carry += all;
        }
        __syncthreads();
    }
}

// Block b of nb takes the run [b * per, (b + 1) * per) of the level's nodes.
__device__ __forceinline__ uint32_t rl_run(uint32_t n, uint32_t& begin) {
    const uint32_t per = ((n + gridDim.x - 1) / gridDim.x + 255u) & ~255u;
    begin = min(blockIdx.x * per, n);
    return min(begin + per, n);
}

__global__ __launch_bounds__(256) void rl_visit_kernel(RlLists r, int l) {
    __shared__ uint64_t shw[256 / 64];
    RlLevel* lv = r.table->lv + l;
    const uint32_t n = lv->n, off = lv->off;
    if (n == 0) return;
    uint32_t begin;
    const uint32_t end = rl_run(n, begin);
    uint64_t sum = 0, total = 0;
    for (uint32_t i = begin + threadIdx.x; i < end; i += 256u) sum += rl_pack(rl_visit(r, lv, off, off + i));
    (void)block_excl_scan<uint64_t, 256>(sum, shw, total);
    if (threadIdx.x == 0) r.parts[blockIdx.x] = make_uint2((uint32_t)total, (uint32_t)(total >> 32));
}

__global__ __launch_bounds__(kParts / 2) void rl_totals_kernel(RlLists r, int l, uint32_t nb) {
    __shared__ uint64_t shw[kParts / 2 / 64];
    RlLevel* lv = r.table->lv;
    const uint32_t n = lv[l].n;
    const uint32_t t = threadIdx.x * 2u;
    const uint2 none = make_uint2(0u, 0u);
    const uint2 p = n && t < nb ? r.parts[t] : none, q = n && t + 1u < nb ? r.parts[t + 1u] : none;
    uint64_t recs, nodes;
    const uint64_t er = block_excl_scan<uint64_t, (int)kParts / 2>((uint64_t)p.x + q.x, shw, recs);
    const uint64_t en = block_excl_scan<uint64_t, (int)kParts / 2>((uint64_t)p.y + q.y, shw, nodes);
    if (n && t < nb) r.parts[t] = make_uint2((uint32_t)er, (uint32_t)en);
    if (n && t + 1u < nb) r.parts[t + 1u] = make_uint2((uint32_t)er + p.x, (uint32_t)en + p.y);
    if (threadIdx.x == 0) rl_next(lv, l, r.nn, recs, (uint32_t)nodes);
}

__global__ __launch_bounds__(256) void rl_gather_kernel(RlLists r, int l) {
    __shared__ uint64_t shw[256 / 64];
    RlLevel* lv = r.table->lv + l;
    const uint32_t n = lv->n, off = lv->off;
    uint32_t begin;
    const uint32_t end = rl_run(n, begin);
    if (begin >= end) return;
    const uint2 carry0 = r.parts[blockIdx.x];
    uint32_t recs = carry0.x, nodes = carry0.y;
    for (uint32_t base = begin; base < end; base += 256u) {
        const uint32_t i = base + threadIdx.x;
        uint64_t mine = 0, all = 0;
        if (i < end) {
            const uint32_t m = r.mask[off + i];
            mine = rl_pack(make_uint2((uint32_t)__popc((m | (m >> 8)) & 0xffu), (uint32_t)__popc(m >> 8)));
        }
        const uint64_t ex = block_excl_scan<uint64_t, 256>(mine, shw, all);
        if (i < end) rl_place(r, lv, off + i, recs + (uint32_t)ex, nodes + (uint32_t)(ex >> 32));
        recs += (uint32_t)all;
        nodes += (uint32_t)(all >> 32);
    }
}

// Channel sums and leaf count of a subtree, as the level above reads them:
// in one 64-bit word up to 64 leaves (4 x 14 bits of at most 64 * 255, then 8
// bits), as 32-bit words up to 8^8 leaves (255 * 8^8 < 2^32), then as 64-bit
// ones. Most nodes hold leaves only, so most sums are 8 bytes.
struct SumsPacked {
    uint64_t w;
    template <class T>
    __device__ void add_to(T acc[5]) const {
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[q] += (T)((w >> (14 * q)) & 0x3FFFu);
        acc[4] += (T)(w >> 56);
    }
    template <class T>
    __device__ void set(const T acc[5]) {
        w = (uint64_t)acc[4] << 56;
#pragma unroll
        for (int q = 0; q < 4; ++q) w |= (uint64_t)acc[q] << (14 * q);
    }
};

template <class S>
struct SumsPlain {
    S v[5];
    template <class T>
    __device__ void add_to(T acc[5]) const {
#pragma unroll
        for (int q = 0; q < 5; ++q) acc[q] += (T)v[q];
    }
    template <class T>
    __device__ void set(const T acc[5]) {
#pragma unroll
        for (int q = 0; q < 5; ++q) v[q] = (S)acc[q];
    }
};

// Records, leaf records and mean colours of one level's n nodes, which start
// at list position off; `below` holds the sums of the next level's nodes. T:
// what this level's sums need.
template <class T, class In, class Out>
__global__ __launch_bounds__(256) void rl_emit_kernel(RlLists r, uint32_t off, uint32_t n, const In* __restrict__ below,
                                                      Out* __restrict__ sums, uint2* __restrict__ recs,
                                                      uint32_t* __restrict__ lod) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= n) return;
    const uint32_t p = off + i, id = r.ids[p], m = r.mask[p], lm = m & 0xffu, cm = m >> 8;
    uint32_t v[10];
    rl_load(r.vox, id, v);
    const uint32_t at = r.rec[p], first = r.first[p];
    T acc[5] = {0, 0, 0, 0, 0};
    uint32_t j = cm ? r.noff[p] : 0u, k = first;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        if ((lm >> c) & 1u) {
            const uint32_t ch = v[2 + c];
            recs[k] = make_uint2(ch, id);
            lod[k] = ch;
            ++k;
#pragma unroll
            for (int q = 0; q < 4; ++q) acc[q] += (ch >> (8 * q)) & 0xffu;
            acc[4] += 1;
        } else if ((cm >> c) & 1u) {
            ++k;
            below[j++].add_to(acc);
        }
    }
    recs[at] = (lm | cm) ? make_uint2(first, cm | (lm << 8)) : make_uint2(0u, 0u);
    sums[i].set(acc);
    uint32_t mean = 0;
    if (acc[4] > 0)
#pragma unroll
        for (int q = 0; q < 4; ++q) mean |= (uint32_t)((acc[q] + acc[4] / 2) / acc[4]) << (8 * q);
    lod[at] = mean;
}

inline dim3 rl_grid(uint64_t n) { return dim3((unsigned)((n + 255u) / 256u)); }

template <class T>
int rl_grow(T** p, size_t* cap, size_t need, const char* what) {
    if (need <= *cap && *p) return YX_OK;
    if (*p) (void)hipFree(*p);
    *p = nullptr;
    *cap = 0;
    if (hipMalloc((void**)p, std::max<size_t>(need, 1) * sizeof(T)) != hipSuccess) {
        *p = nullptr;
        return fail(YX_ERR_OOM, "hipMalloc(%zu) for %s", need * sizeof(T), what);
    }
    *cap = need;
    return YX_OK;
}

}  // namespace

// Device workspace of the re-layout, kept between calls: node-sized arrays
// (level lists laid end to end), the subtree sums of the widest level, the
// level table and a pinned host copy of it. 22 bytes a node.
struct RelayoutWork {
    size_t cap = 0, cap_wide = 0;
    uint32_t *claim = nullptr, *ids = nullptr, *rec = nullptr, *first = nullptr, *noff = nullptr;
    uint16_t* mask = nullptr;
    uint64_t *sa = nullptr, *sb = nullptr;
    uint2* parts = nullptr;
    RlTable* table = nullptr;
    RlTable* h_table = nullptr;  // pinned
    int levels = 0;              // levels with nodes of the last tree: how many to enqueue at first
    ~RelayoutWork() {
        for (void* p : {(void*)claim, (void*)ids, (void*)rec, (void*)first, (void*)noff, (void*)mask, (void*)sa,
                        (void*)sb, (void*)parts, (void*)table})
            if (p) (void)hipFree(p);
        if (h_table) (void)hipHostFree(h_table);
    }
};

RelayoutWork* relayout_work_create() { return new (std::nothrow) RelayoutWork(); }
void relayout_work_free(RelayoutWork* w) { delete w; }

int gpu_relayout(const uint32_t* d_vox, uint32_t nn, uint32_t root, void* stream, RelayoutWork* w,
                 uint32_t** recs_io, uint32_t** lod_io, size_t* cap_io, GpuLayout& out) {
    const hipStream_t st = (hipStream_t)stream;
    out = GpuLayout();
    if (!w) return fail(YX_ERR_INVALID_ARG, "no re-layout workspace");
    if (root & kNull) return YX_OK;  // EmptyNode / FullNode root: nothing to hit
    if (root >= nn) return fail(YX_ERR_FORMAT, "root id %u out of range (%u nodes)", root, nn);
    if (nn >= (1u << 29)) return fail(YX_ERR_RANGE, "at most 2^29 nodes");
    int rc;
    if (w->cap < nn) {
        size_t c = 0;
        for (uint32_t** p : {&w->claim, &w->ids, &w->rec, &w->first, &w->noff}) {
            c = w->cap;
            if ((rc = rl_grow(p, &c, nn, "the re-layout workspace")) != YX_OK) {
                w->cap = 0;
                return rc;
            }
        }
        c = w->cap;
        if ((rc = rl_grow(&w->mask, &c, nn, "the re-layout workspace")) != YX_OK) {
            w->cap = 0;
            return rc;
        }
        w->cap = nn;
    }
    if (!w->h_table) {
        size_t c = 0;
        if ((rc = rl_grow(&w->parts, &c, kParts, "block sums")) != YX_OK) return rc;
        c = 0;
        if ((rc = rl_grow(&w->table, &c, 1, "the level table")) != YX_OK) return rc;
        if (hipHostMalloc((void**)&w->h_table, sizeof(RlTable), hipHostMallocDefault) != hipSuccess) {
            w->h_table = nullptr;
            return fail(YX_ERR_OOM, "pinned host memory for the re-layout");
        }
    }
    RlLists r;
    r.vox = d_vox;
    r.nn = nn;
    r.root = root;
    r.ids = w->ids;
    r.rec = w->rec;
    r.first = w->first;
    r.noff = w->noff;
    r.mask = w->mask;
    r.claim = w->claim;
    r.parts = w->parts;
    r.table = w->table;
    hipLaunchKernelGGL(rl_top_kernel, dim3(1), dim3(1024), 0, st, r);
    RL_HIP(hipGetLastError());
    // levels enqueued up to `upto`, then one wait for the table; a tree as deep
    // as the last one needs no other
    const RlLevel* lv = w->h_table->lv;
    int l = kTopLevels, upto = w->levels > 0 ? w->levels : kTopLevels + 4;
    for (;;) {
        upto = std::min(upto, kMaxDepth + 1);
        for (; l < upto; ++l) {
            const uint64_t most = std::min<uint64_t>(nn, l < 10 ? (uint64_t)1 << (3 * l) : nn);
            const uint32_t nb = (uint32_t)std::min<uint64_t>(kParts, (most + 255) / 256);
            hipLaunchKernelGGL(rl_visit_kernel, dim3(nb), dim3(256), 0, st, r, l);
            hipLaunchKernelGGL(rl_totals_kernel, dim3(1), dim3(kParts / 2), 0, st, r, l, nb);
            hipLaunchKernelGGL(rl_gather_kernel, dim3(nb), dim3(256), 0, st, r, l);
            RL_HIP(hipGetLastError());
        }
        RL_HIP(hipMemcpyAsync(w->h_table, w->table, sizeof(RlTable), hipMemcpyDeviceToHost, st));
        RL_HIP(hipStreamSynchronize(st));
        if (l > kMaxDepth || lv[l].n == 0) break;
        upto = l + 4;
    }
    uint64_t total = 1;  // records (the root's first)
    int depth = 0;
    uint32_t widest = 1;
    size_t levels = 0;  // levels with nodes
    std::vector<uint32_t> level_records(1, 1u);
    for (int q = 0; q < l && lv[q].n > 0; ++q) {
        if (lv[q].bad_id)
            return fail(YX_ERR_FORMAT, "child id %u out of range (%u nodes)", lv[q].bad_id - 1u, nn);
        if (lv[q].shared) return fail(YX_ERR_FORMAT, "node %u reached twice (not a tree)", lv[q].shared - 1u);
        if (lv[q].too_deep) return fail(YX_ERR_RANGE, "tree deeper than %d levels", kMaxDepth);
        if (lv[q].child_recs > lv[q].child_nodes) depth = q + 1;  // some child is a leaf
        if (lv[q].too_many) return fail(YX_ERR_RANGE, "more than 2^32 records");
        total += lv[q].child_recs;
        level_records.push_back((uint32_t)total);
        widest = std::max(widest, lv[q].n);
        ++levels;
    }
    w->levels = (int)levels;
    if (depth == 0) return YX_OK;  // no leaf anywhere: nothing to hit

    // bottom-up subtree sums: two buffers of 5 u64 per node of the widest level
    if (w->cap_wide < widest) {
        // growing frees first, so there is none until both have grown
        w->cap_wide = 0;
        for (uint64_t** p : {&w->sa, &w->sb}) {
            size_t c = 0;
            if ((rc = rl_grow(p, &c, (size_t)widest * 5, "subtree sums")) != YX_OK) return rc;
        }
        w->cap_wide = widest;
    }

    // the caller's record arrays, grown only when too small, and last: after a
    // failure the caller goes on with the records that it has
    if (*cap_io < total || !*recs_io || !*lod_io) {
        uint32_t *nr = nullptr, *nl = nullptr;
        if (hipMalloc((void**)&nr, total * 8u) != hipSuccess)
            return fail(YX_ERR_OOM, "hipMalloc(%zu) for the records", (size_t)(total * 8u));
        if (hipMalloc((void**)&nl, total * 4u) != hipSuccess) {
            (void)hipFree(nr);
            return fail(YX_ERR_OOM, "hipMalloc(%zu) for the LOD colours", (size_t)(total * 4u));
        }
        if (*recs_io) (void)hipFree(*recs_io);
        if (*lod_io) (void)hipFree(*lod_io);
        *recs_io = nr;
        *lod_io = nl;
        *cap_io = (size_t)total;
    }
    uint2* d_recs = reinterpret_cast<uint2*>(*recs_io);
    uint32_t* d_lod = *lod_io;
    uint64_t *sa = w->sa, *sb = w->sb;
    for (int q = (int)levels; q-- > 0;) {
        // a level's nodes are this many levels above the leaves at most
        const int height = (int)levels - q;
        const uint32_t off = lv[q].off, n = lv[q].n;
#define RL_EMIT(T, IN, OUT)                                                                                     \
    hipLaunchKernelGGL((rl_emit_kernel<T, IN, OUT>), rl_grid(n), dim3(256), 0, st, r, off, n, (const IN*)sb, \
                       (OUT*)sa, d_recs, d_lod)
        if (height <= 2)
            RL_EMIT(uint32_t, SumsPacked, SumsPacked);
        else if (height == 3)
            RL_EMIT(uint32_t, SumsPacked, SumsPlain<uint32_t>);
        else if (height <= 8)
            RL_EMIT(uint32_t, SumsPlain<uint32_t>, SumsPlain<uint32_t>);
        else if (height == 9)
            RL_EMIT(uint64_t, SumsPlain<uint32_t>, SumsPlain<uint64_t>);
        else
            RL_EMIT(uint64_t, SumsPlain<uint64_t>, SumsPlain<uint64_t>);
#undef RL_EMIT
        RL_HIP(hipGetLastError());
        std::swap(sa, sb);
    }
    RL_HIP(hipStreamSynchronize(st));
    out.recs = *recs_io;
    out.lod = *lod_io;
    out.n_recs = (size_t)total;
    out.depth = depth;
    out.node_levels = (int)levels;
    out.level_records = level_records;
    out.empty = false;
    return YX_OK;
}

}  // namespace yx
