// The host side of the GPU re-layout (csrc/relayout.hip) on the CPU: the file is
// compiled for the host alone and linked to the few HIP calls below, in which
// "device" memory is host memory, kernels are recorded instead of run, and an
// allocation can be made to fail. Checks that what the kernels are given stays
// valid after an allocation failed.
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>

#include "../../yoxel-voxel_amd/csrc/relayout.hip"

namespace {

std::map<char*, size_t> g_live;  // allocations
size_t g_fail_bytes = 0;         // fail the g_fail_nth next allocation of this size
int g_fail_nth = 0;
yx::RlTable g_table;  // what the device's level table "holds"
int g_emits = 0, g_bad = 0;

// whether [p, p + bytes) lies in a live allocation
bool valid(const void* p, size_t bytes) {
    auto it = g_live.upper_bound((char*)p);
    if (!p || it == g_live.begin()) return false;
    --it;
    return (char*)p + bytes <= it->first + it->second;
}

template <class T, class In, class Out>
bool emit_of(const void* f, void** args) {
    if (f != (const void*)yx::rl_emit_kernel<T, In, Out>) return false;
    ++g_emits;
    const uint32_t n = *(uint32_t*)args[2];
    const void* below = *(void**)args[3];
    const void* sums = *(void**)args[4];
    // the lowest level reads nothing from below, the others a word at least
    if (!valid(sums, n * sizeof(Out)) || !valid(below, 1)) ++g_bad;
    return true;
}

}  // namespace

namespace yx {
int fail(int code, const char* fmt, ...) {
    (void)fmt;
    return code;
}
}  // namespace yx

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
    if (n == g_fail_bytes && g_fail_nth > 0 && --g_fail_nth == 0) return hipErrorOutOfMemory;
    *p = std::calloc(1, n);
    g_live[(char*)*p] = n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    if (p && !g_live.erase((char*)p)) ++g_bad;
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipMemcpyAsync(void* dst, const void*, size_t n, hipMemcpyKind, hipStream_t) {
    if (n == sizeof(g_table)) std::memcpy(dst, &g_table, n);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return ""; }

static dim3 s_grid, s_block;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t, hipStream_t) {
    s_grid = g;
    s_block = b;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* shared, hipStream_t* st) {
    *g = s_grid;
    *b = s_block;
    *shared = 0;
    *st = nullptr;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t) {
    using namespace yx;
    (void)(emit_of<uint32_t, SumsPacked, SumsPacked>(f, args) ||
           emit_of<uint32_t, SumsPacked, SumsPlain<uint32_t>>(f, args) ||
           emit_of<uint32_t, SumsPlain<uint32_t>, SumsPlain<uint32_t>>(f, args) ||
           emit_of<uint64_t, SumsPlain<uint32_t>, SumsPlain<uint64_t>>(f, args) ||
           emit_of<uint64_t, SumsPlain<uint64_t>, SumsPlain<uint64_t>>(f, args));
    return hipSuccess;
}
void** __hipRegisterFatBinary(const void*) {
    static void* h;
    return &h;
}
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}
extern const char __hip_fatbin[] = "";
}

// One re-layout of a tree whose levels have 1, 8 and `wide` nodes, the last
// ones with a leaf each.
static int layout(yx::RelayoutWork* w, uint32_t nn, uint32_t wide, uint32_t** recs, uint32_t** lod, size_t* cap) {
    const uint32_t n[3] = {1, 8, wide};
    std::memset(&g_table, 0, sizeof(g_table));
    uint32_t off = 0, rec = 1;
    for (int l = 0; l < 3; ++l) {
        yx::RlLevel& q = g_table.lv[l];
        q.n = n[l];
        q.off = off;
        q.first_rec = rec;
        q.child_nodes = l < 2 ? n[l + 1] : 0;
        q.child_recs = l < 2 ? n[l + 1] : wide;
        off += n[l];
        rec += (uint32_t)q.child_recs;
    }
    static uint32_t vox[10];
    yx::GpuLayout out;
    return yx::gpu_relayout(vox, nn, 0, nullptr, w, recs, lod, cap, out);
}

int main() {
    int failed = 0;
    auto expect = [&](bool ok, const char* what) {
        if (!ok) std::printf("FAILED: %s\n", what), ++failed;
    };
    for (int nth = 1; nth <= 2; ++nth) {  // the first, then the second sums buffer cannot grow
        yx::RelayoutWork* w = yx::relayout_work_create();
        uint32_t *recs = nullptr, *lod = nullptr;
        size_t cap = 0;
        g_fail_nth = 0;
        expect(layout(w, 200, 50, &recs, &lod, &cap) == YX_OK && g_emits == 3 && !g_bad, "a first tree");
        g_fail_bytes = (size_t)90 * 5 * 8;
        g_fail_nth = nth;
        g_emits = g_bad = 0;
        uint32_t *const recs0 = recs, *const lod0 = lod;
        const size_t cap0 = cap;
        expect(layout(w, 200, 90, &recs, &lod, &cap) == YX_ERR_OOM && g_emits == 0, "a wider tree without memory");
        expect(recs == recs0 && lod == lod0 && cap == cap0, "the records in use after it");
        g_fail_nth = 0;
        expect(layout(w, 200, 50, &recs, &lod, &cap) == YX_OK && g_emits == 3, "the first tree again");
        expect(!g_bad, "its kernels' sums");
        g_emits = g_bad = 0;
        expect(layout(w, 200, 90, &recs, &lod, &cap) == YX_OK && g_emits == 3 && !g_bad, "the wider tree with memory");
        g_emits = g_bad = 0;
        // the node arrays: the third of them cannot grow
        g_fail_bytes = (size_t)300 * 4;
        g_fail_nth = 3;
        expect(layout(w, 300, 50, &recs, &lod, &cap) == YX_ERR_OOM && g_emits == 0, "more nodes without memory");
        g_fail_nth = 0;
        expect(layout(w, 200, 50, &recs, &lod, &cap) == YX_OK && g_emits == 3 && !g_bad, "fewer nodes again");
        g_emits = g_bad = 0;
        yx::relayout_work_free(w);
        (void)hipFree(recs);
        (void)hipFree(lod);
        expect(g_live.empty() && !g_bad, "everything freed once");
    }
    std::printf(failed ? "%d failed\n" : "ok\n", failed);
    return failed != 0;
}
