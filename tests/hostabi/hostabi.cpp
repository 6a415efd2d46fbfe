// CPU build of the renderer's host code and C ABI (pt_renderer.cpp) over a
// stand-in HIP runtime, for tests of what it does with memory and where an
// allocation fails. Ray queries run the device code on the CPU; the other kernels of
// a render do nothing. Test infrastructure: the product never links this.
#include <algorithm>
#include <new>
#include <vector>

#include "pt_renderer.cpp"
#include "pt_path.h"

namespace fake {
thread_local long until_failure = -1;  // allocations of this thread before the one that fails (-1: none does)
}
void* operator new(size_t n) {
    const bool fail = fake::until_failure >= 0 && fake::until_failure-- == 0;
    void* p = fail ? nullptr : std::malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

extern "C" {
void fake_device_limit(size_t bytes) { fake::state().limit = bytes; }
size_t fake_device_used() { return fake::state().used; }
// High water mark since the last call.
size_t fake_device_peak() {
    const size_t p = fake::state().peak;
    fake::state().peak = fake::state().used;
    return p;
}
void fake_refuse_pinned(int on) { fake::state().refuse_pinned = on != 0; }
void fake_fail_new(long after) { fake::until_failure = after; }
long fake_fail_new_left() { return fake::until_failure; }
size_t fake_pinned() { return fake::state().pinned; }
}

namespace ptk {
using namespace ptd;
int persistent_blocks(int kind, int, int, bool, int num_cu, size_t) {
    return (kind == KIND_FINISH || kind == KIND_FINISH_INLINE ? 8 : 2) * num_cu;
}
LayoutSizes layout_sizes() { return layout_sizes_here(); }
TlasLayout tlas_layout() { return tlas_layout_here(); }
size_t env_cdf_scratch_bytes(int n) { return env_cdf_scratch_size(n); }
void launch_plain(hipStream_t, int, int, const DevScene&, const DevOpts&, float4*, int, int, int, int, int*, int, int*,
                  unsigned long long*, int*, bool, bool, const int2*) {}
void launch_tiles(hipStream_t, const DevScene&, const DevOpts&, const JobDev*, int, int, int2*) {}
void launch_extend(hipStream_t, int, int, const DevScene&, const DevOpts&, const PathBuf&, bool, const int*, const int*,
                   int, int, int, int*, int*, int*, int, int*, unsigned long long*, int*, bool, int, const ContBuf*,
                   int*, int, const int2*) {}
void launch_extend_resume(hipStream_t, int, int, const DevScene&, const DevOpts&, const PathBuf&, const ContBuf&,
                          const int*, int*, int*, int, int*, int*) {}
void launch_finish(hipStream_t, int, const DevScene&, const DevOpts&, const PathBuf&, const BatchBuf*, bool, bool,
                   const int*, const int*, const int*, int, int, int, int, int, int, int*, int*, int*, const int2*, int,
                   const Record*) {}
void launch_shade(hipStream_t, int, int, const DevScene&, const DevOpts&, const PathBuf&, const ShadowBuf&,
                  const BatchBuf*, bool, bool, const int*, const int*, int, int, int*, int*, int*, int*, bool, int, int*,
                  unsigned long long*, int*) {}
void launch_shadow(hipStream_t, int, int, const DevScene&, const DevOpts&, const PathBuf&, const ShadowBuf&, const int*,
                   int*, int, int*, unsigned long long*, int*, bool, unsigned*, int) {}
void launch_replay_shade(hipStream_t, int, int, const DevScene&, const DevOpts&, const PathBuf&, bool, const int*,
                         const int*, int, int, int*, int*, int*, bool, const ReplayBuf&, int) {}
void launch_accum(hipStream_t, const DevOpts&, const PathBuf&, float4*, int, int) {}
void launch_pass_begin(hipStream_t, const BatchBuf&, int*, int) {}
void launch_pass_end(hipStream_t, const BatchBuf&) {}
void launch_extend_batch(hipStream_t, int, int, const DevScene&, const DevOpts&, const PathBuf&, const BatchBuf&, int*,
                         int*, int*, int, int*, int*, const int2*) {}
void launch_accum_batch(hipStream_t, int, const PathBuf&, const BatchBuf&) {}
void launch_plain_batch(hipStream_t, int, int, const DevScene&, const DevOpts&, const JobDev*, int, int, int, float4*,
                        int*, int, int*, int*, bool, const int2*) {}
void launch_env_cdf(hipStream_t, const float*, int, float*, float*, int*, void*) {}
void launch_zero_cells(hipStream_t, int* cells, int n) {
    for (int i = 0; i < n; ++i) cells[static_cast<size_t>(i) * CELL] = 0;
}
void launch_roll_cells(hipStream_t s, int* cells, int n, const int* from) {
    const int first = *from;
    launch_zero_cells(s, cells, n);
    cells[0] = first;
}
void launch_fill(hipStream_t, int* p, int n, int v) { std::fill_n(p, n, v); }
void launch_tonemap(hipStream_t, const float4*, int, int, float, int, int, int, int, const float*, uchar4*) {}
void launch_tlas_rebuild(hipStream_t, const TlasBuild&) {}
void launch_tlas4(hipStream_t, const GNode*, int, GNode4*, int, int, int*, int*) {}

// The query kernels: a thread per ray, its stack's S entries in LDS, the rest
// at its slot of the backing store.
template <class F>
static void rays(int n, int S, int* spill, int* ovf, F&& ray) {
    std::vector<int> lds(S);
    const size_t threads = (static_cast<size_t>(n) + 255) / 256 * 256;
    for (int i = 0; i < n; ++i) {
        Stack stk{lds.data(), spill, 0, 1, S, static_cast<size_t>(i), threads};
        TravCount cnt{0, 0, 0, 0, 0, 0};
        bool o = false;
        ray(i, stk, cnt, o);
        if (o) *ovf = 1;
    }
}
void launch_query_closest(hipStream_t, const DevScene& sc, const DevOpts& op, const float* o, const float* d, int n,
                          float* t, int* inst, int* tri, int* light, float* uv, int S, int* spill, int* ovf) {
    rays(n, S, spill, ovf, [&](int i, Stack& stk, TravCount& cnt, bool& of) {
        const Hit h = closest<false>(sc, op, V(o[3 * i], o[3 * i + 1], o[3 * i + 2]),
                                     V(d[3 * i], d[3 * i + 1], d[3 * i + 2]), 1, stk, cnt, of);
        t[i] = h.t;
        inst[i] = h.inst;
        tri[i] = h.tri;
        light[i] = h.light;
        uv[2 * i] = h.tri >= 0 ? h.u : 0.f;
        uv[2 * i + 1] = h.tri >= 0 ? h.v : 0.f;
    });
}
void launch_query_any(hipStream_t, const DevScene& sc, const DevOpts& op, const float* o, const float* d,
                      const float* maxd, int n, int* occ, int S, int* spill, int* ovf) {
    rays(n, S, spill, ovf, [&](int i, Stack& stk, TravCount& cnt, bool& of) {
        occ[i] = occluded<false, true>(sc, op, V(o[3 * i], o[3 * i + 1], o[3 * i + 2]),
                                       V(d[3 * i], d[3 * i + 1], d[3 * i + 2]), maxd[i], stk, cnt, of);
    });
}
}  // namespace ptk
