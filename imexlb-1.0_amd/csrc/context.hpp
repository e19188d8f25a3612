// context.hpp -- internal: the lattice context behind the C ABI, shared by
// capi.cpp (single lattice) and batch.cpp (batched ensemble).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdlib>
#include <string>
#include <vector>

#include "../../include/imexlb.h"
#include "geometry.hpp"
#include "kernels.hpp"

namespace imexlb {

inline std::string &last_error()
{
    thread_local std::string s;
    return s;
}

inline int fail(int code, const std::string &msg)
{
    last_error() = msg;
    return code;
}

#define HIP_TRY(expr)                                                                                  \
    do {                                                                                               \
        hipError_t e_ = (expr);                                                                        \
        if (e_ != hipSuccess)                                                                          \
            return fail(e_ == hipErrorOutOfMemory ? IMEXLB_E_OOM : IMEXLB_E_HIP,                       \
                        std::string(#expr) + ": " + hipGetErrorString(e_));                            \
    } while (0)

enum Stage { S_NONE, S_PRE, S_COLLIDED, S_FILLED, S_PENDING, S_STREAMED, S_FUSED };

struct TimedLaunch {
    int cls, steps;  // steps: lattice steps the launch makes (counted as so many launches)
    hipEvent_t a, b;
};


// Pinned buffers of the downloads, one per thread, kept by the object that
// downloads (its calls are not concurrent) and freed with it: at most 16 MiB.
struct Staging {
    static constexpr int kWorkers = 8;
    double *host[kWorkers] = {};
    hipEvent_t done[kWorkers] = {};
    int64_t values = 0;  // of each buffer
    void release();
};

struct FieldCopy {
    const double *from;  // padded device array
    double *to;          // the caller's dense interior array
};

// Test hook: IMEXLB_FAIL_ALLOC=N (read when a lattice or an ensemble is
// created) makes its N-th device allocation fail.
struct AllocHook {
    int64_t calls = 0, fail_at = 0;
    void read()
    {
        if (const char *v = std::getenv("IMEXLB_FAIL_ALLOC")) fail_at = std::atoll(v);
    }
    bool fails() { return fail_at > 0 && ++calls == fail_at; }
};

// Device memory of a plan that its owner does without if there is none: no
// error is left behind, and what the plan keeps is counted while it does.
struct PlanMemory {
    size_t bytes = 0;
    bool get(AllocHook &hook, void **ptr, size_t n)
    {
        if (!temp(hook, ptr, n)) return false;
        bytes += n;
        return true;
    }
    static bool temp(AllocHook &hook, void **ptr, size_t n)
    {
        *ptr = nullptr;
        if (hook.fails()) return false;
        if (hipMalloc(ptr, n) == hipSuccess) return true;
        (void)hipGetLastError();
        *ptr = nullptr;
        return false;
    }
};

struct DeviceTemp {  // freed on every return
    void *p = nullptr;
    ~DeviceTemp()
    {
        if (p) (void)hipFree(p);
    }
};

// The interior of padded device arrays to dense host arrays, after the work on
// the stream; false if there is no memory for the buffers, or the fields are
// small enough for a plain copy (nothing was copied).
bool download_interior(Staging &s, int device, hipStream_t stream, int dim, const KParams &kp,
                       const std::vector<FieldCopy> &fields, hipError_t &err);

}  // namespace imexlb

using namespace imexlb;

struct imexlb_ctx {
    int dim = 2, Q = 9, device = -1, prec = 0;
    bool host_only = true;
    RefGeometry g;
    BcTable bc;
    bool geom_set = false;
    double ome = 0.0, rho0 = 1.0, uu = 0.0;

    // device layout
    int64_t Px = 0, Py = 0, Pz = 1, PxPy = 0, o0 = 0, plane = 0;
    size_t ssz = 8;
    KParams kp{};
    uint32_t skip_c = 0xffffffffu;

    hipStream_t stream = nullptr;
    void *fb[2] = {nullptr, nullptr};
    void *f = nullptr;
    double *p = nullptr, *ux = nullptr, *uy = nullptr, *uz = nullptr, *rv = nullptr;
    uint8_t *geo = nullptr;
    void *fill_dst = nullptr, *fill_src = nullptr;  // int32 (fill32) or int64 slots
    bool fill32 = false;
    // boundary copies pushed by the fused step (grouped resolved table)
    int32_t *push_beg = nullptr;
    uint8_t *push_q = nullptr;
    void *push_dst = nullptr;   // int32 (fill32) or int64 slots
    uint16_t *push_lds = nullptr;  // LDS position of each entry's value
    bool push_enabled = true;   // IMEXLB_PUSH=0 keeps the separate fill
    bool push_on = false;       // enabled and the table qualifies
    bool prefilled = false;     // buffer cur already holds its boundary copies
    int64_t nfill = 0;
    unsigned long long *red = nullptr;
    // body links for the momentum-exchange force
    int64_t *link_out = nullptr, *link_back = nullptr;
    int8_t *link_q = nullptr;
    int64_t nlink = 0;
    double *force_partial = nullptr, *force_out = nullptr;
    Staging staging;
    double *mass_partial = nullptr;  // MASS_BLOCKS partial sums, then the total
    size_t dev_bytes = 0;
    AllocHook hook;

    // Forget the geometry after a failed SetGeometry: every call that needs
    // one (InitUP, the phases, Monitor, downloads) then returns
    // IMEXLB_E_STATE until SetGeometry succeeds.
    void forget_geometry()
    {
        geom_set = false;
        nfill = nlink = 0;
        push_on = prefilled = dbl_on = multi_on = false;
        stage = S_NONE;
        have_pu = have_f = have_fb = false;
        lazy_src = -1;
        drop_graphs();
    }

    // phase state
    Stage stage = S_NONE;
    int cur = 0;
    bool fused = true;
    bool have_pu = false, have_f = false, have_fb = false;
    int lazy_src = -1;

    // replay of pairs of fused steps as HIP graphs of kGraphPairs[j] pairs,
    // one per size and starting buffer (cur); advance() takes the largest
    // that fit first (longer graphs: fewer gaps between replays, 3 % on the
    // 400x100 cylinder from 16 to 64 pairs)
    bool graphs = true;
    static constexpr int kGraphSizes = 3;
    static constexpr int kGraphPairs[kGraphSizes] = {64, 8, 1};
    hipGraphExec_t graph[kGraphSizes][2] = {};
    void drop_graphs()
    {
        for (auto *all : {&graph, &quad_graph, &multi_graph})
            for (auto &set : *all)
                for (int k = 0; k < 2; ++k)
                    if (set[k]) {
                        (void)hipGraphExecDestroy(set[k]);
                        set[k] = nullptr;
                    }
    }

    // Fused steps asked for through the phase calls (PostProcessing of a
    // lattice whose step writes its own boundary copies) and not launched
    // yet: they run as graph replays once kDeferChunk are pending (one graph
    // of kDeferChunk / 2 pairs, so the GPU works while the caller goes on)
    // and when the state is next needed (any other call that launches work
    // or reads device memory).  Step k of them reads fb[defer_src ^ (k & 1)].
    int64_t deferred = 0;
    int defer_src = 0;
    static constexpr int64_t kDeferChunk = 16;
    int64_t defer_chunk() const { return multi_on ? 2 * multi.halo + 1 : kDeferChunk; }
    bool can_defer() const { return fused && graphs && !prof && push_on; }

    // Two steps in one pass over memory, for lattices that do not stay in the
    // caches (built with the geometry; IMEXLB_DOUBLE=0 keeps single steps)
    DoublePlan dbl;
    PlanMemory dbl_mem;
    bool dbl_enabled = true, dbl_on = false;
    hipGraphExec_t quad_graph[kGraphSizes][2] = {};  // kQuads[j] pairs of double steps, by starting buffer
    static constexpr int kQuads[kGraphSizes] = {16, 4, 1};
    // Several steps in one launch (built with the geometry; IMEXLB_MULTI=0
    // keeps the other forms)
    MultiPlan multi;
    PlanMemory multi_mem;
    int32_t *multi_table = nullptr;
    uint16_t *multi_place = nullptr;
    bool multi_enabled = true, multi_on = false;
    hipGraphExec_t multi_graph[kGraphSizes][2] = {};  // kMulti[j] launches of multi.halo steps
    static constexpr int kMulti[kGraphSizes] = {16, 4, 2};  // even: they end in the buffer they began in
    void drop_multi()
    {
        for (void *q : {(void *)multi_table, (void *)multi_place})
            if (q) (void)hipFree(q);
        multi_table = nullptr;
        multi_place = nullptr;
        multi = MultiPlan{};
        multi_mem = PlanMemory{};
        multi_on = false;
    }
    void drop_double()
    {
        for (void *q : {(void *)dbl.list[0], (void *)dbl.list[1], dbl.scratch})
            if (q) (void)hipFree(q);
        dbl = DoublePlan{};
        dbl_mem = PlanMemory{};
        dbl_on = false;
    }

    // profiling
    bool prof = false;
    std::vector<TimedLaunch> timed;
    static constexpr size_t kMaxTimed = 512;
    int64_t prof_n[3] = {0, 0, 0};
    double prof_ms[3] = {0, 0, 0};

    int64_t pidx(int x, int y, int z) const { return o0 + x + Px * y + PxPy * z; }

    StepArgs args() const
    {
        StepArgs a;
        a.kp = kp;
        a.p = p;
        a.ux = ux;
        a.uy = uy;
        a.uz = uz;
        a.geo = geo;
        a.push.beg = push_beg;
        a.push.q = push_q;
        a.push.dst = push_dst;
        a.push.lds = push_lds;
        return a;
    }

    int begin(int cls, hipEvent_t &b)
    {
        (void)cls;
        if (!prof) return IMEXLB_OK;
        HIP_TRY(hipEventCreate(&b));
        HIP_TRY(hipEventRecord(b, stream));
        return IMEXLB_OK;
    }
    int end(int cls, hipEvent_t b, int steps)
    {
        if (!prof) return IMEXLB_OK;
        hipEvent_t e;
        HIP_TRY(hipEventCreate(&e));
        HIP_TRY(hipEventRecord(e, stream));
        timed.push_back(TimedLaunch{cls, steps, b, e});
        // bound the live event pairs of a long timed run: fold the oldest
        // half into the totals (waiting for them) once kMaxTimed are held
        if (timed.size() >= kMaxTimed) return harvest(kMaxTimed / 2);
        return IMEXLB_OK;
    }

    // add the elapsed time of all but the newest `keep` event pairs to
    // prof_n / prof_ms and destroy them (waits for those launches)
    int harvest(size_t keep)
    {
        const size_t n = timed.size() > keep ? timed.size() - keep : 0;
        for (size_t k = 0; k < n; ++k) {
            TimedLaunch &t = timed[k];
            HIP_TRY(hipEventSynchronize(t.b));
            float v = 0.0f;
            HIP_TRY(hipEventElapsedTime(&v, t.a, t.b));
            prof_n[t.cls] += t.steps;
            prof_ms[t.cls] += double(v);
            (void)hipEventDestroy(t.a);
            (void)hipEventDestroy(t.b);
        }
        timed.erase(timed.begin(), timed.begin() + std::ptrdiff_t(n));
        return IMEXLB_OK;
    }

    template <class F>
    int launch(int cls, F &&fn, int steps = 1)
    {
        hipEvent_t b = nullptr;
        int rc = begin(cls, b);
        if (rc) return rc;
        hipError_t e = fn();
        if (e != hipSuccess) return fail(IMEXLB_E_HIP, std::string("kernel launch: ") + hipGetErrorString(e));
        return end(cls, b, steps);
    }

    // BoundaryCondition on buffer `buf`; the other buffer holds the previous
    // step's state (every Collision writes the buffer the previous step did
    // not use)
    int run_fill(int buf)
    {
        return launch(1, [&] {
            return launch_fill(prec, fb[buf], fb[1 - buf], fill_dst, fill_src, fill32, nfill, stream);
        });
    }

    // mode bits of the fused collide step for this lattice (K_SMALL in 2D and
    // K_CACHED in 3D for lattices of at most small_cells cells)
    int collide_mode() const
    {
        if (!push_on) return K_COLLIDE;
        if (!fill32) return K_COLLIDE | K_PUSH | K_IDX64;
        if (cells > small_cells) return K_COLLIDE | K_PUSH;
        return K_COLLIDE | K_PUSH | (dim == 2 ? K_SMALL : K_CACHED);
    }
    int64_t cells = 0;        // with the ghost layer, without padding of rows
    int64_t small_cells = 0;  // set at creation (IMEXLB_SMALL_CELLS)
    int64_t multi_cells = 0;  // up to it several steps per launch

    int run_step(int mode, const void *src, void *dst, void *fout)
    {
        StepArgs a = args();
        a.src = src;
        a.dst = dst;
        a.fout = fout;
        return launch((mode & K_COLLIDE) ? 0 : 2, [&] { return launch_step(dim, prec, mode, a, stream); });
    }

    // rebuild f, p, u of the current pre-collision state if the fused
    // kernel skipped writing them
    int materialize()
    {
        if (have_pu && have_f) return IMEXLB_OK;
        if (lazy_src < 0) {
            if (have_pu) return IMEXLB_OK;
            return fail(IMEXLB_E_STATE, "fields requested before InitUP/upload");
        }
        int rc = run_step(K_WRITE_F | K_WRITE_PU, fb[lazy_src], nullptr, f);
        if (rc) return rc;
        have_pu = have_f = true;
        return IMEXLB_OK;
    }

    void release()
    {
        if (host_only) return;
        (void)hipSetDevice(device);
        if (stream) (void)hipStreamSynchronize(stream);
        drop_graphs();
        for (auto &t : timed) {
            (void)hipEventDestroy(t.a);
            (void)hipEventDestroy(t.b);
        }
        timed.clear();
        void *ptrs[] = {fb[0],     fb[1],  f,         p,        ux,       uy,        uz,     rv,
                        geo,       fill_dst, fill_src, red,     link_out, link_back, link_q, force_partial,
                        force_out, push_beg, push_q,   push_dst, push_lds, mass_partial};
        for (void *q : ptrs)
            if (q) (void)hipFree(q);
        drop_double();
        drop_multi();
        staging.release();
        fb[0] = fb[1] = f = nullptr;
        push_beg = nullptr;
        push_q = nullptr;
        push_dst = nullptr;
        push_lds = nullptr;
        p = ux = uy = uz = rv = nullptr;
        geo = nullptr;
        fill_dst = fill_src = nullptr;
        red = nullptr;
        link_out = link_back = nullptr;
        link_q = nullptr;
        force_partial = force_out = nullptr;
        mass_partial = nullptr;
        if (stream) (void)hipStreamDestroy(stream);
        stream = nullptr;
    }
};

namespace imexlb {

inline int dev_alloc(imexlb_ctx *c, void **ptr, size_t bytes)
{
    if (c->hook.fails()) {
        *ptr = nullptr;
        return fail(IMEXLB_E_OOM, "hipMalloc(" + std::to_string(bytes) + "): failure injected by IMEXLB_FAIL_ALLOC");
    }
    hipError_t e = hipMalloc(ptr, bytes);
    if (e != hipSuccess) {
        *ptr = nullptr;
        return fail(e == hipErrorOutOfMemory ? IMEXLB_E_OOM : IMEXLB_E_HIP,
                    "hipMalloc(" + std::to_string(bytes) + "): " + hipGetErrorString(e));
    }
    c->dev_bytes += bytes;
    e = hipMemset(*ptr, 0, bytes);
    if (e != hipSuccess) return fail(IMEXLB_E_HIP, std::string("hipMemset: ") + hipGetErrorString(e));
    return IMEXLB_OK;
}

// Device-layout tables of one lattice, built on the host from its geometry:
// node types, the resolved boundary fill (dst, src in FillEntry encoding
// with device slots) and the body links of the force.
struct DeviceTables {
    std::vector<uint8_t> geo;
    uint32_t skip_c = 0xffffffffu;
    std::vector<int64_t> fill_dst, fill_src;
    std::vector<int32_t> push_beg;  // ncell + 1 offsets
    std::vector<uint8_t> push_q;
    std::vector<int64_t> push_dst;
    std::vector<uint16_t> push_lds;
    bool push_ok = true;  // every copy's source is a fluid node or a body cell
    std::vector<int64_t> link_out, link_back;
    std::vector<int8_t> link_q;
};
int build_device_tables(const imexlb_ctx *c, DeviceTables &t);

// Whether every boundary copy of a previous step's body value is always 0: such
// values mostly go round among body cells (a mirror's mirror is the cell
// itself) and stay the 0 they start with.
bool body_copies_zero(const DeviceTables &t);

// A run of several steps per launch.
struct MultiRun {
    int64_t full = 0;  // launches of m.halo steps before the last one
    int last = 0;      // steps of the last launch, which leaves the boundary copies (0: no launch at all)
    int64_t done = 0;  // steps in all
};
// n steps as launches of an odd number of steps each, the last one of m.least
// or more, with at least one single step left: the buffers end up as after as
// many single steps.
inline MultiRun multi_run(const MultiPlan &m, int64_t n)
{
    MultiRun r;
    if (n < m.from) return r;
    r.full = (n - 1) / m.halo;
    r.last = int((n - 1) % m.halo);
    if (!(r.last & 1)) --r.last;
    if (r.last < m.least) r.last = 0;
    r.done = r.full * m.halo + r.last;
    if (r.last == 0 && r.full > 0) {
        r.last = m.halo;
        --r.full;
    }
    return r;
}

// The boundary fill's slot tables fit int32 entries when every slot and its
// previous-step encoding (-slot-2) do.
inline bool fill_fits_32(int64_t nslots) { return nslots < (int64_t(1) << 31) - 2; }

// test hook: IMEXLB_SLOTS64=1 (read when the boundary tables are built)
// stores them with int64 slots also where int32 would do
inline bool force_slots64()
{
    const char *v = std::getenv("IMEXLB_SLOTS64");
    return v && v[0] == '1';
}

// copy a slot table to the device as int32 or int64 entries
inline hipError_t upload_slots(void *dev, const std::vector<int64_t> &v, bool idx32)
{
    if (v.empty()) return hipSuccess;
    if (!idx32) return hipMemcpy(dev, v.data(), v.size() * sizeof(int64_t), hipMemcpyHostToDevice);
    std::vector<int32_t> n(v.begin(), v.end());
    return hipMemcpy(dev, n.data(), n.size() * sizeof(int32_t), hipMemcpyHostToDevice);
}

}  // namespace imexlb
