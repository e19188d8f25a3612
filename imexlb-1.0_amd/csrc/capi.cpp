// capi.cpp -- the C ABI (include/imexlb.h): context, device memory, and the
// phase state machine that maps the reference's four per-step procedures
// (main.f90:57-61) onto the gfx950 kernels.
//
// Fused mode (default): Collision of step t+1, Propagation and
// PostProcessing of step t run as one pull kernel launched from
// PostProcessing; the post-collision populations ping-pong between two
// buffers.  f, p and u of step t are not written by that kernel; when a
// caller reads them (Monitor, downloads) one stream+moments pass rebuilds
// them from the buffer the fused kernel streamed from, which stays intact
// until the next PostProcessing.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <limits>
#include <memory>
#include <new>
#include <string>
#include <vector>

#include "context.hpp"



namespace {

#define CHECK_CTX(c)                                                       \
    do {                                                                   \
        if (!(c)) return fail(IMEXLB_E_ARG, "null context");              \
    } while (0)
#define CHECK_DEV(c)                                                                   \
    do {                                                                               \
        CHECK_CTX(c);                                                                  \
        if ((c)->host_only) return fail(IMEXLB_E_NODEV, "host-only context");         \
        HIP_TRY(hipSetDevice((c)->device));                                            \
    } while (0)

size_t storage_bytes(int prec) { return prec == 0 ? 8 : prec == 1 ? 4 : 2; }

const std::vector<int32_t> *pick_list(const imexlb_ctx *c, int list)
{
    const RefGeometry &g = c->g;
    switch (list) {
    case IMEXLB_LIST_FLUID: return &g.fluid_id;
    case IMEXLB_LIST_BL: return &g.bl;
    case IMEXLB_LIST_BR: return &g.br;
    case IMEXLB_LIST_BU: return &g.bu;
    case IMEXLB_LIST_BD: return &g.bd;
    case IMEXLB_LIST_BF: return &g.bf;
    case IMEXLB_LIST_BB: return &g.bb;
    case IMEXLB_LIST_USER: return &g.b_user;
    default: return nullptr;
    }
}

// host staging helpers: interior node (x,y,z) <-> reference id / dense index
template <class Fn>
static void for_interior(const imexlb_ctx *c, Fn fn)
{
    const int nx = c->kp.nx, ny = c->kp.ny, nz = c->dim == 3 ? c->kp.nz : 0;
    int64_t k = 0;
    for (int z = 0; z <= nz; ++z)
        for (int y = 0; y <= ny; ++y)
            for (int x = 0; x <= nx; ++x, ++k) fn(x, y, z, k, c->g.id(x, y, z), c->pidx(x, y, z));
}

double load_value(const uint8_t *base, size_t i, int prec)
{
    switch (prec) {
    case 0: {
        double v;
        std::memcpy(&v, base + i * 8, 8);
        return v;
    }
    case 1: {
        float v;
        std::memcpy(&v, base + i * 4, 4);
        return double(v);
    }
    case 2: {
        _Float16 v;
        std::memcpy(&v, base + i * 2, 2);
        return double(float(v));
    }
    default: {
        uint16_t b;
        std::memcpy(&b, base + i * 2, 2);
        uint32_t w = uint32_t(b) << 16;
        float v;
        std::memcpy(&v, &w, 4);
        return double(v);
    }
    }
}

}  // namespace

namespace imexlb {

int build_device_tables(const imexlb_ctx *c, DeviceTables &t)
{
    const RefGeometry &g = c->g;
    // node types: 1 on interior fluid nodes
    t.geo.assign(size_t(c->plane), 0);
    for (int32_t id : g.fluid_id) {
        int x, y, z;
        g.coords(id, x, y, z);
        t.geo[size_t(c->pidx(x, y, z))] = G_FLUID;
    }
    if (!g.fluid_id.empty()) {
        int x, y, z;
        g.coords(g.fluid_id[0], x, y, z);
        t.skip_c = uint32_t(c->pidx(x, y, z));
    }
    // resolved boundary table in device slots
    auto dev_slot = [&](int64_t ref_slot) {
        int x, y, z;
        g.coords(ref_slot / c->Q, x, y, z);
        return pop_slot(ref_slot % c->Q, c->pidx(x, y, z), c->plane, c->Q);
    };
    const int64_t nslots = int64_t(c->Q) * c->plane;
    t.fill_dst.clear();
    t.fill_src.clear();
    t.fill_dst.reserve(c->bc.entries.size());
    t.fill_src.reserve(c->bc.entries.size());
    for (const FillEntry &e : c->bc.entries) {
        const int64_t d = dev_slot(e.ref_slot);
        int64_t s = -1;  // zero
        if (e.ref_src >= 0) s = dev_slot(e.ref_src);
        else if (e.ref_src <= -2) s = encode_prev(dev_slot(decode_prev(e.ref_src)));
        const int64_t sabs = s >= 0 ? s : s == -1 ? 0 : decode_prev(s);
        if (d < 0 || d >= nslots || sabs < 0 || sabs >= nslots)
            return fail(IMEXLB_E_ARG, "boundary table slot outside the population arrays");
        t.fill_dst.push_back(d);
        t.fill_src.push_back(s);
    }
    // destination order: consecutive fill threads write consecutive slots
    {
        std::vector<size_t> order(t.fill_dst.size());
        for (size_t k = 0; k < order.size(); ++k) order[k] = k;
        std::sort(order.begin(), order.end(), [&](size_t a, size_t b) { return t.fill_dst[a] < t.fill_dst[b]; });
        std::vector<int64_t> d(order.size()), s(order.size());
        for (size_t k = 0; k < order.size(); ++k) {
            d[k] = t.fill_dst[order[k]];
            s[k] = t.fill_src[order[k]];
        }
        t.fill_dst.swap(d);
        t.fill_src.swap(s);
    }
    // the same table grouped by source node (padded cell, direction) for the
    // fused step's push copies; zero entries are left out (never written,
    // the buffers start at 0)
    {
        struct Copy {
            uint32_t cell;
            uint8_t q;
            int64_t dst;
        };
        std::vector<Copy> v;
        v.reserve(c->bc.entries.size());
        t.push_ok = true;
        for (const FillEntry &e : c->bc.entries) {
            if (e.ref_src == -1) continue;
            const bool prev = e.ref_src <= -2;
            const int64_t rs = prev ? decode_prev(e.ref_src) : e.ref_src;
            int x, y, z;
            g.coords(rs / c->Q, x, y, z);
            const uint32_t cell = uint32_t(c->pidx(x, y, z));
            // this step's value comes from a fluid node, a previous one from a
            // body cell, and either is an interior node (the step has no
            // thread on ghost cells)
            if (bool(t.geo[cell] & G_FLUID) == prev) t.push_ok = false;
            if (!g.interior(x, y, z)) t.push_ok = false;
            v.push_back({cell, uint8_t(rs % c->Q), dev_slot(e.ref_slot)});
        }
        std::sort(v.begin(), v.end(), [](const Copy &a, const Copy &b) {
            return a.cell != b.cell ? a.cell < b.cell : a.q != b.q ? a.q < b.q : a.dst < b.dst;
        });
        t.push_beg.assign(size_t(c->kp.ncell) + 1, 0);
        t.push_q.resize(v.size());
        t.push_dst.resize(v.size());
        t.push_lds.resize(v.size());
        for (size_t k = 0; k < v.size(); ++k) {
            ++t.push_beg[size_t(v[k].cell) + 1];
            t.push_q[k] = v[k].q;
            t.push_dst[k] = v[k].dst;
            t.push_lds[k] = uint16_t(v[k].q * 64u + (v[k].cell & 63u));
            t.geo[v[k].cell] |= G_PUSH;
        }
        for (size_t k = 1; k < t.push_beg.size(); ++k) t.push_beg[k] += t.push_beg[k - 1];
    }
    // body links: fluid node x, direction q, interior solid neighbour x+e_q
    t.link_out.clear();
    t.link_back.clear();
    t.link_q.clear();
    const int nzmax = c->dim == 3 ? c->kp.nz : 0;
    for (int z = 0; z <= nzmax; ++z)
        for (int y = 0; y <= c->kp.ny; ++y)
            for (int x = 0; x <= c->kp.nx; ++x) {
                if (g.geo[size_t(g.id(x, y, z))] != 0) continue;
                for (int q = 0; q < c->Q; ++q) {
                    const int fx = x - g.lat.e[q][0], fy = y - g.lat.e[q][1], fz = z - g.lat.e[q][2];
                    if (!g.interior(fx, fy, fz) || g.geo[size_t(g.id(fx, fy, fz))] != 1) continue;
                    t.link_out.push_back(pop_slot(q, c->pidx(fx, fy, fz), c->plane, c->Q));
                    t.link_back.push_back(pop_slot(c->Q - 1 - q, c->pidx(x, y, z), c->plane, c->Q));
                    t.link_q.push_back(int8_t(q));
                }
            }
    return IMEXLB_OK;
}

bool body_copies_zero(const DeviceTables &t)
{
    const size_t n = t.fill_dst.size();
    std::vector<uint8_t> seen(n, 0);  // entries found to be 0, or on the way there (a ring)
    for (size_t k = 0; k < n; ++k) {
        size_t at = k;
        while (!seen[at] && t.fill_src[at] <= -2) {
            seen[at] = 1;
            const int64_t s = decode_prev(t.fill_src[at]);
            const auto it = std::lower_bound(t.fill_dst.begin(), t.fill_dst.end(), s);  // in order
            if (it == t.fill_dst.end() || *it != s) break;  // never written
            at = size_t(it - t.fill_dst.begin());
            if (t.fill_src[at] >= 0) return false;
        }
    }
    return true;
}

}  // namespace imexlb

extern "C" {

const char *imexlb_strerror(int code)
{
    switch (code) {
    case IMEXLB_OK: return "success";
    case IMEXLB_E_ARG: return "invalid argument";
    case IMEXLB_E_HIP: return "HIP runtime error";
    case IMEXLB_E_OOM: return "out of memory";
    case IMEXLB_E_STATE: return "call out of the Collision..PostProcessing order";
    case IMEXLB_E_UB: return "result depends on a read past the end of the reference arrays";
    case IMEXLB_E_NODEV: return "compute call on a host-only context";
    case IMEXLB_E_NAN: return "non-finite velocity (the lattice has diverged)";
    default: return "unknown error";
    }
}

const char *imexlb_last_error(void) { return last_error().c_str(); }

// Launches the fused steps the phase calls deferred (defined with the graph
// replay below); every entry point that launches other work or reads the
// device state runs it first.
static int flush_deferred(imexlb_ctx *c);
#define FLUSH(c)                                            \
    do {                                                    \
        if (int rf_ = flush_deferred(c)) return rf_;        \
    } while (0)

int imexlb_device_count(int *n)
{
    if (!n) return fail(IMEXLB_E_ARG, "null pointer");
    int k = 0;
    hipError_t e = hipGetDeviceCount(&k);
    *n = e == hipSuccess ? k : 0;
    return IMEXLB_OK;
}

int imexlb_create(imexlb_ctx **out, int dim, int nx, int ny, int nz, int device, int precision)
{
    if (!out) return fail(IMEXLB_E_ARG, "null output pointer");
    *out = nullptr;
    if (dim != 2 && dim != 3) return fail(IMEXLB_E_ARG, "dim must be 2 or 3");
    if (nx < 2 || ny < 2 || (dim == 3 && nz < 2))
        return fail(IMEXLB_E_ARG, "every axis needs at least 3 nodes (cart_mpi.f90:107-110)");
    if (precision < IMEXLB_F64 || precision > IMEXLB_BF16SR_F32) return fail(IMEXLB_E_ARG, "unknown precision");
    std::unique_ptr<imexlb_ctx> c(new (std::nothrow) imexlb_ctx);
    if (!c) return fail(IMEXLB_E_OOM, "context");
    c->dim = dim;
    c->Q = dim == 2 ? 9 : 27;
    c->prec = precision;
    c->ssz = storage_bytes(precision);
    c->g.init(dim, nx, ny, dim == 3 ? nz : 0);
    if (c->g.A >= (int64_t(1) << 31)) return fail(IMEXLB_E_ARG, "array_size exceeds the reference's 32-bit ids");

    // padded device layout, one ghost layer; rows optionally padded to a
    // multiple of `align` cells (IMEXLB_ROW_ALIGN) so that the y- and
    // z-shifted pulls of a tile start on a tile boundary
    int64_t align = 1;
    // The small-lattice step form pays while the two population buffers stay
    // in the 256 MB Infinity Cache from step to step: up to 240 MiB of them
    // and 5 Mi cells (measured on MI355X from 400x100 to 8192x2048 in every
    // storage form; against two steps per pass FP64 2048x512 23.4 and 26.3 us
    // a step, 2560x640 35.0 and 33.4, FP16 4096x1024 25.3 and 29.0, 5001x1251
    // 40.0 and 38.0 us); IMEXLB_SMALL_CELLS overrides the cell limit (and
    // that of several steps per launch).
    c->small_cells = std::min<int64_t>(int64_t(5) << 20, (int64_t(240) << 20) / (2 * 9 * int64_t(c->ssz)));
    // 3D lattices of the same size store their outputs through the caches
    // (us a step: 129x49x49 FP64 41 and 31 (25 with LDS copies), 161x65x65 FP32 37 and 27, 201x81x81
    // FP16 37 and 28; above, where they leave the cache before they are read
    // again, 201x81x81 FP32 62 and 65, FP64 121 and 138).
    if (dim == 3) c->small_cells = (int64_t(240) << 20) / (2 * 27 * int64_t(c->ssz));
    if (const char *sv = std::getenv("IMEXLB_SMALL_CELLS")) c->small_cells = std::atoll(sv);
    // Several steps per launch pay in FP32 at every size, in 16-bit storage up
    // to 8 Mi cells and in FP64 up to 2.5 Mi; above, the cells that neighbouring
    // windows both compute cost more than a second pass (against two steps per
    // pass, us a step: FP32 8192x2048 97 and 129, FP16 5001x1251 32.1 and 38.1,
    // 8192x2048 83.6 and 82.8, FP64 3000x750 39.8 and 41.5, 8192x2048 285 and
    // 244); with stochastic rounding, more arithmetic per cell, up to 0.75 Mi
    // (1000x250 3.60 and, single steps, 4.45; 2000x500 9.73 and 9.24).
    c->multi_cells = c->ssz == 4                     ? INT64_MAX
                     : precision == IMEXLB_BF16SR_F32 ? int64_t(3) << 18
                     : c->ssz == 2                    ? int64_t(8) << 20
                                                      : int64_t(5) << 19;
    if (std::getenv("IMEXLB_SMALL_CELLS")) c->multi_cells = c->small_cells;
    const char *mv = std::getenv("IMEXLB_MULTI");
    c->multi_enabled = !(mv && mv[0] == '0');
    c->cells = int64_t(nx + 3) * (ny + 3) * (dim == 3 ? nz + 3 : 1);
    // Two steps per pass (k_double2) take rows of whole tiles and populations
    // that 32 bits address.  They pay from the width on where most of a strip
    // of 256 columns does work and the frame beside it is a small part: us a
    // step, single and two per pass, of 6 M cells (16 M): FP64 120 wide 180 and
    // 174 (484 and 489), 190 168 and 147, 500 154 and 115; FP32 300 77 and 81,
    // 380 77 and 71, 500 75 and 64; FP16, of which it takes those above 8 Mi cells,
    // (640 110 and 120, 760 108 and 102, 1100 106 and 100, 2000 102 and 87); with
    // stochastic rounding 640 48.2 and 51.1, 760 47.2 and 47.4, 2000 45.5 and
    // 41.0; 20 wide 349 and 753, FP16 72 and 380.  IMEXLB_DOUBLE=1, and IMEXLB_SMALL_CELLS
    // for lattices above it, take them at every width from 16 on.
    const char *dv = std::getenv("IMEXLB_DOUBLE");
    const bool everywhere = (dv && dv[0] == '1') || std::getenv("IMEXLB_SMALL_CELLS");
    const int64_t tiles = (int64_t(nx) + 3 + 63) / 64 * 64;
    c->dbl_enabled = !(dv && dv[0] == '0') && device >= 0 && dim == 2 && IMEXLB_TILE == 64 && nx >= 16 && ny >= 16 &&
                     c->cells > c->small_cells &&
                     (everywhere || nx >= (c->ssz == 8 ? 120 : c->ssz == 4 ? 360 : 720)) &&
                     size_t(c->Q) * size_t(tiles * (ny + 3) + 128) * c->ssz < (size_t(1) << 32) - (size_t(1) << 16);
    // Where several steps per launch are tried first, two per pass only serve
    // the bodies that those do not suit: rows are padded for them if that adds
    // at most a sixteenth.
    if (c->dbl_enabled && !(c->multi_enabled && c->cells <= c->multi_cells && (tiles - nx - 3) * 16 > nx + 3)) align = 64;
    if (const char *av = std::getenv("IMEXLB_ROW_ALIGN")) align = std::max<int64_t>(1, std::atoll(av));
    if (align > 4096) return fail(IMEXLB_E_ARG, "IMEXLB_ROW_ALIGN above 4096 cells");
    c->Px = ((int64_t(nx) + 3 + align - 1) / align) * align;
    c->Py = int64_t(ny) + 3;
    c->Pz = dim == 3 ? int64_t(nz) + 3 : 1;
    c->PxPy = c->Px * c->Py;
    c->o0 = 1 + c->Px + (dim == 3 ? c->PxPy : 0);
    // whole tiles in the tiled layout (and 128-value alignment of planes)
    constexpr int64_t kRound = IMEXLB_TILE > 128 ? IMEXLB_TILE : 128;
    c->plane = ((c->Px * c->Py * c->Pz + kRound - 1) / kRound) * kRound;
    const int64_t nodes = int64_t(nx + 1) * (ny + 1) * (dim == 3 ? nz + 1 : 1);
    if (c->plane >= (int64_t(1) << 31) || nodes >= (int64_t(1) << 31))
        return fail(IMEXLB_E_ARG, "grid too large for 32-bit node indexing");

    KParams &k = c->kp;
    k.nx = nx;
    k.ny = ny;
    k.nz = dim == 3 ? nz : 0;
    k.N = uint32_t(nodes);
    k.div_x.init(uint32_t(nx + 1));
    k.div_y.init(uint32_t(ny + 1));
    // host self-check of the multiply-high division on the row/plane ends
    const uint32_t probes[] = {0u, uint32_t(nx), uint32_t(nx + 1), k.N - 1u, k.N / 2u, 0xfffffffeu};
    for (uint32_t n : probes) {
        if (k.div_x.host_div(n) != n / uint32_t(nx + 1) || k.div_y.host_div(n) != n / uint32_t(ny + 1))
            return fail(IMEXLB_E_ARG, "fast division self-check failed");
    }
    k.o0 = c->o0;
    k.Px = c->Px;
    k.PxPy = dim == 3 ? c->PxPy : 0;
    k.plane = c->plane;
    k.ncell = uint32_t(c->Px * c->Py * c->Pz);
    k.Py = c->Py;
    k.row_pad = uint32_t(c->Px - (int64_t(nx) + 3));
    k.div_px.init(uint32_t(c->Px));
    k.div_py.init(uint32_t(c->Py));
    for (uint32_t n : {0u, uint32_t(c->Px), k.ncell - 1u, 0xfffffffeu})
        if (k.div_px.host_div(n) != n / uint32_t(c->Px) || k.div_py.host_div(n) != n / uint32_t(c->Py))
            return fail(IMEXLB_E_ARG, "fast division self-check failed");
    k.back_tiles = uint32_t((1 + k.Px + k.PxPy + 63) / 64);
    k.rdy = c->g.dy;
    k.rdz = c->g.dz;
    // XCD-contiguous block order (each XCD steps the same eighth of the
    // lattice every step, so a step reads the previous one's output from its
    // own L2) pays for the lattices that stay in the caches between steps;
    // larger ones take the hardware's order (D3Q27 FP64 us a step, contiguous
    // and hardware order: 513x129x129 707 and 693, 258x132x130 389 and 376,
    // 513x257x257 2744 and 2734; FP16 208 and 187, 113 and 103, 794 and 717);
    // IMEXLB_XCD_REMAP=0/1/R overrides
    const char *xv = std::getenv("IMEXLB_XCD_REMAP");
    k.xcd_remap = xv ? uint32_t(std::max(0, std::atoi(xv)))
                     : uint32_t(c->cells <= c->small_cells);

    c->hook.read();
    if (device >= 0) {
        int ndev = 0;
        HIP_TRY(hipGetDeviceCount(&ndev));
        if (device >= ndev) return fail(IMEXLB_E_ARG, "device index out of range");
        c->device = device;
        c->host_only = false;
        const char *gv = std::getenv("IMEXLB_GRAPHS");
        c->graphs = !(gv && gv[0] == '0');
        const char *pv = std::getenv("IMEXLB_PUSH");
        c->push_enabled = !(pv && pv[0] == '0');
        HIP_TRY(hipSetDevice(device));
        HIP_TRY(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
        const size_t pop = size_t(c->Q) * size_t(c->plane) * c->ssz;
        const size_t fld = size_t(c->plane) * sizeof(double);
        int rc;
        if ((rc = dev_alloc(c.get(), &c->fb[0], pop)) || (rc = dev_alloc(c.get(), &c->fb[1], pop)) ||
            (rc = dev_alloc(c.get(), &c->f, pop)) || (rc = dev_alloc(c.get(), (void **)&c->p, fld)) ||
            (rc = dev_alloc(c.get(), (void **)&c->ux, fld)) || (rc = dev_alloc(c.get(), (void **)&c->uy, fld)) ||
            (dim == 3 && (rc = dev_alloc(c.get(), (void **)&c->uz, fld))) ||
            (rc = dev_alloc(c.get(), (void **)&c->geo, size_t(c->plane))) ||
            (rc = dev_alloc(c.get(), (void **)&c->rv, 100 * sizeof(double))) ||
            (rc = dev_alloc(c.get(), (void **)&c->red, 64)) ||
            (rc = dev_alloc(c.get(), (void **)&c->mass_partial, (MASS_BLOCKS + 1) * sizeof(double)))) {
            c->release();
            return rc;
        }
    }
    *out = c.release();
    return IMEXLB_OK;
}

int imexlb_destroy(imexlb_ctx *c)
{
    if (!c) return IMEXLB_OK;
    c->release();
    delete c;
    return IMEXLB_OK;
}

int imexlb_set_params(imexlb_ctx *c, double ome, double rho0, double uu)
{
    CHECK_CTX(c);
    if (!std::isfinite(ome) || !std::isfinite(rho0) || !std::isfinite(uu) || rho0 == 0.0)
        return fail(IMEXLB_E_ARG, "non-finite parameter or rho0 == 0");
    FLUSH(c);  // deferred steps keep the parameters they were asked with
    if (!c->host_only && c->stage == S_FUSED && (ome != c->ome || rho0 != c->rho0 || uu != c->uu)) {
        // The fused kernel of the last step has already relaxed the next one
        // with the old parameters, where the reference's Collision reads
        // them when it runs (lbm.f90:52-76).  Rebuild f, p, u of the current
        // step (PostProcessing with the old parameters) and continue through
        // the per-phase path: the next Collision relaxes them anew.
        HIP_TRY(hipSetDevice(c->device));
        int rc = c->materialize();
        if (rc) return rc;
        c->lazy_src = -1;
        c->stage = S_PRE;
    }
    c->ome = c->kp.ome = ome;
    c->rho0 = c->kp.rho0 = rho0;
    c->kp.inv_rho0 = 1.0 / rho0;
    c->uu = c->kp.uu = uu;
    c->kp.ome_f = float(ome);
    c->kp.rho0_f = float(rho0);
    c->kp.uu_f = float(uu);
    c->kp.inv_rho0_f = float(c->kp.inv_rho0);
    if (!c->host_only) {
        HIP_TRY(hipSetDevice(c->device));
        HIP_TRY(hipStreamSynchronize(c->stream));
        c->drop_graphs();
    }
    return IMEXLB_OK;
}

// The two-steps-per-pass plan of the new geometry: the frame's lists, the
// bulk's marks in the node types, the scratch buffer.  A lattice it does not
// suit, or without memory for it, keeps single steps.
static int build_double(imexlb_ctx *c)
{
    c->drop_double();
    const size_t pop = size_t(c->Q) * size_t(c->plane) * c->ssz, n = size_t(c->plane);
    if (!c->dbl_enabled || !c->push_on || !c->fill32 || c->multi_on || c->Px % 64 != 0 ||
        pop >= (size_t(1) << 32) - (size_t(1) << 16))  // (IMEXLB_ROW_ALIGN)
        return IMEXLB_OK;
    DoublePlan &d = c->dbl;
    DeviceTemp zones, counts;
    const auto no_memory = [&] {
        c->drop_double();
        return IMEXLB_OK;
    };
    if (!c->dbl_mem.get(c->hook, &d.scratch, pop) || !PlanMemory::temp(c->hook, &zones.p, 3 * n) ||
        !PlanMemory::temp(c->hook, &counts.p, 4 * sizeof(uint32_t)))
        return no_memory();
    HIP_TRY(hipMemset(d.scratch, 0, pop));
    HIP_TRY(hipMemset(zones.p, 0, 3 * n));
    HIP_TRY(hipMemset(counts.p, 0, 4 * sizeof(uint32_t)));
    uint8_t *const z = static_cast<uint8_t *>(zones.p);
    uint32_t *const cnt = static_cast<uint32_t *>(counts.p);
    const StepArgs a = c->args();
    // special nodes, the second step's frame (one node around them), the
    // first step's (one more)
    HIP_TRY(launch_zone(0, a, c->geo, nullptr, z, nullptr, nullptr, 0, nullptr));
    HIP_TRY(launch_zone(1, a, c->geo, z, z + n, nullptr, nullptr, 0, nullptr));
    HIP_TRY(launch_zone(1, a, c->geo, z + n, z + 2 * n, nullptr, nullptr, 0, nullptr));
    for (int k = 0; k < 2; ++k)
        HIP_TRY(launch_zone(2, a, c->geo, z + (2 - k) * n, nullptr, cnt + k, nullptr, k, nullptr));
    HIP_TRY(hipMemcpy(d.count, cnt, sizeof(d.count), hipMemcpyDeviceToHost));
    for (int k = 0; k < 2; ++k) {
        if (!c->dbl_mem.get(c->hook, (void **)&d.list[k], std::max<size_t>(d.count[k], 1) * sizeof(uint32_t)))
            return no_memory();
        HIP_TRY(launch_zone(2, a, c->geo, z + (2 - k) * n, nullptr, cnt + 2 + k, d.list[k], 0, nullptr));
    }
    HIP_TRY(hipDeviceSynchronize());
    plan_double(int(c->ssz), c->kp, d);
    c->dbl_on = true;
    return IMEXLB_OK;
}

// The several-steps-per-launch plan of the new geometry.  A lattice it does
// not suit, or without memory for its tables, keeps single steps.
static int build_multi(imexlb_ctx *c, const DeviceTables &t)
{
    c->drop_multi();
    if (!c->multi_enabled || !c->push_on || !c->fill32 || c->dim != 2 || IMEXLB_TILE != 64 ||
        c->cells > c->multi_cells || !body_copies_zero(t))
        return IMEXLB_OK;
    std::vector<MultiPlan> plans;
    plan_multi(int(c->ssz), {&c->kp}, plans);
    c->multi = plans[0];
    DeviceTemp dfrom, dbad;
    const MultiPlan &m = c->multi;
    const size_t nw = size_t(m.nx) * size_t(m.ny), nslots = size_t(c->Q) * size_t(c->plane);
    const auto no_memory = [&] {
        c->drop_multi();
        return IMEXLB_OK;
    };
    if (!c->multi_mem.get(c->hook, (void **)&c->multi_table, nw * sizeof(int32_t)) ||
        !PlanMemory::temp(c->hook, &dfrom.p, nslots * sizeof(int32_t)) || !PlanMemory::temp(c->hook, &dbad.p, 4))
        return no_memory();
    uint32_t bad = 0;
    std::vector<int32_t> mark(nw);
    HIP_TRY(hipMemset(dbad.p, 0, 4));
    HIP_TRY(launch_multi_from(c->args(), static_cast<int32_t *>(dfrom.p), int64_t(nslots),
                              static_cast<const int32_t *>(c->fill_dst), static_cast<const int32_t *>(c->fill_src),
                              c->nfill, nullptr));
    const auto plan = [&](uint16_t *place) {
        return launch_multi_plan(c->args(), static_cast<int32_t *>(dfrom.p), m, c->multi_table, place,
                                 static_cast<uint32_t *>(dbad.p), nullptr);
    };
    HIP_TRY(plan(nullptr));
    HIP_TRY(hipMemcpy(&bad, dbad.p, 4, hipMemcpyDeviceToHost));
    HIP_TRY(hipMemcpy(mark.data(), c->multi_table, nw * sizeof(int32_t), hipMemcpyDeviceToHost));
    if (bad) {
        c->drop_multi();
        return IMEXLB_OK;
    }
    int32_t tables = 0;
    for (int32_t &v : mark) v = v ? tables++ : -1;
    if (!c->multi_mem.get(c->hook, (void **)&c->multi_place,
                          std::max<size_t>(1, size_t(place_base(tables, uint32_t(m.wx * m.wy))) * 2)))
        return no_memory();
    HIP_TRY(hipMemcpy(c->multi_table, mark.data(), nw * sizeof(int32_t), hipMemcpyHostToDevice));
    HIP_TRY(plan(c->multi_place));
    HIP_TRY(hipDeviceSynchronize());
    // A launch of three steps takes as long as three or more single ones where
    // loading and storing the windows is most of it (single steps' time = 1: FP16
    // 1.0 M nodes 0.87, 1.5 M 1.08, 5 M 1.06 to 1.9; FP64 1.06 M 0.75, 1.4 M 1.05
    // to 1.54; FP32 0.6 to 1.0 at every size), and so do short runs of 16-bit
    // lattices most of whose windows read tables, while their single steps
    // stay in the caches (5 steps of 43 x 111109 nodes 1.28, 91 x 53761 1.40).
    if (c->ssz != 4 && c->cells > (int64_t(5) << 18)) c->multi.least = 5;
    if (c->ssz == 2 && c->cells > (int64_t(4) << 20) && c->cells <= c->small_cells &&
        5 * int64_t(tables) >= 3 * int64_t(nw))
        c->multi.from = 3 * m.halo + 1;
    c->multi.table = c->multi_table;
    c->multi.place = c->multi_place;
    c->multi_on = true;
    return IMEXLB_OK;
}

int imexlb_set_geometry(imexlb_ctx *c, double pos, double radius)
{
    return imexlb_set_geometry_shape(c, pos, radius, 1.0, 0.0);
}

int imexlb_set_geometry_shape(imexlb_ctx *c, double pos, double radius, double aspect, double angle_deg)
{
    CHECK_CTX(c);
    FLUSH(c);
    if (!std::isfinite(pos) || !std::isfinite(radius) || !std::isfinite(aspect) || !std::isfinite(angle_deg))
        return fail(IMEXLB_E_ARG, "non-finite geometry");
    if (aspect <= 0.0) return fail(IMEXLB_E_ARG, "ellipse axis ratio must be positive");
    if (c->dim == 3 && (aspect != 1.0 || angle_deg != 0.0)) return fail(IMEXLB_E_ARG, "ellipses are 2D");
    if (!c->host_only) {
        HIP_TRY(hipSetDevice(c->device));
        HIP_TRY(hipStreamSynchronize(c->stream));
    }
    // From here on the old geometry is gone: every return before the end
    // leaves the context without one (forget_geometry), so later calls get
    // IMEXLB_E_STATE instead of running on half-built tables.
    c->forget_geometry();
    struct Commit {
        imexlb_ctx *c;
        bool done = false;
        ~Commit()
        {
            if (!done) c->forget_geometry();
        }
    } commit{c};
    c->g.build(pos, radius, aspect, angle_deg);
    c->bc = resolve_boundary(c->g);
    if (c->bc.undefined) return fail(IMEXLB_E_UB, c->bc.error);
    if (c->host_only) {
        commit.done = c->geom_set = true;
        return IMEXLB_OK;
    }

    DeviceTables t;
    int rc = build_device_tables(c, t);
    if (rc) return rc;
    c->skip_c = t.skip_c;
    HIP_TRY(hipMemcpy(c->geo, t.geo.data(), t.geo.size(), hipMemcpyHostToDevice));
    for (void *q : {(void *)c->fill_dst, (void *)c->fill_src, (void *)c->link_out, (void *)c->link_back,
                    (void *)c->link_q, (void *)c->force_partial, (void *)c->force_out, (void *)c->push_beg,
                    (void *)c->push_q, c->push_dst, (void *)c->push_lds})
        if (q) (void)hipFree(q);
    c->fill_dst = c->fill_src = c->link_out = c->link_back = nullptr;
    c->link_q = nullptr;
    c->force_partial = c->force_out = nullptr;
    c->push_beg = nullptr;
    c->push_q = nullptr;
    c->push_dst = nullptr;
    c->push_lds = nullptr;
    // boundary slots whose value is 0 are never written by the pushed copies:
    // start both buffers from 0 for this geometry
    const size_t pop = size_t(c->Q) * size_t(c->plane) * c->ssz;
    HIP_TRY(hipMemset(c->fb[0], 0, pop));
    HIP_TRY(hipMemset(c->fb[1], 0, pop));
    c->nfill = int64_t(t.fill_dst.size());
    c->nlink = int64_t(t.link_out.size());
    const size_t nf = std::max<size_t>(t.fill_dst.size(), 1), nl = std::max<size_t>(t.link_out.size(), 1);
    const size_t nblk = (nl + 255) / 256;
    c->fill32 = fill_fits_32(int64_t(c->Q) * c->plane) && !force_slots64();
    const size_t isz = c->fill32 ? 4 : 8;
    if ((rc = dev_alloc(c, &c->fill_dst, nf * isz)) || (rc = dev_alloc(c, &c->fill_src, nf * isz)) ||
        (rc = dev_alloc(c, (void **)&c->link_out, nl * 8)) || (rc = dev_alloc(c, (void **)&c->link_back, nl * 8)) ||
        (rc = dev_alloc(c, (void **)&c->link_q, nl)) ||
        (rc = dev_alloc(c, (void **)&c->force_partial, nblk * 3 * sizeof(double))) ||
        (rc = dev_alloc(c, (void **)&c->force_out, 4 * sizeof(double))))
        return rc;
    HIP_TRY(upload_slots(c->fill_dst, t.fill_dst, c->fill32));
    HIP_TRY(upload_slots(c->fill_src, t.fill_src, c->fill32));
    c->push_on = c->push_enabled && t.push_ok;
    const size_t np = std::max<size_t>(t.push_q.size(), 1);
    if ((rc = dev_alloc(c, (void **)&c->push_beg, t.push_beg.size() * sizeof(int32_t))) ||
        (rc = dev_alloc(c, (void **)&c->push_q, np)) || (rc = dev_alloc(c, &c->push_dst, np * isz)) ||
        (rc = dev_alloc(c, (void **)&c->push_lds, np * sizeof(uint16_t))))
        return rc;
    HIP_TRY(hipMemcpy(c->push_beg, t.push_beg.data(), t.push_beg.size() * sizeof(int32_t), hipMemcpyHostToDevice));
    if (!t.push_q.empty()) HIP_TRY(hipMemcpy(c->push_q, t.push_q.data(), t.push_q.size(), hipMemcpyHostToDevice));
    HIP_TRY(upload_slots(c->push_dst, t.push_dst, c->fill32));
    if (!t.push_lds.empty())
        HIP_TRY(hipMemcpy(c->push_lds, t.push_lds.data(), t.push_lds.size() * sizeof(uint16_t), hipMemcpyHostToDevice));
    if (c->nlink) {
        HIP_TRY(hipMemcpy(c->link_out, t.link_out.data(), t.link_out.size() * 8, hipMemcpyHostToDevice));
        HIP_TRY(hipMemcpy(c->link_back, t.link_back.data(), t.link_back.size() * 8, hipMemcpyHostToDevice));
        HIP_TRY(hipMemcpy(c->link_q, t.link_q.data(), t.link_q.size(), hipMemcpyHostToDevice));
    }
    if ((rc = build_multi(c, t)) || (rc = build_double(c))) return rc;
    commit.done = c->geom_set = true;
    return IMEXLB_OK;
}


int imexlb_geometry_size(imexlb_ctx *c, int list, int64_t *n)
{
    CHECK_CTX(c);
    if (!n) return fail(IMEXLB_E_ARG, "null pointer");
    if (!c->geom_set) return fail(IMEXLB_E_STATE, "SetGeometry not called");
    if (list == -1) {  // array_size
        *n = c->g.A;
        return IMEXLB_OK;
    }
    const auto *v = pick_list(c, list);
    if (!v) return fail(IMEXLB_E_ARG, "unknown list");
    *n = int64_t(v->size());
    return IMEXLB_OK;
}

int imexlb_geometry_list(imexlb_ctx *c, int list, int32_t *out, int64_t cap)
{
    CHECK_CTX(c);
    if (!c->geom_set) return fail(IMEXLB_E_STATE, "SetGeometry not called");
    const auto *v = pick_list(c, list);
    if (!v) return fail(IMEXLB_E_ARG, "unknown list");
    if (cap < int64_t(v->size()) || (!out && !v->empty())) return fail(IMEXLB_E_ARG, "output too small");
    if (!v->empty()) std::memcpy(out, v->data(), v->size() * sizeof(int32_t));
    return IMEXLB_OK;
}

int imexlb_geometry_geo(imexlb_ctx *c, int32_t *geo, int64_t cap)
{
    CHECK_CTX(c);
    if (!c->geom_set) return fail(IMEXLB_E_STATE, "SetGeometry not called");
    if (!geo || cap < c->g.A) return fail(IMEXLB_E_ARG, "output too small");
    std::memcpy(geo, c->g.geo.data(), size_t(c->g.A) * sizeof(int32_t));
    return IMEXLB_OK;
}

int imexlb_bc_table(imexlb_ctx *c, int64_t *slot, int64_t *src, int64_t cap, int64_t stats[2])
{
    CHECK_CTX(c);
    if (!c->geom_set) return fail(IMEXLB_E_STATE, "SetGeometry not called");
    const int64_t n = int64_t(c->bc.entries.size());
    if (stats) {
        stats[0] = n;
        stats[1] = c->bc.order_sensitive;
    }
    if (slot || src) {
        if (cap < n) return fail(IMEXLB_E_ARG, "output too small");
        for (int64_t i = 0; i < n; ++i) {
            if (slot) slot[i] = c->bc.entries[size_t(i)].ref_slot;
            if (src) src[i] = c->bc.entries[size_t(i)].ref_src;
        }
    }
    return IMEXLB_OK;
}

int imexlb_init_up(imexlb_ctx *c, const double *r_vec)
{
    CHECK_DEV(c);
    FLUSH(c);
    if (!r_vec) return fail(IMEXLB_E_ARG, "null r_vec");
    if (!c->geom_set) return fail(IMEXLB_E_STATE, "SetGeometry before InitUP");
    HIP_TRY(hipMemcpyAsync(c->rv, r_vec, 100 * sizeof(double), hipMemcpyHostToDevice, c->stream));
    StepArgs a = c->args();
    int rc = c->launch(2, [&] { return launch_init_up(c->dim, a, c->rv, c->stream); });
    if (rc) return rc;
    HIP_TRY(hipStreamSynchronize(c->stream));  // r_vec is the caller's
    c->have_pu = true;
    c->have_f = c->have_fb = false;
    c->lazy_src = -1;
    c->stage = S_NONE;
    return IMEXLB_OK;
}


int imexlb_init_fields_f32(imexlb_ctx *c, const float *fields, int H, int W, double p_scale, double u_scale,
                           const double *r_vec)
{
    CHECK_DEV(c);
    FLUSH(c);
    if (c->dim != 2) return fail(IMEXLB_E_ARG, "FP32 field stacks are for 2D lattices");
    if (!fields || H <= 0 || W <= 0) return fail(IMEXLB_E_ARG, "fields");
    if (!c->geom_set) return fail(IMEXLB_E_STATE, "SetGeometry before setting fields");
    if (r_vec) HIP_TRY(hipMemcpyAsync(c->rv, r_vec, 100 * sizeof(double), hipMemcpyHostToDevice, c->stream));
    StepArgs a = c->args();
    int rc = c->launch(2, [&] {
        return launch_init_given(a, r_vec ? c->rv : nullptr, fields, H, W, p_scale, u_scale, c->stream);
    });
    if (rc) return rc;
    HIP_TRY(hipStreamSynchronize(c->stream));  // r_vec is the caller's
    c->have_pu = true;
    c->have_f = c->have_fb = false;
    c->lazy_src = -1;
    c->stage = S_NONE;
    return IMEXLB_OK;
}

int imexlb_body_mask_f32(imexlb_ctx *c, float *out, int H, int W)
{
    CHECK_DEV(c);
    FLUSH(c);
    if (c->dim != 2) return fail(IMEXLB_E_ARG, "body masks are for 2D lattices");
    if (!out || H <= 0 || W <= 0 || H > c->kp.ny + 1 || W > c->kp.nx + 1) return fail(IMEXLB_E_ARG, "mask size");
    if (!c->geom_set) return fail(IMEXLB_E_STATE, "SetGeometry before the body mask");
    StepArgs a = c->args();
    return c->launch(2, [&] { return launch_body_mask(a, out, H, W, c->stream); });
}

int imexlb_upload_fields(imexlb_ctx *c, const double *p, const double *u, int layout)
{
    CHECK_DEV(c);
    FLUSH(c);
    if (!p || !u) return fail(IMEXLB_E_ARG, "null field");
    if (layout != IMEXLB_LAYOUT_REF && layout != IMEXLB_LAYOUT_INTERIOR) return fail(IMEXLB_E_ARG, "layout");
    if (!c->geom_set) return fail(IMEXLB_E_STATE, "SetGeometry before upload");
    const int dim = c->dim;
    const int64_t N = c->kp.N;
    std::vector<double> hp(size_t(c->plane), 0.0), hu[3];
    for (int d = 0; d < dim; ++d) hu[d].assign(size_t(c->plane), 0.0);
    for_interior(c, [&](int, int, int, int64_t k, int64_t rid, int64_t pi) {
        if (layout == IMEXLB_LAYOUT_REF) {
            hp[size_t(pi)] = p[rid];
            for (int d = 0; d < dim; ++d) hu[d][size_t(pi)] = u[rid * dim + d];
        } else {
            hp[size_t(pi)] = p[k];
            for (int d = 0; d < dim; ++d) hu[d][size_t(pi)] = u[int64_t(d) * N + k];
        }
    });
    const size_t bytes = size_t(c->plane) * sizeof(double);
    HIP_TRY(hipMemcpy(c->p, hp.data(), bytes, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(c->ux, hu[0].data(), bytes, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(c->uy, hu[1].data(), bytes, hipMemcpyHostToDevice));
    if (dim == 3) HIP_TRY(hipMemcpy(c->uz, hu[2].data(), bytes, hipMemcpyHostToDevice));
    c->have_pu = true;
    c->have_f = c->have_fb = false;
    c->lazy_src = -1;
    c->stage = S_NONE;
    return IMEXLB_OK;
}

int imexlb_init_pdf(imexlb_ctx *c)
{
    CHECK_DEV(c);
    FLUSH(c);
    if (!c->have_pu || c->lazy_src >= 0) {
        int rc = c->materialize();
        if (rc) return rc;
    }
    StepArgs a = c->args();
    a.fout = c->f;
    int rc = c->launch(2, [&] { return launch_init_pdf(c->dim, c->prec, a, c->stream); });
    if (rc) return rc;
    c->have_f = true;
    c->have_fb = false;
    c->lazy_src = -1;
    c->stage = S_PRE;
    return IMEXLB_OK;
}

int imexlb_collision(imexlb_ctx *c)
{
    CHECK_DEV(c);
    if (c->stage == S_FUSED) {  // the fused kernel already relaxed this step
        c->cur = 1 - c->cur;
        c->stage = S_COLLIDED;
        c->prefilled = c->push_on;  // and wrote the boundary copies of its output
        return IMEXLB_OK;
    }
    if (c->stage != S_PRE) return fail(IMEXLB_E_STATE, "Collision needs InitPDF or a completed step");
    FLUSH(c);
    // write the buffer the previous step did not use: its body cells are
    // the previous values BoundaryCondition may read
    StepArgs a = c->args();
    a.src = c->f;
    a.dst = c->fb[1 - c->cur];
    int rc = c->launch(2, [&] { return launch_collide(c->dim, c->prec, a, c->stream); });
    if (rc) return rc;
    c->cur = 1 - c->cur;
    c->have_fb = true;
    c->stage = S_COLLIDED;
    c->prefilled = false;
    return IMEXLB_OK;
}

int imexlb_boundary_condition(imexlb_ctx *c)
{
    CHECK_DEV(c);
    if (c->stage != S_COLLIDED) return fail(IMEXLB_E_STATE, "BoundaryCondition must follow Collision");
    if (!c->prefilled) {
        FLUSH(c);
        int rc = c->run_fill(c->cur);
        if (rc) return rc;
    }
    c->prefilled = false;
    c->stage = S_FILLED;
    return IMEXLB_OK;
}

int imexlb_propagation(imexlb_ctx *c)
{
    CHECK_DEV(c);
    if (c->stage != S_FILLED) return fail(IMEXLB_E_STATE, "Propagation must follow BoundaryCondition");
    if (c->fused) {
        c->stage = S_PENDING;
        return IMEXLB_OK;
    }
    FLUSH(c);
    int rc = c->run_step(K_WRITE_F, c->fb[c->cur], nullptr, c->f);
    if (rc) return rc;
    c->have_f = true;
    c->lazy_src = -1;
    c->stage = S_STREAMED;
    return IMEXLB_OK;
}

int imexlb_post_processing(imexlb_ctx *c)
{
    CHECK_DEV(c);
    if (c->stage == S_PENDING) {
        if (c->can_defer()) {  // launched later, as a graph replay with its neighbours
            if (c->deferred == 0) c->defer_src = c->cur;
            ++c->deferred;
        } else {
            FLUSH(c);
            int rc = c->run_step(c->collide_mode(), c->fb[c->cur], c->fb[1 - c->cur], nullptr);
            if (rc) return rc;
        }
        c->lazy_src = c->cur;
        c->have_f = c->have_pu = false;
        c->stage = S_FUSED;
        if (c->deferred >= c->defer_chunk()) FLUSH(c);
        return IMEXLB_OK;
    }
    if (c->stage != S_STREAMED) return fail(IMEXLB_E_STATE, "PostProcessing must follow Propagation");
    FLUSH(c);
    int rc = c->run_step(K_NOSHIFT | K_WRITE_PU, c->f, nullptr, nullptr);
    if (rc) return rc;
    c->have_pu = true;
    c->stage = S_PRE;
    return IMEXLB_OK;
}

int imexlb_set_fused(imexlb_ctx *c, int fused)
{
    CHECK_CTX(c);
    FLUSH(c);
    if (c->stage == S_PENDING || c->stage == S_STREAMED)
        return fail(IMEXLB_E_STATE, "cannot switch between Propagation and PostProcessing");
    c->fused = fused != 0;
    return IMEXLB_OK;
}

static int one_step(imexlb_ctx *c)
{
    int rc;
    if ((rc = imexlb_collision(c)) || (rc = imexlb_boundary_condition(c)) || (rc = imexlb_propagation(c)) ||
        (rc = imexlb_post_processing(c)))
        return rc;
    return IMEXLB_OK;
}

// Pairs of fused steps from the steady state (stage S_FUSED, cur == X) as
// one HIP graph: per pair fill(1-X) pull(1-X -> X) fill(X) pull(X -> 1-X),
// or without the fills when the pulls push their boundary copies.  After it
// the state is again S_FUSED with cur == X, so the graph replays.
// Only kernels are recorded (no memset or copy nodes).  size: index into
// kGraphPairs (the graph's number of pairs).
static int step_graph(imexlb_ctx *c, int size, int X, hipGraphExec_t *out)
{
    const int pairs = imexlb_ctx::kGraphPairs[size];
    hipGraphExec_t &slot = c->graph[size][X];
    if (slot) {
        *out = slot;
        return IMEXLB_OK;
    }
    StepArgs a = c->args();
    HIP_TRY(hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
    hipError_t e = hipSuccess;
    for (int k = 0; k < 2 * pairs && e == hipSuccess; ++k) {
        const int b = k % 2 == 0 ? 1 - X : X;
        if (!c->push_on) {  // with pushed copies every buffer is complete already
            e = launch_fill(c->prec, c->fb[b], c->fb[1 - b], c->fill_dst, c->fill_src, c->fill32, c->nfill,
                            c->stream);
            if (e != hipSuccess) break;
        }
        a.src = c->fb[b];
        a.dst = c->fb[1 - b];
        a.fout = nullptr;
        e = launch_step(c->dim, c->prec, c->collide_mode(), a, c->stream);
    }
    hipGraph_t g = nullptr;
    hipError_t e2 = hipStreamEndCapture(c->stream, &g);
    if (e != hipSuccess || e2 != hipSuccess) {
        if (g) (void)hipGraphDestroy(g);
        return fail(IMEXLB_E_HIP, std::string("graph capture: ") + hipGetErrorString(e != hipSuccess ? e : e2));
    }
    hipGraphExec_t x = nullptr;
    e = hipGraphInstantiate(&x, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (e != hipSuccess) return fail(IMEXLB_E_HIP, std::string("graph instantiate: ") + hipGetErrorString(e));
    slot = x;
    *out = x;
    return IMEXLB_OK;
}

// n launches of `one` from fb[A], one after the other between the two buffers,
// as a graph
extern "C++" template <class F>
static int capture_passes(imexlb_ctx *c, int n, int A, hipGraphExec_t &slot, F &&one)
{
    if (slot) return IMEXLB_OK;
    StepArgs a = c->args();
    HIP_TRY(hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
    hipError_t e = hipSuccess;
    for (int k = 0; k < n && e == hipSuccess; ++k) {
        a.src = c->fb[A ^ (k & 1)];
        a.dst = c->fb[A ^ 1 ^ (k & 1)];
        e = one(a);
    }
    hipGraph_t g = nullptr;
    hipError_t e2 = hipStreamEndCapture(c->stream, &g);
    if (e != hipSuccess || e2 != hipSuccess) {
        if (g) (void)hipGraphDestroy(g);
        return fail(IMEXLB_E_HIP, std::string("graph capture: ") + hipGetErrorString(e != hipSuccess ? e : e2));
    }
    e = hipGraphInstantiate(&slot, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (e != hipSuccess) {
        slot = nullptr;
        return fail(IMEXLB_E_HIP, std::string("graph instantiate: ") + hipGetErrorString(e));
    }
    return IMEXLB_OK;
}

// The part of n fused steps from fb[A] that runs two steps per pass: fours,
// which end in the buffer they began in, leaving at least one single step
// (the last step's source buffer has to hold the step before).  Returns the
// steps taken in *done.
static int run_double_steps(imexlb_ctx *c, int A, int64_t n, int64_t *done)
{
    int64_t quads = c->dbl_on ? (n - 1) / 4 : 0;
    *done = 4 * quads;
    if (!c->graphs || c->prof) {
        for (int64_t k = 0; k < 2 * quads; ++k) {
            StepArgs a = c->args();
            a.src = c->fb[A ^ int(k & 1)];
            a.dst = c->fb[A ^ 1 ^ int(k & 1)];
            int rc = c->launch(0, [&] { return launch_double(c->prec, a, c->dbl, c->stream); }, 2);
            if (rc) return rc;
        }
        return IMEXLB_OK;
    }
    for (int j = 0; j < imexlb_ctx::kGraphSizes && quads > 0; ++j) {
        const int64_t reps = quads / imexlb_ctx::kQuads[j];
        if (reps <= 0) continue;
        hipGraphExec_t &g = c->quad_graph[j][A];
        int rc = capture_passes(c, 2 * imexlb_ctx::kQuads[j], A, g,
                                [&](const StepArgs &a) { return launch_double(c->prec, a, c->dbl, c->stream); });
        if (rc) return rc;
        for (int64_t k = 0; k < reps; ++k) HIP_TRY(hipGraphLaunch(g, c->stream));
        quads -= reps * imexlb_ctx::kQuads[j];
    }
    return IMEXLB_OK;
}

// The part of n fused steps from fb[A] that runs several steps per launch;
// only the last launch leaves the boundary copies that single steps read.
static int run_multi_steps(imexlb_ctx *c, int A, int64_t n, int64_t *done)
{
    *done = 0;
    if (!c->multi_on) return IMEXLB_OK;
    const int K = c->multi.halo;
    const MultiRun run = multi_run(c->multi, n);
    int64_t full = run.full;
    *done = run.done;
    if (run.done == 0) return IMEXLB_OK;
    if (c->graphs && !c->prof) {
        for (int j = 0; j < imexlb_ctx::kGraphSizes; ++j)
            for (; full >= imexlb_ctx::kMulti[j]; full -= imexlb_ctx::kMulti[j]) {
                hipGraphExec_t &g = c->multi_graph[j][A];
                int rc = capture_passes(c, imexlb_ctx::kMulti[j], A, g, [&](const StepArgs &a) {
                    return launch_multi(c->prec, a, c->multi, K, false, c->stream);
                });
                if (rc) return rc;
                HIP_TRY(hipGraphLaunch(g, c->stream));
            }
    }
    for (; full >= 0; --full, A = 1 - A) {
        const int steps = full > 0 ? K : run.last;
        StepArgs a = c->args();
        a.src = c->fb[A];
        a.dst = c->fb[1 - A];
        int rc = c->launch(0, [&] { return launch_multi(c->prec, a, c->multi, steps, full == 0, c->stream); }, steps);
        if (rc) return rc;
    }
    return IMEXLB_OK;
}

// n fused steps, the first reading fb[A]: two steps per pass where the
// lattice has the plan for it, then one alone if an odd number is left, then
// pairs as replays of the largest graphs that fit (the state they leave is
// the one n launches one by one would)
static int run_fused_steps(imexlb_ctx *c, int A, int64_t n)
{
    int64_t done = 0;
    int rd = c->dbl_on ? run_double_steps(c, A, n, &done) : run_multi_steps(c, A, n, &done);
    if (rd) return rd;
    n -= done;
    A ^= int(done & 1);
    if (!c->graphs || c->prof) {
        for (; n > 0; --n, A = 1 - A) {
            int rc = c->run_step(c->collide_mode(), c->fb[A], c->fb[1 - A], nullptr);
            if (rc) return rc;
        }
        return IMEXLB_OK;
    }
    if (n & 1) {
        int rc = c->run_step(c->collide_mode(), c->fb[A], c->fb[1 - A], nullptr);
        if (rc) return rc;
        A = 1 - A;
        --n;
    }
    int64_t pairs = n / 2;
    // the two steps after several per launch as they are: replaying a graph of
    // two costs more (9.9 and 8.0 us a step of five, 401 x 101 nodes)
    for (; pairs == 1 && done > 0; --pairs)
        for (int k = 0; k < 2; ++k, A = 1 - A) {
            int rc = c->run_step(c->collide_mode(), c->fb[A], c->fb[1 - A], nullptr);
            if (rc) return rc;
        }
    for (int j = 0; j < imexlb_ctx::kGraphSizes && pairs > 0; ++j) {
        const int64_t reps = pairs / imexlb_ctx::kGraphPairs[j];
        if (reps <= 0) continue;
        hipGraphExec_t g;
        int rc = step_graph(c, j, 1 - A, &g);  // from cur == X a pair first reads fb[1 - X]
        if (rc) return rc;
        for (int64_t k = 0; k < reps; ++k) HIP_TRY(hipGraphLaunch(g, c->stream));
        pairs -= reps * imexlb_ctx::kGraphPairs[j];
    }
    return IMEXLB_OK;
}

static int flush_deferred(imexlb_ctx *c)
{
    if (c->deferred == 0) return IMEXLB_OK;
    const int64_t n = c->deferred;
    c->deferred = 0;
    HIP_TRY(hipSetDevice(c->device));
    return run_fused_steps(c, c->defer_src, n);
}

int imexlb_advance(imexlb_ctx *c, int64_t nsteps)
{
    CHECK_DEV(c);
    if (nsteps < 0) return fail(IMEXLB_E_ARG, "negative step count");
    int64_t i = 0;
    // timed (profiled) runs launch kernel by kernel so each one is bracketed
    if (c->can_defer() || (c->fused && (c->dbl_on || c->multi_on))) {
        for (; i < nsteps && c->stage != S_FUSED; ++i) {
            int rc = one_step(c);
            if (rc) return rc;
        }
        if (i < nsteps) {  // the rest joins the deferred steps: from cur == X the next step reads fb[1 - X]
            if (c->deferred == 0) c->defer_src = 1 - c->cur;
            c->deferred += nsteps - i;
            c->cur ^= int((nsteps - i) & 1);  // each step's Collision flips it
            c->lazy_src = c->cur;
            c->have_f = c->have_pu = false;
            i = nsteps;
        }
        return flush_deferred(c);  // advance launches everything it was asked for
    }
    FLUSH(c);
    if (c->fused && c->graphs && !c->prof) {  // a boundary fill before every pull: graphs of whole pairs
        for (; i < nsteps && c->stage != S_FUSED; ++i) {
            int rc = one_step(c);
            if (rc) return rc;
        }
        for (int j = 0; j < imexlb_ctx::kGraphSizes; ++j) {
            const int per = imexlb_ctx::kGraphPairs[j];
            const int64_t reps = (nsteps - i) / (2 * per);
            if (reps <= 0) continue;
            hipGraphExec_t g;
            int rc = step_graph(c, j, c->cur, &g);
            if (rc) return rc;
            for (int64_t k = 0; k < reps; ++k) HIP_TRY(hipGraphLaunch(g, c->stream));
            i += 2 * per * reps;
            c->have_f = c->have_pu = false;
        }
    }
    for (; i < nsteps; ++i) {
        int rc = one_step(c);
        if (rc) return rc;
    }
    return IMEXLB_OK;
}

int imexlb_monitor(imexlb_ctx *c, double *um)
{
    CHECK_DEV(c);
    FLUSH(c);
    if (!um) return fail(IMEXLB_E_ARG, "null pointer");
    int rc = c->materialize();
    if (rc) return rc;
    StepArgs a = c->args();
    rc = c->launch(2, [&] { return launch_monitor(c->dim, a, c->skip_c, c->red, c->stream); });
    if (rc) return rc;
    unsigned long long words[2] = {0, 0};  // maximum of ux^2+uy^2, non-finite count
    HIP_TRY(hipMemcpyAsync(words, c->red, sizeof(words), hipMemcpyDeviceToHost, c->stream));
    HIP_TRY(hipStreamSynchronize(c->stream));
    if (words[1] != 0) {
        *um = std::numeric_limits<double>::quiet_NaN();
        return fail(IMEXLB_E_NAN, std::to_string(words[1]) + " fluid node(s) with a non-finite velocity");
    }
    double m;
    std::memcpy(&m, &words[0], sizeof(m));
    *um = std::sqrt(m);
    return IMEXLB_OK;
}

int imexlb_forces(imexlb_ctx *c, double F[3])
{
    CHECK_DEV(c);
    FLUSH(c);
    if (!F) return fail(IMEXLB_E_ARG, "null pointer");
    const void *buf;
    if (c->stage == S_FUSED)
        buf = c->fb[c->lazy_src];
    else if (c->have_fb && (c->stage == S_FILLED || c->stage == S_PENDING || c->stage == S_STREAMED ||
                            c->stage == S_PRE))
        buf = c->fb[c->cur];
    else
        return fail(IMEXLB_E_STATE, "forces need a step's BoundaryCondition to have run");
    int rc = c->launch(2, [&] {
        return launch_forces(c->dim, c->prec, buf, c->link_out, c->link_back, c->link_q, c->nlink, c->force_partial,
                             c->force_out, c->stream);
    });
    if (rc) return rc;
    double h[3];
    HIP_TRY(hipMemcpyAsync(h, c->force_out, sizeof(h), hipMemcpyDeviceToHost, c->stream));
    HIP_TRY(hipStreamSynchronize(c->stream));
    F[0] = h[0];
    F[1] = h[1];
    F[2] = c->dim == 3 ? h[2] : 0.0;
    return IMEXLB_OK;
}

int imexlb_mass(imexlb_ctx *c, double *m)
{
    CHECK_DEV(c);
    FLUSH(c);
    if (!m) return fail(IMEXLB_E_ARG, "null pointer");
    if (c->stage == S_NONE) return fail(IMEXLB_E_STATE, "no populations yet");
    int rc = c->materialize();
    if (rc) return rc;
    StepArgs a = c->args();
    a.src = c->f;
    double *out = c->mass_partial + MASS_BLOCKS;
    rc = c->launch(2, [&] { return launch_mass(c->dim, c->prec, a, c->mass_partial, out, c->stream); });
    if (rc) return rc;
    HIP_TRY(hipMemcpyAsync(m, out, sizeof(double), hipMemcpyDeviceToHost, c->stream));
    HIP_TRY(hipStreamSynchronize(c->stream));
    return IMEXLB_OK;
}

int imexlb_download_fields(imexlb_ctx *c, double *p, double *u, int layout)
{
    CHECK_DEV(c);
    FLUSH(c);
    if (layout != IMEXLB_LAYOUT_REF && layout != IMEXLB_LAYOUT_INTERIOR) return fail(IMEXLB_E_ARG, "layout");
    int rc = c->materialize();
    if (rc) return rc;
    const int dim = c->dim;
    const size_t bytes = size_t(c->plane) * sizeof(double);
    const int64_t N = c->kp.N;
    double *srcs[4] = {c->p, c->ux, c->uy, c->uz};
    if (layout == IMEXLB_LAYOUT_INTERIOR) {
        std::vector<FieldCopy> fields;
        for (int k = 0; k <= dim; ++k)
            if (k == 0 ? p != nullptr : u != nullptr) fields.push_back({srcs[k], k == 0 ? p : u + int64_t(k - 1) * N});
        hipError_t e;
        if (fields.empty()) return IMEXLB_OK;
        if (download_interior(c->staging, c->device, c->stream, dim, c->kp, fields, e))
            return e == hipSuccess ? IMEXLB_OK
                                   : fail(IMEXLB_E_HIP, std::string("field download: ") + hipGetErrorString(e));
    }
    std::vector<double> h(size_t(c->plane));
    for (int k = 0; k <= dim; ++k) {
        double *out = k == 0 ? p : u;
        if (!out) continue;
        HIP_TRY(hipMemcpyAsync(h.data(), srcs[k], bytes, hipMemcpyDeviceToHost, c->stream));
        HIP_TRY(hipStreamSynchronize(c->stream));
        for_interior(c, [&](int, int, int, int64_t n, int64_t rid, int64_t pi) {
            const double v = h[size_t(pi)];
            if (layout == IMEXLB_LAYOUT_REF)
                out[k == 0 ? rid : rid * dim + (k - 1)] = v;
            else
                out[k == 0 ? n : int64_t(k - 1) * N + n] = v;
        });
    }
    return IMEXLB_OK;
}


int imexlb_download_pdf(imexlb_ctx *c, int which, double *out, int layout)
{
    CHECK_DEV(c);
    FLUSH(c);
    if (!out) return fail(IMEXLB_E_ARG, "null output");
    if (layout != IMEXLB_LAYOUT_REF && layout != IMEXLB_LAYOUT_INTERIOR) return fail(IMEXLB_E_ARG, "layout");
    const void *src;
    if (which == IMEXLB_PDF_F) {
        if (c->stage == S_NONE) return fail(IMEXLB_E_STATE, "no populations yet");
        int rc = c->materialize();
        if (rc) return rc;
        src = c->f;
    } else if (which == IMEXLB_PDF_FB) {
        if (!c->have_fb) return fail(IMEXLB_E_STATE, "no post-collision state yet");
        src = c->stage == S_FUSED ? c->fb[c->lazy_src] : c->fb[c->cur];
    } else {
        return fail(IMEXLB_E_ARG, "which");
    }
    const int Q = c->Q;
    const int64_t N = c->kp.N;
    // the whole population array, then every direction of every interior node
    std::vector<uint8_t> h(size_t(Q) * size_t(c->plane) * c->ssz);
    HIP_TRY(hipMemcpyAsync(h.data(), src, h.size(), hipMemcpyDeviceToHost, c->stream));
    HIP_TRY(hipStreamSynchronize(c->stream));
    for (int q = 0; q < Q; ++q) {
        for_interior(c, [&](int, int, int, int64_t n, int64_t rid, int64_t pi) {
            const double v = load_value(h.data(), size_t(pop_slot(q, pi, c->plane, Q)), c->prec);
            if (layout == IMEXLB_LAYOUT_REF)
                out[rid * Q + q] = v;
            else
                out[int64_t(q) * N + n] = v;
        });
    }
    if (which == IMEXLB_PDF_FB && layout == IMEXLB_LAYOUT_REF) {
        for (const FillEntry &e : c->bc.entries) {
            int x, y, z;
            c->g.coords(e.ref_slot / Q, x, y, z);
            out[e.ref_slot] = load_value(h.data(), size_t(pop_slot(e.ref_slot % Q, c->pidx(x, y, z), c->plane, Q)),
                                         c->prec);
        }
    }
    return IMEXLB_OK;
}

int imexlb_synchronize(imexlb_ctx *c)
{
    CHECK_DEV(c);
    FLUSH(c);
    HIP_TRY(hipStreamSynchronize(c->stream));
    return IMEXLB_OK;
}

int imexlb_profile(imexlb_ctx *c, int enable)
{
    CHECK_DEV(c);
    FLUSH(c);
    HIP_TRY(hipStreamSynchronize(c->stream));
    for (auto &t : c->timed) {
        (void)hipEventDestroy(t.a);
        (void)hipEventDestroy(t.b);
    }
    c->timed.clear();
    for (int k = 0; k < 3; ++k) {
        c->prof_n[k] = 0;
        c->prof_ms[k] = 0.0;
    }
    c->prof = enable != 0;
    return IMEXLB_OK;
}

int imexlb_profile_read(imexlb_ctx *c, int64_t launches[3], double ms[3])
{
    CHECK_DEV(c);
    HIP_TRY(hipStreamSynchronize(c->stream));
    int rc = c->harvest(0);
    if (rc) return rc;
    for (int k = 0; k < 3; ++k) {
        if (launches) launches[k] = c->prof_n[k];
        if (ms) ms[k] = c->prof_ms[k];
    }
    return IMEXLB_OK;
}

int imexlb_info(imexlb_ctx *c, int64_t out[6])
{
    CHECK_CTX(c);
    if (!out) return fail(IMEXLB_E_ARG, "null pointer");
    out[0] = int64_t(c->kp.N);
    out[1] = int64_t(c->g.fluid_id.size());
    out[2] = int64_t(c->plane) * int64_t(c->ssz);
    out[3] = int64_t(c->dev_bytes + c->dbl_mem.bytes + c->multi_mem.bytes);
    out[4] = int64_t(c->ssz);
    out[5] = int64_t(c->bc.entries.size());
    return IMEXLB_OK;
}

int imexlb_step_form(imexlb_ctx *c, int32_t out[4])
{
    CHECK_DEV(c);
    if (!out) return fail(IMEXLB_E_ARG, "null pointer");
    if (!c->geom_set) return fail(IMEXLB_E_STATE, "SetGeometry not called");
    out[0] = c->multi_on ? c->multi.halo : c->dbl_on ? 2 : 1;
    out[1] = c->multi_on ? c->multi.wx : 0;
    out[2] = c->multi_on ? c->multi.wy : 0;
    out[3] = int32_t(c->Px);
    return IMEXLB_OK;
}

}  // extern "C"
