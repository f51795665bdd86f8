// Batched steady solves (include/cfd_hip.h, cfd_batch_*): many independent meshes of uneven
// size concatenated into one tiled device mesh, marched together with local time stepping.
//
// Every stage kernel runs once over the tiles of all instances still marching (a compacted
// tile list rebuilt on the device after each step), so large and small instances share the
// machine without per-instance launches. One whole step -- gradient and flux/stage passes of
// each RK stage, the per-instance error norm and convergence test, and the tile-list rebuild --
// is captured once in a hipGraph and replayed; the host only reads the instance status every
// `check_every` steps.
#include "../../include/cfd_hip.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <fstream>
#include <sstream>
#include <string>
#include <thread>
#include <vector>

#include "fv_kernels.h"
#include "host_ahead.h"
#include "host_rows.h"
#include "mesh_host.h"

using namespace cfd;

namespace cfd {
int capi_fail(int code, const std::string &msg);
int capi_hip_fail(hipError_t e, const char *where);
int capi_check_viscous(const cfd_config_t *c, const char *who);
void capi_fill_viscous(DevCfg &d, const cfd_config_t &c);
}  // namespace cfd

namespace {

#define BHIP(expr)                                               \
    do {                                                         \
        hipError_t _e = (expr);                                  \
        if (_e != hipSuccess) return cfd::capi_hip_fail(_e, #expr); \
    } while (0)

template <typename T>
hipError_t dalloc(T **p, size_t n) {
    *p = nullptr;
    if (n == 0) return hipSuccess;
    return hipMalloc((void **)p, n * sizeof(T));
}

template <typename T>
hipError_t h2d(T *d, const T *h, size_t n) {
    if (n == 0) return hipSuccess;
    return hipMemcpy(d, h, n * sizeof(T), hipMemcpyHostToDevice);
}

double now_s() {
    return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count();
}

}  // namespace

struct cfd_batch_s {
    int ninst = 0;
    cfd_config_t cfg{};
    DevCfg dcfg{};
    int tile = 0, face_budget = 0, block = 0;
    int nc = 0, ntiles = 0, nfe = 0, max_tile_faces = 0;
    std::vector<int> cell_off;   // [ninst+1]
    std::vector<int> inst_tile;  // [ninst+1]
    std::vector<int> iperm;      // caller cell (global) -> renumbered cell (global)
    // device mesh
    int *d_tile_cstart = nullptr, *d_tile_fstart = nullptr;
    double *d_fgeo = nullptr, *d_cw = nullptr, *d_cn = nullptr, *d_ghost_n = nullptr, *d_fd = nullptr, *d_area = nullptr, *d_inv_area = nullptr;
    double *d_fnx = nullptr, *d_fny = nullptr, *d_fdl = nullptr;
    int *d_fLR = nullptr;
    int *d_fst = nullptr;  // WENO line stencils, 4 per face entry (order 3)
    uint16_t *d_slots = nullptr;
    // tile neighbourhoods (TileRings), order 2
    int *d_rings = nullptr, *d_ring_cell = nullptr, *d_ghost = nullptr;
    uint16_t *d_own_nbr = nullptr, *d_ring_nbr = nullptr, *d_floc = nullptr;
    int *d_tile_inst = nullptr, *d_inst_tile = nullptr, *d_tile_list = nullptr, *d_tile_count = nullptr;
    int *d_status = nullptr, *d_steps = nullptr;
    int *d_fz = nullptr, *d_fz_since = nullptr;  // per instance limiter-freezing state
    double *d_fz_best = nullptr;
    float *psi = nullptr;  // [8 * face entries] frozen limiter factors
    double4 *d_inst_fs = nullptr;
    double *d_err4 = nullptr;
    // solver state
    double4 *Un = nullptr, *Ua = nullptr, *Ub = nullptr, *acc = nullptr;
    // positivity fallback: the last stage's output (copied into Un over the marching tiles), the
    // second RK4 accumulator, per-cell flags, per-tile marks with the list of marked tiles
    double4 *Uc = nullptr, *acc2 = nullptr;
    uint8_t *pflag = nullptr;
    int *dirty = nullptr;
    double *grad = nullptr, *hbuf = nullptr, *err_partial = nullptr;
    DevMesh dev{};
    hipStream_t stream = nullptr;
    hipGraph_t graph = nullptr, graph_many = nullptr;
    hipGraphExec_t exec = nullptr, exec_many = nullptr;  // one step, kGraphSteps steps
    double graph_tol = -1.0;
    int graph_tiles = 0;         // tiles the captured step's launch grids cover
    std::vector<int> fz_start;   // per instance freeze mode each solve starts with (empty: 0)
    std::vector<double> hist;    // Error[0] per instance at each check of the last solve
    int hist_checks = 0;
    cfd_progress_fn progress = nullptr;  // called every progress_every checks of a solve
    void *progress_user = nullptr;
    int progress_every = 0;
    HostRows rows;
    double build_s = 0.0, tune_s = 0.0;
    int tune_src = 0;  // launch shape: 0 given, 1 timed by the autotuner, 2 from the autotune cache
    ~cfd_batch_s() {
        for (hipGraphExec_t e : {exec, exec_many})
            if (e) (void)hipGraphExecDestroy(e);
        for (hipGraph_t g : {graph, graph_many})
            if (g) (void)hipGraphDestroy(g);
        if (stream) (void)hipStreamDestroy(stream);
        void *ps[] = {d_tile_cstart, d_tile_fstart, d_fgeo, d_cw, d_cn, d_ghost_n, d_fd, d_rings, d_ring_cell, d_ghost, d_own_nbr, d_ring_nbr, d_floc, d_fnx, d_fny, d_fdl, d_fLR, d_fst, d_area, d_inv_area, d_slots, d_tile_inst, d_inst_tile,
                      d_tile_list, d_tile_count, d_status, d_steps, d_inst_fs, d_err4,
                      Un, Ua, Ub, acc, grad, hbuf, err_partial, d_fz, d_fz_since, d_fz_best, psi,
                      Uc, acc2, pflag, dirty};
        for (void *p : ps)
            if (p) (void)hipFree(p);
    }
};

namespace {

struct InstanceInput {
    int npts, ncells;
    const double *pts;
    const int *cells;
};

int check_batch_config(const cfd_config_t *c) {
    if (c->flux < 0 || c->flux > 3) return capi_fail(CFD_E_ARG, "batch config: flux must be 0..3");
    if (c->order < 1 || c->order > 3) return capi_fail(CFD_E_ARG, "batch config: order must be 1, 2 or 3 (WENO5)");
    if (c->order == 3 && (c->freeze_tol > 0.0 || c->freeze_stall > 0))
        return capi_fail(CFD_E_ARG, "batch config: limiter freezing needs order 2");
    if (c->limiter < 0 || c->limiter > 4) return capi_fail(CFD_E_ARG, "batch config: limiter must be 0..4");
    if (c->gradient < 0 || c->gradient > 1) return capi_fail(CFD_E_ARG, "batch config: gradient must be 0 or 1");
    if (c->xcd_remap < 0 || c->xcd_remap > 4096) return capi_fail(CFD_E_ARG, "batch config: xcd_remap must be in 0..4096");
    if (!(c->cfl > 0.0)) return capi_fail(CFD_E_ARG, "batch config: cfl must be positive");
    if (c->rk != 3 && c->rk != 4) return capi_fail(CFD_E_ARG, "batch config: rk must be 3 or 4");
    if (c->ref_mode) return capi_fail(CFD_E_ARG, "batch config: the reference iteration is not batched");
    if (!(c->freeze_tol >= 0.0) || c->freeze_stall < 0)
        return capi_fail(CFD_E_ARG, "batch config: freeze_tol and freeze_stall must be >= 0");
    if (!c->lts) return capi_fail(CFD_E_ARG, "batch config: batched steady solves use local time stepping (lts = 1)");
    if (c->positivity < 0 || c->positivity > 2)
        return capi_fail(CFD_E_ARG, "batch config: positivity must be 0, 1 or 2");
    if (c->positivity && (c->order != 2 || c->viscous))
        return capi_fail(CFD_E_ARG, "batch config: the positivity fallback needs order 2, inviscid");
    for (int k = 1; k <= 5; k++)
        if (c->bc[k] < 1 || c->bc[k] > 10) return capi_fail(CFD_E_ARG, "batch config: bc types must be 1..10");
    if (!(c->p_exit >= 0.0) || !std::isfinite(c->p_exit))
        return capi_fail(CFD_E_ARG, "batch config: p_exit must be finite and >= 0");
    return capi_check_viscous(c, "batch config");
}

// Builds connectivity and tiled layouts of the instances (in parallel), concatenates them on
// the device and allocates the solver state.
int build_batch(const std::vector<InstanceInput> &in, const double *fs4, const cfd_config_t &cfg,
                int tile, int face_budget, int block, int nthreads, cfd_batch_s **out) {
    *out = nullptr;
    const int ni = (int)in.size();
    std::vector<Layout> lays(ni);
    std::vector<std::vector<int>> sts(ni);  // WENO line stencils (order 3)
    std::vector<TileRings> rgs(ni);         // tile neighbourhoods (order 2)
    std::vector<std::string> errs(ni);
    {
        std::atomic<int> next{0};
        auto work = [&]() {
            for (;;) {
                const int i = next.fetch_add(1);
                if (i >= ni) break;
                try {
                    RefMesh rm;
                    build_ref_mesh(in[i].npts, in[i].pts, in[i].ncells, in[i].cells, rm);
                    build_layout(rm, tile, 1, lays[i], face_budget);
                    if (cfg.order == 3) line_stencils(rm, lays[i], sts[i]);
                    if (cfg.order == 2) tile_rings(rm, lays[i], rgs[i]);
                } catch (const std::exception &e) {
                    errs[i] = e.what();
                }
            }
        };
        const int nt = std::max(1, std::min(nthreads, ni));
        std::vector<std::thread> th;
        for (int t = 1; t < nt; t++) th.emplace_back(work);
        work();
        for (auto &t : th) t.join();
    }
    for (int i = 0; i < ni; i++)
        if (!errs[i].empty()) return capi_fail(CFD_E_MESH, "cfd_batch_create: instance " + std::to_string(i) + ": " + errs[i]);

    cfd_batch_s *b = new cfd_batch_s();
    b->ninst = ni;
    b->cfg = cfg;
    b->tile = tile;
    b->face_budget = face_budget;
    b->block = block;
    b->cell_off.assign(ni + 1, 0);
    b->inst_tile.assign(ni + 1, 0);
    std::vector<int> fe_off(ni + 1, 0);
    for (int i = 0; i < ni; i++) {
        b->cell_off[i + 1] = b->cell_off[i] + (int)lays[i].area.size();
        b->inst_tile[i + 1] = b->inst_tile[i] + lays[i].ntiles;
        fe_off[i + 1] = fe_off[i] + (int)lays[i].fL.size();
        b->max_tile_faces = std::max(b->max_tile_faces, lays[i].max_tile_faces);
    }
    // offsets of the instances' ring cells and ghosts
    bool rings = cfg.order == 2;
    std::vector<size_t> rc_off(ni + 1, 0), gh_off(ni + 1, 0);
    for (int i = 0; i < ni; i++) {
        rings = rings && rgs[i].ok;
        rc_off[i + 1] = rc_off[i] + rgs[i].cell.size();
        gh_off[i + 1] = gh_off[i] + rgs[i].ghost.size() / 2;
        b->dev.max_local = std::max(b->dev.max_local, rgs[i].max_local);
        b->dev.max_grad = std::max(b->dev.max_grad, rgs[i].max_grad);
        b->dev.first_ring += rgs[i].first_ring;
    }
    rings = rings && rc_off[ni] <= 0x7FFFFFFFu;
    b->nc = b->cell_off[ni];
    b->ntiles = b->inst_tile[ni];
    b->nfe = fe_off[ni];
    const size_t nc = b->nc, nt = b->ntiles, nfe = b->nfe;
    hipError_t e = hipSuccess;
#define BALLOC(p, n)                                   \
    if ((e = dalloc(&(p), (n))) != hipSuccess) {       \
        delete b;                                      \
        return capi_hip_fail(e, "cfd_batch_create alloc"); \
    }
    BALLOC(b->d_tile_cstart, nt + 1);
    BALLOC(b->d_tile_fstart, nt + 1);
    BALLOC(b->d_fgeo, 6 * nfe);
    if (cfg.order >= 2) BALLOC(b->d_cw, 8 * nc);
    if (rings) {
        BALLOC(b->d_rings, 4 * nt);
        BALLOC(b->d_ring_cell, rc_off[ni]);
        BALLOC(b->d_own_nbr, 4 * nc);
        BALLOC(b->d_ring_nbr, 4 * rc_off[ni]);
        BALLOC(b->d_ghost, 2 * gh_off[ni]);
        BALLOC(b->d_ghost_n, 2 * gh_off[ni]);
        BALLOC(b->d_floc, 2 * nfe);
        BALLOC(b->d_fd, 2 * nfe);
        if (cfg.gradient == GRAD_GG) BALLOC(b->d_cn, 12 * nc);
    }
    BALLOC(b->d_fLR, 2 * nfe);
    BALLOC(b->d_fnx, nfe);
    BALLOC(b->d_fny, nfe);
    BALLOC(b->d_fdl, nfe);
    BALLOC(b->d_slots, 4 * nc);
    BALLOC(b->d_area, nc);
    BALLOC(b->d_inv_area, nc);
    BALLOC(b->d_tile_inst, nt);
    BALLOC(b->d_inst_tile, (size_t)ni + 1);
    BALLOC(b->d_tile_list, nt);
    BALLOC(b->d_tile_count, 1);
    BALLOC(b->d_status, (size_t)ni);
    BALLOC(b->d_steps, (size_t)ni);
    BALLOC(b->d_inst_fs, (size_t)ni);
    BALLOC(b->d_err4, 4 * (size_t)ni);
    BALLOC(b->Un, nc);
    BALLOC(b->Ua, nc);
    BALLOC(b->Ub, nc);
    if (cfg.rk == 4) BALLOC(b->acc, nc);
    if (cfg.positivity) {
        BALLOC(b->Uc, nc);
        if (cfg.rk == 4) BALLOC(b->acc2, nc);
        BALLOC(b->pflag, nc);
        BALLOC(b->dirty, 2 * nt + 4);
        if ((e = hipMemset(b->dirty, 0, (2 * nt + 4) * sizeof(int))) != hipSuccess) {
            delete b;
            return capi_hip_fail(e, "cfd_batch_create alloc");
        }
    }
    if (cfg.order >= 2) BALLOC(b->grad, 8 * nc);
    if (cfg.order == 3) BALLOC(b->d_fst, 4 * nfe);
    BALLOC(b->hbuf, nc);
    BALLOC(b->err_partial, 4 * nt);
    if (cfg.order == 2 && (cfg.freeze_tol > 0.0 || cfg.freeze_stall > 0)) {
        BALLOC(b->d_fz, (size_t)ni);
        BALLOC(b->d_fz_since, (size_t)ni);
        BALLOC(b->d_fz_best, (size_t)ni);
        BALLOC(b->psi, 8 * nfe);
    }
#undef BALLOC
    b->iperm.resize(nc);
    // The device records, 200 to 300 bytes a cell beside the layouts: packed by other threads, a few groups
    // of instances ahead, while the groups before are copied. A group is an instance, or several small ones
    // in a row, whose arrays go in one copy each (creating 256 instances of 2k cells: 95 ms with copies of
    // every instance's, 36 so).
    constexpr size_t kGroupCells = 32768;
    std::vector<int> group(1, 0);  // first instance of each group, and the end
    for (int i = 1; i <= ni; i++)
        if (i == ni || (size_t)(b->cell_off[i + 1] - b->cell_off[group.back()]) > kGroupCells) group.push_back(i);
    struct Packed {
        std::vector<double> geo, cw, cn, fd, fnx, fny, fdl, area, inv_area, ghost_n;
        std::vector<int> lr, tc, tf, ti, st, rings, ring_cell, ghost;
        std::vector<uint16_t> slots, own, ring, face;
    };
    auto pack = [&](int g) {
        Packed pk;
        auto add = [](auto &all, auto &&part) {
            if (all.empty()) all = std::move(part);
            else all.insert(all.end(), part.begin(), part.end());
        };
        for (int i = group[g]; i < group[g + 1]; i++) {
            Layout L = std::move(lays[i]);
            TileRings rg = std::move(rgs[i]);
            std::vector<int> st = std::move(sts[i]);
            const int cb = b->cell_off[i], fb = fe_off[i];
            std::vector<double> geo, v;
            std::vector<int> lr;
            pack_face_geometry(L, cb, geo, lr);
            add(pk.geo, std::move(geo));
            add(pk.lr, std::move(lr));
            if (cfg.order >= 2) {
                cell_face_vectors(L, v);
                add(pk.cw, std::move(v));
            }
            if (rings) {
                face_offsets(L, v);
                add(pk.fd, std::move(v));
                if (cfg.gradient == GRAD_GG) {
                    cell_face_normals(L, v);
                    add(pk.cn, std::move(v));
                }
                for (size_t t = 0; t < (size_t)L.ntiles; t++) {
                    rg.tiles[4 * t] += (int)rc_off[i];
                    rg.tiles[4 * t + 3] += (int)gh_off[i];
                }
                for (int &c : rg.cell) c += cb;
                for (size_t k = 0; k < rg.ghost.size(); k += 2) rg.ghost[k] += cb;
                add(pk.rings, std::move(rg.tiles));
                add(pk.ring_cell, std::move(rg.cell));
                add(pk.own, std::move(rg.own));
                add(pk.ring, std::move(rg.ring));
                add(pk.ghost, std::move(rg.ghost));
                add(pk.ghost_n, std::move(rg.ghost_n));
                add(pk.face, std::move(rg.face));
            }
            for (int &c : st)
                if (c >= 0) c += cb;
            add(pk.st, std::move(st));
            pk.ti.insert(pk.ti.end(), L.ntiles, i);
            for (int t = 0; t < L.ntiles; t++) {
                pk.tc.push_back(L.tile_cstart[t] + cb);
                pk.tf.push_back(L.tile_fstart[t] + fb);
            }
            for (size_t c = 0; c < L.iperm.size(); c++) b->iperm[cb + c] = cb + L.iperm[c];
            add(pk.fnx, std::move(L.fnx));
            add(pk.fny, std::move(L.fny));
            add(pk.fdl, std::move(L.fdl));
            add(pk.slots, std::move(L.slots));
            add(pk.area, std::move(L.area));
            add(pk.inv_area, std::move(L.inv_area));
        }
        return pk;
    };
    auto copy = [&](int g, const Packed &pk) {
        const int i = group[g];
        const size_t cb = b->cell_off[i], tb = b->inst_tile[i], fb = fe_off[i];
        auto put = [&](auto *d, size_t at, const auto &v) {
            if (e == hipSuccess && d) e = h2d(d + at, v.data(), v.size());
        };
        put(b->d_tile_cstart, tb, pk.tc);
        put(b->d_tile_fstart, tb, pk.tf);
        put(b->d_tile_inst, tb, pk.ti);
        put(b->d_fgeo, 6 * fb, pk.geo);
        put(b->d_cw, 8 * cb, pk.cw);
        put(b->d_fLR, 2 * fb, pk.lr);
        put(b->d_fst, 4 * fb, pk.st);
        put(b->d_fnx, fb, pk.fnx);
        put(b->d_fny, fb, pk.fny);
        put(b->d_fdl, fb, pk.fdl);
        put(b->d_slots, 4 * cb, pk.slots);
        put(b->d_area, cb, pk.area);
        put(b->d_inv_area, cb, pk.inv_area);
        put(b->d_rings, 4 * tb, pk.rings);
        put(b->d_ring_cell, rc_off[i], pk.ring_cell);
        put(b->d_own_nbr, 4 * cb, pk.own);
        put(b->d_ring_nbr, 4 * rc_off[i], pk.ring);
        put(b->d_ghost, 2 * gh_off[i], pk.ghost);
        put(b->d_ghost_n, 2 * gh_off[i], pk.ghost_n);
        put(b->d_floc, 2 * fb, pk.face);
        put(b->d_fd, 2 * fb, pk.fd);
        put(b->d_cn, 12 * cb, pk.cn);
        return e == hipSuccess;
    };
    try {
        const int groups = (int)group.size() - 1;
        in_turn(groups, std::max(1, std::min(nthreads, groups)) - 1, pack, copy);
    } catch (const std::exception &x) {
        delete b;
        return capi_fail(CFD_E_MESH, std::string("cfd_batch_create: ") + x.what());
    }
    if (e != hipSuccess) {
        delete b;
        return capi_hip_fail(e, "cfd_batch_create upload");
    }
    const int last_c = b->nc, last_f = b->nfe;
    std::vector<double4> fsv(ni);
    for (int i = 0; i < ni; i++) fsv[i] = make_double4(fs4[4 * i], fs4[4 * i + 1], fs4[4 * i + 2], fs4[4 * i + 3]);
    if ((e = h2d(b->d_tile_cstart + nt, &last_c, 1)) != hipSuccess ||
        (e = h2d(b->d_tile_fstart + nt, &last_f, 1)) != hipSuccess ||
        (e = h2d(b->d_inst_tile, b->inst_tile.data(), (size_t)ni + 1)) != hipSuccess ||
        (e = h2d(b->d_inst_fs, fsv.data(), (size_t)ni)) != hipSuccess ||
        (e = hipStreamCreate(&b->stream)) != hipSuccess) {
        delete b;
        return capi_hip_fail(e, "cfd_batch_create upload");
    }
    DevMesh &d = b->dev;
    d.nc = b->nc;
    d.ntiles = b->ntiles;
    d.tile = tile;
    d.max_tile_faces = b->max_tile_faces;
    d.nfe = b->nfe;
    d.tile_cstart = b->d_tile_cstart;
    d.tile_fstart = b->d_tile_fstart;
    d.fgeo = reinterpret_cast<const double2 *>(b->d_fgeo);
    d.cw = reinterpret_cast<const double2 *>(b->d_cw);
    if (rings) {
        d.rings = reinterpret_cast<const int4 *>(b->d_rings);
        d.ring_cell = b->d_ring_cell;
        d.own_nbr = reinterpret_cast<const ushort4 *>(b->d_own_nbr);
        d.ring_nbr = reinterpret_cast<const ushort4 *>(b->d_ring_nbr);
        d.ghost = reinterpret_cast<const int2 *>(b->d_ghost);
        d.ghost_n = reinterpret_cast<const double2 *>(b->d_ghost_n);
        d.fd = reinterpret_cast<const double2 *>(b->d_fd);
        d.floc = reinterpret_cast<const ushort2 *>(b->d_floc);
        d.cn = b->d_cn;
    }
    d.fLR = reinterpret_cast<const int2 *>(b->d_fLR);
    d.fst = reinterpret_cast<const int4 *>(b->d_fst);
    d.fnx = b->d_fnx;
    d.fny = b->d_fny;
    d.fdl = b->d_fdl;
    d.slots = b->d_slots;
    d.area = b->d_area;
    d.inv_area = b->d_inv_area;
    d.tile_inst = b->d_tile_inst;
    d.inst_fs = b->d_inst_fs;
    d.tile_list = b->d_tile_list;
    d.tile_count = b->d_tile_count;
    for (int k = 0; k < 6; k++) b->dcfg.bc[k] = cfg.bc[k];
    for (int k = 0; k < 4; k++) b->dcfg.fs[k] = 0.0;
    b->dcfg.cfl = cfg.cfl;
    b->dcfg.roe_bdiss = cfg.roe_bdiss;
    b->dcfg.xcd_remap = cfg.xcd_remap;
    b->dcfg.grad_lds = cfg.grad_lds;
    b->dcfg.p_exit = cfg.p_exit;  // 0: each instance's prescribed p
    capi_fill_viscous(b->dcfg, cfg);
    const size_t sm = flux_smem_bytes(d, cfg.order, cfg.grad_lds);
    if (sm > 65536 || grad_smem_bytes(d, cfg.gradient) > 65536) {
        delete b;
        return capi_fail(CFD_E_ARG, "cfd_batch_create: tile too large for 64 KiB of LDS per workgroup");
    }
    *out = b;
    return 0;
}

// Marks every instance as marching and rebuilds the full tile list.
int batch_reset(cfd_batch_s *b) {
    std::vector<int> ones(b->ninst, 1), zeros(b->ninst, 0);
    BHIP(h2d(b->d_status, ones.data(), ones.size()));
    BHIP(h2d(b->d_steps, zeros.data(), zeros.size()));
    if (b->d_fz) {
        std::vector<double> big(b->ninst, 1.7976931348623157e308);
        BHIP(h2d(b->d_fz, b->fz_start.empty() ? zeros.data() : b->fz_start.data(), zeros.size()));
        BHIP(h2d(b->d_fz_since, zeros.data(), zeros.size()));
        BHIP(h2d(b->d_fz_best, big.data(), big.size()));
    }
    BHIP(launch_batch_list(b->ninst, b->ntiles, b->d_inst_tile, b->d_tile_inst, b->d_status, b->d_tile_list,
                           b->d_tile_count, b->stream));
    return 0;
}

// The launches of one step on b->stream (captured into the graph). The tile passes' grids cover
// `grid_tiles` tiles (at least the tiles still marching: the compacted list never grows during a
// solve), so that a batch whose instances have mostly converged launches few empty workgroups.
int batch_step_launches(cfd_batch_s *b, double tol, int grid_tiles) {
    const cfd_config_t &c = b->cfg;
    const DevMesh &dm = b->dev;
    DevCfg dc = b->dcfg;
    dc.grid_tiles = grid_tiles;
    const int nst = (c.rk == 4) ? 4 : 3;
    // With the positivity fallback no stage writes an array it reads (its recomputation reads the
    // stage inputs again): the last stage writes Uc, copied into Un over the marching tiles after
    // the step, and the RK4 accumulator alternates between acc and acc2.
    const bool pos = c.positivity != 0;
    double4 *last = pos ? b->Uc : b->Un;
    const double4 *ins3[3] = {b->Un, b->Ua, b->Ub};
    double4 *outs3[3] = {b->Ua, b->Ub, last};
    const double4 *ins4[4] = {b->Un, b->Ua, b->Ub, b->Ua};
    double4 *outs4[4] = {b->Ua, b->Ub, b->Ua, last};
    double4 *acc_w[4] = {b->acc, pos ? b->acc2 : b->acc, b->acc, b->acc};
    const double4 *acc_r[4] = {b->acc, b->acc, pos ? b->acc2 : b->acc, b->acc};
    for (int k = 0; k < nst; k++) {
        const double4 *in = (nst == 4) ? ins4[k] : ins3[k];
        double4 *out = (nst == 4) ? outs4[k] : outs3[k];
        if (c.order == 3) BHIP(launch_grad(dm, dc, c.gradient, in, b->grad, b->block, b->stream));
        StageArgs a{};
        a.rk = nst;
        a.stage = k;
        a.lts = 1;
        a.last = (k == nst - 1);
        a.Un = b->Un;
        a.Uout = out;
        a.acc_in = acc_r[k];
        a.acc_out = acc_w[k];
        a.hbuf = b->hbuf;
        a.err_partial = a.last ? b->err_partial : nullptr;
        a.freeze = b->d_fz;
        a.psi = b->psi;
        if (pos) {
            // the stages of one captured step use the marked-tile counts 0 .. nst-1 in turn
            a.pflag = b->pflag;
            a.dirty = b->dirty;
            a.pos_range = (c.positivity == 1 ? 1 : 0) | (k << 1) | (((k + 1) % nst) << 3);
            for (int pass = 1; pass <= 2; pass++)
                BHIP(launch_second_order(dm, dc, c.flux, c.limiter, c.gradient, MODE_STAGE, in, b->grad, false, a, pass,
                                         b->block, b->stream));
        } else if (c.order == 2) {
            BHIP(launch_second_order(dm, dc, c.flux, c.limiter, c.gradient, MODE_STAGE, in, b->grad, false, a, 0, b->block,
                                     b->stream));
        } else {
            BHIP(launch_flux(dm, dc, c.flux, c.order, c.limiter, MODE_STAGE, in, b->grad, a, b->block, b->stream));
        }
    }
    if (pos) BHIP(launch_batch_commit(dm, grid_tiles, b->Uc, b->Un, b->stream));
    BHIP(launch_batch_status(b->ninst, b->d_inst_tile, b->err_partial, tol, b->d_status, b->d_steps, b->d_err4,
                             b->d_fz, b->d_fz_best, b->d_fz_since, c.freeze_tol, c.freeze_stall, b->stream));
    BHIP(launch_batch_list(b->ninst, b->ntiles, b->d_inst_tile, b->d_tile_inst, b->d_status, b->d_tile_list,
                           b->d_tile_count, b->stream));
    return 0;
}

// Captures `steps` steps into *g and *exec (replacing what they held).
int batch_capture(cfd_batch_s *b, double tol, int grid_tiles, int steps, hipGraph_t *g, hipGraphExec_t *exec) {
    if (*exec) BHIP(hipGraphExecDestroy(*exec));
    *exec = nullptr;
    if (*g) BHIP(hipGraphDestroy(*g));
    *g = nullptr;
    BHIP(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
    int rc = 0;
    for (int k = 0; k < steps && !rc; k++) rc = batch_step_launches(b, tol, grid_tiles);
    hipGraph_t got = nullptr;
    hipError_t e = hipStreamEndCapture(b->stream, &got);
    if (rc) {
        if (got) (void)hipGraphDestroy(got);
        return rc;
    }
    if (e != hipSuccess) return capi_hip_fail(e, "hipStreamEndCapture");
    *g = got;
    BHIP(hipGraphInstantiate(exec, *g, nullptr, nullptr, 0));
    return 0;
}

int batch_graph(cfd_batch_s *b, double tol, int grid_tiles = -1) {
    if (grid_tiles < 0) grid_tiles = b->ntiles;
    if (b->exec && b->graph_tol == tol && b->graph_tiles == grid_tiles) return 0;
    if (b->exec_many) BHIP(hipGraphExecDestroy(b->exec_many));
    b->exec_many = nullptr;
    if (int rc = batch_capture(b, tol, grid_tiles, 1, &b->graph, &b->exec)) return rc;
    b->graph_tol = tol;
    b->graph_tiles = grid_tiles;
    return 0;
}

// `n` steps of the captured kind. The device idles 9 us between two graphs, so longer runs replay
// graphs of several steps (captured when a run first has kMany of them).
constexpr int kGraphSteps = 8, kMany = 2 * kGraphSteps;
int batch_many(cfd_batch_s *b, int n) {
    if (n < kMany || b->exec_many) return 0;
    return batch_capture(b, b->graph_tol, b->graph_tiles, kGraphSteps, &b->graph_many, &b->exec_many);
}
int batch_launch(cfd_batch_s *b, int n) {
    if (int rc = batch_many(b, n)) return rc;
    for (; n >= kGraphSteps && b->exec_many; n -= kGraphSteps) BHIP(hipGraphLaunch(b->exec_many, b->stream));
    for (; n > 0; n--) BHIP(hipGraphLaunch(b->exec, b->stream));
    return 0;
}

// Time of `n` steps (after one warm-up step) on the current state, in milliseconds.
int batch_time_steps(cfd_batch_s *b, int n, double *ms) {
    int rc = batch_reset(b);
    if (rc) return rc;
    rc = batch_graph(b, -1.0);  // tol < 0: nothing converges while timing
    if (rc) return rc;
    if ((rc = batch_many(b, n)) || (rc = batch_launch(b, 1))) return rc;
    hipEvent_t e0, e1;
    BHIP(hipEventCreate(&e0));
    BHIP(hipEventCreate(&e1));
    BHIP(hipEventRecord(e0, b->stream));
    if ((rc = batch_launch(b, n))) return rc;
    BHIP(hipEventRecord(e1, b->stream));
    BHIP(hipEventSynchronize(e1));
    float f = 0.f;
    BHIP(hipEventElapsedTime(&f, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    *ms = f;
    return 0;
}

// Steps the autotuner marches each candidate from freestream before timing it.
constexpr int kTuneDevelop = 200;

// `n` graph-launched steps of the current state (tolerance -1: nothing converges), then a wait.
int batch_march(cfd_batch_s *b, int n) {
    int rc = batch_reset(b);
    if (rc) return rc;
    rc = batch_graph(b, -1.0);
    if (rc) return rc;
    if ((rc = batch_launch(b, n))) return rc;
    BHIP(hipStreamSynchronize(b->stream));
    return 0;
}

// ---- autotune cache --------------------------------------------------------------------------
// One JSON object in a file, one entry per line: "key": [tile, face budget, block, ms per cell].
// The key names the GPU (architecture, compute units), the batch's statistics (instances, total
// and largest cell counts in powers of two), the scheme and the kernels, so a batch of the same shape
// on the same GPU reuses the measured choice. Path: CFD_AUTOTUNE_CACHE, else $HOME/.cache/cfdhip_autotune.json;
// an unreadable or unwritable file only disables the cache.
std::string tune_cache_path() {
    if (const char *p = std::getenv("CFD_AUTOTUNE_CACHE")) return p;
    if (const char *h = std::getenv("HOME")) return std::string(h) + "/.cache/cfdhip_autotune.json";
    return "";
}

int ilog2(long v) {
    int k = 0;
    while (v > 1) {
        v >>= 1;
        k++;
    }
    return k;
}

// The kernels that a cached shape was timed with: the build gives a digest of their sources and flags, so
// that an entry of other kernels is not found. (The one-launch second-order pass moved the ramps' best
// shape from 128-cell to 256-cell tiles.)
#ifndef CFD_KERNELS
#error "CFD_KERNELS: digest of the kernel sources (build.py)"
#endif
#define CFD_TEXT_(x) #x
#define CFD_TEXT(x) CFD_TEXT_(x)

std::string tune_key(const cfd_config_t &c, const std::vector<InstanceInput> &in) {
    int dev = 0;
    hipDeviceProp_t p{};
    std::string arch = "unknown";
    int cus = 0;
    if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&p, dev) == hipSuccess) {
        arch = p.gcnArchName;
        cus = p.multiProcessorCount;
    }
    long total = 0, largest = 0;
    for (const auto &x : in) {
        total += x.ncells;
        largest = std::max<long>(largest, x.ncells);
    }
    std::ostringstream k;
    k << arch << ":" << cus << "|inst2^" << ilog2((long)in.size()) << "|cells2^" << ilog2(total) << "|max2^"
      << ilog2(largest) << "|order" << c.order << "|flux" << c.flux << "|lim" << c.limiter << "|grad"
      << c.gradient << "|visc" << c.viscous << "|rk" << c.rk << "|pos" << c.positivity << "|freeze"
      << (c.freeze_tol > 0.0 || c.freeze_stall > 0) << "|kernels" CFD_TEXT(CFD_KERNELS);
    std::string s = k.str();
    for (char &ch : s)
        if (ch == '"' || ch == '\\') ch = '_';
    return s;
}

// entries of the cache file: key -> "[tile, budget, block, per_cell]"
std::vector<std::pair<std::string, std::string>> tune_cache_load(const std::string &path) {
    std::vector<std::pair<std::string, std::string>> out;
    if (path.empty()) return out;
    std::ifstream f(path);
    std::string line;
    while (std::getline(f, line)) {
        const size_t a = line.find('"'), b = line.find("\": [");
        const size_t e = line.find(']', b == std::string::npos ? 0 : b);
        if (a == std::string::npos || b == std::string::npos || e == std::string::npos || b < a) continue;
        out.emplace_back(line.substr(a + 1, b - a - 1), line.substr(b + 3, e - b - 2));
    }
    return out;
}

bool tune_cache_get(const std::string &path, const std::string &key, int *tile, int *budget, int *block) {
    for (const auto &kv : tune_cache_load(path)) {
        if (kv.first != key) continue;
        int t = 0, bu = 0, bl = 0;
        if (std::sscanf(kv.second.c_str(), "[%d, %d, %d", &t, &bu, &bl) == 3 && t > 0 && bu > 0 &&
            (bl == 64 || bl == 128 || bl == 256) && t <= bl) {
            *tile = t;
            *budget = bu;
            *block = bl;
            return true;
        }
    }
    return false;
}

void tune_cache_put(const std::string &path, const std::string &key, int tile, int budget, int block,
                    double per_cell) {
    if (path.empty()) return;
    auto entries = tune_cache_load(path);
    char val[128];
    std::snprintf(val, sizeof(val), "[%d, %d, %d, %.6e]", tile, budget, block, per_cell);
    bool found = false;
    for (auto &kv : entries)
        if (kv.first == key) {
            kv.second = val;
            found = true;
        }
    if (!found) entries.emplace_back(key, val);
    const std::string tmp = path + ".tmp" + std::to_string((long)std::chrono::steady_clock::now().time_since_epoch().count());
    {
        std::ofstream f(tmp);
        if (!f) return;
        f << "{\n";
        for (size_t i = 0; i < entries.size(); i++)
            f << "\"" << entries[i].first << "\": " << entries[i].second << (i + 1 < entries.size() ? ",\n" : "\n");
        f << "}\n";
        if (!f) return;
    }
    (void)std::rename(tmp.c_str(), path.c_str());
}

int set_freestream(cfd_batch_s *b, const double *fs4) {
    std::vector<double4> U(b->nc);
    const double gm1 = 1.4 - 1.0;  // formed as the reference forms gamma - 1 (include/definitions.h:62-64)
    for (int i = 0; i < b->ninst; i++) {
        const double r = fs4[4 * i], u = fs4[4 * i + 1], v = fs4[4 * i + 2], p = fs4[4 * i + 3];
        const double4 q = make_double4(r, r * u, r * v, p / gm1 + 0.5 * r * (u * u + v * v));
        for (int c = b->cell_off[i]; c < b->cell_off[i + 1]; c++) U[c] = q;
    }
    BHIP(h2d(b->Un, U.data(), U.size()));
    return 0;
}

}  // namespace

extern "C" {

int cfd_batch_create(int ninst, const int *pt_off, const double *pts3, const int *cell_off,
                     const int *cells4, const double *fs4, const cfd_config_t *cfg, int nthreads,
                     cfd_batch_t **out) {
    if (!out || !pt_off || !pts3 || !cell_off || !cells4 || !fs4 || !cfg || ninst <= 0)
        return capi_fail(CFD_E_ARG, "cfd_batch_create: bad arguments");
    *out = nullptr;
    int rc = check_batch_config(cfg);
    if (rc) return rc;
    std::vector<InstanceInput> in(ninst);
    for (int i = 0; i < ninst; i++) {
        const int np = pt_off[i + 1] - pt_off[i], nc = cell_off[i + 1] - cell_off[i];
        if (np <= 0 || nc <= 0) return capi_fail(CFD_E_ARG, "cfd_batch_create: empty instance " + std::to_string(i));
        in[i] = InstanceInput{np, nc, pts3 + 3 * (size_t)pt_off[i], cells4 + 4 * (size_t)cell_off[i]};
    }
    const double t0 = now_s();
    int tile = 0, budget = 0, block = cfg->block;
    double tune_s = 0.0;
    int tune_src = 0;
    const std::string cache = (block == 0) ? tune_cache_path() : std::string();
    const std::string key = (block == 0) ? tune_key(*cfg, in) : std::string();
    if (block == 0 && tune_cache_get(cache, key, &tile, &budget, &block)) {
        tune_src = 2;
    } else if (block == 0) {
        // Autotune: time each (tile, face budget, block) candidate on a sample of the instances
        // (the largest ones, up to ~1.5M cells) and keep the fastest per cell.
        std::vector<int> order(ninst);
        for (int i = 0; i < ninst; i++) order[i] = i;
        std::sort(order.begin(), order.end(), [&](int a, int c) { return in[a].ncells > in[c].ncells; });
        std::vector<InstanceInput> sample;
        std::vector<double> sfs;
        long cells = 0;
        for (int i : order) {
            if (cells > 1500000 && !sample.empty()) break;
            sample.push_back(in[i]);
            for (int k = 0; k < 4; k++) sfs.push_back(fs4[4 * i + k]);
            cells += in[i].ncells;
        }
        const int cand[][3] = {{64, 128, 64}, {128, 256, 128}, {128, 320, 128}, {256, 512, 256}};
        double best = 1e300;
        for (const auto &cd : cand) {
            cfd_batch_s *sb = nullptr;
            cfd_config_t sc = *cfg;
            sc.block = cd[2];
            rc = build_batch(sample, sfs.data(), sc, cd[0], cd[1], cd[2], nthreads, &sb);
            if (rc) continue;  // e.g. a candidate that does not fit in LDS
            double ms = 0.0;
            // timed on a developing flow, not on the uniform start (where every limiter skips its
            // division and every face takes the same flux branch)
            rc = set_freestream(sb, sfs.data());
            if (!rc) rc = batch_march(sb, kTuneDevelop);
            if (!rc) rc = batch_time_steps(sb, 5, &ms);
            delete sb;
            if (rc) return rc;
            const double per_cell = ms / (double)cells;
            if (per_cell < best) {
                best = per_cell;
                tile = cd[0];
                budget = cd[1];
                block = cd[2];
            }
        }
        if (block == 0) return capi_fail(CFD_E_ARG, "cfd_batch_create: no autotune candidate fits");
        tune_s = now_s() - t0;
        tune_src = 1;
        tune_cache_put(cache, key, tile, budget, block, best);
    } else {
        if (block != 64 && block != 128 && block != 256)
            return capi_fail(CFD_E_ARG, "cfd_batch_create: block must be 0 (autotune), 64, 128 or 256");
        tile = block;
        budget = 2 * block;
    }
    cfd_config_t c = *cfg;
    c.block = block;
    cfd_batch_s *b = nullptr;
    rc = build_batch(in, fs4, c, tile, budget, block, nthreads, &b);
    if (rc) return rc;
    b->tune_s = tune_s;
    b->tune_src = tune_src;
    b->build_s = now_s() - t0 - tune_s;
    rc = set_freestream(b, fs4);
    if (rc) {
        delete b;
        return rc;
    }
    *out = b;
    return 0;
}

void cfd_batch_destroy(cfd_batch_t *b) { delete b; }

int cfd_batch_info(const cfd_batch_t *b, int *out8, double *secs2) {
    if (!b) return capi_fail(CFD_E_ARG, "cfd_batch_info: null batch");
    if (out8) {
        const int v[8] = {b->ninst, b->nc, b->ntiles, b->nfe, b->tile, b->face_budget, b->block, b->max_tile_faces};
        std::memcpy(out8, v, sizeof(v));
    }
    if (secs2) {
        secs2[0] = b->build_s;
        secs2[1] = b->tune_s;
    }
    return 0;
}

int cfd_batch_tuning(const cfd_batch_t *b, int *source) {
    if (!b || !source) return capi_fail(CFD_E_ARG, "cfd_batch_tuning: null argument");
    *source = b->tune_src;
    return 0;
}

int cfd_batch_set_state(cfd_batch_t *b, const double *U) {
    if (!b || !U) return capi_fail(CFD_E_ARG, "cfd_batch_set_state: null argument");
    std::vector<double4> h(b->nc);
    for (int c = 0; c < b->nc; c++)
        h[b->iperm[c]] = make_double4(U[4 * (size_t)c], U[4 * (size_t)c + 1], U[4 * (size_t)c + 2], U[4 * (size_t)c + 3]);
    BHIP(h2d(b->Un, h.data(), h.size()));
    return 0;
}

int cfd_batch_get_state(cfd_batch_t *b, double *U) {
    if (!b || !U) return capi_fail(CFD_E_ARG, "cfd_batch_get_state: null argument");
    BHIP(b->rows.get(b->iperm, 4, reinterpret_cast<const double *>(b->Un), U, b->stream));
    return 0;
}

int cfd_batch_solve(cfd_batch_t *b, double tol, int max_steps, int check_every, int *steps,
                    double *err4, int *status, double *conv_s, double *wall_s, void *stream) {
    if (!b || max_steps < 0 || check_every <= 0) return capi_fail(CFD_E_ARG, "cfd_batch_solve: bad arguments");
    BHIP(hipStreamSynchronize((hipStream_t)stream));
    int rc = batch_reset(b);
    if (rc) return rc;
    rc = batch_graph(b, tol);
    if (rc) return rc;
    const int ni = b->ninst;
    std::vector<int> st(ni, 1);
    std::vector<double> conv(ni, -1.0);
    BHIP(hipStreamSynchronize(b->stream));
    const double t0 = now_s();
    int done = 0;
    bool all = false;
    std::vector<double> e4(4 * (size_t)ni);
    b->hist.clear();
    b->hist_checks = 0;
    while (done < max_steps && !all) {
        const int k = std::min(check_every, max_steps - done);
        if ((rc = batch_launch(b, k))) return rc;
        done += k;
        BHIP(hipMemcpyAsync(st.data(), b->d_status, ni * sizeof(int), hipMemcpyDeviceToHost, b->stream));
        BHIP(hipMemcpyAsync(e4.data(), b->d_err4, e4.size() * sizeof(double), hipMemcpyDeviceToHost, b->stream));
        BHIP(hipStreamSynchronize(b->stream));
        for (int i = 0; i < ni; i++) b->hist.push_back(e4[4 * (size_t)i]);
        b->hist_checks++;
        const double t = now_s() - t0;
        all = true;
        int marching = 0;
        for (int i = 0; i < ni; i++) {
            if (st[i] != 1 && conv[i] < 0.0) conv[i] = t;
            if (st[i] == 1) {
                all = false;
                marching++;
            }
        }
        if (b->progress && b->progress_every > 0 && b->hist_checks % b->progress_every == 0)
            b->progress(done, marching, b->progress_user);
        if (!all && !b->dcfg.persist) {
            // once the marching instances hold half the tiles the launch grids cover or fewer,
            // capture the step again with grids sized to them
            int active = 0;
            for (int i = 0; i < ni; i++)
                if (st[i] == 1) active += b->inst_tile[i + 1] - b->inst_tile[i];
            if (2 * active <= b->graph_tiles && (rc = batch_graph(b, tol, active))) return rc;
        }
    }
    const double wall = now_s() - t0;
    if (steps) BHIP(hipMemcpy(steps, b->d_steps, ni * sizeof(int), hipMemcpyDeviceToHost));
    if (err4) BHIP(hipMemcpy(err4, b->d_err4, 4 * (size_t)ni * sizeof(double), hipMemcpyDeviceToHost));
    if (status) std::memcpy(status, st.data(), ni * sizeof(int));
    if (conv_s) std::memcpy(conv_s, conv.data(), ni * sizeof(double));
    if (wall_s) *wall_s = wall;
    for (int i = 0; i < ni; i++)
        if (st[i] != 0) return CFD_E_NOTCONV;
    return 0;
}

int cfd_batch_set_freeze(cfd_batch_t *b, const int *mode) {
    if (!b) return capi_fail(CFD_E_ARG, "cfd_batch_set_freeze: null batch");
    if (!b->d_fz) return capi_fail(CFD_E_ARG, "cfd_batch_set_freeze: limiter freezing is off (freeze_tol, freeze_stall)");
    if (!mode) {
        b->fz_start.clear();
        return 0;
    }
    for (int i = 0; i < b->ninst; i++)
        if (mode[i] != 0 && mode[i] != 1) return capi_fail(CFD_E_ARG, "cfd_batch_set_freeze: mode must be 0 or 1");
    b->fz_start.assign(mode, mode + b->ninst);
    return 0;
}

int cfd_batch_set_progress(cfd_batch_t *b, cfd_progress_fn fn, void *user, int every_checks) {
    if (!b || every_checks < 0) return capi_fail(CFD_E_ARG, "cfd_batch_set_progress: bad arguments");
    b->progress = fn;
    b->progress_user = user;
    b->progress_every = every_checks;
    return 0;
}

int cfd_batch_set_cfl(cfd_batch_t *b, double cfl) {
    if (!b || !(cfl > 0.0) || !std::isfinite(cfl)) return capi_fail(CFD_E_ARG, "cfd_batch_set_cfl: cfl must be positive");
    b->cfg.cfl = cfl;
    b->dcfg.cfl = cfl;
    b->graph_tol = std::nan("");  // the captured step holds the old value: capture again
    return 0;
}

int cfd_batch_set_launch(cfd_batch_t *b, int mode) {
    if (!b || (mode != 0 && mode != 1)) return capi_fail(CFD_E_ARG, "cfd_batch_set_launch: mode must be 0 or 1");
    if (mode == 1 && (b->cfg.order > 2 || b->cfg.viscous || b->cfg.positivity))
        return capi_fail(CFD_E_ARG, "cfd_batch_set_launch: persistent workgroups need order 1 or 2, inviscid, "
                                    "without the positivity fallback");
    if (b->dcfg.persist != mode) {
        b->dcfg.persist = mode;
        b->graph_tol = std::nan("");  // the captured step holds the old launches: capture again
    }
    return 0;
}

int cfd_batch_history(const cfd_batch_t *b, int *nchecks, double *e0) {
    if (!b || !nchecks) return capi_fail(CFD_E_ARG, "cfd_batch_history: null argument");
    *nchecks = b->hist_checks;
    if (e0) std::memcpy(e0, b->hist.data(), b->hist.size() * sizeof(double));
    return 0;
}

int cfd_batch_time_steps(cfd_batch_t *b, int nsteps, float *ms) {
    if (!b || !ms || nsteps <= 0) return capi_fail(CFD_E_ARG, "cfd_batch_time_steps: bad arguments");
    double m = 0.0;
    int rc = batch_time_steps(b, nsteps, &m);
    *ms = (float)m;
    return rc;
}

}  // extern "C"
