// One-launch second-order pass: a workgroup forms the gradients of its tile's cells and of the ring
// of cells around it itself, so that a residual evaluation needs no gradient pass and no gradient
// array. Shared by the translation units that instantiate it (fv_fused.hip: inviscid;
// fv_fused_visc.hip: with viscous terms; fv_fused_pos.hip: the positivity fallback's two passes;
// fv_fused_freeze.hip: limiter freezing).
//
// Why: the two-pass form (grad_tile_kernel + flux_tile_kernel) moves 128 B per cell of gradients
// through HBM, reads the state of every tile and its ring twice and pays two launches. Here the
// ring's gradients are formed again by every tile that needs them (0.37 of a cell per cell in tiles
// of 128 Hilbert-ordered cells, each at about a sixth of a face flux's arithmetic), which costs less
// than the traffic. Measured on MI355X, whole steps, two-pass to one launch: 7.97M-cell forward
// step, RK4 with the positivity fallback 3.83 to 2.80 ms; 1.27M-cell bump, RK3 0.423 to 0.332 ms;
// 320k-cell viscous bump 161 to 118 us; 2.5k cells 50 to 32 us (and with stage_update's states kept
// in registers to 2.61 ms, 0.307 ms, 113 us and 31 us).
//
// What bounds it (forward step, 0.65 ms a stage): FP64 issue, about 2,000 vector instructions a wave or
// 70-75 % of the launch; the L2 fills run at 4.4-4.9 TB/s, the rate (4.7) of a copy of arrays beyond the last-level cache.
// Neither leaves room for less occupancy: 128 registers and 20 KB of LDS give 4 waves per SIMD, and
// every variant that spilled (a second prefetched stencil for Green-Gauss, initialised records) lost
// more than it hid.
//
// The recomputing pass forms a marked tile's gradients again, where the two-pass form reads them. With few
// marked tiles that is free; with nearly all of them marked (a 2.6M-cell bump with 30 % noise in every cell,
// RK4 steps in tiles of 128) the two-pass form takes 3.36 ms with HLLC and 3.56 with Roe and Green-Gauss,
// this one 3.50 and 3.91 (3.61 and 4.10 with a flux evaluation for each kind of face).
//
// Local cells of a tile: its own cells, the first ring (whose gradients the tile's faces read), the
// second ring (whose states the first ring's gradients read) and the ghosts of boundary faces
// (mesh_host.h, TileRings). Phases:
//   A  primitives of all local cells into LDS (one 32-byte load per cell);
//   G  gradients of own and first-ring cells into LDS, each in its own face order;
//   F  one flux per face, every operand from LDS; a thread keeps its (at most two) fluxes in
//      registers until all gradients have been read, and they then take the gradients' LDS;
//   C  gather per cell, time step and stage update, as flux_tile_kernel's.
// Every value is formed by the same operations in the same order as in the two-pass form, so both
// give the same bits.
#pragma once
#include "fv_flux.h"

namespace cfd {

struct FusedArgs {
    DevMesh m;
    DevCfg cfg;
    const double4 *Us;
    double *grad;  // residual mode: the tile's gradients are written here when set
    StageArgs st;
    int gg;        // Green-Gauss gradients (weighted least squares otherwise)
    int block;     // threads of the error sums' tree (its order does not follow the launch's threads)
};

// LDS of one launch, in doubles: primitives of the local cells, then the gradients, whose space the
// fluxes of a thread's first two faces take over, then the fluxes of further faces (tiles with
// more faces than two per thread); at least the block reductions' 4 per thread of the tree.
__host__ __device__ __forceinline__ int fused_held(int FT, int threads) { return FT < 2 * threads ? FT : 2 * threads; }
__host__ __device__ __forceinline__ int fused_space(int max_grad, int FT, int threads) {
    const int g = 8 * max_grad, f = 4 * fused_held(FT, threads);
    return g > f ? g : f;
}
__host__ __device__ __forceinline__ size_t fused_doubles(int max_local, int max_grad, int FT, int threads, int block) {
    const size_t d = 4 * (size_t)max_local + fused_space(max_grad, FT, threads) + 4 * (size_t)(FT - fused_held(FT, threads));
    return d < 4 * (size_t)block ? 4 * (size_t)block : d;
}

namespace {

// The launch's arguments, read again from the kernel-argument segment. Each phase takes its own
// copy: values that phases share through one copy would stay in scalar registers from the first
// phase to the last, and there are not enough of them (the two-pass kernels spill 140).
__device__ __forceinline__ const FusedArgs &fused_args() {
    const __attribute__((address_space(4))) void *p =
        (const __attribute__((address_space(4))) void *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const FusedArgs *)p;
}

// Primitives (rho, u, v, p) of a conserved state, with state_from_U's arithmetic.
__device__ __forceinline__ void prim4(const double4 &u, double2 &a, double2 &b) {
    const double Rho = u.x;
    const double inv = 1.0 / Rho;
    double v1 = u.y * inv;
    double v2 = u.z * inv;
    if (fabs(v1) <= 1e-10) v1 = 0.0;
    if (fabs(v2) <= 1e-10) v2 = 0.0;
    const double vmag = (v1 * v1 + v2 * v2);
    a = make_double2(Rho, v1);
    b = make_double2(v2, kGm1 * (u.w - 0.5 * Rho * vmag));
}

// Ghost of state `in` across a boundary face of kind `kind` of a tile.
__device__ __forceinline__ void ghost_of_tile(const FusedArgs &A, int tile, int kind, const FState &in, double nx,
                                              double ny, FState &g) {
    double fsv[5];
    tile_fs(A.m, A.cfg, tile, fsv);
    ghost_state(A.cfg.bc[kind], in, nx, ny, fsv, g);
}

// What a weighted least-squares gradient of one local cell reads: its local neighbours and the
// vector of each face.
struct Stencil {
    ushort4 nb;
    double2 w[4];
};

__device__ __forceinline__ int local_cell(const DevMesh &m, int l, int c0, int nct, int r0) {
    return l < nct ? c0 + l : m.ring_cell[r0 + l - nct];
}

__device__ __forceinline__ void load_stencil(const DevMesh &m, int i, int c, int nct, int r0, Stencil &s) {
    s.nb = i < nct ? m.own_nbr[c] : m.ring_nbr[r0 + i - nct];
    const double2 *__restrict__ p = m.cw + 4 * (size_t)c;
    for (int q = 0; q < 4; q++) s.w[q] = p[q];
}

// Geometry of a face entry, and its local cells.
struct LocalFace {
    ushort2 c;
    double nx, ny, dl, dx, dy;
};

__device__ __forceinline__ void load_local_face(const DevMesh &m, int e, LocalFace &f) {
    f.c = m.floc[e];
    f.nx = m.fnx[e];
    f.ny = m.fny[e];
    f.dl = m.fdl[e];
    const double2 d = m.fd[e];
    f.dx = d.x;
    f.dy = d.y;
}

// The tile's ranges, as the phases hand them on.
struct TileRange {
    int tile, c0, nct, r0, nr, g0;
};

template <int FLUX, int LIM, bool VISC, int POS>
__device__ __forceinline__ void fused_face(const FusedArgs &A, const double2 *sWa, const double2 *sWb,
                                           const double2 *sG, int NG, const TileRange &t, const LocalFace &f,
                                           int fz, int e, double *F) {
    const double nx = f.nx, ny = f.ny, dl = f.dl;
    const ushort2 lc = f.c;
    const bool boundary = lc.y >= t.nct + t.nr;
    int kind = 0;
    if (boundary) kind = A.m.ghost[t.g0 + lc.y - t.nct - t.nr].y;
    FState SL, SR, fL, fR;
    double gL[8], gR[8];
    bool first = false;
    if constexpr (POS == 2) {
        // positivity fallback, recomputation: a face of a flagged cell takes the two cells'
        // first-order states (conserved values as stored, ghost of the left state). Both kinds of face
        // share the flux below, which a wave of both would otherwise go through twice
        const uint8_t *pflag = A.st.pflag;
        const int L = local_cell(A.m, lc.x, t.c0, t.nct, t.r0);
        const int R = boundary ? L : local_cell(A.m, lc.y, t.c0, t.nct, t.r0);
        first = pflag[L] || pflag[R];
        if (first) {
            load_state(A.Us, L, fL);
            if (boundary) ghost_of_tile(A, t.tile, kind, fL, nx, ny, fR);
            else load_state(A.Us, R, fR);
        }
    }
    auto prims = [&](int l, FState &s) {
        const double2 a = sWa[l], b = sWb[l];
        s.W[0] = a.x;
        s.W[1] = a.y;
        s.W[2] = b.x;
        s.W[3] = b.y;
    };
    auto gradient = [&](int l, double *g) {
        for (int q = 0; q < 4; q++) {
            const double2 v = sG[q * NG + l];
            g[2 * q] = v.x;
            g[2 * q + 1] = v.y;
        }
    };
    if (!first) {
        prims(lc.x, SL);
        prims(lc.y, SR);
        // frozen limiter factors of this face entry (8 floats, two 16-byte loads)
        float pv[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        float4 *p4 = fz ? reinterpret_cast<float4 *>(A.st.psi) + 2 * (size_t)e : nullptr;
        if (fz == 2) {
            const float4 a = p4[0], b = p4[1];
            pv[0] = a.x; pv[1] = a.y; pv[2] = a.z; pv[3] = a.w;
            pv[4] = b.x; pv[5] = b.y; pv[6] = b.z; pv[7] = b.w;
        }
        gradient(lc.x, gL);
        reconstruct_side<LIM, false>(SL, SR, gL, f.dx, f.dy, 1.0, fz, pv, fL);
        if (boundary) {
            ghost_of_tile(A, t.tile, kind, fL, nx, ny, fR);
            if constexpr (VISC)
                for (int q = 0; q < 8; q++) gR[q] = gL[q];
        } else {
            gradient(lc.y, gR);
            reconstruct_side<LIM, false>(SR, SL, gR, f.dx, f.dy, -1.0, fz, pv + 4, fR);
        }
        if (fz == 1) {
            p4[0] = make_float4(pv[0], pv[1], pv[2], pv[3]);
            p4[1] = make_float4(pv[4], pv[5], pv[6], pv[7]);
        }
    }
    face_flux<FLUX>(boundary, A.cfg.roe_bdiss, fL, fR, nx, ny, dl, F);
    if constexpr (VISC) {
        double Fv[4];
        viscous_flux(A.cfg, SL.W, SR.W, gL, gR, nx, ny, dl, f.dx, f.dy, Fv);
        for (int q = 0; q < 4; q++) F[q] = F[q] - Fv[q];
    }
}

}  // namespace

// FZ, POS: as flux_tile_kernel (POS 1 detects, 2 recomputes the marked tiles with persistent
// workgroups, each finding those of its share by their marks: no list, no launch to make one).
template <int FLUX, int LIM, int MODE, bool VISC, int POS = 0, bool FZ = false>
__global__ void __launch_bounds__(VISC || POS == 2 ? 512 : 1024) fused_tile_kernel(FusedArgs) {
    extern __shared__ double2 smem2[];
    constexpr bool REDO = (POS == 2);
    // a face's record travels during the previous face's arithmetic, where registers allow it
    // (the viscous variants drop to 2 waves per SIMD with it, and Roe's spill)
    constexpr bool PREFETCH = !VISC && FLUX != FLUX_ROE;
    int tile, next = blockIdx.x;
    if constexpr (REDO) {
        // the two-pass form's counts of listed tiles start from zero wherever it takes over
        const FusedArgs &A = fused_args();
        if (blockIdx.x == 0 && threadIdx.x < 4) A.st.dirty[2 * A.m.ntiles + threadIdx.x] = 0;
    }
    do {
    if constexpr (REDO) {
        // the next marked tile of this workgroup's share (every gridDim.x-th tile): 64 marks a look
        const FusedArgs &A = fused_args();
        for (tile = -1; tile < 0 && next < A.m.ntiles;) {
            const int t = next + (threadIdx.x & 63) * gridDim.x;
            const unsigned long long hit = __ballot(t < A.m.ntiles && A.st.dirty[t] != 0);
            if (hit) tile = next + (__ffsll(hit) - 1) * gridDim.x;
            next = hit ? tile + gridDim.x : next + 64 * gridDim.x;
        }
        if (tile < 0) return;
        __syncthreads();  // every wave has looked, and read the previous tile's LDS
    }
    int c0, nct, fs, nft, r0, n1, nr, g0, NL, NG, FT;
    int fz = 0;
    bool geom;
    const int k = threadIdx.x, B = blockDim.x;
    LocalFace f;        // loaded where they are used
    Stencil st0, st1;
    double2 *sWa = smem2, *sWb, *sG;
    // ---- A: primitives of the local cells -------------------------------------------------
    {
        const FusedArgs &A = fused_args();
        const DevMesh &m = A.m;
        if constexpr (!REDO) {
            tile = virtual_tile(m, blockIdx.x, tiles_to_run(m), A.cfg.xcd_remap);
            if (tile < 0) return;
        }
        c0 = m.tile_cstart[tile];
        nct = m.tile_cstart[tile + 1] - c0;
        fs = m.tile_fstart[tile];
        nft = m.tile_fstart[tile + 1] - fs;
        const int4 rg = m.rings[tile];
        r0 = rg.x;
        n1 = rg.y & 0xFFFF;
        nr = rg.z;
        const int ng = rg.y >> 16;
        g0 = rg.w;
        NL = m.max_local;
        NG = m.max_grad;
        FT = m.max_tile_faces;
        sWb = sWa + NL;
        sG = sWb + NL;
        geom = (MODE == MODE_RESID) || (A.st.lts && A.st.stage == 0) || (A.st.last && A.st.dt_partial);
        if (FZ && A.st.freeze) fz = A.st.freeze[m.tile_inst ? m.tile_inst[tile] : 0];
        const double4 *__restrict__ Us = A.Us;
        const int *__restrict__ ring = m.ring_cell + r0;
        // ghosts first (tiles at the boundary only): their code would spill what is held below
        for (int i = k; i < ng; i += B) {
            const int2 gh = m.ghost[g0 + i];
            const double2 n = m.ghost_n[g0 + i];
            FState in, g;
            load_state(Us, gh.x, in);
            ghost_of_tile(A, tile, gh.y, in, n.x, n.y, g);
            sWa[nct + nr + i] = make_double2(g.W[0], g.W[1]);
            sWb[nct + nr + i] = make_double2(g.W[2], g.W[3]);
        }
        // this thread's first face record travels while the states are staged
        if (k < nft) load_local_face(m, fs + k, f);
        auto stage = [&](int l, int c) {
            double2 a, b;
            prim4(Us[c], a, b);
            sWa[l] = a;
            sWb[l] = b;
        };
        if (k < nct) stage(k, c0 + k);
        // and so do the stencils of its first two gradients
        if (!A.gg) {
            if (k < nct + n1) load_stencil(m, k, local_cell(m, k, c0, nct, r0), nct, r0, st0);
            if (k + B < nct + n1) load_stencil(m, k + B, local_cell(m, k + B, c0, nct, r0), nct, r0, st1);
        }
        for (int i = k; i < nr; i += B) stage(nct + i, ring[i]);
    }
    __syncthreads();
    // ---- G: gradients of own and first-ring cells ------------------------------------------
    {
        const FusedArgs &A = fused_args();
        const DevMesh &m = A.m;
        auto put_gradient = [&](int i, const double *g) {
            for (int q = 0; q < 4; q++) sG[q * NG + i] = make_double2(g[2 * q], g[2 * q + 1]);
            if constexpr (MODE == MODE_RESID) {
                if (A.grad && i < nct) {
                    double2 *out = reinterpret_cast<double2 *>(A.grad + 8 * (size_t)(c0 + i));
                    for (int q = 0; q < 4; q++) out[q] = make_double2(g[2 * q], g[2 * q + 1]);
                }
            }
        };
        if (A.gg) {
            // the face values times the outward normal and length; a boundary face takes the cell's
            // own value
#pragma unroll 1
            for (int i = k; i < nct + n1; i += B) {
                const int c = local_cell(m, i, c0, nct, r0);
                const ushort4 nb = i < nct ? m.own_nbr[c] : m.ring_nbr[r0 + i - nct];
                const uint16_t nbs[4] = {nb.x, nb.y, nb.z, nb.w};
                const double2 *__restrict__ p = reinterpret_cast<const double2 *>(m.cn) + 6 * (size_t)c;
                double cn[12];
                for (int q = 0; q < 6; q++) {
                    const double2 v = p[q];
                    cn[2 * q] = v.x;
                    cn[2 * q + 1] = v.y;
                }
                const double ia = m.inv_area[c];
                const double2 a = sWa[i], b = sWb[i];
                double g[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
                for (int s = 0; s < 4; s++) {
                    if (nbs[s] == 0xFFFF) break;
                    const int j = nbs[s] >= nct + nr ? i : nbs[s];
                    const double nx = cn[3 * s], ny = cn[3 * s + 1], dl = cn[3 * s + 2];
                    const double2 u = sWa[j], w = sWb[j];
                    const double phi[4] = {0.5 * (a.x + u.x), 0.5 * (a.y + u.y), 0.5 * (b.x + w.x), 0.5 * (b.y + w.y)};
                    for (int q = 0; q < 4; q++) {
                        g[2 * q] += phi[q] * nx * dl;
                        g[2 * q + 1] += phi[q] * ny * dl;
                    }
                }
                for (int q = 0; q < 8; q++) g[q] = g[q] * ia;
                put_gradient(i, g);
            }
        } else {
            auto wlsq = [&](int i, const Stencil &st) {
                const uint16_t nbs[4] = {st.nb.x, st.nb.y, st.nb.z, st.nb.w};
                const double2 a = sWa[i], b = sWb[i];
                double g[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
                for (int s = 0; s < 4; s++) {
                    if (nbs[s] == 0xFFFF) break;
                    const int j = nbs[s];
                    const double2 u = sWa[j], w = sWb[j];
                    const double d[4] = {u.x - a.x, u.y - a.y, w.x - b.x, w.y - b.y};
                    for (int q = 0; q < 4; q++) {
                        g[2 * q] += st.w[s].x * d[q];
                        g[2 * q + 1] += st.w[s].y * d[q];
                    }
                }
                put_gradient(i, g);
            };
            if (k < nct + n1) wlsq(k, st0);
            if (k + B < nct + n1) wlsq(k + B, st1);
#pragma unroll 1
            for (int i = k + 2 * B; i < nct + n1; i += B) {
                load_stencil(m, i, local_cell(m, i, c0, nct, r0), nct, r0, st0);
                wlsq(i, st0);
            }
        }
    }
    __syncthreads();
    // ---- F: one flux per face ---------------------------------------------------------------
    const int held = fused_held(FT, B), more_faces = FT - held;
    double2 *sX = sG + fused_space(NG, FT, B) / 2;  // fluxes of faces beyond the held ones
    // the two halves of face j's flux
    auto flux_at = [&](int j, double2 *&lo, double2 *&hi) {
        lo = sG + j;
        hi = lo + held;
        if (more_faces && j >= held) {
            lo = sX + (j - held);
            hi = lo + more_faces;
        }
    };
    auto put_flux = [&](int j, const double *F) {
        double2 *lo, *hi;
        flux_at(j, lo, hi);
        *lo = make_double2(F[0], F[1]);
        *hi = make_double2(F[2], F[3]);
    };
    ushort4 sl4;
    double4 un4, us4;
    double ar, ia, hprev;
    double gnx[4], gny[4], gdl[4];  // normal and length of the cell's faces (time steps)
    auto load_cell = [&]() {
        const FusedArgs &A = fused_args();
        const int c = c0 + k;
        sl4 = reinterpret_cast<const ushort4 *>(A.m.slots)[c];
        if (geom) {
            ar = A.m.area[c];
            const uint16_t sls[4] = {sl4.x, sl4.y, sl4.z, sl4.w};
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const int e = fs + (sls[s] == 0xFFFF ? 0 : sls[s] >> 1);
                gnx[s] = A.m.fnx[e];
                gny[s] = A.m.fny[e];
                gdl[s] = A.m.fdl[e];
            }
        }
        if constexpr (MODE == MODE_STAGE) {
            un4 = A.st.Un[c];
            ia = A.m.inv_area[c];
            // the stage input (TVD-RK3) or the sum of net fluxes (RK4) of the later stages
            if (A.st.stage > 0) us4 = (A.st.rk == 4) ? A.st.acc_in[c] : A.Us[c];
            if (A.st.lts && A.st.stage > 0) hprev = A.st.hbuf[c];
        }
    };
    {
        const FusedArgs &A = fused_args();
        double Fa[4], Fb[4];
#pragma unroll 1
        for (int j = k; j < nft; j += B) {
            LocalFace fn;
            const bool more = j + B < nft;
            if (PREFETCH && more) load_local_face(A.m, fs + j + B, fn);
            double F[4];
            fused_face<FLUX, LIM, VISC, POS>(A, sWa, sWb, sG, NG, TileRange{tile, c0, nct, r0, nr, g0}, f, fz, fs + j, F);
            if (j < B) {
                for (int q = 0; q < 4; q++) Fa[q] = F[q];
            } else if (j < 2 * B) {
                for (int q = 0; q < 4; q++) Fb[q] = F[q];
            } else {
                put_flux(j, F);
            }
            if (PREFETCH) f = fn;
            else if (more) load_local_face(A.m, fs + j + B, f);
        }
        // the cell's own inputs of phase C travel during the barriers
        if (k < nct) load_cell();
        __syncthreads();
        if (k < nft) put_flux(k, Fa);
        if (k + B < nft) put_flux(k + B, Fb);
        __syncthreads();
    }
    // ---- C: gather per cell, time step, stage update ---------------------------------------
    double errp[4] = {0.0, 0.0, 0.0, 0.0};
    double dtmin = 1.7976931348623157e308;
    const FusedArgs &A = fused_args();
    const DevMesh &m = A.m;
    const StageArgs &st = A.st;
    if (k < nct) {
        const int c = c0 + k;
        double r[4] = {0.0, 0.0, 0.0, 0.0};
        const uint16_t sls[4] = {sl4.x, sl4.y, sl4.z, sl4.w};
        for (int s = 0; s < 4; s++) {
            const uint16_t sl = sls[s];
            if (sl == 0xFFFF) break;
            const int j = sl >> 1;
            const bool isR = sl & 1;
            double2 *lo, *hi;
            flux_at(j, lo, hi);
            const double2 a = *lo, b = *hi;
            r[0] += isR ? -a.x : a.x;
            r[1] += isR ? -a.y : a.y;
            r[2] += isR ? -b.x : b.x;
            r[3] += isR ? -b.y : b.y;
        }
        // local time step of the cell state (rho, u, v, p) with sound speed a
        auto time_step = [&](double rho, double u, double w, double p, double a) {
            double den = 0.0, sdl2 = 0.0;
#pragma unroll
            for (int s = 0; s < 4; s++) {
                if (sls[s] == 0xFFFF) break;
                den += (fabs(u * gnx[s] + w * gny[s]) + a) * gdl[s];
                if constexpr (VISC) sdl2 += gdl[s] * gdl[s];
            }
            if constexpr (VISC) den += viscous_dt_term(A.cfg, rho, p, sdl2, ar);
            return (den <= 0.0 || !isfinite(den)) ? 0.0 : A.cfg.cfl * ar / den;
        };
        double dtc = 0.0;
        if (MODE == MODE_RESID || (st.lts && st.stage == 0)) {
            const double2 a = sWa[k], b = sWb[k];
            dtc = time_step(a.x, a.y, b.x, b.y, sound_speed(a.x, b.y));
        }
        if constexpr (MODE == MODE_RESID) {
            reinterpret_cast<double4 *>(st.R_out)[c] = make_double4(r[0], r[1], r[2], r[3]);
            if (st.dt_out) st.dt_out[c] = dtc;
            dtmin = fmin(dtmin, dtc);
        } else {
            double h;
            if (st.lts) {
                h = (st.stage == 0) ? dtc * ia : hprev;
                if (st.stage == 0) st.hbuf[c] = h;
            } else {
                h = (*st.dt_global) * ia;
            }
            const double Un[4] = {un4.x, un4.y, un4.z, un4.w};
            const double us[4] = {us4.x, us4.y, us4.z, us4.w};
            const double4 o4 = stage_update(st, c, h, Un, us, us4, r);
            const double Uo[4] = {o4.x, o4.y, o4.z, o4.w};
            if constexpr (POS == 1) {
                // positivity fallback, detection (the same test as flux_tile_kernel's): the range of
                // the cell's and its face neighbours' stage inputs, rounded to FP32
                const ushort4 nb4 = m.own_nbr[c];
                const uint16_t nbs[4] = {nb4.x, nb4.y, nb4.z, nb4.w};
                double rlo = (double)(float)sWa[k].x, rhi = rlo, plo = (double)(float)sWb[k].y, phi = plo;
                for (int s = 0; s < 4; s++) {
                    if (nbs[s] >= nct + nr) continue;  // unused slot, or a ghost
                    const double rj = (double)(float)sWa[nbs[s]].x;
                    const double pj = (double)(float)sWb[nbs[s]].y;
                    rlo = fmin(rlo, rj);
                    rhi = fmax(rhi, rj);
                    plo = fmin(plo, pj);
                    phi = fmax(phi, pj);
                }
                const bool bad = inadmissible(Uo, rlo, rhi, plo, phi, st.pos_range & 1);
                st.pflag[c] = bad ? 1 : 0;
                if (bad) mark_dirty(m, st, tile, c0, nct, fs, sls);
            }
            st.Uout[c] = o4;
            if (st.last) {
                if (st.err_partial) {
                    for (int q = 0; q < 4; q++) errp[q] += err_term(Uo[q] - Un[q], Un[q]);
                }
                if (st.dt_partial) {
                    // time step of the new state, for the next step's global dt
                    FState s;
                    state_from_U(Uo[0], Uo[1], Uo[2], Uo[3], s);
                    dtmin = fmin(dtmin, time_step(s.W[0], s.W[1], s.W[2], s.W[3], s.W[4]));
                }
            }
        }
    }
    // block reductions reuse LDS from its base (the allocation holds >= 4 * blockDim doubles)
    double *red = reinterpret_cast<double *>(smem2);
    if constexpr (MODE == MODE_STAGE) {
        if (st.last && st.err_partial) {
            __syncthreads();
            double out[4];
            block_sum4(red, errp, out, A.block);
            if (k == 0)
                for (int q = 0; q < 4; q++) st.err_partial[4 * tile + q] = out[q];
        }
    }
    if ((MODE == MODE_RESID || st.last) && st.dt_partial) {
        __syncthreads();
        const double b = block_min(red, dtmin, A.block);
        if (k == 0) st.dt_partial[tile] = b;
    }
    if constexpr (POS == 2) {
        if (k == 0) st.dirty[tile] = 0;
    }
    } while (REDO);
}

template <int FLUX, int LIM, int MODE, bool VISC, int POS, bool FZ>
static hipError_t launch_fused_t(const FusedArgs &a, int threads, size_t sm, hipStream_t s) {
    auto kern = fused_tile_kernel<FLUX, LIM, MODE, VISC, POS, FZ>;
    const int grid = (POS == 2) ? grid_persist(kern, a.m, a.cfg, threads, sm) : grid_of(a.m, a.cfg);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(threads), sm, s, a);
    return hipGetLastError();
}

// Every flux and limiter of one variant.
template <int MODE, bool VISC, int POS, bool FZ>
static hipError_t launch_fused_family(const FusedArgs &a, int flux, int lim, int threads, size_t sm, hipStream_t s) {
    auto by_lim = [&](auto fluxc) {
        constexpr int F = decltype(fluxc)::value;
        switch (lim) {
        case LIM_NONE: return launch_fused_t<F, LIM_NONE, MODE, VISC, POS, FZ>(a, threads, sm, s);
        case LIM_MINMOD: return launch_fused_t<F, LIM_MINMOD, MODE, VISC, POS, FZ>(a, threads, sm, s);
        case LIM_VANLEER: return launch_fused_t<F, LIM_VANLEER, MODE, VISC, POS, FZ>(a, threads, sm, s);
        case LIM_VANALBADA: return launch_fused_t<F, LIM_VANALBADA, MODE, VISC, POS, FZ>(a, threads, sm, s);
        default: return launch_fused_t<F, LIM_SUPERBEE, MODE, VISC, POS, FZ>(a, threads, sm, s);
        }
    };
    switch (flux) {
    case FLUX_ROE: return by_lim(std::integral_constant<int, FLUX_ROE>{});
    case FLUX_HLLC: return by_lim(std::integral_constant<int, FLUX_HLLC>{});
    case FLUX_LLF: return by_lim(std::integral_constant<int, FLUX_LLF>{});
    default: return by_lim(std::integral_constant<int, FLUX_AUSM>{});
    }
}

// The variants, one translation unit each.
hipError_t launch_fused_plain(const FusedArgs &a, int flux, int lim, int mode, int threads, size_t sm, hipStream_t s);
hipError_t launch_fused_visc(const FusedArgs &a, int flux, int lim, int mode, int threads, size_t sm, hipStream_t s);
hipError_t launch_fused_pos(const FusedArgs &a, int flux, int lim, int pass, int threads, size_t sm, hipStream_t s);
hipError_t launch_fused_freeze(const FusedArgs &a, int flux, int lim, bool visc, int threads, size_t sm, hipStream_t s);

}  // namespace cfd
