// Checks of the tiles' neighbourhoods (TileRings) on meshes read from binary files (npts, ncells,
// points [3*npts], cells [4*ncells]): every local index names the cell, or the ghost, that the
// global connectivity names, and every index is in range.
#include <cstdint>
#include <cstdio>
#include <vector>

#include "../../cfd_solver_withcuda_amd/csrc/mesh_host.h"

using namespace cfd;

static int fails = 0;
#define CHECK(x)                                                          \
    do {                                                                  \
        if (!(x)) {                                                       \
            if (fails++ < 20) std::printf("failed: %s (line %d)\n", #x, __LINE__); \
        }                                                                 \
    } while (0)

static void check_rings(const RefMesh &m, int tile, int renumber, int budget) {
    Layout L;
    build_layout(m, tile, renumber, L, budget);
    TileRings r;
    tile_rings(m, L, r);
    CHECK(r.ok && (int)r.tiles.size() == 4 * L.ntiles && r.face.size() == 2 * L.fL.size());
    CHECK(r.own.size() == 4 * (size_t)m.nc && r.ring.size() == 4 * r.cell.size());
    int most_local = 0, most_grad = 0;
    size_t at = 0, ghosts = 0;
    for (int t = 0; t < L.ntiles; t++) {
        const int k0 = L.tile_cstart[t], nct = L.tile_cstart[t + 1] - k0;
        const int r0 = r.tiles[4 * t], n1 = r.tiles[4 * t + 1] & 0xFFFF, ng = r.tiles[4 * t + 1] >> 16;
        const int nr = r.tiles[4 * t + 2], g0 = r.tiles[4 * t + 3];
        CHECK((size_t)r0 == at && (size_t)g0 == ghosts && n1 <= nr);
        at += nr;
        ghosts += ng;
        most_local = nct + nr + ng > most_local ? nct + nr + ng : most_local;
        most_grad = nct + n1 > most_grad ? nct + n1 : most_grad;
        std::vector<char> seen(m.nc, 0);
        auto global = [&](int l) { return l < nct ? k0 + l : r.cell[r0 + l - nct]; };
        for (int l = 0; l < nct + nr; l++) {
            const int c = global(l);
            CHECK(c >= 0 && c < m.nc && !seen[c]);
            seen[c] = 1;
        }
        // local index `l` names the neighbour of renumbered cell k across its face f
        auto names = [&](int l, int k, int f) {
            const int c = L.perm[k], j = m.nbr[4 * (size_t)c + f];
            if (j < m.nc) return l < nct + nr && global(l) == L.iperm[j];
            const int g = l - nct - nr;
            if (g < 0 || g >= ng) return false;
            const size_t q = 2 * (size_t)(g0 + g);
            return r.ghost[q] == k && r.ghost[q + 1] == m.kind[4 * (size_t)c + f] &&
                   r.ghost_n[q] == m.nrm[8 * (size_t)c + 2 * f] && r.ghost_n[q + 1] == m.nrm[8 * (size_t)c + 2 * f + 1];
        };
        for (int i = 0; i < nct + n1; i++) {
            const int k = global(i);
            const uint16_t *nb = i < nct ? &r.own[4 * (size_t)k] : &r.ring[4 * (size_t)(r0 + i - nct)];
            for (int f = 0; f < 4; f++) {
                if (f >= m.nf[L.perm[k]]) CHECK(nb[f] == 0xFFFF);
                else CHECK(names(nb[f], k, f));
            }
        }
        for (int e = L.tile_fstart[t]; e < L.tile_fstart[t + 1]; e++) {
            const int l = r.face[2 * (size_t)e], q = r.face[2 * (size_t)e + 1];
            CHECK(l < nct + n1 && global(l) == L.fL[e]);
            if (L.fR[e] >= 0) CHECK(q < nct + n1 && global(q) == L.fR[e]);
            else CHECK(q >= nct + nr && q < nct + nr + ng && r.ghost[2 * (size_t)(g0 + q - nct - nr)] == L.fL[e] &&
                       r.ghost[2 * (size_t)(g0 + q - nct - nr) + 1] == -L.fR[e] &&
                       r.ghost_n[2 * (size_t)(g0 + q - nct - nr)] == L.fnx[e]);
        }
    }
    CHECK(at == r.cell.size() && 2 * ghosts == r.ghost.size() && most_local == r.max_local && most_grad == r.max_grad);
    // per-slot vectors and outward normals are the face entries'
    std::vector<double> w, n;
    cell_face_vectors(L, w);
    cell_face_normals(L, n);
    for (int k = 0; k < m.nc; k++) {
        const int c = L.perm[k];
        for (int f = 0; f < m.nf[c]; f++) {
            CHECK(n[12 * (size_t)k + 3 * f + 2] == m.len[4 * (size_t)c + f] || m.nbr[4 * (size_t)c + f] < c);
            const double x = n[12 * (size_t)k + 3 * f], y = n[12 * (size_t)k + 3 * f + 1];
            CHECK(x * m.nrm[8 * (size_t)c + 2 * f] + y * m.nrm[8 * (size_t)c + 2 * f + 1] > 0.999999);
        }
    }
}

int main(int argc, char **argv) {
    for (int a = 1; a < argc; a++) {
        std::FILE *f = std::fopen(argv[a], "rb");
        int32_t h[2];
        if (!f || std::fread(h, sizeof(int32_t), 2, f) != 2) return 2;
        std::vector<double> pts(3 * (size_t)h[0]);
        std::vector<int> cells(4 * (size_t)h[1]);
        if (std::fread(pts.data(), sizeof(double), pts.size(), f) != pts.size() ||
            std::fread(cells.data(), sizeof(int), cells.size(), f) != cells.size())
            return 2;
        std::fclose(f);
        RefMesh m;
        build_ref_mesh(h[0], pts.data(), h[1], cells.data(), m);
        const int shapes[6][3] = {{128, 1, 256}, {64, 1, 128}, {256, 1, 0}, {32, 0, 0}, {16, 1, 0}, {256, 0, 512}};
        for (const auto &s : shapes) check_rings(m, s[0], s[1], s[2]);
        std::printf("%s: %d cells checked\n", argv[a], m.nc);
    }
    return fails ? 1 : 0;
}
