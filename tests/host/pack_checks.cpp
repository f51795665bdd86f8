// Values of the records that are copied to the device (mesh_host.h) on a mesh file (npts, ncells, points
// [3*npts], cells [4*ncells]): face geometry and cell ids with an offset, centre offsets, and per cell
// and face slot the least-squares vector, normal and length.
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <vector>

#include "../../cfd_solver_withcuda_amd/csrc/mesh_host.h"

using namespace cfd;

static int fails = 0;
#define CHECK(x)                                                                        \
    do {                                                                                \
        if (!(x) && fails++ < 20) std::printf("failed: %s (line %d)\n", #x, __LINE__); \
    } while (0)

static void check(const RefMesh &m, int tile, int renumber, int off) {
    Layout L;
    build_layout(m, tile, renumber, L, 0);
    const size_t ne = L.fL.size();
    std::vector<double> geo, fd, w, n;
    std::vector<int> lr;
    pack_face_geometry(L, off, geo, lr);
    face_offsets(L, fd);
    cell_face_vectors(L, w);
    cell_face_normals(L, n);
    CHECK(geo.size() == 6 * ne && lr.size() == 2 * ne && fd.size() == 2 * ne);
    CHECK(w.size() == 8 * (size_t)m.nc && n.size() == 12 * (size_t)m.nc);
    for (size_t e = 0; e < ne; e++) {
        int32_t id[2];
        std::memcpy(id, &geo[6 * e], sizeof(id));
        CHECK(id[0] == L.fL[e] + off && id[1] == (L.fR[e] < 0 ? L.fR[e] : L.fR[e] + off));
        CHECK(lr[2 * e] == id[0] && lr[2 * e + 1] == id[1]);
        CHECK(geo[6 * e + 1] == L.fnx[e] && geo[6 * e + 2] == L.fny[e] && geo[6 * e + 3] == L.fdl[e]);
        CHECK(geo[6 * e + 4] == L.fdx[e] && geo[6 * e + 5] == L.fdy[e]);
        CHECK(fd[2 * e] == L.fdx[e] && fd[2 * e + 1] == L.fdy[e]);
    }
    for (int t = 0; t < L.ntiles; t++)
        for (int k = L.tile_cstart[t]; k < L.tile_cstart[t + 1]; k++)
            for (int s = 0; s < 4; s++) {
                const double *wk = &w[8 * (size_t)k + 2 * s], *nk = &n[12 * (size_t)k + 3 * s];
                const uint16_t sl = L.slots[4 * (size_t)k + s];
                if (sl == 0xFFFF) {
                    CHECK(wk[0] == 0 && wk[1] == 0 && nk[0] == 0 && nk[1] == 0 && nk[2] == 0);
                    continue;
                }
                const size_t e = (size_t)L.tile_fstart[t] + (sl >> 1);
                const double *v = (sl & 1) ? &L.fwR[2 * e] : &L.fwL[2 * e];
                const double sign = (sl & 1) ? -1.0 : 1.0;
                CHECK(wk[0] == v[0] && wk[1] == v[1]);
                CHECK(nk[0] == sign * L.fnx[e] && nk[1] == sign * L.fny[e] && nk[2] == L.fdl[e]);
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
        check(m, 128, 1, 0);
        check(m, 64, 1, 100000);
        check(m, 256, 0, 7);
        std::printf("checked %s\n", argv[a]);
    }
    return fails ? 1 : 0;
}
