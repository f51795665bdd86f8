// Prints, for a mesh file (npts, ncells, points [3*npts], cells [4*ncells]) and tiles of so many cells
// in its own or in Hilbert order, whether the one-launch second-order pass is taken with workgroups of
// so many threads:  form_checks <mesh.bin> [<tile> <renumber> <block> ...]
#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../../cfd_solver_withcuda_amd/csrc/mesh_host.h"

using namespace cfd;

int main(int argc, char **argv) {
    std::FILE *f = argc > 1 ? std::fopen(argv[1], "rb") : nullptr;
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
    for (int a = 2; a + 2 < argc; a += 3) {
        const int block = std::atoi(argv[a + 2]);
        Layout L;
        build_layout(m, std::atoi(argv[a]), std::atoi(argv[a + 1]), L, 0);
        TileRings r;
        tile_rings(m, L, r);
        long first = 0;
        for (int t = 0; t < L.ntiles; t++) first += r.tiles[4 * t + 1] & 0xFFFF;
        if (first != r.first_ring) return 1;
        // the launch's LDS: primitives of the local cells, then gradients or the fluxes of a thread's first
        // two faces, then the other faces' fluxes
        const int held = std::min(L.max_tile_faces, 2 * block);
        const size_t lds = 8 * (size_t)(4 * r.max_local + std::max(8 * r.max_grad, 4 * held) + 4 * (L.max_tile_faces - held));
        std::printf("%d\n", (int)one_launch_pays(m.nc, L.ntiles, r.first_ring, lds, block));
    }
    return 0;
}
