// Host driver of qg_sphere_plan.hpp: prints what the sphere passes' size rules give.
//   chunks <nbands> <ntile> <max_col> <nc> <ncoef> <bands per workgroup> <nz> <capacity>
//       -> chunk, then for every chunk "bands slabs planes doubles"
//   lists <nv> <trips> <slots> <room>
//       -> "vals slot_vals words slot_words bytes fit", all but the last in bytes
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include "../../qumasun_amd/csrc/qg_sphere_plan.hpp"

int main(int argc, char** argv) {
    if (argc == 10 && !std::strcmp(argv[1], "chunks")) {
        const int nbands = std::atoi(argv[2]), ntile = std::atoi(argv[3]), max_col = std::atoi(argv[4]);
        const int nc = std::atoi(argv[5]), ncoef = std::atoi(argv[6]), nb = std::atoi(argv[7]), nz = std::atoi(argv[8]);
        const size_t cap = std::strtoull(argv[9], nullptr, 10), slab1 = (size_t)ntile * max_col * nc;
        const int chunk = qg::sphere_chunk_bands(nbands, slab1, ncoef, cap);
        std::printf("%d\n", chunk);
        for (int b0 = 0; chunk > 0 && b0 < nbands; b0 += chunk) {
            const int n = nbands - b0 < chunk ? nbands - b0 : chunk;
            const size_t room = cap - (size_t)n * ncoef;
            const qg::SphereSlabs s =
                qg::sphere_project_slabs(nz, (int64_t)ntile * ((n + nb - 1) / nb), slab1 * n, room);
            std::printf("%d %d %d %zu\n", n, s.nslab, s.tz, slab1 * n * s.nslab + (size_t)n * ncoef);
        }
        return 0;
    }
    if (argc == 6 && !std::strcmp(argv[1], "lists")) {
        const int nv = std::atoi(argv[2]);
        const size_t trips = std::strtoull(argv[3], nullptr, 10), slots = std::strtoull(argv[4], nullptr, 10);
        const qg::SphereListLayout l = qg::sphere_list_layout(nv, trips, slots);
        std::printf("%zu %zu %zu %zu %zu %d\n", l.vals, l.slot_vals, l.words, l.slot_words, l.bytes,
                    qg::sphere_lists_that_fit(nv, trips, slots, std::strtoull(argv[5], nullptr, 10)));
        return 0;
    }
    return 2;
}
