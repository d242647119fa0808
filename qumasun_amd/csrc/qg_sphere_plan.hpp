// qg_sphere_plan.hpp — sizes of the sphere passes (qg_sphere.hip) that follow from counts alone: host
// arithmetic without HIP, also compiled by the tests.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace qg {

// planes of one epoch of the projection's lists
constexpr int kProjPlanes = 8;

struct SphereSlabs {
    int tz, nslab;      // planes per slab (whole epochs), slabs
};

// Slabs of a projection of nz planes with wg workgroups per slab: about 4096 workgroups, but no more
// slabs than `most` doubles of partials hold (per_slab doubles each; one slab at least).
inline SphereSlabs sphere_project_slabs(int nz, int64_t wg, size_t per_slab, size_t most) {
    const int nep = (nz + kProjPlanes - 1) / kProjPlanes;
    const int64_t fit = (int64_t)std::min<size_t>(most / std::max<size_t>(1, per_slab), (size_t)nep);
    const int64_t want = std::max<int64_t>(1, std::min({(4096 + wg - 1) / wg, (int64_t)nep, fit}));
    SphereSlabs s;
    s.tz = (int)((nep + want - 1) / want) * kProjPlanes;
    s.nslab = (nz + s.tz - 1) / s.tz;
    return s;
}

// Bands of the equal chunks (the last may be shorter) in which nbands bands go through a scratch of
// `capacity` doubles: a band needs at least per_band doubles of partials (one slab) and its ncoef
// coefficients, and fewer slabs than the chunk would have without the limit are taken where they do not
// fit.  0: not even one band fits.
inline int sphere_chunk_bands(int nbands, size_t per_band, size_t ncoef, size_t capacity) {
    const size_t most = capacity / std::max<size_t>(1, per_band + ncoef);
    if (most == 0) return 0;
    const int64_t chunks = ((int64_t)nbands + (int64_t)std::min<size_t>(most, (size_t)INT32_MAX) - 1) /
                           (int64_t)std::min<size_t>(most, (size_t)INT32_MAX);
    return (int)((nbands + chunks - 1) / std::max<int64_t>(1, chunks));
}

// Byte offsets of the entry lists of one tile height and type in their one allocation: values and words
// of the apply's trips and of the projection's slots (nv radial vectors each).
//
// The kernels issue the loads of their first kSphereAhead entries of a plane or epoch without a look at
// their number, through buffer resources that end at the last one.  Whether the offset of such a load
// counts in the range check is the hardware's affair: the slack keeps what the loads can address inside
// the allocation either way.
constexpr int kSphereAhead = 4;

struct SphereListLayout {
    size_t vals, slot_vals, words, slot_words, bytes;
};

inline SphereListLayout sphere_list_layout(int nv, size_t trips, size_t slots) {
    SphereListLayout l;
    l.vals = 0;
    l.slot_vals = (size_t)1024 * nv * trips;
    l.words = l.slot_vals + (size_t)1024 * nv * slots * kProjPlanes;
    l.slot_words = l.words + (size_t)256 * trips;
    l.bytes = l.slot_words + (size_t)256 * slots + (size_t)1024 * nv * kSphereAhead;
    return l;
}

// What of a tile height's lists may be built where `room` bytes are left: 2 trips and slots, 1 the trips
// alone (another projection serves), 0 neither.
inline int sphere_lists_that_fit(int nv, size_t trips, size_t slots, size_t room) {
    if (sphere_list_layout(nv, trips, slots).bytes <= room) return 2;
    return sphere_list_layout(nv, trips, 0).bytes <= room ? 1 : 0;
}

}  // namespace qg
