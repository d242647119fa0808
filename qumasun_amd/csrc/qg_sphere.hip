// qg_sphere.hip — H·psi apply on MI355X (gfx950): stencil + local potential + projector term in
// one pass over psi, the projector values read from per-lane entry lists.
//
// Reference semantics (QUMASUN source/):
//   H psi = V psi + V_NL psi - 1/2 Lap8 psi   qumasun_mpi.matrix.h:21-43
//   V_NL psi = sum_aj E_j c_aj beta_j         PseudoPotOperator_mpi_v2.h:465-570
//   beta_j = p(r) Y_lm(r), Y_1m = sqrt(3/4pi) (y, z, x)/r, Y_1m(r^2 < 1e-14) = 0
//                                             RealSphericalHarmonics.h:149-161, SetBlockYlm.h:41
//
// A workgroup owns a tile of ty x-rows, a slab of planes and NB bands.  Every thread owns one
// group of VN = 16 / sizeof(T) consecutive x-points of one row for all NB bands and streams
// through the slab in z: the 9 z-neighbours in a register queue, the current plane (with 4
// wrapped columns and rows each side) in LDS, double buffered, one barrier per plane.
//
// Projector term.  For every (tile, plane, wavefront) the sphere images that touch a lane's
// group are listed lane by lane ("trips": entry k of all 64 lanes stored together, lanes with
// fewer entries padded with an empty image), each entry holding the radial functions at the
// lane's VN points (s channels: p(r) Y00; p channels: p(r) sqrt(3/4pi) / r, both zero outside
// the cutoff) and the group's integer displacement from the image centre.  The owner of a point
// adds
//   sum_s f_s (E c)_s + sum_p f_p [(E c)_y dy + (E c)_z dz + (E c)_x dx]
// to it from registers, so the term needs no exponentials, no LDS exchange, no barrier and no
// atomics, and every radial form (Gaussian or tabulated) costs the same.
//
// Infinities and NaN: those of psi outside every sphere reach no projection and no force.  A coefficient
// that is not finite (one inside its sphere) makes its spheres' points so, and with them the other points
// of the groups they touch (zero times the coefficient), at most VN - 1 beyond a sphere's end.
#include <algorithm>
#include <cmath>
#include <map>
#include <tuple>
#include <type_traits>
#include "qg_internal.hpp"
#include "qg_radial.hpp"

namespace qg {

namespace {

using rsrc_t = __amdgpu_buffer_rsrc_t;
using u4 = __attribute__((ext_vector_type(4))) uint32_t;

template <class T>
struct alignas(16) Row {
    T v[16 / sizeof(T)];
};

__device__ __forceinline__ rsrc_t rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}
template <class T>
__device__ __forceinline__ Row<T> vload(rsrc_t r, int voff, int soff) {
    return __builtin_bit_cast(Row<T>, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}
template <class T>
__device__ __forceinline__ void vstore(rsrc_t r, const Row<T>& v, int voff, int soff) {
    // cache policy nt: the results are not read back here, and keeping them out of L2 leaves it to
    // the halo rows and entry lists (3.42 -> 3.21 ms per application at 120^3 / 512 FP32 bands)
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, v), r, voff, soff, 2);
}

// hardware workgroup ids go round-robin over the 8 XCDs; give each XCD one contiguous range of
// logical ids (the tiles and bands of a range share halo rows and entry lists in its L2)
__device__ __forceinline__ int xcd_order(int i, int n) {
    const int xcd = i & 7, slot = i >> 3;
    const int per = n >> 3, rem = n & 7;
    return ((xcd < rem) ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + slot;
}

template <class T>
struct Coef8 {
    T c0;
    T cx[4], cy[4], cz[4];
};

template <class T>
Coef8<T> coef8(const qg_grid& g, double coef) {
    const double w[4] = {8064.0, -1008.0, 128.0, -9.0};
    Coef8<T> s;
    s.c0 = (T)(-14350.0 / 5040.0 * coef *
               (1.0 / (g.h[0] * g.h[0]) + 1.0 / (g.h[1] * g.h[1]) + 1.0 / (g.h[2] * g.h[2])));
    for (int m = 0; m < 4; ++m) {
        s.cx[m] = (T)(w[m] * coef / (5040.0 * g.h[0] * g.h[0]));
        s.cy[m] = (T)(w[m] * coef / (5040.0 * g.h[1] * g.h[1]));
        s.cz[m] = (T)(w[m] * coef / (5040.0 * g.h[2] * g.h[2]));
    }
    return s;
}

int round64i(int v) { return (v + 63) / 64 * 64; }

// buffer offset of lanes with nothing to load or store: beyond every band's num_records, so
// the hardware returns zero for the load and drops the store
constexpr int kOOB = 0x7ffffff0;
constexpr int kMaxThreads = 512;

// entry word: column image | dy offset << 10 | dx offset << 21 (the last two signed 11-bit, in
// grid points from the image's nearest grid point)
__host__ __device__ constexpr uint32_t entry_word(int li, int dx, int dy) {
    return (uint32_t)li | ((uint32_t)(dy & 2047) << 10) | ((uint32_t)(dx & 2047) << 21);
}

}  // namespace

struct SphereArgs {
    int nx, ny, nz;
    int ty, tz, ntile, nslab, nbands;
    int tg;                     // tiles per group of the workgroup order
    int nq, tpb;                // groups per row, threads per workgroup
    int64_t ld_in, ld_out;
    int nw;                     // wavefronts per workgroup
    const int* col_off;         // per tile: first column image
    const int* col_img;         // sphere image ids
    const SphereImage* images;
    const int* trip_off;        // per (tile, plane, wavefront): first trip
    int ntrips;                 // all trips, at least 1
    const void* vals;           // [trip][radial vector][lane] 16-byte vectors
    const uint32_t* words;      // [trip][lane]
    const double* coef;         // nbands x ncoef, this application's bands
    const double* coef_energy;
    const int* atom_coef_off;
    const int* atom_chan;       // [atom][4]: coefficient slots of its s, s, p, p channels (-1: none)
    int ncoef;
    int max_col;
    double h[3];
    // force pass: the occupied bands and their weights -2 occ; per workgroup and column image the
    // partial force (part[((tile * nslab + slab) * bandgroups + bandgroup) * max_col + image][3])
    const int* band_idx;
    const double* weight;
    double* part;
};

// LDS bytes of an apply workgroup; of a force workgroup with nw wavefronts (0: apply)
template <class T>
static size_t sphere_lds(int nx, int ty, int nb, int ns, int np, int max_col, int nw = 0) {
    constexpr int VN = 16 / sizeof(T);
    const size_t W = (size_t)(nx + 8 + VN - 1) / VN * VN;
    const size_t b = sizeof(T) * (2 * (size_t)nb * (ty + 8) * W + (size_t)(max_col + 1) * (4 + nb * (ns + 3 * np)));
    return (b + 15) / 16 * 16 + sizeof(double) * 3 * (size_t)nw * (max_col + 1);
}

// One workgroup of the apply pass.  NB bands; NS s and NP p channels per image; RAG: Nx is not a
// multiple of VN (the last group of a row then overlaps its neighbour: both owners compute and
// write the same values, to the bit, so a point's x displacement is formed from its own grid index
// and not from its group's; LDS is accessed by element); HV halo vectors per thread and band.
//
// FORCE: instead of H psi, the nonlocal forces F_a = sum_b (-2 occ_b) sum_i v_ba(i) D psi_b(i), with
// v_ba = sum_j E_j c_baj beta_aj the value an entry contributes to V_NL psi and D the 8th-order
// gradient: an entry's three sums stay with its lane while consecutive planes list the same image,
// then go to the wavefront's own LDS sums.
template <class T, int NB, int NS, int NP, bool RAG, int HV, bool FORCE = false>
__device__ __forceinline__ void sphere_body(const SphereArgs& a, const Coef8<T>& sc, const T* __restrict__ V,
                                            const T* __restrict__ psi, T* __restrict__ out, const int wg,
                                            unsigned char* smem) {
    constexpr int VN = 16 / sizeof(T);
    constexpr int S = sizeof(T);
    constexpr int NC = NS + 3 * NP;
    constexpr int NV = NS + NP;            // 16-byte vectors per entry
    const int nx = a.nx, ny = a.ny, nz = a.nz;
    const int W = RAG ? (nx + 8 + VN - 1) / VN * VN : nx + 8;
    const int ty = a.ty;
    const int lband = (ty + 8) * W;
    const int nthr = a.tpb;
    T* planes = reinterpret_cast<T*>(smem);                    // [2][NB][ty + 8][W]
    T* imf = planes + (size_t)2 * NB * lband;                  // [max_col + 1][4]: f.x f.y f.z, n.z
    T* ec = imf + (size_t)(a.max_col + 1) * 4;                 // [max_col + 1][NB][NC]
    // force pass: [wavefront][max_col + 1][3] sums
    const size_t foff = (sizeof(T) * (2 * (size_t)NB * lband + (size_t)(a.max_col + 1) * (4 + NB * NC)) + 15) / 16 * 16;
    double* facc = reinterpret_cast<double*>(smem + foff);

    // order: tiles of a group of tg, then bands, then slabs, then groups
    const int nbg = (a.nbands + NB - 1) / NB;
    const int grp = wg / (a.tg * nbg * a.nslab);
    const int in_grp = wg - grp * (a.tg * nbg * a.nslab);
    const int tgw = min(a.tg, a.ntile - grp * a.tg);
    const int tile = grp * a.tg + in_grp % tgw;
    const int rest = in_grp / tgw;
    const int slab = rest / nbg;
    const int b0 = (rest - slab * nbg) * NB;
    const int y0 = tile * ty;
    const int rows = min(ty, ny - y0);
    const int z0 = slab * a.tz, z1 = min(z0 + a.tz, nz);
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int nq = a.nq;
    const int r = tid / nq, xq = tid - r * nq;
    const int x = RAG ? min(xq * VN, nx - VN) : xq * VN;
    const bool own = r < rows;
    const int plane = nx * ny;
    const uint32_t band_bytes = (uint32_t)((int64_t)plane * nz * S);
    rsrc_t rin[NB], rout[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        // bands past the block read the last one and store nothing
        int band = min(b0 + b, a.nbands - 1);
        if constexpr (FORCE) band = __builtin_amdgcn_readfirstlane(a.band_idx[band]);
        rin[b] = rsrc(psi + (int64_t)band * a.ld_in, band_bytes);
        if constexpr (!FORCE) rout[b] = rsrc(out + (int64_t)band * a.ld_out, b0 + b < a.nbands ? band_bytes : 0u);
    }
    const rsrc_t rv = rsrc(V, FORCE ? 0u : band_bytes);
    const int vo = own ? ((y0 + r) * nx + x) * S : kOOB;
    const int lc = (r + 4) * W + 4 + x;
    const int lw = (x < 4) ? lc + nx : ((x >= nx - 4) ? lc - nx : -1);   // wrapped copy (whole vectors)
    int ho[HV], hl[HV];
#pragma unroll
    for (int k = 0; k < HV; ++k) {
        const int v = tid + k * nthr;
        ho[k] = kOOB;
        hl[k] = -1;
        if (v < 8 * nq) {
            const int hr = v / nq, hq = v - hr * nq;
            const int hx = RAG ? min(hq * VN, nx - VN) : hq * VN;
            int gy = (hr < 4) ? y0 - 4 + hr : y0 + rows + (hr - 4);
            gy = ((gy % ny) + ny) % ny;
            ho[k] = (gy * nx + hx) * S;
            hl[k] = ((hr < 4) ? hr : rows + hr) * W + 4 + hx;
        }
    }
    // byte offset of plane z, -nz <= z < 2 nz
    auto zoff = [&](int z) { return (z < 0 ? z + nz : (z >= nz ? z - nz : z)) * plane * S; };
    const T hx = (T)a.h[0], hy = (T)a.h[1], hz = (T)a.h[2];

    // image centres and E c of the tile's column; image ncol is the empty one of the padding
    const int c0 = a.col_off[tile];
    const int ncol = a.col_off[tile + 1] - c0;
    for (int li = tid; li <= ncol; li += nthr) {
        const SphereImage* im = a.images + a.col_img[c0 + min(li, ncol - 1)];
        const bool ok = li < ncol;
        imf[4 * li] = ok ? (T)im->f[0] : T(0);
        imf[4 * li + 1] = ok ? (T)im->f[1] : T(0);
        imf[4 * li + 2] = ok ? (T)im->f[2] : T(0);
        imf[4 * li + 3] = ok ? (T)im->n[2] : T(0);
    }
    for (int i = tid; i < (ncol + 1) * NB * NC; i += nthr) {
        const int li = i / (NB * NC), b = (i / NC) % NB, j = i % NC;
        T v = T(0);
        if (li < ncol && b0 + b < a.nbands) {
            const int at = a.images[a.col_img[c0 + li]].atom;
            const int ch = j < NS ? j : 2 + (j - NS) / 3;
            const int slot = a.atom_chan[4 * at + ch];
            if (slot >= 0) {
                const int cb = a.atom_coef_off[at] + slot + (j < NS ? 0 : (j - NS) % 3);
                double e = a.coef_energy[cb] * a.coef[(int64_t)(b0 + b) * a.ncoef + cb];
                if constexpr (FORCE) e *= a.weight[b0 + b];
                v = (T)e;
            }
        }
        ec[i] = v;
    }
    if constexpr (FORCE)
        for (int i = tid; i < 3 * a.nw * (a.max_col + 1); i += nthr) facc[i] = 0.0;

    // z-queue: step k of three planes holds the planes z - 4 .. z + 4 in q[k] .. q[k + 8] and
    // loads z + 5 into q[k + 9] (step 2: into the free q[0]); the queue moves once per three planes
    Row<T> q[NB][11];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int d = 0; d < 8; ++d) q[b][d] = vload<T>(rin[b], vo, zoff(z0 - 4 + d));
    Row<T> hn[NB][HV], vn;
    auto load_halo = [&](int z) {
        if constexpr (!FORCE) vn = vload<T>(rv, vo, zoff(z));
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int k = 0; k < HV; ++k) hn[b][k] = vload<T>(rin[b], ho[k], zoff(z));
    };
#pragma unroll
    for (int b = 0; b < NB; ++b) q[b][8] = vload<T>(rin[b], vo, zoff(z0 + 4));
    load_halo(z0);

    // the first K trips of a plane in registers, loaded a plane ahead: through buffer resources
    // of exactly the plane's trips, so that those past its last one cost no traffic and every
    // plane issues the same number of loads
    constexpr int K = 3;
    static_assert(K <= kSphereAhead, "the lists' slack covers the loads ahead");
    struct Entry {
        Row<T> f[NV];
        uint32_t w;
    };
    Entry en[K];
    const int* toff = a.trip_off + (size_t)tile * nz * a.nw + wave;
    int tb, n;      // first trip and number of trips of the plane whose entries are held
    auto load_entry = [&](rsrc_t rvals, rsrc_t rwords, int k) {
        Entry e;
#pragma unroll
        for (int v = 0; v < NV; ++v) e.f[v] = vload<T>(rvals, lane * 16, (k * NV + v) * 1024);
        e.w = __builtin_amdgcn_raw_buffer_load_b32(rwords, lane * 4, k * 256, 0);
        return e;
    };
    auto load_entries = [&](int z) {
        tb = __builtin_amdgcn_readfirstlane(toff[(size_t)z * a.nw]);
        n = __builtin_amdgcn_readfirstlane(toff[(size_t)z * a.nw + 1]) - tb;
        const rsrc_t rvals = rsrc((const unsigned char*)a.vals + (int64_t)tb * NV * 1024, (uint32_t)n * NV * 1024);
        const rsrc_t rwords = rsrc(a.words + (int64_t)tb * 64, (uint32_t)n * 256);
#pragma unroll
        for (int k = 0; k < K; ++k) en[k] = load_entry(rvals, rwords, k);
    };
    load_entries(z0);
    // force pass: the image whose sums each of the first K trips holds
    double fa[K][3];
    int cur[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        cur[k] = ncol;
        fa[k][0] = fa[k][1] = fa[k][2] = 0.0;
    }
    auto flush = [&](int li, const double (&f)[3]) {
        double* d = facc + 3 * ((size_t)wave * (a.max_col + 1) + li);
#pragma unroll
        for (int k = 0; k < 3; ++k) __hip_atomic_fetch_add(d + k, f[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    };

    auto step = [&](auto kc, int z) __attribute__((always_inline)) {
        constexpr int k0 = decltype(kc)::value;
        T* Lp = planes + (size_t)((z - z0) & 1) * NB * lband;
        const int zn = min(z + 1, z1 - 1);
        const Row<T> vcur = vn;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            T* Lb = Lp + b * lband;
            const Row<T>& cur = q[b][k0 + 4];
            if (own) {
                if constexpr (!RAG) {
                    *reinterpret_cast<Row<T>*>(Lb + lc) = cur;
                    if (lw >= 0) *reinterpret_cast<Row<T>*>(Lb + lw) = cur;
                } else {
#pragma unroll
                    for (int i = 0; i < VN; ++i) {
                        Lb[lc + i] = cur.v[i];
                        if (x + i < 4) Lb[lc + i + nx] = cur.v[i];
                        if (x + i >= nx - 4) Lb[lc + i - nx] = cur.v[i];
                    }
                }
            }
#pragma unroll
            for (int k = 0; k < HV; ++k)
                if (hl[k] >= 0) {
                    if constexpr (!RAG) {
                        *reinterpret_cast<Row<T>*>(Lb + hl[k]) = hn[b][k];
                    } else {
#pragma unroll
                        for (int i = 0; i < VN; ++i) Lb[hl[k] + i] = hn[b][k].v[i];
                    }
                }
        }
        // the next plane: every load unconditional (the slab's last plane loads one too many)
#pragma unroll
        for (int b = 0; b < NB; ++b) q[b][k0 < 2 ? k0 + 9 : 0] = vload<T>(rin[b], vo, zoff(z + 5));
        load_halo(zn);
        __syncthreads();

        Row<T> res[NB], gx[NB], gz[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            // V psi and the stencil: centre and z from the register queue, x and y from LDS
            const T* Lc = Lp + b * lband + (own ? (r + 4) * W + x : 4 * W);   // Lc[4 + i] is point x + i
            T d[VN], e[VN];
            const Row<T>* qb = q[b] + k0;
#pragma unroll
            for (int i = 0; i < VN; ++i) {
                // force pass: d, e and res are the z, x and y derivatives (weights in sc)
                if constexpr (FORCE)
                    d[i] = sc.cz[3] * (qb[8].v[i] - qb[0].v[i]) + sc.cz[2] * (qb[7].v[i] - qb[1].v[i]) +
                           sc.cz[1] * (qb[6].v[i] - qb[2].v[i]) + sc.cz[0] * (qb[5].v[i] - qb[3].v[i]);
                else
                    d[i] = sc.cz[3] * (qb[8].v[i] + qb[0].v[i]) + sc.cz[2] * (qb[7].v[i] + qb[1].v[i]) +
                           sc.cz[1] * (qb[6].v[i] + qb[2].v[i]) + sc.cz[0] * (qb[5].v[i] + qb[3].v[i]);
            }
            {
                T xsv[VN + 8];
                if constexpr (!RAG) {
#pragma unroll
                    for (int k = 0; k < (VN + 8) / VN; ++k) {
                        const Row<T> w = *reinterpret_cast<const Row<T>*>(Lc + k * VN);
#pragma unroll
                        for (int u = 0; u < VN; ++u) xsv[k * VN + u] = w.v[u];
                    }
                } else {
#pragma unroll
                    for (int k = 0; k < VN + 8; ++k) xsv[k] = Lc[k];
                }
#pragma unroll
                for (int i = 0; i < VN; ++i) {
                    if constexpr (FORCE)
                        e[i] = sc.cx[3] * (xsv[i + 8] - xsv[i]) + sc.cx[2] * (xsv[i + 7] - xsv[i + 1]) +
                               sc.cx[1] * (xsv[i + 6] - xsv[i + 2]) + sc.cx[0] * (xsv[i + 5] - xsv[i + 3]);
                    else
                        d[i] += sc.cx[3] * (xsv[i + 8] + xsv[i]) + sc.cx[2] * (xsv[i + 7] + xsv[i + 1]) +
                                sc.cx[1] * (xsv[i + 6] + xsv[i + 2]) + sc.cx[0] * (xsv[i + 5] + xsv[i + 3]);
                }
            }
            if constexpr (FORCE) res[b] = Row<T>{};
#pragma unroll
            for (int m = 3; m >= 0; --m) {
                Row<T> ym, yp;
                if constexpr (!RAG) {
                    ym = *reinterpret_cast<const Row<T>*>(Lc + 4 - (m + 1) * W);
                    yp = *reinterpret_cast<const Row<T>*>(Lc + 4 + (m + 1) * W);
                } else {
#pragma unroll
                    for (int i = 0; i < VN; ++i) {
                        ym.v[i] = Lc[4 + i - (m + 1) * W];
                        yp.v[i] = Lc[4 + i + (m + 1) * W];
                    }
                }
#pragma unroll
                for (int i = 0; i < VN; ++i) {
                    if constexpr (FORCE) res[b].v[i] += sc.cy[m] * (yp.v[i] - ym.v[i]);
                    else d[i] += sc.cy[m] * (yp.v[i] + ym.v[i]);
                }
            }
#pragma unroll
            for (int i = 0; i < VN; ++i) {
                if constexpr (FORCE) {
                    // a point of two overlapping groups counts once
                    const bool mine = !RAG || x + i >= xq * VN;
                    gx[b].v[i] = mine ? e[i] : T(0);
                    gz[b].v[i] = mine ? d[i] : T(0);
                    if (!mine) res[b].v[i] = T(0);
                } else {
                    // the large centre term last: the sums before it round at their own size
                    res[b].v[i] = vcur.v[i] * qb[4].v[i] + (sc.c0 * qb[4].v[i] + d[i]);
                }
            }
            // one band's LDS values live at a time
            __builtin_amdgcn_sched_barrier(0);
        }

        // projector term: one trip per list entry, the same number for all lanes of the wavefront
        // (an entry's channels are summed before they meet the larger stencil value)
        auto trip = [&](const Entry& e, int slot) {
            double f[3];
            const int li = (int)(e.w & 1023u);
            const int dyi = ((int)(e.w << 11)) >> 21, dxi = ((int)e.w) >> 21;
            const T* im = imf + 4 * li;
            T fx, fy, fz, nzf;
            if constexpr (VN == 4) {
                const Row<T> w = *reinterpret_cast<const Row<T>*>(im);
                fx = w.v[0]; fy = w.v[1]; fz = w.v[2]; nzf = w.v[3];
            } else {
                const Row<T> w0 = *reinterpret_cast<const Row<T>*>(im), w1 = *reinterpret_cast<const Row<T>*>(im + 2);
                fx = w0.v[0]; fy = w0.v[1]; fz = w1.v[0]; nzf = w1.v[1];
            }
            const T dx0 = hx * ((T)dxi - fx), dy = hy * ((T)dyi - fy), dz = hz * (((T)z - nzf) - fz);
            auto dx = [&](int u) { return RAG && !FORCE ? hx * ((T)(dxi + u) - fx) : dx0 + (T)u * hx; };
            // inside: leave out points outside the image
            auto bands = [&](auto inside) __attribute__((always_inline)) {
#pragma unroll
                for (int k = 0; k < 3; ++k) f[k] = 0.0;
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    T c[NC];
                    const Row<T>* ep = reinterpret_cast<const Row<T>*>(ec + ((size_t)li * NB + b) * NC);
#pragma unroll
                    for (int k = 0; k < NC / VN; ++k) {
                        const Row<T> w = ep[k];
#pragma unroll
                        for (int u = 0; u < VN; ++u) c[k * VN + u] = w.v[u];
                    }
                    T val[VN];
#pragma unroll
                    for (int u = 0; u < VN; ++u) val[u] = e.f[0].v[u] * c[0];
#pragma unroll
                    for (int s = 1; s < NS; ++s)
#pragma unroll
                        for (int u = 0; u < VN; ++u) val[u] += e.f[s].v[u] * c[s];
#pragma unroll
                    for (int p = 0; p < NP; ++p) {
                        const T cy = c[NS + 3 * p], cz = c[NS + 3 * p + 1], cx = c[NS + 3 * p + 2];
                        const T ayz = cy * dy + cz * dz;
#pragma unroll
                        for (int u = 0; u < VN; ++u) val[u] += e.f[NS + p].v[u] * (ayz + cx * dx(u));
                    }
#pragma unroll
                    for (int u = 0; u < VN; ++u) {
                        if constexpr (FORCE) {
                            if constexpr (decltype(inside)::value) {
                                bool on = false;
#pragma unroll
                                for (int v = 0; v < NV; ++v) on = on || e.f[v].v[u] != T(0);
                                if (!on) continue;
                            }
                            f[0] += (double)val[u] * (double)gx[b].v[u];
                            f[1] += (double)val[u] * (double)res[b].v[u];
                            f[2] += (double)val[u] * (double)gz[b].v[u];
                        } else {
                            res[b].v[u] += val[u];
                        }
                    }
                }
            };
            bands(std::false_type{});
            // a list's zero times an infinite or undefined gradient is not zero
            if constexpr (FORCE)
                if (__builtin_expect(__ballot(!__builtin_isfinite(f[0] + f[1] + f[2])) != 0, 0)) bands(std::true_type{});
            if constexpr (FORCE) {
                if (slot < 0) {
                    flush(li, f);
                } else {
                    if (li != cur[slot]) {
                        flush(cur[slot], fa[slot]);
                        cur[slot] = li;
                        fa[slot][0] = fa[slot][1] = fa[slot][2] = 0.0;
                    }
#pragma unroll
                    for (int k = 0; k < 3; ++k) fa[slot][k] += f[k];
                }
            }
        };
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (k < n) trip(en[k], k);
        if (n > K) {
            const rsrc_t rvals = rsrc((const unsigned char*)a.vals + (int64_t)tb * NV * 1024, (uint32_t)n * NV * 1024);
            const rsrc_t rwords = rsrc(a.words + (int64_t)tb * 64, (uint32_t)n * 256);
            for (int k = K; k < n; ++k) trip(load_entry(rvals, rwords, k), -1);
        }
        load_entries(zn);
        // lanes without a point store out of range (dropped)
        if constexpr (!FORCE)
#pragma unroll
        for (int b = 0; b < NB; ++b) vstore<T>(rout[b], res[b], vo, zoff(z));
    };
    for (int z = z0;;) {
        step(std::integral_constant<int, 0>{}, z);
        if (++z >= z1) break;
        step(std::integral_constant<int, 1>{}, z);
        if (++z >= z1) break;
        step(std::integral_constant<int, 2>{}, z);
        if (++z >= z1) break;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const Row<T> next = q[b][0];
#pragma unroll
            for (int d = 0; d < 8; ++d) q[b][d] = q[b][d + 3];
            q[b][8] = next;
        }
    }
    if constexpr (FORCE) {
#pragma unroll
        for (int k = 0; k < K; ++k) flush(cur[k], fa[k]);
        __syncthreads();
        double* part = a.part + (((size_t)tile * a.nslab + slab) * nbg + b0 / NB) * a.max_col * 3;
        for (int i = tid; i < 3 * ncol; i += nthr) {
            double s = 0.0;
            for (int w = 0; w < a.nw; ++w) s += facc[(size_t)3 * w * (a.max_col + 1) + i];
            part[i] = s;
        }
    }
}

template <class T, int NB, int NS, int NP, bool RAG, int HV>
__global__ __launch_bounds__(kMaxThreads) void sphere_hpsi_kernel(SphereArgs a, Coef8<T> sc, const T* __restrict__ V,
                                                                  const T* __restrict__ psi, T* __restrict__ out) {
    extern __shared__ __align__(16) unsigned char smem[];
    sphere_body<T, NB, NS, NP, RAG, HV>(a, sc, V, psi, out, xcd_order(blockIdx.x, gridDim.x), smem);
}

// The nonlocal force pass of FP64 bands: psi is read once (the chain of gradient blocks and their
// projections moved psi eight times: 64 atoms, 80^3, 137 occupied bands 1.45 ms after the projection of
// psi, 0.53 ms here).
template <int NB, int NS, int NP, bool RAG, int HV>
__global__ __launch_bounds__(kMaxThreads) void sphere_force_kernel(SphereArgs a, Coef8<double> sc,
                                                                   const double* __restrict__ psi) {
    extern __shared__ __align__(16) unsigned char smem[];
    sphere_body<double, NB, NS, NP, RAG, HV, true>(a, sc, nullptr, psi, nullptr, xcd_order(blockIdx.x, gridDim.x), smem);
}

// force[atom][3]: the atom's partials, over its (tile, column image) pairs and their workgroups in
// a fixed order
__global__ __launch_bounds__(256) void sphere_force_reduce_kernel(const double* __restrict__ part,
                                                                  const int* __restrict__ atom_ref_off,
                                                                  const int2* __restrict__ atom_ref, int per_tile,
                                                                  int max_col, double* __restrict__ force) {
    __shared__ double red[4][3];
    const int at = blockIdx.x;
    double f[3] = {0.0, 0.0, 0.0};
    for (int k = atom_ref_off[at]; k < atom_ref_off[at + 1]; ++k) {
        const int2 ref = atom_ref[k];
        for (int w = threadIdx.x; w < per_tile; w += 256) {
            const double* p = part + (((size_t)ref.x * per_tile + w) * max_col + ref.y) * 3;
            for (int d = 0; d < 3; ++d) f[d] += p[d];
        }
    }
    for (int d = 0; d < 3; ++d) {
        for (int s = 32; s >= 1; s >>= 1) f[d] += __shfl_xor(f[d], s, 64);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][d] = f[d];
    }
    __syncthreads();
    if (threadIdx.x < 3)
        force[3 * at + threadIdx.x] =
            red[0][threadIdx.x] + red[1][threadIdx.x] + red[2][threadIdx.x] + red[3][threadIdx.x];
}

// ------------------------------------------------------------------------ projection ----
// Bloch phases of a k-point projection: k_d h_d per grid step (real blocks: unused)
struct SpherePhase {
    double kh[3];
};

struct SphereProjArgs {
    int nx, ny, nz;
    int ty, tz, ntile, nslab, nbands;     // tz: a multiple of kProjPlanes
    int nq, tpb, nw, nepoch;
    int64_t ld;                 // in T elements per band (complex blocks: 2 per point)
    const int* col_off;
    const int* col_img;
    const SphereImage* images;
    const int* slot_off;        // per (tile, epoch, wavefront): first slot
    const uint32_t* mask;       // per (tile, epoch, wavefront, plane of the epoch): slots with points
    const void* vals;           // [slot][plane of the epoch][radial vector][lane] 16-byte vectors
    const uint32_t* words;      // [slot][lane]
    int max_col;
    double h[3];
    double* part;               // [((tile * nslab + slab) * max_col + image) * NC + c][real bands]
};

// LDS bytes of a projection workgroup: image centres, phases of the slab's planes, sums, and the
// wavefronts' exchange buffers
template <class T>
static size_t sphere_proj_lds(int max_col, int tz, int nw, int nbr, int nc, bool cplx) {
    const size_t b = sizeof(T) * (4 * (size_t)(max_col + 1) + (cplx ? 2 * (size_t)tz : 0));
    return (b + 15) / 16 * 16 + sizeof(double) * (size_t)nw * (max_col + 1) * nc * nbr +
           (size_t)nw * 64 * (sizeof(T) * nc * nbr + 16 + sizeof(int));
}

// c_aj = dV sum_i beta_j(i) psi(i).  A workgroup owns a tile, a slab of planes and NB bands; every
// lane reads its own points' psi (each value once, 16 bytes a lane, two planes ahead) and adds the
// radial values times psi to running sums.  The lists of this pass give an image the same slot
// for all planes of an epoch (kProjPlanes planes), so a slot's sums stay in registers for the
// epoch; per channel they are sum f psi (s), and sum f psi, sum u f psi, sum z f psi (p; u the
// point of the lane's group, z the plane of the epoch), which at the epoch's end give
//   c_s,  c_y = dy P0, c_z = dz0 P0 + hz Pz, c_x = dx0 P0 + hx Pu
// and go to the wavefront's own LDS sums (FP64), and at the slab's end to one partial per
// (workgroup, image, coefficient, band).  Slots beyond the K held at once take another walk of
// the epoch.  No barrier inside the loop and no projector value is evaluated.
// psi is read once; measured against the row projection (projector values evaluated per item): 120^3 /
// 512 FP32 bands 1.0 against 1.1 ms (3.5 TB/s), 24^3 / 8 FP64 bands 12 against 38 us, 40^3 / 16 FP32
// bands 15 against 41 us, tables on 77x41x117 / 72 FP64 bands 190 against 290 us (per-point tables).
// CPLX: complex bands (re, im interleaved) times exp(i k.x) of the point; the two parts are then
// two real bands (the image's own phase is applied by the reduction).
template <class T, int NB, int NS, int NP, bool RAG, bool CPLX>
__global__ __launch_bounds__(kMaxThreads) void sphere_project_kernel(SphereProjArgs a, SpherePhase ph,
                                                                     const T* __restrict__ psi) {
    constexpr int VN = 16 / sizeof(T);
    constexpr int S = sizeof(T);
    constexpr int NC = NS + 3 * NP;
    constexpr int NV = NS + NP;
    constexpr int NR = CPLX ? 2 * NB : NB;      // real bands
    constexpr int PW = CPLX ? 2 : 1;            // 16-byte vectors per lane and band
    constexpr int K = CPLX && NS == 2 && sizeof(T) == 8 ? 2 : 4;   // slots held at once (4 would spill there)
    static_assert(K <= kSphereAhead, "the lists' slack covers the loads ahead");
    constexpr int E = kProjPlanes;
    extern __shared__ __align__(16) unsigned char smem[];
    const int nx = a.nx, ny = a.ny, nz = a.nz;
    T* imf = reinterpret_cast<T*>(smem);                      // [max_col + 1][4]
    T* ez = imf + 4 * (size_t)(a.max_col + 1);                // [tz][2]
    const size_t aoff = (sizeof(T) * (4 * (size_t)(a.max_col + 1) + (CPLX ? 2 * (size_t)a.tz : 0)) + 15) / 16 * 16;
    double* sums = reinterpret_cast<double*>(smem + aoff);    // [nw][max_col + 1][NC][NR]

    // order: bands fastest (they share the tile's lists in an XCD's L2), then slabs, then tiles
    const int wg = xcd_order(blockIdx.x, gridDim.x);
    const int nbg = (a.nbands + NB - 1) / NB;
    const int b0 = wg % nbg * NB;
    const int slab = wg / nbg % a.nslab;
    const int tile = wg / (nbg * a.nslab);
    const int y0 = tile * a.ty;
    const int rows = min(a.ty, ny - y0);
    const int z0 = slab * a.tz, z1 = min(z0 + a.tz, nz);
    const int tid = threadIdx.x, nthr = a.tpb;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int r = tid / a.nq, xq = tid - r * a.nq;
    const int x = RAG ? min(xq * VN, nx - VN) : xq * VN;
    const bool own = r < rows;
    const int plane = nx * ny;
    const uint32_t band_bytes = (uint32_t)((int64_t)plane * nz * S * PW);
    rsrc_t rin[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) rin[b] = rsrc(psi + (int64_t)min(b0 + b, a.nbands - 1) * a.ld, band_bytes);
    const int vo = own ? ((y0 + r) * nx + x) * S * PW : kOOB;

    const int c0 = a.col_off[tile];
    const int ncol = a.col_off[tile + 1] - c0;
    for (int li = tid; li <= ncol; li += nthr) {
        const SphereImage* im = a.images + a.col_img[c0 + max(min(li, ncol - 1), 0)];
        const bool ok = li < ncol;
        imf[4 * li] = ok ? (T)im->f[0] : T(0);
        imf[4 * li + 1] = ok ? (T)im->f[1] : T(0);
        imf[4 * li + 2] = ok ? (T)im->f[2] : T(0);
        imf[4 * li + 3] = ok ? (T)im->n[2] : T(0);
    }
    T exy[VN][2];
    if constexpr (CPLX) {
        for (int i = tid; i < z1 - z0; i += nthr) {
            double s, c;
            sincos(ph.kh[2] * (double)(z0 + i), &s, &c);
            ez[2 * i] = (T)c;
            ez[2 * i + 1] = (T)s;
        }
#pragma unroll
        for (int u = 0; u < VN; ++u) {
            double s, c;
            sincos(ph.kh[0] * (double)(x + u) + ph.kh[1] * (double)(y0 + r), &s, &c);
            exy[u][0] = (T)c;
            exy[u][1] = (T)s;
        }
    }
    for (int i = tid; i < a.nw * (a.max_col + 1) * NC * NR; i += nthr) sums[i] = 0.0;
    __syncthreads();

    const T hx = (T)a.h[0], hy = (T)a.h[1], hz = (T)a.h[2];
    const int ep1 = (z1 + E - 1) / E;
    // one step: a plane of one walk (K slots from s0) of an epoch; uniform over the wavefront
    struct Step {
        int ep, z, s0, ns, off;     // epoch, plane, first slot of the walk, slots of the epoch, its first slot
    };
    const size_t lists = (size_t)tile * a.nepoch * a.nw + wave;
    auto open = [&](int ep) {       // the first step of the first epoch from ep on that has slots
        Step s{ep, ep * E, 0, 0, 0};
        while (s.ep < ep1) {
            s.off = __builtin_amdgcn_readfirstlane(a.slot_off[lists + (size_t)s.ep * a.nw]);
            s.ns = __builtin_amdgcn_readfirstlane(a.slot_off[lists + (size_t)s.ep * a.nw + 1]) - s.off;
            if (s.ns > 0) break;
            ++s.ep;
        }
        s.z = s.ep * E;
        return s;
    };
    auto next = [&](Step s) {
        if (s.ep >= ep1) return s;
        ++s.z;
        if (s.z < min((s.ep + 1) * E, z1)) return s;
        s.s0 += K;
        s.z = s.ep * E;
        return s.s0 < s.ns ? s : open(s.ep + 1);
    };
    auto mask_of = [&](const Step& s) -> uint32_t {
        if (s.ep >= ep1) return 0u;
        return __builtin_amdgcn_readfirstlane(a.mask[(lists + (size_t)s.ep * a.nw) * E + (s.z - s.ep * E)]) >> s.s0;
    };
    struct Vals {
        Row<T> f[NV];
    };
    constexpr int D = 2;            // planes of psi in flight (3 and 4: no faster)
    Row<T> p[D][NB][PW];
    Vals en[K];
    uint32_t wd[K];
    auto load_psi = [&](Row<T> (&q)[NB][PW], const Step& s) {
        const int z = min(s.z, nz - 1);     // past the last step: a load that is not used
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int h = 0; h < PW; ++h) q[b][h] = vload<T>(rin[b], vo + (own ? 16 * h : 0), z * plane * S * PW);
    };
    // a slot without points in the plane is loaded through an empty resource (zeros, no traffic)
    auto load_vals = [&](const Step& s, uint32_t m, int k) {
        const int64_t at = ((int64_t)(s.off + s.s0 + k) * E + (s.z - s.ep * E)) * NV * 1024;
        const bool on = (m >> k) & 1u;
        const rsrc_t rv = rsrc((const unsigned char*)a.vals + (on ? at : 0), on ? NV * 1024u : 0u);
        Vals e;
#pragma unroll
        for (int v = 0; v < NV; ++v) e.f[v] = vload<T>(rv, lane * 16, v * 1024);
        return e;
    };
    auto load_words = [&](const Step& s) {
        const int cnt = s.ep < ep1 ? min(K, s.ns - s.s0) : 0;
        const rsrc_t rw = rsrc(a.words + (cnt > 0 ? (int64_t)(s.off + s.s0) * 64 : 0), (uint32_t)max(cnt, 0) * 256);
#pragma unroll
        for (int k = 0; k < K; ++k) wd[k] = __builtin_amdgcn_raw_buffer_load_b32(rw, lane * 4, k * 256, 0);
    };

    T acc[K][NC][NR];
    auto clear = [&] {
#pragma unroll
        for (int k = 0; k < K; ++k)
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int b = 0; b < NR; ++b) acc[k][c][b] = T(0);
    };
    clear();
    // the plane's values of the lane's points as real bands; a point of two overlapping groups counts once
    auto values = [&](const Row<T> (&q)[NB][PW], int z, T (&v)[NR][VN]) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < VN; ++u) {
            const bool mine = !RAG || x + u >= xq * VN;
            if constexpr (CPLX) {
                const T cz = ez[2 * (z - z0)], sz = ez[2 * (z - z0) + 1];
                const T er = exy[u][0] * cz - exy[u][1] * sz, ei = exy[u][0] * sz + exy[u][1] * cz;
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    const T re = q[b][2 * u / VN].v[2 * u % VN], im = q[b][2 * u / VN].v[2 * u % VN + 1];
                    v[2 * b][u] = mine ? er * re - ei * im : T(0);
                    v[2 * b + 1][u] = mine ? er * im + ei * re : T(0);
                }
            } else {
#pragma unroll
                for (int b = 0; b < NB; ++b) v[b][u] = mine ? q[b][0].v[u] : T(0);
            }
        }
    };
    // the sums of one walk into the wavefront's LDS sums, a slot at a time: every lane puts its CN
    // coefficients and its image into the wavefront's buffer; then lane l owns coefficient l % CN of
    // CN neighbouring lanes, adds up runs of one image and the runs to the sums.  (Straight atomics
    // from every lane met on one address per image: 130 cycles an instruction, the time of the pass.)
    constexpr int CN = NC * NR;
    static_assert(64 % CN == 0 && CN % VN == 0, "coefficients of a slot must divide the wavefront");
    constexpr int BS = CN + VN;                              // buffer stride: 16-byte rows, no bank conflicts
    T* buf = reinterpret_cast<T*>(sums + (size_t)a.nw * (a.max_col + 1) * CN) + (size_t)wave * 64 * BS;
    int* lis = reinterpret_cast<int*>(reinterpret_cast<T*>(sums + (size_t)a.nw * (a.max_col + 1) * CN) +
                                      (size_t)a.nw * 64 * BS) + wave * 64;
    auto flush = [&](const Step& s) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            if (s.s0 + k < s.ns) {
                const int li = (int)(wd[k] & 1023u);
                const int dyi = ((int)(wd[k] << 11)) >> 21, dxi = ((int)wd[k]) >> 21;
                const T* im = imf + 4 * li;
                const T dx0 = hx * ((T)dxi - im[0]), dy = hy * ((T)dyi - im[1]);
                const T dz0 = hz * (((T)(s.ep * E) - im[3]) - im[2]);
                T c[CN];
                auto coefficients = [&]() __attribute__((always_inline)) {
                    T all = T(0);
#pragma unroll
                    for (int b = 0; b < NR; ++b) {
#pragma unroll
                        for (int q = 0; q < NS; ++q) c[q * NR + b] = acc[k][q][b];
#pragma unroll
                        for (int q = 0; q < NP; ++q) {
                            const double p0 = (double)acc[k][NS + 3 * q][b];
                            c[(NS + 3 * q) * NR + b] = (T)((double)dy * p0);
                            c[(NS + 3 * q + 1) * NR + b] =
                                (T)((double)dz0 * p0 + (double)hz * (double)acc[k][NS + 3 * q + 2][b]);
                            c[(NS + 3 * q + 2) * NR + b] =
                                (T)((double)dx0 * p0 + (double)hx * (double)acc[k][NS + 3 * q + 1][b]);
                        }
                    }
#pragma unroll
                    for (int i = 0; i < CN; ++i) all += c[i];
                    return __builtin_isfinite(all);
                };
                if (__builtin_expect(__ballot(!coefficients()) != 0, 0)) {
                    // a list's zero times an infinity or NaN at a point outside the image is not zero: the
                    // slot's epoch once more, point by point, without those
#pragma unroll
                    for (int i = 0; i < CN; ++i) c[i] = T(0);
                    for (Step t{s.ep, s.ep * E, s.s0, s.ns, s.off}; t.z < min((s.ep + 1) * E, z1); ++t.z) {
                        Row<T> q[NB][PW];
                        load_psi(q, t);
                        const Vals e = load_vals(t, mask_of(t), k);
                        T v[NR][VN];
                        values(q, t.z, v);
                        const T dz = hz * (((T)t.z - im[3]) - im[2]);
#pragma unroll
                        for (int u = 0; u < VN; ++u) {
                            const T dx = dx0 + (T)u * hx;
#pragma unroll
                            for (int b = 0; b < NR; ++b) {
#pragma unroll
                                for (int q = 0; q < NS; ++q)
                                    if (e.f[q].v[u] != T(0)) c[q * NR + b] += e.f[q].v[u] * v[b][u];
#pragma unroll
                                for (int q = 0; q < NP; ++q)
                                    if (e.f[NS + q].v[u] != T(0)) {
                                        const T w = e.f[NS + q].v[u] * v[b][u];
                                        c[(NS + 3 * q) * NR + b] += w * dy;
                                        c[(NS + 3 * q + 1) * NR + b] += w * dz;
                                        c[(NS + 3 * q + 2) * NR + b] += w * dx;
                                    }
                            }
                        }
                    }
                }
#pragma unroll
                for (int v = 0; v < CN / VN; ++v) {
                    Row<T> w;
#pragma unroll
                    for (int u = 0; u < VN; ++u) w.v[u] = c[v * VN + u];
                    *reinterpret_cast<Row<T>*>(buf + lane * BS + v * VN) = w;
                }
                lis[lane] = li;
                __builtin_amdgcn_wave_barrier();
                const int own_c = lane % CN, l0 = lane - own_c;
                auto add = [&](int row, double v) {
                    __hip_atomic_fetch_add(sums + ((size_t)wave * (a.max_col + 1) + row) * CN + own_c, v, __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_WORKGROUP);
                };
                int run = lis[l0];
                double sum = (double)buf[l0 * BS + own_c];
#pragma unroll
                for (int i = 1; i < CN; ++i) {
                    const int l = lis[l0 + i];
                    const double v = (double)buf[(l0 + i) * BS + own_c];
                    if (l != run) {
                        add(run, sum);
                        run = l;
                        sum = 0.0;
                    }
                    sum += v;
                }
                add(run, sum);
                __builtin_amdgcn_wave_barrier();
            }
        }
        clear();
    };

    Step cur = open(z0 / E), nx1 = next(cur), nx2 = next(nx1);
    uint32_t mcur = mask_of(cur), m1 = mask_of(nx1);
    load_psi(p[0], cur);
    load_words(cur);
#pragma unroll
    for (int k = 0; k < K; ++k) en[k] = load_vals(cur, mcur, k);
    Step far = nx1;
#pragma unroll
    for (int i = 1; i < D; ++i) {
        load_psi(p[i], far);
        far = next(far);
    }
    auto step = [&](auto ic) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value;
        T v[NR][VN];
        values(p[i], cur.z, v);
        const T zr = (T)(cur.z - cur.ep * E);
#pragma unroll
        for (int k = 0; k < K; ++k) {
            if ((mcur >> k) & 1u) {
#pragma unroll
                for (int b = 0; b < NR; ++b) {
#pragma unroll
                    for (int s = 0; s < NS; ++s)
#pragma unroll
                        for (int u = 0; u < VN; ++u) acc[k][s][b] += en[k].f[s].v[u] * v[b][u];
#pragma unroll
                    for (int q = 0; q < NP; ++q) {
                        T t[VN], s0 = T(0);
#pragma unroll
                        for (int u = 0; u < VN; ++u) {
                            t[u] = en[k].f[NS + q].v[u] * v[b][u];
                            s0 += t[u];
                        }
                        acc[k][NS + 3 * q][b] += s0;
#pragma unroll
                        for (int u = 1; u < VN; ++u) acc[k][NS + 3 * q + 1][b] += (T)u * t[u];
                        acc[k][NS + 3 * q + 2][b] += zr * s0;
                    }
                }
            }
            en[k] = load_vals(nx1, m1, k);
        }
        if (nx1.ep != cur.ep || nx1.s0 != cur.s0) {
            flush(cur);
            load_words(nx1);
        }
        // after the next plane's values: waiting for those leaves this load in flight
        load_psi(p[i], far);
        far = next(far);
        cur = nx1;
        nx1 = nx2;
        mcur = m1;
        m1 = mask_of(nx1);
        nx2 = next(nx2);
    };
    while (cur.ep < ep1) {
        step(std::integral_constant<int, 0>{});
        if (cur.ep >= ep1) break;
        step(std::integral_constant<int, 1>{});
    }
    __syncthreads();
    const int nbr = (CPLX ? 2 : 1) * a.nbands;
    double* part = a.part + ((size_t)tile * a.nslab + slab) * a.max_col * NC * nbr;
    for (int i = tid; i < ncol * NC * NR; i += nthr) {
        const int b = (CPLX ? 2 : 1) * b0 + i % NR;
        double s = 0.0;
        for (int w = 0; w < a.nw; ++w) s += sums[(size_t)w * (a.max_col + 1) * NC * NR + i];
        if (b < nbr) part[(size_t)(i / NR) * nbr + b] = s;
    }
}

// coef[b * ncoef + j] = dV * sum of the atom's partials over its (tile, column image) pairs and the
// slabs, in a fixed order; complex: times exp(-i k.h shift) of the image
// 64 bands by 4 parts of the sum per workgroup (the parts of one coefficient are added in order), so
// that the dependent loads of a small problem's many partials run side by side
template <bool CPLX>
__global__ __launch_bounds__(256) void sphere_coef_reduce_kernel(
    const double* __restrict__ part, int nslab, int max_col, int ns, int np, int nbands, const int* __restrict__ atom_ref_off,
    const int2* __restrict__ atom_ref, const int* __restrict__ col_off, const int* __restrict__ col_img,
    const SphereImage* __restrict__ images, const int* __restrict__ atom_chan, const int* __restrict__ atom_coef_off,
    SpherePhase ph, double dv, double* __restrict__ coef, int ncoef) {
    __shared__ double red[4][64][CPLX ? 2 : 1];
    const int nc = ns + 3 * np;
    const int at = blockIdx.x / nc, c = blockIdx.x % nc;
    const int lb = threadIdx.x & 63, q = threadIdx.x >> 6;
    const int b = blockIdx.y * 64 + lb;
    const int slot = atom_chan[4 * at + (c < ns ? c : 2 + (c - ns) / 3)];
    if (slot < 0) return;
    const int nbr = (CPLX ? 2 : 1) * nbands;
    double re = 0.0, im = 0.0;
    const int k0 = atom_ref_off[at], n = (atom_ref_off[at + 1] - k0) * nslab;
    if (b < nbands) {
#pragma unroll 4
        for (int i = q; i < n; i += 4) {
            const int2 ref = atom_ref[k0 + i / nslab];
            const double* p = part + ((((size_t)ref.x * nslab + i % nslab) * max_col + ref.y) * nc + c) * nbr;
            if constexpr (CPLX) {
                const SphereImage& g = images[col_img[col_off[ref.x] + ref.y]];
                const double sr = p[2 * b], si = p[2 * b + 1];
                double sn = 0.0, cs = 1.0;
                if (g.shift[0] | g.shift[1] | g.shift[2])
                    sincos(-(ph.kh[0] * g.shift[0] + ph.kh[1] * g.shift[1] + ph.kh[2] * g.shift[2]), &sn, &cs);
                re += cs * sr - sn * si;
                im += cs * si + sn * sr;
            } else {
                re += p[b];
            }
        }
    }
    red[q][lb][0] = re;
    if constexpr (CPLX) red[q][lb][1] = im;
    __syncthreads();
    if (q != 0 || b >= nbands) return;
    const int64_t o = (int64_t)b * ncoef + atom_coef_off[at] + slot + (c < ns ? 0 : (c - ns) % 3);
    constexpr int W = CPLX ? 2 : 1;
#pragma unroll
    for (int w = 0; w < W; ++w)
        coef[W * o + w] = dv * (((red[0][lb][w] + red[1][lb][w]) + red[2][lb][w]) + red[3][lb][w]);
}

// -------------------------------------------------------------------------- k points ----
// H_k u = coef [L8 - |k|^2 + 2 i k . D8] u + V u + sum_j E_j conj(P_j) c_j for one complex band per
// workgroup (re, im interleaved), the structure of sphere_body with the two parts in place of two
// bands: a part of a point is a fixed element of the lane's two 16-byte vectors, so the z-queue holds
// the block's own layout; LDS holds the parts in separate planes.
// The phase of P_j = beta_j exp(i k.x_u), x_u the image-frame coordinate, is the grid point's
// exp(i k.h i) times the image's exp(-i k.h shift): the second sits in the staged E c, the first is
// applied once per point to the sum over its images.
// One pass replaces stencil, projection gather and their read-modify-write: 64 atoms, 80^3, 64
// complex128 bands 465 us against 398 (stencil) + 347 (gather); occupancy (two halves of the
// z-queue, ~200 VGPRs) and L2 traffic of halo rows and lists bound it.
template <class T>
struct SphereKStencil {
    T c0;
    T a[3][4], b[3][4];     // second- and first-difference weights of offsets 1..4
};

template <class T>
static size_t sphere_kpoint_lds(int nx, int ty, int tz, int ns, int np, int max_col) {
    return sphere_lds<T>(nx, ty, 2, ns, np, max_col) + sizeof(T) * 2 * (size_t)tz;
}

template <class T, int NS, int NP, bool RAG, int HV>
__global__ __launch_bounds__(kMaxThreads) void sphere_kpoint_kernel(SphereArgs a, SphereKStencil<T> ks, SpherePhase ph,
                                                                    const T* __restrict__ V, const T* __restrict__ psi,
                                                                    T* __restrict__ out) {
    constexpr int VN = 16 / sizeof(T);
    constexpr int S = sizeof(T);
    constexpr int NC = NS + 3 * NP;
    constexpr int NV = NS + NP;
    constexpr int K = 3;
    static_assert(K <= kSphereAhead, "the lists' slack covers the loads ahead");
    extern __shared__ __align__(16) unsigned char smem[];
    const int nx = a.nx, ny = a.ny, nz = a.nz;
    const int W = RAG ? (nx + 8 + VN - 1) / VN * VN : nx + 8;
    const int ty = a.ty;
    const int lband = (ty + 8) * W;
    const int nthr = a.tpb;
    T* planes = reinterpret_cast<T*>(smem);                    // [2][re, im][ty + 8][W]
    T* imf = planes + (size_t)4 * lband;                       // [max_col + 1][4]
    T* ec = imf + (size_t)(a.max_col + 1) * 4;                 // [max_col + 1][re, im][NC]
    T* ez = ec + (size_t)(a.max_col + 1) * 2 * NC;             // [tz][2]

    const int wg = xcd_order(blockIdx.x, gridDim.x);
    const int grp = wg / (a.tg * a.nbands * a.nslab);
    const int in_grp = wg - grp * (a.tg * a.nbands * a.nslab);
    const int tgw = min(a.tg, a.ntile - grp * a.tg);
    const int tile = grp * a.tg + in_grp % tgw;
    const int rest = in_grp / tgw;
    const int slab = rest / a.nbands;
    const int band = rest - slab * a.nbands;
    const int y0 = tile * ty;
    const int rows = min(ty, ny - y0);
    const int z0 = slab * a.tz, z1 = min(z0 + a.tz, nz);
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int nq = a.nq;
    const int r = tid / nq, xq = tid - r * nq;
    const int x = RAG ? min(xq * VN, nx - VN) : xq * VN;
    const bool own = r < rows;
    const int plane = nx * ny;
    const uint32_t v_bytes = (uint32_t)((int64_t)plane * nz * S);
    const rsrc_t rin = rsrc(psi + (int64_t)band * a.ld_in, 2 * v_bytes);
    const rsrc_t rout = rsrc(out + (int64_t)band * a.ld_out, 2 * v_bytes);
    const rsrc_t rv = rsrc(V, v_bytes);
    const int pt = (y0 + r) * nx + x;
    const int vo = own ? pt * S : kOOB;                        // V
    const int vc[2] = {own ? 2 * pt * S : kOOB, own ? 2 * pt * S + 16 : kOOB};
    const int lc = (r + 4) * W + 4 + x;
    const int lw = (x < 4) ? lc + nx : ((x >= nx - 4) ? lc - nx : -1);
    int ho[HV][2], hl[HV];
#pragma unroll
    for (int k = 0; k < HV; ++k) {
        const int v = tid + k * nthr;
        ho[k][0] = ho[k][1] = kOOB;
        hl[k] = -1;
        if (v < 8 * nq) {
            const int hr = v / nq, hq = v - hr * nq;
            const int hx = RAG ? min(hq * VN, nx - VN) : hq * VN;
            int gy = (hr < 4) ? y0 - 4 + hr : y0 + rows + (hr - 4);
            gy = ((gy % ny) + ny) % ny;
            ho[k][0] = 2 * (gy * nx + hx) * S;
            ho[k][1] = ho[k][0] + 16;
            hl[k] = ((hr < 4) ? hr : rows + hr) * W + 4 + hx;
        }
    }
    auto wrapz = [&](int z) { return (z < 0 ? z + nz : (z >= nz ? z - nz : z)) * plane * S; };
    const T hx = (T)a.h[0], hy = (T)a.h[1], hz = (T)a.h[2];

    const int c0 = a.col_off[tile];
    const int ncol = a.col_off[tile + 1] - c0;
    for (int li = tid; li <= ncol; li += nthr) {
        const SphereImage* im = a.images + a.col_img[c0 + max(min(li, ncol - 1), 0)];
        const bool ok = li < ncol;
        imf[4 * li] = ok ? (T)im->f[0] : T(0);
        imf[4 * li + 1] = ok ? (T)im->f[1] : T(0);
        imf[4 * li + 2] = ok ? (T)im->f[2] : T(0);
        imf[4 * li + 3] = ok ? (T)im->n[2] : T(0);
    }
    for (int i = tid; i < (ncol + 1) * NC; i += nthr) {
        const int li = i / NC, j = i % NC;
        double er = 0.0, ei = 0.0;
        if (li < ncol) {
            const SphereImage& im = a.images[a.col_img[c0 + li]];
            const int slot = a.atom_chan[4 * im.atom + (j < NS ? j : 2 + (j - NS) / 3)];
            if (slot >= 0) {
                const int cb = a.atom_coef_off[im.atom] + slot + (j < NS ? 0 : (j - NS) % 3);
                const double e = a.coef_energy[cb];
                const double cr = e * a.coef[2 * ((int64_t)band * a.ncoef + cb)];
                const double ci = e * a.coef[2 * ((int64_t)band * a.ncoef + cb) + 1];
                double sn, cs;
                sincos(ph.kh[0] * im.shift[0] + ph.kh[1] * im.shift[1] + ph.kh[2] * im.shift[2], &sn, &cs);
                er = cr * cs - ci * sn;
                ei = cr * sn + ci * cs;
            }
        }
        ec[(size_t)li * 2 * NC + j] = (T)er;
        ec[(size_t)li * 2 * NC + NC + j] = (T)ei;
    }
    for (int i = tid; i < z1 - z0; i += nthr) {
        double s, c;
        sincos(ph.kh[2] * (double)(z0 + i), &s, &c);
        ez[2 * i] = (T)c;
        ez[2 * i + 1] = (T)s;
    }
    T exy[VN][2];
#pragma unroll
    for (int u = 0; u < VN; ++u) {
        double s, c;
        sincos(ph.kh[0] * (double)(x + u) + ph.kh[1] * (double)(y0 + r), &s, &c);
        exy[u][0] = (T)c;
        exy[u][1] = (T)s;
    }

    // part c of point u of a pair of vectors
#define QG_PART(pair, c, u) ((pair)[(2 * (u) + (c)) / VN].v[(2 * (u) + (c)) % VN])
    struct Pair {
        Row<T> h[2];
    };
    Pair q[11];     // the z-queue of sphere_body
    auto load_pair = [&](const int (&off)[2], int zo) {
        Pair p;
        p.h[0] = vload<T>(rin, off[0], 2 * zo);
        p.h[1] = vload<T>(rin, off[1], 2 * zo);
        return p;
    };
#pragma unroll
    for (int d = 0; d < 9; ++d) q[d] = load_pair(vc, wrapz(z0 - 4 + d));
    Pair hn[HV];
    Row<T> vn;
    auto load_halo = [&](int z) {
        vn = vload<T>(rv, vo, wrapz(z));
#pragma unroll
        for (int k = 0; k < HV; ++k) hn[k] = load_pair(ho[k], wrapz(z));
    };
    load_halo(z0);
    struct Entry {
        Row<T> f[NV];
        uint32_t w;
    };
    Entry en[K];
    const int* toff = a.trip_off + (size_t)tile * nz * a.nw + wave;
    int tb, n;
    auto load_entry = [&](rsrc_t rvals, rsrc_t rwords, int k) {
        Entry e;
#pragma unroll
        for (int v = 0; v < NV; ++v) e.f[v] = vload<T>(rvals, lane * 16, (k * NV + v) * 1024);
        e.w = __builtin_amdgcn_raw_buffer_load_b32(rwords, lane * 4, k * 256, 0);
        return e;
    };
    auto load_entries = [&](int z) {
        tb = __builtin_amdgcn_readfirstlane(toff[(size_t)z * a.nw]);
        n = __builtin_amdgcn_readfirstlane(toff[(size_t)z * a.nw + 1]) - tb;
        const rsrc_t rvals = rsrc((const unsigned char*)a.vals + (int64_t)tb * NV * 1024, (uint32_t)n * NV * 1024);
        const rsrc_t rwords = rsrc(a.words + (int64_t)tb * 64, (uint32_t)n * 256);
#pragma unroll
        for (int k = 0; k < K; ++k) en[k] = load_entry(rvals, rwords, k);
    };
    load_entries(z0);
    auto stage = [&](T* L, int at, const Pair& p, int c) __attribute__((always_inline)) {
        if constexpr (!RAG) {
            Row<T> w;
#pragma unroll
            for (int u = 0; u < VN; ++u) w.v[u] = QG_PART(p.h, c, u);
            *reinterpret_cast<Row<T>*>(L + at) = w;
        } else {
#pragma unroll
            for (int u = 0; u < VN; ++u) L[at + u] = QG_PART(p.h, c, u);
        }
    };

    auto step = [&](auto kc, int z) __attribute__((always_inline)) {
        constexpr int k0 = decltype(kc)::value;
        T* Lp = planes + (size_t)((z - z0) & 1) * 2 * lband;
        const int zn = min(z + 1, z1 - 1);
        const Row<T> vcur = vn;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            T* Lb = Lp + c * lband;
            if (own) {
                stage(Lb, lc, q[k0 + 4], c);
                if constexpr (!RAG) {
                    if (lw >= 0) stage(Lb, lw, q[k0 + 4], c);
                } else {
#pragma unroll
                    for (int u = 0; u < VN; ++u) {
                        if (x + u < 4) Lb[lc + u + nx] = QG_PART(q[k0 + 4].h, c, u);
                        if (x + u >= nx - 4) Lb[lc + u - nx] = QG_PART(q[k0 + 4].h, c, u);
                    }
                }
            }
#pragma unroll
            for (int k = 0; k < HV; ++k)
                if (hl[k] >= 0) stage(Lb, hl[k], hn[k], c);
        }
        q[k0 < 2 ? k0 + 9 : 0] = load_pair(vc, wrapz(z + 5));
        load_halo(zn);
        __syncthreads();

        // the stencil: d[c] collects part c; a first difference of one part enters the other
        T d[2][VN];
#pragma unroll
        for (int u = 0; u < VN; ++u) {
#pragma unroll
            for (int c = 0; c < 2; ++c) d[c][u] = T(0);
#pragma unroll
            for (int m = 3; m >= 0; --m)
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    const T up = QG_PART(q[k0 + 5 + m].h, c, u), dn = QG_PART(q[k0 + 3 - m].h, c, u);
                    d[c][u] += ks.a[2][m] * (up + dn);
                    d[1 - c][u] += (c == 0 ? ks.b[2][m] : -ks.b[2][m]) * (up - dn);
                }
        }
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const T* Lc = Lp + c * lband + (own ? (r + 4) * W + x : 4 * W);   // Lc[4 + i] is point x + i
            T xsv[VN + 8];
            if constexpr (!RAG) {
#pragma unroll
                for (int k = 0; k < (VN + 8) / VN; ++k) {
                    const Row<T> w = *reinterpret_cast<const Row<T>*>(Lc + k * VN);
#pragma unroll
                    for (int u = 0; u < VN; ++u) xsv[k * VN + u] = w.v[u];
                }
            } else {
#pragma unroll
                for (int k = 0; k < VN + 8; ++k) xsv[k] = Lc[k];
            }
#pragma unroll
            for (int u = 0; u < VN; ++u)
#pragma unroll
                for (int m = 3; m >= 0; --m) {
                    d[c][u] += ks.a[0][m] * (xsv[u + 5 + m] + xsv[u + 3 - m]);
                    d[1 - c][u] += (c == 0 ? ks.b[0][m] : -ks.b[0][m]) * (xsv[u + 5 + m] - xsv[u + 3 - m]);
                }
#pragma unroll
            for (int m = 3; m >= 0; --m) {
                Row<T> ym, yp;
                if constexpr (!RAG) {
                    ym = *reinterpret_cast<const Row<T>*>(Lc + 4 - (m + 1) * W);
                    yp = *reinterpret_cast<const Row<T>*>(Lc + 4 + (m + 1) * W);
                } else {
#pragma unroll
                    for (int i = 0; i < VN; ++i) {
                        ym.v[i] = Lc[4 + i - (m + 1) * W];
                        yp.v[i] = Lc[4 + i + (m + 1) * W];
                    }
                }
#pragma unroll
                for (int u = 0; u < VN; ++u) {
                    d[c][u] += ks.a[1][m] * (yp.v[u] + ym.v[u]);
                    d[1 - c][u] += (c == 0 ? ks.b[1][m] : -ks.b[1][m]) * (yp.v[u] - ym.v[u]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int u = 0; u < VN; ++u) {
            const T cv = ks.c0 + vcur.v[u];
#pragma unroll
            for (int c = 0; c < 2; ++c) d[c][u] += cv * QG_PART(q[k0 + 4].h, c, u);
        }
        // keep the stencil here: moved behind the projector term it would hold its operands for it
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int u = 0; u < VN; ++u) asm volatile("" : "+v"(d[c][u]));

        T nl[2][VN];
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int u = 0; u < VN; ++u) nl[c][u] = T(0);
        auto trip = [&](const Entry& e) __attribute__((always_inline)) {
            const int li = (int)(e.w & 1023u);
            const int dyi = ((int)(e.w << 11)) >> 21, dxi = ((int)e.w) >> 21;
            const T* im = imf + 4 * li;
            T fx, fy, fz, nzf;
            if constexpr (VN == 4) {
                const Row<T> w = *reinterpret_cast<const Row<T>*>(im);
                fx = w.v[0]; fy = w.v[1]; fz = w.v[2]; nzf = w.v[3];
            } else {
                const Row<T> w0 = *reinterpret_cast<const Row<T>*>(im), w1 = *reinterpret_cast<const Row<T>*>(im + 2);
                fx = w0.v[0]; fy = w0.v[1]; fz = w1.v[0]; nzf = w1.v[1];
            }
            const T dx0 = hx * ((T)dxi - fx), dy = hy * ((T)dyi - fy), dz = hz * (((T)z - nzf) - fz);
            // as in sphere_body: the same bits from both owners of a point
            auto dx = [&](int u) { return RAG ? hx * ((T)(dxi + u) - fx) : dx0 + (T)u * hx; };
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                T c[NC];
                const Row<T>* ep = reinterpret_cast<const Row<T>*>(ec + ((size_t)li * 2 + b) * NC);
#pragma unroll
                for (int k = 0; k < NC / VN; ++k) {
                    const Row<T> w = ep[k];
#pragma unroll
                    for (int u = 0; u < VN; ++u) c[k * VN + u] = w.v[u];
                }
#pragma unroll
                for (int s = 0; s < NS; ++s)
#pragma unroll
                    for (int u = 0; u < VN; ++u) nl[b][u] += e.f[s].v[u] * c[s];
#pragma unroll
                for (int p = 0; p < NP; ++p) {
                    const T ayz = c[NS + 3 * p] * dy + c[NS + 3 * p + 1] * dz;
#pragma unroll
                    for (int u = 0; u < VN; ++u)
                        nl[b][u] += e.f[NS + p].v[u] * (ayz + c[NS + 3 * p + 2] * dx(u));
                }
            }
        };
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (k < n) trip(en[k]);
        if (n > K) {
            const rsrc_t rvals = rsrc((const unsigned char*)a.vals + (int64_t)tb * NV * 1024, (uint32_t)n * NV * 1024);
            const rsrc_t rwords = rsrc(a.words + (int64_t)tb * 64, (uint32_t)n * 256);
            for (int k = K; k < n; ++k) trip(load_entry(rvals, rwords, k));
        }
        load_entries(zn);
        // conj(phase) of the point times the sum of its images
        const T cz = ez[2 * (z - z0)], sz = ez[2 * (z - z0) + 1];
        Pair o;
#pragma unroll
        for (int u = 0; u < VN; ++u) {
            const T er = exy[u][0] * cz - exy[u][1] * sz, ei = exy[u][0] * sz + exy[u][1] * cz;
            QG_PART(o.h, 0, u) = d[0][u] + (er * nl[0][u] + ei * nl[1][u]);
            QG_PART(o.h, 1, u) = d[1][u] + (er * nl[1][u] - ei * nl[0][u]);
        }
        vstore<T>(rout, o.h[0], vc[0], 2 * wrapz(z));
        vstore<T>(rout, o.h[1], vc[1], 2 * wrapz(z));
    };
    for (int z = z0;;) {
        step(std::integral_constant<int, 0>{}, z);
        if (++z >= z1) break;
        step(std::integral_constant<int, 1>{}, z);
        if (++z >= z1) break;
        step(std::integral_constant<int, 2>{}, z);
        if (++z >= z1) break;
        const Pair next = q[0];
#pragma unroll
        for (int d = 0; d < 8; ++d) q[d] = q[d + 3];
        q[8] = next;
    }
#undef QG_PART
}

// ------------------------------------------------------------------ entry lists ----
// radial function of a channel at squared distance rr (inside its cutoff), FP64
__device__ double radial_dev(const DevProj& d, const double* tables, double rr) {
    if (d.kind == QG_RADIAL_GAUSSIAN) return d.amp * exp(-rr * d.inv_2s2);
    const double* v = tables + d.table_off;
    if (d.r_min2 > rr) return v[0];
    return radial_by_rel(0.5 * log(rr) - d.xi_min, v, d.n_table, d.xi_delta);
}

struct BuildArgs {
    int nx, ny, nz, ty, ntile, nq, tpb, nw;
    double h[3];
    const int* col_off;
    const int* col_img;
    const SphereImage* images;
    const DevImage* parts;       // the per-cutoff images a sphere image is made of
    const int2* intervals;
    const DevProj* projs;
    const double* tables;
    const int* atom_chan;
    int* trips;                  // counting pass: trips per (tile, plane, wavefront)
    const int* trip_off;         // filling pass
    uint32_t* words;
    void* vals;
};

// the in-cutoff x range of part p on row (y, z), or an empty one
__device__ __forceinline__ int2 part_row(const BuildArgs& a, const DevImage& p, int y, int z) {
    if (z < p.b[2] || z >= p.e[2] || y < p.b[1] || y >= p.e[1]) return make_int2(0, 0);
    return a.intervals[p.row_base + (y - p.b[1]) + (p.e[1] - p.b[1]) * (z - p.b[2])];
}

// radial functions of image im at the VN points from (x, y, z), per channel (f zero on entry)
template <class T, int NS, int NP>
__device__ __forceinline__ void radial_rows(const BuildArgs& a, const SphereImage& im, int x, int y, int z,
                                            Row<T> (&f)[NS + NP]) {
    constexpr int VN = 16 / sizeof(T);
    for (int k = 0; k < im.nparts; ++k) {
        const DevImage& p = a.parts[im.part[k]];
        const int2 iv = part_row(a, p, y, z);
        const double dz = a.h[2] * (double)(z - p.shift[2]) - p.R[2];
        const double dy = a.h[1] * (double)(y - p.shift[1]) - p.R[1];
        for (int pj = p.proj_begin; pj < p.proj_end; ++pj) {
            const DevProj& d = a.projs[pj];
#pragma unroll
            for (int c = 0; c < NS + NP; ++c) {
                // the channel of this projector: the one whose coefficient slot it fills
                if (a.atom_chan[4 * im.atom + (c < NS ? c : 2 + c - NS)] != d.coef_rel) continue;
                if ((d.l == 0) != (c < NS)) continue;
#pragma unroll
                for (int u = 0; u < VN; ++u) {
                    if (x + u < iv.x || x + u >= iv.y) continue;
                    const double dx = a.h[0] * (double)(x + u - p.shift[0]) - p.R[0];
                    const double rr = dx * dx + (dy * dy + dz * dz);
                    const double rad = radial_dev(d, a.tables, rr);
                    if (d.l == 0) f[c].v[u] = (T)(rad * 0.28209479177387814);          // Y00
                    else f[c].v[u] = 1.0e-14 > rr ? T(0) : (T)(rad * 0.48860251190291992 / sqrt(rr));
                }
            }
        }
    }
}

// One workgroup per (tile, plane), one thread per lane of the apply workgroup.  FILL false:
// counts the images touching each lane's group and records the wavefront's largest count; FILL
// true: writes the lane's entries and pads to that count with the empty image.
template <class T, int NS, int NP, bool FILL>
__global__ __launch_bounds__(kMaxThreads) void sphere_build_kernel(BuildArgs a) {
    constexpr int VN = 16 / sizeof(T);
    constexpr int NV = NS + NP;
    const int tile = blockIdx.x, z = blockIdx.y;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int y0 = tile * a.ty;
    const int r = tid / a.nq;
    const int x = min((tid - r * a.nq) * VN, a.nx - VN);
    const int y = y0 + r;
    const bool own = r < min(a.ty, a.ny - y0);
    const int c0 = a.col_off[tile], ncol = a.col_off[tile + 1] - c0;
    const size_t w = ((size_t)tile * a.nz + z) * a.nw + wave;
    int n = 0;
    const int base = FILL ? a.trip_off[w] : 0;
    Row<T>* vals = reinterpret_cast<Row<T>*>(a.vals);
    for (int li = 0; own && li < ncol; ++li) {
        const SphereImage& im = a.images[a.col_img[c0 + li]];
        if (y < im.b[1] || y >= im.e[1] || x + VN <= im.b[0] || x >= im.e[0] || z < im.b[2] || z >= im.e[2]) continue;
        bool touch = false;
        for (int k = 0; k < im.nparts; ++k) {
            const int2 iv = part_row(a, a.parts[im.part[k]], y, z);
            touch = touch || (iv.x < x + VN && iv.y > x);
        }
        if (!touch) continue;
        if constexpr (FILL) {
            Row<T> f[NV];
#pragma unroll
            for (int c = 0; c < NV; ++c) f[c] = Row<T>{};
            radial_rows<T, NS, NP>(a, im, x, y, z, f);
#pragma unroll
            for (int c = 0; c < NV; ++c) vals[((size_t)(base + n) * NV + c) * 64 + lane] = f[c];
            a.words[(size_t)(base + n) * 64 + lane] = entry_word(li, x - im.n[0], y - im.n[1]);
        }
        ++n;
    }
    if constexpr (FILL) {
        const int cnt = a.trip_off[w + 1] - base;
        for (; n < cnt; ++n) {
#pragma unroll
            for (int c = 0; c < NV; ++c) vals[((size_t)(base + n) * NV + c) * 64 + lane] = Row<T>{};
            a.words[(size_t)(base + n) * 64 + lane] = entry_word(ncol, 0, 0);
        }
    } else {
#pragma unroll
        for (int s = 32; s >= 1; s >>= 1) n = max(n, __shfl_xor(n, s, 64));
        if (lane == 0) a.trips[w] = n;
    }
}

// The projection's lists: one workgroup per (tile, epoch).  A lane gives every image that touches its
// group in the epoch a slot, in image order.  FILL false: records the wavefront's number of slots;
// FILL true (a workgroup per plane of the epoch): writes words, values of every (slot, plane) and the
// planes' slot masks.
template <class T, int NS, int NP, bool FILL>
__global__ __launch_bounds__(kMaxThreads) void sphere_slots_kernel(BuildArgs a, uint32_t* __restrict__ mask) {
    constexpr int VN = 16 / sizeof(T);
    constexpr int NV = NS + NP;
    constexpr int E = kProjPlanes;
    const int tile = blockIdx.x, ep = blockIdx.y;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int y0 = tile * a.ty;
    const int r = tid / a.nq;
    const int x = min((tid - r * a.nq) * VN, a.nx - VN);
    const int y = y0 + r;
    const bool own = r < min(a.ty, a.ny - y0);
    const int c0 = a.col_off[tile], ncol = a.col_off[tile + 1] - c0;
    const size_t w = ((size_t)tile * gridDim.y + ep) * a.nw + wave;
    const int zb = ep * E, ze = min(zb + E, a.nz);
    int n = 0;
    const int base = FILL ? a.trip_off[w] : 0;
    const int cnt = FILL ? a.trip_off[w + 1] - base : 0;
    Row<T>* vals = reinterpret_cast<Row<T>*>(a.vals);
    const int e = blockIdx.z;     // filling: one plane of the epoch
    uint32_t has = 0u;
    for (int li = 0; own && li < ncol; ++li) {
        const SphereImage& im = a.images[a.col_img[c0 + li]];
        if (y < im.b[1] || y >= im.e[1] || x + VN <= im.b[0] || x >= im.e[0] || ze <= im.b[2] || zb >= im.e[2]) continue;
        uint32_t in = 0u;     // planes of the epoch where the image touches the group
        for (int k = 0; k < im.nparts; ++k) {
            const DevImage& part = a.parts[im.part[k]];
#pragma unroll
            for (int d = 0; d < E; ++d) {
                const int2 iv = part_row(a, part, y, zb + d);
                if (iv.x < x + VN && iv.y > x) in |= 1u << d;
            }
        }
        if (!in) continue;
        if constexpr (FILL) {
            Row<T> f[NV];
#pragma unroll
            for (int c = 0; c < NV; ++c) f[c] = Row<T>{};
            if ((in >> e) & 1u) radial_rows<T, NS, NP>(a, im, x, y, zb + e, f);
#pragma unroll
            for (int c = 0; c < NV; ++c) vals[(((size_t)(base + n) * E + e) * NV + c) * 64 + lane] = f[c];
            has |= ((in >> e) & 1u) << n;
            if (e == 0) a.words[(size_t)(base + n) * 64 + lane] = entry_word(li, x - im.n[0], y - im.n[1]);
        }
        ++n;
    }
    if constexpr (FILL) {
        for (; n < cnt; ++n) {
#pragma unroll
            for (int c = 0; c < NV; ++c) vals[(((size_t)(base + n) * E + e) * NV + c) * 64 + lane] = Row<T>{};
            if (e == 0) a.words[(size_t)(base + n) * 64 + lane] = entry_word(ncol, 0, 0);
        }
#pragma unroll
        for (int s = 32; s >= 1; s >>= 1) has |= __shfl_xor(has, s, 64);
        if (lane == 0) mask[w * E + e] = has;
    } else {
#pragma unroll
        for (int s = 32; s >= 1; s >>= 1) n = max(n, __shfl_xor(n, s, 64));
        if (lane == 0) a.trips[w] = n;
    }
}

// ------------------------------------------------------------------------ host side ----
// Tile rows for groups of nq per row: the largest product of lane use, the share of the staged
// rows that are the tile's own (8 halo rows), the share of tile rows inside the grid, and the
// wavefront slots filled (two bands per workgroup take ~175 VGPRs, so a CU holds 8 wavefronts;
// one workgroup of 8 stalls at its barriers where two of 4 overlap: 2.59 against 2.30 ms at
// 120^3, ty 16 and 8, while 12 rows beat 8 by 183 to 214 us at 80^3 / 128 FP32 bands and by 0.88
// to 1.0 ms at 80 x 80 x 120 / 192 FP64 bands)
static int sphere_pick_ty(int nq, int ny, int want) {
    if (nq > kMaxThreads) return 0;
    const int most = std::max(1, std::min(ny, kMaxThreads / nq));
    if (want > 0) return std::max(1, std::min(most, std::min(32, want)));
    int best = 1;
    double bests = -1.0;
    for (int ty = 1; ty <= std::min(most, 16); ++ty) {
        const int tpb = round64i(ty * nq), w = tpb / 64, ntile = (ny + ty - 1) / ty;
        const double slots = w <= 4 ? (8 / w) * w / 8.0 : 0.75 * w / 8.0;
        const double score = (double)ty * nq / tpb * ty / (ty + 8.0) * ny / ((double)ntile * ty) * slots;
        if (score > bests) { bests = score; best = ty; }
    }
    return best;
}

// Tile rows of the complex passes: 4 wavefronts where that leaves 6 rows or more (two workgroups of
// ~175 VGPRs a CU instead of one: 64 atoms, 80^3, 64 complex128 bands 709 us with 6 rows, 812 with 12),
// the real passes' height otherwise
static int sphere_kpoint_ty(int nq, int ny) {
    const int four = std::min(ny, 256 / std::max(1, nq));
    return four >= 6 && four < sphere_pick_ty(nq, ny, 0) ? four : sphere_pick_ty(nq, ny, 0);
}

static SphereForm sphere_form(const NlGeometry& geo, std::vector<int>& chan) {
    // coefficient slots of every atom's s, s, p, p channels; the kernels hold up to 2 + 2
    chan.assign((size_t)std::max(1, geo.natoms) * 4, -1);
    int ns = 0, np = 0;
    std::vector<char> seen(geo.natoms, 0);
    for (const DevImage& im : geo.images) {
        int* c = &chan[4 * (size_t)im.atom];
        for (int pj = im.proj_begin; pj < im.proj_end; ++pj) {
            const DevProj& d = geo.projs[pj];
            const int first = d.l == 0 ? 0 : 2;
            int k = 0;
            while (k < 2 && c[first + k] >= 0 && c[first + k] != d.coef_rel) ++k;
            if (k == 2) return SphereForm{};
            c[first + k] = d.coef_rel;
            (d.l == 0 ? ns : np) = std::max(d.l == 0 ? ns : np, k + 1);
        }
    }
    return (ns <= 1 && np <= 1) ? SphereForm{1, 1} : SphereForm{2, 2};
}

bool sphere_serves(const qg_grid& g, const qg_nonlocal* nl) {
    if (g.n[0] < 8 || g.n[0] > 1024 || g.n[2] < 8) return false;
    if (g.ng() * 8 > (int64_t)kOOB - 64) return false;   // band bytes below the out-of-range offset
    return nl->geo.ncoef > 0 && !nl->geo.images.empty() && nl->sphere_form.ns > 0;
}

// Sphere images of the whole cell (one per atom and periodic shift, all cutoffs together) and
// the channel slots, from the per-cutoff images of the geometry.
static void sphere_images(qg_nonlocal* nl) {
    const NlGeometry& geo = nl->geo;
    std::vector<int> chan;
    nl->sphere_form = sphere_form(geo, chan);
    nl->sphere_img.clear();
    if (nl->sphere_form.ns == 0) return;
    std::map<std::tuple<int, int, int, int>, int> at;
    for (int i = 0; i < (int)geo.images.size(); ++i) {
        const DevImage& im = geo.images[i];
        const auto key = std::make_tuple(im.atom, im.shift[0], im.shift[1], im.shift[2]);
        auto it = at.find(key);
        if (it == at.end()) {
            it = at.emplace(key, (int)nl->sphere_img.size()).first;
            SphereImage s{};
            s.atom = im.atom;
            for (int d = 0; d < 3; ++d) {
                const double u = im.R[d] / nl->gcopy.h[d], nn = std::rint(u);
                s.n[d] = im.shift[d] + (int)nn;
                s.shift[d] = im.shift[d];
                s.f[d] = u - nn;
                s.b[d] = im.b[d];
                s.e[d] = im.e[d];
            }
            nl->sphere_img.push_back(s);
        }
        SphereImage& s = nl->sphere_img[it->second];
        if (s.nparts == 4) { nl->sphere_form = SphereForm{}; return; }
        s.part[s.nparts++] = i;
        for (int d = 0; d < 3; ++d) {
            s.b[d] = std::min(s.b[d], im.b[d]);
            s.e[d] = std::max(s.e[d], im.e[d]);
            // the image's points, and those up to a group's start before them, as displacements from its
            // centre (which may lie outside the grid): the entry word has signed 11-bit fields
            if (s.n[d] - s.b[d] > 1000 || s.e[d] - s.n[d] > 1000) { nl->sphere_form = SphereForm{}; return; }
        }
    }
    nl->d_sphere_img.upload(nl->sphere_img.data(), nl->sphere_img.size());
    nl->d_atom_chan.upload(chan.data(), chan.size());
}

// Bytes the lists of one projector set may take, all its tile heights and types together: a sixteenth of
// the device's memory (18 GB of 288; 216 atoms on 120^3 take 250 MB in both types).  QG_SPHERE_KB: another number of
// KiB (measurement switch).
static size_t sphere_list_budget() {
    const int kb = env_int("QG_SPHERE_KB", -1);
    if (kb >= 0) return (size_t)kb << 10;
    static std::mutex mu;
    static size_t total[64] = {};
    int dev = 0;
    QG_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= 64) return (size_t)4 << 30;
    std::lock_guard<std::mutex> lk(mu);
    if (!total[dev]) {
        size_t free = 0;
        QG_HIP(hipMemGetInfo(&free, &total[dev]));
    }
    return total[dev] / 16;
}

// Entry lists of tile rows ty for the block type, built on the device on first use.  Lists beyond the
// budget, or that the device has no memory for, are left out until the next update of the nuclei: the
// row or table kernels serve in their place (ok, slots_ok false).
static SphereGeo* sphere_geometry(qg_nonlocal* nl, int dtype, int ty, bool build) {
    std::lock_guard<std::mutex> lk(nl->rows_mu);
    for (auto& c : nl->sphere)
        if (c->ty == ty && c->dtype == dtype) return c.get();
    if (!build) return nullptr;
    const qg_grid& g = nl->gcopy;
    auto c = std::make_unique<SphereGeo>();
    const int VN = dtype == QG_F32 ? 4 : 2;
    c->ty = ty;
    c->dtype = dtype;
    c->nq = (g.n[0] + VN - 1) / VN;
    c->tpb = round64i(ty * c->nq);
    c->ntile = (g.n[1] + ty - 1) / ty;
    const int nw = c->tpb / 64, nz = g.n[2];
    std::vector<std::vector<int>> col(c->ntile);
    for (int i = 0; i < (int)nl->sphere_img.size(); ++i) {
        const SphereImage& im = nl->sphere_img[i];
        for (int t = im.b[1] / ty; t <= (im.e[1] - 1) / ty; ++t) col[t].push_back(i);
    }
    std::vector<int> off(1, 0), img;
    for (auto& v : col) {
        img.insert(img.end(), v.begin(), v.end());
        off.push_back((int)img.size());
        c->max_col = std::max(c->max_col, (int)v.size());
    }
    // (tile, column image) pairs of every atom
    std::vector<std::vector<int2>> refs(nl->geo.natoms);
    for (int t = 0; t < c->ntile; ++t)
        for (int k = 0; k < (int)col[t].size(); ++k) refs[nl->sphere_img[col[t][k]].atom].push_back(make_int2(t, k));
    std::vector<int> ref_off(1, 0);
    std::vector<int2> ref;
    for (auto& v : refs) {
        ref.insert(ref.end(), v.begin(), v.end());
        ref_off.push_back((int)ref.size());
    }
    if (c->max_col < 1023) {
        // one upload for the index arrays, one read and one write of the counts, one allocation for the
        // lists: their number is what a small cell's set-up costs
        std::vector<int> meta(off);
        auto put = [&](const int* p, size_t n) {
            const size_t at = (meta.size() + 1) / 2 * 2;
            meta.resize(at + std::max<size_t>(n, 2), 0);
            std::copy(p, p + n, meta.begin() + at);
            return at;
        };
        const size_t at_img = put(img.data(), img.size()), at_roff = put(ref_off.data(), ref_off.size());
        const size_t at_ref = put(reinterpret_cast<const int*>(ref.data()), 2 * ref.size());
        c->meta.alloc(meta.size());
        QG_HIP(hipMemcpyAsync(c->meta.p, meta.data(), meta.size() * sizeof(int), hipMemcpyHostToDevice, nullptr));
        c->col_off = c->meta.p;
        c->col_img = c->meta.p + at_img;
        c->atom_ref_off = c->meta.p + at_roff;
        c->atom_ref = reinterpret_cast<const int2*>(c->meta.p + at_ref);
        const int nep = (nz + kProjPlanes - 1) / kProjPlanes;
        const size_t nwv = (size_t)c->ntile * nz * nw, ne = (size_t)c->ntile * nep * nw;
        std::vector<int> cnt(nwv + 1 + ne + 1, 0);
        c->counts.alloc(cnt.size() + ne * kProjPlanes);
        c->trip_off = c->counts.p;
        c->slot_off = c->counts.p + nwv + 1;
        uint32_t* mask = reinterpret_cast<uint32_t*>(c->counts.p + cnt.size());
        c->slot_mask = mask;
        BuildArgs a{};
        a.nx = g.n[0]; a.ny = g.n[1]; a.nz = nz;
        a.ty = ty; a.ntile = c->ntile; a.nq = c->nq; a.tpb = c->tpb; a.nw = nw;
        for (int d = 0; d < 3; ++d) a.h[d] = g.h[d];
        a.col_off = c->col_off; a.col_img = c->col_img;
        a.images = nl->d_sphere_img.p; a.parts = nl->d_images.p; a.intervals = nl->d_intervals.p;
        a.projs = nl->d_projs.p; a.tables = nl->d_tables.p; a.atom_chan = nl->d_atom_chan.p;
        BuildArgs s = a;     // the projection's lists
        a.trips = c->counts.p;
        s.trips = c->counts.p + nwv + 1;
        const bool two = nl->sphere_form.ns == 2;
        auto build = [&](auto tag, auto fill, bool slots) {
            using T = decltype(tag);
            constexpr bool F = decltype(fill)::value;
            const dim3 blk(c->tpb), tg(c->ntile, nz), sgr(c->ntile, nep, F ? kProjPlanes : 1);
            if (two) {
                hipLaunchKernelGGL((sphere_build_kernel<T, 2, 2, F>), tg, blk, 0, nullptr, a);
                if (slots) hipLaunchKernelGGL((sphere_slots_kernel<T, 2, 2, F>), sgr, blk, 0, nullptr, s, mask);
            } else {
                hipLaunchKernelGGL((sphere_build_kernel<T, 1, 1, F>), tg, blk, 0, nullptr, a);
                if (slots) hipLaunchKernelGGL((sphere_slots_kernel<T, 1, 1, F>), sgr, blk, 0, nullptr, s, mask);
            }
            QG_HIP(hipGetLastError());
        };
        dtype == QG_F32 ? build(float{}, std::false_type{}, true) : build(double{}, std::false_type{}, true);
        QG_HIP(hipMemcpy(cnt.data(), c->counts.p, cnt.size() * sizeof(int), hipMemcpyDeviceToHost));
        // counts -> offsets; a word of the masks holds 32 slots (more: the other projections serve)
        auto scan = [](int* v, size_t n, int& most) {
            int64_t sum = 0;
            for (size_t k = 0; k <= n; ++k) {
                const int m = k < n ? v[k] : 0;
                v[k] = (int)std::min<int64_t>(sum, INT32_MAX);
                sum += m;
                most = std::max(most, m);
            }
            return sum;
        };
        int most_trips = 0, most_slots = 0;
        const int64_t trips = scan(cnt.data(), nwv, most_trips), slots = scan(cnt.data() + nwv + 1, ne, most_slots);
        const int nv = nl->sphere_form.ns + nl->sphere_form.np;
        const size_t nt = (size_t)std::max<int64_t>(1, trips);
        const bool may_slots = most_slots <= 32 && slots < (1LL << 28);
        const size_t budget = sphere_list_budget(), room = budget - std::min(budget, nl->sphere_bytes);
        int fit = trips < (1LL << 30)
                      ? sphere_lists_that_fit(nv, nt, may_slots ? (size_t)std::max<int64_t>(1, slots) : 0, room)
                      : 0;
        if (fit == 2 && !may_slots) fit = 1;
        SphereListLayout l{};
        for (; fit > 0; --fit) {
            l = sphere_list_layout(nv, nt, fit == 2 ? (size_t)std::max<int64_t>(1, slots) : 0);
            if (c->lists.try_alloc(l.bytes)) break;
        }
        if (fit > 0) {
            c->slots_ok = fit == 2;
            c->ntrips = (int)nt;
            nl->sphere_bytes += l.bytes;
            QG_HIP(hipMemcpyAsync(c->counts.p, cnt.data(), cnt.size() * sizeof(int), hipMemcpyHostToDevice, nullptr));
            unsigned char* v = c->lists.p;
            c->vals = v + l.vals;
            c->slot_vals = v + l.slot_vals;
            c->words = reinterpret_cast<uint32_t*>(v + l.words);
            c->slot_words = reinterpret_cast<uint32_t*>(v + l.slot_words);
            a.trip_off = c->trip_off;
            a.words = const_cast<uint32_t*>(c->words);
            a.vals = const_cast<void*>(c->vals);
            s.trip_off = c->slot_off;
            s.words = const_cast<uint32_t*>(c->slot_words);
            s.vals = const_cast<void*>(c->slot_vals);
            dtype == QG_F32 ? build(float{}, std::true_type{}, c->slots_ok) : build(double{}, std::true_type{}, c->slots_ok);
            c->ok = true;
        }
        QG_HIP(hipStreamSynchronize(nullptr));
    }
    nl->sphere.push_back(std::move(c));
    return nl->sphere.back().get();
}

// Device state of the geometry just built into nl, with the entry lists of the default tile
// heights where the allocation-free application may need them (other lists are built at their first
// use).
void sphere_prepare(qg_nonlocal* nl) {
    nl->sphere.clear();
    nl->sphere_bytes = 0;
    sphere_images(nl);
    if (!sphere_serves(nl->gcopy, nl)) return;
    for (int dtype : {QG_F32, QG_F64}) {
        const int VN = dtype == QG_F32 ? 4 : 2;
        const int ty = sphere_pick_ty((nl->gcopy.n[0] + VN - 1) / VN, nl->gcopy.n[1], 0);
        if (ty > 0 && rows_serve(nl, dtype)) sphere_geometry(nl, dtype, ty, true);
    }
}

// 16-byte vectors of the 8 halo rows each thread stages
static int sphere_halo_vectors(int nq, int tpb) { return (8 * nq + tpb - 1) / tpb; }

template <class T, int NB, int NS, int NP>
static void sphere_launch(const SphereArgs& a, const Coef8<T>& sc, const T* V, const T* psi, T* out, size_t lds,
                          hipStream_t s) {
    const int64_t nwg = (int64_t)a.ntile * a.nslab * ((a.nbands + NB - 1) / NB);
    QG_REQUIRE(nwg < (1LL << 31), "too many workgroups");
    const dim3 grid((unsigned)nwg), blk(a.tpb);
    const bool rag = a.nx % (16 / (int)sizeof(T)) != 0;
    const int hv = sphere_halo_vectors(a.nq, a.tpb);
    QG_REQUIRE(hv <= (NB == 1 ? 8 : 1), "row tile too low for its halo");
#define QG_SPHERE_GO(RAG, HV) \
    hipLaunchKernelGGL((sphere_hpsi_kernel<T, NB, NS, NP, RAG, HV>), grid, blk, lds, s, a, sc, V, psi, out)
    if (hv <= 1) {
        if (rag) QG_SPHERE_GO(true, 1);
        else QG_SPHERE_GO(false, 1);
    } else if constexpr (NB == 1) {
        if (hv == 2) {
            if (rag) QG_SPHERE_GO(true, 2);
            else QG_SPHERE_GO(false, 2);
        } else {
            if (rag) QG_SPHERE_GO(true, 8);
            else QG_SPHERE_GO(false, 8);
        }
    }
#undef QG_SPHERE_GO
    QG_HIP(hipGetLastError());
}

template <class T>
static size_t sphere_lds_of(const qg_nonlocal* nl, const SphereGeo& sg, int nb) {
    return sphere_lds<T>(nl->gcopy.n[0], sg.ty, nb, nl->sphere_form.ns, nl->sphere_form.np, sg.max_col);
}

// Whether the apply pass of the block type runs on the entry lists prepared with the geometry
// (with one band per workgroup at least).
bool sphere_prepared(qg_nonlocal* nl, int dtype) {
    if (!sphere_serves(nl->gcopy, nl)) return false;
    const int VN = dtype == QG_F32 ? 4 : 2;
    const int nq = (nl->gcopy.n[0] + VN - 1) / VN;
    const int ty = sphere_pick_ty(nq, nl->gcopy.n[1], 0);
    const SphereGeo* sg = ty > 0 ? sphere_geometry(nl, dtype, ty, false) : nullptr;
    return sg && sg->ok && sphere_halo_vectors(nq, sg->tpb) <= 8 &&
           (dtype == QG_F32 ? sphere_lds_of<float>(nl, *sg, 1) : sphere_lds_of<double>(nl, *sg, 1)) <= lds_limit();
}

// Arguments of a launch over nbands bands, nb per workgroup, except the blocks and coefficients;
// want_tz: planes per slab (0: automatic)
static SphereArgs sphere_args(const qg_nonlocal* nl, const SphereGeo& sg, int nbands, int nb, int want_tz) {
    const qg_grid& g = nl->gcopy;
    SphereArgs a{};
    a.nx = g.n[0]; a.ny = g.n[1]; a.nz = g.n[2];
    a.ty = sg.ty;
    a.ntile = sg.ntile;
    // two neighbouring tiles, then all bands: the workgroups an XCD runs together share the
    // entry lists and V in its L2 (per application of 512 FP32 bands at 120^3 the pass reads
    // 8.0 GB so, 10.2 GB with 4 tiles, more with all)
    a.tg = std::min(sg.ntile, 2);
    a.nq = sg.nq; a.tpb = sg.tpb; a.nw = sg.tpb / 64;
    // z-slabs for about 2048 workgroups, of at least 8 planes (a slab re-reads 8), or of 3 where
    // the workgroups are too few to fill the chip: then a workgroup's chain of planes is the time
    // (24^3, 8 bands: 12.9 us in slabs of 8, 8.8 of 3; 40^3, 16 FP32 bands: 14.8 us of 8, 11.8 of 4)
    const int64_t wg = (int64_t)a.ntile * ((nbands + nb - 1) / nb);
    const int least = wg * std::max(1, g.n[2] / 8) < 512 ? 3 : 8;
    const int nslab = (int)std::max<int64_t>(1, std::min<int64_t>((2048 + wg - 1) / wg, std::max(1, g.n[2] / least)));
    a.tz = want_tz > 0 ? std::min(g.n[2], want_tz) : (g.n[2] + nslab - 1) / nslab;
    a.nslab = (g.n[2] + a.tz - 1) / a.tz;
    a.nbands = nbands;
    a.col_off = sg.col_off; a.col_img = sg.col_img;
    a.images = nl->d_sphere_img.p;
    a.trip_off = sg.trip_off;
    a.ntrips = sg.ntrips;
    a.vals = sg.vals; a.words = sg.words;
    a.coef_energy = nl->d_coef_energy.p; a.atom_coef_off = nl->d_atom_coef_off.p;
    a.atom_chan = nl->d_atom_chan.p;
    a.ncoef = nl->geo.ncoef;
    a.max_col = sg.max_col;
    for (int d = 0; d < 3; ++d) a.h[d] = g.h[d];
    return a;
}

// Two bands per workgroup (an entry is loaded once for both) where that leaves two workgroups per CU
static int sphere_pick_nb(const SphereGeo& sg, int nbands) {
    return (int64_t)sg.ntile * ((nbands + 1) / 2) >= 512 ? 2 : 1;
}

// Launch shape of a projection over nbands bands: bands per workgroup, planes per slab, partials
struct SphereProjShape {
    const SphereGeo* sg = nullptr;
    int nb = 0, tz = 0, nslab = 0;
    size_t lds = 0, npart = 0;     // npart: doubles of the partials
};

template <class T>
static bool sphere_proj_shape(qg_nonlocal* nl, int nbands, bool cplx, bool may_build, size_t most, SphereProjShape& sh) {
    if (!sphere_serves(nl->gcopy, nl)) return false;
    const qg_grid& g = nl->gcopy;
    if (cplx && g.ng() * 16 > (int64_t)kOOB - 64) return false;   // band bytes below the out-of-range offset
    constexpr int VN = 16 / sizeof(T);
    const int nq = (g.n[0] + VN - 1) / VN;
    const int ty = cplx ? sphere_kpoint_ty(nq, g.n[1]) : sphere_pick_ty(nq, g.n[1], 0);
    sh.sg = ty > 0 ? sphere_geometry(nl, sizeof(T) == 4 ? QG_F32 : QG_F64, ty, may_build) : nullptr;
    if (!sh.sg || !sh.sg->slots_ok) return false;
    const int nc = nl->sphere_form.ns + 3 * nl->sphere_form.np;
    const int nw = sh.sg->tpb / 64;
    // real bands per workgroup: 4 FP32 or 2 FP64 with 1 + 1 channels, half with 2 + 2 (their running
    // sums fill the registers)
    const int nbr = (sizeof(T) == 4 ? 4 : 2) / (nl->sphere_form.ns == 2 ? 2 : 1);
    sh.nb = cplx ? std::max(1, nbr / 2) : nbr;
    const size_t per_slab = (size_t)sh.sg->ntile * std::max(1, sh.sg->max_col) * nc * nbands * (cplx ? 2 : 1);
    auto shape = [&] {
        const SphereSlabs sl =
            sphere_project_slabs(g.n[2], (int64_t)sh.sg->ntile * ((nbands + sh.nb - 1) / sh.nb), per_slab, most);
        sh.tz = sl.tz;
        sh.nslab = sl.nslab;
        sh.lds = sphere_proj_lds<T>(sh.sg->max_col, sh.tz, nw, cplx ? 2 * sh.nb : sh.nb, nc, cplx);
    };
    shape();
    if (sh.lds > lds_limit() && sh.nb > 1) {
        sh.nb = 1;
        shape();
    }
    if (sh.lds > lds_limit()) return false;
    sh.npart = per_slab * sh.nslab;
    return true;
}

// Doubles of partials a projection of nbands bands needs; 0 where the entry lists do not serve it.
// most: the doubles there are; the slabs are fewer where they would need more (more than `most` is
// returned only where one slab does not fit).
size_t sphere_project_need(qg_nonlocal* nl, int dtype, int nbands, bool cplx, bool may_build, size_t most) {
    SphereProjShape sh;
    const bool ok = dtype == QG_F32 ? sphere_proj_shape<float>(nl, nbands, cplx, may_build, most, sh)
                                    : sphere_proj_shape<double>(nl, nbands, cplx, may_build, most, sh);
    return ok ? std::max<size_t>(1, sh.npart) : 0;
}

template <class T, int NB, int NS, int NP, bool CPLX>
static void sphere_project_launch(const SphereProjArgs& a, const SpherePhase& ph, const T* psi, size_t lds, hipStream_t s) {
    const int64_t nwg = (int64_t)a.ntile * a.nslab * ((a.nbands + NB - 1) / NB);
    QG_REQUIRE(nwg < (1LL << 31), "too many workgroups");
    const dim3 grid((unsigned)nwg), blk(a.tpb);
    if (a.nx % (16 / (int)sizeof(T)) != 0)
        hipLaunchKernelGGL((sphere_project_kernel<T, NB, NS, NP, true, CPLX>), grid, blk, lds, s, a, ph, psi);
    else
        hipLaunchKernelGGL((sphere_project_kernel<T, NB, NS, NP, false, CPLX>), grid, blk, lds, s, a, ph, psi);
    QG_HIP(hipGetLastError());
}

template <class T>
static bool sphere_project_t(qg_nonlocal* nl, int nbands, const T* psi, int64_t ld, const double* k, double* part,
                             double* coef, bool may_build, size_t most, hipStream_t s) {
    const bool cplx = k != nullptr;
    SphereProjShape sh;
    if (!sphere_proj_shape<T>(nl, nbands, cplx, may_build, most, sh)) return false;
    const qg_grid& g = nl->gcopy;
    const SphereGeo& sg = *sh.sg;
    SphereProjArgs a{};
    a.nx = g.n[0]; a.ny = g.n[1]; a.nz = g.n[2];
    a.ty = sg.ty; a.tz = sh.tz; a.ntile = sg.ntile; a.nslab = sh.nslab; a.nbands = nbands;
    a.nq = sg.nq; a.tpb = sg.tpb; a.nw = sg.tpb / 64;
    a.ld = cplx ? 2 * ld : ld;
    a.col_off = sg.col_off; a.col_img = sg.col_img; a.images = nl->d_sphere_img.p;
    a.nepoch = (g.n[2] + kProjPlanes - 1) / kProjPlanes;
    a.slot_off = sg.slot_off; a.mask = sg.slot_mask;
    a.vals = sg.slot_vals; a.words = sg.slot_words;
    a.max_col = std::max(1, sg.max_col);
    for (int d = 0; d < 3; ++d) a.h[d] = g.h[d];
    a.part = part;
    SpherePhase ph{};
    if (cplx)
        for (int d = 0; d < 3; ++d) ph.kh[d] = k[d] * g.h[d];
    constexpr int F = sizeof(T) == 4 ? 4 : 2;    // real bands with 1 + 1 channels
    const bool two = nl->sphere_form.ns == 2;
#define QG_SPHERE_PROJ(NB, NS, NP, C) sphere_project_launch<T, NB, NS, NP, C>(a, ph, psi, sh.lds, s)
    if (cplx) {
        if (two) QG_SPHERE_PROJ(1, 2, 2, true);
        else if (sh.nb == F / 2) QG_SPHERE_PROJ(F / 2, 1, 1, true);
        else QG_SPHERE_PROJ(1, 1, 1, true);
    } else if (two) {
        if (sh.nb == F / 2) QG_SPHERE_PROJ(F / 2, 2, 2, false);
        else QG_SPHERE_PROJ(1, 2, 2, false);
    } else {
        if (sh.nb == F) QG_SPHERE_PROJ(F, 1, 1, false);
        else QG_SPHERE_PROJ(1, 1, 1, false);
    }
#undef QG_SPHERE_PROJ
    const int nc = nl->sphere_form.ns + 3 * nl->sphere_form.np;
    const dim3 rgrid((unsigned)(nl->geo.natoms * nc), (unsigned)((nbands + 63) / 64));
    QG_REQUIRE(rgrid.y <= 65535, "too many bands in one projection");
    auto reduce = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, rgrid, dim3(256), 0, s, part, sh.nslab, a.max_col, nl->sphere_form.ns,
                           nl->sphere_form.np, nbands, sg.atom_ref_off, sg.atom_ref, a.col_off, a.col_img,
                           a.images, nl->d_atom_chan.p, nl->d_atom_coef_off.p, ph, g.dvol(), coef, nl->geo.ncoef);
    };
    if (cplx) reduce(sphere_coef_reduce_kernel<true>);
    else reduce(sphere_coef_reduce_kernel<false>);
    QG_HIP(hipGetLastError());
    return true;
}

// coef[b * ncoef + j] = dV sum beta_j psi_b through the entry lists, part holding
// sphere_project_need doubles (of the same `most`); k non-null: complex blocks (dtype the type of a part, ld and coef in
// complex elements) with the Bloch phases of k.  False (nothing launched) where not served.
bool sphere_project(qg_nonlocal* nl, int dtype, int nbands, const void* psi, int64_t ld, const double* k, double* part,
                    double* coef, bool may_build, hipStream_t s, size_t most) {
    if (dtype == QG_F32)
        return sphere_project_t<float>(nl, nbands, (const float*)psi, ld, k, part, coef, may_build, most, s);
    return sphere_project_t<double>(nl, nbands, (const double*)psi, ld, k, part, coef, may_build, most, s);
}

template <int NB, int NS, int NP>
static void sphere_force_launch(const SphereArgs& a, const Coef8<double>& sc, const double* psi, size_t lds, hipStream_t s) {
    const int64_t nwg = (int64_t)a.ntile * a.nslab * ((a.nbands + NB - 1) / NB);
    QG_REQUIRE(nwg < (1LL << 31), "too many workgroups");
    const dim3 grid((unsigned)nwg), blk(a.tpb);
    const bool rag = a.nx % 2 != 0;
    const int hv = sphere_halo_vectors(a.nq, a.tpb);
    QG_REQUIRE(hv <= (NB == 1 ? 8 : 1), "row tile too low for its halo");
    if (hv <= 1) {
        if (rag) hipLaunchKernelGGL((sphere_force_kernel<NB, NS, NP, true, 1>), grid, blk, lds, s, a, sc, psi);
        else hipLaunchKernelGGL((sphere_force_kernel<NB, NS, NP, false, 1>), grid, blk, lds, s, a, sc, psi);
    } else if constexpr (NB == 1) {
        if (rag) hipLaunchKernelGGL((sphere_force_kernel<NB, NS, NP, true, 8>), grid, blk, lds, s, a, sc, psi);
        else hipLaunchKernelGGL((sphere_force_kernel<NB, NS, NP, false, 8>), grid, blk, lds, s, a, sc, psi);
    }
    QG_HIP(hipGetLastError());
}

// force[atom][3] (device) = sum_b weight_b sum_j E_j c_baj dV sum_i beta_aj D psi_b over the FP64 bands
// band_idx[0 .. nocc) of psi (device arrays), coef their projections in that order.  False (nothing
// launched) where the entry lists do not serve the grid or projector set; run false only says so.
bool sphere_nonlocal_force(qg_nonlocal* nl, int nocc, const int* band_idx, const double* weight, const double* psi,
                           int64_t ld, const double* coef, DevBuf<double>& part, double* force, bool run, hipStream_t s) {
    if (!sphere_serves(nl->gcopy, nl)) return false;
    const qg_grid& g = nl->gcopy;
    const int nq = (g.n[0] + 1) / 2;
    const int ty = sphere_pick_ty(nq, g.n[1], 0);
    const SphereGeo* sg = ty > 0 ? sphere_geometry(nl, QG_F64, ty, true) : nullptr;
    if (!sg || !sg->ok || sphere_halo_vectors(nq, sg->tpb) > 8) return false;
    const int nw = sg->tpb / 64;
    auto lds_of = [&](int b) {
        return sphere_lds<double>(g.n[0], ty, b, nl->sphere_form.ns, nl->sphere_form.np, sg->max_col, nw);
    };
    // two bands share an entry, its running sums and their LDS updates (64 atoms, 80^3, 137 FP64
    // bands: 0.84 ms a call against 1.0 with one); 2 + 2 channels of two bands would spill
    int nb = nl->sphere_form.ns == 2 || (int64_t)sg->ntile * ((nocc + 1) / 2) < 256 ? 1 : 2;
    if (nb > 1 && (sphere_halo_vectors(nq, sg->tpb) > 1 || lds_of(nb) > lds_limit())) nb = 1;
    if (lds_of(nb) > lds_limit()) return false;
    if (!run) return true;
    SphereArgs a = sphere_args(nl, *sg, nocc, nb, 0);
    a.ld_in = ld;
    a.coef = coef;
    a.band_idx = band_idx;
    a.weight = weight;
    const int per_tile = a.nslab * ((nocc + nb - 1) / nb);
    part.alloc((size_t)a.ntile * per_tile * std::max(1, a.max_col) * 3);
    a.part = part.p;
    // 8th-order first-difference weights, dV of the projection's dot product in them
    Coef8<double> sc{};
    const double w[4] = {672.0, -168.0, 32.0, -3.0};
    for (int m = 0; m < 4; ++m) {
        sc.cx[m] = g.dvol() * w[m] / (840.0 * g.h[0]);
        sc.cy[m] = g.dvol() * w[m] / (840.0 * g.h[1]);
        sc.cz[m] = g.dvol() * w[m] / (840.0 * g.h[2]);
    }
    const size_t lds = lds_of(nb);
    if (nl->sphere_form.ns == 2) {
        sphere_force_launch<1, 2, 2>(a, sc, psi, lds, s);
    } else {
        if (nb == 2) sphere_force_launch<2, 1, 1>(a, sc, psi, lds, s);
        else sphere_force_launch<1, 1, 1>(a, sc, psi, lds, s);
    }
    hipLaunchKernelGGL(sphere_force_reduce_kernel, dim3(nl->geo.natoms), dim3(256), 0, s, a.part, sg->atom_ref_off,
                       sg->atom_ref, per_tile, a.max_col, force);
    QG_HIP(hipGetLastError());
    return true;
}

template <class T>
static bool sphere_apply_t(qg_ham* h, int nbands, const T* psi, int64_t ld, T* hpsi, int64_t ld_out,
                           const double* coef, bool may_build, bool run, hipStream_t s) {
    const qg_grid& g = h->grid;
    qg_nonlocal* nl = h->nl;
    constexpr int VN = 16 / sizeof(T);
    const int dtype = sizeof(T) == 4 ? QG_F32 : QG_F64;
    const int nq = (g.n[0] + VN - 1) / VN;
    int ty = sphere_pick_ty(nq, g.n[1], h->plan.rows_ty);
    if (ty == 0) return false;
    const SphereGeo* sg = sphere_geometry(nl, dtype, ty, may_build);
    if ((!sg || !sg->ok) && h->plan.rows_ty > 0) {
        // nothing may be built now, or not these: the tile height prepared with the geometry
        ty = sphere_pick_ty(nq, g.n[1], 0);
        sg = sphere_geometry(nl, dtype, ty, may_build);
    }
    if (!sg || !sg->ok) return false;
    const bool two = nl->sphere_form.ns == 2;
    int nb = h->plan.rows_bands > 0 ? std::min(2, h->plan.rows_bands) : sphere_pick_nb(*sg, nbands);
    auto lds_of = [&](int b) { return sphere_lds_of<T>(nl, *sg, b); };
    if (nb > 1 && (sphere_halo_vectors(nq, sg->tpb) > 1 || lds_of(nb) > lds_limit())) nb = 1;
    if (lds_of(nb) > lds_limit() || sphere_halo_vectors(nq, sg->tpb) > 8) return false;
    if (!run) return true;
    SphereArgs a = sphere_args(nl, *sg, nbands, nb, h->plan.rows_tz);
    a.ld_in = ld; a.ld_out = ld_out;
    a.coef = coef;
    const T* V = sizeof(T) == 4 ? (const T*)(const void*)h->V32.p : (const T*)(const void*)h->V64.p;
    const Coef8<T> sc = coef8<T>(g, -0.5);
    const size_t lds = lds_of(nb);
    if (two) {
        if (nb == 2) sphere_launch<T, 2, 2, 2>(a, sc, V, psi, hpsi, lds, s);
        else sphere_launch<T, 1, 2, 2>(a, sc, V, psi, hpsi, lds, s);
    } else {
        if (nb == 2) sphere_launch<T, 2, 1, 1>(a, sc, V, psi, hpsi, lds, s);
        else sphere_launch<T, 1, 1, 1>(a, sc, V, psi, hpsi, lds, s);
    }
    return true;
}

// H psi = V psi - 1/2 Lap8 psi + sum E c beta from the coefficients coef (nbands x ncoef), in
// one launch; false (nothing launched) where the entry lists do not serve the grid or projector
// set.  may_build: the lists of this tile height may be built now.  run false: only says whether
// the call would be served.
bool sphere_hamiltonian_apply(qg_ham* h, int dtype, int nbands, const void* psi, int64_t ld, void* hpsi,
                              int64_t ld_out, const double* coef, bool may_build, bool run,
                              hipStream_t s) {
    if (!h->nl || !sphere_serves(h->grid, h->nl)) return false;
    if (dtype == QG_F32)
        return sphere_apply_t<float>(h, nbands, (const float*)psi, ld, (float*)hpsi, ld_out, coef, may_build,
                                     run, s);
    return sphere_apply_t<double>(h, nbands, (const double*)psi, ld, (double*)hpsi, ld_out, coef, may_build,
                                  run, s);
}

template <class T, int NS, int NP>
static void sphere_kpoint_launch(const SphereArgs& a, const SphereKStencil<T>& ks, const SpherePhase& ph, const T* V,
                                 const T* psi, T* out, size_t lds, int hv, hipStream_t s) {
    const int64_t nwg = (int64_t)a.ntile * a.nslab * a.nbands;
    QG_REQUIRE(nwg < (1LL << 31), "too many workgroups");
    const dim3 grid((unsigned)nwg), blk(a.tpb);
    const bool rag = a.nx % (16 / (int)sizeof(T)) != 0;
    if (hv <= 1) {
        if (rag) hipLaunchKernelGGL((sphere_kpoint_kernel<T, NS, NP, true, 1>), grid, blk, lds, s, a, ks, ph, V, psi, out);
        else hipLaunchKernelGGL((sphere_kpoint_kernel<T, NS, NP, false, 1>), grid, blk, lds, s, a, ks, ph, V, psi, out);
    } else {
        if (rag) hipLaunchKernelGGL((sphere_kpoint_kernel<T, NS, NP, true, 2>), grid, blk, lds, s, a, ks, ph, V, psi, out);
        else hipLaunchKernelGGL((sphere_kpoint_kernel<T, NS, NP, false, 2>), grid, blk, lds, s, a, ks, ph, V, psi, out);
    }
    QG_HIP(hipGetLastError());
}

template <class T>
static bool sphere_kpoint_t(qg_ham* h, const double* k, int nbands, const T* psi, int64_t ld, T* out, int64_t ld_out,
                            DevBuf<double>& part, double* coef, hipStream_t s) {
    qg_nonlocal* nl = h->nl;
    const qg_grid& g = h->grid;
    constexpr int VN = 16 / sizeof(T);
    const int dtype = sizeof(T) == 4 ? QG_F32 : QG_F64;
    const size_t need = sphere_project_need(nl, dtype, std::max(1, nbands), true, true);
    if (need == 0) return false;
    const int nq = (g.n[0] + VN - 1) / VN;
    const int ty = sphere_kpoint_ty(nq, g.n[1]);
    const SphereGeo* sg = sphere_geometry(nl, dtype, ty, true);
    const int hv = sphere_halo_vectors(nq, sg->tpb);
    if (!sg->ok || hv > 2) return false;
    if (sphere_kpoint_lds<T>(g.n[0], ty, g.n[2], nl->sphere_form.ns, nl->sphere_form.np, sg->max_col) > lds_limit())
        return false;
    if (nbands == 0) return true;
    SphereArgs a = sphere_args(nl, *sg, nbands, 1, 0);
    const size_t lds = sphere_kpoint_lds<T>(g.n[0], ty, a.tz, nl->sphere_form.ns, nl->sphere_form.np, sg->max_col);
    part.alloc(need);
    (void)sphere_project(nl, dtype, nbands, psi, ld, k, part.p, coef, true, s);
    a.ld_in = 2 * ld; a.ld_out = 2 * ld_out;
    a.coef = coef;
    const double cf = -0.5, k2 = k[0] * k[0] + k[1] * k[1] + k[2] * k[2];
    SphereKStencil<T> ks;
    ks.c0 = (T)(-14350.0 / 5040.0 * cf * (1.0 / (g.h[0] * g.h[0]) + 1.0 / (g.h[1] * g.h[1]) + 1.0 / (g.h[2] * g.h[2])) -
                cf * k2);
    const double w2[4] = {8064.0, -1008.0, 128.0, -9.0}, w1[4] = {672.0, -168.0, 32.0, -3.0};
    for (int d = 0; d < 3; ++d)
        for (int m = 0; m < 4; ++m) {
            ks.a[d][m] = (T)(w2[m] * cf / (5040.0 * g.h[d] * g.h[d]));
            ks.b[d][m] = (T)(2.0 * cf * k[d] * w1[m] / (840.0 * g.h[d]));
        }
    SpherePhase ph;
    for (int d = 0; d < 3; ++d) ph.kh[d] = k[d] * g.h[d];
    const T* V = sizeof(T) == 4 ? (const T*)(const void*)h->V32.p : (const T*)(const void*)h->V64.p;
    if (nl->sphere_form.ns == 2) sphere_kpoint_launch<T, 2, 2>(a, ks, ph, V, psi, out, lds, hv, s);
    else sphere_kpoint_launch<T, 1, 1>(a, ks, ph, V, psi, out, lds, hv, s);
    return true;
}

// H_k of complex blocks (interleaved; dtype the type of a part, ld in complex elements): projection
// into coef (complex, nbands x ncoef) and one apply pass.  False (nothing launched) where the entry
// lists do not serve; nbands 0: prepares the lists and says so.
bool sphere_kpoint_apply(qg_ham* h, const double* k, int dtype, int nbands, const void* psi, int64_t ld, void* out,
                         int64_t ld_out, DevBuf<double>& part, double* coef, hipStream_t s) {
    if (!h->nl || !sphere_serves(h->grid, h->nl)) return false;
    if (h->grid.ng() * (dtype == QG_F32 ? 8 : 16) > (int64_t)kOOB - 64) return false;
    if (dtype == QG_F32)
        return sphere_kpoint_t<float>(h, k, nbands, (const float*)psi, ld, (float*)out, ld_out, part, coef, s);
    return sphere_kpoint_t<double>(h, k, nbands, (const double*)psi, ld, (double*)out, ld_out, part, coef, s);
}

}  // namespace qg
