// FP64 products of tall blocks (K grid points x a few hundred bands) on the FP64 matrix cores: the Gram
// blocks C = A^T B of the Rayleigh-Ritz step and the Ritz update Out = A C.  Columns (bands) are
// contiguous over the grid.
#include "qg_gram64_split.hpp"
#include "qg_internal.hpp"

#include <algorithm>
#include <type_traits>

namespace qg {

typedef double f64x2 __attribute__((ext_vector_type(2)));
typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(1))) void* global_ptr;
typedef __attribute__((address_space(3))) void* lds_ptr;

constexpr int kGramThreads = 512;
constexpr int kGramSlabs = 2;      // slabs of 8 points of one step
constexpr int kGramStages = 3;     // steps in LDS: one in use, two on their way

struct GramArgs {
    const double *A, *B;
    double* ws;
    int64_t lda, ldb, K, per;
    int M, N, mb, nb;              // bands; blocks of rows and of columns
};

// Ends a step: this wavefront's reads of LDS are done, all but its newest n (at most 6) loads to LDS have
// landed, and every wavefront has come this far.  __syncthreads would wait for the newest too.
__device__ __forceinline__ void step_barrier(int n) {
    asm volatile("" ::: "memory");
    switch (n) {    // lgkmcnt(0) vmcnt(n)
        case 0: __builtin_amdgcn_s_waitcnt(0x0070); break;
        case 1: __builtin_amdgcn_s_waitcnt(0x0071); break;
        case 2: __builtin_amdgcn_s_waitcnt(0x0072); break;
        case 3: __builtin_amdgcn_s_waitcnt(0x0073); break;
        case 4: __builtin_amdgcn_s_waitcnt(0x0074); break;
        case 5: __builtin_amdgcn_s_waitcnt(0x0075); break;
        default: __builtin_amdgcn_s_waitcnt(0x0076); break;
    }
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// A wavefront's part: NI x NJ tiles from tile row i0 and column j0 of the block.  Every wavefront of the
// workgroup passes the same number of barriers (one per step and one before them).
template <int NI, int NJ>
__device__ __forceinline__ void gram64_wave(const GramArgs& g, unsigned char* smem, int chunk, int m0, int n0, int tm,
                                            int tn, int w, int i0, int j0) {
    constexpr int KS = kGramSlabs;
    const int lane = threadIdx.x & 63, lb = lane & 15, lp = (lane >> 4) * 2;
    const int nt = tm + tn;                            // staged tiles: A's, then B's
    const int64_t p0 = chunk * g.per, p1 = min(g.K, p0 + g.per);
    const int steps = (int)((p1 - p0 + 8 * KS - 1) / (8 * KS));
    const int loads = (nt * KS - w + 7) / 8;           // of this wavefront per step
    auto load = [&](int st) __attribute__((always_inline)) {
        unsigned char* base = smem + (size_t)(st % kGramStages) * nt * KS * 1024;
        const int64_t p = p0 + (int64_t)st * 8 * KS + lp;
        for (int c = w; c < nt * KS; c += 8) {
            const int t = c / KS, k = c - t * KS;
            const bool a = t < tm;
            const int band = a ? min(m0 + 16 * t + lb, g.M - 1) : min(n0 + 16 * (t - tm) + lb, g.N - 1);
            const double* src = (a ? g.A + (int64_t)band * g.lda : g.B + (int64_t)band * g.ldb) + min(p + 8 * k, g.K - 2);
            __builtin_amdgcn_global_load_lds((global_ptr)src, (lds_ptr)(base + (size_t)c * 1024), 16, 0, 0);
        }
    };
    f64x4 acc[NI > 0 ? NI : 1][NJ > 0 ? NJ : 1];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = f64x4{0.0, 0.0, 0.0, 0.0};

    struct Slab {
        f64x2 a[NI > 0 ? NI : 1], b[NJ > 0 ? NJ : 1];
    };
    auto read = [&](int st, int k, Slab& o) __attribute__((always_inline)) {
        const unsigned char* base = smem + (size_t)(st % kGramStages) * nt * KS * 1024 + lane * 16;
#pragma unroll
        for (int i = 0; i < NI; ++i) o.a[i] = *reinterpret_cast<const f64x2*>(base + (size_t)((i0 + i) * KS + k) * 1024);
#pragma unroll
        for (int j = 0; j < NJ; ++j)
            o.b[j] = *reinterpret_cast<const f64x2*>(base + (size_t)((tm + j0 + j) * KS + k) * 1024);
    };
    auto multiply = [&](int st, int k, Slab& o) __attribute__((always_inline)) {
        if (p0 + (int64_t)(st + 1) * 8 * KS > p1) {
            const bool ok = p0 + (int64_t)st * 8 * KS + 8 * k + lp < p1;    // K is even: both points or neither
#pragma unroll
            for (int i = 0; i < NI; ++i) o.a[i] = ok ? o.a[i] : f64x2{0.0, 0.0};
#pragma unroll
            for (int j = 0; j < NJ; ++j) o.b[j] = ok ? o.b[j] : f64x2{0.0, 0.0};
        }
#pragma unroll
        for (int i = 0; i < NI; ++i) {
#pragma unroll
            for (int j = 0; j < NJ; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(o.a[i].x, o.b[j].x, acc[i][j], 0, 0, 0);
#pragma unroll
            for (int j = 0; j < NJ; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(o.a[i].y, o.b[j].y, acc[i][j], 0, 0, 0);
        }
    };

    // a slab's operands are read ahead of the products of the one before it, so that products cover the
    // reads and the barrier
    static_assert(KS == 2, "two slabs a step");
    load(0);
    if (steps > 1) load(1);
    step_barrier(steps > 1 ? loads : 0);
    Slab s0, s1;
    read(0, 0, s0);
    for (int st = 0; st < steps; ++st) {
        if (st + 2 < steps) load(st + 2);
        read(st, 1, s1);
        __builtin_amdgcn_sched_barrier(0);
        multiply(st, 0, s0);
        step_barrier(st + 2 < steps ? loads : 0);
        if (st + 1 < steps) read(st + 1, 0, s0);
        __builtin_amdgcn_sched_barrier(0);
        multiply(st, 1, s1);
    }
    double* out = g.ws + (size_t)chunk * g.M * g.N;
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int n = n0 + 16 * (j0 + j) + lb;
            if (n >= g.N) continue;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = m0 + 16 * (i0 + i) + (lane >> 4) + 4 * r;
                if (m < g.M) out[m + (int64_t)g.M * n] = acc[i][j][r];
            }
        }
}

// One workgroup: a block of 2 TM - 2 to 2 TM by 4 TN - 4 to 4 TN tiles (16 x 16) of C over one range of
// points, summed in registers.  Wavefront w holds a half of the rows (w / 4) and a quarter of the columns
// (the second half takes the quarters in reverse, so that the two wavefronts of a SIMD hold a large and a
// small share); the code of each share's size is its own, as products under conditions cost more.
// A slab of a 16-band tile (8 points) is 1 KB of LDS in operand order: lane l's 16 bytes are band l % 16,
// points 2 (l / 16) and + 1, which a direct load to LDS fills and one 16-byte read hands to two
// v_mfma_f64_16x16x4 (the order of the points within a product is free).  Two steps are on their way
// while one is in use.  Bands past the last read the last one, points past the last become zeros.
// Bound by the FP64 matrix rate and, below ~100 bands, by memory; the wavefronts of a step are uneven
// (144 bands: 23 of 20.25 tiles on the fullest SIMD).  Against the library's strided-batched product in
// 64 ranges, us: 512,000 points x 8 x 8 75 : 269, 64 x 64 163 : 336, 96 x 96 257 : 338, 144 x 144
// 490 : 757 (300 at 71 TFLOP/s); 13,824 x 16 x 16 25 : 138; where the library's tiles are full it is the
// faster one (gram64_faster).
template <int TM, int TN>
__global__ __launch_bounds__(kGramThreads, 2) void gram64_kernel(GramArgs g) {
    extern __shared__ __align__(16) unsigned char gsmem[];
    const int chunk = blockIdx.x / (g.mb * g.nb), blk = blockIdx.x - chunk * g.mb * g.nb;
    const int bi = blk % g.mb, bj = blk / g.mb, mt = (g.M + 15) / 16, ntl = (g.N + 15) / 16;
    const int tm0 = mt * bi / g.mb, tm = mt * (bi + 1) / g.mb - tm0;
    const int tn0 = ntl * bj / g.nb, tn = ntl * (bj + 1) / g.nb - tn0;
    const int m0 = 16 * tm0, n0 = 16 * tn0;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rh = w >> 2, cq = rh ? 3 - (w & 3) : (w & 3);
    const int mh = (tm + 1) / 2;
    const int i0 = rh * mh, ni = rh ? tm - mh : mh;
    const int j0 = tn * cq / 4, nj = tn * (cq + 1) / 4 - j0;
    if (ni == TM) {
        if (nj == TN) gram64_wave<TM, TN>(g, gsmem, chunk, m0, n0, tm, tn, w, i0, j0);
        else gram64_wave<TM, TN - 1>(g, gsmem, chunk, m0, n0, tm, tn, w, i0, j0);
    } else {
        if (nj == TN) gram64_wave<TM - 1, TN>(g, gsmem, chunk, m0, n0, tm, tn, w, i0, j0);
        else gram64_wave<TM - 1, TN - 1>(g, gsmem, chunk, m0, n0, tm, tn, w, i0, j0);
    }
}

// C[m + ldc n] = sum over the ranges: 64 entries per workgroup, four lanes' shares of the ranges each
__global__ __launch_bounds__(256) void gram64_reduce_kernel(const double* __restrict__ ws, int nch, int M, int N,
                                                            double* __restrict__ C, int ldc) {
    __shared__ double part[4][64];
    const int64_t i = blockIdx.x * (int64_t)64 + (threadIdx.x & 63), nn = (int64_t)M * N;
    const int q = threadIdx.x >> 6;
    double s = 0.0;
    if (i < nn)
        for (int c = q; c < nch; c += 4) s += ws[(int64_t)c * nn + i];
    part[q][threadIdx.x & 63] = s;
    __syncthreads();
    if (q == 0 && i < nn)
        C[(i % M) + (int64_t)ldc * (i / M)] = ((part[0][threadIdx.x] + part[1][threadIdx.x]) + part[2][threadIdx.x]) +
                                              part[3][threadIdx.x];
}

size_t gram64_workspace(int64_t K, int M, int N) { return (size_t)gram64_split(K, M, N).nch * M * N * sizeof(double); }

// Whether the operands suit the kernel (whole 16-byte vectors) and it is the faster one against the
// library's product in `chunks` chunks
bool gram64_serves(const double* A, int64_t lda, const double* B, int64_t ldb, int64_t K, int M, int N, int64_t chunks) {
    return K >= 2 && K % 2 == 0 && M > 0 && N > 0 && lda % 2 == 0 && ldb % 2 == 0 && reinterpret_cast<uintptr_t>(A) % 16 == 0 &&
           reinterpret_cast<uintptr_t>(B) % 16 == 0 && gram64_faster(K, M, N, chunks);
}

// C (M x N, column stride ldc) = A^T B over K points
void gram64(const double* A, int64_t lda, const double* B, int64_t ldb, int64_t K, int M, int N, double* C, int ldc,
            double* ws, size_t ws_bytes, hipStream_t s) {
    const GramSplit g = gram64_split(K, M, N);
    QG_REQUIRE(ws_bytes >= gram64_workspace(K, M, N), "Gram workspace too small");
    const size_t lds = (size_t)kGramStages * (g.bm + g.bn) * kGramSlabs * 1024;
    const GramArgs a{A, B, ws, lda, ldb, K, g.per, M, N, g.mb, g.nb};
    auto go = [&](auto kernel) {
        QG_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)lds));
        hipLaunchKernelGGL(kernel, dim3((unsigned)(g.nch * g.mb * g.nb)), dim3(kGramThreads), lds, s, a);
    };
    auto rows = [&](auto tn) {
        constexpr int TN = decltype(tn)::value;
        switch ((g.bm + 1) / 2) {
            case 1: go(gram64_kernel<1, TN>); break;
            case 2: go(gram64_kernel<2, TN>); break;
            case 3: go(gram64_kernel<3, TN>); break;
            case 4: go(gram64_kernel<4, TN>); break;
            default: go(gram64_kernel<5, TN>); break;
        }
    };
    switch ((g.bn + 3) / 4) {
        case 1: rows(std::integral_constant<int, 1>{}); break;
        case 2: rows(std::integral_constant<int, 2>{}); break;
        default: rows(std::integral_constant<int, 3>{}); break;
    }
    hipLaunchKernelGGL(gram64_reduce_kernel, dim3((unsigned)(((int64_t)M * N + 63) / 64)), dim3(256), 0, s, ws, (int)g.nch,
                       M, N, C, ldc);
    QG_HIP(hipGetLastError());
}

// ------------------------------------------------------------------- Ritz update ----
constexpr int kUpdThreads = 256;
constexpr int kUpdPoints = 128;    // of a workgroup, 32 per wavefront

struct UpdateArgs {
    const double *A, *C;
    double* out;
    int64_t lda, ldo, K;
    double alpha, beta;
    int N, ldc;
};

// Out = alpha A C + beta Out (A, Out: K points x N bands, C: N x N): a wavefront's 32 points by all
// N <= 16 NT output bands in registers, as rows C^T x columns A^T, so that a lane stores two neighbouring
// points of a band.  A lane's 16 bytes of A are points 2 (l % 16) and + 1 of one band, products for the
// even and the odd points apart; a step is 8 bands of A, brought to registers two steps ahead (each value
// is read once).  The step's 8 x 16 NT coefficients lie in LDS in operand order, the next step's written
// while this one's are in use.  Bands past the last have zero coefficients.
// Products and memory share the time (512,000 points x 144 bands: floors 300 us of the matrix rate and 250
// of memory, 380 with beta): 634 us, the library's product 730.
template <int NT>
__global__ __launch_bounds__(kUpdThreads, 2) void update64_kernel(UpdateArgs g) {
    __shared__ f64x2 coef[2][NT * 64];
    const int tid = threadIdx.x, lane = tid & 63, lb = lane & 15, kg = lane >> 4;
    const int64_t p = (int64_t)blockIdx.x * kUpdPoints + (tid >> 6) * 32 + 2 * lb;
    const int steps = (g.N + 7) / 8;
    const double* src = g.A + min(p, g.K - 2);
    constexpr int SL = (NT * 64 + kUpdThreads - 1) / kUpdThreads;

    f64x2 cr[SL];
    auto fetch_c = [&](int st) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < SL; ++k) {
            const int slot = tid + k * kUpdThreads, l = slot & 63;
            const int n = 16 * (slot >> 6) + (l & 15), m = 8 * st + 2 * (l >> 4);
            const double* c = g.C + (int64_t)min(n, g.N - 1) * g.ldc;
            cr[k] = f64x2{c[min(m, g.N - 1)], c[min(m + 1, g.N - 1)]};
        }
    };
    auto put_c = [&](int st) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < SL; ++k) {
            const int slot = tid + k * kUpdThreads;
            const int l = slot & 63, n = 16 * (slot >> 6) + (l & 15), m = 8 * st + 2 * (l >> 4);
            if (NT * 64 % kUpdThreads == 0 || slot < NT * 64)
                coef[st & 1][slot] = f64x2{n < g.N && m < g.N ? cr[k].x : 0.0, n < g.N && m + 1 < g.N ? cr[k].y : 0.0};
        }
    };
    struct Pair {
        f64x2 even, odd;       // bands 2 kg and 2 kg + 1 of a step
    };
    auto fetch_a = [&](int st) __attribute__((always_inline)) {
        const int m = 8 * st + 2 * kg;
        return Pair{*reinterpret_cast<const f64x2*>(src + (int64_t)min(m, g.N - 1) * g.lda),
                    *reinterpret_cast<const f64x2*>(src + (int64_t)min(m + 1, g.N - 1) * g.lda)};
    };
    f64x4 acc[NT][2];
#pragma unroll
    for (int i = 0; i < NT; ++i) acc[i][0] = acc[i][1] = f64x4{0.0, 0.0, 0.0, 0.0};

    // one step: products of x, the bands of two steps on into y.  The coefficients are loaded first, so that
    // waiting for them does not wait for those bands.
    auto step = [&](int st, const Pair& x, Pair& y) __attribute__((always_inline)) {
        fetch_c(st + 1);
        __builtin_amdgcn_sched_barrier(0);
        y = fetch_a(st + 2);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            const f64x2 c = coef[st & 1][i * 64 + lane];
            acc[i][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(c.x, x.even.x, acc[i][0], 0, 0, 0);
            acc[i][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(c.x, x.even.y, acc[i][1], 0, 0, 0);
            acc[i][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(c.y, x.odd.x, acc[i][0], 0, 0, 0);
            acc[i][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(c.y, x.odd.y, acc[i][1], 0, 0, 0);
        }
        put_c(st + 1);
        __syncthreads();
    };
    Pair x0 = fetch_a(0), x1 = fetch_a(1), x2;
    fetch_c(0);
    put_c(0);
    __syncthreads();
    // in threes, the registers of a step by name (moving them would wait for their loads); steps past the
    // last multiply the last band by zeros
    for (int st = 0; st < steps; st += 3) {
        step(st, x0, x2);
        step(st + 1, x1, x0);
        step(st + 2, x2, x1);
    }
    if (p >= g.K) return;
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int n = 16 * i + kg + 4 * r;
            if (n >= g.N) continue;
            f64x2* o = reinterpret_cast<f64x2*>(g.out + (int64_t)n * g.ldo + p);
            f64x2 v{g.alpha * acc[i][0][r], g.alpha * acc[i][1][r]};
            if (g.beta != 0.0) {
                const f64x2 w = *o;
                v.x += g.beta * w.x;
                v.y += g.beta * w.y;
            }
            *o = v;
        }
}

// Out = alpha A C + beta Out; A, Out: N bands of K points, not overlapping.  False (nothing launched)
// where a band is not 16-byte aligned, and where the library's product is as fast: its tiles are 128 bands
// wide, these 16, so this one serves where at most 0.6 of the library's tiles are bands (17-76 and 129-153).
// Mean us of a solve's updates (with and without beta) on 512,000 points, this : library: 32 bands 65 : 115,
// 64 147 : 193, 76 197 : 227, 96 278 : 277, 112 323 : 323, 128 469 : 366, 144 556 : 689, 153 673 : 757,
// 176 1429 : 841, 192 853 : 909; on 64,000 points 64 22 : 37, 76 31 : 44, 112 49 : 62, 128 60 : 48,
// 144 69 : 95, 153 84 : 105.
bool update64(const double* A, int64_t lda, const double* C, int ldc, int64_t K, int N, double alpha, double beta,
              double* out, int64_t ldo, hipStream_t s) {
    if (K < 2 || K % 2 || lda % 2 || ldo % 2 || reinterpret_cast<uintptr_t>(A) % 16 ||
        reinterpret_cast<uintptr_t>(out) % 16)
        return false;
    if (N <= 16 || N > 153 || 10 * N > 6 * ((N + 127) / 128 * 128)) return false;
    const int64_t wgs = (K + kUpdPoints - 1) / kUpdPoints;
    if (wgs > 0x7fffffff) return false;
    const UpdateArgs a{A, C, out, lda, ldo, K, alpha, beta, N, ldc};
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3((unsigned)wgs), dim3(kUpdThreads), 0, s, a); };
    switch ((N + 15) / 16) {
        case 2: go(update64_kernel<2>); break;
        case 3: go(update64_kernel<3>); break;
        case 4: go(update64_kernel<4>); break;
        case 5: go(update64_kernel<5>); break;
        case 9: go(update64_kernel<9>); break;
        default: go(update64_kernel<10>); break;
    }
    QG_HIP(hipGetLastError());
    return true;
}

}  // namespace qg
